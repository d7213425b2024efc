"""The wide-tile kernel (configs 3-6) and the launch plan of calls on codes
above 16 tokens, at the edges of their tiles, against the CPU oracle."""
import numpy as np
import pytest
import torch

from actune_amd import _native
from oracle import oracle as O
from tests.helpers import bits, canonical_bounds, oracle_activation, oracle_weight, seeded_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _weights(w, W, A):
    codes, scale = oracle_weight(w, W, A)
    return codes, scale, torch.from_numpy(O.pack_rows(codes, W)).to(DEV), torch.from_numpy(scale).to(DEV)


# K: one group; a ragged last quad; 17 quads (chunks of one and two quads:
# the sets of a K split walk rounds of unequal length); 19 quads, ragged
@pytest.mark.parametrize("W,A", [(2, 2), (2, 8), (4, 8), (4, 4), (8, 8), (8, 2)])
@pytest.mark.parametrize("m,n,k", [(1, 31, 64), (33, 64, 320), (65, 129, 4352), (130, 70, 4672), (257, 34, 1088)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_wide_tile_edges(W, A, m, n, k, dtype):
    x, w, b = seeded_inputs(m, k, n, seed=m + n + k, dtype=dtype, bias=True)
    packed, scales, a_codes = oracle_activation(x, A)
    codes, wscale, w_dev, ws_dev = _weights(w, W, A)
    bias = b.float() if A == 4 else b
    want = O.linear(a_codes, scales, codes, wscale, bias.float().numpy(), bounds=canonical_bounds(k // 64))
    a_dev, s_dev = torch.from_numpy(packed).to(DEV), torch.from_numpy(scales).to(DEV)
    for config in (3, 4, 5, 6, _native.CONFIG_AUTO):
        out = _native.grouped_linear(a_dev, s_dev, w_dev, ws_dev, bias.to(DEV), x, W, A, config)
        name = "bf16" if dtype == torch.bfloat16 else "f32"
        np.testing.assert_array_equal(bits(out), O.round_out(want, name), err_msg=f"config {config}")


# sibling problems of unequal N: one wide launch (grid y; the narrow ones leave
# early), or one prefill launch each
@pytest.mark.parametrize("W,A", [(4, 8), (8, 4)])
@pytest.mark.parametrize("m", [17, 40, 100, 513])
@pytest.mark.parametrize("ns,k", [((200, 1500, 37), 4096), ((3000, 2990), 1088)])
def test_planned_siblings_match_single_calls(W, A, m, ns, k):
    x, _, _ = seeded_inputs(m, k, 1, seed=m + k)
    xd = x.to(DEV)
    _, scales, a_codes = oracle_activation(x, A)
    targets, side = [], []
    for j, n in enumerate(ns):
        _, w, _ = seeded_inputs(1, k, n, seed=70 + j)
        codes, wscale, w_dev, ws_dev = _weights(w, W, A)
        targets.append((w_dev, ws_dev, None, None, W))
        side.append((codes, wscale))
    for config in (_native.CONFIG_AUTO, 4):
        outs = _native.grouped_forward_multi(xd, targets, W, A, config=config)
        for (w_dev, ws_dev, *_), (codes, wscale), out in zip(targets, side, outs):
            n = w_dev.shape[0]
            assert torch.equal(out, _native.grouped_forward(xd, w_dev, ws_dev, None, W, A, config=13)), (config, n)
            cols = np.sort(np.random.default_rng(n).choice(n, size=24, replace=False))
            want = O.linear(a_codes, scales, codes, wscale, None, bounds=canonical_bounds(k // 64), cols=cols)
            np.testing.assert_array_equal(bits(out)[:, cols], O.round_out(want, "bf16"), err_msg=f"n={n}")


# The dots mode of configs 3-6 runs the prefill kernel, so the integer dots of the wide-tile kernel are read from its fp32
# outputs: with a weight scale of 1 and an activation scale of 1 in one group and 0 in the others an output is that
# group's dot (at most 2^20: exact). Ragged quads; 17 quads (chunks of one and two quads, sets of a K split out of step).
@pytest.mark.parametrize("W,A", [(w, a) for w in (2, 4, 8) for a in (2, 4, 8)])
@pytest.mark.parametrize("m,n,k", [(35, 70, 448), (130, 33, 4352)])
def test_wide_tile_group_dots_are_exact(W, A, m, n, k):
    gen = torch.Generator().manual_seed(m + n + k)
    a_codes = torch.randint(-(1 << (A - 1)), 1 << (A - 1), (m, k), generator=gen, dtype=torch.int8)
    w_codes = torch.randint(-(1 << (W - 1)), 1 << (W - 1), (n, k), generator=gen, dtype=torch.int8)
    a_codes[0], w_codes[0] = -(1 << (A - 1)), -(1 << (W - 1))  # the largest dot
    packed_a = torch.from_numpy(O.pack_rows(a_codes.numpy(), A)).to(DEV)
    packed_w = torch.from_numpy(O.pack_rows(w_codes.numpy(), W)).to(DEV)
    ones = torch.ones(n, device=DEV)
    groups = k // 64
    for g in range(groups) if groups < 8 else (0, 3, 4, 30, 35, 63, 66, 67):
        scales = torch.zeros(m, groups, device=DEV)
        scales[:, g] = 1
        part = slice(64 * g, 64 * g + 64)
        want = (a_codes[:, part].double() @ w_codes[:, part].double().T).float()
        for config in (3, 4, 5, 6):
            out = _native.grouped_linear(packed_a, scales, packed_w, ones, None, (m, k), W, A, config, out_dtype=torch.float32)
            assert torch.equal(out.cpu(), want), (config, g)
