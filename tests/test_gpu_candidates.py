"""The calibration kernels at their edges: packed weight candidates against the
oracle's codebooks, losses and choices against numpy in float64."""
import numpy as np
import pytest
import torch

from actune_amd import _native
from oracle import oracle as O
from tests.helpers import PAIRS, seeded_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one group; a ragged pass of the row loop (2048 elements); more than one pass
@pytest.mark.parametrize("W,A", PAIRS)
@pytest.mark.parametrize("n,k", [(1, 64), (3, 2048), (5, 2112), (2, 6400)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_weight_candidates_match_the_codebooks(W, A, n, k, dtype):
    _, w, _ = seeded_inputs(1, k, n, seed=n + k, dtype=dtype)
    w[0, :64] = 0
    ratios = torch.tensor([1.0, 0.9, 0.75])
    packed, scales = _native.weight_candidates(w.to(DEV), ratios.to(DEV), W, A)
    for r, ratio in enumerate(ratios.tolist()):
        codes, scale = O.weight_codes(w.float().numpy(), W, A, ratio, gpu_division=True)
        np.testing.assert_array_equal(packed[r * n:(r + 1) * n].cpu().numpy(), O.pack_rows(codes, W))
        np.testing.assert_array_equal(scales[r * n:(r + 1) * n].cpu().numpy(), scale)


@pytest.mark.parametrize("m,n,r", [(1, 1, 1), (17, 63, 3), (127, 65, 2), (129, 200, 9)])
def test_candidate_select(m, n, r):
    g = torch.Generator().manual_seed(m + n + r)
    y, ref = torch.randn(m, r * n, generator=g), torch.randn(m, n, generator=g)
    ratios = torch.linspace(1, 0.5, r)
    best, chosen = torch.full((n,), float("inf")), torch.full((n,), 0.25)
    best[0] = 0.0  # nothing improves on it
    y[:, n - 1] = float("nan")
    bd, cd = best.to(DEV), chosen.to(DEV)
    loss = _native.candidate_select(y.to(DEV), ref.to(DEV), ratios.to(DEV), bd, cd).cpu().numpy()
    # squares in fp32, sums in fp64: one rounding of the square, one of the mean
    d = (y.reshape(m, r, n) - ref[:, None, :]).numpy()
    want = np.square(d).astype(np.float64).mean(0)
    np.testing.assert_allclose(loss, want, rtol=2 ** -22)
    for j in range(n):
        b, c = float(best[j]), float(chosen[j])
        for i in range(r):
            if loss[i, j] < b:
                b, c = float(loss[i, j]), float(ratios[i])
        assert float(bd[j]) == b and float(cd[j]) == c
