"""Tile sizes and orders of the per-row ring kernel: every row of a large call
has the bits of the same row in a call of at most 32 rows, whose kernel the
oracle tests cover."""
import pytest
import torch

from actune_amd import _native as N
from actune_amd.kernels import tokenwise as T

LAYERS = [T.W4A8TritonLinear, T.W8A8TritonLinear, T.W2A8TritonLinear, T.W4A4NativeLinear, T.W2A4NativeLinear, T.W8A4NativeLinear]


# tiles of 64 x 128: below 257, below 512, then 64, 96 (192 rows for W8), 128 rows, and a last tile of one row and column
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(33, 130, 128), (300, 8193, 256), (1000, 4096, 128), (1000, 4097, 384), (1990, 4092, 256),
                                   (1153, 3970, 640)])
@pytest.mark.parametrize("layer", LAYERS)
def test_rows_do_not_depend_on_the_tile(layer, m, n, k):
    torch.manual_seed(m + n)
    lin = torch.nn.Linear(k, n, bias=n % 2 == 0, device="cuda:0", dtype=torch.float32)
    lay = layer(lin)
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        x = torch.randn(m, k, device="cuda:0").to(dtype)
        assert torch.equal(lay(x), torch.cat([lay(part) for part in x.split(32)]))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(5, 64, 128), (70, 256, 2048), (1000, 4096, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_misaligned_outputs(dtype, m, n, k):
    torch.manual_seed(1)
    w = torch.randint(-127, 128, (k, n), device="cuda:0", dtype=torch.int8)
    ws, x = torch.rand(n, device="cuda:0"), torch.randn(m, k, device="cuda:0")
    codes, scales = N.tokenwise_quantize(x, 8)
    size = N.tokenwise_workspace_bytes(m, n, k, N.TW_KMAJOR_W8, N.TW_ACT_A8)
    outs = []
    for shift in (0, 1):
        buf = torch.full((m * n + 2,), 7.0, device="cuda:0", dtype=dtype)
        out = buf[shift:shift + m * n].view(m, n)
        work = torch.empty(size, device="cuda:0", dtype=torch.uint8) if size else None
        N.tokenwise_linear(codes, N.TW_ACT_A8, scales, w, N.TW_KMAJOR_W8, ws, None, n, k, N.TW_EPI_A8, out, work)
        outs.append(out)
        assert torch.equal(buf[m * n + shift:], torch.full((2 - shift,), 7.0, device="cuda:0", dtype=dtype))
        assert shift == 0 or buf[0] == 7.0
    want = (codes.double() @ w.double()).float() * scales.view(-1, 1) * ws
    assert torch.equal(outs[0], want.to(dtype)) and torch.equal(outs[1], outs[0])
