"""Tile sizes and orders of the per-row ring kernel: every row of a large call
has the bits of the same row in a call of at most 32 rows, whose kernel the
oracle tests cover."""
import pytest
import torch

from actune_amd import _native as N
from actune_amd.kernels import tokenwise as T

LAYERS = [T.W4A8TritonLinear, T.W8A8TritonLinear, T.W2A8TritonLinear, T.W4A4NativeLinear, T.W2A4NativeLinear, T.W8A4NativeLinear]


# the rows of the tile at each size, by layout (W8, K-major fields, row-major): below 257 and below 512 tiles of 64 x 128,
# then 128/64/128, 192/96/96, 128/64/128, 192/96/96, 64/64/64 and 96/96/96; ragged sizes end in a tile of one row or column
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(33, 130, 128), (300, 8193, 256), (1000, 4096, 128), (1000, 4097, 384), (1990, 4092, 256),
                                   (1153, 3970, 640), (512, 11008, 128), (1500, 5504, 128)])
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


# scales and biases at every alignment that the call takes: one row without and with a K split, the ring without and with
# one (its reduce with one and with four columns a thread); 130 rows of weights: no whole groups of four columns
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 144, 256), (3, 4096, 512), (1, 1024, 4096), (40, 130, 256), (300, 1024, 4096),
                                   (600, 8192, 256)])
@pytest.mark.parametrize("bias_dtype", [torch.float32, torch.bfloat16, torch.float16, None])
@pytest.mark.parametrize("layout", [N.TW_KMAJOR_W8, N.TW_ROWS_S4])
def test_scales_and_biases_at_any_alignment(layout, bias_dtype, m, n, k):
    if layout == N.TW_KMAJOR_W8:
        n = -(-n // 16) * 16
    torch.manual_seed(m + n)
    act, size = (N.TW_ACT_A8, k * n) if layout == N.TW_KMAJOR_W8 else (N.TW_ACT_A4, k // 2 * n)
    w = torch.randint(-128, 128, (size,), device="cuda:0", dtype=torch.int8)
    codes, scales = N.tokenwise_quantize(torch.randn(m, k, device="cuda:0"), 8 if act == N.TW_ACT_A8 else 4)
    work = torch.empty(N.tokenwise_workspace_bytes(m, n, k, layout, act), device="cuda:0", dtype=torch.uint8)
    outs = []
    for shift in range(3):
        gen = torch.Generator(device="cuda:0").manual_seed(9)
        values, biases = torch.rand(n, device="cuda:0", generator=gen), torch.randn(n, device="cuda:0", generator=gen)
        ws = torch.full((n + 4,), 1e30, device="cuda:0")
        ws[shift:shift + n] = values
        bias = None
        if bias_dtype is not None:
            bias = torch.full((n + 4,), 1e4, device="cuda:0", dtype=bias_dtype)
            bias[shift:shift + n] = biases.to(bias_dtype)
        out = torch.empty(m, n, device="cuda:0")
        N.tokenwise_linear(codes, act, scales, w, layout, ws[shift:shift + n], None if bias is None else bias[shift:shift + n],
                           n, k, N.TW_EPI_A8, out, work)
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    if layout == N.TW_KMAJOR_W8:
        acc = (codes.double() @ w.view(k, n).double()).float() * scales.view(-1, 1)
        want = acc * values if bias is None else (acc.double() * values.double() + biases.to(bias_dtype).double()).float()
        # one fma; the reference's sum in double rounds once more
        torch.testing.assert_close(outs[0], want, rtol=0 if bias is None else 2 ** -22, atol=0)


# the tile order of the ring: one band of tile rows or several, a last band of one, two or all eight, tiles that do not
# divide over the XCDs, up to 1024 columns (row order, but for W8 columns that end inside a line) and past them
@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(33, 1104), (190, 2064), (512, 1168), (513, 1040), (640, 1552), (1090, 1040), (600, 608),
                                 (600, 1024)])
@pytest.mark.parametrize("layer", [T.W8A8TritonLinear, T.W4A8TritonLinear, T.W2A4NativeLinear])
def test_tile_order_reaches_every_tile(layer, m, n):
    torch.manual_seed(m + n)
    lay = layer(torch.nn.Linear(256, n, device="cuda:0", dtype=torch.bfloat16))
    x = torch.randn(m, 256, device="cuda:0", dtype=torch.bfloat16)
    assert torch.equal(lay(x), torch.cat([lay(part) for part in x.split(32)]))


# row-major layouts at 257, 384 (64 x 64 tiles) and 385 tiles of 64 x 128
@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(16448, 70), (1022, 3010), (4900, 530)])
@pytest.mark.parametrize("layer", [T.W4A4NativeLinear, T.W2A4NativeLinear])
def test_row_major_tiles(layer, m, n):
    torch.manual_seed(m + n)
    lay = layer(torch.nn.Linear(128, n, device="cuda:0", dtype=torch.bfloat16))
    x = torch.randn(m, 128, device="cuda:0", dtype=torch.bfloat16)
    assert torch.equal(lay(x), torch.cat([lay(part) for part in x.split(32)]))
