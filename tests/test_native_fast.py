"""The native call path (csrc/binding.cpp) against the ctypes path it stands
in for: None for whatever it does not take, equal results for what it does."""
import pytest
import torch

from actune_amd import _native as N

DEV = "cuda:0"


def test_host_tensors_are_left_to_the_ctypes_path():
    f = N.fast()
    x, w, ws = torch.zeros(2, 64, dtype=torch.bfloat16), torch.zeros(4, 32, dtype=torch.uint8), torch.zeros(4)
    codes, scales = torch.zeros(2, 64, dtype=torch.uint8), torch.zeros(2, 1)
    assert f.quantize_groups(x, 8, None) is None
    assert f.quantize_gated(x, x, 0, 8, None) is None
    assert f.grouped_linear(codes, scales, w, ws, None, 2, 64, 0, 4, 8, -1) is None
    assert f.grouped_forward(x, w, ws, None, 4, 8, None, -1) is None
    assert f.grouped_forward_multi(x, [(w, ws, None, None)], 4, 8, None, -1) is None
    assert f.tokenwise_quantize(x, 8) is None
    assert f.tokenwise_linear(codes.view(torch.int8), 0, torch.zeros(2), w, 1, ws, None, 4, 64, 0, 0) is None
    assert f.tokenwise_linear_x(x, w, 1, ws, None, 4, 64, 0) is None
    assert f.tokenwise_decode(x[:1], [w], [None], [ws], [None], 1, 4, 64, 0) is None
    with pytest.raises(RuntimeError, match="CUDA required"):
        N.grouped_forward(x, w, ws, None, 4, 8)


def _layer(n, k, w, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    packed = torch.randint(0, 256, (n, k * w // 8), device=DEV, dtype=torch.uint8, generator=g)
    return packed, torch.rand(n, device=DEV, generator=g) * 0.01


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,n,k,w,a", [(1, 37, 64, 4, 8), (3, 512, 4096, 8, 4), (17, 130, 192, 2, 2), (130, 96, 1088, 4, 4),
                                       (0, 16, 64, 4, 8)])
def test_equals_the_ctypes_path(dtype, m, n, k, w, a):
    packed, ws = _layer(n, k, w)
    x = torch.randn(m, k, device=DEV).to(dtype)
    for bias in (None, torch.randn(n, device=DEV).to(dtype), torch.randn(n, device=DEV)):
        for scale in (None, (torch.rand(k, device=DEV) + 0.5).to(dtype)):
            want = N.grouped_forward(x, packed, ws, bias, w, a, scale, out=torch.empty(m, n, device=DEV, dtype=dtype))
            got = N.fast().grouped_forward(x, packed, ws, bias, w, a, scale, -1)
            assert got is not None and torch.equal(got, want) and got.dtype == dtype
            both = N.fast().grouped_forward_multi(x, [(packed, ws, bias, None, w)] * 2, w, a, scale, -1)
            assert all(torch.equal(o, want) for o in both)
    codes, scales = N.fast().quantize_groups(x, a, None)
    empty = torch.empty_like(codes)
    assert torch.equal(codes, N.quantize_groups(x, a, packed=empty)[0])
    for out in (torch.bfloat16, torch.float32):
        want = N.grouped_linear(codes, scales, packed, ws, None, (m, k), w, a, out=torch.empty(m, n, device=DEV, dtype=out),
                                out_dtype=out)
        assert torch.equal(N.fast().grouped_linear(codes, scales, packed, ws, None, m, k, N.DTYPE_CODES[out], w, a, -1), want)


@pytest.mark.gpu
def test_what_it_does_not_take_behaves_as_before():
    packed, ws = _layer(48, 128, 4)
    base = torch.randn(4, 136, device=DEV, dtype=torch.bfloat16)
    rows = torch.randn(4 * 128 + 1, device=DEV, dtype=torch.bfloat16)[1:].reshape(4, 128)  # contiguous, misaligned
    f = N.fast()
    assert f.grouped_forward(rows, packed, ws, None, 4, 8, None, -1) is None
    assert torch.equal(N.grouped_forward(rows, packed, ws, None, 4, 8), N.grouped_forward(rows.clone(), packed, ws, None, 4, 8))
    assert f.grouped_forward(base[:, :128], packed, ws, None, 4, 8, None, -1) is None
    for bad, error, match in (
            (lambda: N.grouped_forward(base[:, :128], packed, ws, None, 4, 8), RuntimeError, "contiguous"),
            (lambda: N.grouped_forward(rows, packed[:, :32], ws, None, 4, 8), RuntimeError, "packed shape mismatch"),
            (lambda: N.grouped_forward(rows, packed, ws[:4], None, 4, 8), RuntimeError, "scale shape mismatch"),
            (lambda: N.grouped_forward(rows, packed, ws.double(), None, 4, 8), RuntimeError, "float scales"),
            (lambda: N.grouped_forward(rows, packed, ws, ws.long(), 4, 8), RuntimeError, "float scales/bias"),
            (lambda: N.grouped_forward(rows.clone(), packed, ws, None, 4, 3), ValueError, "integer width"),
            (lambda: N.grouped_forward(rows.clone(), packed, ws, None, 4, 8, config=99), ValueError, "configuration"),
            (lambda: N.tokenwise_quantize(rows.clone(), 2), ValueError, "A8 or A4")):
        with pytest.raises(error, match=match):
            bad()


def test_arguments_of_another_kind_are_left_to_the_ctypes_path():
    """Targets may be any sequence of sequences, and an argument of a type that the native call path does not take
    reaches the checks that name what is wrong."""
    f = N.fast()
    x, w, ws = torch.zeros(2, 64, dtype=torch.bfloat16), torch.zeros(4, 32, dtype=torch.uint8), torch.zeros(4)
    for targets in ([[w, ws, None, None]], ((w, ws, None, None),), [(w, ws, None)], [None], [(None, ws, None, None)],
                    [(w, ws, 1, None)], [(w, ws, None, None, 4.0)], None, 5):
        assert f.grouped_forward_multi(x, targets, 4, 8, None, -1) is None
    for call in (lambda: f.quantize_groups(None, 8, None), lambda: f.quantize_groups(x, 8.0, None),
                 lambda: f.quantize_gated(x, None, 0, 8, None),
                 lambda: f.grouped_linear(None, ws, w, ws, None, 2, 64, 0, 4, 8, -1),
                 lambda: f.grouped_linear(w, ws, w, ws, None, 2.0, 64, 0, 4, 8, -1),
                 lambda: f.grouped_forward(x, None, ws, None, 4, 8, None, -1),
                 lambda: f.grouped_forward(x, w, ws, None, 4, 8, None, 2 ** 40), lambda: f.tokenwise_quantize(x, "8"),
                 lambda: f.tokenwise_linear(None, 0, ws, w, 1, ws, None, 4, 64, 0, 0),
                 lambda: f.tokenwise_linear_x(x, None, 1, ws, None, 4, 64, 0),
                 lambda: f.tokenwise_decode(x[:1], [None], [None], [ws], [None], 1, 4, 64, 0)):
        assert call() is None
    with pytest.raises(RuntimeError, match="CUDA required"):
        N.grouped_forward_multi(x, [[w, ws, None, None]], 4, 8)
    with pytest.raises(RuntimeError, match="CUDA required"):
        N.grouped_forward_multi(x, [[None, ws, None, None]], 4, 8)


@pytest.mark.gpu
def test_target_sequences_and_empty_outputs():
    packed, ws = _layer(48, 128, 4)
    x = torch.randn(4, 128, device=DEV, dtype=torch.bfloat16)
    want = N.grouped_forward(x, packed, ws, None, 4, 8)
    for targets in ([[packed, ws, None, None]], ((packed, ws, None, None),), ([packed, ws, None, None, 4],)):
        assert torch.equal(N.fast().grouped_forward_multi(x, targets, 4, 8, None, -1)[0], want)
        assert torch.equal(N.grouped_forward_multi(x, targets, 4, 8)[0], want)
    codes, scales = N.quantize_groups(x, 8)
    assert torch.equal(N.grouped_linear(codes, scales, packed, ws, None, iter((4, 128)), 4, 8), want)
    with pytest.raises(RuntimeError, match="invalid dimensions"):
        N.grouped_linear(codes, scales, packed[:0], ws[:0], None, x, 4, 8)


@pytest.mark.parametrize("kind", ["missing", "unloadable", "other torch"])
def test_calls_run_without_the_extension(kind, monkeypatch, tmp_path):
    """Without a native call path that loads (none built, or one of another torch) the ctypes path serves every call,
    after one warning."""
    path = tmp_path / "_actune_fast.so"
    if kind == "unloadable":
        path.write_bytes(b"not a library")
    elif kind == "other torch":
        path = N.FAST_PATH
        monkeypatch.setattr(N.torch, "__version__", "1.0.0")
    monkeypatch.setattr(N, "FAST_PATH", path)
    monkeypatch.setattr(N, "_FAST", None)
    x, w, ws = torch.zeros(2, 64, dtype=torch.bfloat16), torch.zeros(4, 32, dtype=torch.uint8), torch.zeros(4)
    with pytest.warns(RuntimeWarning, match="native call path"):
        f = N.fast()
    assert f is N.fast()
    assert f.grouped_forward(x, w, ws, None, 4, 8, None, -1) is None and f.tokenwise_quantize(x, 8) is None
    with pytest.raises(RuntimeError, match="CUDA required"):
        N.grouped_forward(x, w, ws, None, 4, 8)


@pytest.mark.gpu
def test_results_without_the_extension(monkeypatch, tmp_path):
    packed, scales = _layer(48, 128, 4)
    rows = torch.randn(4, 128, device=DEV, dtype=torch.bfloat16)
    want = N.grouped_forward(rows, packed, scales, None, 4, 8)
    monkeypatch.setattr(N, "FAST_PATH", tmp_path / "missing.so")
    monkeypatch.setattr(N, "_FAST", None)
    with pytest.warns(RuntimeWarning, match="native call path"):
        assert torch.equal(N.grouped_forward(rows, packed, scales, None, 4, 8), want)
    codes, s = N.quantize_groups(rows, 8)
    assert torch.equal(N.grouped_linear(codes, s, packed, scales, None, rows, 4, 8), want)


def test_the_extension_is_built_again_for_another_torch(monkeypatch, tmp_path):
    from actune_amd import build as B
    lib = tmp_path / B.BINDING_LIB.name
    lib.write_bytes(b"")
    monkeypatch.setattr(B, "BINDING_LIB", lib)
    monkeypatch.setattr(B, "BINDING_STAMP", tmp_path / "stamp")
    assert B._binding_stale()  # of an unknown torch
    B.BINDING_STAMP.write_text(B._binding_target())
    assert not B._binding_stale()
    B.BINDING_STAMP.write_text(B._binding_target().replace(torch.__version__, "1.0.0"))
    assert B._binding_stale()


@pytest.mark.gpu
def test_a_first_decode_launches_once(monkeypatch):
    from actune_amd.kernels import tokenwise as T
    layer = T.W4A8TritonLinear(torch.nn.Linear(256, 128, device=DEV, dtype=torch.bfloat16))
    x = torch.randn(1, 256, device=DEV, dtype=torch.bfloat16)
    launches = []

    class Counting:
        def __getattr__(self, name):
            launches.append(name)
            return getattr(fast, name)

    fast = N.fast()
    monkeypatch.setattr(N, "_FAST", Counting())
    first = layer(x)
    assert launches.count("tokenwise_decode") == 1
    assert torch.equal(first, layer(x)) and launches.count("tokenwise_decode") == 2
    with pytest.raises(RuntimeError):
        T.graph_decode_linear(layer, x, layer.packed_weight, None, layer.weight_scale[16:32], layer.bias)
    assert T.decode_workspace_summary(layer)["decode_graph_plan_count"] == 1
