"""The operators' native host path (csrc/arcq_host.cpp) against the general route it stands in front of: what it does not take it
leaves alone (None, nothing raised, nothing launched), and what it takes gives the same bits."""
import pytest
import torch

import recipes


def test_what_is_not_taken_on_the_cpu():
    """CPU tensors, wrong types and counts, subclasses, active modes: None, and the operators raise what they always raised"""
    from arcquant_amd import _lib, agemm
    h = _lib.host
    x, idx = torch.zeros(4, 64, dtype=torch.bfloat16), torch.arange(64, dtype=torch.int16)
    codes, sf = torch.zeros(4, 32, dtype=torch.uint8), torch.zeros(16, dtype=torch.uint8)
    assert h.quantize(0, x, None, 0.0, idx, 0, "NVFP4", None) is None
    assert h.quantize(0, "x", None, 0.0, idx, 0, "NVFP4", None) is None
    assert h.quantize(0, x, None, 0.0, idx, 1 << 80, "NVFP4", None) is None
    assert h.quantize(2, x, x[0], 1e-5, idx, 0, "other", None) is None
    assert h.swiglu_quantize(x, x, idx, 0, "NVFP4", "absmax") is None
    assert h.matmul(codes, codes, sf, sf, 1.0, None, None) is None
    assert h.decode_step(x, 1, x, x, idx, codes, codes, idx, idx, idx, 0) is None
    with pytest.raises(TypeError):
        h.matmul(codes)
    with pytest.raises(RuntimeError, match="must be on the GPU"):
        agemm.reorder_quantize_x(x, idx, 0)
    with pytest.raises(RuntimeError, match="must be on the GPU"):
        agemm.matmul(codes, codes, sf, sf, 1.0)


@pytest.mark.parametrize("how", ["missing", "another torch", "not a library"])
def test_without_the_native_host_path(monkeypatch, tmp_path, how):
    """no _arcq_host.so, one of another torch, one that does not load: a warning, and every operator by its general route"""
    from arcquant_amd import _lib, agemm
    assert _lib.host_lib_is_current()
    path = tmp_path / "_arcq_host.so"
    if how == "another torch":
        with open(_lib.HOST_LIB_PATH, "rb") as f:
            path.write_bytes(f.read().replace(_lib.host_lib_mark(), b"x" * len(_lib.host_lib_mark())))
    elif how == "not a library":
        path.write_bytes(_lib.host_lib_mark())
    monkeypatch.setattr(_lib, "HOST_LIB_PATH", str(path))
    h = _lib._Host()
    with pytest.warns(RuntimeWarning, match="general route"):
        assert h.matmul() is None
    assert h.quantize(1, 2) is None and h.swiglu_quantize() is None and h.decode_step() is None
    monkeypatch.setattr(agemm, "_host", h)
    codes, sf = torch.zeros(4, 32, dtype=torch.uint8), torch.zeros(16, dtype=torch.uint8)
    with pytest.raises(RuntimeError, match="must be on the GPU"):
        agemm.matmul(codes, codes, sf, sf, 1.0)
    with pytest.raises(AttributeError):
        h.nothing


def _general(monkeypatch, call):
    """the call by the general route"""
    from arcquant_amd import _lib, agemm

    class Nothing:
        def __getattr__(self, name):
            return lambda *a: None

    with monkeypatch.context() as m:
        m.setattr(agemm, "_host", Nothing())
        m.setattr(_lib, "host", Nothing())
        return call()


def _same(a, b):
    a, b = (t if isinstance(t, tuple) else (t,) for t in (a, b))
    return len(a) == len(b) and all(torch.equal(u, v) and u.dtype == v.dtype and u.shape == v.shape for u, v in zip(a, b))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["NVFP4", "MXFP4"])
def test_same_bits_as_the_general_route(monkeypatch, fmt):
    """every form of the arguments, each also in a form that only the general route takes"""
    from arcquant_amd import _lib, agemm
    M, N, K, S = 33, 256, 1024, 128
    x, w = recipes.activations(M, K, seed=1).cuda(), recipes.weights(N, K, seed=2).cuda()
    gam, idx = recipes.gamma(K, seed=3).cuda(), recipes.reorder_index(x.cpu()).cuda()
    two = torch.cat([x, x.flip(0)], dim=1)                        # strided halves
    gs = torch.tensor(0.37, device="cuda")
    calls = [lambda: agemm.rmsnorm_quantize_x(x, gam, 1e-5, idx, S, fmt=fmt),
             lambda: agemm.rmsnorm_quantize_x(x, torch.nn.Parameter(gam, requires_grad=False), 1e-5, idx, S, fmt=fmt, global_scale=0.5),
             lambda: agemm.reorder_quantize_x(x, idx, S, fmt=fmt, global_scale=gs),
             lambda: agemm.reorder_quantize_x(x, idx, S, fmt=fmt, global_scale=gs.double()),   # converted by the general route
             lambda: agemm.reorder_quantize_x(x, idx, S, fmt=fmt, global_scale="absmax"),
             lambda: agemm.reorder_quantize_x(x[:0], idx, S, fmt=fmt, global_scale="absmax"),
             lambda: agemm.reorder_quantize_w(w, idx, S, fmt=fmt, global_scale=3),
             lambda: agemm.swiglu_quantize_x(two[:, :K], two[:, K:], idx, S, fmt=fmt, global_scale="absmax"),
             lambda: agemm.swiglu_quantize_x(two[:1, :K], two[:1, K:], idx, S, fmt=fmt, global_scale=gs)]
    (a, sfa), (b, sfb) = agemm.reorder_quantize_x(x, idx, S, fmt=fmt), agemm.reorder_quantize_w(w, idx, S, fmt=fmt)
    res = recipes.activations(M, N, seed=4).cuda()
    calls += [lambda: agemm.matmul(a, b, sfa, sfb, 0.3),
              lambda: agemm.matmul(a, b, sfa, sfb, (gs, gs), fmt=fmt, residual=res),
              lambda: agemm.matmul(a, b, sfa, sfb, (0.1, gs), fmt=fmt),
              lambda: agemm.matmul(a, b, sfa, sfb, (0.1, 0.3), fmt=fmt),
              lambda: agemm.matmul(a, b, sfa, sfb, [gs, gs.cpu()], fmt=fmt)]                   # a list, a CPU scalar
    for i, call in enumerate(calls):
        assert _same(call(), _general(monkeypatch, call)), i
    with pytest.raises(RuntimeError):
        agemm.reorder_quantize_x(x, idx[:-32], S, fmt=fmt)
    with pytest.raises(RuntimeError):
        agemm.reorder_quantize_x(x, idx, 3, fmt=fmt)
    with pytest.raises(RuntimeError, match="residual"):
        agemm.matmul(a, b, sfa, sfb, 1.0, residual=res[:-1])
    assert _lib.host.quantize(0, x.t(), None, 0.0, idx, S, fmt, None) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_decode_step_same_bits(monkeypatch, dtype):
    from arcquant_amd.kv_cache import MultiLayerPagedKVCache4Bit
    g = torch.Generator(device="cuda").manual_seed(5)
    qkv = torch.randn(3, (8 + 2 * 2) * 128, generator=g, device="cuda").to(dtype)
    kv = torch.randn(2, 3, 37, 2, 128, generator=g, device="cuda").to(dtype)

    def call():
        cache = MultiLayerPagedKVCache4Bit(3, 16, 64, "cuda", 1, 2, 128, dtype=dtype)
        cache.update(kv[0], kv[1], 0)
        return cache.decode_step(qkv, 8, 0), cache.pages, cache.scales

    assert _same(call(), _general(monkeypatch, call))
