"""Host-side checks of arcquant_amd.layers that need no GPU: the module imports, its callers keep the
reference's names and argument order, and building a layer from CPU weights fails loudly."""
import copy
import inspect
import os

import pytest
import torch
import torch.nn as nn

from arcquant_amd import layers


def test_qlinear_signature_follows_the_reference():
    # model/qLinearLayer.py:31-38
    params = list(inspect.signature(layers.QLinearLayer.__init__).parameters)
    assert params == ["self", "originalLayer", "select_num", "reorder_index", "out_reorder_index", "quant_type"]
    # model/qLlamaLayer.py:79
    params = list(inspect.signature(layers.reorder_quantize_x).parameters)
    assert params == ["x", "reorder_index", "select_num", "quant_type"]
    assert inspect.signature(layers.reorder_quantize_x).parameters["quant_type"].default == "NVFP4"


def test_tensor_scale_rule():
    t = torch.tensor([[-8.0, 2.0], [1.0, -0.5]])
    assert float(layers._tensor_scale(t, signed=False)) == pytest.approx(8.0 / 2688.0, rel=1e-7)   # max|x|
    assert float(layers._tensor_scale(t, signed=True)) == pytest.approx(2.0 / 2688.0, rel=1e-7)    # signed max
    assert float(layers._tensor_scale(torch.zeros(4), signed=False)) == 1.0


def test_cpu_weights_are_refused():
    lin = nn.Linear(64, 32, bias=False)
    with pytest.raises(RuntimeError, match="GPU"):
        layers.QLinearLayer(lin, 0, torch.arange(64))


def test_rotary_matches_closed_form():
    q = torch.zeros(1, 1, 3, 4)
    q[..., 0] = 1.0                                   # pairs (0, 2) and (1, 3) rotate together
    qe, _ = layers.rotary_pos_emb(q, q.clone(), beg=2)
    # position p, frequency 1 for the first pair: (1, 0) -> (cos p, sin p)
    for i, p in enumerate((2, 3, 4)):
        assert qe[0, 0, i, 0].item() == pytest.approx(torch.cos(torch.tensor(float(p))).item(), abs=1e-6)
        assert qe[0, 0, i, 2].item() == pytest.approx(torch.sin(torch.tensor(float(p))).item(), abs=1e-6)


def _quantized_linear(out_features, half, bias=None):
    """a QLinearLayer over given codes (its constructor quantizes on the GPU)"""
    lin = layers.QLinearLayer.__new__(layers.QLinearLayer)
    nn.Module.__init__(lin)
    lin.in_features, lin.out_features, lin.select_num, lin.quant_type = 2 * half, out_features, 0, "NVFP4"
    g = torch.Generator().manual_seed(out_features)
    lin.register_buffer("W", torch.randint(0, 256, (out_features, half), generator=g, dtype=torch.uint8))
    lin.register_buffer("scale_w", torch.randint(0, 256, (out_features * half // 8,), generator=g, dtype=torch.uint8))
    lin.register_buffer("scale", torch.tensor(0.5))
    if bias is None:
        lin.bias = None
    else:
        lin.register_buffer("bias", bias)
    return lin


def test_buffers_replaced_by_parameters(monkeypatch):
    """torch moves a name out of the buffers when a Parameter is assigned to it: the layers find it all the same"""
    seen = []
    monkeypatch.setattr(layers.agemm, "matmul", lambda *a, **kw: seen.append(a) or torch.zeros(2, 32, dtype=torch.bfloat16))
    monkeypatch.setattr(layers.agemm, "rmsnorm_quantize_x", lambda *a, **kw: seen.append(a) or (None, None))
    param = lambda t: nn.Parameter(t, requires_grad=False)
    x = torch.randn(1, 2, 64).to(torch.bfloat16)
    lin = _quantized_linear(32, 32, torch.ones(32, dtype=torch.bfloat16))
    quantized = (torch.zeros(2, 32, dtype=torch.uint8), torch.zeros(8, dtype=torch.uint8), 0.25, 1, 2)
    want = lin(quantized)
    for name in ("W", "scale_w", "scale", "bias"):
        setattr(lin, name, param(getattr(lin, name)))
    assert torch.equal(lin(quantized), want) and not lin._buffers
    assert all(a is b for a, b in zip((seen[1][1], seen[1][3], seen[1][4][1]), (lin.W, lin.scale_w, lin.scale)))
    norm = layers.RMSNormQuant(torch.ones(64), 1e-5, 0, torch.arange(64))
    norm.weight, norm.reorder_index = param(norm.weight), param(norm.reorder_index)
    norm(x)
    assert seen[2][1] is norm.weight and seen[2][3] is norm.reorder_index
    plain = layers.LlamaRMSNorm(torch.linspace(0.5, 1.5, 64), 1e-5)
    want = plain(x)
    plain.weight = param(plain.weight)
    assert torch.equal(plain(x), want)


def _one_behind_the_other(split, name):
    ts = [p._buffers[name] for p in split.parts]
    assert all(t.untyped_storage().nbytes() == t.numel() * t.element_size() for t in ts)
    return all(a.data_ptr() + a.numel() * a.element_size() == b.data_ptr() for a, b in zip(ts, ts[1:])) and \
        torch.equal(split._joint(name), torch.cat(ts))


def test_split_linear_joins_its_parts_again_when_moved():
    parts = [_quantized_linear(n, 64, torch.full((n,), float(n), dtype=torch.bfloat16)) for n in (96, 32, 64)]
    want = [{k: v.clone() for k, v in p.state_dict().items()} for p in parts]
    split = layers.SplitQLinear(parts)
    names = ("W", "scale_w", "bias")
    assert all(_one_behind_the_other(split, n) for n in names)
    held = split._joint("W").data_ptr()
    split.to(torch.device("cpu"))                                 # nothing moves: nothing is copied
    assert split._joint("W").data_ptr() == held
    shared = copy.deepcopy(split).share_memory()                  # not joined anew, which would take them out of the shared memory
    assert all(p.W.is_shared() for p in shared.parts) and shared._joint("W") is None
    for moved in (split._apply(torch.clone), copy.deepcopy(split), nn.Sequential(parts[1], split)._apply(torch.clone)[1]):
        assert all(_one_behind_the_other(moved, n) and moved._joint(n) is not None for n in names)
        assert all(torch.equal(v, w[k]) for p, w in zip(moved.parts, want) for k, v in p.state_dict().items())
    split.load_state_dict({k: v + 1 for k, v in split.state_dict().items()})
    assert all(_one_behind_the_other(split, n) for n in names) and torch.equal(split.parts[2].bias, want[2]["bias"] + 1)
    first = split._first["W"]
    split.parts[0].W = split.parts[0].W.clone()                   # the joint tensor goes with the pieces
    assert first() is None and split._joint("W") is None
    assert split._apply(torch.empty_like).to("meta").parts[0].W.is_meta


class _TwoNames(nn.Module):
    """its parts under two names, as the attention layers have them"""

    def __init__(self, parts):
        super().__init__()
        self.qkv_proj = layers.SplitQLinear(parts)
        self.q_proj, self.k_proj = parts


def test_split_linear_is_saved_as_its_parts_are(tmp_path):
    """the pieces of a joint allocation are tensors of their own for whoever saves them: no part carries the others' bytes, and
    safetensors finds a name for each where a part has two"""
    model = _TwoNames([_quantized_linear(96, 64), _quantized_linear(32, 64)])
    state = {k: v.clone() for k, v in model.state_dict().items()}
    torch.save(model.k_proj.state_dict(), tmp_path / "k.pt")
    assert (tmp_path / "k.pt").stat().st_size < 96 * 64
    torch.save(model, tmp_path / "model.pt")
    again = torch.load(tmp_path / "model.pt", weights_only=False)
    assert again.q_proj is again.qkv_proj.parts[0] and _one_behind_the_other(again.qkv_proj, "W")
    safetensors = pytest.importorskip("safetensors.torch")
    safetensors.save_model(model, str(tmp_path / "model.safetensors"))
    model.load_state_dict({k: torch.zeros_like(v) for k, v in state.items()})
    safetensors.load_model(model, str(tmp_path / "model.safetensors"))
    for m in (model, again):
        assert all(torch.equal(v, state[k]) for k, v in m.state_dict().items()) and _one_behind_the_other(m.qkv_proj, "scale_w")


def test_split_linear_leaves_other_parts_as_they_are(monkeypatch):
    """parts that one GEMM does not take: odd row counts (whose scale bytes would lie unaligned), Parameters, biases of two types, one
    part twice, other modules; each is built, keeps its tensors, and runs part by part"""
    class Other(nn.Module):
        select_num, out_features = 0, 8

        def forward(self, x):
            return torch.ones(x[0].shape[0], 8, dtype=torch.bfloat16)

    monkeypatch.setattr(layers.agemm, "matmul", lambda A, B, *a, **kw: torch.ones(A.shape[0], B.shape[0], dtype=torch.bfloat16))
    monkeypatch.setattr(layers.agemm, "matmul_parts", lambda *a, **kw: pytest.fail("run as one"))
    bf = lambda n, t=torch.bfloat16: torch.ones(n, dtype=t)
    held = _quantized_linear(32, 32)
    held.W = nn.Parameter(held.W, requires_grad=False)
    mixed = [_quantized_linear(32, 32, bf(32)), _quantized_linear(32, 32, bf(32, torch.float32))]
    one = _quantized_linear(32, 32)
    for parts in ([_quantized_linear(33, 32), _quantized_linear(40, 32)], [held, _quantized_linear(64, 32)], mixed,
                  [one, one], [_quantized_linear(32, 32, bf(32)), _quantized_linear(32, 32)], [Other(), one],
                  [_quantized_linear(32, 32) for _ in range(5)], [_quantized_linear(32, 32), _quantized_linear(32, 64)]):
        before = [dict(p._buffers) for p in parts]
        split = layers.SplitQLinear(parts)
        assert all(p._buffers[k] is v for p, b in zip(parts, before) for k, v in b.items())
        y = split((torch.zeros(2, 32, dtype=torch.uint8), torch.zeros(8, dtype=torch.uint8), 1.0, None, 2))
        assert y.shape == (2, split.out_features)
    assert mixed[1].bias.dtype == torch.float32


def test_split_linear_runs_part_by_part_where_a_part_is_not_itself(monkeypatch):
    """hooks, a replaced forward and tensors put in the joint ones' place: the parts are called as the modules that they are"""
    ran = []
    monkeypatch.setattr(layers.agemm, "matmul", lambda A, B, *a, **kw: ran.append("part") or torch.ones(A.shape[0], B.shape[0], dtype=torch.bfloat16))
    monkeypatch.setattr(layers.agemm, "matmul_parts", lambda A, B, *a, **kw: ran.append("one") or torch.ones(A.shape[0], B.shape[0], dtype=torch.bfloat16))
    x = (torch.zeros(2, 32, dtype=torch.uint8), torch.zeros(8, dtype=torch.uint8), 1.0, 1, 2)

    def run(change):
        split = layers.SplitQLinear([_quantized_linear(64, 32), _quantized_linear(32, 32)])
        undo = change(split)
        ran.clear()
        assert split(x).shape == (1, 2, 96)
        if undo is not None:
            undo.remove()
        return ran == ["one"]

    assert run(lambda s: None)
    assert not run(lambda s: s.parts[1].register_forward_hook(lambda *a: None))
    assert not run(lambda s: s.parts[0].register_forward_pre_hook(lambda *a: None))
    assert not run(lambda s: nn.modules.module.register_module_forward_hook(lambda *a: None))
    assert not run(lambda s: setattr(s.parts[0], "forward", s.parts[0].forward))
    assert not run(lambda s: setattr(s.parts[0], "_compiled_call_impl", s.parts[0].forward))     # what .compile() sets
    assert not run(lambda s: setattr(s.parts[1], "W", s.parts[1].W.clone()))
    assert not run(lambda s: setattr(s.parts[0], "scale_w", nn.Parameter(s.parts[0].scale_w, requires_grad=False)))
    assert not run(lambda s: setattr(s.parts[0], "scale", s.parts[0].scale.double()))
    own = layers.QLinearLayer.forward
    monkeypatch.setattr(layers.QLinearLayer, "forward", lambda self, *a, **kw: own(self, *a, **kw))
    assert not run(lambda s: None)


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
def test_split_linear_runs_part_by_part_where_that_is_faster(monkeypatch):
    """one GEMM over all parts, but for up to 80 rows where each part by itself is a stream of one tile of them and all parts together are not
    (the measured times stand at parts_pay)"""
    for M, rows, kp, one in ((300, (18944, 18944), 4352, True), (384, (18944, 18944), 4352, True), (600, (11008, 11008), 4352, True),
                             (1500, (4096, 4096, 4096), 4352, True), (65, (28672, 28672), 8320, False), (80, (28672, 28672), 8320, False),
                             (81, (28672, 28672), 8320, True), (128, (28672, 28672), 8320, True), (80, (38016, 38016), 4352, False),
                             (64, (28672, 28672), 8320, True), (80, (18944, 18944), 4352, True), (200, (18944, 18944), 4352, True),
                             (300, (14336, 14336), 4352, True), (2331, (3584, 512, 512), 3712, True), (2331, (18944, 18944), 3712, True)):
        assert layers.agemm.parts_pay(M, rows, kp, "NVFP4") == one, (M, rows)
        assert layers.agemm.parts_pay(M, rows, kp, "MXFP4")
    ran = []
    monkeypatch.setattr(layers.agemm, "matmul", lambda A, B, *a, **kw: ran.append("part") or torch.ones(A.shape[0], B.shape[0], dtype=torch.bfloat16))
    monkeypatch.setattr(layers.agemm, "matmul_parts", lambda A, B, *a, **kw: ran.append("one") or torch.ones(A.shape[0], B.shape[0], dtype=torch.bfloat16))
    split = layers.SplitQLinear([_quantized_linear(64, 32), _quantized_linear(32, 32)])
    x = (torch.zeros(2, 32, dtype=torch.uint8), torch.zeros(8, dtype=torch.uint8), 1.0, 1, 2)
    split(x)
    monkeypatch.setattr(layers.agemm, "parts_pay", lambda M, rows, kp, fmt: (M, rows, kp, fmt) != (2, (64, 32), 64, "NVFP4"))
    split(x)
    assert ran == ["one", "part", "part"]


def _mlp(projection, down, quant_type):
    """a LlamaMLP over given linears"""
    mlp = layers.LlamaMLP.__new__(layers.LlamaMLP)
    nn.Module.__init__(mlp)
    mlp.gate_up_proj, mlp.down_proj, mlp.quant_type = projection, down, quant_type
    mlp.inter, mlp.interleaved = 64, False
    mlp.register_buffer("down_reorder_index", torch.arange(64, dtype=torch.int16))
    return mlp


@pytest.mark.parametrize("split", [False, True])
def test_mlp_projection_of_another_format(monkeypatch, split):
    """gate and up in another format than the MLP's own (projections or quant_type assigned after construction), or of other sizes: the
    projection is called by itself and its output quantized in the MLP's format, never the epilogue's output with the other's scale"""
    ran = []
    epilogue = lambda *a, tensor_scale=False, **kw: ran.append("epilogue") or (("t", "scale") if tensor_scale else "t")
    monkeypatch.setattr(layers.agemm, "swiglu_halves_pay", lambda *a: True)
    monkeypatch.setattr(layers.agemm, "matmul_swiglu", epilogue)
    monkeypatch.setattr(layers.agemm, "matmul_parts", lambda A, B, *a, swiglu=False, **kw: epilogue(**kw) if swiglu else
                        ran.append("projection") or torch.zeros(A.shape[0], B.shape[0], dtype=torch.bfloat16))
    monkeypatch.setattr(layers.agemm, "matmul", lambda A, B, *a, **kw: ran.append("projection") or
                        torch.zeros(A.shape[0], B.shape[0], dtype=torch.bfloat16))
    monkeypatch.setattr(layers.agemm, "reorder_quantize_x", lambda t, *a, fmt, global_scale=None: ran.append((t, fmt, global_scale)) or ("q", "s"))
    monkeypatch.setattr(layers, "swiglu_quantize_tokens", lambda gu, inter, index, select, fmt: ran.append(("gate_up", fmt)) or
                        ("q", "s", 0.5, None, 100))

    class Down(nn.Module):
        select_num, out_features = 0, 32

        def forward(self, x, residual=None):
            return x

    def run(fmt, own, sizes=(64, 64)):
        parts = [_quantized_linear(n, 32) for n in (sizes if split else [sum(sizes)])]
        for p in parts:
            p.quant_type = fmt
        mlp = _mlp(layers.SplitQLinear(parts) if split else parts[0], Down(), own)
        ran.clear()
        return mlp((torch.zeros(100, 32, dtype=torch.uint8), torch.zeros(400, dtype=torch.uint8), 1.0, None, 100))

    assert run("NVFP4", "NVFP4")[2] == "scale" and ran == ["epilogue", ("t", "NVFP4", "scale")]
    assert run("MXFP4", "MXFP4")[2] == 1.0 and ran == ["epilogue", ("t", "MXFP4", None)]
    for fmt, own, sizes in (("NVFP4", "MXFP4", (64, 64)), ("MXFP4", "NVFP4", (64, 64)), ("NVFP4", "NVFP4", (96, 96))):
        assert run(fmt, own, sizes)[2] == 0.5 and ran == ["projection", ("gate_up", own)], (fmt, own, sizes)


def test_norm_ahead_of_a_quantizer_is_the_module(monkeypatch):
    """the norm's launch that also forms the tensor scale stands in for LlamaRMSNorm's own forward alone"""
    layer = layers.QLlamaDecoderLayer.__new__(layers.QLlamaDecoderLayer)
    nn.Module.__init__(layer)
    layer.fuse_norm, layer.quant_type = False, "NVFP4"
    norm, x = layers.LlamaRMSNorm(torch.ones(64), 1e-5), torch.randn(1, 2, 64).to(torch.bfloat16)
    monkeypatch.setattr(layers, "quantize_tokens", lambda t, *a: t)
    monkeypatch.setattr(layers.agemm, "reorder_quantize_x", lambda t, *a, **kw: ("codes", "scales"))
    monkeypatch.setattr(layers.LlamaRMSNorm, "forward_with_scale", lambda self, t: (t, 1.0))
    quantize = lambda: layer._norm_and_quantize(norm, x, None, 0)
    want = norm(x)
    assert quantize() == ("codes", "scales", 1.0, 1, 2)
    handle = norm.register_forward_hook(lambda m, i, y: y + 1)
    assert torch.equal(quantize(), want + 1)
    handle.remove()
    own = layers.LlamaRMSNorm.forward
    monkeypatch.setattr(layers.LlamaRMSNorm, "forward", lambda self, t: own(self, t) + 2)
    assert torch.equal(quantize(), want + 2)


def test_rmsnorm_of_tensors_without_memory():
    """GPU tensors that only stand for some (a shape propagation ahead of a compilation): torch's operators, not an address"""
    from torch._subclasses.fake_tensor import FakeTensorMode
    norm = layers.LlamaRMSNorm(torch.ones(64), 1e-5)
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        norm.weight = torch.empty(64, dtype=torch.bfloat16, device="cuda")
        y = norm(torch.empty(2, 3, 64, dtype=torch.bfloat16, device="cuda"))
        assert y.shape == (2, 3, 64) and y.dtype == torch.bfloat16 and y.fake_mode is mode
