"""GPU parity of the augmented-K FP4 GEMM: within 1e-2 relative Frobenius error of
dequantize-then-matmul in fp32/fp64 (the stated tolerance; bf16 output rounding alone is
~2e-3), on seeded inputs quantized by the GPU quantizers (themselves bit-exact, see
test_gpu_quantize.py)."""
import os

import numpy as np
import pytest
import torch

import recipes

pytestmark = pytest.mark.gpu
FMTS = ["NVFP4", "MXFP4"]
TOL = 1e-2


@pytest.fixture(scope="module")
def agemm():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from arcquant_amd import agemm as m
    return m


def rel_fro(got, want):
    got, want = got.double(), want.double()
    return float((got - want).norm() / want.norm())


def oracle_dq(oracle, codes, sf, fmt):
    """fp32 values of codes + scale bytes from the CPU oracle's dequantizer, back on the GPU (the
    library's own dequantizer stays out of the GEMM checks)"""
    c = codes.cpu().numpy()
    return torch.from_numpy(oracle.dequantize(c, sf.cpu().numpy().reshape(c.shape[0], -1), fmt)).cuda()


def assert_kernel(M, N, Kp, fmt, kernel, n_seg=0, swiglu=0):
    """The dispatch takes this kernel for the problem (a kernel forced through the environment aside)"""
    from arcquant_amd import _lib
    if "ARCQ_GEMM_KERNEL" not in os.environ:
        assert _lib.lib().arcq_gemm_kernel(M, N, Kp, _lib.FORMATS[fmt], n_seg, swiglu) == kernel


def assert_route(M, N, Kp, fmt, route):
    from arcquant_amd import _lib
    if "ARCQ_GEMM_KERNEL" not in os.environ:
        assert _lib.lib().arcq_gemm_route(M, N, Kp, _lib.FORMATS[fmt], 0, 0) == route


def quantized_pair(agemm, M, N, K, S, fmt, seed):
    x = recipes.activations(M, K, seed=seed)
    w = recipes.weights(N, K, seed=seed + 1)
    idx = recipes.reorder_index(x)
    gx, gw = recipes.tensor_scale(x, fmt), recipes.tensor_scale(w, fmt)
    xd, wd, idxd = x.cuda(), w.cuda(), idx.cuda()
    a, sfa = agemm.reorder_quantize_x(xd, idxd, S, fmt=fmt, global_scale=gx)
    b, sfb = agemm.reorder_quantize_w(wd, idxd, S, fmt=fmt, global_scale=gw)
    return (x, w, idx, gx, gw), (a, sfa, b, sfb)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M,N,K,S", [(1, 128, 256, 64), (16, 256, 512, 0), (37, 200, 1024, 128), (128, 128, 4096, 256),
                                     (130, 384, 448, 64)])
def test_matmul_vs_oracle_fp64(agemm, oracle, fmt, M, N, K, S):
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, fmt, seed=40 + M + N)
    print(f"matmul {fmt} M={M} N={N} K={K} S={S}", flush=True)
    y = agemm.matmul(a, b, sfa, sfb, gx * gw)
    assert y.shape == (M, N) and y.dtype == torch.bfloat16
    G = 16 if fmt == "NVFP4" else 32
    want = oracle.matmul(a.cpu().numpy(), sfa.cpu().numpy().reshape(M, -1), b.cpu().numpy(),
                         sfb.cpu().numpy().reshape(N, -1), fmt, alpha=gx * gw)
    assert sfa.numel() == M * (K + S) // G
    err = rel_fro(y.cpu().float(), torch.from_numpy(want))
    assert err < TOL, err
    # elementwise: bf16 rounding of an fp32-accumulated sum
    assert torch.allclose(y.cpu().float(), torch.from_numpy(want), rtol=2 ** -7, atol=1e-3 * float(np.abs(want).max()))


@pytest.mark.parametrize("fmt", FMTS)
def test_matmul_scale_argument_forms(agemm, fmt):
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, 48, 256, 512, 64, fmt, seed=5)
    y0 = agemm.matmul(a, b, sfa, sfb, gx * gw)
    y1 = agemm.matmul(a, b, sfa, sfb, torch.tensor(gx * gw))                       # CPU tensor, like .item()
    y2 = agemm.matmul(a, b, sfa, sfb, torch.tensor(gx * gw, device="cuda"))        # device scalar, no sync
    y3 = agemm.matmul(a, b, sfa, sfb, (torch.tensor(gx, device="cuda"), torch.tensor(gw, device="cuda")))
    assert torch.equal(y0, y1)
    for y in (y2, y3):
        assert rel_fro(y.float(), y0.float()) < 1e-2 and torch.allclose(y.float(), y0.float(), rtol=2 ** -6, atol=0)
    with pytest.raises(RuntimeError):
        agemm.matmul(a, b[:, :-32], sfa, sfb, 1.0)
    with pytest.raises(RuntimeError):
        agemm.matmul(a.float(), b, sfa, sfb, 1.0)


@pytest.mark.parametrize("fmt", FMTS)
def test_identity_weights_recover_activations(agemm, oracle, fmt):
    """W = I on the reordered channels: Y = d * (dq(x) main + residual) with d = dq(1.0) (1.0 for
    MXFP4, 1.03125 for NVFP4 whose 1/6 block scale rounds to 0.171875): at most two exact
    products per output, so the fp32 sum is exact and the bf16 result is determined."""
    M, K, S = 64, 256, 64
    x = recipes.activations(M, K, seed=12)
    idx = torch.arange(K).to(torch.int16)
    w = torch.eye(K).to(torch.bfloat16)
    a, sfa = agemm.reorder_quantize_x(x.cuda(), idx.cuda(), S, fmt=fmt)
    b, sfb = agemm.reorder_quantize_w(w.cuda(), idx.cuda(), S, fmt=fmt)
    y = agemm.matmul(a, b, sfa, sfb, 1.0).cpu().float()
    dq = oracle.quantize_x(x, idx, S, fmt, 1.0, want_dq=True)["dq"].astype(np.float64)
    d = {"NVFP4": 1.03125, "MXFP4": 1.0}[fmt]
    assert np.all(np.diag(oracle.quantize_w(w, idx, 0, fmt, 1.0, want_dq=True)["dq"]) == d)
    folded = dq[:, :K].copy()
    folded[:, K - S:] += dq[:, K:]
    want = torch.from_numpy(folded * d).to(torch.bfloat16).float()
    assert torch.equal(y, want)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M,N,K,S", [(512, 4096, 4096, 256), (2048, 6144, 4096, 256), (256, 4096, 14336, 256),
                                     (512, 6144, 1024, 128), (448, 6200, 768, 256), (128, 28672, 1024, 256),
                                     (100, 4096, 4096, 256), (384, 4100, 8192, 128)])
def test_matmul_llama_shapes_vs_torch_fp32(agemm, oracle, fmt, M, N, K, S):
    """Benchmark shapes, and shapes of one round of workgroups (at most 256 tiles of 128x64 or 128x128, also
    ragged and with K' % 256 == 128, and K cut into slices for a few hundred rows): compare with torch's
    fp32 matmul on the GPU of the operands as the CPU oracle dequantizes them."""
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, fmt, seed=3)
    print(f"matmul {fmt} M={M} N={N} K={K} S={S}", flush=True)
    y = agemm.matmul(a, b, sfa, sfb, gx * gw)
    prev = torch.backends.cuda.matmul.allow_tf32
    torch.backends.cuda.matmul.allow_tf32 = False
    try:
        want = (oracle_dq(oracle, a, sfa, fmt) @ oracle_dq(oracle, b, sfb, fmt).T) * (gx * gw)
    finally:
        torch.backends.cuda.matmul.allow_tf32 = prev
    err = rel_fro(y.float(), want)
    assert err < TOL, err
    # and the whole scheme tracks the unquantized product
    y_true = x.cuda().float() @ w.cuda().float().T
    assert rel_fro(y.float(), y_true) < 0.2


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M", [1, 5, 16, 17, 32, 48, 64])
@pytest.mark.parametrize("N,K,S", [(6144, 4096, 256), (202, 384, 0), (4100, 1024, 128), (4100, 8192, 128),
                                   (8324, 1024, 256), (8450, 768, 256), (16500, 1024, 128)])
def test_matmul_decode_batches(agemm, oracle, fmt, M, N, K, S):
    """M <= 64 (decode batches) at a benchmark shape and at shapes whose N is not a multiple of the
    16-row strips or of the 4-wide stores: against torch's fp32 matmul of the dequantized operands,
    and, row by row, against the same call on a 128-row batch that contains these rows (another
    kernel computes that one).  The long-K shape and the wider batches of the benchmark shape take the
    split-K path (partial tiles in a workspace, added by a second launch): a repeated call must give
    the same bits.  The two wide shapes take the 128x64 tiles with a ragged last workgroup, one of them
    with N % 4 != 0."""
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, 128, N, K, S, fmt, seed=11)
    print(f"matmul decode {fmt} M={M} N={N} K={K} S={S}", flush=True)
    a_m = a[:M].contiguous()
    sfa_m = sfa.view(128, -1)[:M].contiguous().view(-1)
    y = agemm.matmul(a_m, b, sfa_m, sfb, gx * gw)
    assert y.shape == (M, N)
    assert torch.equal(y, agemm.matmul(a_m, b, sfa_m, sfb, gx * gw))
    prev = torch.backends.cuda.matmul.allow_tf32
    torch.backends.cuda.matmul.allow_tf32 = False
    try:
        want = (oracle_dq(oracle, a_m, sfa_m, fmt) @ oracle_dq(oracle, b, sfb, fmt).T) * (gx * gw)
    finally:
        torch.backends.cuda.matmul.allow_tf32 = prev
    assert rel_fro(y.float(), want) < TOL
    y_big = agemm.matmul(a, b, sfa, sfb, gx * gw)[:M]
    # same operands, fp32 accumulation in another order, one bf16 rounding each
    assert rel_fro(y.float(), y_big.float()) < 4e-3


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M,N,K,S", [
    (1, 4096, 4096, 256),      # skinny, eight waves
    (48, 6144, 4096, 256),     # split-K: the second launch adds
    (64, 4100, 8192, 128),     # split-K with a ragged last tile
    (33, 28672, 1024, 128),    # tiled 128x64
    (40, 8324, 1024, 256),     # tiled 128x64, ragged last workgroup
    (300, 1000, 2048, 128),    # tiled, ragged M and N: transposed epilogue and the per-element one
    (512, 6144, 1024, 128),    # one round of 128x128 tiles
    (200, 4096, 8448, 256),    # a few hundred rows, long K: slices
    (1100, 1024, 1024, 0),     # 256x256 tiles (MXFP4 cost model may take smaller ones) with a ragged M
    (130, 384, 448, 64),       # K' % 128 != 0: direct kernels
    (5, 202, 384, 0),          # N % 4 != 0: scalar stores
])
def test_matmul_with_residual_equals_separate_add(agemm, fmt, M, N, K, S):
    """arcq_matmul_add through every epilogue: the same bits as matmul(...) + residual in bf16."""
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, fmt, seed=90 + M)
    g = torch.Generator().manual_seed(M * 7 + N)
    r = (torch.randn(M, N, generator=g) * 0.7).to(torch.bfloat16).cuda()
    print(f"matmul + residual {fmt} M={M} N={N} K={K} S={S}", flush=True)
    y = agemm.matmul(a, b, sfa, sfb, gx * gw)
    z = agemm.matmul(a, b, sfa, sfb, gx * gw, residual=r)
    assert torch.equal(z, y + r)
    with pytest.raises(RuntimeError):
        agemm.matmul(a, b, sfa, sfb, gx * gw, residual=r[:, :-1].contiguous())


def oracle_dq(oracle, q, sf, fmt):
    """fp32 values of quantized rows from the CPU oracle's dequantizer, on the GPU"""
    rows = q.shape[0]
    return torch.from_numpy(oracle.dequantize(q.cpu().numpy(), sf.cpu().numpy().reshape(rows, -1), fmt)).cuda()


def test_matmul_operand_of_more_than_4_gib(agemm, oracle):
    """An activation operand of 4.35 GB (2 000 000 rows of K' = 4352): the eight-wave MXFP4 kernels address rows
    with 32-bit byte offsets, so the dispatch must hand this one to the kernels with 64-bit addresses.  Random
    codes and scale bytes near 2^0; first, middle and last rows against the product of the operands as the CPU
    oracle dequantizes them."""
    M, N, Kp = 2_000_000, 512, 4352
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randint(0, 256, (M, Kp // 2), dtype=torch.uint8, device="cuda", generator=g)
    b = torch.randint(0, 256, (N, Kp // 2), dtype=torch.uint8, device="cuda", generator=g)
    sfa = torch.randint(124, 130, (M * (Kp // 32),), dtype=torch.uint8, device="cuda", generator=g)
    sfb = torch.randint(124, 130, (N * (Kp // 32),), dtype=torch.uint8, device="cuda", generator=g)
    assert a.numel() >= 1 << 32
    print(f"matmul MXFP4 M={M} N={N} K'={Kp}: operand of {a.numel()} bytes", flush=True)
    c = agemm.matmul(a, b, sfa, sfb, 1.0, fmt="MXFP4")
    db = oracle_dq(oracle, b, sfb, "MXFP4")
    prev = torch.backends.cuda.matmul.allow_tf32
    torch.backends.cuda.matmul.allow_tf32 = False
    for r0 in (0, M // 2 + 3, 1_999_000, M - 64):
        da = oracle_dq(oracle, a[r0:r0 + 64], sfa.view(M, -1)[r0:r0 + 64], "MXFP4")
        want = da @ db.T
        err = float((c[r0:r0 + 64].float() - want).norm() / want.norm())
        assert err < 5e-3, (r0, err)
    torch.backends.cuda.matmul.allow_tf32 = prev
    del a, c
    torch.cuda.empty_cache()


@pytest.mark.parametrize("seed", [1, 7])
def test_matmul_random_shapes(agemm, oracle, seed):
    """Forty random (format, M, N, K, select_num) problems per seed, sizes around the tile edges of every
    kernel the dispatch knows: quantize both operands, multiply, compare the whole output with the fp32 product
    of the operands as the CPU oracle dequantizes them (the rounding of the bf16 output bounds the error)."""
    import random
    rnd = random.Random(seed)
    done = 0
    while done < 40:
        fmt = rnd.choice(FMTS)
        M = rnd.choice([1, 2, 7, 16, 17, 31, 32, 33, 63, 64, 65, 100, 127, 128, 129, 200, 255, 256, 257, 300, 511, 512, 513, 700,
                        1000, 1024, 1500, 2048, 2100, 3000])
        N = rnd.choice([8, 16, 24, 64, 100, 128, 136, 200, 256, 264, 500, 512, 520, 1000, 1024, 2048, 2056, 4096, 4104, 6144,
                        8192, 8200, 16384, 28672])
        K = rnd.choice([64, 128, 192, 256, 320, 384, 448, 512, 640, 768, 896, 1024, 1152, 2048, 3072, 4096])
        S = min(rnd.choice([0, 64, 128, 256]), K)
        if M * N > 12_000_000 or N * K > 60_000_000:
            continue
        x = recipes.activations(M, K, seed=seed * 1000 + done, outlier_frac=0.01, outlier_gain=30.0).cuda()
        w = recipes.weights(N, K, seed=seed * 2000 + done).cuda()
        idx = torch.randperm(K, generator=torch.Generator().manual_seed(done)).to(torch.int16).cuda()
        print(f"random shape {done}: {fmt} M={M} N={N} K={K} S={S}", flush=True)
        a, sfa = agemm.reorder_quantize_x(x, idx, S, fmt=fmt)
        b, sfb = agemm.reorder_quantize_w(w, idx, S, fmt=fmt)
        y = agemm.matmul(a, b, sfa, sfb, 1.0, fmt=fmt)
        want = oracle_dq(oracle, a, sfa, fmt) @ oracle_dq(oracle, b, sfb, fmt).T
        err = float((y.float() - want).norm() / max(1e-20, float(want.norm())))
        assert err < 6e-3, (fmt, M, N, K, S, err)
        done += 1


@pytest.mark.parametrize("M,N,K,S", [(300, 28672, 512, 128), (8300, 1030, 448, 64), (257, 33000, 1152, 256),
                                     (6017, 2200, 1024, 128), (2048, 4352, 768, 0)])
def test_nvfp4_one_operand_decoded_ahead(agemm, oracle, M, N, K, S):
    """NVFP4 problems beyond one round of 256x128 tiles: the operand with fewer rows is decoded to fp16 ahead of the
    GEMM (rows of either operand ending inside a 256-row tile, N not a multiple of 8, K' from two pairs of steps on,
    with and without a residual).  Products are exact and sums fp32, so against fp32 matmul of the oracle's values only
    the bf16 rounding (2^-9 per element, 1.7e-3 in norm) and the order of the sum remain."""
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, "NVFP4", seed=17)
    assert_kernel(M, N, K + S, "NVFP4", 168)
    want = oracle_dq(oracle, a, sfa, "NVFP4") @ oracle_dq(oracle, b, sfb, "NVFP4").T * (gx * gw)
    scale = (torch.tensor(gx, device="cuda"), torch.tensor(gw, device="cuda"))
    y = agemm.matmul(a, b, sfa, sfb, scale)
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul(a, b, sfa, sfb, scale, residual=res), y + res)


@pytest.mark.parametrize("M,N,K,S", [(3900, 4090, 8192, 128), (4096, 4096, 8192, 0), (4000, 4095, 8320, 128), (4000, 4095, 8448, 128)])
def test_mxfp4_long_rows(agemm, oracle, M, N, K, S):
    """MXFP4 with K' of 8192 and more on problems that fill the chip with 256x256 tiles: the ping-pong kernel, with K' a
    multiple of 256 and not (half a stage at the end; the window of scale bytes that ends with the row is shifted by 12, 0, 8
    and 4 bytes), rows of either operand ending inside a tile, N odd and not a multiple of 8.  Exact products, fp32 sums: the bf16 rounding (1.7e-3 in norm) and the sum's order remain."""
    assert_kernel(M, N, K + S, "MXFP4", 88)
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, "MXFP4", seed=23)
    want = oracle_dq(oracle, a, sfa, "MXFP4") @ oracle_dq(oracle, b, sfb, "MXFP4").T * 0.5
    y = agemm.matmul(a, b, sfa, sfb, 0.5, fmt="MXFP4")
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul(a, b, sfa, sfb, 0.5, fmt="MXFP4", residual=res), y + res)


@pytest.mark.parametrize("form", ["plain", "residual", "swiglu", "grouped"])
def test_gemm_without_memory_for_the_workspace(agemm, monkeypatch, form):
    """No memory for the decoded operand: the kernels that need none compute the same product (the sum in another order, one
    bf16 rounding), and nothing is raised."""
    M, N, K = 2100, 6400, 512
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, 128, "NVFP4", seed=31)
    assert_kernel(M, N, K + 128, "NVFP4", 168, int(form == "grouped"), int(form == "swiglu"))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    seg = torch.tensor([0, M], dtype=torch.int32, device="cuda")
    call = {"plain": lambda: agemm.matmul(a, b, sfa, sfb, gx * gw),
            "residual": lambda: agemm.matmul(a, b, sfa, sfb, gx * gw, residual=res),
            "swiglu": lambda: agemm.matmul_swiglu(a, b, sfa, sfb, gx * gw),
            "grouped": lambda: agemm.grouped_matmul(a, b[None], sfa, sfb, seg)}[form]
    want, refused, empty = call(), [], torch.empty

    def full(*size, **kw):
        if kw.get("dtype") is torch.uint8:
            refused.append(size)
            raise torch.OutOfMemoryError("no memory for the workspace")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", full)
    got = call()
    monkeypatch.undo()
    assert len(refused) == 1 or "ARCQ_GEMM_KERNEL" in os.environ
    # a sum in another order moves fewer than one value in a hundred to the neighbouring bf16 number (2^-8 of it at most)
    assert rel_fro(got.float(), want.float()) < 1e-3


def test_gemm_with_memory_for_the_smaller_workspace(agemm, monkeypatch):
    """Memory for the decoded operand, but not for the sums of the last round's parts beside it: the kernel that takes that much,
    bit for bit, and not the ones that take none"""
    import ctypes
    from arcquant_amd import _lib
    L, (M, N, kp) = _lib.lib(), (4100, 4096, 8192)
    g = torch.Generator(device="cuda").manual_seed(9)
    codes = lambda rows: (torch.randint(0, 256, (rows, kp // 2), generator=g, device="cuda", dtype=torch.uint8),
                          torch.randint(60, 90, (rows * (kp // 16),), generator=g, device="cuda", dtype=torch.uint8))
    (a, sfa), (b, sfb) = codes(M), codes(N)
    sizes = [L.arcq_gemm_scratch_bytes(M, N, kp, 0, 0), L.arcq_gemm_workspace_bytes(M, N, kp, 0, 0)]
    if "ARCQ_GEMM_KERNEL" in os.environ:
        pytest.skip("another kernel is forced")
    assert sizes[0] > sizes[1] > 0
    want = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    work = torch.empty(sizes[1], dtype=torch.uint8, device="cuda")
    args = _lib.GemmArgs(a.data_ptr(), sfa.data_ptr(), b.data_ptr(), sfb.data_ptr(), M, N, kp, 0, 2.0 ** -9, 0, None, None, None, want.data_ptr(),
                         None, 0, None, work.data_ptr(), sizes[1])
    assert L.arcq_gemm(args, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    asked, empty = [], torch.empty

    def scarce(*size, **kw):
        if kw.get("dtype") is torch.uint8:
            asked.append(size[0])
            if size[0] > sizes[1]:
                raise torch.OutOfMemoryError("no memory for the larger workspace")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", scarce)
    got = agemm.matmul(a, b, sfa, sfb, 2.0 ** -9)
    monkeypatch.undo()
    assert asked == sizes and torch.equal(got, want)


def test_gemm_workspace_too_small(agemm):
    """A workspace one byte short of what arcq_gemm_workspace_bytes says is not used: the result of the call without one,
    bit for bit, and not a byte of it written."""
    import ctypes
    from arcquant_amd import _lib
    M, N, K = 2100, 6400, 512
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, 128, "NVFP4", seed=31)
    L, Kp = _lib.lib(), K + 128
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    work = torch.full((2 * M * Kp,), 77, dtype=torch.uint8, device="cuda")
    out = []
    for nbytes in (0, 2 * M * Kp - 1):
        c = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        args = _lib.GemmArgs(a.data_ptr(), sfa.data_ptr(), b.data_ptr(), sfb.data_ptr(), M, N, Kp, 0, 0.5, 0, None, None, None,
                             c.data_ptr(), None, 0, None, work.data_ptr() if nbytes else None, nbytes)
        assert L.arcq_gemm(args, stream) == 0
        out.append(c)
    assert torch.equal(*out) and bool((work == 77).all())


@pytest.mark.parametrize("N", [24, 101, 4096, 4104, 8192, 12286, 14336, 18944, 20482, 28672, 33000])
@pytest.mark.parametrize("M,K,S", [(5, 512, 0), (16, 640, 0), (17, 1024, 128), (32, 832, 64), (33, 1024, 256), (48, 2048, 128), (64, 576, 64)])
def test_nvfp4_decode_batches(agemm, oracle, M, N, K, S):
    """NVFP4 decode batches, one pass over the weights: every number of 16-row tiles of either operand, the last ones partly
    empty, N not a multiple of 4, K' from one step on, ending inside a step and inside a 16-byte window of scale bytes.  Exact
    products and fp32 sums: the bf16 rounding (2^-9 per element, 1.7e-3 in norm) and the sum's order remain."""
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, "NVFP4", seed=41)
    want = oracle_dq(oracle, a, sfa, "NVFP4") @ oracle_dq(oracle, b, sfb, "NVFP4").T * (gx * gw)
    scale = (torch.tensor(gx, device="cuda"), torch.tensor(gw, device="cuda"))
    y = agemm.matmul(a, b, sfa, sfb, scale)
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul(a, b, sfa, sfb, scale, residual=res), y + res)
    if N % 16 == 0:
        t, gs = agemm.matmul_swiglu(a, b, sfa, sfb, scale, tensor_scale=True)
        h = torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2]
        assert torch.equal(t, h) and float(gs) == float(h.abs().max().float().cpu() / torch.tensor(2688.0))


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M,rows", [(1, (512, 64, 32)), (17, (4096, 32, 520)), (64, (96, 100)), (64, (4096,)), (100, (3584, 512, 512)), (512, (1024, 2048, 512, 512)),
                                    (300, (256, 260)), (700, (2048, 2048)), (2100, (6400, 1000))])
def test_matmul_parts(agemm, M, rows, fmt):
    """Several linears as one GEMM: the columns of each under its own scale (in every epilogue: decode batches, split-K, tiles
    inside C and across its edge, parts that end inside a tile), against a GEMM per part; the bias exactly as a bf16 add.
    Another tile sums in another order: one bf16 rounding at most, in fewer than one value in a hundred."""
    N, K, S = sum(rows), 1024, 128
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, fmt, seed=51)
    dgx = torch.tensor(gx, device="cuda")
    scales = [torch.tensor(0.5 + k, device="cuda") for k in range(len(rows))]
    y = agemm.matmul_parts(a, b, sfa, sfb, dgx, rows, scales, fmt=fmt)
    at, ones = 0, []
    for n, s in zip(rows, scales):
        ones.append(agemm.matmul(a, b[at:at + n], sfa, sfb.view(N, -1)[at:at + n].reshape(-1), (dgx, s), fmt=fmt))
        at += n
    one = torch.cat(ones, dim=1)
    assert rel_fro(y.float(), one.float()) < 1e-3
    assert torch.allclose(y.float(), one.float(), rtol=2 ** -7, atol=1e-4 * float(one.float().abs().max()))
    bias = torch.randn(N, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul_parts(a, b, sfa, sfb, dgx, rows, scales, fmt=fmt, bias=bias), y + bias)
    with pytest.raises(RuntimeError):
        agemm.matmul_parts(a, b, sfa, sfb, dgx, (N - 16, 16), scales[:1] * 2, fmt=fmt)


@pytest.mark.parametrize("M,N,kp,counts", [(4100, 4096, 8192, None), (3000, 6144, 8320, None), (6144, 3000, 8320, None), (5000, 4090, 10240, None),
                                           (4096, 4352, 9088, [900, 2100, 0, 96, 1000]), (4096, 4360, 8192, [1, 4095])])
def test_nvfp4_last_round_cut(agemm, oracle, M, N, kp, counts):
    """NVFP4 problems of a few rounds of tiles with a long K': the last round's tiles shared by workgroups along K, either operand
    decoded ahead, rows and columns ending inside a tile, experts without rows; against the kernels without a workspace (the
    sum in another order: one bf16 rounding at most) and the 64-bit product of some rows."""
    import ctypes
    from arcquant_amd import _lib
    L, E = _lib.lib(), len(counts) if counts else 0
    g = torch.Generator(device="cuda").manual_seed(9)
    codes = lambda rows: (torch.randint(0, 256, (rows, kp // 2), generator=g, device="cuda", dtype=torch.uint8),
                          torch.randint(60, 90, (rows * (kp // 16),), generator=g, device="cuda", dtype=torch.uint8))
    (a, sfa), (b, sfb) = codes(M), codes(N * max(E, 1))
    seg = torch.tensor([0] + list(np.cumsum(counts)), dtype=torch.int32, device="cuda") if counts else None
    res = torch.randn(M, N, generator=g, device="cuda").to(torch.bfloat16)
    need = L.arcq_gemm_scratch_bytes(M, N, kp, 0, E)
    if "ARCQ_GEMM_KERNEL" not in os.environ:
        assert need >= 512 * 65536 * 4
    out = []
    for residual in (None, res):
        for nbytes in (need, 0):
            c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
            work = torch.full((nbytes,), 0xff, dtype=torch.uint8, device="cuda") if nbytes else None
            args = _lib.GemmArgs(a.data_ptr(), sfa.data_ptr(), b.data_ptr(), sfb.data_ptr(), M, N, kp, 0, 2.0 ** -9, 0, None, None,
                                 None if residual is None else residual.data_ptr(), c.data_ptr(), None if seg is None else seg.data_ptr(), E,
                                 None, None if work is None else work.data_ptr(), nbytes)
            assert L.arcq_gemm(args, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
            out.append(c)
    assert rel_fro(out[0].float(), out[1].float()) < 1e-3
    assert torch.equal(out[2], out[0] + res)
    rows = torch.tensor([0, 255, 256, M // 2, M - 1])
    e = torch.bucketize(rows, seg.cpu()[1:].long(), right=True) if counts else torch.zeros(5, dtype=torch.long)
    da = oracle_dq(oracle, a[rows.cuda()], sfa.view(M, -1)[rows.cuda()].reshape(-1), "NVFP4")
    for i in range(5):
        w = slice(int(e[i]) * N, (int(e[i]) + 1) * N)
        want = da[i].double() @ oracle_dq(oracle, b[w], sfb.view(-1, kp // 16)[w].reshape(-1), "NVFP4").double().T * 2.0 ** -9
        assert rel_fro(out[0][rows[i]].float(), want) < 2.5e-3


@pytest.mark.parametrize("M,N,K,S", [(65, 1000, 512, 0), (128, 6144, 576, 64), (100, 4096, 1024, 0), (200, 6144, 640, 0), (256, 4096, 1024, 128), (333, 6145, 1152, 0),
                                     (333, 4096, 8192, 128), (400, 6144, 1024, 128), (400, 4100, 2048, 0), (80, 28672, 512, 128), (777, 6144, 1024, 128),
                                     (1000, 4608, 1024, 0), (112, 20500, 640, 0), (512, 4096, 8192, 0), (1024, 3000, 512, 0)])
def test_nvfp4_a_few_hundred_rows(agemm, oracle, M, N, K, S):
    """NVFP4 problems of 65 to 1024 rows: shapes of up to 112 rows per workgroup in the place of the plan's tiles, rows and
    columns ending inside them; exact products and fp32 sums as for decode batches."""
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, "NVFP4", seed=71)
    want = oracle_dq(oracle, a, sfa, "NVFP4") @ oracle_dq(oracle, b, sfb, "NVFP4").T * (gx * gw)
    scale = (torch.tensor(gx, device="cuda"), torch.tensor(gw, device="cuda"))
    y = agemm.matmul(a, b, sfa, sfb, scale)
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul(a, b, sfa, sfb, scale, residual=res), y + res)


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
@pytest.mark.parametrize("M,N,kp,shape", [
    (65, 4101, 512, 0), (83, 6145, 512, 1), (79, 6145, 640, 2), (137, 6145, 1152, 3), (197, 4101, 1152, 4), (197, 6145, 2176, 5),
    (902, 4101, 640, 6), (449, 4101, 2176, 7), (323, 6145, 4352, 8),                   # N % 4 != 0
    (65, 256, 512, 0), (100, 8192, 1152, 1), (144, 4096, 4352, 2), (113, 6144, 1152, 0), (520, 2048, 640, 4), (65, 18944, 512, 5), (161, 18944, 640, 6),
    (333, 6144, 4352, 7), (83, 18944, 640, 7), (65, 28672, 512, 8), (333, 4096, 8192, 3)])
def test_nvfp4_every_shape_of_a_few_hundred_rows(agemm, oracle, M, N, kp, shape):
    """Each shape of the kernel for 65 to 1024 rows, on problems that are given to it: rows and columns ending inside its tile, columns
    that are no multiple of four, plain and with a residual; exact products and fp32 sums."""
    from arcquant_amd import _lib
    assert _lib.lib().arcq_gemm_route(M, N, kp, 0, 0, 0) == 16 + shape
    S = 64 if kp % 256 else 0
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, kp - S, S, "NVFP4", seed=83)
    want = oracle_dq(oracle, a, sfa, "NVFP4") @ oracle_dq(oracle, b, sfb, "NVFP4").T * (gx * gw)
    scale = (torch.tensor(gx, device="cuda"), torch.tensor(gw, device="cuda"))
    y = agemm.matmul(a, b, sfa, sfb, scale)
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul(a, b, sfa, sfb, scale, residual=res), y + res)


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
@pytest.mark.parametrize("M,N,kp,route", [
    (5, 4096, 10240, 3), (5, 4096, 10112, 0), (16, 2048, 10240, 3), (16, 2048, 10112, 0), (9, 4096, 8192, 3), (17, 2048, 4096, 3),
    (17, 2048, 3968, 0), (5, 8192, 4096, 3), (5, 8192, 3968, 0), (1, 12288, 2560, 3), (1, 12288, 2432, 0), (4, 28672, 512, 3),
    (64, 1024, 12288, 0), (64, 1024, 12160, 3), (64, 4096, 16384, 0), (64, 37888, 1408, 0), (64, 28672, 512, 3)])
def test_nvfp4_decode_batches_at_the_edges_of_the_stream(agemm, oracle, M, N, kp, route):
    """both sides of the lines between the stream of the weights and the kernels that begin and end sooner"""
    from arcquant_amd import _lib
    assert _lib.lib().arcq_gemm_route(M, N, kp, 0, 0, 0) == route
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, kp - 64, 64, "NVFP4", seed=85)
    want = oracle_dq(oracle, a, sfa, "NVFP4") @ oracle_dq(oracle, b, sfb, "NVFP4").T * (gx * gw)
    y = agemm.matmul(a, b, sfa, sfb, gx * gw)
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))


@pytest.mark.parametrize("M,N,kp", [(64, 1024, 12288), (64, 2048, 16384), (130, 256, 8320)])
def test_nvfp4_captured_without_scratch(agemm, oracle, M, N, kp):
    """a plan with slices of K on a stream that is captured and was not prepared: there is no memory for their sums, and a kernel
    that needs none has the problem (M = 130: the plan's slices, or a shape that needs none, by their times)"""
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, kp - 64, 64, "NVFP4", seed=87)
    want = oracle_dq(oracle, a, sfa, "NVFP4") @ oracle_dq(oracle, b, sfb, "NVFP4").T * (gx * gw)
    if "ARCQ_GEMM_KERNEL" in os.environ:
        pytest.skip("another kernel is forced")
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        y = agemm.matmul(a, b, sfa, sfb, gx * gw)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert rel_fro(y.float(), want) < 2.5e-3
        assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
@pytest.mark.parametrize("M,N,kp,decoded", [
    (70, 49160, 512, 70), (128, 49152, 640, 128),                                   # tiles of 128 activation rows
    (300, 22100, 512, 300), (385, 20480, 768, 385), (192, 33000, 640, 192),         # of 192, the last one of 108, 1 and 192
    (385, 24576, 768, 385),                                                          # of 256, the last one of 129
    (3900, 4096, 512, 3900), (3960, 4090, 640, 3960), (4020, 4096, 512, 4020), (4090, 4096, 512, 4090),   # of 256: 60, 120, 180, 250
    (3841, 4096, 512, 3841), (5331, 3584, 640, 5331), (4096, 3584, 512, 3584)])     # more rows than weights: either one decoded
def test_nvfp4_decoded_ahead_tiles(agemm, oracle, M, N, kp, decoded):
    """Every tile of the kernel on one operand decoded ahead, and every smaller one that the last rows take: against the kernels
    without a workspace (exact products, sums in another order: one bf16 rounding at most), the residual exactly, and some rows
    against the 64-bit product."""
    import ctypes
    from arcquant_amd import _lib
    L = _lib.lib()
    assert L.arcq_gemm_route(M, N, kp, 0, 0, 0) == 1 and L.arcq_gemm_workspace_bytes(M, N, kp, 0, 0) == 2 * decoded * kp
    g = torch.Generator(device="cuda").manual_seed(M + N)
    codes = lambda rows: (torch.randint(0, 256, (rows, kp // 2), generator=g, device="cuda", dtype=torch.uint8),
                          torch.randint(60, 90, (rows * (kp // 16),), generator=g, device="cuda", dtype=torch.uint8))
    (a, sfa), (b, sfb) = codes(M), codes(N)
    res = torch.randn(M, N, generator=g, device="cuda").to(torch.bfloat16)
    out = []
    for residual, nbytes in ((None, 2 * decoded * kp), (None, 0), (res, 2 * decoded * kp)):
        c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        work = torch.full((nbytes,), 0xff, dtype=torch.uint8, device="cuda") if nbytes else None
        args = _lib.GemmArgs(a.data_ptr(), sfa.data_ptr(), b.data_ptr(), sfb.data_ptr(), M, N, kp, 0, 2.0 ** -9, 0, None, None,
                             None if residual is None else residual.data_ptr(), c.data_ptr(), None, 0, None,
                             None if work is None else work.data_ptr(), nbytes)
        assert L.arcq_gemm(args, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        out.append(c)
    assert rel_fro(out[0].float(), out[1].float()) < 1e-3
    assert torch.allclose(out[0].float(), out[1].float(), rtol=2 ** -7, atol=1e-4 * float(out[1].float().abs().max()))
    assert torch.equal(out[2], out[0] + res)
    rows = torch.tensor([0, min(127, M - 1), M // 2, M - 1])
    da = oracle_dq(oracle, a[rows.cuda()], sfa.view(M, -1)[rows.cuda()].reshape(-1), "NVFP4").double()
    want = da @ oracle_dq(oracle, b, sfb, "NVFP4").double().T * 2.0 ** -9
    assert rel_fro(out[0][rows.cuda()].float(), want) < 2.5e-3


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
@pytest.mark.parametrize("counts", [[830, 40, 2130], [1000, 950, 0, 1122], [2304, 1, 191, 1088]])
def test_nvfp4_decoded_ahead_tiles_of_experts(agemm, counts):
    """experts that end in a tile of 64, 128, 192 or 256 rows: each as a GEMM of its own (other tiles: one bf16 rounding at most),
    and the fused SwiGLU epilogue's bits and maxima from the plain one's output"""
    E, M, N, kp = len(counts), sum(counts), 6160, 512
    g = torch.Generator(device="cuda").manual_seed(M)
    codes = lambda rows: (torch.randint(0, 256, (rows, kp // 2), generator=g, device="cuda", dtype=torch.uint8),
                          torch.randint(40, 60, (rows * (kp // 16),), generator=g, device="cuda", dtype=torch.uint8))
    (a, sfa), (b, sfb) = codes(M), codes(E * N)
    b, seg = b.view(E, N, -1), torch.tensor([0] + list(np.cumsum(counts)), dtype=torch.int32, device="cuda")
    y = agemm.grouped_matmul(a, b, sfa, sfb, seg)
    t, scales = agemm.grouped_matmul_swiglu(a, b, sfa, sfb, seg, tensor_scale=True)
    assert torch.equal(t, torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2])
    at = 0
    for e, n in enumerate(counts):
        if n == 0:
            assert float(scales[e]) == 1.0
            continue
        rows = slice(at, at + n)
        one = agemm.matmul(a[rows], b[e], sfa.view(M, -1)[rows].reshape(-1), sfb.view(E, -1)[e], 1.0)
        assert rel_fro(y[rows].float(), one.float()) < 1e-3
        assert float(scales[e]) == float(t[rows].abs().max().float().cpu() / torch.tensor(2688.0))
        at += n


@pytest.mark.parametrize("M,N,K,S", [(4096, 4352, 512, 0), (4096, 4352, 512, 128), (4352, 4096, 2048, 0), (2048, 16384, 3328, 256), (4096, 4352, 2048, 256)])
def test_mxfp4_persistent_workgroups(agemm, oracle, M, N, K, S):
    """MXFP4 on whole 256x256 tiles, more than one for every CU, with a short K': one workgroup per CU walks its tiles; the bf16 rounding and
    the fp32 sum's order remain."""
    assert_kernel(M, N, K + S, "MXFP4", 84)
    assert_route(M, N, K + S, "MXFP4", 0)
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, "MXFP4", seed=37)
    want = oracle_dq(oracle, a, sfa, "MXFP4") @ oracle_dq(oracle, b, sfb, "MXFP4").T * 0.5
    y = agemm.matmul(a, b, sfa, sfb, 0.5, fmt="MXFP4")
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul(a, b, sfa, sfb, 0.5, fmt="MXFP4", residual=res), y + res)


@pytest.mark.parametrize("M,N,K,S", [(2300, 4600, 2048, 128), (2304, 4608, 2048, 256), (2049, 4601, 2304, 128), (2300, 4610, 2304, 256),
                                     (2304, 4608, 2048, 128), (4096, 4352, 2304, 256)])
def test_mxfp4_rows_of_medium_length(agemm, oracle, M, N, K, S):
    """MXFP4 on 256x256 tiles from K' = 2176 on: the ping-pong kernel (2304 excepted) with an odd and an even number of stages, the last one
    whole and half; the bf16 rounding (1.7e-3 in norm) and the fp32 sum's order remain."""
    assert_kernel(M, N, K + S, "MXFP4", 84)
    assert_route(M, N, K + S, "MXFP4", 0 if K + S == 2304 else 4)
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, S, "MXFP4", seed=29)
    want = oracle_dq(oracle, a, sfa, "MXFP4") @ oracle_dq(oracle, b, sfb, "MXFP4").T * 0.5
    y = agemm.matmul(a, b, sfa, sfb, 0.5, fmt="MXFP4")
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul(a, b, sfa, sfb, 0.5, fmt="MXFP4", residual=res), y + res)


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
@pytest.mark.parametrize("fmt,M,N,kp", [
    ("NVFP4", 70, 49184, 512), ("NVFP4", 300, 22112, 640), ("NVFP4", 3900, 4096, 512), ("NVFP4", 3960, 4064, 512), ("NVFP4", 257, 43968, 512),
    ("NVFP4", 8192, 3616, 512), ("NVFP4", 4100, 4096, 8192), ("NVFP4", 6144, 3008, 8320),          # the weights decoded; the last round cut
    ("MXFP4", 2300, 4608, 2176), ("MXFP4", 2304, 4640, 2304), ("MXFP4", 4000, 3936, 8320)])
def test_swiglu_of_weights_as_they_are(agemm, fmt, M, N, kp):
    """gate rows and then up rows with the SwiGLU epilogue: the bits of the GEMM followed by silu and multiply in bf16, and the tensor scale
    of the result; N / 2 a multiple of 16 that ends inside a tile, one scale for both and one each (parts), special activations
    (5.9375 and beyond 87, where the epilogue leaves its estimate) among the gates.  Where the last round of tiles is cut along K, other
    columns are in it: one bf16 rounding (2^-9, 1.7e-3 in norm) of a few gates and ups."""
    from arcquant_amd import _lib
    assert agemm.swiglu_halves_pay(M, N, kp, fmt)
    cut = _lib.lib().arcq_gemm_route(M, N, kp, _lib.FORMATS[fmt], 0, 0) == 2
    g, F, nv = torch.Generator(device="cuda").manual_seed(M + N), N // 2, fmt == "NVFP4"
    lo, hi, G = (30, 60, 16) if nv else (118, 124, 32)
    codes = lambda rows: (torch.randint(0, 256, (rows, kp // 2), generator=g, device="cuda", dtype=torch.uint8),
                          torch.randint(lo, hi, (rows * (kp // G),), generator=g, device="cuda", dtype=torch.uint8))
    (a, sfa), (b, sfb) = codes(M), codes(N)
    y = agemm.matmul(a, b, sfa, sfb, 1.0, fmt=fmt)
    big = 100.0 / float(y[:, :F].float().abs().max())      # gates of up to 100 in magnitude, most of them small
    y = agemm.matmul(a, b, sfa, sfb, big, fmt=fmt)
    want = torch.nn.functional.silu(y[:, :F]) * y[:, F:]
    t, scale = agemm.matmul_swiglu(a, b, sfa, sfb, big, fmt=fmt, tensor_scale=True, halves=True)
    assert rel_fro(t.float(), want.float()) < 1.7e-3 if cut else torch.equal(t, want)
    assert float(scale) == float(t.abs().max().float().cpu() / torch.tensor(2688.0))
    assert torch.equal(agemm.matmul_swiglu(a, b, sfa, sfb, big, fmt=fmt, halves=True), t)
    scales = [torch.tensor(s, device="cuda") for s in (big, 0.5 * big)]
    one = torch.tensor(1.0, device="cuda")
    if F % 32 == 0:
        y = agemm.matmul_parts(a, b, sfa, sfb, one, (F, F), scales, fmt=fmt)
        want = torch.nn.functional.silu(y[:, :F]) * y[:, F:]
        t, scale = agemm.matmul_parts(a, b, sfa, sfb, one, (F, F), scales, fmt=fmt, swiglu=True, tensor_scale=True)
        assert rel_fro(t.float(), want.float()) < 1.7e-3 if cut else torch.equal(t, want)
        assert float(scale) == float(t.abs().max().float().cpu() / torch.tensor(2688.0))


def test_swiglu_of_weights_as_they_are_for_others(agemm, monkeypatch):
    """problems that have no such epilogue are refused, and without memory for the scratch there is no result to be had"""
    import ctypes
    from arcquant_amd import _lib
    L = _lib.lib()
    for M, N, kp, f in ((64, 28672, 4352, 0), (16, 28672, 4352, 1), (4096, 28672, 1152, 1), (4096, 28688, 4352, 0), (4096, 28672, 448, 0)):
        assert L.arcq_gemm_swiglu_halves(M, N, kp, f) == 0
        ok = 0x1000
        args = _lib.GemmArgs(ok, ok, ok, ok, M, N, kp, f, 1.0, _lib.SWIGLU_HALVES, None, None, None, ok, None, 0, None, None, 0)
        assert L.arcq_gemm(args, None) == 2
    if "ARCQ_GEMM_KERNEL" in os.environ:
        pytest.skip("another kernel is forced")
    M, N, K = 2100, 6400, 512
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, K, 128, "NVFP4", seed=31)
    few, scale, one = 64, torch.tensor(1.0, device="cuda"), torch.tensor(1.0, device="cuda")
    with pytest.raises(RuntimeError):
        agemm.matmul_swiglu(a[:few], b, sfa.view(M, -1)[:few].reshape(-1), sfb, 1.0, tensor_scale=True, halves=True)
    with pytest.raises(RuntimeError):
        agemm.matmul_parts(a[:few], b, sfa.view(M, -1)[:few].reshape(-1), sfb, one, (N // 2, N // 2), (scale, scale), fmt="NVFP4", swiglu=True)
    empty = torch.empty

    def full(*size, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no memory for the workspace")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", full)
    assert agemm.matmul_swiglu(a, b, sfa, sfb, gx * gw, tensor_scale=True, halves=True) is None


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
@pytest.mark.parametrize("M,N,kp,route", [
    (8, 8192, 4224, 3), (5, 5121, 4096, 3), (17, 6145, 2176, 3), (33, 6144, 1152, 3), (48, 5121, 1152, 3), (64, 8190, 4224, 3), (64, 4112, 8320, 3),
    (64, 8190, 6016, 3), (49, 4112, 6144, 3), (48, 8177, 6144, 3),                   # (more than 48 rows from K' = 6144 on: 64 elements)
    (523, 3001, 1792, 21), (349, 4099, 2048, 21), (375, 5122, 2432, 22), (297, 6145, 1664, 22), (644, 3001, 1536, 23), (326, 6144, 1792, 23),
    (333, 6144, 1152, 23), (556, 4099, 2048, 24), (80, 28672, 640, 24)])
def test_nvfp4_steps_of_128_elements_per_wave(agemm, oracle, M, N, kp, route):
    """the streams whose waves take 128 elements of a step: K' ending after any number of waves' shares of the last step and inside a
    16-byte piece of scale bytes, rows and columns ending inside a tile; exact products and fp32 sums as for the other shapes"""
    from arcquant_amd import _lib
    assert _lib.lib().arcq_gemm_route(M, N, kp, 0, 0, 0) == route
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, kp - 64, 64, "NVFP4", seed=91)
    want = oracle_dq(oracle, a, sfa, "NVFP4") @ oracle_dq(oracle, b, sfb, "NVFP4").T * (gx * gw)
    scale = (torch.tensor(gx, device="cuda"), torch.tensor(gw, device="cuda"))
    y = agemm.matmul(a, b, sfa, sfb, scale)
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul(a, b, sfa, sfb, scale, residual=res), y + res)


@pytest.mark.parametrize("M,N,kp", [(1, 24, 128), (3, 100, 256), (8, 4096, 384), (16, 513, 640), (5, 4096, 8320), (16, 4090, 8448), (8, 2048, 8576), (1, 4096, 8192),
                                    (17, 1000, 896), (40, 4096, 1408), (64, 333, 4352), (4, 8200, 1152), (33, 4096, 8320), (8, 6144, 8576),
                                    (1, 8208, 1280), (2, 8200, 2304), (3, 9000, 2176), (4, 8193, 2432), (20, 300, 384), (48, 2048, 256), (33, 100, 128)])
def test_mxfp4_decode_batches(agemm, oracle, M, N, kp):
    """MXFP4 decode batches straight from global memory: K' ending after one to four steps of a wave's run, fewer runs than waves and many
    more, sixteen waves for long rows, runs of two steps for short rows of wide layers and for those of less than four steps; the bf16
    rounding and the order of the fp32 sum remain"""
    (x, w, idx, gx, gw), (a, sfa, b, sfb) = quantized_pair(agemm, M, N, kp - 64, 64, "MXFP4", seed=93)
    want = oracle_dq(oracle, a, sfa, "MXFP4") @ oracle_dq(oracle, b, sfb, "MXFP4").T * 0.5
    y = agemm.matmul(a, b, sfa, sfb, 0.5, fmt="MXFP4")
    assert rel_fro(y.float(), want) < 2.5e-3
    assert torch.allclose(y.float(), want, rtol=2 ** -7, atol=1e-4 * float(want.abs().max()))
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(agemm.matmul(a, b, sfa, sfb, 0.5, fmt="MXFP4", residual=res), y + res)
