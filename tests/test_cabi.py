"""CPU-only checks of the C-ABI library: it loads, exports every symbol include/arcq.h declares,
sizes buffers as documented and rejects bad arguments before touching a GPU."""
import ctypes
import os
import re

import pytest

from arcquant_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols(header="arcq.h"):
    text = open(os.path.join(ROOT, "include", header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(arcq_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    L = _lib.lib()
    names = declared_symbols()
    assert {"arcq_reorder_quantize_x", "arcq_reorder_quantize_w", "arcq_rmsnorm_quantize_x", "arcq_matmul"} <= set(
        names)
    for n in names:
        assert hasattr(L, n), f"{n} is declared in include/arcq.h but not exported"
    assert L.arcq_version() >= 100


def test_buffer_sizes():
    L = _lib.lib()
    assert L.arcq_group_size(0) == 16 and L.arcq_group_size(1) == 32 and L.arcq_group_size(7) == 0
    assert L.arcq_codes_bytes(2048, 4096, 128) == 2048 * 4224 // 2
    assert L.arcq_scales_bytes(2048, 4096, 128, 0) == 2048 * 4224 // 16
    assert L.arcq_scales_bytes(2048, 4096, 128, 1) == 2048 * 4224 // 32
    assert L.arcq_scales_bytes(1, 64, 0, 9) == 0


@pytest.mark.parametrize("K,S,fmt,want", [
    (4096, 128, 2, 3),      # unknown format
    (4100, 0, 0, 2),        # K not a multiple of 32
    (16, 0, 0, 2),          # K too small
    (32768, 0, 0, 2),       # beyond int16 indices
    (4096, 8, 0, 2),        # select_num not a multiple of the block
    (4096, 48, 1, 2),       # ... of 32 for MXFP4
    (4096, 8192, 0, 2),     # select_num > K
])
def test_argument_errors_need_no_gpu(K, S, fmt, want):
    L = _lib.lib()
    dummy = ctypes.c_void_p(0x1000)
    for fn in (L.arcq_reorder_quantize_x, L.arcq_reorder_quantize_w):
        assert fn(dummy, 4, K, dummy, S, fmt, 1.0, None, dummy, dummy, None) == want
    assert L.arcq_rmsnorm_quantize_x(dummy, dummy, 1e-5, 4, K, dummy, S, fmt, 1.0, None, dummy, dummy, None) == want
    assert L.arcq_reorder_quantize_x_absmax(dummy, 4, K, dummy, S, fmt, 2688.0, dummy, dummy, dummy, None) == want


def test_null_alignment_and_matmul_errors():
    L = _lib.lib()
    ok, odd = ctypes.c_void_p(0x1000), ctypes.c_void_p(0x1004)
    assert L.arcq_reorder_quantize_x(None, 4, 4096, ok, 0, 0, 1.0, None, ok, ok, None) == 1
    assert L.arcq_reorder_quantize_x(odd, 4, 4096, ok, 0, 0, 1.0, None, ok, ok, None) == 4
    assert L.arcq_reorder_quantize_x(ok, 0, 4096, ok, 0, 0, 1.0, None, ok, ok, None) == 0   # zero rows: nothing to do
    absmax = L.arcq_reorder_quantize_x_absmax                                                # scale + quantizer as one call
    assert absmax(ok, 4, 4096, ok, 0, 0, 2688.0, None, ok, ok, None) == 1                    # nowhere to put the scale
    assert absmax(None, 4, 4096, ok, 0, 0, 2688.0, ok, ok, ok, None) == 1
    assert absmax(odd, 4, 4096, ok, 0, 0, 2688.0, ok, ok, ok, None) == 4
    assert absmax(ok, 4, 4096, ok, 0, 0, 0.0, ok, ok, ok, None) == 2                         # divisor must be positive
    assert L.arcq_matmul(ok, ok, ok, ok, 4, 4, 100, 0, 1.0, None, None, ok, None) == 2       # K' % 64
    assert L.arcq_matmul(ok, ok, ok, ok, 4, 4, 128, 5, 1.0, None, None, ok, None) == 3
    assert L.arcq_matmul(ok, None, ok, ok, 4, 4, 128, 0, 1.0, None, None, ok, None) == 1
    assert L.arcq_matmul(ok, ok, ok, ok, 0, 4, 128, 0, 1.0, None, None, ok, None) == 0
    assert b"16-byte" in L.arcq_status_string(4)


def test_grouped_entry_points_reject_bad_arguments():
    """the MoE entry points check shapes, pointers and alignment before any launch"""
    L = _lib.lib()
    ok, odd = ctypes.c_void_p(0x1000), ctypes.c_void_p(0x1004)
    gq = L.arcq_grouped_reorder_quantize_x
    assert gq(ok, 8, 4096, ok, 0, ok, 128, 0, None, ok, ok, None) == 2          # no segment
    assert gq(ok, 8, 4100, ok, 2, ok, 128, 0, None, ok, ok, None) == 2          # K % 32
    assert gq(ok, 8, 4096, ok, 2, ok, 8, 0, None, ok, ok, None) == 2            # select_num % 16
    assert gq(ok, 8, 4096, ok, 2, ok, 128, 7, None, ok, ok, None) == 3          # format
    assert gq(ok, 8, 4096, None, 2, ok, 128, 0, None, ok, ok, None) == 1        # no offsets
    assert gq(odd, 8, 4096, ok, 2, ok, 128, 0, None, ok, ok, None) == 4
    assert gq(ok, 0, 4096, ok, 2, ok, 128, 0, None, ok, ok, None) == 0          # no rows: nothing to do
    gs = L.arcq_grouped_swiglu_quantize_x
    assert gs(ok, ok, 4000, 8, 4096, ok, 2, ok, 128, 0, None, ok, ok, None) == 2  # row stride below K
    assert gs(ok, None, 8192, 8, 4096, ok, 2, ok, 128, 0, None, ok, ok, None) == 1
    ts = L.arcq_grouped_tensor_scale
    assert ts(ok, None, 4096, 8, 4096, ok, 0, 2688.0, ok, None) == 2
    assert ts(ok, None, 4096, 8, 4096, ok, 2, 0.0, ok, None) == 2
    assert ts(ok, None, 4096, 8, 4096, ok, 2, 2688.0, None, None) == 1
    gm = L.arcq_grouped_matmul
    assert gm(ok, ok, ok, ok, ok, 2, 8, 256, 448, 1, 1.0, None, None, None, ok, None) == 2    # K' % 128
    assert gm(ok, ok, ok, ok, ok, 2, 8, 256, 384, 1, 1.0, None, None, None, ok, None) == 2    # K' < 512
    assert gm(ok, ok, ok, ok, ok, 0, 8, 256, 512, 1, 1.0, None, None, None, ok, None) == 2    # no segment
    assert gm(ok, ok, ok, ok, None, 2, 8, 256, 512, 1, 1.0, None, None, None, ok, None) == 1
    assert gm(ok, odd, ok, ok, ok, 2, 8, 256, 512, 1, 1.0, None, None, None, ok, None) == 4   # scale bytes unaligned
    assert gm(ok, ok, ok, ok, ok, 2, 0, 256, 512, 1, 1.0, None, None, None, ok, None) == 0
    sw = L.arcq_grouped_matmul_swiglu
    assert sw(ok, ok, ok, ok, ok, 2, 8, 250, 512, 1, 1.0, None, None, ok, None, None) == 2    # N % 16
    assert L.arcq_matmul_swiglu(ok, ok, ok, ok, 8, 256, 448, 1, 1.0, None, None, ok, None, None) == 2
    assert L.arcq_scales_from_absmax(None, 4, 2688.0, None) == 1
    assert L.arcq_scales_from_absmax(ok, 4, -1.0, None) == 2
    mc = L.arcq_moe_combine
    assert mc(ok, ok, ok, 8, 4100, 2, 16, ok, None) == 2                                      # H % 8
    assert mc(ok, ok, ok, 8, 4096, 9, 72, ok, None) == 2                                      # top_k > 8
    assert mc(ok, None, ok, 8, 4096, 2, 16, ok, None) == 1
    assert mc(ok, ok, ok, 0, 4096, 2, 0, ok, None) == 0
    mr = L.arcq_moe_route
    assert L.arcq_moe_route_workspace_bytes(4096, 8) == 64 * 8 * 4
    assert mr(ok, 0, 16, 65, 2, ok, ok, ok, ok, ok, ok, ok, 1 << 20, None) == 2               # more than 64 experts
    assert mr(ok, 0, 16, 8, 9, ok, ok, ok, ok, ok, ok, ok, 1 << 20, None) == 2                # top_k > 8
    assert mr(ok, 0, 16, 4, 5, ok, ok, ok, ok, ok, ok, ok, 1 << 20, None) == 2                # top_k > experts
    assert mr(None, 0, 16, 8, 2, ok, ok, ok, ok, ok, ok, ok, 1 << 20, None) == 1
    assert mr(ok, 0, 4096, 8, 2, ok, ok, ok, ok, ok, ok, ok, 16, None) == 7                   # workspace too small
    P = _lib.probe_lib()                 # the measurement-only library (include/arcq_probe.h)
    assert P.arcq_stream_probe_variants() >= 2
    assert P.arcq_stream_probe_variant(ok, ok, 1024, 512, 99, None) == 2


def test_decode_batches_fit_the_no_alloc_array():
    """arcq_matmul and arcq_matmul_noalloc share one planner: every decode batch (M <= 64) of the Llama-3-8B
    projection shapes must get a plan whose split-K partial tiles fit the fixed array, in both formats"""
    L = _lib.lib()
    limit = L.arcq_matmul_noalloc_limit()
    assert limit == 8 << 20
    for fmt in (0, 1):
        for N, K in ((6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336)):
            for S in (64, 128, 256):
                for M in range(1, 65):
                    need = L.arcq_matmul_scratch_bytes(M, N, K + S, fmt)
                    assert need <= limit, (fmt, M, N, K + S, need)


@pytest.mark.parametrize("rows,n,kp,n_seg,decoded_rows", [
    (8 * 1024, 28672, 4224, 8, 8192), (8 * 1024, 6144, 4224, 8, 8192), (64 * 768, 4096, 2176, 64, 64 * 768),
    (64 * 768, 2816, 2176, 64, 64 * 768),
    (8 * 767, 28672, 4224, 8, 0),         # too few rows per expert
    (64 * 1024, 2048, 1536, 64, 0),       # too few columns to pay for decoding the activations
    (8 * 1024, 4096, 14464, 8, 0),        # few columns and few rounds of tiles
    (3000, 528, 640, 3, 0),
])
def test_grouped_gemm_workspace(rows, n, kp, n_seg, decoded_rows):
    """which grouped NVFP4 problems multiply activations decoded to fp16 ahead (two bytes per value of the workspace)"""
    ask = _lib.lib().arcq_gemm_workspace_bytes
    assert ask(rows, n, kp, 0, n_seg) == 2 * decoded_rows * kp
    assert ask(rows, n, kp, 1, n_seg) == 0  # MXFP4 decodes nothing


@pytest.mark.parametrize("rows,n,kp,n_seg,cut", [
    (4 * 512, 4096, 14464, 4, False), (2 * 512, 4096, 14464, 2, False), (3072, 4096, 8192, 4, False),   # never more than a round of tiles
    (3073, 4096, 8192, 4, True), (8 * 512, 4096, 14464, 8, True), (2 * 650, 14336, 8320, 2, True), (8 * 1024, 4096, 14464, 8, True),
    (8 * 511, 4096, 14464, 8, False), (8 * 1024, 2048, 14464, 8, False), (8 * 1024, 4096, 8064, 8, False), (16 * 4096, 4096, 8192, 16, False),
    (3000, 6144, 10240, 0, True), (4096, 4096, 14592, 0, False), (2331, 4096, 14592, 0, False),        # whole rounds; less than one
])
def test_gemm_scratch_for_a_cut_round(rows, n, kp, n_seg, cut):
    """which NVFP4 problems take 128 MiB behind the decoded operand, to cut their last round of tiles along K': only where more than
    a round of 256 is possible at all"""
    L = _lib.lib()
    operand = 2 * kp * (rows if n_seg else min(rows, n))
    assert L.arcq_gemm_scratch_bytes(rows, n, kp, 0, n_seg) == (operand + (128 << 20) if cut else L.arcq_gemm_workspace_bytes(rows, n, kp, 0, n_seg))


@pytest.mark.parametrize("M,N,kp,decoded_rows", [
    (2049, 4096, 4352, 2049), (257, 28672, 4352, 257), (33000, 64, 1152, 64), (65, 70000, 1152, 65),
    (2048, 4096, 4352, 0), (256, 28672, 4352, 0),                                 # one round of 256x128 tiles
    (64, 70000, 1152, 0), (16, 70000, 4352, 0), (1, 128256, 4352, 0),             # decode batches
    (4096, 4096, 448, 0), (4096, 4096, 4160, 0),                                  # K' short, or not a multiple of 128
])
def test_gemm_workspace(M, N, kp, decoded_rows):
    """which NVFP4 problems multiply the operand with fewer rows decoded to fp16 ahead"""
    ask = _lib.lib().arcq_gemm_workspace_bytes
    assert ask(M, N, kp, 0, 0) == 2 * decoded_rows * kp
    assert ask(M, N, kp, 1, 0) == 0


@pytest.mark.parametrize("M,N,decoded_rows", [
    (8100, 3072, 3072),      # two rounds of 256 rows (less the decoding of fewer rows), and not three of 128: 1.88 to 2.1
    (8300, 6144, 6144),      # four of 256 rows, and not five of 192: 3.95 to 4.1
    (6216, 3584, 6216),      # two of 192 rows, and not two of 256: 1.64 to 1.94
])
def test_gemm_workspace_by_rounds_of_tiles(M, N, decoded_rows):
    """more rows of activations than of weights: the weights are decoded for tiles of 256 rows of activations, the activations for
    smaller ones, whichever make the fewest rounds, counted by what a round of each was measured to take"""
    for kp in (512, 1152, 4352):
        assert _lib.lib().arcq_gemm_workspace_bytes(M, N, kp, 0, 0) == 2 * decoded_rows * kp


def test_gemm_rejects_bad_arguments():
    """arcq_gemm checks the forms against each other, alignment, shapes and pointers before any launch"""
    L, ok, odd = _lib.lib(), 0x1000, 0x1004

    def gemm(**kw):
        a = dict(a_codes=ok, a_scales=ok, b_codes=ok, b_scales=ok, M=8, N=256, Kp=512, fmt=0, alpha=1.0, c=ok)
        return L.arcq_gemm(_lib.GemmArgs(**{**a, **kw}), None)

    assert L.arcq_gemm(None, None) == 1
    assert gemm(c=None) == 1 and gemm(a_codes=None) == 1
    assert gemm(n_seg=2) == 1                                                        # no offsets
    assert gemm(Kp=100) == 2 and gemm(M=-1) == 2 and gemm(n_seg=-1) == 2
    assert gemm(swiglu=1, residual=ok) == 2 and gemm(swiglu=1, N=250) == 2 and gemm(swiglu=1, Kp=448) == 2
    assert gemm(n_seg=2, seg_offsets=ok, Kp=448) == 2
    assert gemm(fmt=2) == 3
    assert gemm(workspace=odd, workspace_bytes=1 << 20) == 4 and gemm(residual=odd) == 4 and gemm(a_codes=odd) == 4
    assert gemm(n_seg=2, seg_offsets=ok, a_scales=odd) == 4 and gemm(swiglu=1, b_scales=odd) == 4
    assert gemm(M=0) == 0 and gemm(N=0) == 0


def test_gemm_kernel_of_a_problem():
    """the dispatch as arcq_gemm_kernel reports it: decode batches, one round of tiles, the formats' large tiles, operands
    beyond 4 GiB, grouped and fused forms, refused arguments"""
    k = _lib.lib().arcq_gemm_kernel
    assert [k(M, 4096, 4352, 0, 0, 0) for M in (1, 16, 128, 1024, 4096)] == [1, 1, 21, 22, 168]
    assert [k(M, 28672, 4352, 1, 0, 0) for M in (1, 16, 300, 4096)] == [1, 214, 22, 84]
    assert k(4096, 4096, 14592, 1, 0, 0) == 88 and k(4096, 4096, 8064, 1, 0, 0) == 84
    assert k(2_000_000, 4096, 8192, 1, 0, 0) == 44                             # rows beyond 32-bit byte offsets
    assert [k(M, 28672, 4224, 0, 8, 0) for M in (64, 800, 8192)] == [21, 22, 168]
    assert [k(M, 28672, 4224, 1, 8, 0) for M in (64, 800, 8192)] == [21, 22, 84]
    assert k(8192, 4096, 13312, 1, 8, 0) == 84 and k(8192, 4096, 14464, 1, 8, 0) == 88
    assert k(16, 28672, 4352, 0, 0, 1) == 21 and k(16, 28672, 4352, 0, 0, 0) == 11   # split-K has no fused epilogue
    for bad in ((4096, 4096, 4352, 2, 0, 0), (0, 4096, 4352, 0, 0, 0), (4096, 4096, 100, 0, 0, 0), (4096, 4096, 4352, 0, -1, 0),
                (64, 256, 448, 1, 2, 0), (64, 256, 448, 1, 0, 1)):
        assert k(*bad) == -1


PLAN, AHEAD, CUT, STREAM, SHAPE = 0, 1, 2, 3, 16


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
@pytest.mark.parametrize("N,edges", [
    # by rows: the K' below which the weights are not streamed (0: always, None: never)
    (2048, {1: None, 8: None, 9: 10240, 16: 10240, 17: 4096, 32: 4096, 33: 0, 48: 0}),
    (4096, {4: None, 5: 10240, 8: 10240, 9: 8192, 16: 8192, 17: 4096, 33: 0}),
    (8192, {4: None, 5: 4096, 16: 4096, 17: 2048, 32: 2048, 33: 0, 64: 0}),
    (12288, {1: 2560, 16: 2560, 17: 0, 64: 0}), (14336, {8: 2560, 9: 1536, 16: 1536, 17: 0}),
    (18944, {4: 2560, 5: 2048, 7: 2048, 8: 0, 64: 0}), (28672, {8: 0, 64: 0}), (37888, {8: 0, 48: 0, 49: 1536, 64: 1536}),
    (49152, {8: 0, 64: 0}),
])
def test_route_of_nvfp4_decode_batches(N, edges):
    """where a decode batch is a stream of the weights, and where the kernels that begin and end sooner have it; a fused SwiGLU
    epilogue, which those have not, always is one"""
    route = _lib.lib().arcq_gemm_route
    for M, edge in edges.items():
        for kp in ((512, 8192) if edge == 0 else (512, 16256) if edge is None else (edge - 128, edge)):
            want = STREAM if edge is not None and kp >= edge else PLAN
            assert route(M, N, kp, 0, 0, 0) == want, (M, kp)
            assert route(M, N, kp, 0, 0, 1) == STREAM
            assert route(M, N, kp, 1, 0, 0) == PLAN                         # MXFP4
    assert route(4, 28672, 512, 0, 0, 0) == STREAM and route(4, 28672, 640, 0, 0, 0) == PLAN   # one step of a wide layer
    for (M, N, kp), want in {(64, 1024, 12160): STREAM, (64, 1024, 12288): PLAN, (64, 4096, 16256): STREAM, (64, 4096, 16384): PLAN,
                             (48, 4096, 16384): STREAM, (64, 4096, 448): PLAN, (64, 4096, 4160): PLAN}.items():
        assert route(M, N, kp, 0, 0, 0) == want, (M, N, kp)


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
def test_route_of_other_nvfp4_problems():
    """as arcq_gemm launches them, given the scratch that it asks for"""
    route = _lib.lib().arcq_gemm_route
    for (M, N, kp, E), want in {
            (4096, 4096, 4352, 0): AHEAD, (3000, 6144, 10240, 0): CUT, (2048, 4096, 4352, 0): PLAN,
            (8 * 1024, 4096, 14464, 8): CUT, (8 * 1024, 28672, 4224, 8): AHEAD, (4 * 512, 4096, 14464, 4): PLAN}.items():
        assert route(M, N, kp, 0, E, 0) == want, (M, N, kp, E)
    # experts: 40 rows on average, 95 where a layer is wide or all experts together are small, 32 where K' is short
    for (rows, N, kp, E), want in {
            (40, 4096, 14464, 8): STREAM, (41, 4096, 14464, 8): PLAN, (95, 8208, 2048, 8): STREAM, (96, 8208, 2048, 8): PLAN,
            (95, 2048, 8320, 8): STREAM, (41, 2064, 8320, 8): PLAN, (32, 2048, 1536, 64): STREAM, (33, 2048, 1536, 64): PLAN,
            (40, 2048, 1536, 8): STREAM, (41, 2048, 1536, 8): PLAN, (40, 28672, 1920, 8): PLAN}.items():
        assert route(rows * E, N, kp, 0, E, 0) == route(rows * E, N, kp, 0, E, 1) == want, (rows, N, kp, E)
    assert route(0, 4096, 4352, 0, 0, 0) == route(64, 256, 448, 0, 2, 0) == route(64, 256, 512, 2, 0, 0) == -1


@pytest.mark.skipif("ARCQ_GEMM_KERNEL" in os.environ, reason="another kernel is forced")
def test_route_of_mxfp4_problems_on_large_tiles():
    """what a plan of 84 is launched as: the ping-pong kernel from K' = 2176 on, of multiples of 256 from 2560, 3840 where persistent workgroups
    walk many columns; not with the interleaved SwiGLU epilogue or over experts, and not where rows lie beyond 32-bit offsets"""
    L, PINGPONG = _lib.lib(), 4
    for M, N, first, before in ((2300, 4600, 2176, 2048), (2304, 4608, 2560, 2304), (2300, 4610, 2560, 2304), (2300, 4610, 2432, 2048), (4096, 28672, 3840, 3584),
                                (4096, 28672, 2176, 2048), (4090, 28672, 2560, 2304), (8192, 28672, 2560, 2304), (4096, 14336, 2560, 2304)):
        assert L.arcq_gemm_kernel(M, N, first, 1, 0, 0) == L.arcq_gemm_kernel(M, N, before, 1, 0, 0) == 84
        assert L.arcq_gemm_route(M, N, first, 1, 0, 0) == PINGPONG and L.arcq_gemm_route(M, N, before, 1, 0, 0) == PLAN, (M, N)
        assert L.arcq_gemm_route(M, N, first, 1, 0, 1) == L.arcq_gemm_route(8 * 800, N, first, 1, 8, 0) == PLAN
    assert L.arcq_gemm_kernel(4096, 4096, 14592, 1, 0, 0) == 88 and L.arcq_gemm_route(4096, 4096, 14592, 1, 0, 0) == PLAN
    assert L.arcq_gemm_route(2_000_000, 4096, 8064, 1, 0, 0) == L.arcq_gemm_route(16, 4096, 4352, 1, 0, 0) == PLAN


def test_release_stream_without_buffers_needs_no_gpu_work():
    assert hasattr(_lib.lib(), "arcq_release_stream")


def test_probe_library_is_separate_from_the_product_library():
    """the copy kernels used for measurement live in their own library with their own header"""
    P, L = _lib.probe_lib(), _lib.lib()
    names = declared_symbols("arcq_probe.h")
    assert names == ["arcq_mfma_rate_probe", "arcq_mfma_rate_probe_flops", "arcq_stream_probe", "arcq_stream_probe_variant",
                     "arcq_stream_probe_variants"]
    assert P.arcq_mfma_rate_probe(3, 1, 10, ctypes.c_void_p(0x1000), ctypes.c_void_p(0x1000), None) == 2
    assert P.arcq_mfma_rate_probe_flops(0, 2, 1) == 256.0 * 4 * 2 * 4 * 8 * 2.0 * 32 * 32 * 64
    assert P.arcq_mfma_rate_probe_flops(1, 1, 3) == 256.0 * 4 * 1 * 3 * 4 * 8 * 2.0 * 32 * 32 * 16
    for n in names:
        assert hasattr(P, n) and not hasattr(L, n)
