"""The pipelined MFMA products (gemm_pipe.h): every kernel at the edges of its
tile against a plain fp32 product, and the calls of tm_matmul / tm_linear /
tm_dot that select them."""
import ctypes

import pytest
import torch

import triton_metal_amd as tm

KINDS = {"f16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn,
         "e5m2": torch.float8_e5m2}
TILES = {"44": (4, 4), "42": (4, 2), "22": (2, 2), "22d": (2, 2), "21": (2, 1), "11": (1, 1)}
DTC = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
# unit roundoff of an output dtype; fp32 outputs carry the sums' own error
U = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


class Params(ctypes.Structure):
    """struct MmParams of gemm_pipe.h"""
    _fields_ = ([(n, ctypes.c_void_p) for n in ("A", "B", "C", "Z")]
                + [(n, ctypes.c_longlong) for n in ("sa_b", "sb_b", "sc_b", "sz_b", "sc_m",
                                                    "sc_n", "sz_m", "sz_n")]
                + [(n, ctypes.c_int) for n in ("M", "N", "K", "lda", "ldb", "tiles_m", "tiles_n",
                                               "epi", "out_dt", "z_dt", "vec_z", "fix")])


def _operand(b, rows, cols, dt, transposed, seed, al):
    """[b, rows, cols] of small random values, stored [b, cols, rows] if
    transposed; stored rows padded with NaN to a multiple of al elements."""
    g = torch.Generator().manual_seed(seed)
    d0, d1 = (cols, rows) if transposed else (rows, cols)
    t = torch.full((b, d0, -(-d1 // al) * al), float("nan")).to(dt)
    t[:, :, :d1] = torch.randn(b, d0, d1, generator=g).to(dt)
    t = t.cuda()[:, :, :d1]
    return t.transpose(1, 2) if transposed else t


def _close(got, ref, bound, odt):
    """|got - ref| <= one rounding of the result + the bound on a K-term fp32
    sum (K u sum |a||b|; the MFMA sums in fp32 in some order)."""
    err = (got.double() - ref).abs()
    tol = 1.01 * U[odt] * ref.abs() + bound + 1e-30
    assert bool((err <= tol).all()), float((err / tol).max())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("layout", ["kk", "kr", "rk", "rr"])
@pytest.mark.parametrize("kind", KINDS)
def test_every_kernel(kind, layout, tile):
    """Remainders of the tile in M and N, a last k step that is partial (or the
    only one), two batches, with each kind of Z and output."""
    from triton_metal_amd import _lib
    from triton_metal_amd.driver import HipUtils
    hu = HipUtils()
    rt, ct = TILES[tile]
    bm, bn, dt = 64 * rt, 64 * ct, KINDS[kind]
    fp8 = dt.itemsize == 1
    al, bk = (16, 128) if fp8 else (8, 64)
    fn = hu.builtin_function(f"mm_{kind}_{layout}_{tile}")
    rb = layout[1] == "r"
    shapes = ((bm + 5, bn - 3, 3 * bk + al, torch.float32, None),
              (bm - 1, bn + 9, al, torch.bfloat16, "rows"),
              (3, 2 * bn + 1, 9 * bk, torch.float16, "cols"),
              (bm, bn, 2 * bk, torch.float32, "matrix"))
    for i, (M, N, K, odt, zk) in enumerate(shapes):
        b = 1 + i % 2
        # row-contiguous operands of any row count, their k rows padded to pieces
        A = _operand(b, M, K, dt, layout[0] == "r", 3 * i, al)
        B = _operand(b, K, N, dt, not rb, 3 * i + 1, al)
        C = torch.full((b, M, N), float("nan"), device="cuda", dtype=odt)
        p = Params(A.data_ptr(), B.data_ptr(), C.data_ptr(), None)
        p.sa_b, p.sb_b, p.sc_b = A.stride(0), B.stride(0), C.stride(0)
        p.sc_m, p.sc_n, p.M, p.N, p.K = N, 1, M, N, K
        p.lda = A.stride(2) if layout[0] == "r" else A.stride(1)
        p.ldb = B.stride(1) if rb else B.stride(2)
        p.tiles_m, p.tiles_n = -(-M // bm), -(-N // bn)
        p.out_dt = DTC[odt]
        ref = A.double() @ B.double().contiguous()
        bound = K * U[torch.float32] * (A.double().abs() @ B.double().abs().contiguous())
        if zk:
            Z = torch.randn(b, 1 if zk == "cols" else M, 1 if zk == "rows" else N).to(odt).cuda()
            p.Z, p.epi, p.z_dt, p.sz_b = Z.data_ptr(), 1, DTC[odt], Z.stride(0)
            p.sz_m = 0 if zk == "cols" else Z.stride(1)
            p.sz_n = 0 if zk == "rows" else 1
            p.vec_z = int(zk != "rows")
            ref = ref + Z.double()
        args = (ctypes.c_void_p * 1)(ctypes.cast(ctypes.pointer(p), ctypes.c_void_p))
        rc = hu._lib.tm_launch(fn, p.tiles_m * p.tiles_n, b, 1, 256, 1, 1, 0,
                               torch.cuda.current_stream().cuda_stream, args)
        assert rc == 0, _lib.last_error()
        torch.cuda.synchronize()
        # the fp32 sum and the addition of Z each round once more
        _close(C, ref, bound + 2 * U[torch.float32] * ref.abs(), odt)


def _unaligned(b, rows, cols, dt, transposed, seed, off=1):
    """[b, rows, cols] of small random values without any padding: the first
    element `off` past an aligned address, one element (NaN) between the batches
    and after the last."""
    g = torch.Generator().manual_seed(seed)
    d0, d1 = (cols, rows) if transposed else (rows, cols)
    step = d0 * d1 + 1
    flat = torch.full((off + b * step,), float("nan")).to(dt)
    for i in range(b):
        flat[off + i * step:][:d0 * d1] = torch.randn(d0 * d1, generator=g).to(dt)
    t = flat.cuda().as_strided((b, d0, d1), (step, d1, 1), off)
    return t.transpose(1, 2) if transposed else t


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("layout", ["kk", "kr", "rk", "rr"])
@pytest.mark.parametrize("kind", KINDS)
def test_every_kernel_fills_by_elements(kind, layout, tile):
    """The pieces that no copy may take whole (MmParams::fix, as mm_plan sets it for
    operands like these), in the only k step and in the last of several: K no whole
    number of pieces, row-contiguous rows that end inside one, an odd batch stride."""
    from triton_metal_amd import _lib
    from triton_metal_amd.driver import HipUtils
    hu = HipUtils()
    rt, ct = TILES[tile]
    bm, bn, dt = 64 * rt, 64 * ct, KINDS[kind]
    al, bk = (16, 128) if dt.itemsize == 1 else (8, 64)
    fn = hu.builtin_function(f"mm_{kind}_{layout}_{tile}")
    ar, br = layout[0] == "r", layout[1] == "r"
    for i, (M, N, K) in enumerate(((bm + 5, bn - 3, 2 * bk + al // 2 + 1), (bm - 1, bn + 9, al - 1),
                                   (al + 3, 2 * bn + 1, 4 * bk + 1), (bm + 1, al + 7, bk - 3),
                                   (bm, bn, 3 * bk))):
        b = 1 + i % 2
        A = _unaligned(b, M, K, dt, ar, 3 * i)
        B = _unaligned(b, K, N, dt, not br, 3 * i + 1)
        C = torch.full((b, M, N), float("nan"), device="cuda")
        p = Params(A.data_ptr(), B.data_ptr(), C.data_ptr(), None)
        p.sa_b, p.sb_b, p.sc_b = A.stride(0), B.stride(0), C.stride(0)
        p.sc_m, p.sc_n, p.M, p.N, p.K = N, 1, M, N, K
        p.lda, p.ldb = A.stride(2 if ar else 1), B.stride(1 if br else 2)
        p.tiles_m, p.tiles_n = -(-M // bm), -(-N // bn)
        p.out_dt = DTC[torch.float32]
        p.fix = (4 if ar else 1 if K % al else 0) | (8 if br else 2 if K % al else 0)
        args = (ctypes.c_void_p * 1)(ctypes.cast(ctypes.pointer(p), ctypes.c_void_p))
        rc = hu._lib.tm_launch(fn, p.tiles_m * p.tiles_n, b, 1, 256, 1, 1, 0,
                               torch.cuda.current_stream().cuda_stream, args)
        assert rc == 0, _lib.last_error()
        torch.cuda.synchronize()
        ref = A.double() @ B.double().contiguous()
        bound = K * U[torch.float32] * (A.double().abs() @ B.double().abs().contiguous())
        _close(C, ref, bound, torch.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.float8_e4m3fn])
@pytest.mark.parametrize("M,N,K", [(72, 136, 208), (300, 520, 1040)])
def test_odd_batch_stride(dt, M, N, K):
    """tm.dot on batches of aligned rows whose batch stride alone is odd."""
    for ta in (False, True):
        for tb in (False, True):
            a = _unaligned(3, M, K, dt, ta, 1, off=0)
            b = _unaligned(3, K, N, dt, tb, 2, off=0)
            c = torch.full((3, M, N), 7.0, device="cuda")
            tm.dot(a, b, c)
            torch.cuda.synchronize()
            ref = a.double().contiguous() @ b.double().contiguous()
            bound = K * U[torch.float32] * (a.double().abs().contiguous()
                                            @ b.double().abs().contiguous())
            _close(c, ref, bound, torch.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", KINDS.values(), ids=KINDS)
@pytest.mark.parametrize("M,N,K", [(5, 70, 33), (129, 257, 131), (64, 33, 1), (300, 190, 1027),
                                   (131, 515, 575), (1, 1, 200)])
def test_any_alignment(dt, M, N, K):
    """Operands that start anywhere, with any row length and any K, in every
    layout; NaN around them (and in the row after the one a piece crosses into)
    never reaches the result."""
    for ta in (False, True):
        for tb in (False, True):
            for off, pad in ((0, 0), (1, 3), (3, 1)):
                def place(rows, cols, seed):
                    g = torch.Generator().manual_seed(seed)
                    flat = torch.full((off + rows * (cols + pad),), float("nan")).to(dt)
                    t = flat[off:].view(rows, cols + pad)
                    t[:, :cols] = torch.randn(rows, cols, generator=g).to(dt)
                    return flat.cuda()[off:].view(rows, cols + pad)[:, :cols]
                a = place(K, M, 1).t() if ta else place(M, K, 1)
                b = place(N, K, 2).t() if tb else place(K, N, 2)
                c = torch.full((M, N), 7.0, device="cuda")
                tm.dot(a, b, c)
                torch.cuda.synchronize()
                ref = a.double() @ b.double().contiguous()
                bound = K * U[torch.float32] * (a.double().abs() @ b.double().abs().contiguous())
                _close(c, ref, bound, torch.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_fp8_codes_are_exact(dt):
    """Every code through the product (a diagonal of codes times ones), the NaN
    and infinite ones included."""
    codes = torch.arange(256, dtype=torch.int32).to(torch.uint8).cuda()
    A = torch.zeros(256, 256, dtype=torch.uint8, device="cuda")
    A[torch.arange(256), torch.arange(256)] = codes
    B = torch.ones(256, 256, device="cuda").to(dt)
    C = torch.empty(256, 256, device="cuda")
    tm.matmul(A.view(dt), B, C, 256, 256, 256)
    want = codes.view(dt).float()
    assert torch.equal(torch.nan_to_num(C[:, 7], nan=3e38), torch.nan_to_num(want, nan=3e38))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("M,N,K", [(130, 264, 1040), (1, 336, 2064), (520, 72, 528)])
def test_padded_operands_and_in_place_bias(dt, M, N, K):
    """tm.dot on views of larger tensors (leading dimensions past the matrix, NaN
    around it: nothing outside the operands reaches the result), all four
    layouts, the bias read in place from the output; the output's padding
    stays as it was."""
    for ta in (False, True):
        for tb in (False, True):
            def padded(rows, cols, seed):
                g = torch.Generator().manual_seed(seed)
                t = torch.full((rows + 3, cols + 16), float("nan")).to(dt)
                t[:rows, :cols] = torch.randn(rows, cols, generator=g).to(dt)
                return t.cuda()[:rows, :cols]
            a = padded(K, -(-M // 16) * 16, 1).t()[:M] if ta else padded(M, K, 1)
            bm = padded(N, K, 2).t() if tb else padded(K, N, 2)
            out = torch.full((M, N + 8), 3.0, device="cuda")
            c = out[:, :N]
            tm.dot(a, bm, c, "add-matrix", z=c)
            torch.cuda.synchronize()
            ref = a.double() @ bm.double().contiguous() + 3.0
            bound = (K + 2) * U[torch.float32] * (a.double().abs() @ bm.double().abs().contiguous()
                                                  + 3.0)
            _close(c, ref, bound, torch.float32)
            assert bool((out[:, N:] == 3.0).all())


def test_selection():
    """Which sizes take the pipelined kernels and which keep the others, and
    the layouts and alignments they refuse (no device is touched)."""
    k = lambda *a, **kw: tm.gemm_kernel_for(*a, **kw)[0]
    assert k(4096, 4096, 4096) == "gemm_t256_nn_f16_same"
    assert k(2048, 11008, 4096) == "mm_f16_kr_42" and k(4096, 4352, 4096)[:9] == "mm_f16_kr"
    assert k(4096, 4096, 4096, trans_b=True, in_dtype=torch.bfloat16) == "mm_bf16_kk_44"
    assert k(16, 11008, 4096, trans_b=True, bias=True) == "mm_f16_kk_11"
    assert k(2000, 11008, 4096, trans_b=True) == "mm_f16_kk_42"
    assert {k(M, 4096, 4096, trans_b=True)[-2:] for M in (64, 512, 1024, 2048, 4096)} >= {"11", "44"}
    # odd N is fine for [N, K] weights, not for rows of [K, N]
    assert k(300, 1001, 1024, trans_b=True).startswith("mm_f16_kk_")
    assert k(300, 1001, 1024) == "tm_dot"
    assert k(300, 1000, 1001) == "tm_dot"
    assert k(300, 1000, 1024, lda=1028) == "tm_dot"
    assert k(512, 512, 512).startswith("gemm_s32k128_")
    assert k(4096, 4096, 64).startswith("gemm_t256_")
    # 256-tile problems on both sides of its rules (rounds of CUs filled; K)
    t256 = lambda *a, **kw: k(*a, **kw).startswith("gemm_t256_")
    assert not t256(2048, 4096, 1024) and t256(2304, 4096, 1024) and t256(2304, 4096, 4096)
    assert not t256(4096, 5120, 1024) and t256(5120, 5120, 1024) and not t256(5120, 5120, 4096)
    assert t256(8192, 4096, 4096) and not t256(8192, 4096, 4096 + 32) and not t256(8192, 4095, 4096)
    assert t256(3584, 4096, 3072, trans_b=True) and not t256(3584, 4096, 4096, trans_b=True)
    # few rows of [N, K] weights, and the K-split kernel past two workgroups a CU
    assert k(4, 8192, 384, trans_b=True).startswith("gemm_t32k_")
    assert k(4, 16384, 384, trans_b=True).startswith("mm_") and k(33, 8192, 384, trans_b=True)[:3] == "mm_"
    assert k(100, 2048, 648, trans_b=True).startswith("gemm_t32_")
    assert k(128, 2048, 1152, trans_b=True).startswith("mm_") and k(100, 2048, 648).startswith("mm_")
    assert k(16, 768, 1536, trans_b=True).startswith("gemm_t32_")
    assert k(1024, 1024, 256).startswith("gemm_s32k64_") and k(4096, 256, 256).startswith("mm_")
    assert k(768, 768, 512).startswith("gemm_s32k128_") and k(1024, 768, 512).startswith("mm_")
