"""The pipelined weight-only kernels (wq_pipe.hip): edges of their tiles and k
slices against the fp32 product, and the calls that select them."""
import pytest
import torch

import triton_metal_amd as tm

ACT = {"f16": torch.float16, "bf16": torch.bfloat16}


def _problem(qbits, M, N, K, act, zeros, seed):
    """x, weights, scales, zero-points, the dequantised weights, and the largest
    terms the kernels sum in fp32: (OFF + q + z) s, OFF the operands' offset (a
    single fp16 row: the GEMV kernels, 1024)."""
    off = 0 if qbits == 8 else 128 if act == torch.bfloat16 else 64 if M > 1 else 1024
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(act)
    cols = K // 128 if qbits == 4 else 1
    if qbits == 4:
        w = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8)
        q = torch.stack((w & 15, w >> 4), -1).reshape(N, K).double()
    else:
        w = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8)
        q = w.double()
    s = ((0.5 + torch.rand(N, cols, generator=g)) / 64).to(act)
    z = None
    if zeros == "u":
        z = torch.randint(0, 256, (N, cols), generator=g).to(torch.uint8)
    elif zeros == "s":  # fractional zero-points too
        z = (torch.rand(N, cols, generator=g) * 15).to(act)
    rep = K // cols
    deq = s.double().repeat_interleave(rep, 1)
    mag = (q.abs() + (0 if z is None else z.double().repeat_interleave(rep, 1)) + off) * deq
    deq = deq * (q - (0 if z is None else z.double().repeat_interleave(rep, 1)))
    return x, w, s if qbits == 4 else s.reshape(N), z, deq, mag


def _sum_bound(x, deq, mag):
    """How far the fp32 sums may be off: each addition rounds a partial sum whose
    size is that of the terms' 2-norm, in groups of 128 k (|x| mag) and then over the
    groups (|x| deq); 16 and 4 for the largest of many outputs."""
    x2 = x.double() ** 2
    return 2.0 ** -24 * (16 * (x2 @ (mag ** 2).t()).sqrt()
                         + 4 * (x.shape[1] / 128) ** 0.5 * (x2 @ (deq ** 2).t()).sqrt())


@pytest.mark.gpu
@pytest.mark.parametrize("act", ACT)
@pytest.mark.parametrize("qbits,zeros", [(4, None), (4, "s"), (4, "u"), (8, None)])
@pytest.mark.parametrize("M,N,K", [(1, 144, 640), (2, 48, 128), (1, 4112, 640), (2, 4112, 128),
                                   (9, 144, 384), (40, 272, 1152), (64, 128, 384),
                                   (65, 400, 896), (129, 16, 2176), (200, 1040, 3200),
                                   (1300, 2064, 384)])
def test_against_the_fp32_product(qbits, zeros, act, M, N, K):
    dt = ACT[act]
    x, w, s, z, deq, mag = _problem(qbits, M, N, K, dt, zeros, M + N)
    if not (qbits == 4 and M == 1):
        name = tm.wq_kernel_for(qbits, M, N, K, act_dtype=dt, details=True, zero_dtype=None if z is
                                None else z.dtype)["name"]
        assert name == (f"wq_pipe_q{qbits}_{act}_z{zeros or 'n'}_r{1 if M <= 64 else 2}"
                        if M > 2 or N > 4096 else "wq_general"), name
    bias = torch.randn(N).to(dt)
    xd, wd, sd, bd = x.cuda(), w.cuda(), s.cuda(), bias.cuda()
    zd = None if z is None else z.cuda()
    y = torch.full((M, N), float("nan"), dtype=dt, device="cuda")
    if qbits == 4:
        tm.int4_linear(xd, wd, bd, y, sd, zd, M, N, K, 128)
    else:
        tm.int8_linear(xd, wd, bd, y, sd, zd, M, N, K)
    ref = x.double() @ deq.t() + bias.double()
    # one rounding of the result on top of the sums'
    u = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    tol = 1.01 * u * ref.abs() + _sum_bound(x, deq, mag) + 1e-6
    err = (y.cpu().double() - ref).abs()
    assert bool((err <= tol).all()), float((err / tol).max())
    # the sums themselves: equal rows with a bias that cancels them up to its own
    # rounding leave a result small enough for the output type to show the error
    x = x[:1].expand(M, K).contiguous()
    ref = x[:1].double() @ deq.t()
    bias = (-ref[0]).to(dt)
    rest = ref + bias.double()
    err = (_call(qbits, x, w, s, z, bias) - rest).abs()
    tol = 1.01 * u * rest.abs() + _sum_bound(x[:1], deq, mag) + 1e-7
    assert bool((err <= tol).all()), float((err / tol).max())


@pytest.mark.parametrize("act", ACT)
@pytest.mark.parametrize("zeros", [None, "s", "u"])
@pytest.mark.parametrize("K", [128, 640, 3200])
def test_the_bound_on_the_sums_sees_lost_bits(K, zeros, act):
    """The bound of the test above holds for fp32 sums of the kernels' form and fails
    for sums that lose bits: rounded to bf16 after each group (two groups and more),
    or a scale that is 2^-12 off."""
    dt = ACT[act]
    M, N = 4, 64
    x, w, s, z, deq, mag = _problem(4, M, N, K, dt, zeros, K)
    off = 128.0 if act == "bf16" else 64.0
    q = torch.stack((w & 15, w >> 4), -1).reshape(N, K).float()
    zf = torch.zeros(N, K // 128) if z is None else z.float()
    ref = x.double() @ deq.t()

    def sums(keep, scale):
        y = torch.zeros(M, N)
        for g in range(K // 128):
            xg, k = x[:, 128 * g:128 * g + 128].float(), slice(128 * g, 128 * g + 128)
            acc = -(zf[:, g] + off) * xg.sum(1, keepdim=True)
            for e in range(0, 128, 16):
                acc = acc + xg[:, e:e + 16] @ (off + q[:, k][:, e:e + 16]).t()
            y = keep(y + s[:, g].float() * scale * acc)
        return (y.double() - ref).abs()

    same = lambda t: t
    bound = _sum_bound(x, deq, mag)
    assert bool((sums(same, 1.0) <= bound).all())
    assert not bool((sums(same, 1 + 2.0 ** -12) <= bound).all())
    if K > 128:
        assert not bool((sums(lambda t: t.bfloat16().float(), 1.0) <= bound).all())


def _call(qbits, x, w, s, z, bias, general=False):
    """y = x @ dequant(w)^T + bias; general: x two bytes off its alignment, which
    leaves every kernel but wq_general (the sizes' former route)."""
    M, K = x.shape
    N = w.shape[0]
    xd = x.cuda()
    if general:
        xd = torch.empty(M * K + 1, dtype=x.dtype, device="cuda")[1:].view(M, K).copy_(xd)
        assert xd.data_ptr() % 4 == 2
    y = torch.full((M, N), float("nan"), dtype=x.dtype, device="cuda")
    wd, sd, zd, bd = (None if t is None else t.cuda() for t in (w, s, z, bias))
    if qbits == 4:
        tm.int4_linear(xd, wd, bd, y, sd, zd, M, N, K, 128)
    else:
        tm.int8_linear(xd, wd, bd, y, sd, zd, M, N, K)
    return y.cpu().double()


# (qbits, M, N, K): sizes that wq_general took before these kernels, K no
# multiple of 256 or N of 64: the pipelined one and the short-K streaming ones
NEW_ROUTES = [(4, 228, 272, 1152), (4, 100, 272, 7040), (4, 40, 144, 3200), (4, 3, 48, 640),
              (4, 12, 4112, 1152), (4, 32, 272, 2176), (8, 5, 144, 1088), (8, 24, 272, 3264)]


@pytest.mark.gpu
@pytest.mark.parametrize("mean", [0.0, 1.0])
@pytest.mark.parametrize("act", ACT)
@pytest.mark.parametrize("zeros", [None, "s", "u"])
@pytest.mark.parametrize("qbits,M,N,K", NEW_ROUTES)
def test_no_further_from_64_bits_than_the_general_kernel(qbits, M, N, K, zeros, act, mean):
    """The error against 64 bits (2-norm) is wq_general's, up to the few results
    whose fp32 sum falls on the other side of a rounding (5e-4 of the error).
    Zero-points near the middle of the weights, activations with a mean too."""
    dt = ACT[act]
    x, w, s, z, deq, _ = _problem(qbits, M, N, K, dt, None, M + N)
    x = (x.float() + mean).to(dt)
    if zeros:
        z = 5 + 6 * torch.rand(s.shape, generator=torch.Generator().manual_seed(K))
        z = z.round().to(torch.uint8) if zeros == "u" else z.to(dt)
        rep = (1, 128) if qbits == 4 else (1, K)
        wide = lambda t: t.double().reshape(N, -1).repeat_interleave(rep[1], 1)
        deq = deq - wide(z) * wide(s)
    name = tm.wq_kernel_for(qbits, M, N, K, act_dtype=dt, zero_dtype=None if z is None else z.dtype)
    assert name[0] != "wq_general"
    ref = x.double() @ deq.t()
    err = [float((_call(qbits, x, w, s, z, None, general=g) - ref).norm()) for g in (False, True)]
    assert err[0] <= err[1] * (1 + 5e-4), (name[0], err[0] / err[1])


@pytest.mark.gpu
@pytest.mark.parametrize("act", ACT)
@pytest.mark.parametrize("zeros", [None, "s", "u"])
@pytest.mark.parametrize("qbits,M,N,K", NEW_ROUTES + [(4, 700, 7168, 512), (8, 40, 272, 1152)])
def test_infinite_activations(qbits, M, N, K, zeros, act):
    """An infinite activation gives an infinity of the weight's sign (NaN for a weight
    of exactly its zero-point), two of opposite signs NaN where they meet, and
    activations whose multiples overflow the sums stay finite: all as wq_general.
    Rows without one are untouched."""
    dt = ACT[act]
    x, w, s, z, deq, mag = _problem(qbits, M, N, K, dt, zeros, M + K)
    inf = float("inf")
    clean = _call(qbits, x, w, s, z, None)
    x[0, 5] = inf
    x[1, K - 1] = -inf
    x[2, 7], x[2, K - 70] = inf, inf
    x[M - 1, 3] = float("nan")
    if M > 4:
        x[3, 100], x[3, 101] = -inf, torch.finfo(dt).max
        x[M - 2, K // 2] = torch.finfo(dt).max / 64
    got, want = _call(qbits, x, w, s, z, None), _call(qbits, x, w, s, z, None, general=True)
    assert bool((got.isnan() == want.isnan()).all())
    assert bool((got.isinf() == want.isinf()).all())
    i = want.isinf()
    assert i.any() and torch.equal(got[i], want[i])
    f = want.isfinite()
    u = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    # a rounding apart, and the sums' own error (partial sums of at most x (OFF + q + z) s)
    tol = 2 * u * want[f].abs() + 2 * _sum_bound(x.nan_to_num(0, 0, 0), deq, mag)[f]
    assert bool(((got[f] - want[f]).abs() <= tol + 1e-6).all())
    assert torch.equal(got[4:M - 2], clean[4:M - 2])


@pytest.mark.gpu
def test_more_rows_than_a_grid_dimension_holds():
    """65536 rows and more (y and z of a grid end at 65535) on the pipelined int4
    path, whose copy of X has one row of workgroups per row of X."""
    M, N, K = 65600, 128, 256
    assert tm.wq_kernel_for(4, M, N, K)[0] == "wq_pipe_q4_f16_zn_r2"
    x, w, s, z, deq, _ = _problem(4, M, N, K, torch.float16, None, 9)
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    tm.int4_matmul(x.cuda(), w.cuda(), y, s.cuda(), None, M, N, K, 128)
    ref = x.cuda().double() @ deq.t().contiguous().cuda()
    err = (y.double() - ref).norm() / ref.norm()
    assert err < 2 * 2.0 ** -11, float(err)  # one rounding to fp16


def test_selection():
    """Sizes on both sides of the pipelined kernels' rules (no device is touched)."""
    k = lambda *a, **kw: tm.wq_kernel_for(*a, **kw, details=True)
    f16, bf16, u8 = torch.float16, torch.bfloat16, torch.uint8
    assert k(4, 228, 2816, 7040, act_dtype=bf16)["name"] == "wq_pipe_q4_bf16_zn_r2"
    assert k(4, 1000, 4096, 11008, zero_dtype=u8)["name"] == "wq_pipe_q4_f16_zu_r2"
    assert k(4, 1000, 4096, 4096, zero_dtype=u8)["name"].startswith("wq_wide_")
    assert k(8, 40, 1280, 3456)["name"] == "wq_pipe_q8_f16_zn_r1"
    # few rows and columns, on both sides
    pipe = lambda *a, **kw: k(*a, **kw)["name"].startswith("wq_pipe_")
    assert pipe(8, 1, 4112, 640) and not pipe(8, 1, 4096, 640) and not pipe(8, 1, 4096, 2432)
    assert pipe(4, 9, 2448, 384) and not pipe(4, 8, 2448, 384) and not pipe(8, 8, 272, 384)
    assert pipe(4, 5, 272, 128) and not pipe(4, 4, 272, 128) and pipe(8, 3, 272, 128)
    # without the workspace int4 stays where it was
    assert k(4, 228, 2816, 7040, with_workspace=False)["name"] == "wq_general"
    assert k(8, 700, 22016, 4096, with_workspace=False)["workspace_bytes"] == 0
    d = k(4, 40, 1280, 3712)
    assert d["splits"] > 1 and d["workspace_bytes"] >= d["splits"] * 40 * 1280 * 4 + 40 * 3712 * 2
    # short K with few columns streams 16- / 32-column workgroups: K a multiple of
    # 512 up to 64 rows, others up to 32
    assert k(4, 64, 4096, 4096)["name"] == "wq_streamk_q4_f16_zn_t1_x16m_c4"
    assert k(8, 16, 8192, 4096)["name"] == "wq_streamk_q8_f16_zn_t2_x16s_c8"
    assert k(8, 32, 1280, 3456)["name"] == "wq_streamk_q8_f16_zn_t1_x16m_c8"
    assert k(8, 16, 8208, 4096)["name"] == "wq_stream_q8_f16_zn_x16s"
    # zero-points of int8, and groups other than 128, are not theirs
    assert not k(8, 40, 1280, 3456, zero_dtype=f16)["name"].startswith("wq_pipe")
    assert not k(4, 40, 1280, 3456, 64)["name"].startswith("wq_pipe")


@pytest.mark.gpu
def test_small_workspace_keeps_the_other_kernels():
    """A workspace that the pipelined plan does not fit (too small for the slice
    sums, then for the permuted X) is no error: one slice, then the kernels that
    need none."""
    import ctypes
    from triton_metal_amd import _lib
    L = _lib.lib()
    M, N, K = 40, 272, 1152
    x, w, s, z, deq, mag = _problem(4, M, N, K, torch.float16, "u", 3)
    xd, wd, sd, zd = x.cuda(), w.cuda(), s.cuda(), z.cuda()
    need = tm.wq_kernel_for(4, M, N, K, zero_dtype=torch.uint8, details=True)["workspace_bytes"]
    ref = x.double() @ deq.t()
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    for nbytes in (need, need - 1, M * K * 2 + 4096, 1024):
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        y = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        rc = L.tm_wq_matmul_ws(4, p(xd), p(wd), None, p(y), p(sd), p(zd), M, N, K, 128,
                               _lib.TM_DT_F16, _lib.TM_DT_F16, _lib.TM_DT_U8, p(ws), nbytes, None)
        assert rc == 0, _lib.last_error()
        torch.cuda.synchronize()
        tol = 2.0 ** -11 * 1.01 * ref.abs() + _sum_bound(x, deq, mag) + 1e-6
        assert bool(((y.cpu().double() - ref).abs() <= tol).all()), nbytes


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["int4", "decode", "kda"])
def test_workspace_belongs_to_the_plans_stream(op):
    """A plan bound to a stream other than the current one takes its workspace from
    that stream's memory: not what the current stream freed a moment ago (its work
    there may still run), and what a dropped plan gives back (its own work may still
    run) does not go to the current stream's tensors.  Nothing is launched."""
    side = torch.cuda.Stream()
    zeros = lambda *s, dt=torch.float16: torch.zeros(*s, dtype=dt, device="cuda")
    if op == "int4":
        M, N, K = 300, 2816, 7040
        a = [zeros(M, K), zeros(N, K // 2, dt=torch.uint8), zeros(M, N), zeros(N, K // 128)]
        plan = lambda s: tm.plan_int4_matmul(*a, None, M, N, K, 128, stream=s)
        ws = lambda p: p._keep
    elif op == "decode":
        q, kv = zeros(2, 8, 128), zeros(2, 8, 8192, 128)
        o = torch.empty_like(q)
        plan = lambda s: tm.plan_decode_attention(q, kv, kv, o, stream=s)
        ws = lambda p: p._keep[1]
    else:
        bf = torch.bfloat16
        q, g, b = zeros(1, 640, 4, 128, dt=bf), zeros(1, 640, 4, 128, dt=torch.float32), zeros(
            1, 640, 4, dt=torch.float32)
        o = torch.empty_like(q)
        plan = lambda s: tm.plan_chunk_kda(q, q, q, g, b, o, stream=s)
        ws = lambda p: p._keep
    size = ws(plan(None)).numel()
    freed = torch.empty(size, dtype=torch.uint8, device="cuda")
    at = freed.data_ptr()
    del freed
    p = plan(side.cuda_stream)
    w = ws(p)
    assert w.numel() == size and w.data_ptr() != at
    at = w.data_ptr()
    del p, w
    assert torch.empty(size, dtype=torch.uint8, device="cuda").data_ptr() != at
    with torch.cuda.stream(side):
        assert torch.empty(size, dtype=torch.uint8, device="cuda").data_ptr() == at
