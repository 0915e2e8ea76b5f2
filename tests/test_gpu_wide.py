"""The wide parallel kernel (bf16, d <= 64 and dv <= 128 in eights; at d = 16 with dv <= 64 on small grids) at
the edges of its tiles, against 64 bits.  Bound: p = 1 + r with r rounded to fp16 (2^-11 relative) and
everything else in fp32, in the numerator and in the row sum, so |y - y64| <= (2^-11 + 2^-13)
(sum |r| |v| + |y| sum |r|) / den + N 2^-24 sum p |v| / den."""

import math

import pytest
import torch

from tests.helpers import rand_qkv

pytestmark = pytest.mark.gpu


def _check(q, k, v, y, den, scale, eps=1e-6):
    q, k, v = (x.double().cpu() for x in (q, k, v))
    N = q.shape[2]
    s = scale * q @ k.transpose(-2, -1)
    r = torch.tril(s + 0.5 * s * s)
    one = torch.tril(torch.ones(N, N, dtype=torch.float64))
    d64 = (r + one).sum(-1, keepdim=True)
    y64 = (r + one) @ v / (d64 + eps)
    mag = r.abs().sum(-1, keepdim=True)
    bound = (2.0 ** -11 + 2.0 ** -13) * (r.abs() @ v.abs() + y64.abs() * mag) / d64
    bound = bound + (N + 64) * 2.0 ** -24 * ((r.abs() + one) @ v.abs()) / d64 + 1e-30
    off = ((y.double().cpu() - y64).abs() / bound).max().item()
    offd = ((den.double().cpu() - d64[..., 0]).abs() / ((2.0 ** -11 + 2.0 ** -13) * mag[..., 0] + N * 2.0 ** -24 * d64[..., 0])).max().item()
    return off, offd


@pytest.mark.parametrize("B,H,N,d,dv", [
    (1, 1, 1, 64, 64), (1, 2, 31, 8, 8), (2, 1, 63, 24, 40), (1, 3, 64, 32, 32), (1, 1, 65, 40, 64), (1, 2, 127, 64, 72),
    (3, 1, 128, 16, 128), (1, 8, 129, 48, 96), (1, 1, 255, 56, 16), (2, 2, 257, 64, 128), (1, 2, 515, 32, 64),
    (4, 128, 257, 64, 64), (4, 128, 200, 32, 32), (2, 256, 130, 16, 72)])   # the last three: 256-query work-groups
@pytest.mark.parametrize("scale", [None, 0.09])
def test_edges(B, H, N, d, dv, scale):
    import kernels as K
    q, k, v = (x.cuda() for x in rand_qkv(B, H, N, d, dv, seed=N + d + dv, dtype=torch.bfloat16, scale_qk=0.7))
    y, den = K.based_parallel(q, k, v, scale=scale, out_dtype=torch.float32, return_den=True)
    off, offd = _check(q, k, v, y, den, 1.0 / math.sqrt(d) if scale is None else scale)
    assert off < 1 and offd < 1, (off, offd)
    assert torch.equal(K.based_parallel(q, k, v, scale=scale), y.bfloat16())


@pytest.mark.parametrize("H,N,dv,wide", [(2, 43520, 32, True), (2, 43777, 32, False), (3, 43520, 64, True), (32, 4090, 64, False),
                                         (8, 16128, 32, True), (8, 16129, 32, False)])
def test_d16_grids_on_both_sides_of_the_route_limits(H, N, dv, wide):
    """Fewer 256-query work-groups than two per CU (4/3 with fewer than 8 heads and dv <= 32) run the wide
    kernel, others the packed one; fp64 rows of the last head on either side."""
    import ctypes

    import kernels as K
    from kernels import _lib
    from tests.helpers import rows_fp64
    S = ctypes.c_longlong * 3
    s = [S(0, N * w, w) for w in (16, dv)]
    assert (_lib.lib().la_based_parallel_strided_workspace_bytes(1, H, N, 16, dv, s[0], s[1], s[1]) > 0) == wide
    q, k, v = rand_qkv(1, H, N, 16, dv, seed=N, dtype=torch.bfloat16, scale_qk=0.25)
    y = K.based_parallel(q.cuda(), k.cuda(), v.cuda(), out_dtype=torch.float32).cpu()
    rows = torch.tensor([0, 63, 255, 256, N // 2, N - 1])
    want = rows_fp64(q, k, v, 0, H - 1, rows)
    assert ((y[0, H - 1, rows].double() - want).norm() / want.norm()).item() < 1e-4


@pytest.mark.parametrize("dv", [32, 64])
@pytest.mark.parametrize("scale", [None, 0.3])
def test_d16_denominators_from_fp32_sums(dv, scale):
    """d = 16 calls on small grids that return denominators sum u in fp32: q.k sums 17 products in fp32, whose
    error e moves p by (1 + |s|) e, and N fp32 sums; nothing of fp16's 2^-11.  The output is that of a call
    without."""
    import kernels as K
    N = 900
    q, k, v = rand_qkv(1, 4, N, 16, dv, seed=dv, dtype=torch.bfloat16, scale_qk=1.0)
    y, den = K.based_parallel(q.cuda(), k.cuda(), v.cuda(), scale=scale, out_dtype=torch.float32, return_den=True)
    assert torch.equal(y, K.based_parallel(q.cuda(), k.cuda(), v.cuda(), scale=scale, out_dtype=torch.float32))
    q, k, c = q.double(), k.double(), 0.25 if scale is None else scale
    s = c * q @ k.transpose(-2, -1)
    one = torch.tril(torch.ones(N, N, dtype=torch.float64))
    p = (1.0 + s + 0.5 * s * s) * one
    reach = c * q.abs() @ k.abs().transpose(-2, -1) + 1.0
    bound = ((1.0 + s.abs()) * 18 * 2.0 ** -24 * reach * one + (N / 8 + 16) * 2.0 ** -24 * (p + 2 * one)).sum(-1)
    off = ((den.double().cpu() - p.sum(-1)).abs() / bound).max().item()
    assert off < 1, off


@pytest.mark.parametrize("dv", [32, 64, 128])
def test_v_exponents(dv):
    """Blocks of V that differ by many powers of two (one of them zero): each wave takes the largest
    exponent among its blocks, and smaller ones multiply apart."""
    import kernels as K
    q, k, v = rand_qkv(2, 2, 400, 64, dv, seed=dv, dtype=torch.bfloat16, scale_qk=0.7)
    f = torch.ones(400)
    # whole 64-key blocks: inside a block fp16 V^T holds 2^-14 of its largest value in full (bf16's 8 bits
    # down to 2^-24), so the bound, relative to each row's own terms, needs one magnitude per block
    f[64:128], f[128:192], f[192:256], f[256:320], f[320:] = 2.0 ** -30, 0.0, 2.0 ** 40, 2.0 ** 41, 2.0 ** 90
    v = (v.float() * f[:, None]).bfloat16()
    qd, kd, vd = (x.cuda() for x in (q, k, v))
    y, den = K.based_parallel(qd, kd, vd, out_dtype=torch.float32, return_den=True)
    off, offd = _check(q, k, v, y, den, 0.125)
    assert off < 1 and offd < 1, (off, offd)


@pytest.mark.parametrize("B,H,d,dv", [(2, 2, 64, 64), (1, 3, 16, 128), (4, 128, 32, 32), (4, 128, 64, 64)])
@pytest.mark.parametrize("std", [0.13, 2.0 ** -9])
def test_v_exponents_a_step_apart(B, H, d, dv, std):
    """V whose blocks lie on both sides of a step of their exponents (largest values 0.3 to 0.7), and 2^8
    below it every third block: lower blocks take u by 2^-8, rounded at 2^-25 (2^-16 of W = 0.18 to 0.71, the
    weight of the 1 of p), and by 2^-16 they multiply apart.  Parallel and chunked calls."""
    import kernels as K
    N = 4500 if B * H < 8 else 700          # more than 64 blocks
    q, k, v = rand_qkv(B, H, N, d, dv, seed=dv, dtype=torch.bfloat16, scale_qk=0.7)
    v = v.float() * std
    v[:, :, (torch.arange(N) // 64) % 3 == 1] *= 0.13 / 2.0 ** 7
    v = v.bfloat16()
    qd, kd, vd = (x.cuda() for x in (q, k, v))
    y, den = K.based_parallel(qd, kd, vd, scale=0.09, out_dtype=torch.float32, return_den=True)
    num = K.based_chunked(qd, kd, vd, scale=0.09, normalize=False, out_dtype=torch.float32)
    y, den, num = (x[-1:, -2:].double().cpu() for x in (y, den, num))
    q, k, v = (x[-1:, -2:].double() for x in (q, k, v))
    n64, d64, en, ed = _chunked_terms(q, k, v, 0.09)
    one = torch.tril(torch.ones(N, N, dtype=torch.float64))
    r = (0.09 * q @ k.transpose(-2, -1)) * one
    r = r + 0.5 * r * r
    step = 2.0 ** -15 * one + (2.0 ** -11 + 2.0 ** -13) * r.abs()     # fp16 u in every row, or by 2^-8
    en = en + step @ v.abs() + (N + 64) * 2.0 ** -24 * ((r.abs() + one) @ v.abs())
    ed = ed + step.sum(-1, keepdim=True)
    off = ((num - n64).abs() / en).max().item()
    assert off < 1, off
    y64 = n64 / (d64 + 1e-6)
    off = ((y - y64).abs() / ((en + y64.abs() * ed) / d64)).max().item()
    offd = ((den[..., None] - d64).abs() / ed).max().item()
    assert off < 1.01 and offd < 1, (off, offd)


def test_pre_pass_apart_and_misaligned():
    """The two halves apart equal the whole call; an output that is not 16-byte aligned takes the
    register-staged kernel, after the same pre-pass too."""
    from kernels import _lib
    L = _lib.lib()
    B, H, N, d, dv = 1, 3, 300, 64, 64
    q, k, v = (x.cuda() for x in rand_qkv(B, H, N, d, dv, seed=5, dtype=torch.bfloat16, scale_qk=0.7))
    n = int(L.la_based_parallel_workspace_bytes(B, H, N, d, dv, 1))
    st = torch.cuda.current_stream().cuda_stream
    buf = torch.empty(B * H * N * dv + 8, device="cuda")
    outs = []
    for skew, apart in ((0, False), (0, True), (1, False), (1, True)):
        ws = torch.full((n,), 0x7f, dtype=torch.uint8, device="cuda")
        out = buf[skew:skew + B * H * N * dv]
        args = (B, H, N, d, dv)
        if apart:
            assert L.la_based_parallel_pack(k.data_ptr(), v.data_ptr(), 1, *args, ws.data_ptr(), n, st) == 0
        f = L.la_based_parallel_fwd_packed if apart else L.la_based_parallel_fwd
        assert f(q.data_ptr(), k.data_ptr(), v.data_ptr(), 1, out.data_ptr(), 0, None, *args, 0.125, 1e-6, 1, ws.data_ptr(),
                 n, st) == 0
        outs.append(out.clone().view(B, H, N, dv))
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[2], outs[3])
    for y in outs[::2]:
        assert _check(q, k, v, y, torch.zeros(1), 0.125)[0] < 1


def _chunked_terms(q, k, v, c):
    """Numerator and denominator in 64 bits, and what a chunked call may be off them by: below row 512 p is
    bf16 hi + lo (2^-17 relative), from there on r = p - 1 of earlier blocks fp16 (2^-11); q.k sums d + 1
    products in fp32, p turns an error e of s into (1 + |s|) e; N fp32 sums."""
    N, d = q.shape[-2], q.shape[-1]
    s = c * q @ k.transpose(-2, -1)
    one = torch.tril(torch.ones(N, N, dtype=torch.float64))
    r = (s + 0.5 * s * s) * one
    reach = c * q.abs() @ k.abs().transpose(-2, -1)
    ep = (1.0 + s.abs()) * (d + 2) * 2.0 ** -23 * (reach + 1.0) * one + (N + 64) * 2.0 ** -23 * (r.abs() + one)
    rel = torch.where(torch.arange(N) < 512, 2.0 ** -17, 2.0 ** -11 + 2.0 ** -13).double()[:, None]
    ep = ep + rel * torch.where(rel > 2.0 ** -17, r.abs(), r + one)
    return (r + one) @ v, (r + one).sum(-1, keepdim=True), ep @ v.abs(), ep.sum(-1, keepdim=True)


@pytest.mark.parametrize("big", [1.0, 30.0, 3000.0])
@pytest.mark.parametrize("B,H,N,d,dv", [(1, 2, 513, 64, 64), (1, 2, 700, 32, 128), (4, 128, 514, 64, 32), (1, 3, 1024, 24, 16),
                                        (4, 128, 1100, 8, 72), (4, 128, 800, 64, 64)])
def test_chunked_calls_any_scores(B, H, N, d, dv, big):
    """Chunked calls of several segments take this kernel too, with scores of any size: some queries and
    keys are `big` times the others; numerator and normalised."""
    import kernels as K
    q, k, v = rand_qkv(B, H, N, d, dv, seed=N + d, dtype=torch.float32, scale_qk=0.7)
    q[:, :, 5::7] *= big
    k[:, :, 3::11] *= big
    q, k, v = (x.bfloat16() for x in (q, k, v))
    qd, kd, vd = (x.cuda() for x in (q, k, v))
    y = K.based_chunked(qd, kd, vd, out_dtype=torch.float32)
    num = K.based_chunked(qd, kd, vd, normalize=False, out_dtype=torch.float32)
    heads = slice(0, 2)          # the oracle's N x N in 64 bits: two heads of the last batch
    q, k, v = (x[-1:, heads].double() for x in (q, k, v))
    n64, d64, en, ed = _chunked_terms(q, k, v, 1.0 / math.sqrt(d))
    off = ((num[-1:, heads].double().cpu() - n64).abs() / en).max().item()
    assert off < 1, off
    y64 = n64 / (d64 + 1e-6)
    off = ((y[-1:, heads].double().cpu() - y64).abs() / ((en + y64.abs() * ed) / d64)).max().item()
    assert off < 1.01, off


@pytest.mark.parametrize("N,d,dv", [(900, 64, 64), (1300, 16, 128), (700, 32, 32)])
def test_chunked_calls_as_exact_as_the_segment_path(N, d, dv):
    """Relative errors of fp32 outputs, q and k four times the benchmark's: 2.6e-6 in the first 512 rows and
    1.6e-4 to 2e-4 after them on the segment path (with u in fp16 for all rows: 5e-5 to 1.4e-4 in the first)."""
    import kernels as K
    q, k, v = rand_qkv(1, 3, N, d, dv, seed=N, dtype=torch.bfloat16, scale_qk=4.0 / math.sqrt(d))
    y = K.based_chunked(q.cuda(), k.cuda(), v.cuda(), out_dtype=torch.float32).double().cpu()
    n64, d64, _, _ = _chunked_terms(q.double(), k.double(), v.double(), 1.0 / math.sqrt(d))
    y64 = n64 / (d64 + 1e-6)
    first, rest = (((y - y64)[:, :, r].norm() / y64[:, :, r].norm()).item() for r in (slice(0, 512), slice(512, N)))
    assert first < 4e-6 and rest < 2e-4, (first, rest)


@pytest.mark.parametrize("d,dv", [(64, 64), (32, 128), (64, 32)])
def test_chunked_calls_are_causal(d, dv):
    """A huge key or value changes no bit of an earlier row, in its own 64-token block or before."""
    import kernels as K
    N = 1090
    q, k, v = (x.cuda() for x in rand_qkv(1, 2, N, d, dv, seed=d, dtype=torch.bfloat16, scale_qk=0.7))
    want = K.based_chunked(q, k, v, out_dtype=torch.float32)
    for t in (50, 500, 520, 690, 1000, 1085):
        kb, vb = k.clone(), v.clone()
        kb[:, :, t] *= 3e5
        vb[:, :, t] *= 1e20
        y = K.based_chunked(q, kb, vb, out_dtype=torch.float32)
        assert torch.equal(y[:, :, :t], want[:, :, :t]), t


def test_chunked_calls_small_value_columns():
    """A column of V 2^-30 below the others, which one fp16 exponent per block could not hold."""
    import kernels as K
    q, k, v = rand_qkv(1, 2, 1100, 64, 64, seed=3, dtype=torch.bfloat16, scale_qk=0.7)
    v = (v.float() * torch.where(torch.arange(64) % 8 == 3, 2.0 ** -30, 1.0)).bfloat16()
    num = K.based_chunked(q.cuda(), k.cuda(), v.cuda(), normalize=False, out_dtype=torch.float32).double().cpu()
    n64, _, en, _ = _chunked_terms(q.double(), k.double(), v.double(), 0.125)
    off = ((num - n64).abs() / en).max().item()
    assert off < 1, off


@pytest.mark.parametrize("B,N,H,d", [(1, 65, 2, 64), (3, 200, 4, 24), (2, 257, 16, 16), (2, 2048, 32, 64), (1, 130, 3, 8)])
def test_strided_projection_equals_copies(B, N, H, d):
    """q, k, v read in place in a (b, t, 3, h, d) projection and the heads written merged: bit for bit
    what the same kernel gives on contiguous copies."""
    import kernels as K
    from kernels import pytorch_attention as P
    g = torch.Generator(device="cuda").manual_seed(N)
    qkv = (torch.randn(B, N, 3, H, d, generator=g, device="cuda") / math.sqrt(math.sqrt(d))).bfloat16()
    y = P.parallel_from_projection(qkv, 1e-6)
    q, k, v = qkv.permute(2, 0, 3, 1, 4).contiguous().unbind(0)
    assert y is not None and torch.equal(y, K.solution_nki(q, k, v).transpose(1, 2).reshape(B, N, H * d))


@pytest.mark.parametrize("B,H,N,d,dv", [(2, 3, 65, 64, 40), (3, 2, 200, 24, 72), (1, 5, 130, 16, 48), (2, 128, 257, 8, 24)])
def test_strides_wider_than_the_data(B, H, N, d, dv):
    """q and k, v and the output each with batch, head and token strides of their own that leave gaps, the
    output inside a buffer of sentinels: values of the contiguous call, every element between, before and
    after them untouched."""
    import ctypes

    import kernels as K
    from kernels import _lib
    L = _lib.lib()
    q, k, v = (x.cuda() for x in rand_qkv(B, H, N, d, dv, seed=N + d, dtype=torch.bfloat16, scale_qk=0.7))
    S = ctypes.c_longlong * 3

    def strides(w, head_gap, row_gap, batch_gap):
        head = w + head_gap
        row = H * head + row_gap
        return (N * row + batch_gap, head, row)

    def place(x, st, lead, fill=float("nan")):
        buf = torch.full((lead + B * st[0] + 64,), fill, dtype=torch.bfloat16, device="cuda")
        view = buf[lead:].as_strided((B, H, N, x.shape[-1]), (*st, 1))
        view.copy_(x)
        return buf, view

    sk, sv, so = strides(d, 8, 16, 24), strides(dv, 0, 8, 64), strides(dv, 16, 40, 8)
    (_, qv), (_, kv), (_, vv) = place(q, sk, 64), place(k, sk, 8), place(v, sv, 16)
    out, ov = place(torch.full_like(v, -7.0), so, 64, -7.0)
    n = int(L.la_based_parallel_workspace_bytes(B, H, N, d, dv, 1))
    ws = torch.full((n + 64,), 0x7f, dtype=torch.uint8, device="cuda")
    assert L.la_based_parallel_fwd_strided(qv.data_ptr(), kv.data_ptr(), vv.data_ptr(), ov.data_ptr(), B, H, N, d, dv,
                                           S(*sk), S(*sv), S(*so), 1.0 / math.sqrt(d), 1e-6, ws.data_ptr(), n,
                                           torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(ov, K.based_parallel(q, k, v))
    ov.fill_(-7.0)
    assert (out == -7.0).all() and (ws[n:] == 0x7f).all()


@pytest.mark.parametrize("B,N,H,d", [(8, 4096, 16, 16), (1, 64, 2, 64), (1, 300, 2, 72)])
def test_refused_projections_allocate_nothing(B, N, H, d):
    """Shapes that the strided kernel does not take (the packed kernel's grids, one block, other dims)."""
    from kernels import pytorch_attention as P
    qkv = torch.zeros(B, N, 3, H, d, dtype=torch.bfloat16, device="cuda")
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    assert P.parallel_from_projection(qkv, 1e-6) is None
    assert torch.cuda.memory_stats()["allocation.all.allocated"] == before


def test_strided_arguments():
    import ctypes

    from kernels import _lib
    L = _lib.lib()
    x = torch.zeros(1, 128, 3, 2, 64, dtype=torch.bfloat16, device="cuda")
    n = int(L.la_based_parallel_workspace_bytes(1, 2, 128, 64, 64, 1))
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    S = ctypes.c_longlong * 3

    def call(N=128, d=64, k=(49152, 64, 384), ptr=x.data_ptr(), bytes_=n):
        return L.la_based_parallel_fwd_strided(ptr, ptr, ptr, x.data_ptr(), 1, 2, N, d, 64, S(*k), S(*k), S(*k), 0.125, 1e-6,
                                               ws.data_ptr(), bytes_, torch.cuda.current_stream().cuda_stream)

    assert call(k=(49152, 64, 380)) == -8 and call(ptr=x.data_ptr() + 2) == -8 and call(k=(0, -64, 384)) == -2
    assert call(N=64) == -5 and call(d=60) == -5 and call(d=72) == -5 and call(k=(49152, 64, 56)) == -5
    assert call(bytes_=n - 1) == -6 and call(N=0) == 0

    def need(N=128, d=64, k=(49152, 64, 384), out=(8192, 64, 128)):
        return L.la_based_parallel_strided_workspace_bytes(1, 2, N, d, 64, S(*k), S(*k), S(*out))

    assert need() == n and need(k=(49152, 64, 380)) == 0 and need(k=(0, -64, 384)) == 0 and need(N=0) == 0
    assert need(N=64) == 0 and need(d=72) == 0 and need(out=(8192, 64, 56)) == 0 and need(N=-1) == 0


@pytest.mark.parametrize("B,H,N,dv", [(1, 1, 65, 64), (2, 3, 200, 40), (1, 2, 1100, 64), (2, 4, 129, 24), (1, 3, 640, 32)])
def test_v_aligned_to_8_bytes_only(B, H, N, dv):
    """d = 16 calls on small grids whose V is not 16-byte aligned stay on the packed kernel, with 128-query
    work-groups; the whole call and the pre-pass apart."""
    from kernels import _lib
    L = _lib.lib()
    q, k, v = (x.cuda() for x in rand_qkv(B, H, N, 16, dv, seed=N, dtype=torch.bfloat16, scale_qk=0.7))
    buf = torch.empty(v.numel() + 4, dtype=torch.bfloat16, device="cuda")
    buf[4:] = v.view(-1)
    n = int(L.la_based_parallel_workspace_bytes(B, H, N, 16, dv, 1))
    st = torch.cuda.current_stream().cuda_stream
    outs = []
    for apart in (False, True):
        ws = torch.full((n,), 0x7f, dtype=torch.uint8, device="cuda")
        out, den = torch.empty(B, H, N, dv, device="cuda"), torch.empty(B, H, N, device="cuda")
        if apart:
            assert L.la_based_parallel_pack(k.data_ptr(), buf[4:].data_ptr(), 1, B, H, N, 16, dv, ws.data_ptr(), n, st) == 0
        f = L.la_based_parallel_fwd_packed if apart else L.la_based_parallel_fwd
        assert f(q.data_ptr(), k.data_ptr(), buf[4:].data_ptr(), 1, out.data_ptr(), 0, den.data_ptr(), B, H, N, 16, dv,
                 0.25, 1e-6, 1, ws.data_ptr(), n, st) == 0
        outs.append(out)
    off, offd = _check(q, k, v, outs[0], den, 0.25)
    assert off < 1 and offd < 1 and torch.equal(*outs), (off, offd)


@pytest.mark.parametrize("apart", [False, True])
def test_workspace_of_the_maxima_alone(apart):
    """256 bytes a head, which these shapes took before the wide kernel, still suffice."""
    from kernels import _lib
    L = _lib.lib()
    B, H, N, d, dv = 1, 3, 300, 64, 64
    q, k, v = (x.cuda() for x in rand_qkv(B, H, N, d, dv, seed=5, dtype=torch.bfloat16, scale_qk=0.7))
    assert int(L.la_based_parallel_workspace_bytes(B, H, N, d, dv, 1)) > 256 * H
    st = torch.cuda.current_stream().cuda_stream
    ws = torch.full((256 * H + 64,), 0x7f, dtype=torch.uint8, device="cuda")
    out = torch.empty(B, H, N, dv, device="cuda")
    f = L.la_based_parallel_fwd_packed if apart else L.la_based_parallel_fwd

    def call(n):
        if apart:
            assert L.la_based_parallel_pack(k.data_ptr(), v.data_ptr(), 1, B, H, N, d, dv, ws.data_ptr(), 256 * H, st) == 0
        return f(q.data_ptr(), k.data_ptr(), v.data_ptr(), 1, out.data_ptr(), 0, None, B, H, N, d, dv, 0.125, 1e-6, 1,
                 ws.data_ptr(), n, st)

    assert call(256 * H) == 0 and call(256 * H - 1) == -6
    assert _check(q, k, v, out, torch.zeros(1), 0.125)[0] < 1
    assert (ws[256 * H:] == 0x7f).all()
