"""The state kernels of the segment-state shapes (la_based_state_export, la_based_state_apply) at the
edges of their tiles, against 64 bits.  Bounds: every output is a fp32 sum of exact products, so it is off
by at most steps 2^-24 times the sum of the magnitudes of its terms, steps the additions in a row (two
MFMAs for each 16 tokens, and the parts; three for each 16 features)."""

import math

import pytest
import torch

from oracle import reference as ref
from tests.helpers import rand_qkv

pytestmark = pytest.mark.gpu


def _call(fn, *args):
    from kernels import _lib
    _lib.check(getattr(_lib.lib(), fn)(*args, torch.cuda.current_stream().cuda_stream), fn)


def _ws(B, H, N, d, dv):
    from kernels import _lib
    n = int(_lib.lib().la_based_state_workspace_bytes(B, H, N, d, dv))
    return torch.full((n,), 0x7f, dtype=torch.uint8, device="cuda"), n


def _phi(x, scale):
    d = x.shape[-1]
    return ref.taylor_feature_map(x.double() * math.sqrt(scale * math.sqrt(d)))


def _inputs(B, H, N, d, dv, kscale=1.0, vscale=1.0):
    q, k, v = rand_qkv(B, H, N, d, dv, seed=N + 131 * d + dv, dtype=torch.float32, scale_qk=0.7)
    return (q * kscale).bfloat16(), (k * kscale).bfloat16(), (v * vscale).bfloat16()


CASES = [(1, 1, 1, 64, 64), (2, 1, 63, 33, 31), (1, 3, 64, 32, 32), (1, 2, 65, 31, 33), (2, 2, 129, 64, 65),
         (1, 2, 300, 16, 128), (1, 1, 513, 17, 1), (3, 1, 257, 1, 7), (1, 1, 1100, 63, 100), (4, 16, 200, 48, 64),
         (8, 12, 130, 64, 96)]


@pytest.mark.parametrize("with_state", [False, True])
@pytest.mark.parametrize("B,H,N,d,dv", CASES)
def test_export(B, H, N, d, dv, with_state):
    _, k, v = _inputs(B, H, N, d, dv)
    scale = 1.0 / math.sqrt(d)
    ph, vx = _phi(k, scale).transpose(-2, -1), torch.cat([v.double(), torch.ones(B, H, N, 1, dtype=torch.float64)], -1)
    old = torch.randn(B, H, ph.shape[-2], dv + 1) if with_state else torch.zeros(B, H, ph.shape[-2], dv + 1)
    want, mag = ph @ vx + old.double(), ph.abs() @ vx.abs() + old.abs().double()
    ws, n = _ws(B, H, N, d, dv)
    old_d, out = old.cuda(), torch.full_like(old, float("nan"), device="cuda")
    kd, vd = k.cuda(), v.cuda()
    _call("la_based_state_export", kd.data_ptr(), vd.data_ptr(), 1, old_d.data_ptr() if with_state else None,
          out.data_ptr(), B, H, N, d, dv, scale, ws.data_ptr(), n)
    off = ((out.cpu().double() - want).abs() / mag.clamp_min(1e-30)).max().item()
    assert off < (N / 8 + 16) * 2.0 ** -24, off
    if with_state:   # in place
        _call("la_based_state_export", kd.data_ptr(), vd.data_ptr(), 1, old_d.data_ptr(), old_d.data_ptr(), B, H, N, d,
              dv, scale, ws.data_ptr(), n)
        assert torch.equal(old_d, out)


@pytest.mark.parametrize("normalize", [0, 1])
@pytest.mark.parametrize("B,H,N,d,dv", CASES + [(2, 8, 4200, 64, 32)])
def test_apply(B, H, N, d, dv, normalize):
    q, _, _ = _inputs(B, H, N, d, dv)
    scale, eps = 0.8 / math.sqrt(d), 1e-6
    F = 1 + d + d * (d + 1) // 2
    g = torch.Generator().manual_seed(N)
    st = torch.randn(B, H, F, dv + 1, generator=g) * torch.exp(torch.randn(B, H, F, 1, generator=g))
    st[..., dv] = st[..., dv].abs()
    st[:, :, 0, dv] += 4.0 * F      # denominators away from zero
    num, den = torch.randn(B, H, N, dv, generator=g), torch.rand(B, H, N, generator=g) + 1
    ph = _phi(q, scale)
    tot, mag = ph @ st.double(), ph.abs() @ st.abs().double()
    tn, td = tot[..., :dv] + num.double(), tot[..., dv] + den.double()
    rel = (F / 8 + 16) * 2.0 ** -24 + 2.0 ** -21
    en, ed = rel * (mag[..., :dv] + num.abs().double()), rel * (mag[..., dv] + den.double())
    if normalize:
        want = tn / (td + eps).unsqueeze(-1)
        bound = (en + want.abs() * ed.unsqueeze(-1)) / td.abs().unsqueeze(-1)
    else:
        want, bound = tn, en
    ws, n = _ws(B, H, N, d, dv)
    nd, dd, qd, sd = num.cuda(), den.cuda(), q.cuda(), st.cuda()
    out = torch.full((B, H, N, dv), float("nan"), device="cuda")
    args = (qd.data_ptr(), 1, sd.data_ptr(), nd.data_ptr(), dd.data_ptr())
    tail = (0, B, H, N, d, dv, scale, eps, normalize, ws.data_ptr(), n)
    _call("la_based_state_apply", *args, out.data_ptr(), *tail)
    off = ((out.cpu().double() - want).abs() / bound).max().item()
    assert off < 1.1, off      # 1.1: the quotient's own rounding
    _call("la_based_state_apply", *args, nd.data_ptr(), *tail)   # over the numerator
    assert torch.equal(nd, out)


@pytest.mark.parametrize("kscale,vscale", [(1e-12, 1e-20), (1e3, 1e20), (0.0, 1.0), (1.0, 0.0), (64.0, 2.0 ** -100)])
def test_scales(kscale, vscale):
    """Powers far from one and zeros."""
    B, H, N, d, dv = 1, 2, 200, 64, 64
    q, k, v = _inputs(B, H, N, d, dv, kscale, vscale)
    scale = 1.0 / math.sqrt(d)
    vx = torch.cat([v.double(), torch.ones(B, H, N, 1, dtype=torch.float64)], -1)
    ph = _phi(k, scale).transpose(-2, -1)
    want, mag = ph @ vx, ph.abs() @ vx.abs()
    ws, n = _ws(B, H, N, d, dv)
    st = torch.full(want.shape, float("nan"), device="cuda", dtype=torch.float32)
    kd, vd, qd = k.cuda(), v.cuda(), q.cuda()
    _call("la_based_state_export", kd.data_ptr(), vd.data_ptr(), 1, None, st.data_ptr(), B, H, N, d, dv, scale,
          ws.data_ptr(), n)
    off = (st.cpu().double() - want).abs() - (N / 8 + 16) * 2.0 ** -24 * mag
    assert float(off.max()) <= 1e-36      # fp32 subnormals
    num, den = torch.zeros(B, H, N, dv, device="cuda"), torch.zeros(B, H, N, device="cuda")
    out = torch.empty_like(num)
    _call("la_based_state_apply", qd.data_ptr(), 1, st.data_ptr(), num.data_ptr(), den.data_ptr(), out.data_ptr(), 0, B,
          H, N, d, dv, scale, 0.0, 1, ws.data_ptr(), n)
    pq, s64 = _phi(q, scale), st.cpu().double()
    z = (pq @ s64[..., dv:])
    y, m = (pq @ s64[..., :dv]) / z, (pq.abs() @ s64.abs()[..., :dv]) / z
    rel = 2 * ((ph.shape[-2] / 8 + 16) * 2.0 ** -24 + 2.0 ** -21)
    assert float(((out.cpu().double() - y).abs() - rel * m).max()) <= 1e-36


def _export(k, v, scale=0.125):
    B, H, N, d = k.shape
    dv = v.shape[-1]
    ws, n = _ws(B, H, N, d, dv)
    st = torch.full((B, H, 1 + d + d * (d + 1) // 2, dv + 1), float("nan"), device="cuda")
    kd, vd = k.cuda(), v.cuda()
    _call("la_based_state_export", kd.data_ptr(), vd.data_ptr(), 1, None, st.data_ptr(), B, H, N, d, dv, scale,
          ws.data_ptr(), n)
    return st.cpu().double()


@pytest.mark.parametrize("big", [1e3, 1e5, 1e12])
@pytest.mark.parametrize("what", ["channel", "token", "sink", "column"])
@pytest.mark.parametrize("d,dv", [(64, 64), (32, 40)])
def test_export_of_uneven_inputs(d, dv, what, big):
    """One key channel, one token's keys (with its values, or with zeros as of an attention sink) or one
    value column far above the rest: every entry still within the bound of its own terms."""
    _, k, v = (x.float() for x in _inputs(1, 2, 1100, d, dv))
    if what == "channel":
        k[..., d // 3] *= big
    elif what == "column":
        v[..., dv // 3] *= big
    else:
        k[:, :, 500] *= big
        v[:, :, 500] *= what == "token"
    k, v = k.bfloat16(), v.bfloat16()
    vx = torch.cat([v.double(), torch.ones(1, 2, 1100, 1, dtype=torch.float64)], -1)
    ph = _phi(k, 0.125).transpose(-2, -1)
    off = ((_export(k, v) - ph @ vx).abs() / (ph.abs() @ vx.abs())).max().item()
    assert off < (1100 / 8 + 16) * 2.0 ** -24, off


def test_export_of_infinite_keys():
    """The rows of an infinite key are infinite (its K-sums too), of the sign of their products, and so are
    sums that overflow (another head); the others as without it."""
    _, k, v = _inputs(1, 2, 300, 64, 64)
    k[0, 0, 70, 5] = float("inf")
    k[0, 1, 200], v[0, 1, 200] = 1.0, 64.0
    k[0, 1, 200, 9] = 3e38
    got = _export(k, v)
    vx = torch.cat([v.double(), torch.ones(1, 2, 300, 1, dtype=torch.float64)], -1)
    ph = _phi(k, 0.125).transpose(-2, -1)
    want, m = ph @ vx, ph.abs() @ vx.abs()
    inf = want.abs() > 2e38
    assert inf[0, 0].any() and inf[0, 1].any() and not want.isnan().any()
    big = got.abs() > 2e38
    assert torch.equal(big, inf) and torch.equal(got[big].sign(), want[inf].sign())
    assert ((got - want).abs()[~inf] / m[~inf]).max().item() < (300 / 8 + 16) * 2.0 ** -24


def _apply(q, st, num, den, scale, eps, normalize):
    B, H, N, d = q.shape
    dv = num.shape[-1]
    ws, n = _ws(B, H, N, d, dv)
    qd, sd, nd, dd = (x.cuda() for x in (q, st, num, den))
    out = torch.full((B, H, N, dv), float("nan"), device="cuda")
    _call("la_based_state_apply", qd.data_ptr(), 1, sd.data_ptr(), nd.data_ptr(), dd.data_ptr(), out.data_ptr(), 0, B, H,
          N, d, dv, scale, eps, normalize, ws.data_ptr(), n)
    return out.cpu().double()


@pytest.mark.parametrize("N,d,dv", [(300, 64, 64), (130, 32, 128), (70, 16, 24)])
@pytest.mark.parametrize("what", ["columns", "entries", "queries"])
def test_apply_of_uneven_inputs(N, d, dv, what):
    """Value columns 2^-28 below the others, entries of the state of any power, one query channel far above
    the rest: every output within the bound of its own terms (exact entries: no 2^-21)."""
    q, _, _ = _inputs(1, 2, N, d, dv)
    F = 1 + d + d * (d + 1) // 2
    g = torch.Generator().manual_seed(N + len(what))
    st = torch.randn(1, 2, F, dv + 1, generator=g)
    if what == "columns":
        st[..., 2:dv:8] *= 2.0 ** -28
    elif what == "entries":
        st = torch.ldexp(st, torch.randint(-40, 40, st.shape, generator=g))
    else:
        q[..., d // 3] *= 3e4
    num, den = torch.zeros(1, 2, N, dv), torch.zeros(1, 2, N)
    ph = _phi(q, 0.8 / math.sqrt(d))
    want, mag = ph @ st[..., :dv].double(), ph.abs() @ st[..., :dv].abs().double()
    off = ((_apply(q, st, num, den, 0.8 / math.sqrt(d), 0.0, 0) - want).abs() / mag).max().item()
    assert off < (F / 8 + 16) * 2.0 ** -24, off


def test_apply_of_infinite_entries():
    """Infinite entries of the state make their column's numerators infinite, of the sign of the feature."""
    q, _, _ = _inputs(1, 1, 200, 64, 64)
    st = torch.randn(1, 1, 2145, 65, generator=torch.Generator().manual_seed(3))
    rows = (3, 70, 1000)        # a linear, a square and an off-diagonal feature
    for f, c in zip(rows, (0, 5, 40)):
        st[0, 0, f, c] = float("inf")
    num, den = torch.zeros(1, 1, 200, 64), torch.zeros(1, 1, 200)
    ph = _phi(q, 0.125)
    assert (ph != 0).all()
    got = _apply(q, st, num, den, 0.125, 0.0, 0)
    want, mag = ph @ st[..., :64].double(), ph.abs() @ st[..., :64].abs().double()
    inf = want.isinf()
    assert inf[..., [0, 5, 40]].all() and torch.equal(got[inf], want[inf])
    assert ((got - want).abs()[~inf] / mag[~inf]).max().item() < (2145 / 8 + 16) * 2.0 ** -24


def _need_gib(n):
    if torch.cuda.mem_get_info()[0] < n * 2 ** 30:
        pytest.skip(f"needs {n} GiB of device memory")


def test_export_of_a_sequence_past_2_32_bytes_of_chunks():
    """One part of 11.3 M tokens, 24 KB of converted rows per 64: the last tokens' offsets pass 2^32.  Zeros
    but for the first and the last tokens, whose state alone is the reference."""
    _need_gib(120)
    B, H, N, d, dv, n1 = 1, 8, 11_300_000, 64, 128, 640
    k = torch.zeros(B, H, N, d, dtype=torch.bfloat16, device="cuda")
    v = torch.zeros(B, H, N, dv, dtype=torch.bfloat16, device="cuda")
    _, k1, v1 = (x.cuda() for x in _inputs(B, H, 2 * n1, d, dv))
    for x, x1 in ((k, k1), (v, v1)):
        x[:, :, :n1] = x1[:, :, :n1]
        x[:, :, N - n1:] = x1[:, :, n1:]
    out = []
    for kk, vv, n in ((k, v, N), (k1, v1, 2 * n1)):
        ws, nb = _ws(B, H, n, d, dv)
        st = torch.empty(B, H, 2145, dv + 1, device="cuda")
        _call("la_based_state_export", kk.data_ptr(), vv.data_ptr(), 1, None, st.data_ptr(), B, H, n, d, dv, 0.125,
              ws.data_ptr(), nb)
        out.append(st)
        del ws
    assert (out[0][:, :, 0, dv] == N).all()
    out[1][:, :, 0, dv] = N
    assert ((out[0] - out[1]).norm() / out[1][:, :, 1:].norm()).item() < 1e-5
    del k, v, out
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_chunked_sequence_past_2_32_bytes(dtype):
    """The segment states of 10.9 M tokens (25 KB of converted rows per 64; fp32 rows of v past 2^32 bytes):
    the last row's numerator against the 512 tokens that are not zero.  In bf16 the fp16 prefix holds them with
    one exponent beside the count of all tokens: 5 % off at this length, 2e-4 at 20000 (resources that wrapped
    gave zeros, 100 %)."""
    _need_gib(120)
    import kernels as K
    N, d, dv, n1, at = 10_900_000, 64, 128, 512, 10_800_000
    q = torch.zeros(1, 1, N, d, dtype=dtype, device="cuda")
    k, v = torch.zeros_like(q), torch.zeros(1, 1, N, dv, dtype=dtype, device="cuda")
    q1, k1, v1 = (x.to(dtype).cuda() for x in rand_qkv(1, 1, n1, d, dv, seed=1, dtype=torch.bfloat16, scale_qk=0.7))
    k[:, :, at:at + n1], v[:, :, at:at + n1], q[:, :, N - 1] = k1, v1, q1[:, :, 0]
    num = K.based_chunked(q, k, v, normalize=False, out_dtype=torch.float32)[0, 0, N - 1].double().cpu()
    s = (k1[0, 0].double() @ q1[0, 0, 0].double()).cpu() / 8
    p = 1 + s + 0.5 * s * s
    want = p @ v1[0, 0].double().cpu()
    assert ((num - want).norm() / want.norm()).item() < (0.1 if dtype == torch.bfloat16 else 1e-6)
    del q, k, v
    torch.cuda.empty_cache()
