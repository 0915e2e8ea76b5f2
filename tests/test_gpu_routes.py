"""The packed parallel kernel and the segment-state chunked kernels at sizes that reach them.  Smaller grids of
the packed kernel's shapes (fewer than two 256-query work-groups per CU) and aligned chunked calls up to a
length that depends on the head dims and heads run the wide kernel instead, which the smaller cases of the
other files cover.  Value scales, score ranges, zero regions and heads, against fp64."""

import pytest
import torch

from oracle import reference as ref
from tests.helpers import err, head_errs, rand_qkv, rows_fp64, to_dev

pytestmark = pytest.mark.gpu

TOL = 2e-2
CASES = ["plain", "v_x1e5", "v_x1e-6", "v_x1e-36", "v_x1e30", "v_steps", "tiny_prefix", "zero_leading", "zero_inner",
         "zero_head", "large_scores", "unbalanced"]


def _kernels():
    import kernels
    return kernels


def _inputs(case, H, N, d, dv, seed):
    q, k, v = rand_qkv(1, H, N, d, dv, seed=seed, dtype=torch.float32, scale_qk=0.5)
    t = torch.ones(1, H, N, 1)
    if case.startswith("v_x"):
        t *= float(case[3:])
    elif case == "v_steps":            # 512-token segments on both sides of the exponents' steps, |v| near 128
        t *= torch.tensor([40.0, 0.01, 4000.0, 0.3])[(torch.arange(N) // 512) % 4].view(1, 1, N, 1)
    elif case == "tiny_prefix":
        t[:, :, :600] = 1e-20
    elif case == "zero_leading":
        t[:, :, :600] = 0
    elif case == "zero_inner":
        t[:, :, 64:320] = t[:, :, 1000:1100] = 0
    elif case == "zero_head":
        t[:, 0] = 0
    elif case == "large_scores":       # |s| to about 300 at d = 16
        q, k = q * 15, k * 15
    elif case == "unbalanced":
        q, k = q / 30, k * 30
    return q.bfloat16(), k.bfloat16(), (v * t).bfloat16()


def _off8(x):
    """A copy 8 bytes off a 16-byte boundary."""
    buf = torch.empty(x.numel() + 4, dtype=x.dtype, device=x.device)
    buf[4:] = x.reshape(-1)
    return buf[4:].view(x.shape)


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("H,N,dv", [(128, 1100, 64), (160, 1030, 40)])
def test_packed_kernel(case, H, N, dv):
    """At least 512 work-groups of 256 queries; normalised, numerator, and the two halves apart."""
    from kernels import _lib
    K, L = _kernels(), _lib.lib()
    q, k, v = _inputs(case, H, N, 16, dv, seed=N + dv)
    qd, kd, vd = to_dev(q, k, v)
    y, den = K.based_parallel(qd, kd, vd, out_dtype=torch.float32, return_den=True)
    num = K.based_parallel(qd, kd, vd, normalize=False, out_dtype=torch.float32)
    assert torch.isfinite(y).all() and torch.isfinite(num).all()
    n = int(L.la_based_parallel_workspace_bytes(1, H, N, 16, dv, 1))
    ws, st = torch.full((n,), 0x7f, dtype=torch.uint8, device="cuda"), torch.cuda.current_stream().cuda_stream
    apart = torch.empty_like(y)
    assert L.la_based_parallel_pack(kd.data_ptr(), vd.data_ptr(), 1, 1, H, N, 16, dv, ws.data_ptr(), n, st) == 0
    assert L.la_based_parallel_fwd_packed(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), 1, apart.data_ptr(), 0, None, 1, H,
                                          N, 16, dv, 0.25, 1e-6, 1, ws.data_ptr(), n, st) == 0
    assert torch.equal(apart, y)
    if case == "zero_head":
        assert y[0, 0].abs().max().item() == 0.0
    for h in (1, 77, H - 1):
        want, want_num, want_den = ref.based_dense(q[:, h:h + 1], k[:, h:h + 1], v[:, h:h + 1])
        assert max(head_errs(y[:, h:h + 1], want)) < TOL and max(head_errs(num[:, h:h + 1], want_num)) < TOL
        assert err(den[:, h:h + 1], want_den) < TOL


def test_packed_kernel_heads_of_different_scales():
    K = _kernels()
    H, N = 128, 1100
    q, k, v = _inputs("plain", H, N, 16, 64, seed=13)
    v = (v.float() * torch.tensor([1e5, 1.0, 1e-6, 1e-3]).repeat(H // 4).view(1, H, 1, 1)).bfloat16()
    y = K.based_parallel(*to_dev(q, k, v), out_dtype=torch.float32)
    for h in (0, 1, 2, 3, 126):
        want, _, _ = ref.based_dense(q[:, h:h + 1], k[:, h:h + 1], v[:, h:h + 1])
        assert max(head_errs(y[:, h:h + 1], want)) < TOL


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("N,d,dv", [(12300, 16, 128), (12800, 32, 32), (13400, 48, 64), (15700, 64, 64), (15300, 64, 128)])
def test_segment_path(case, N, d, dv):
    """Beyond the lengths at which aligned calls take the wide kernel: 16-byte and element-wise loads give the
    same bits (so both ran this path), fp64 rows at segment edges and across the sequence."""
    K = _kernels()
    H = 2
    q, k, v = _inputs(case, H, N, d, dv, seed=N)
    qd, kd, vd = to_dev(q, k, v)
    y = K.based_chunked(qd, kd, vd, out_dtype=torch.float32)
    assert torch.isfinite(y).all()
    assert torch.equal(y, K.based_chunked(_off8(qd), _off8(kd), _off8(vd), out_dtype=torch.float32))
    y = y.cpu()
    rows = torch.tensor([0, 1, 63, 255, 256, 511, 512, 513, 700, 1023, 1024, 1100, 2047, 2048, 5000, 8191, 8192, N - 513, N - 2, N - 1])
    for h in range(H):
        if case == "zero_head" and h == 0:
            assert y[0, 0].abs().max().item() == 0.0
            continue
        # rows on one side of a step of V's scale have an rms of their own
        for r in (rows[rows < 512], rows[(rows >= 512) & (rows < 1536)], rows[rows >= 1536]):
            want = rows_fp64(q, k, v, 0, h, r)
            if want.abs().max() > 0:
                assert ref.rel_err(y[0, h, r], want) < TOL, (h, r)


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("d,dv", [(64, 64), (48, 40), (17, 128)])
def test_segment_path_short(case, d, dv):
    """The same path by alignment (8 bytes off) at a few segments, every row, numerator too."""
    K = _kernels()
    q, k, v = _inputs(case, 2, 1800, d, dv, seed=d)
    a = [_off8(x) for x in to_dev(q, k, v)]
    want, want_num, _ = ref.based_dense(q, k, v)
    hs = slice(1, 2) if case == "zero_head" else slice(0, 2)
    e = max(head_errs(K.based_chunked(*a, out_dtype=torch.float32)[:, hs], want[:, hs]))
    en = max(head_errs(K.based_chunked(*a, normalize=False, out_dtype=torch.float32)[:, hs], want_num[:, hs]))
    assert e < TOL and en < TOL, (e, en)


def test_segment_path_zero_key_dims():
    """Keys zero in dims 16 .. 63 over the first segment, V x 1e10: work-groups whose prefix is all zeros."""
    K = _kernels()
    q, k, v = _inputs("v_x1e10", 2, 1500, 64, 64, seed=18)
    k[:, :, :512, 16:] = 0
    y = K.based_chunked(*(_off8(x) for x in to_dev(q, k, v)), out_dtype=torch.float32)
    want, _, _ = ref.based_dense(q, k, v)
    assert torch.isfinite(y).all() and max(head_errs(y, want)) < TOL


@pytest.mark.parametrize("d,dv", [(64, 64), (32, 128)])
def test_segment_path_many_heads(d, dv):
    """More state work-groups than CUs (two share one, with alternating wave priorities): 32 heads by alignment,
    the first 700 rows of every head and later rows of three."""
    K = _kernels()
    q, k, v = rand_qkv(2, 16, 4096, d, dv, seed=41, dtype=torch.bfloat16)
    y = K.based_chunked(*(_off8(x) for x in to_dev(q, k, v)), out_dtype=torch.float32).cpu()
    want, _, _ = ref.based_dense(q[:, :, :700], k[:, :, :700], v[:, :, :700])
    assert max(head_errs(y[:, :, :700], want)) < TOL
    rows = torch.tensor([1500, 2047, 2048, 3583, 3584, 4095])
    for b, h in ((0, 0), (1, 7), (1, 15)):
        assert ref.rel_err(y[b, h, rows], rows_fp64(q, k, v, b, h, rows)) < TOL
