"""GPU parity of the Taylor feature map kernel (la_taylor_feature_map)."""

import pytest
import torch

from oracle import reference as ref
from tests.helpers import load_golden

pytestmark = pytest.mark.gpu


def _kernels():
    import kernels
    return kernels


@pytest.mark.parametrize("name", ["phi_d4", "phi_d16"])
def test_golden(name):
    K = _kernels()
    g = load_golden(name)
    x = torch.from_numpy(g["x"])
    y = K.taylor_feature_map(x.cuda()).cpu()
    assert y.dtype == torch.float32
    assert torch.allclose(y.double(), torch.from_numpy(g["phi"]), rtol=2e-7, atol=1e-7)


@pytest.mark.parametrize("d", [1, 2, 3, 5, 16, 17, 64, 128])
def test_matches_reference_fp32(d):
    K = _kernels()
    x = torch.randn(3, 7, d)
    y = K.taylor_feature_map(x.cuda()).cpu()
    want = ref.taylor_feature_map(x)
    assert y.shape == want.shape
    ulp = torch.finfo(torch.float32).eps * want.abs().clamp_min(1e-30)
    print(f"d={d} exact={torch.equal(y, want)} max_ulp={((y - want).abs() / ulp).max().item():.2f}")
    assert ((y - want).abs() <= ulp).all()


def test_bf16_input():
    K = _kernels()
    x = torch.randn(50, 16).to(torch.bfloat16)
    y = K.taylor_feature_map(x.cuda()).cpu()
    assert y.dtype == torch.bfloat16
    want = ref.taylor_feature_map(x.double())
    assert torch.allclose(y.double(), want, rtol=8e-3, atol=1e-6)


@pytest.mark.parametrize("rows,d,off", [
    (1, 1, 0),            # a row shorter than a thread's four outputs
    (7, 2, 0),            # an incomplete eight-row work-group
    (33, 16, 1),          # an output pointer that takes no wide stores
    (16385, 16, 0),       # 32-row work-groups (from 64 rows per CU on), one row in the last
    (32775, 5, 0),        # the same for a divisor that is no power of two
    (17000, 64, 3),
    (16387, 128, 0),      # the largest table
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_and_alignment(rows, d, off, dtype):
    """Every work-group size and store width; fp32 within an ulp of the reference's fp32 evaluation, bf16 the
    rounding of such a value (8 significand bits: half an ulp is at most 2^-8 of the value)."""
    from kernels import _lib
    g = torch.Generator().manual_seed(rows + d)
    x = torch.randn(rows, d, generator=g).to(dtype)
    F = 1 + d + d * (d + 1) // 2
    buf = torch.full((rows * F + 8,), -7.0, device="cuda", dtype=dtype)
    xc, out = x.cuda(), buf[off:off + rows * F]
    code = _lib.dtype_code(dtype)
    rc = _lib.lib().la_taylor_feature_map(_lib.ptr(xc), code, _lib.ptr(out), code, rows, d, 0)
    assert rc == 0
    torch.cuda.synchronize()
    y = out.cpu().view(rows, F).float()
    want = ref.taylor_feature_map(x.float())
    rel = torch.finfo(torch.float32).eps + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)
    assert ((y - want).abs() <= rel * 1.001 * want.abs() + 1e-37).all()
    assert (buf[:off] == -7.0).all() and (buf[off + rows * F:] == -7.0).all()
