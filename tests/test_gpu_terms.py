"""fp16 / fp32 activations as two bf16 terms: the split and the sum bit for
bit against torch, aligned and not, and the product through bf16x_gemm."""
import pytest
import torch

from oracle import dict_codec as dc
from tests.test_gpu_dict import DEV, bits_tensor, bx  # noqa: F401

pytestmark = pytest.mark.gpu


def same(a, b):
    """Equal values, NaN equal to NaN (an fp16 infinity splits into inf + NaN)."""
    return a.dtype == b.dtype and torch.allclose(a, b, rtol=0, atol=0, equal_nan=True)


def specials(n, dt, seed):
    x = torch.randn(n, generator=torch.Generator().manual_seed(seed)) * 10.0
    x[::7] *= 1e-6
    x[::11] *= 3000.0
    x[1::13] = 0.0
    return x.to(dt).to(DEV)


@pytest.mark.parametrize("dt", [torch.float16, torch.float32])
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 4096 * 5])
@pytest.mark.parametrize("off", [0, 1, 2])
def test_split_and_add_terms(bx, dt, n, off):  # noqa: F811
    L, code = bx._lib.lib(), bx.ops._X_DTYPES[dt]
    x = specials(n + off, dt, n)[off:]
    hi = torch.empty(n + off, dtype=torch.bfloat16, device=DEV)[off:]
    lo = torch.empty(n + off, dtype=torch.bfloat16, device=DEV)[off:]
    st = bx._lib.stream_of(x.device)
    assert L.bf16x_split_terms(x.data_ptr(), code, n, hi.data_ptr(), lo.data_ptr(), st) == 0
    want = x.float().to(torch.bfloat16)
    assert same(hi, want)
    assert same(lo, (x.float() - want.float()).to(torch.bfloat16))
    a, b = specials(n + off, torch.float32, 1)[off:], specials(n + off, torch.float32, 2)[off:]
    y = torch.empty(n + off, dtype=dt, device=DEV)[off:]
    assert L.bf16x_add_terms(a.data_ptr(), b.data_ptr(), n, y.data_ptr(), code, st) == 0
    assert same(y, (a + b).to(dt))


# 2 M rows on each kernel of the dispatch: 2 (one row), 16 / 18, 64; from 33
# rows, or 17 where the weight has 2^25 elements, the kernel that takes both
# terms (tiles of 64 and 128 tokens, whole K and split), except at in_f % 256
# != 0; a row-offset view (contiguous, its
# start aligned to one element only), which a 2-byte type splits first
@pytest.mark.parametrize("dt", [torch.float16, torch.float32])
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("M,out_f,in_f,split,off", [
    (1, 520, 2048, -1, 1), (8, 520, 2048, -1, 0), (9, 520, 2048, -1, 1), (32, 520, 2048, -1, 0),
    (33, 520, 2048, -1, 0), (33, 520, 2048, -1, 1), (64, 130, 1024, 1, 0), (65, 300, 1024, 3, 2),
    (128, 128, 256, -1, 0), (129, 200, 768, -1, 0), (200, 520, 2048, -1, 0), (300, 96, 4096, 2, 0),
    (100, 520, 2112, -1, 0), (16, 2048, 16384, -1, 0), (17, 2048, 16384, -1, 0), (17, 2048, 16384, -1, 1),
    (32, 2048, 16384, -1, 0)])
def test_gemm_terms(bx, tune, dt, exact, M, out_f, in_f, split, off):  # noqa: F811
    tune(gemm_ws_split=split)
    w = bits_tensor(dc.bench_weight_bits(out_f, in_f, seed=M))
    d = bx.bf16x_quantize(w.to(DEV))
    plan = bx.build_plan_host(d, device=DEV) if exact else None
    if not exact:
        w = bits_tensor(dc.decode_saturated({k: (v.cpu().numpy() if isinstance(v, torch.Tensor) else v)
                                             for k, v in d.items()}).reshape(out_f, in_f))
    x = torch.randn(M * in_f + off, generator=torch.Generator().manual_seed(M)).to(dt).to(DEV)[off:].view(M, in_f)
    y = bx.bf16x_gemm(x, d["sign_packed"], d["mant_packed"], d["delta_packed"], d["emax"], out_f, in_f, plan=plan,
                      path="fused")
    assert y.dtype == dt and y.shape == (M, out_f)
    hi = x.float().to(torch.bfloat16)
    xs = hi.double() + (x.float() - hi.float()).to(torch.bfloat16).double()
    ref = xs @ w.to(DEV).double().t().contiguous()
    # fp32 sums of in_f products: half an ulp per addition over in_f of them is
    # far above what pairwise sums show; 2^-24 sqrt(in_f) of the magnitude, x 4,
    # and one rounding to fp16
    mag = xs.abs() @ w.to(DEV).double().abs().t().contiguous()
    tol = 4 * 2.0 ** -24 * in_f ** 0.5 * mag + (2.0 ** -11 * ref.abs() + 2.0 ** -25 if dt == torch.float16 else 0)
    assert bool(((y.double() - ref).abs() <= tol).all())
