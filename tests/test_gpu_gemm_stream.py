"""The streaming few-row GEMM (up to 16 rows, small weights) against float64 of
the weight it decodes: dict and GGUF, exact / lossless and not."""
import numpy as np
import pytest
import torch

from oracle import dict_codec as dc
from oracle import gguf_codec as go
from tests.gemm_abi import check_product as check
from tests.test_gpu_dict import DEV, bits_tensor, bx  # noqa: F401

pytestmark = pytest.mark.gpu


def spread(out_f, in_f, seed):
    """Exponents uniform over 28 values: most elements are in the plan."""
    rng = np.random.default_rng(seed)
    return ((rng.integers(0, 2, (out_f, in_f)) << 15) | (rng.integers(100, 128, (out_f, in_f)) << 7)
            | rng.integers(0, 128, (out_f, in_f))).astype(np.uint16)


# fewer steps than the 16 waves, exactly one each, one more (waves with an
# empty last step), several; rows around a 16-row group, more groups than CUs
# (a workgroup's second group); one token to 16
@pytest.mark.parametrize("out_f,in_f", [(1, 128), (17, 640), (64, 2048), (33, 2176), (100, 8192), (4100, 1152),
                                        (8300, 128)])
@pytest.mark.parametrize("M", [1, 2, 15, 16])
@pytest.mark.parametrize("kind", ["bench", "spread"])
def test_stream_dict(bx, tune, out_f, in_f, M, kind):  # noqa: F811
    tune(gemm_stream_max=16)
    w = bits_tensor(dc.bench_weight_bits(out_f, in_f, seed=M) if kind == "bench" else spread(out_f, in_f, M))
    d = bx.bf16x_quantize(w.to(DEV))
    plan = bx.build_plan_host(d, device=DEV)
    kp = plan.kplan()
    sat = bx.bf16x_decode(d["sign_packed"], d["mant_packed"], d["delta_packed"], d["emax"], out_f, in_f)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    L = bx._lib.lib()
    assert L.bf16x_gemm_workspace(M, out_f, in_f) == 0
    for wr, ko, ke, mode in ((w.to(DEV), kp[0].data_ptr(), kp[1].data_ptr(), bx._lib.EXACT),
                             (sat, None, None, bx._lib.SATURATED)):
        for dt, code in ((torch.bfloat16, bx._lib.BF16), (torch.float32, bx._lib.F32)):
            y = torch.full((M + 1, out_f), 7.0, dtype=dt, device=DEV)
            args = [v for k in ("sign_packed", "mant_packed", "delta_packed", "emax")
                    for v in (d[k].data_ptr(), d[k].numel())]
            assert L.bf16x_gemm(x.data_ptr(), bx._lib.BF16, M, *args, ko, ke, out_f, in_f, 16, mode, y.data_ptr(),
                                code, None, 0, bx._lib.stream_of(x.device)) == 0
            check(y[:M], x, wr)
            assert bool((y[M] == 7.0).all())                    # nothing past the last token


@pytest.mark.parametrize("out_f,in_f", [(17, 640), (130, 2048), (4100, 256)])
@pytest.mark.parametrize("M", [2, 16])
def test_stream_gguf(bx, tune, out_f, in_f, M):  # noqa: F811
    tune(gemm_stream_max=16)
    g = bx.gguf
    w = (np.random.default_rng(M).standard_t(3, (out_f, in_f)) * 0.015).astype(np.float32)
    wb = go.bf16_bits_to_fp32(go.fp32_to_bf16_bits(w)).astype(np.float64).reshape(out_f, in_f)
    packed = g.quantize_blocks(w)
    wnl = go.dequantize_blocks(packed).astype(np.float64).reshape(out_f, in_f)
    t = g.device_ovf(g.pack_ovf(w), packed, DEV)
    blocks = g.device_blocks(packed, DEV)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    for ovf, ref in ((t, wb), (None, wnl)):
        for dt in (torch.float32, torch.bfloat16):
            y = g.gguf_gemm_fused(x, blocks, out_f, in_f, out_dtype=dt, ovf=ovf)
            check(y, x, torch.from_numpy(ref).to(DEV))


# both sides of the dispatch's line (a wave's steps x tokens <= 32, <= 4 steps)
@pytest.mark.parametrize("M,out_f,in_f", [(16, 512, 1024), (16, 512, 5120), (8, 512, 8192), (9, 512, 8192),
                                          (2, 512, 8192), (2, 512, 10240), (17, 512, 1024)])
def test_dispatch_line(bx, M, out_f, in_f):  # noqa: F811
    w = bits_tensor(dc.bench_weight_bits(out_f, in_f, seed=M))
    d = bx.bf16x_quantize(w.to(DEV))
    plan = bx.build_plan_host(d, device=DEV)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    y = bx.bf16x_gemm(x, d["sign_packed"], d["mant_packed"], d["delta_packed"], d["emax"], out_f, in_f, plan=plan)
    check(y, x, w.to(DEV))
