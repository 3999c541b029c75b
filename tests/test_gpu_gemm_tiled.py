"""The tiled fused GEMM (33 to 191 rows at in_f % 256 != 0, 65 to 191 where
in_f % 128 == 0), pinned for every tile height and K split: products against
float64, the weight it decodes bit for bit, and dense plans."""
import numpy as np
import pytest
import torch

from oracle import dict_codec as dc
from tests.gemm_abi import check_product, columns_bit_for_bit, product
from tests.test_gpu_dict import DEV, bits_tensor, bx, to_dev, with_specials  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture
def tiled(tune):
    tune(gemm_ws_min_rows=1 << 30, gemm_skinny2_max=0, gemm_skinny_max=0, gemm_stream_max=0)


def weight(bx, bits):  # noqa: F811
    bits[(bits & 0x7F00) == 0x7F00] = 0x3F80            # finite products
    d = bx.bf16x_quantize(bits_tensor(bits))
    sat = dc.decode_saturated({k: (v.numpy() if isinstance(v, torch.Tensor) else v) for k, v in d.items()})
    return to_dev(d), bx.build_plan_host(d, device=DEV), sat.reshape(bits.shape)


def dense(out_f, in_f, seed, share=0.35):
    rng = np.random.default_rng(seed)
    bits = dc.bench_weight_bits(out_f, in_f, seed=seed)
    tiny = rng.random(bits.shape) < share
    bits[tiny] = (bits[tiny] & 0x807F) | 0x0080
    return bits


# each tile height (32, 64, 128, 256 rows) below, at and past its rows; one K
# range and several; out_f around a 128-row tile; odd step counts
@pytest.mark.parametrize("M", [1, 32, 33, 64, 65, 128, 129, 191])
@pytest.mark.parametrize("out_f,in_f,split", [(640, 1088, -1), (130, 2112, 3), (127, 640, 1), (300, 64, -1)])
@pytest.mark.parametrize("kind", ["bench", "dense"])
def test_tiled_products(bx, tiled, tune, M, out_f, in_f, split, kind):  # noqa: F811
    tune(gemm_split=split)
    bits = with_specials(dc.bench_weight_bits(out_f, in_f, seed=M), 3) if kind == "bench" else dense(out_f, in_f, M)
    g, plan, sat = weight(bx, bits)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    for p, b in ((plan, bits), (None, sat)):
        flushed = np.where((b & 0x7F80) == 0, 0, b).astype(np.uint16)       # the MFMA's subnormal inputs
        for dt in (torch.bfloat16, torch.float32):
            check_product(product(bx, x, g, out_f, in_f, p, dt), x, bits_tensor(flushed).to(DEV))


@pytest.mark.parametrize("M", [40, 128, 191])
@pytest.mark.parametrize("kind", ["bench", "dense"])
def test_tiled_weight_bit_for_bit(bx, tiled, M, kind):  # noqa: F811
    out_f, in_f = 200, 832
    bits = with_specials(dc.bench_weight_bits(out_f, in_f, seed=M), 3) if kind == "bench" else dense(out_f, in_f, M)
    g, plan, sat = weight(bx, bits)
    columns_bit_for_bit(bx, g, bits, plan, M)
    columns_bit_for_bit(bx, g, sat, None, M)


# without any key: these shapes run it
@pytest.mark.parametrize("M,in_f", [(33, 1088), (64, 2112), (65, 640), (128, 1088), (129, 1088), (191, 2112)])
def test_dispatch_to_the_tiled_kernel(bx, M, in_f):  # noqa: F811
    out_f = 384
    bits = dc.bench_weight_bits(out_f, in_f, seed=M)
    g, plan, sat = weight(bx, bits)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    for p, b in ((plan, bits), (None, sat)):
        w = bits_tensor(b).to(DEV)
        check_product(product(bx, x, g, out_f, in_f, p, torch.float32), x, w)
        check_product(bx.bf16x_gemm(x, g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                                    plan=p, path="fused"), x, w)
