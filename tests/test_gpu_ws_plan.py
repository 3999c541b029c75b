"""The overflow entries inside the grouped wave-specialised GEMM, bit for bit:
x = rows of the identity pick W's columns, for every tile of tokens and for
plans from empty to half of all elements."""
import numpy as np
import pytest
import torch

from tests.gemm_abi import product
from tests.test_gpu_dict import DEV, bits_tensor, bx, gpu_bits  # noqa: F401

pytestmark = pytest.mark.gpu

OUT_F, IN_F = 200, 768                 # a ragged 128-row tile, three 256-column groups


def with_entries(share, seed):
    """Exponent 127 throughout but for a share of elements, 10 to 26 below."""
    rng = np.random.default_rng(seed)
    shape = (OUT_F, IN_F)
    e = np.where(rng.random(shape) < share, rng.integers(101, 118, shape), 127)
    return ((rng.integers(0, 2, shape) << 15) | (e << 7) | rng.integers(0, 128, shape)).astype(np.uint16)


# entries of a decode wave's rows and a 256-column group against what it loads
# ahead, one in 32 elements always and up to one in 16 behind a branch: none,
# below the first, between them, around and far above the second
@pytest.mark.parametrize("share", [0.0, 0.02, 0.045, 0.0625, 0.1, 0.5])
@pytest.mark.parametrize("bm", [64, 128, 256])
@pytest.mark.parametrize("kind", ["dict", "gguf"])
def test_entries_bit_for_bit(bx, tune, kind, bm, share):  # noqa: F811
    tune(gemm_ws_bm=bm, gemm_ws_min_rows=1, gemm_skinny2_max=0, gemm_skinny_max=0, gemm_stream_max=0)
    bits = with_entries(share, bm)
    w = bits_tensor(bits)
    if kind == "dict":
        d = bx.bf16x_quantize(w.to(DEV))
        plan = bx.build_plan_host(d, device=DEV)
        n = plan.n_fix
    else:
        blocks = bx.gguf.device_blocks(bx.gguf.quantize_blocks(w), DEV)
        t = bx.gguf.device_ovf(bx.gguf.pack_ovf(w), bx.gguf.quantize_blocks(w), DEV)
        n = t.n_entries
    assert abs(n - share * bits.size) <= 6 * (share * bits.size) ** 0.5 + 1e-3
    for start in range(0, IN_F, bm):
        eye = torch.zeros(bm, IN_F, dtype=torch.bfloat16, device=DEV)
        eye[torch.arange(bm), start + torch.arange(bm)] = 1
        if kind == "dict":
            y = product(bx, eye, d, OUT_F, IN_F, plan)
        else:
            y = bx.gguf.gguf_gemm_fused(eye, blocks, OUT_F, IN_F, ovf=t)
        assert np.array_equal(gpu_bits(y).T, bits[:, start:start + bm]), start

