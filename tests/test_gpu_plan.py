"""The device plan builder against the host builder: equal plans, word for
word, and the same refusals."""
import numpy as np
import pytest
import torch

from oracle import dict_codec as dc
from tests.test_gpu_dict import DEV, bits_tensor, bx, to_dev, with_specials  # noqa: F401

pytestmark = pytest.mark.gpu


def sparse_bits(shape, seed, n):
    """A flat weight with n elements far below their block's exponent, at
    random positions: long runs of rows without an entry."""
    b = np.full(shape, 0x3C01, np.uint16).reshape(-1)
    rng = np.random.default_rng(seed)
    at = rng.choice(b.size, n, replace=False)
    b[at] = 0x8005 | (rng.integers(100, 110, n).astype(np.uint16) << 7)
    return b.reshape(shape)


def same_plan(p, q):
    assert (p.n_fix, p.out_f, p.in_f) == (q.n_fix, q.out_f, q.in_f)
    assert torch.equal(p.tile_off.cpu(), q.tile_off.cpu())
    assert torch.equal(p.tile_ent[:p.n_fix].cpu(), q.tile_ent[:q.n_fix].cpu())
    assert torch.equal(p.tile_sat[:p.n_fix].cpu(), q.tile_sat[:q.n_fix].cpu())
    assert p.tile_ent.shape == q.tile_ent.shape and p.tile_sat.shape == q.tile_sat.shape


# rows shorter and longer than a wave's 64 entries, two tiles per row (in_f >
# 65536), odd widths, more entries than one workgroup per count of the scan
@pytest.mark.parametrize("shape", [(7, 9), (33, 40), (256, 32), (64, 4096), (3, 70016), (300, 577), (4096, 3000)])
@pytest.mark.parametrize("kind", ["bench", "special", "sparse", "one"])
def test_device_plan_equals_host(bx, shape, kind):  # noqa: F811
    bits = {"bench": lambda: dc.bench_weight_bits(*shape, seed=2),
            "special": lambda: with_specials(dc.bench_weight_bits(*shape, seed=3), 4, k=shape[0] * shape[1] // 3),
            "sparse": lambda: sparse_bits(shape, 5, max(2, shape[0] // 20)),
            "one": lambda: sparse_bits(shape, 6, 1)}[kind]()
    d = bx.bf16x_quantize(bits_tensor(bits))
    want = bx.build_plan_host(d)
    got = bx.build_plan_host(to_dev(d), device=DEV)
    assert got.tile_off.is_cuda
    same_plan(got, want)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1024, 256 * 4096, 256 * 4096 + 1])
def test_device_plan_entry_counts(bx, n):  # noqa: F811
    """Table sizes at the edges of a workgroup and of the scan's capacity."""
    shape = (1024, 2048) if n > 1024 else (64, 256)
    w = torch.full(shape, 0x3C01, dtype=torch.int16, device=DEV).reshape(-1)
    w[(torch.arange(n, device=DEV) // 15) * 16 + torch.arange(n, device=DEV) % 15] = 0x3405
    d = bx.bf16x_quantize(w.view(torch.bfloat16).view(shape))
    assert d["delta_ovf_idx"].numel() == n
    host = {k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in d.items()}
    same_plan(bx.build_plan_host(d, device=DEV), bx.build_plan_host(host))


def test_device_plan_refuses_bad_tables(bx):  # noqa: F811
    d = bx.bf16x_quantize(bits_tensor(dc.bench_weight_bits(64, 4096, seed=7)))
    n = d["delta_ovf_idx"].numel()
    code7 = np.zeros(64 * 4096, bool)
    code7[d["delta_ovf_idx"].numpy()] = True

    def bad(name, i, v):
        t = dict(d)
        t[name] = d[name].clone()
        t[name][i] = v
        return t
    cases = [bad("delta_ovf_idx", n - 1, 64 * 4096), bad("delta_ovf_idx", 0, -1),
             bad("delta_ovf_idx", 5, int(d["delta_ovf_idx"][4])), bad("delta_ovf_val", n // 2, 6),
             bad("delta_ovf_val", 3, 255), bad("delta_ovf_idx", 0, int(np.flatnonzero(~code7)[0]))]
    for t in cases:
        for where, device in ((t, None), (to_dev(t), DEV)):
            with pytest.raises(bx.Bf16xError) as e:
                bx.build_plan_host(where, device=device)
            assert e.value.status == -4
