"""The step-major plan (bf16x_kplan_build, bf16x_gguf_kplan_build) and the scan
behind it, from plans made here, word for word against numpy."""
import numpy as np
import pytest
import torch

from tests.test_gpu_dict import DEV, bx  # noqa: F401

pytestmark = pytest.mark.gpu


def make_plan(out_f, in_f, per_row, seed):
    """Row plan with about per_row entries a row (0 .. in_f), columns
    ascending; a few rows empty, a few full of entries."""
    rng = np.random.default_rng(seed)
    off, cols = [0], []
    for r in range(out_f):
        n = 0 if r % 7 == 3 else min(in_f, int(rng.integers(0, 2 * per_row + 1)))
        if r % 31 == 5:
            n = min(in_f, 40 * per_row)
        cols.append(np.sort(rng.choice(in_f, n, replace=False)))
        off.append(off[-1] + n)
    cols = np.concatenate(cols).astype(np.uint32)
    bits = rng.integers(0, 65536, cols.size).astype(np.uint32)
    return np.array(off, np.uint32), cols, bits


def walk_reference(off, cols, bits, out_f, in_f):
    """Runs (step, 16-row group); a row's entries are taken in order while
    their steps do not go down."""
    S, G2 = in_f // 64, 2 * ((out_f + 31) // 32)
    runs = {}
    for r in range(out_f):
        p, s = int(off[r]), 0
        for s in range(S):
            while p < off[r + 1] and cols[p] >> 6 == s:
                runs.setdefault((s, r // 16), []).append((r & 255) << 22 | int(cols[p] & 63) << 16 | int(bits[p]))
                p += 1
    kp_off, ent = np.zeros(S * G2 + 1, np.int64), []
    for i in range(S * G2):
        run = runs.get((i // G2, i % G2), [])
        ent += run
        kp_off[i + 1] = kp_off[i] + len(run)
    return kp_off, np.array(ent, np.int64)


def build(bx, off, cols, bits, out_f, in_f, gguf):  # noqa: F811
    L = bx._lib.lib()
    ent = (cols | bits << 16) if gguf else (cols << 16 | bits)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.uint32).view(np.int32)).to(DEV)
    d_off, d_ent = to(off), to(ent if ent.size else np.zeros(1))
    kp_off = torch.empty(int(L.bf16x_kplan_size(out_f, in_f)), dtype=torch.int32, device=DEV)
    kp_ent = torch.zeros(max(ent.size, 1), dtype=torch.int32, device=DEV)
    f = L.bf16x_gguf_kplan_build if gguf else L.bf16x_kplan_build
    st = f(d_off.data_ptr(), d_ent.data_ptr(), out_f, in_f, kp_off.data_ptr(), kp_ent.data_ptr(),
           bx._lib.stream_of(kp_off.device))
    assert st == 0
    return [t.cpu().numpy().view(np.uint32).astype(np.int64) for t in (kp_off, kp_ent)]


# rows around a 16-row group and a 32-row pair, one step to 1024 (65536
# columns, the largest), odd step counts, empty and full rows
@pytest.mark.parametrize("out_f,in_f,per_row", [(1, 64, 3), (15, 64, 2), (16, 192, 6), (17, 4096, 90), (33, 320, 20),
                                                (70, 65536, 300), (300, 1024, 25), (48, 128, 0)])
@pytest.mark.parametrize("gguf", [False, True])
def test_kplan(bx, out_f, in_f, per_row, gguf):  # noqa: F811
    off, cols, bits = make_plan(out_f, in_f, per_row, out_f)
    kp_off, kp_ent = build(bx, off, cols, bits, out_f, in_f, gguf)
    ref_off, ref_ent = walk_reference(off, cols, bits, out_f, in_f)
    assert np.array_equal(kp_off, ref_off)
    assert np.array_equal(kp_ent[:ref_ent.size], ref_ent)


# entries out of order in one row, and twice the same column: that row's group
# is walked as before, the others are not affected
@pytest.mark.parametrize("kind", ["swapped", "repeated", "past the row"])
def test_kplan_out_of_order(bx, kind):  # noqa: F811
    out_f, in_f = 100, 512
    off, cols, bits = make_plan(out_f, in_f, 12, 3)
    j = int(off[40])
    assert off[41] - j >= 3
    if kind == "swapped":
        cols[[j, j + 2]] = cols[[j + 2, j]]
    elif kind == "repeated":
        cols[j + 1] = cols[j]
    else:
        cols[off[41] - 1] = 5000
    kp_off, kp_ent = build(bx, off, cols, bits, out_f, in_f, False)
    ref_off, ref_ent = walk_reference(off, cols, bits, out_f, in_f)
    assert np.array_equal(kp_off, ref_off)
    assert np.array_equal(kp_ent[:ref_ent.size], ref_ent)


# a CSR whose offsets fall back: its plan's rows share no entry, so the
# regrouped plans stay inside their n entries; a well-formed one is unchanged
@pytest.mark.parametrize("kind", ["ascending", "falling", "out of range"])
def test_csr_offsets(bx, kind):  # noqa: F811
    out_f, in_f = 64, 512
    d = bx.bf16x_quantize(torch.randn(out_f, in_f, generator=torch.Generator().manual_seed(1)).to(DEV))
    off, cols, _ = make_plan(out_f, in_f, 9, 4)
    n, good = cols.size, off.astype(np.int32)
    bad = good.copy()
    if kind == "falling":
        bad[1::2] = n
        bad[2::2] = 0
    elif kind == "out of range":
        bad[10], bad[20], bad[30] = -7, 2 ** 30, 3
    to = lambda a: torch.from_numpy(a.astype(np.int32)).to(DEV)
    plan = bx.codec.build_plan_from_csr(to(cols), torch.full((n,), 9, dtype=torch.int32, device=DEV), to(bad),
                                        d["sign_packed"], d["mant_packed"], d["emax"], out_f, in_f)
    t = plan.tile_off.cpu().numpy()
    assert t.min() >= 0 and t.max() <= n and np.all(np.diff(t) >= 0)
    assert kind != "ascending" or np.array_equal(t, good)
    for o, e in (plan.kplan(), plan.cplan()):
        assert 0 <= int(o[-1]) <= n <= e.numel()
    torch.cuda.synchronize()


# the scan at its tile's edges and with more tiles than one pass over their
# first elements takes (1024), through the chunk plan's offsets
@pytest.mark.parametrize("out_f,in_f", [(1, 256), (4095, 256), (4096, 256), (4097, 256), (8192, 256), (140000, 8192)])
def test_scan(bx, out_f, in_f):  # noqa: F811
    L = bx._lib.lib()
    rng = np.random.default_rng(out_f)
    n = min(out_f * 3, 60000)
    rows = np.sort(rng.integers(0, out_f, n))
    cols = np.zeros(n, np.int64)
    at = np.arange(n) - np.searchsorted(rows, rows)             # distinct, ascending columns of a row
    cols = at * (in_f // 64)
    keep = cols < in_f
    rows, cols = rows[keep], cols[keep]
    off = np.searchsorted(rows, np.arange(out_f + 1))
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.uint32).view(np.int32)).to(DEV)
    d_off, d_ent = to(off), to(cols << 16 | 7)
    size = int(L.bf16x_cplan_size(out_f, in_f))
    cp_off = torch.empty(size, dtype=torch.int32, device=DEV)
    cp_ent = torch.zeros(rows.size + 1, dtype=torch.int32, device=DEV)
    assert L.bf16x_cplan_build(d_off.data_ptr(), d_ent.data_ptr(), out_f, in_f, cp_off.data_ptr(), cp_ent.data_ptr(),
                               bx._lib.stream_of(cp_off.device)) == 0
    counts = np.bincount((cols // 256) * out_f + rows, minlength=size - 1)
    assert np.array_equal(cp_off.cpu().numpy().astype(np.int64), np.concatenate([[0], np.cumsum(counts)]))
