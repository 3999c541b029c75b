"""GPU parity of the fused decode+GEMM (bf16x_fused_gemm, bf16x_gemm_fused.py:97)
against the oracle: saturated (the reference kernel's numerics) and exact
(with the plan), through the C ABI."""
import numpy as np
import pytest
import torch

from oracle import dict_codec as dc
from tests.test_gpu_dict import DEV, bits_tensor, check_tol, to_dev, with_specials

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bx():
    import bfloat16x_amd as m
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return m


def _np(d):
    return {k: (v.numpy() if isinstance(v, torch.Tensor) else v) for k, v in d.items()}


# (M, out_f, in_f): the dispatch's kernels from one row to 2048 (few-row, grouped
# wave-specialised with its token tiles, one step at a time at 300 x 640),
# ragged M and out_f, the C3 prefill shapes at reduced out_f; the tiled kernel
# has its tests in test_gpu_gemm_tiled.py
CASES = [(1, 128, 64), (5, 96, 128), (16, 512, 4096), (33, 200, 1536), (64, 1024, 4096), (100, 300, 1536),
         (128, 256, 14336), (256, 1024, 4096), (300, 130, 640), (512, 512, 4096), (2048, 256, 4096)]


@pytest.mark.parametrize("path", ["fused", "auto"])
@pytest.mark.parametrize("M,out_f,in_f", CASES)
def test_gemm_saturated_and_exact(bx, M, out_f, in_f, path):
    print("gemm", M, out_f, in_f, path, flush=True)
    bits = with_specials(dc.bench_weight_bits(out_f, in_f, seed=M), seed=3) if out_f * in_f < 1 << 20 else \
        dc.bench_weight_bits(out_f, in_f, seed=M)
    bits[(bits & 0x7F00) == 0x7F00] = 0x3F80        # no inf/nan/near-max: keep the products finite
    d = bx.bf16x_quantize(bits_tensor(bits))
    g = to_dev(d)
    dn = _np(d)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16)
    xn = x.float().numpy()
    y = bx.bf16x_fused_gemm(x.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                            path=path)
    assert y.dtype == torch.bfloat16 and y.shape == (M, out_f)
    check_tol(y.float().cpu().numpy(), dc.gemm_ref(dn, xn, saturated=True))
    plan = bx.build_plan_host(d, device=DEV)
    ye = bx.bf16x_fused_gemm(x.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                             plan=plan, path=path)
    check_tol(ye.float().cpu().numpy(), dc.gemm_ref(dn, xn, saturated=False))


def test_gemm_exact_dense_overflow(bx):
    """A weight with many overflow entries per row (every atom has several):
    runs longer than the few-row kernel's preload (48 rows) and than the
    grouped kernel's lists (256 rows)."""
    out_f, in_f, M = 64, 1024, 48
    rng = np.random.default_rng(7)
    bits = dc.bench_weight_bits(out_f, in_f, seed=7)
    tiny = rng.random(bits.shape) < 0.3
    bits[tiny] = (bits[tiny] & 0x807F) | 0x0080              # exponent 1: delta >= 7 next to normal values
    d = bx.bf16x_quantize(bits_tensor(bits))
    plan = bx.build_plan_host(d, device=DEV)
    assert plan.n_fix > out_f * in_f // 32 * 2
    g = to_dev(d)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16)
    y = bx.bf16x_gemm(x.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                      plan=plan, path="fused")
    # bit-level check of the weight the kernel used: x = unit rows picks W columns
    eye = torch.eye(in_f, dtype=torch.bfloat16)[:256]
    w_cols = bx.bf16x_gemm(eye.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                           plan=plan, path="fused")
    assert np.array_equal(w_cols.contiguous().view(torch.int16).cpu().numpy().view(np.uint16).T, bits[:, :256])
    check_tol(y.float().cpu().numpy(), dc.gemm_ref(_np(d), x.float().numpy(), saturated=False))


def test_gemm_identity_is_bit_exact(bx):
    """x = I: the GEMM returns W^T element for element (one product per output,
    fp32 accumulate, bf16 store), so the decode inside the GEMM is bit exact."""
    out_f, in_f = 320, 512
    bits = dc.bench_weight_bits(out_f, in_f, seed=12)
    d = bx.bf16x_quantize(bits_tensor(bits))
    g = to_dev(d)
    plan = bx.build_plan_host(d, device=DEV)
    for start in range(0, in_f, 256):
        eye = torch.zeros(256, in_f, dtype=torch.bfloat16)
        eye[torch.arange(256), start + torch.arange(256)] = 1
        for p, ref in ((plan, bits), (None, dc.decode_saturated(_np(d)))):
            y = bx.bf16x_gemm(eye.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f,
                              in_f, plan=p, path="fused")
            got = y.contiguous().view(torch.int16).cpu().numpy().view(np.uint16).T
            assert np.array_equal(got, ref[:, start:start + 256]), start


@pytest.mark.parametrize("xdt", [torch.float16, torch.float32])
def test_gemm_fp16_fp32_activations(bx, xdt):
    out_f, in_f, M = 256, 2048, 40
    bits = dc.bench_weight_bits(out_f, in_f, seed=5)
    d = bx.bf16x_quantize(bits_tensor(bits))
    g = to_dev(d)
    plan = bx.build_plan_host(d, device=DEV)
    x = torch.randn(2, M // 2, in_f, generator=torch.Generator().manual_seed(6)).to(xdt)
    y = bx.bf16x_gemm(x.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                      plan=plan, path="fused")
    assert y.dtype == xdt and y.shape == (2, M // 2, out_f)
    y_ref = dc.gemm_ref(_np(d), x.double().numpy().reshape(M, in_f), saturated=False)
    # fp16 splits exactly into two bf16; fp32 keeps 16 of its 24 mantissa bits
    # (max 1e-2 / median 2e-3, covers both)
    tol = dict(max_tol=2e-3, med_tol=5e-4) if xdt == torch.float16 else dict(max_tol=1e-2, med_tol=1e-5)
    check_tol(y.float().cpu().numpy().reshape(M, out_f), y_ref, **tol)


def test_gemm_unfused_shapes(bx):
    """in_f not a multiple of 64 (and > 65536) goes through decode + matmul."""
    for out_f, in_f, M in ((40, 96, 7), (3, 70016, 4)):
        bits = dc.bench_weight_bits(out_f, in_f, seed=in_f)
        d = bx.bf16x_quantize(bits_tensor(bits))
        g = to_dev(d)
        plan = bx.build_plan_host(d, device=DEV)
        x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
        y = bx.bf16x_gemm(x.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                          plan=plan)
        check_tol(y.float().cpu().numpy(), dc.gemm_ref(_np(d), x.float().numpy(), saturated=False))


def test_gemm_full_size(bx):
    """C3 shape 14336x4096 at M = 512, exact: against fp32 matmul of the
    original weight on the device."""
    out_f, in_f, M = 14336, 4096, 512
    print("gemm full", M, out_f, in_f, flush=True)
    bits = dc.bench_weight_bits(out_f, in_f, seed=0)
    w = bits_tensor(bits)
    d = bx.bf16x_quantize(w)
    g = to_dev(d)
    plan = bx.build_plan_host(d, device=DEV)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(DEV)
    y_ref = (x.float() @ w.to(DEV).float().t()).double().cpu().numpy()
    for path in ("fused", "auto"):
        y = bx.bf16x_gemm(x, g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f, plan=plan,
                          path=path)
        mx, med = check_tol(y.float().cpu().numpy(), y_ref)
        print("full-size gemm (%s) rel err max %.2e median %.2e" % (path, mx, med), flush=True)


@pytest.mark.parametrize("M", [32, 64, 100])
def test_gemm_few_rows_identity_is_bit_exact(bx, M):
    """The chunked, 16x16x32 and grouped kernels the dispatch takes at these
    rows: x = rows of I select W columns, so the decode that feeds the MFMA is
    checked bit for bit, exact and saturated."""
    out_f, in_f = 96, 1024
    bits = with_specials(dc.bench_weight_bits(out_f, in_f, seed=M), seed=M)
    bits[(bits & 0x7F00) == 0x7F00] = 0x3F80
    bits[(bits & 0x7F80) == 0] = 0                       # MFMA inputs: no subnormals
    d = bx.bf16x_quantize(bits_tensor(bits))
    g = to_dev(d)
    plan = bx.build_plan_host(d, device=DEV)
    sat = dc.decode_saturated(_np(d))
    sat[(sat & 0x7F80) == 0] = 0
    for start in range(0, in_f, M):
        cols = min(M, in_f - start)
        eye = torch.zeros(M, in_f, dtype=torch.bfloat16)
        eye[torch.arange(cols), start + torch.arange(cols)] = 1
        for p, ref in ((plan, bits), (None, sat)):
            y = bx.bf16x_gemm(eye.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f,
                              in_f, plan=p, path="fused")
            got = y.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)[:cols].T
            assert np.array_equal(got, ref[:, start:start + cols]), (start, p is None)


# The wave-specialised kernel at 192 rows and more: four-step groups when in_f % 256 == 0
# (grouped = 1, the default there) and one-step tiles otherwise or when forced
# (grouped = 0); K splits forced to 1 and 3 (3 leaves a shorter last split).
@pytest.mark.parametrize("grouped", [1, 0])
@pytest.mark.parametrize("split", [-1, 1, 3])
@pytest.mark.parametrize("M,out_f,in_f", [(300, 300, 4096), (192, 136, 1024), (260, 256, 3072)])
def test_gemm_ws_groups_and_splits(bx, tune, grouped, split, M, out_f, in_f):
    print("gemm ws", M, out_f, in_f, "grouped", grouped, "split", split, flush=True)
    tune(gemm_ws_grouped=grouped, gemm_ws_split=split)
    bits = dc.bench_weight_bits(out_f, in_f, seed=out_f + split)
    d = bx.bf16x_quantize(bits_tensor(bits))
    g = to_dev(d)
    dn = _np(d)
    plan = bx.build_plan_host(d, device=DEV)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(M + split)).to(torch.bfloat16)
    for p, sat in ((plan, False), (None, True)):
        y = bx.bf16x_gemm(x.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                          plan=p, path="fused")
        check_tol(y.float().cpu().numpy(), dc.gemm_ref(dn, x.float().numpy(), saturated=sat))
    # the weight the kernel used, bit for bit: x = rows of I select W columns
    eye = torch.zeros(M, in_f, dtype=torch.bfloat16)
    cols = torch.arange(M) * (in_f // M)
    eye[torch.arange(M), cols] = 1
    w_cols = bx.bf16x_gemm(eye.to(DEV), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                           plan=plan, path="fused")
    got = w_cols.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)
    want = bits[:, cols.numpy()].T
    flush = (want & 0x7F80) == 0                # zeros and subnormals (the MFMA flushes these) come back as 0
    assert np.array_equal(np.where(flush, 0, got), np.where(flush, 0, want))
    assert not np.any(got[flush] & 0x7FFF)


# Whole-K tiles in full rounds, then the last round's tiles split over K: with
# the resident block count forced to 4 or 5, the 6 tiles of 300 x 300 run as
# 4 whole tiles + 2 tiles x 2 K ranges, or 5 whole tiles + 1 tile x 5 ranges
# (4 with four-step groups: 16 groups in ranges of 4); 520 rows x 200 columns
# (6 tiles, 3 M tiles) with 4 resident leaves the split tiles in two M rows.
@pytest.mark.parametrize("grouped", [1, 0])
@pytest.mark.parametrize("resident", [4, 5])
@pytest.mark.parametrize("M,out_f,in_f", [(300, 300, 4096), (520, 200, 1024)])
def test_gemm_ws_mixed_rounds(bx, tune, grouped, resident, M, out_f, in_f):
    print("gemm ws mixed", M, out_f, in_f, "grouped", grouped, "resident", resident, flush=True)
    tune(gemm_ws_grouped=grouped, gemm_ws_resident=resident)
    bits = dc.bench_weight_bits(out_f, in_f, seed=resident)
    d = bx.bf16x_quantize(bits_tensor(bits))
    g = to_dev(d)
    dn = _np(d)
    plan = bx.build_plan_host(d, device=DEV)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(M + resident)).to(torch.bfloat16)
    for p, sat in ((plan, False), (None, True)):
        for dt in (torch.bfloat16, torch.float32):
            y = bx.bf16x_gemm(x.to(DEV).to(dt), g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"],
                              out_f, in_f, plan=p, path="fused")
            assert y.dtype == dt
            check_tol(y.float().cpu().numpy(), dc.gemm_ref(dn, x.float().numpy(), saturated=sat))


# Split tiles' fp32 partials are summed in K-range order by the reduction
# launch: repeated launches give the same bits, fp32 and bf16, and the
# result is the product to the north-star tolerance.
@pytest.mark.parametrize("split", [2, 5])
def test_gemm_ws_split_sum_is_deterministic(bx, tune, split):
    M, out_f, in_f = 256, 1024, 4096
    print("gemm ws split determinism", split, flush=True)
    tune(gemm_ws_split=split)
    bits = dc.bench_weight_bits(out_f, in_f, seed=split)
    d = bx.bf16x_quantize(bits_tensor(bits))
    g = to_dev(d)
    plan = bx.build_plan_host(d, device=DEV)
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(split)).to(torch.bfloat16).to(DEV)
    for dt in (torch.float32, torch.bfloat16):
        xs = x.to(dt)
        ys = [bx.bf16x_gemm(xs, g["sign_packed"], g["mant_packed"], g["delta_packed"], g["emax"], out_f, in_f,
                            plan=plan, path="fused") for _ in range(4)]
        for yk in ys[1:]:
            assert torch.equal(yk.view(torch.int32 if dt == torch.float32 else torch.int16),
                               ys[0].view(torch.int32 if dt == torch.float32 else torch.int16))
    mx, med = dc.rel_err(ys[0].float().cpu().numpy(), dc.gemm_ref(_np(d), x.float().cpu().numpy(), saturated=False))
    assert mx <= 1e-2 and med <= 2e-3, (mx, med)


# Token tiles of the grouped kernel: one token, a tile less one / whole / plus
# one token, two tiles, ragged out_f; K in one range, three, and the dispatch's
# own; "spread" exponents put most elements in the plan (lists longer than the
# entries a decode wave reads ahead).  Against float64 of the same weight:
# outputs are fp32 sums of in_f exact products rounded once to bf16.
@pytest.mark.parametrize("bm", [64, 128, 256])
@pytest.mark.parametrize("M", [1, 63, 64, 65, 128, 129, 257])
@pytest.mark.parametrize("kind,out_f,in_f,split", [("bench", 300, 1024, -1), ("bench", 130, 4096, 3),
                                                   ("bench", 256, 256, 1), ("spread", 200, 768, -1)])
def test_gemm_ws_token_tiles(bx, tune, bm, M, kind, out_f, in_f, split):
    tune(gemm_ws_bm=bm, gemm_ws_split=split, gemm_skinny2_max=0, gemm_skinny_max=0, gemm_ws_min_rows=1)
    if kind == "bench":
        bits = dc.bench_weight_bits(out_f, in_f, seed=M)
    else:
        rng = np.random.default_rng(M)
        bits = ((rng.integers(0, 2, (out_f, in_f)) << 15) | (rng.integers(100, 128, (out_f, in_f)) << 7)
                | rng.integers(0, 128, (out_f, in_f))).astype(np.uint16)
    w = bits_tensor(bits)
    d = bx.bf16x_quantize(w)
    g = to_dev(d)
    plan = bx.build_plan_host(d, device=DEV)
    sat = bits_tensor(dc.decode_saturated(_np(d)).reshape(out_f, in_f))
    x = torch.randn(M, in_f, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16)
    L = bx._lib.lib()
    kp = plan.kplan()
    for p, wr in ((plan, w), (None, sat)):
        ref = (x.to(DEV).double() @ wr.to(DEV).double().t().contiguous()).cpu().numpy()
        ws = torch.empty(int(L.bf16x_gemm_workspace(M, out_f, in_f)) // 4 + 4, dtype=torch.float32, device=DEV)
        for dt, code in ((torch.bfloat16, bx._lib.BF16), (torch.float32, bx._lib.F32)):
            y = torch.empty(M, out_f, dtype=dt, device=DEV)
            xd = x.to(DEV)
            st = L.bf16x_gemm(xd.data_ptr(), bx._lib.BF16, M, g["sign_packed"].data_ptr(), g["sign_packed"].numel(),
                              g["mant_packed"].data_ptr(), g["mant_packed"].numel(), g["delta_packed"].data_ptr(),
                              g["delta_packed"].numel(), g["emax"].data_ptr(), g["emax"].numel(),
                              kp[0].data_ptr() if p is not None else None,
                              kp[1].data_ptr() if p is not None else None, out_f, in_f, 16,
                              bx._lib.EXACT if p is not None else bx._lib.SATURATED, y.data_ptr(), code,
                              ws.data_ptr(), ws.numel() * 4, bx._lib.stream_of(xd.device))
            assert st == 0
            check_tol(y.double().cpu().numpy(), ref)


# The dispatch's own choice on both sides of its lines: 64 / 65 rows, 32 / 33
# rows of a weight of 2^25 elements, in_f not a multiple of 256 (no four-step
# groups)
@pytest.mark.parametrize("M,out_f,in_f", [(64, 640, 1024), (65, 640, 1024), (191, 640, 1024), (65, 640, 1088),
                                          (32, 2048, 16384), (33, 2048, 16384), (64, 2048, 16384),
                                          (48, 12288, 4096), (33, 16384, 4096)])
def test_gemm_dispatch_lines(bx, M, out_f, in_f):
    g = torch.Generator(device=DEV).manual_seed(M)
    w = (torch.randn(out_f, in_f, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    w[:, ::97] *= 30
    d = bx.bf16x_quantize(w)
    plan = bx.build_plan_host(d, device=DEV)
    x = torch.randn(M, in_f, generator=g, device=DEV).to(torch.bfloat16)
    y = bx.bf16x_gemm(x, d["sign_packed"], d["mant_packed"], d["delta_packed"], d["emax"], out_f, in_f, plan=plan)
    check_tol(y.double().cpu().numpy(), (x.double() @ w.double().t().contiguous()).cpu().numpy())
