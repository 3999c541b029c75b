"""bf16x_gemm through the C ABI, for tests that pin one of its kernels with the
tuning keys: ops.bf16x_gemm would send some of these shapes to entries of its
own before (the GEMV, the row-streaming, chunked and two-term kernels)."""
import torch

DEV = "cuda:0"


def product(bx, x, d, out_f, in_f, plan=None, dt=torch.bfloat16):
    """x (bf16 [M, in_f]) . W^T in dt (bf16 or fp32), exact with a plan; rows
    past the last are checked untouched."""
    L, M = bx._lib.lib(), x.shape[0]
    ko, ke = plan.kplan() if plan is not None else (None, None)
    nb = int(L.bf16x_gemm_workspace(M, out_f, in_f))
    ws = torch.empty(nb // 4 + 4, dtype=torch.int32, device=DEV)
    y = torch.full((M + 1, out_f), 7.0, dtype=dt, device=DEV)
    w = [v for k in ("sign_packed", "mant_packed", "delta_packed", "emax") for v in (d[k].data_ptr(), d[k].numel())]
    st = L.bf16x_gemm(x.data_ptr(), bx._lib.BF16, M, *w, ko.data_ptr() if ko is not None else None,
                      ke.data_ptr() if ke is not None else None, out_f, in_f, 16,
                      bx._lib.EXACT if plan is not None else bx._lib.SATURATED, y.data_ptr(),
                      bx._lib.F32 if dt == torch.float32 else bx._lib.BF16, ws.data_ptr(), nb,
                      bx._lib.stream_of(x.device))
    assert st == 0
    assert bool((y[M] == 7.0).all())
    return y[:M]


def check_product(y, x, w):
    """Against float64 of the weight it decodes, elementwise: one rounding to
    y's type (bf16: at most 2^-8 of the value) and the fp32 sums' own error,
    4 x 2^-24 sqrt(K) of the products' magnitude."""
    x, w = x.double(), w.double().t().contiguous()
    ref, mag = x @ w, x.abs() @ w.abs()
    tol = 4 * 2.0 ** -24 * w.shape[0] ** 0.5 * mag + (2.0 ** -8 * ref.abs() if y.dtype == torch.bfloat16 else 0)
    assert bool(((y.double() - ref).abs() <= tol).all())


def columns_bit_for_bit(bx, d, bits, plan, M):
    """W's columns picked by rows of the identity, M at a time, equal `bits` (a
    numpy uint16 array; subnormals count as zero: the MFMA flushes them)."""
    out_f, in_f = bits.shape
    want = torch.from_numpy(bits.view("int16").copy()).to(DEV)
    want = torch.where((want & 0x7F80) == 0, torch.zeros_like(want), want)
    for start in range(0, in_f, M):
        n = min(M, in_f - start)
        eye = torch.zeros(M, in_f, dtype=torch.bfloat16, device=DEV)
        eye[torch.arange(n), start + torch.arange(n)] = 1
        got = product(bx, eye, d, out_f, in_f, plan)[:n].contiguous().view(torch.int16).t()
        got = torch.where((got & 0x7F80) == 0, torch.zeros_like(got), got)
        assert torch.equal(got, want[:, start:start + n]), start
