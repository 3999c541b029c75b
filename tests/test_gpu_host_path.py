"""The native call path of the wrappers (ordinary tensors) against their Python
path: the same bits for every form both take, and the same refusals."""
import ctypes
import sys
import threading

import pytest
import torch

from oracle import dict_codec as dc
from tests.test_gpu_dict import DEV, bits_tensor, bx  # noqa: F401

pytestmark = pytest.mark.gpu

OUT_F, IN_F = 96, 1024


class Sub(torch.Tensor):
    pass


def strided(t):
    """The same values with a stride of two elements."""
    b = torch.zeros(t.numel() * 2, dtype=t.dtype, device=t.device)
    b[::2] = t.reshape(-1)
    return b[::2]


@pytest.fixture(scope="module")
def weight(bx):  # noqa: F811
    d = bx.bf16x_quantize(bits_tensor(dc.bench_weight_bits(OUT_F, IN_F, seed=1)).to(DEV))
    return [d[k] for k in ("sign_packed", "mant_packed", "delta_packed", "emax")], bx.build_plan_host(d, device=DEV)


FORMS = {"row": lambda x: x.view(1, -1), "strided": strided, "subclass": lambda x: x.as_subclass(Sub),
         "parameter": lambda x: torch.nn.Parameter(x), "offset": lambda x: torch.cat([x[:2], x])[2:]}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("exact", [True, False])
def test_forms_give_the_same_bits(bx, weight, form, dt, exact):  # noqa: F811
    w, plan = weight
    plan = plan if exact else None
    x = torch.randn(IN_F, generator=torch.Generator().manual_seed(2)).to(dt).to(DEV)
    want = bx.bf16x_gemv(x, *w, OUT_F, IN_F, plan=plan)
    assert want.shape == (OUT_F,) and want.dtype == torch.bfloat16 and not want.requires_grad
    got = bx.bf16x_gemv(FORMS[form](x), *w, OUT_F, IN_F, plan=plan)
    assert torch.equal(got, want)
    got = bx.bf16x_gemv(x, strided(w[0]), *w[1:], OUT_F, IN_F, plan=plan)
    assert torch.equal(got, want)
    out = torch.empty(OUT_F + 5, dtype=torch.bfloat16, device=DEV)
    assert bx.bf16x_gemv(FORMS[form](x), *w, OUT_F, IN_F, plan=plan, out=out) is out
    assert torch.equal(out[:OUT_F], want)
    x3 = torch.stack([x, -x, 2 * x])
    want = bx.bf16x_gemm(x3, *w, OUT_F, IN_F, plan=plan)
    y = bx.bf16x_gemm(strided(x3).view(3, IN_F) if form == "strided" else x3.as_subclass(Sub), *w, OUT_F, IN_F,
                      plan=plan)
    assert torch.equal(y.as_subclass(torch.Tensor), want)


def test_refusals(bx, weight):  # noqa: F811
    w, plan = weight
    x = torch.zeros(IN_F, dtype=torch.bfloat16, device=DEV)
    bad = [(ValueError, (x.cpu(), *w)), (ValueError, (x[:-32], *w)), (TypeError, (x.double(), *w)),
           (TypeError, (x, w[0].float(), *w[1:])), (ValueError, (x, w[0].cpu(), *w[1:])),
           (TypeError, ([0.0], *w)), (bx.Bf16xError, (x, w[0][:4], *w[1:]))]
    for err, args in bad:
        with pytest.raises(err):
            bx.bf16x_gemv(*args, OUT_F, IN_F, plan=plan)
        with pytest.raises(err):
            bx.bf16x_gemm(args[0].view(1, -1).expand(3, -1) if isinstance(args[0], torch.Tensor) else args[0],
                          *args[1:], OUT_F, IN_F, plan=plan, path="fused")
    with pytest.raises(ValueError):
        bx.bf16x_gemv(x, *w, OUT_F - 1, IN_F, plan=plan)             # another shape's plan
    for out in (torch.empty(OUT_F, device=DEV), torch.empty(OUT_F - 1, dtype=torch.bfloat16, device=DEV),
                torch.empty(OUT_F, dtype=torch.bfloat16)):
        with pytest.raises(ValueError):
            bx.bf16x_gemv(x, *w, OUT_F, IN_F, plan=plan, out=out)
    with pytest.raises(bx.Bf16xError):
        bx.bf16x_gemv(x, *w, OUT_F, IN_F, plan=plan, sub=32)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda v: bx.bf16x_gemv(v, *w, OUT_F, IN_F, plan=plan))(x.view(1, -1))


def test_stream_and_capture(bx, weight):  # noqa: F811
    """The launch goes to torch's current stream, and into a graph."""
    w, plan = weight
    x = torch.randn(IN_F, device=DEV).to(torch.bfloat16)
    want = bx.bf16x_gemv(x, *w, OUT_F, IN_F, plan=plan)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        assert bx._lib.stream_of(x.device) == side.cuda_stream
        y = bx.bf16x_gemv(x, *w, OUT_F, IN_F, plan=plan)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(y, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = bx.bf16x_gemv(x, *w, OUT_F, IN_F, plan=plan)
    for k in range(3):
        x.neg_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, -want if k % 2 == 0 else want)


def test_gemv_lets_other_threads_run(bx, weight):  # noqa: F811
    """The native GEMV call gives up the GIL: with the interpreter's own
    switching off, a thread that waits for it runs between two instructions of
    a caller that does nothing else."""
    w, plan = weight
    x = torch.zeros(IN_F, dtype=torch.bfloat16, device=DEV)
    out = torch.empty(OUT_F, dtype=torch.bfloat16, device=DEV)       # (freeing a result would give it up too)
    args = (x, *w, plan.tile_off, plan.tile_ent, plan.tile_sat, OUT_F, IN_F, 16, out)
    gemv = bx._lib.host().gemv
    assert gemv(*args) is out
    go, ran = threading.Lock(), []
    go.acquire()
    t = threading.Thread(target=lambda: (go.acquire(), ran.append(1)))
    t.start()
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1000.0)
    try:
        go.release()
        for _ in range(20000):                       # (some tens suffice)
            gemv(*args)
            if ran:
                break
        met = bool(ran)
    finally:
        sys.setswitchinterval(interval)
    t.join()
    torch.cuda.synchronize()
    assert met


def test_runtime_error_is_raised_and_not_launched_again(bx, weight, monkeypatch):  # noqa: F811
    """A runtime error is reported after the kernel was enqueued: the wrapper
    raises it and does not run the GEMV a second time.  The error is one left
    pending in the runtime by a refused host call (no such device)."""
    w, plan = weight
    x = torch.zeros(IN_F, dtype=torch.bfloat16, device=DEV)
    out = torch.empty(OUT_F, dtype=torch.bfloat16, device=DEV)
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(ln.split()[-1] for ln in f if "libamdhip64" in ln))
    lib, again = bx._lib.lib(), []

    class Lib:
        def __getattr__(self, name):
            if name == "bf16x_gemv":
                again.append(name)
            return getattr(lib, name)

    bx.bf16x_gemv(x, *w, OUT_F, IN_F, plan=plan, out=out)
    monkeypatch.setattr(bx._lib, "lib", lambda: Lib())
    pending = hip.hipSetDevice(1 << 12)
    assert pending > 0
    with pytest.raises(bx.Bf16xError) as e:
        bx.bf16x_gemv(x, *w, OUT_F, IN_F, plan=plan, out=out)
    assert e.value.status == pending and not again
    torch.cuda.synchronize()
    bx.bf16x_gemv(x, *w, OUT_F, IN_F, plan=plan, out=out)             # the error was taken with the report
