"""CPU tests around the device plan builders: the dict's GPU is the current
device while one runs, and a CSR's offsets cover no entry twice."""
import contextlib
import ctypes

import pytest
import torch

import bfloat16x_amd as bx
from bfloat16x_amd import _lib, codec


def test_device_builder_runs_on_the_dicts_gpu(monkeypatch):
    """A dict on a GPU that is not the current one: its stream, both launches
    and the wait for the count belong inside a guard for the dict's device.
    (A null stream handle means the current device's default stream.)"""
    d = bx.bf16x_quantize(torch.randn(8, 96, generator=torch.Generator().manual_seed(0)))
    d["delta_ovf_idx"], d["delta_ovf_val"] = torch.tensor([5], dtype=torch.int32), torch.tensor([9], dtype=torch.uint8)
    current, seen = ["another"], []

    @contextlib.contextmanager
    def guard(device):
        before, current[0] = current[0], device
        yield
        current[0] = before

    class Lib:
        def __getattr__(self, name):
            return getattr(_lib._LIB, name)

        def bf16x_plan_device_count(self, *a):
            seen.append(("count", current[0]))
            ctypes.c_int64.from_address(a[9]).value = 0
            return 0

        def bf16x_plan_device_write(self, *a):
            seen.append(("write", current[0]))
            return 0

    _lib.lib()
    monkeypatch.setattr(codec, "_on_device", lambda packed, device: True)
    monkeypatch.setattr(torch.cuda, "device", guard)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(_lib, "lib", lambda stub=Lib(): stub)
    monkeypatch.setattr(_lib, "stream_of", lambda dev: seen.append(("stream", current[0])) or 0)
    plan = bx.build_plan_host(d, device="cuda:1")
    where = d["delta_ovf_idx"].device
    assert seen == [("stream", where), ("count", where), ("write", where)]
    assert plan.n_fix == 0 and current == ["another"]


@pytest.mark.parametrize("off", [[0, 3, 3, 7, 9], [0, 9, 0, 9, 9], [-5, 4, 2, 100, 1], [9, 0, 0, 0, 0], [0, 0, 0, 0, 0]])
def test_csr_offsets_cover_no_entry_twice(off):
    """Well-formed offsets stay; others become ascending inside [0, n], so the
    rows' entries together are at most n."""
    n = 9
    got = codec._csr_offsets(torch.tensor(off, dtype=torch.int32), n)
    assert got.dtype == torch.int32 and got.is_contiguous() and got.numel() == len(off)
    d = got.diff()
    assert int(got.min()) >= 0 and int(got.max()) <= n and bool((d >= 0).all()) and int(d.sum()) <= n
    if sorted(off) == off:
        assert got.tolist() == off
