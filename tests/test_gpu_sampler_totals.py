"""GPU check of the sampler's totals written to a place inside a pinned allocation (the kernel writes through the address
that the device has for it)."""
import pytest
import torch

from neat_amd import _abi

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("at", [0, 1, 5, 1021])
def test_totals_inside_an_allocation(at):
    print("case: sampler totals at", at, flush=True)
    off = torch.tensor([0, 3, 7], dtype=torch.int64, device=DEV)
    smp = torch.tensor([0, 30, 70], dtype=torch.int64, device=DEV)
    buf = torch.full((1024,), -1, dtype=torch.int64).pin_memory()
    _abi.call("neat_raysample_totals", _abi.stream_ptr(), _abi.ptr(off), _abi.ptr(smp), None, 2, _abi.ptr(buf[at:]))
    want = torch.full((1024,), -1, dtype=torch.int64)
    want[at:at + 3] = torch.tensor([7, 70, 0])
    assert torch.equal(buf, want)
