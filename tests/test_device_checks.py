"""Argument checks of DeviceStep that come before any call of the library (the context
is a stand-in whose library calls fail the test)."""

import pytest
import torch

from cs_afqmc_amd.device import DeviceStep

W = 4


class _NoCalls:
    def __getattr__(self, name):
        raise AssertionError(f"library call {name}")


@pytest.fixture
def dev(monkeypatch):
    d = object.__new__(DeviceStep)
    d._lib, d._h = _NoCalls(), None
    monkeypatch.setattr(DeviceStep, "_walkers", lambda self, w: (w, None, W))
    monkeypatch.setattr(DeviceStep, "_prep", lambda self: self._lib.afqmc_set_stream())
    return d


def refuses(dev, overlaps):
    """The kernel writes n_walkers complex128 values at the tensor's address."""
    with pytest.raises(TypeError, match="overlaps"):
        dev.energy(torch.zeros(W, 1, 1), out=torch.zeros(W, dtype=torch.complex128),
                   overlaps=overlaps)


@pytest.mark.parametrize("overlaps", [torch.zeros(W, dtype=torch.complex128), [0j] * W])
def test_energy_refuses_host_overlaps(dev, overlaps):
    refuses(dev, overlaps)


@pytest.mark.gpu
def test_energy_refuses_overlaps_of_other_sizes_and_types(dev, gpu):
    for shape, dtype in ((W, torch.complex64), (W, torch.float64), (W - 1, torch.complex128)):
        refuses(dev, torch.zeros(shape, dtype=dtype, device=gpu))
    refuses(dev, torch.zeros((W, 2), dtype=torch.complex128, device=gpu)[:, 0])
