"""`device_arch` answers for the device it is asked about, now: two fake devices of different
architectures, the current one changing between calls (CPU)."""
import collections

import pytest
import torch

ARCHS = {0: "gfx950:sramecc+:xnack-", 1: "gfx942:sramecc+:xnack-"}
Props = collections.namedtuple("Props", "gcnArchName")


@pytest.fixture
def sk1(monkeypatch):
    import sageattention.sk1_backend as mod
    world = {"current": 0}

    def get_device_properties(device=None):
        if isinstance(device, int):
            index = device
        else:
            d = torch.device(device) if isinstance(device, str) else device
            if d is not None and d.type != "cuda":
                raise ValueError("Expected a cuda device, but got: %s" % d)
            index = world["current"] if d is None or d.index is None else d.index
        if index not in ARCHS:
            raise AssertionError("Invalid device id")
        return Props(ARCHS[index])

    monkeypatch.setattr(torch.cuda, "get_device_properties", get_device_properties)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: world["current"])
    monkeypatch.setattr(mod, "_ARCHS", {})
    return mod, world


@pytest.mark.parametrize("asked", [None, "cuda", torch.device("cuda")], ids=str)
def test_a_device_without_an_index_is_the_current_one(sk1, asked):
    mod, world = sk1
    for current, arch in ((0, "gfx950"), (1, "gfx942"), (0, "gfx950")):
        world["current"] = current
        assert mod.device_arch(asked) == arch
        assert mod.arch_supported(asked) == (arch == "gfx950")


@pytest.mark.parametrize("current", [0, 1])
def test_a_named_device_is_that_one(sk1, current):
    mod, world = sk1
    world["current"] = current
    for _ in range(2):
        for asked in (0, "cuda:0", torch.device("cuda", 0)):
            assert mod.device_arch(asked) == "gfx950"
        for asked in (1, "cuda:1", torch.device("cuda", 1)):
            assert mod.device_arch(asked) == "gfx942"


def test_what_is_no_gpu_has_no_architecture(sk1):
    mod, _ = sk1
    assert mod.device_arch(None) == "gfx950"
    for asked in ("cpu", torch.device("cpu"), 7, torch.device("cuda", 7), "no such device", [0]):
        assert mod.device_arch(asked) == ""
