"""BitLinear's packed weights are kept per weight version and device: a pack for
another device between the key's check and the store (another thread's call)
reaches neither call's weights, and equal padded widths share one packing."""
import copy

import pytest
import torch

import rational_bitnet
from rational_bitnet import BitLinear


@pytest.fixture
def packs(monkeypatch):
    calls = []

    def pack(w):
        calls.append(w.device.type)
        return w
    monkeypatch.setattr(rational_bitnet.ops, "pack_ternary", pack)
    return calls


def test_pack_of_another_device_in_between(packs, monkeypatch):
    layer = BitLinear(24, 8)
    pack = rational_bitnet.ops.pack_ternary

    def pack_with_other(w):
        if w.device.type == "cpu" and "meta" not in packs:
            layer._packed_weights(torch.device("meta"), 64)     # the other thread
        return pack(w)
    monkeypatch.setattr(rational_bitnet.ops, "pack_ternary", pack_with_other)
    assert layer._packed_weights(torch.device("cpu"), 64)[0].device.type == "cpu"
    assert layer._packed_weights(torch.device("meta"), 64)[0].device.type == "meta"
    assert layer._packed_weights(torch.device("cpu"), 64)[0].device.type == "cpu"


def test_new_weights_are_packed_again(packs):
    layer = BitLinear(24, 8)
    a = layer._packed_weights(torch.device("cpu"), 64)[0]
    assert layer._packed_weights(torch.device("cpu"), 64)[0] is a and len(packs) == 1
    with torch.no_grad():
        layer.weight.neg_()
    b = layer._packed_weights(torch.device("cpu"), 64)[0]
    assert torch.equal(a, -b)


@pytest.mark.parametrize("k,count", [(128, 1), (100, 2)])
def test_equal_widths_share_a_packing(packs, k, count):
    layer = BitLinear(k, 8)
    assert layer._packed_weights(torch.device("cpu"), 64)[0].shape[1] == 128
    assert layer._packed_weights(torch.device("cpu"), 16)[0].shape[1] == -(-k // 16) * 16
    assert len(packs) == count


@pytest.mark.parametrize("held", [None, {}, {64: (torch.zeros(8, 16, dtype=torch.uint8), 1.0)}], ids=["none", "empty", "packed"])
def test_module_saved_whole_by_earlier_versions(packs, held):
    layer = BitLinear(24, 8)
    state = dict(layer.__dict__, _packed=held, _packed_key=None)
    loaded = BitLinear.__new__(BitLinear)
    loaded.__setstate__(state)
    assert torch.equal(loaded._packed_weights(torch.device("cpu"), 64)[0], layer._packed_weights(torch.device("cpu"), 64)[0])


def test_copy_packs_its_own_weights(packs):
    layer = BitLinear(24, 8)
    layer._packed_weights(torch.device("cpu"), 64)
    for other in (copy.copy(layer), copy.deepcopy(layer)):
        other._packed_weights(torch.device("cpu"), 16)
        assert set(layer._packed[1]) == {64}
