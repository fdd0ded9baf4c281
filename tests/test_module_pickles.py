"""Modules pickled whole (torch.save(module)), also in the form they had before the native host path kept their counters."""

import copy
import io

import pytest
import torch

import viola_amd


def _saved(module):
    file = io.BytesIO()
    torch.save(module, file)
    file.seek(0)
    return torch.load(file, weights_only=False)                                # a file that this test wrote


def _module(scaling):
    module = viola_amd.nn.Linear(64, 32, dtype=torch.bfloat16, scaling=scaling, weight_dtype="bf16")
    module.input_quantizer.index = 5
    return module


@pytest.mark.parametrize("used", [False, True])
@pytest.mark.parametrize("scaling", ["current", "delayed"])
def test_round_trip(scaling, used):
    module = _module(scaling)
    if used:
        module._operands()                                                     # the native recipe and counters now exist
    for made in (_saved(module), copy.deepcopy(module)):
        assert (made.input_quantizer.index, made.input_quantizer.scaling) == (5, scaling)
        made.input_quantizer.index = 7
        assert module.input_quantizer.index == 5
        counter = made.input_quantizer.counter()
        assert (counter.value, counter.delayed) == (7, scaling == "delayed") and made._operands() is not None


@pytest.mark.parametrize("scaling", ["current", "delayed"])
def test_attributes_of_earlier_pickles(scaling):
    """`scaling` and `index` were plain attributes, and a Linear knew no recipe."""
    module = _module(scaling)
    state = dict(module.input_quantizer.__dict__)
    for held in ("_scaling", "_calls", "_counter"):
        del state[held]
    old = type(module.input_quantizer).__new__(type(module.input_quantizer))
    old.__setstate__(dict(state, scaling=scaling, index=9))
    assert (old.index, old.scaling, old.counter().value, old.counter().delayed) == (9, scaling, 9, scaling == "delayed")
    state = {key: value for key, value in module.__dict__.items() if key != "_recipe"}
    layer = viola_amd.nn.Linear.__new__(viola_amd.nn.Linear)
    layer.__setstate__(state)
    assert layer._operands() is not None


def test_a_quantizer_that_changes_its_scaling_tells_the_counter():
    quantizer = _module("current").input_quantizer
    counter = quantizer.counter()
    quantizer.set_extra_state({"index": 3, "scaling": "delayed"})
    assert (counter.value, counter.delayed, quantizer.get_extra_state()) == (3, True, {"index": 3, "scaling": "delayed"})
