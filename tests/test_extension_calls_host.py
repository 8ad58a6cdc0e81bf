"""The fast form of the extension's operators, on the host: whatever is no plain int or tensor, is missing, too large or named goes to the
general function and fails or passes as it does there."""
import numpy as np
import pytest
import torch

import TAB_CUDA
from tab_amd import _C

X = torch.zeros(1, 8, 8, 64)
CALLS = {"Conv2d": (4, 12), "TAB_Conv2d": (4, 12), "Quantize": (2, 5), "TAB_Quantize": (2, 5), "QuantizeNCHW": (2, 5), "Conv2dPacked": (3, 12)}


class Named(torch.Tensor):
    pass


@pytest.mark.parametrize("name", CALLS)
def test_arguments(name):
    tensors, ints = CALLS[name]
    f = getattr(_C, name)
    assert not hasattr(TAB_CUDA, name) or getattr(TAB_CUDA, name) is f
    assert f.__name__ == name and "torch.Tensor" in f.__doc__
    numbers = [1] * ints
    for args in ([X] * tensors + numbers, [torch.nn.Parameter(X)] * tensors + numbers, [X.as_subclass(Named)] * tensors + numbers,
                 [X] * tensors + [np.int64(1)] * ints, [X] * tensors + [True] * ints):  # taken: the check of the device is the first to fail
        with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
            f(*args)
    for args in ([X] * tensors + numbers[1:], [X] * tensors + numbers + [1], [X] * tensors + [2**31] + numbers[1:], [X] * tensors + [2**80] + numbers[1:],
                 [X] * tensors + [-2**31 - 1] + numbers[1:], [X] * tensors + [1.5] + numbers[1:], [X] * tensors + [None] + numbers[1:],
                 ["x"] + [X] * (tensors - 1) + numbers, [np.zeros(4)] + [X] * (tensors - 1) + numbers, []):
        with pytest.raises(TypeError, match="incompatible function arguments"):
            f(*args)
    with pytest.raises(TypeError, match="incompatible function arguments"):
        f(*([X] * tensors + numbers[1:]), stride=1)


class Watched(torch.Tensor):
    """A tensor whose device an operator has to ask for in Python, where it can be told that it is elsewhere, or fail."""
    asked, fails = 0, False

    @staticmethod
    def __new__(cls):
        return torch.Tensor._make_wrapper_subclass(cls, (1, 8, 8, 64), dtype=torch.float32, device="cpu", dispatch_device=True)

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        assert func is torch.ops.prim.device.default, func
        cls.asked += 1
        if cls.fails:
            raise KeyError("device of a watched tensor")
        return torch.device("cpu")


@pytest.mark.parametrize("fails, error, words", [(False, RuntimeError, "must be a CUDA tensor"), (True, KeyError, "device of a watched tensor")])
@pytest.mark.parametrize("name", CALLS)
def test_an_operator_is_entered_once(name, fails, error, words):
    """Whatever an operator throws reaches the caller: a second try through the general function would launch, allocate and ask again."""
    tensors, ints = CALLS[name]
    x, Watched.fails, Watched.asked = Watched(), fails, 0
    with pytest.raises(error, match=words):
        getattr(_C, name)(x, *[X] * (tensors - 1), *[1] * ints)
    assert Watched.asked == 1


@pytest.mark.parametrize("name", CALLS)
def test_errors_name_the_function_that_was_called(name):
    with pytest.raises(TypeError, match=rf"^{name}\(\): incompatible function arguments"):
        getattr(_C, name)(1)
