"""The native host path (csrc/py_native.cpp) and its callers where they can be tested without a GPU: what is refused before a
tensor is looked at, and which calls take that path."""
import numpy as np
import pytest
import torch

from ternainfer_amd import _lib, linear

#: arguments of every function: T a tensor, o a tensor or None, i an integer, f a number, b a truth value
ATTENTION = "TTTTTiifi"
SIGNATURES = {
    "bit_linear": "ToTTTTTiio", "bit_linear_bf16": "TTTTTTiii", "quant_input": "T", "linear_packed": "TTTTiio", "linear_bf16_packed": "TTTiio",
    "rmsnorm_quant": "TTfob", "relu2_mul_rmsnorm_quant": "TTfb", "quant_from_stats": "TTTf", "fused_linear": "TofTTiiioiioioobb", "fused_linear_own_stats": "TofTTiiioiioioobb",
    "prompt_attention": "T" + ATTENTION + "b", "decode_attention": "T" + ATTENTION + "oooi",
    "block": "To" + ATTENTION + "foo" + "TTTT" + "TTii" * 4 + "o", "attention_merge_rmsnorm_quant": "TiiiTfib", "step_inputs": "TTTTT",
    "prompt_inputs": "TTTT",
}
VALUES = {"T": torch.zeros((1, 64)), "o": None, "i": 1, "f": 1.0, "b": False}


def _arguments(name):
    """Arguments of the right kinds; where shapes are checked between two tensors, of the right shapes too (one token, one head of
    64 columns, 64 columns everywhere), so that every tensor's turn comes."""
    values = [VALUES[k] for k in SIGNATURES[name]]
    bf = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16)
    attention = [torch.zeros((1, 32)), torch.zeros((1, 32)), torch.zeros(1, dtype=torch.int64), bf(1, 1, 4, 64), bf(1, 1, 4, 64), 1, 64, 1.0, 1]
    if name in ("prompt_attention", "decode_attention"):
        values[:10] = [bf(1, 192)] + attention
    if name == "block":
        values[:2] = [bf(1, 64), None]
        values[2:11] = attention
        values[14:18] = [bf(64)] * 4
        for at, n in ((18, 192), (22, 64), (26, 128), (30, 64)):
            values[at:at + 4] = [torch.zeros(n * 16, dtype=torch.int8), bf(4), 1, n]
    if name.startswith("fused_linear"):
        values[7] = 64
    return values


@pytest.mark.parametrize("name", sorted(SIGNATURES))
def test_arguments_that_are_no_tensors_raise_type_error(name):
    """None in the place of a required tensor, and an object of another type in the place of any, raise TypeError (they were read
    through as pointers)."""
    function, kinds = getattr(_lib.native(), name), SIGNATURES[name]
    for at, kind in enumerate(kinds):
        if kind in "To":
            for wrong in ([None] if kind == "T" else []) + [np.zeros((1, 64), np.float32), 7]:
                arguments = _arguments(name)
                arguments[at] = wrong
                with pytest.raises(TypeError):
                    function(*arguments)


def test_wrong_argument_count_raises_type_error():
    for name, kinds in SIGNATURES.items():
        with pytest.raises(TypeError, match="arguments expected"):
            getattr(_lib.native(), name)(*[None] * (len(kinds) + 1))


class _Quantised(Exception):
    pass


def _own_quantiser(*_):
    raise _Quantised


def _module(cls=linear.SpBitLinear):
    """An `SpBitLinear` of 64 x 64 without its weights on a GPU."""
    m = cls.__new__(cls)
    torch.nn.Module.__init__(m)
    m.in_features = m.out_features = 64
    m.ws_num = 1
    for name in ("packed", "bitmap", "TileOffsets_global", "TileOffsets_median", "compressed_val", "scale"):
        m.register_parameter("weight_" + name, torch.nn.Parameter(torch.zeros(1), requires_grad=False))
    return m


@pytest.mark.parametrize("how", ["subclass", "instance", "class"])
def test_spbitlinear_calls_a_quant_input_of_its_own(how, monkeypatch):
    """A `quant_input` that a subclass, an instance or a patch of the class brings is the one that `forward` quantises with; only
    the module's own is left to the native call."""
    taken = []
    monkeypatch.setattr(_lib, "native", lambda: type("Native", (), {"bit_linear": staticmethod(lambda x, *_: taken.append(x) or x)}))
    monkeypatch.setattr(linear, "get_global_workspace", lambda *_: None)
    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    assert _module()(x) is x and len(taken) == 1
    if how == "subclass":
        module = _module(type("Own", (linear.SpBitLinear,), {"quant_input": _own_quantiser}))
    else:
        module = _module()
        if how == "instance":
            module.quant_input = _own_quantiser
        else:
            monkeypatch.setattr(linear.SpBitLinear, "quant_input", _own_quantiser)
    with pytest.raises(_Quantised):
        module(x)
    assert len(taken) == 1
