"""What LstmStack hands to the library: the plans its layers hold at the moment of the call."""
import ctypes

import pytest


class FakeCore:
    """A layer without a GPU: a handle until it is closed."""
    lib = None
    made = 0

    def __init__(self, batch, input_size, hidden_size):
        FakeCore.made += 1
        self._h = ctypes.c_void_p(0x1000 * FakeCore.made)

    def close(self):
        self._h = None


def test_closed_layers_are_null_pointers(monkeypatch):
    from flashlstm_poc_amd import stack
    monkeypatch.setattr(stack, "LstmCore", FakeCore)
    s = stack.LstmStack(2, 3, 4, 3)
    assert list(s._plans()) == [layer._h.value for layer in s.layers]
    s.layers[1].close()
    assert [p is None for p in s._plans()] == [False, True, False]
    s.close()
    assert list(s._plans()) == [None, None, None]


@pytest.mark.gpu
def test_a_closed_stack_refuses_its_passes():
    import torch
    from flashlstm_poc_amd import LstmStack
    s = LstmStack(2, 16, 32, 2)
    n = lambda *shape: torch.randn(*shape, device="cuda") * 0.1
    s.pack([(n(128, 16), n(128, 32), n(128), n(128)), (n(128, 32), n(128, 32), n(128), n(128))])
    x = n(4, 2, 16).half()
    y, _, _ = s.forward(x)
    s.layers[1].close()
    with pytest.raises((RuntimeError, ValueError)):
        s.backward(torch.ones_like(y))
    s.close()
    with pytest.raises(RuntimeError):
        s.forward(x)


@pytest.mark.gpu
def test_a_layer_used_with_accumulation_leaves_the_stack_usable():
    import torch
    from flashlstm_poc_amd import LstmStack
    s = LstmStack(2, 16, 32, 2)
    g = torch.Generator(device="cuda").manual_seed(3)
    n = lambda *shape: torch.randn(*shape, device="cuda", generator=g) * 0.1
    s.pack([(n(128, 16), n(128, 32), n(128), n(128)), (n(128, 32), n(128, 32), n(128), n(128))])
    x, dy = n(4, 2, 16).half(), n(4, 2, 32).half()
    s.forward(x)
    want = s.backward(dy)
    total = tuple(torch.zeros_like(t) for t in want[1][0])
    s.layers[0].backward(x, dy, accumulate_into=total)
    got = s.backward(dy)
    for a, b in zip(want[1][0] + want[1][1], got[1][0] + got[1][1]):
        assert torch.equal(a, b)
    s.close()
