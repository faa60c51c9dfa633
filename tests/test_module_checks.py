"""What kernels that stand in for modules look at first (chunk_attn_c.modules), on the CPU."""
import pytest
import torch
from torch import nn

from chunk_attn.capi import modules

CPU = torch.device("cpu")


def _linear(n_out=8, n_in=64, **kw):
    return nn.Linear(n_in, n_out, bias=False, dtype=torch.float16, **kw)


def _weights(*linears, n_out=-1, n_in=64, device=CPU, grad=False):
    return modules.linear_weights(linears, nn.Linear, nn.Parameter, n_out, n_in, device, grad)


def test_plain_linears_give_their_weights_addresses():
    a, b = _linear(8), _linear(24)
    addresses, kept = _weights(a, b)
    assert addresses == [a.weight.data_ptr(), b.weight.data_ptr()] and kept[0] is a.weight and kept[1] is b.weight
    assert _weights(a, n_out=8) is not None and _weights(a, b, n_out=8) is None
    assert _weights() == ([], [])


class Derived(nn.Linear):
    pass


class DerivedParameter(nn.Parameter):
    pass


def _hidden(name):
    m = _linear()
    m.__dict__[name] = torch.zeros(8, 64)
    return m


def _with(change):
    m = _linear()
    change(m)
    return m


@pytest.mark.parametrize("m", [
    Derived(64, 8, bias=False, dtype=torch.float16), nn.Linear(64, 8, dtype=torch.float16), nn.Linear(64, 8, bias=False), _linear(n_in=128),
    _hidden("weight"), _hidden("bias"), _hidden("forward"), None, torch.zeros(8, 64),
    _with(lambda m: m.register_forward_hook(lambda *a: None)), _with(lambda m: m.register_forward_pre_hook(lambda *a: None)),
    _with(lambda m: m.register_full_backward_hook(lambda *a: None)), _with(lambda m: m.register_full_backward_pre_hook(lambda *a: None)),
    _with(lambda m: m._parameters.__setitem__("weight", torch.zeros(8, 64, dtype=torch.float16))),
    _with(lambda m: m._parameters.__setitem__("weight", DerivedParameter(torch.zeros(8, 64, dtype=torch.float16)))),
    _with(lambda m: m._parameters.pop("weight")), _with(lambda m: m._parameters.pop("bias")),
    _with(lambda m: setattr(m, "weight", nn.Parameter(torch.zeros(64, 8, dtype=torch.float16).t()))),
    _with(lambda m: setattr(m, "weight", nn.Parameter(torch.zeros(8 * 64 + 1, dtype=torch.float16)[1:].view(8, 64)))),
    _with(lambda m: setattr(m, "weight", nn.Parameter(torch.zeros(1, 8, 64, dtype=torch.float16)))),
])
def test_anything_else_is_left_to_the_modules(m):
    assert _weights(_linear(), m) is None


def test_device_gradient_and_removed_hooks():
    m = _linear()
    assert _weights(m, device=torch.device("cuda", 0)) is None and _weights(m, device=torch.device("meta")) is None
    assert _weights(m, grad=True) is None and _weights(m.requires_grad_(False), grad=True) is not None
    m.register_forward_hook(lambda *a: None).remove()
    assert _weights(m) is not None


def test_bare_modules_and_parameters():
    m = nn.Embedding(4, 8)
    assert modules.all_bare(nn.Embedding, (m, nn.Embedding(2, 2))) and modules.all_bare(nn.Linear, [])
    assert not modules.all_bare(nn.Embedding, (m, _linear())) and not modules.all_bare(nn.Linear, [Derived(2, 2)])
    m.forward = lambda x: x
    assert not modules.all_bare(nn.Embedding, (m,))
    good = nn.Parameter(torch.zeros(16, dtype=torch.float16))

    def taken(*t):
        return modules.parameter_addresses(t, nn.Parameter, (16,), CPU)

    assert taken(good, good) == [good.data_ptr()] * 2
    for bad in (None, good.data, nn.Parameter(torch.zeros(16)), nn.Parameter(torch.zeros(1, 16).half()), nn.Parameter(torch.zeros(32).half()[::2]),
                nn.Parameter(torch.zeros(17).half()[1:]), nn.Parameter(torch.zeros(15).half())):
        assert taken(good, bad) is None


def test_attributes_that_hide_a_registered_child_are_the_ones_looked_at():
    class Holder(nn.Module):
        def __init__(self):
            super().__init__()
            self.child = _linear()

    m = Holder()
    assert modules.children_bare(nn.Linear, (m,), "child") and not modules.children_bare(nn.Embedding, (m,), "child")
    with pytest.raises(AttributeError):
        modules.children_bare(nn.Linear, (m,), "other")
    m.__dict__["child"] = Derived(2, 2)
    assert not modules.children_bare(nn.Linear, (m,), "child")
    del m.__dict__["child"]
    Holder.child = property(lambda self: nn.Embedding(2, 2))
    assert not modules.children_bare(nn.Linear, (m,), "child")
