"""Linking a torch tensor gives what the DLPack exchange gives: the same
storage under a version counter of its own, and the same refusals."""
import pytest
import torch

from astra import _core


def _link(obj, shape=(3, 4)):
    return _core.link_data("-vol", None, shape, obj)


@pytest.mark.parametrize("make", [lambda: torch.zeros(3, 4), lambda: torch.zeros(2, 3, 4)[1],
                                  lambda: torch.nn.Parameter(torch.zeros(3, 4), requires_grad=False)])
def test_same_storage_own_version(make):
    t = make()
    d = _link(t)
    v = t._version
    d.store(2.0)
    assert d.linked.data_ptr() == t.data_ptr() and t._version == v
    assert float(t.sum()) == 24.0 and not d.linked.requires_grad


def _made_under_inference_mode():
    with torch.inference_mode():
        return torch.zeros(3, 4)


def test_inference_tensor_is_written_outside_the_mode():
    t = _made_under_inference_mode()
    d = _link(t)
    d.store(2.0)
    d.write_back(torch.full((3, 4), 5.0))
    assert d.linked.data_ptr() == t.data_ptr() and float(t.sum()) == 60.0
    assert not d.linked.is_inference()


@pytest.mark.filterwarnings("ignore:Named tensors")
def test_named_tensor_links_without_its_names():
    t = torch.zeros(3, 4, names=("row", "col"))
    d = _link(t)
    d.store(2.0)
    assert d.linked.data_ptr() == t.data_ptr() and d.linked.names == (None, None)
    assert float(t.rename(None).sum()) == 24.0


@pytest.mark.parametrize("make", [
    lambda: torch.zeros(3, 4, requires_grad=True),
    lambda: torch.zeros(3, 4, dtype=torch.float64),
    lambda: torch.zeros(4, 3),
    lambda: torch.zeros(4, 3).t(),
    lambda: torch.zeros(3, 4, dtype=torch.complex64).conj().imag,
    lambda: torch.zeros(3, 4).to_sparse(),
    lambda: torch.zeros(3, 4, device="meta"),
    lambda: torch.nested.nested_tensor([torch.zeros(4)] * 3),
])
def test_refused(make):
    with pytest.raises(ValueError):
        _link(make())


def test_refused_under_vmap():
    def f(x):
        _link(x)
        return x
    with pytest.raises(ValueError):
        torch.func.vmap(f)(torch.zeros(2, 3, 4))
