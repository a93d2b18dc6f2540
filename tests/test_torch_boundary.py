"""What crosses from torch into the runtime and back without a numpy array in between: only tensors whose memory holds their values."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from ttmlir_amd import runtime as rt


def _fake():
    with FakeTensorMode():
        return torch.randn(4)


@pytest.mark.parametrize("borrowed", [False, True])
@pytest.mark.parametrize("make", [lambda: torch.tensor([1 + 2j]).conj().imag, lambda: torch._neg_view(torch.arange(4.0)),
                                  lambda: torch._efficientzerotensor(4), _fake], ids=["conj_imag", "neg_view", "zero_tensor", "fake"])
def test_tensors_whose_memory_is_not_their_values_are_refused(make, borrowed):
    with pytest.raises(RuntimeError):
        rt.from_torch(make(), borrowed=borrowed)


def test_other_kinds_of_tensors_keep_their_values():
    class Named(torch.Tensor):
        pass
    x = torch.arange(6.0).reshape(2, 3)
    for t in (x.as_subclass(Named), torch.nn.Parameter(x, requires_grad=False), torch.tensor([1 - 2j, 3 + 4j]).imag, x.t(), x.expand(4, 2, 3),
              torch._neg_view(x).resolve_neg(), torch.empty(0, 3)):
        assert torch.equal(rt.to_torch(rt.from_torch(t)), torch.Tensor(t))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.int32, torch.uint8])
def test_results_come_back_to_host_memory_whatever_the_default_device(dtype):
    x = torch.arange(2000).reshape(50, 40).to(dtype)
    host = rt.from_torch(x)
    with torch.device("meta"):
        back = rt.to_torch(host)
    assert back.device.type == "cpu" and torch.equal(back, x)
    with FakeTensorMode():
        fake = rt.to_torch(host)
    assert fake.shape == x.shape and fake.dtype == dtype
