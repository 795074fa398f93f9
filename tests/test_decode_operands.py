"""Which query and token tensors the one-call decode steps accept: tokens on
another device than the query, or of another shape, go to the general path
(the kernel would take their addresses as its own device's)."""
import pytest
import torch

from helm_amd import _native
from helm_amd.runtime import kv_cache as KC

CUDA0, CUDA1, CPU = torch.device("cuda", 0), torch.device("cuda", 1), torch.device("cpu")


class Operand:
    """A 16-bit tensor's description on a device that need not exist."""

    def __init__(self, shape, device, dtype=torch.bfloat16):
        self._meta = torch.empty(shape, dtype=dtype, device="meta")
        self.shape, self.dtype, self.device = self._meta.shape, dtype, device
        self.is_cuda = device.type == "cuda"

    def stride(self):
        return self._meta.stride()

    def is_contiguous(self):
        return True

    def data_ptr(self):
        return 0x1000


def _operands(k_dev=CUDA0, v_dev=CUDA0, k_shape=(2, 8, 1, 128), v_shape=(2, 8, 1, 128)):
    return (Operand((2, 32, 1, 128), CUDA0), Operand(k_shape, k_dev), Operand(v_shape, v_dev))


def test_plain_operands_are_taken():
    assert KC._decode_operands_plain(*_operands())


@pytest.mark.parametrize("case", [
    {"k_dev": CPU}, {"v_dev": CPU}, {"k_dev": CPU, "v_dev": CPU},
    {"k_dev": CUDA1}, {"v_dev": CUDA1}, {"k_dev": CUDA1, "v_dev": CUDA1},
    {"v_shape": (2, 4, 1, 128)}, {"v_shape": (1, 8, 1, 128)},
    {"k_shape": (2, 8, 1, 64), "v_shape": (2, 8, 1, 64)},
])
def test_tokens_elsewhere_or_of_another_shape_are_not(case, monkeypatch):
    def called(*a):
        raise AssertionError("native call")

    monkeypatch.setitem(_native._entries, "helm_decode_step", called)
    q, k, v = _operands(**case)
    assert not KC._decode_operands_plain(q, k, v)
    assert KC._decode_contiguous_fast([None, None], q, k, v, 0, 1.0, None) is None
    assert KC._decode_step_fast([None, None], q, k, v, 0, 1.0, None) is None
