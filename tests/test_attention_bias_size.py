"""The additive bias of an attention call holds every plane that the kernel reads; no kernel is launched here."""
import pytest
import torch

from aidotnet.tensors_amd import ArgumentException, ArgumentOutOfRangeException, Mi355Backend, Mi355Engine
from aidotnet.tensors_amd.backend import GpuBuffer

B, H, Sq, Sk, D = 2, 3, 5, 7, 8


@pytest.fixture
def be():
    backend = object.__new__(Mi355Backend)
    backend.calls = []
    backend._attn = lambda kind, q, k, v, o, lse, bias, mask, weights, d: backend.calls.append((bias, d.bias_batch_stride))
    backend.WrapTensor = GpuBuffer
    return backend


def operands(Hkv=H):
    return torch.zeros(B, H, Sq, D), torch.zeros(B, Hkv, Sk, D), torch.zeros(B, Hkv, Sk, D)


@pytest.mark.parametrize("shape,stride", [((B, H, Sq, Sk), H * Sq * Sk), ((1, H, Sq, Sk), 0), ((H, Sq, Sk), 0)])
def test_planes_of_one_batch_or_of_all(be, shape, stride):
    """A bias of one batch is every batch's, with or without its leading dimension."""
    Mi355Engine(be).FlashAttention(*operands(), attentionBias=torch.zeros(shape))
    assert [s for _, s in be.calls] == [stride]


@pytest.mark.parametrize("shape", [(B, 1, Sq, Sk), (B, H, 1, Sk), (B, H, Sq, Sk - 1), (1, 1, Sq, Sk), (H - 1, Sq, Sk), (Sq, Sk)])
def test_too_few_planes(be, shape):
    with pytest.raises(ArgumentException):
        Mi355Engine(be).FlashAttention(*operands(), attentionBias=torch.zeros(shape))
    assert not be.calls


@pytest.mark.parametrize("elements,stride,error", [(H * Sq * Sk, 0, None), (H * Sq * Sk - 1, 0, ArgumentException), (H * Sq * Sk + 9, 9, None),
                                                  (H * Sq * Sk + 8, 9, ArgumentException), (4 * H * Sq * Sk, -1, ArgumentOutOfRangeException)])
def test_batch_stride(be, elements, stride, error):
    q, k, v = (GpuBuffer(x) for x in operands())
    call = lambda: be.FlashAttentionV2(q, k, v, GpuBuffer(torch.zeros(B, H, Sq, D)), GpuBuffer(torch.zeros(B, H, Sq)), B, H, Sq, Sk, D, 0.5, False,
                                       GpuBuffer(torch.zeros(elements)), stride)
    if error is None:
        call()
    else:
        with pytest.raises(error):
            call()
    assert len(be.calls) == (error is None)
