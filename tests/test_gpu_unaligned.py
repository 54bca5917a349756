"""Attention at head dims 48, 80, 96 and 112 on tensors off a 16-byte boundary
(contiguous views one element into a larger buffer): the same bits as on
aligned ones, in the outputs and the gradients, written and added, with nothing
outside the views touched."""
import pytest
import torch

from femtochat_amd import MFMAExact, MFMAFast, attention_, delta_attention_
from tests.helpers import gpu_backward, gpu_forward

pytestmark = pytest.mark.gpu


def _off(x):
    """A contiguous copy of x one element past a 256-byte boundary, and its buffer."""
    buf = torch.full((x.numel() + 9,), 7.0, dtype=x.dtype, device=x.device)
    view = buf[1:1 + x.numel()].view(x.shape)
    view.copy_(x)
    assert view.is_contiguous() and view.data_ptr() % 16 != 0
    return view, buf


@pytest.mark.parametrize("mode,D", [("fast", 48), ("fast", 80), ("fast", 96), ("fast", 112), ("exact", 48), ("exact", 80), ("exact", 96),
                                    ("exact", 112)])
def test_unaligned_views(gpu, mode, D):
    A, dt = (MFMAFast(), torch.bfloat16) if mode == "fast" else (MFMAExact(), torch.float32)
    B, T, H, Hkv, window = 2, 77, 4, 2, (-1, 0)
    g = torch.Generator(device=gpu).manual_seed(D)
    rand = lambda h: torch.randn(B, T, h, D, device=gpu, generator=g).to(dt)
    Q, K, V, dO, base = rand(H), rand(Hkv), rand(Hkv), rand(H), [rand(H), rand(Hkv), rand(Hkv)]
    O, l, m = gpu_forward(A, Q, K, V, window)
    O2, O2_buf = _off(torch.zeros_like(O))
    l2, m2 = torch.empty_like(l), torch.empty_like(m)
    Qo, Ko, Vo, dOo = (_off(x)[0] for x in (Q, K, V, dO))
    attention_(A, O2, l2, m2, Qo, Ko, Vo, window)
    assert torch.equal(O2, O) and torch.equal(l2, l) and torch.equal(m2, m)
    buffers = [O2_buf]
    for accumulate in (False, True):
        want = gpu_backward(A, dO, Q, K, V, O, l, m, window, accumulate=accumulate, init=base)
        grads = [_off(x) for x in base]
        delta_attention_(A, *(x for x, _ in grads), dOo, Qo, Ko, Vo, O2, l, m, window, accumulate=accumulate)
        for (x, buf), w in zip(grads, want):
            assert torch.equal(x, w)
            buffers.append(buf)
    for buf in buffers:
        assert buf[0] == 7.0 and bool((buf[-8:] == 7.0).all())
