"""Backward of 256-wide heads, whose waves work in pairs: one, two and three tiles a walk, blocks that nobody sees, walks over
several query heads, against the fp32 reference (bounds as in test_attention_edges_gpu.py)."""
import pytest

import torch

from kubernetes_cloud_amd.ops import attention as A

from .test_attention_edges_gpu import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Sq,Sk", [(1, 1), (31, 31), (33, 33), (64, 64), (65, 97), (96, 300), (128, 128), (129, 257), (260, 260)])
def test_walks(Sq, Sk, causal):
    _check(2, Sq, Sk, 3, 3, 256, causal)
    _check(2, Sq, Sk, 4, 2, 256, causal)


@pytest.mark.parametrize("causal", [True, False])
def test_masks(causal):
    _check(7, 290, 290, 2, 2, 256, causal, lens=[290, 0, 1, 127, 128, 129, 33])
    if causal:
        _check(2, 290, 290, 4, 1, 256, True, lens=[200, 31], alibi=True)
        for window in (1, 32, 33, 150):
            _check(2, 290, 290, 4, 2, 256, True, window=window)
        _check(2, 140, 330, 4, 1, 256, True, window=64, alibi=True)


def test_rows_off_16_bytes():
    """Full tiles in rows that 16-byte loads do not fit keep the kernels of one wave a block."""
    g = torch.Generator(device="cuda").manual_seed(1)
    t = [torch.randn(1, 128, 2, 260, device="cuda", generator=g).bfloat16()[..., 2:258] for _ in range(3)]
    grads = []
    for off in (False, True):
        q, k, v = (x.requires_grad_() if off else x.detach().contiguous().requires_grad_() for x in (y.detach() for y in t))
        A.flash_attention(q, k, v, causal=True).float().square().sum().backward()
        grads.append((q.grad, k.grad, v.grad))
    for a, b in zip(*grads):
        assert (a.float() - b.float()).norm() <= 3 * 2.0 ** -9 * b.float().norm()
