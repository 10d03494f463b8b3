"""Layers of other mixes of Q4_K and Q6_K than the decode kernel's under the
automatic choice, around the token counts where it moves from the per-token
kernels to the grouped path (6 with every tensor Q4_K, 12 with every gate and
up tensor Q4_K, 16 otherwise), for each tensor Q6_K by itself, and where the grouped path does not take the call
(Q6_K down weights or the residual 4-byte aligned only).

The grouped path keeps fp32's precision for these layers (the integer operands
exact, activations 22 bits), so it and the per-token kernels agree as two
fp32 sums of 256 and 512 products do: 512 roundings of 2^-24 at most, about
sqrt(512) of them in effect on each side, 4e-6 together with the gate/up sums.
"""
import numpy as np
import pytest
import torch

import breadv2_amd as B
from breadv2_amd import api

from helpers import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
Q4, Q6 = api.QTYPE_Q4_K, api.QTYPE_Q6_K
MIXES = [(Q4,) * 6, (Q6,) * 6] + [tuple(Q6 if j == i else Q4 for j in range(6)) for i in range(6)]


def run(s, d, x, hidden, path):
    T = x.shape[0]
    ctx = B.MoeContext(s, max_tokens=T)
    ctx.set_path(path)
    idx, w, g = ctx.forward(d, x, hidden, T, want_routing=True)
    torch.cuda.synchronize()
    assert ctx.check_device() == 0
    return hidden.cpu().numpy(), idx.cpu().numpy(), w.cpu().numpy(), g.cpu().numpy()


@pytest.mark.parametrize("T", [5, 6, 12, 16, 33])
@pytest.mark.parametrize("mix", MIXES)
@pytest.mark.parametrize("H,I,Ish,off", [(768, 256, 512, 0), (512, 512, 512, 0), (512, 512, 512, 1)])
def test_mix_auto_matches_per_token(mix, T, H, I, Ish, off):
    s = api.shape(hidden=H, expert_inter=I, shared_inter=Ish, n_experts=24, top_k=4)
    t = api.synth_layer_tensors(s, seed=77, layer=0, types=mix)
    gen = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, H, device=DEV, generator=gen)
    got = []
    for path in (api.PATH_AUTO, api.PATH_PER_TOKEN):
        h = torch.zeros(T * H + 4, device=DEV)[off:off + T * H].view(T, H)
        got.append(run(s, t.desc(), x, h, path))
    for a, b in zip(got[0][1:], got[1][1:]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert rel_l2(got[0][0], got[1][0]) < 4e-6
