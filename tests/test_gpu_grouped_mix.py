"""Layers of other mixes of Q4_K and Q6_K than the decode kernel's under the
automatic choice, around the token counts where it moves from the per-token
kernels to the grouped path (moe.hip, grouped_takes_mix): all Q4_K, all Q6_K and
each tensor Q6_K by itself, layers of the size of the reference's and small
ones, and where the grouped path does not take the call (the residual or Q6_K
down weights 4-byte aligned only).

Which path ran shows in the bits: the two sum in different orders, so thousands
of outputs never agree in all of them, and either path repeats itself exactly.

With weights exact and activations of 23 bits they agree as two fp32 sums of
256 and 512 products do: 512 roundings of 2^-24 at most, about sqrt(512) of them
in effect on each side, 4e-6 together with the gate/up sums.
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
SHAPES = [(768, 256, 512, 24, 4), (512, 512, 512, 24, 4), (512, 256, 256, 12, 2), (2048, 512, 512, 16, 8)]


def first_grouped(mix, shape):
    """Tokens from which the grouped path takes a layer."""
    _, I, Ish, _, K = shape
    gu_q4, dn_q4 = {mix[0], mix[1], mix[3], mix[4]} == {Q4}, {mix[2], mix[5]} == {Q4}
    tokens, rows = (6, 15000) if gu_q4 and dn_q4 else (14, 24000) if gu_q4 else (16, 29000)
    return max(tokens, -(-rows // (K * I + Ish)))


def run(s, d, x, hidden, path):
    T = x.shape[0]
    ctx = B.MoeContext(s, max_tokens=T)
    ctx.set_path(path)
    idx, w, g = ctx.forward(d, x, hidden, T, want_routing=True)
    torch.cuda.synchronize()
    assert ctx.check_device() == 0
    return hidden.cpu().numpy(), idx.cpu().numpy(), w.cpu().numpy(), g.cpu().numpy()


def same_bits(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


def auto_and_per_token(s, d, T, off=0):
    gen = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, s.hidden, device=DEV, generator=gen)
    got = []
    for path in (api.PATH_AUTO, api.PATH_PER_TOKEN):
        h = torch.zeros(T * s.hidden + 4, device=DEV)[off:off + T * s.hidden].view(T, s.hidden)
        got.append(run(s, d, x, h, path))
    for a, b in zip(got[0][1:], got[1][1:]):
        assert same_bits(a, b)
    assert rel_l2(got[0][0], got[1][0]) < 4e-6
    return same_bits(got[0][0], got[1][0])


@pytest.mark.parametrize("mix", MIXES)
@pytest.mark.parametrize("shape", SHAPES)
def test_mix_auto_matches_per_token(mix, shape):
    s = api.shape(*shape)
    d = api.synth_layer_tensors(s, seed=77, layer=0, types=mix)
    first = first_grouped(mix, shape)
    for T in (5, first - 1, first, 33, 70):
        assert auto_and_per_token(s, d.desc(), T) == (T < first)
    assert auto_and_per_token(s, d.desc(), 70, off=1)  # the residual not 16-byte aligned


@pytest.mark.parametrize("which", ["routed", "stride", "shared"])
def test_q6k_down_aligned_to_4_bytes(which):
    """The down kernel loads 16-byte pieces: such layers stay per token."""
    s = api.shape(512, 256, 256, 12, 4)
    t = api.synth_layer_tensors(s, seed=78, layer=0, types=(Q4, Q4, Q6, Q4, Q6, Q6))
    d = t.desc()
    assert not auto_and_per_token(s, d, 70)
    one = d.down_expert_bytes
    if which == "stride":
        down = torch.zeros(s.n_experts * (one + 4), dtype=torch.uint8, device=DEV).view(s.n_experts, -1)
        down[:, :one] = t.down_exps.view(s.n_experts, -1)
        d.down_exps, d.down_expert_bytes = down.data_ptr(), one + 4
    else:
        src = t.down_exps if which == "routed" else t.down_sh
        down = torch.zeros(src.numel() + 16, dtype=torch.uint8, device=DEV)
        down[4:4 + src.numel()] = src
        setattr(d, "down_exps" if which == "routed" else "down_shexp", down.data_ptr() + 4)
    assert auto_and_per_token(s, d, 70)
