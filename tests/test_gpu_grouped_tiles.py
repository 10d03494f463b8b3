"""Edges of the grouped GEMMs' tiles (moe_grouped.hip) against the CPU oracle:
identical tokens, so every chosen expert and the shared one take T pairs, at
counts around the 32-pair tile; hidden sizes that end inside a 512-row chunk
of the down kernel; one superblock and two of intermediate size, the shared
expert's equal to the routed one's (one launch) or not (two).

Bound: the Q6_K down weights are fp16 roundings of integers up to 4096, off
by at most 1 above 2048, 2^-12 of the weight; everything else is exact or has
22 bits.  Roundings of one row have random signs, so the relative L2 error of
a token's output stays below twice that, 2^-11.
"""
import numpy as np
import pytest
import torch

import breadv2_amd as B
from breadv2_amd import api
from oracle import oracle as O

from helpers import host_layer, rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T", [1, 31, 32, 33, 65])
@pytest.mark.parametrize("H,I,Ish", [(256, 256, 256), (768, 512, 512), (1280, 256, 512)])
def test_grouped_tile_edges(H, I, Ish, T):
    s = api.shape(hidden=H, expert_inter=I, shared_inter=Ish, n_experts=12, top_k=3)
    t = api.synth_layer_tensors(s, seed=31 + H, layer=0)
    torch.cuda.synchronize()
    hl = host_layer(t)
    x = np.repeat(np.random.default_rng(H + T).standard_normal((1, H)).astype(np.float32), T, axis=0)
    ctx = B.MoeContext(s, max_tokens=T)
    ctx.set_path(api.PATH_GROUPED)
    hd = torch.zeros(T, H, device=DEV)
    idx, _, _ = ctx.forward(t.desc(), torch.from_numpy(x).to(DEV), hd, T, want_routing=True)
    torch.cuda.synchronize()
    assert ctx.check_device() == 0
    ref = np.zeros_like(x)
    ridx, _, _ = O.moe_forward(hl, x, ref, T, nthreads=16)
    assert np.array_equal(idx.cpu().numpy(), np.asarray(ridx).reshape(T, -1))
    got = hd.cpu().numpy()
    assert np.array_equal(got.view(np.uint32), np.repeat(got[:1], T, axis=0).view(np.uint32))
    assert rel_l2(got, ref) < 2.0 ** -11


def test_context_memory_per_token():
    """What a context of the benchmark's shape takes for each token: the fp32
    residual, input and logits, activations in operand order, SwiGLU rows and
    expert outputs of nine pairs come to 115.5 KB; 4 KB more for
    2 MB pages over 8192 tokens."""
    s = api.shape()

    def taken(tokens):
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        ctx = B.MoeContext(s, max_tokens=tokens)
        n = free - torch.cuda.mem_get_info()[0]
        ctx.close()
        return n

    assert (taken(12288) - taken(4096)) / 8192 < 120 * 1024
