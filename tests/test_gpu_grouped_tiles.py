"""Edges of the grouped path (moe_grouped.hip): its GEMMs' tiles, its bucketing
and its workspace.  The tiles against the CPU oracle: identical tokens, so every
chosen expert and the shared one take T pairs, at counts around the 32-pair
tile; hidden sizes that end inside a 512-row chunk of the down kernel; one
superblock and two of intermediate size, the shared expert's equal to the
routed one's (one launch) or not (two).

Bound: the Q6_K down weights are integers up to 4096 rounded to fp16, off by 1
where they are odd and above 2048, so by less than 2^-11 of a weight and by
nothing below; everything else is exact or has 22 bits.  An output's products
have random signs, as their roundings have, so errors of less than 2^-11 of
every product leave a token's output less than 2^-11 off in relative L2.
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


@pytest.mark.parametrize("T,E", [(2048, 24), (2049, 24), (2050, 1000), (4100, 12)])
def test_bucketing_passes(T, E):
    """16,384 pairs are what the bucketing keeps in registers; more of them take
    a second and a third pass, here with ends inside a pass and inside its 1,024
    threads.  A pair in the wrong place gives its token another expert's output.
    Same bound as above."""
    s = api.shape(hidden=256, expert_inter=256, shared_inter=256, n_experts=E, top_k=8)
    t = api.synth_layer_tensors(s, seed=9, layer=0)
    x = torch.randn(T, 256, device=DEV, generator=torch.Generator(device=DEV).manual_seed(T))
    out = []
    for path in (api.PATH_GROUPED, api.PATH_PER_TOKEN):
        ctx = B.MoeContext(s, max_tokens=T)
        ctx.set_path(path)
        hd = torch.zeros(T, 256, device=DEV)
        idx, w, _ = ctx.forward(t.desc(), x, hd, T, want_routing=True)
        torch.cuda.synchronize()
        assert ctx.check_device() == 0
        out.append([v.cpu().numpy() for v in (hd, idx, w)])
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    err = np.linalg.norm(out[0][0] - out[1][0], axis=1) / np.linalg.norm(out[1][0], axis=1)
    assert err.max() < 2.0 ** -11


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
