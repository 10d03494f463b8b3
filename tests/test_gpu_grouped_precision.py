"""What the grouped path keeps of fp32, on layers whose products can be followed
exactly: gate and up rows with one weight in a column each, and down matrices
that pick one SwiGLU value per output row.  Then g, u and the pick are exact
and an output shows the SwiGLU and the split of its value into fp16 terms.

The per-token kernels give the value itself for the same gate and up tensors
with a Q4_K down matrix (a scale of 1, integers 0 and 1, no min: every product
and sum is exact), which makes them the reference here.
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
H = I = 256
E, K = 3, 1


def q4k_block(d, scale, col, q):
    """One superblock without mins: d * scale * q in column col, zero elsewhere."""
    b = np.zeros(144, np.uint8)
    b[0:2] = np.frombuffer(np.float16(d).tobytes(), np.uint8)
    j = col // 32
    if j < 4:
        b[4 + j] = scale
    else:
        b[4 + j + 4] = scale & 15
        b[4 + j - 4] |= (scale >> 4) << 6
    b[16 + 32 * (col // 64) + col % 32] = q << (4 if col % 64 >= 32 else 0)
    return b


def q6k_block(d, scale, col, q):
    """One superblock: d * scale * (q - 32) in column col, zero elsewhere."""
    v = np.full(256, 32, np.int32)
    v[col] = q
    b = np.zeros(210, np.uint8)
    for half in range(2):
        w = v[128 * half:128 * half + 128].reshape(4, 32)
        b[64 * half:64 * half + 32] = (w[0] & 15) | ((w[2] & 15) << 4)
        b[64 * half + 32:64 * half + 64] = (w[1] & 15) | ((w[3] & 15) << 4)
        b[128 + 32 * half:160 + 32 * half] = (w[0] >> 4) | ((w[1] >> 4) << 2) | ((w[2] >> 4) << 4) | ((w[3] >> 4) << 6)
    b[192:208] = np.full(16, scale, np.int8).view(np.uint8)
    b[208:210] = np.frombuffer(np.float16(d).tobytes(), np.uint8)
    return b


def gate_up():
    """Row r: gate d * scale * q in column 0, 1 to 945 of 2^-5; up 1 in column 64."""
    n = np.unique(np.outer(np.arange(1, 64), np.arange(1, 16)))
    n = n[np.linspace(0, n.size - 1, I).astype(int)]
    pairs = [next((v // q, q) for q in range(15, 0, -1) if v % q == 0 and v // q < 64) for v in n]
    return (np.concatenate([q4k_block(2.0 ** -5, s, 0, q) for s, q in pairs]),
            np.concatenate([q4k_block(1.0, 1, 64, 1) for _ in range(I)]))


def layer(down, down_shared):
    """Every expert the same; the shared one's down matrix is zero."""
    gate, up = gate_up()
    rows = {Q4: lambda s, q: np.concatenate([q4k_block(1.0, s, r, q) for r in range(H)]),
            Q6: lambda s, q: np.concatenate([q6k_block(1.0, s, r, 32 + q) for r in range(H)])}
    typ, scale, q = down

    def dev(a, n=1):
        return torch.from_numpy(np.tile(a, n)).to(DEV)

    return api.LayerTensors(api.shape(H, I, I, E, K), dev(gate, E), dev(up, E), dev(rows[typ](scale, q), E),
                            dev(gate), dev(up), dev(rows[down_shared](0, 0)), torch.zeros(E * H, device=DEV), None,
                            (Q4, Q4, typ, Q4, Q4, down_shared))


def inputs(T):
    """13 bits in columns 0 and 64, so that every g (from -29 to 29) and u is exact."""
    x = np.zeros((T, H), np.float32)
    g = np.random.default_rng(T)
    x[:, 0] = np.round(g.uniform(-4096, 4096, T)) / 4096
    x[:, 64] = np.round(g.uniform(4096, 8191, T)) / 4096
    return torch.from_numpy(x).to(DEV)


def run(t, x, path):
    T = x.shape[0]
    ctx = B.MoeContext(t.shape, max_tokens=T)
    ctx.set_path(path)
    hd = torch.zeros_like(x)
    ctx.forward(t.desc(), x, hd, T)
    torch.cuda.synchronize()
    assert ctx.check_device() == 0
    return hd.cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("T", [50, 130])
@pytest.mark.parametrize("down_shared,path,tail", [(Q6, api.PATH_GROUPED, 2.0 ** -38), (Q4, api.PATH_AUTO, 2.0 ** -48)])
def test_swiglu_is_the_per_token_kernels(T, down_shared, path, tail):
    """An output is its SwiGLU value in two fp16 terms: off by at most 2^-23 of
    itself (11 bits and 11 bits of the signed rest: half a unit of the second
    term is 2^-23), or by what fp16's smallest number, 2^-24, leaves of a row
    scaled to 2^13: half of it, and with the second term held times 2^10 (the
    layers of other type mixes) a 2^-10th of that."""
    x = inputs(T)
    ref = run(layer((Q4, 1, 1), Q4), x, api.PATH_PER_TOKEN)
    got = run(layer((Q6, 1, 1), down_shared), x, path)
    bound = 2.0 ** -23 * np.abs(ref) + tail * np.abs(ref).max(1, keepdims=True)
    assert np.count_nonzero(ref) == ref.size
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("T", [50, 130])
def test_q6k_weight_of_12_bits(T):
    """A Q6_K weight of 127 * 31 = 3937, which fp16 rounds to an even integer,
    in a layer of another type mix: the rest meets both terms of the SwiGLU
    value, so what is off is the split (as above) and the rounding of the
    terms' sum, 2^-24."""
    x = inputs(T)
    ref = 3937.0 * run(layer((Q4, 1, 1), Q4), x, api.PATH_PER_TOKEN)
    got = run(layer((Q6, 127, 31), Q4), x, api.PATH_AUTO)
    bound = (2.0 ** -23 + 2.0 ** -24) * np.abs(ref) + 2.0 ** -48 * np.abs(ref).max(1, keepdims=True)
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("typ", [Q4, Q6])
@pytest.mark.parametrize("outlier", [1e3, 1e5, 1e7])
def test_rows_with_an_outlier(typ, outlier):
    """A channel far above the others that no gate, up or router row weighs
    changes nothing but the row's scale, so the layer's output may move by the
    splits of two operands, 2^-23 of a product each."""
    H, T = 512, 50
    s = api.shape(hidden=H, expert_inter=256, shared_inter=256, n_experts=12, top_k=3)
    t = api.synth_layer_tensors(s, seed=5, layer=0, types=(typ,) * 6)
    for name in ("gate_exps", "up_exps", "gate_sh", "up_sh"):  # columns 0..31 of each row
        b = getattr(t, name).view(-1, H // 256, 144 if typ == Q4 else 210)
        if typ == Q4:
            b[:, 0, 4] &= 0xC0
            b[:, 0, 8] &= 0xC0
        else:
            b[:, 0, 192:194] = 0
    t.router.view(-1, H)[:, 0:32] = 0
    t.shgate[0:32] = 0
    x = torch.randn(T, H, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    out = []
    for v, path in ((0.0, api.PATH_AUTO), (outlier, api.PATH_AUTO), (outlier, api.PATH_PER_TOKEN)):
        x[:, 5] = v
        out.append(run(t, x, path))
    assert not np.array_equal(out[1], out[2])  # another path
    assert rel_l2(out[1], out[0]) <= 2.0 ** -22
