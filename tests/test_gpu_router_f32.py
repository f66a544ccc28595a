"""The batch router on the f32 matrix cores (k_router_f32), which takes over at 240 tokens (384 in a stack), against the
oracle's chains and against the chain router on the same tokens in smaller calls, bit for bit: the first sizes on either
side of the switches, ragged token tiles of 16, and with exact logits asked for the sizes past 511 up to the largest. And
the approximate router with its refinement, the default from 512 tokens: one token's results in batches of different sizes, and
logits that decide the top 8 by ties."""
import numpy as np
import pytest

import maplemoe as M
import pyoracle as O
from helpers import SEED, HostLayer, normed_hidden

pytestmark = pytest.mark.gpu
L = 31


@pytest.fixture(scope="module")
def layer():
    lib = M.lib()
    M.check(lib.mmoe_init(2048), "mmoe_init")
    hl = HostLayer(SEED, L)
    M.register_layer(L, hl.blk, hl.router)
    hl.bias = M.zipf_bias(SEED, 1.1)
    yield hl
    M.check(lib.mmoe_set_bias(L, None), "bias off")


def logits(hn):
    lib = M.lib()
    nb = len(hn)
    x = np.zeros((nb, M.H), np.float32)
    M.check(lib.mmoe_moe(L, M.ptr(hn), nb, M.ptr(x), M.ORDER_BATCH), "mmoe_moe")
    return M.read("LOGITS", (nb, 256), np.float32), M.read("TOP", (nb, 8), np.int32), x


@pytest.mark.parametrize("nb,zipf", [(239, 0), (240, 0), (241, 1), (255, 0), (257, 1), (383, 0), (511, 1), (513, 0), (1023, 1), (1024, 0), (2033, 0), (2048, 1)])
def test_router_f32_matches_chains(layer, nb, zipf):
    lib = M.lib()
    M.check(lib.mmoe_set_bias(L, M.ptr(layer.bias) if zipf else None), "bias")
    _, hn = normed_hidden(SEED, 5400 + nb, nb)
    # magnitudes from subnormal products to 2^40, and exact zeros
    hn *= np.exp2(np.random.default_rng(nb).integers(-130, 40, size=(nb, 1))).astype(np.float32)
    hn[nb // 2] = 0
    hn = np.ascontiguousarray(hn)
    M.check(lib.mmoe_set_router_mode(int(nb >= 512)), "router mode")
    try:
        rl, top, x = logits(hn)
        parts = [logits(np.ascontiguousarray(hn[i:i + 239])) for i in range(0, nb, 239)]
    finally:
        M.check(lib.mmoe_set_router_mode(0), "router mode")
    assert np.array_equal(rl.view(np.int32), np.concatenate([p[0] for p in parts]).view(np.int32))
    assert np.array_equal(top, np.concatenate([p[1] for p in parts]))
    assert np.array_equal(x.view(np.int32), np.concatenate([p[2] for p in parts]).view(np.int32))
    for b in (0, nb // 2, nb - 1):
        want = O.router_batch(hn[b:b + 1], layer.router, layer.bias if zipf else None)
        assert np.array_equal(rl[b:b + 1].view(np.int32), want.view(np.int32)), b


@pytest.mark.parametrize("nb", [512, 700, 1023])
def test_default_router_same_at_every_size(layer, nb):
    """the default router from 512 tokens on gives a token the same logits and x whatever the size of its batch: the first
    tokens of a batch of 1100, bit for bit (512 to 1023 tokens run blocks of 128 experts, from 1024 blocks of all 256)"""
    lib = M.lib()
    M.check(lib.mmoe_set_bias(L, M.ptr(layer.bias)), "bias")
    _, hn = normed_hidden(SEED, 5650, 1100)
    want = logits(hn)
    got = logits(np.ascontiguousarray(hn[:nb]))
    for a, b in zip(got, want):
        assert np.array_equal(a.view(np.int32), b[:nb].view(np.int32))


@pytest.mark.parametrize("nb", [383, 384])
def test_stack_switch(layer, nb):
    """a stack of one layer (rmsnorm in the router launch below 384 tokens) = rmsnorm and the layer call"""
    lib = M.lib()
    M.check(lib.mmoe_set_bias(L, None), "bias")
    x0 = M.synth_hidden(SEED, 5500 + nb, nb)
    d = [lib.mmoe_dev_alloc(x0.nbytes) for _ in range(3)]
    try:
        for p in d[:2]:
            M.check(lib.mmoe_h2d(p, M.ptr(x0), x0.nbytes), "h2d")
        M.check(lib.mmoe_stack_dev(L, 1, d[0], nb, M.ORDER_BATCH), "stack")
        M.check(lib.mmoe_rmsnorm_dev(d[1], None, nb, d[2]), "rmsnorm")
        M.check(lib.mmoe_moe_dev(L, d[2], nb, d[1], M.ORDER_BATCH), "layer")
        out = [np.empty_like(x0) for _ in range(2)]
        for o, p in zip(out, d):
            M.check(lib.mmoe_d2h(M.ptr(o), p, x0.nbytes), "d2h")
        assert not np.array_equal(out[0], x0) and np.array_equal(out[0], out[1])
    finally:
        for p in d:
            lib.mmoe_dev_free(p)


@pytest.mark.parametrize("nb", [1023, 1024, 1100])
@pytest.mark.parametrize("kind", ["ties", "large"])
def test_top8_of_close_logits(layer, nb, kind):
    """default against exact logits: a bias of 2^18 plus the Zipf values (many experts within a few ulp of the 8th place) and
    inputs of zero with 253 equal biases (every one a candidate): same top-8 (lowest index first), picked logits and x"""
    lib = M.lib()
    _, hn = normed_hidden(SEED, 5600 + nb, nb)
    if kind == "ties":
        hn[::2] = 0
        bias = np.full(256, 0.5, np.float32); bias[[250, 3, 180]] = (3.0, 2.0, 1.0)
    else:
        bias = (np.float32(262144.0) + layer.bias).astype(np.float32)
    M.check(lib.mmoe_set_bias(L, M.ptr(bias)), "bias")
    out = {}
    try:
        for mode in (1, 0):
            M.check(lib.mmoe_set_router_mode(mode), "router mode")
            out[mode] = logits(hn)
    finally:
        M.check(lib.mmoe_set_router_mode(0), "router mode")
    (r1, t1, x1), (r0, t0, x0) = out[1], out[0]
    assert np.array_equal(t0, t1)
    if kind == "ties":
        assert (t0[::2] == np.array([250, 3, 180, 0, 1, 2, 4, 5])).all()
    assert np.array_equal(np.take_along_axis(r0, t0, 1).view(np.int32), np.take_along_axis(r1, t1, 1).view(np.int32))
    assert np.abs(x0 - x1).max() <= 1e-5 * np.abs(x1).max()   # the other logits reach x through the softmax sum alone


@pytest.mark.parametrize("nb,rc", [(511, 0), (512, -1), (1023, -1)])
def test_route_of_device_logits(layer, nb, rc):
    """mmoe_route without logits: taken below 512 tokens, from there on only with exact logits asked for"""
    lib = M.lib()
    M.check(lib.mmoe_set_bias(L, None), "bias")
    _, hn = normed_hidden(SEED, 5700, nb)
    logits(hn)
    top = np.empty((nb, 8), np.int32); none = [None] * 6
    got = lib.mmoe_route(None, nb, M.ptr(top), *none)
    assert (got == -1) if rc else (got > 0)
