"""gfull_attn at the edges of its row tiles (4 tokens) and position blocks (16), against the oracle, bit for bit: chunks of 1 to
33 tokens whose first and last positions fall on, before and after a block, windows just inside and just past the 576
positions that one workgroup holds on chip (k_att_local; longer ones take the separate kernels), the window's own start
inside a block, and a context length that is no multiple of 16. Positions before the chunk are zero on both sides, except
where an earlier chunk is part of the case."""
import ctypes as C

import numpy as np
import pytest

import maplemoe as M
import pyoracle as O
from helpers import SEED
from test_gpu_attn import LAYERS, gfull_model  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu
H, CTX = 2048, 1003


@pytest.mark.parametrize("nb,pos0", [(1, 0), (3, 14), (4, 16), (5, 13), (33, 500), (5, 555), (2, 558), (3, 558), (6, 571), (13, 990)])
def test_attn_tiles(gfull_model, nb, pos0):  # noqa: F811
    lib, layers, _, _, _, norms, router_all = gfull_model
    cs = O.rope_table(CTX)
    M.check(lib.gfull_init(CTX, 64, O.WIN, M.ptr(norms), M.ptr(router_all), M.ptr(cs)), "gfull_init")
    x0 = np.random.default_rng(SEED + 60 + pos0 + nb).standard_normal((nb, H)).astype(np.float32)
    lib.gfull_begin(M.ptr(x0), nb, pos0)
    for L, glob in LAYERS:
        lib.gfull_write_x(M.ptr(x0))
        assert lib.gfull_attn(L, glob, None) >= 0, lib.mmoe_last_error()
        x = np.empty((nb, H), np.float32)
        kop = C.c_void_p()
        lib.gfull_read(M.ptr(x), C.addressof(kop))
        ko = np.ctypeslib.as_array((C.c_uint16 * (24 * 64 * 1024)).from_address(kop.value)).reshape(24, 64, 1024)[L, :nb]
        kc = np.zeros((CTX, 512), np.uint16); vc = np.zeros((CTX, 512), np.uint16)
        xo, ko_o, _ = O.attn_chunk(layers[L % 2], x0, pos0, glob, kc, vc, cs)
        assert np.array_equal(ko, ko_o), f"layer {L}: k/v"
        assert np.array_equal(x.view(np.uint32), xo.view(np.uint32)), f"layer {L}: x"


@pytest.mark.parametrize("win,nb,lo", [(600, 5, 16), (600, 9, 15), (600, 4, 17), (600, 33, 3), (777, 6, 30), (557, 13, 31)])
def test_attn_window_start(gfull_model, win, nb, lo):  # noqa: F811
    """local layers whose windows are too long for one workgroup (from 557 positions on; 39 to 50 blocks over several
    workgroups): the first token's window starts at position lo, at, before and inside a block of 16, among the 24 positions
    of an earlier chunk"""
    lib, layers, _, _, _, norms, router_all = gfull_model
    cs, L = O.rope_table(CTX), 0
    M.check(lib.gfull_init(CTX, 64, win, M.ptr(norms), M.ptr(router_all), M.ptr(cs)), "gfull_init")
    rng = np.random.default_rng(SEED + 65 + win + nb)
    kc = np.zeros((CTX, 512), np.uint16); vc = np.zeros((CTX, 512), np.uint16)
    for pos0, n in ((max(lo - 10, 0), 24), (lo + win, nb)):
        x0 = rng.standard_normal((n, H)).astype(np.float32)
        lib.gfull_begin(M.ptr(x0), n, pos0)
        assert lib.gfull_attn(L, 0, None) >= 0, lib.mmoe_last_error()
        x = np.empty((n, H), np.float32)
        lib.gfull_read(M.ptr(x), None)
        xo, _, _ = O.attn_chunk(layers[L % 2], x0, pos0, 0, kc, vc, cs, win)
        assert np.array_equal(x.view(np.uint32), xo.view(np.uint32)), f"chunk at {pos0}"


@pytest.mark.parametrize("win,chunks", [(512, [(0, 8, 3)]), (512, [(600, 9, 2)]), (512, [(0, 8, 3), (512, 10, 7)]), (600, [(0, 7, 2), (601, 9, 5)])])
def test_values_past_fp16(gfull_model, win, chunks):  # noqa: F811
    """one token of a chunk (pos0, nb, token) has values past fp16's range, which the cache holds as infinities: the tokens that
    do not see it, in its row tile before it and after it left the window, are the oracle's bit for bit; those that see it
    come out as in the oracle (NaN). Both attention paths: one workgroup, and the separate kernels (global layers from 576
    positions on; a window of 600)"""
    lib, layers, _, _, _, norms, router_all = gfull_model
    cs, c = O.rope_table(CTX), 77
    norms, ln = norms.copy(), [al.in_ln.copy() for al in layers]
    big = np.float32(2.0 ** 24)                       # norm weight of a column that only the token's hidden state has
    norms[:, c] = big
    rng = np.random.default_rng(SEED + 70 + win)
    try:
        for al in layers:
            al.in_ln[c] = big.view(np.uint32) >> 16
        M.check(lib.gfull_init(CTX, 64, win, M.ptr(norms), M.ptr(router_all), M.ptr(cs)), "gfull_init")
        cache = {L: (np.zeros((CTX, 512), np.uint16), np.zeros((CTX, 512), np.uint16)) for L, _ in LAYERS}
        for pos0, nb, bad in chunks:
            x0 = rng.standard_normal((nb, H)).astype(np.float32)
            x0[:, c] = 0
            x0[bad, c] = 1
            lib.gfull_begin(M.ptr(x0), nb, pos0)
            for L, glob in LAYERS:
                lib.gfull_write_x(M.ptr(x0))
                assert lib.gfull_attn(L, glob, None) >= 0, lib.mmoe_last_error()
                x = np.empty((nb, H), np.float32)
                lib.gfull_read(M.ptr(x), None)
                xo, _, att = O.attn_chunk(layers[L % 2], x0, pos0, glob, *cache[L], cs, win)
                assert not np.isfinite(att[bad]).all()
                for b in range(nb):
                    same = (x[b].view(np.uint32) == xo[b].view(np.uint32)) | (np.isnan(x[b]) & np.isnan(xo[b]))
                    assert same.all(), f"pos0 {pos0} layer {L} token {b}: {int((~same).sum())} values differ"
    finally:
        for al, a in zip(layers, ln):
            al.in_ln[:] = a


@pytest.mark.parametrize("win,nb", [(512, 5), (600, 590)])
def test_scores_all_negative_infinity(gfull_model, win, nb):  # noqa: F811
    """keys with a dim past fp16's range: every score is infinite, and where all the scores a token sees are -inf its softmax
    sum is 0 (the positions of its tile that it does not see add nothing), so the attention output is the oracle's NaN,
    which the o projection's quantisation takes as 0. Both attention paths"""
    lib, layers, _, _, _, norms, router_all = gfull_model
    cs, c = O.rope_table(CTX), 100                    # past the dims that rope mixes
    norms, kn = norms.copy(), [al.k_norm.copy() for al in layers]
    big = np.float32(2.0 ** 60)
    norms[:, 4224 + c] = big
    x0 = np.random.default_rng(SEED + 75 + nb).standard_normal((nb, H)).astype(np.float32)
    try:
        for al in layers:
            al.k_norm[c] = big.view(np.uint32) >> 16
        M.check(lib.gfull_init(CTX, 640, win, M.ptr(norms), M.ptr(router_all), M.ptr(cs)), "gfull_init")
        lib.gfull_begin(M.ptr(x0), nb, 0)
        for L, glob in LAYERS:
            lib.gfull_write_x(M.ptr(x0))
            assert lib.gfull_attn(L, glob, None) >= 0, lib.mmoe_last_error()
            x = np.empty((nb, H), np.float32)
            lib.gfull_read(M.ptr(x), None)
            kc = np.zeros((CTX, 512), np.uint16); vc = np.zeros((CTX, 512), np.uint16)
            xo, _, att = O.attn_chunk(layers[L % 2], x0, 0, glob, kc, vc, cs, win)
            assert np.isnan(att[0]).all()
            bad = np.flatnonzero((x.view(np.uint32) != xo.view(np.uint32)).any(1))
            assert len(bad) == 0, f"layer {L}: tokens {bad[:8]}"
    finally:
        for al, a in zip(layers, kn):
            al.k_norm[:] = a
