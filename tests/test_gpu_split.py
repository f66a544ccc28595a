"""Gate/up and down of batches with few pairs, each expert spread over many workgroups (csrc/split.h), against k_group and
the three separate kernels, bit for bit in every intermediate and in x, at the sizes where the dispatch changes: two and
three tokens (the decode down kernel), 24 / 48 pairs (columns over 4, 2 or 1 waves), 256 pairs (the last batch whose pairs
find their own tiles) and the one above it; 240 to 359 tokens (tiles of 16 with the grouping of k_group) and the one above;
host groupings of 1 to 193 tiles (192 is the last on the split kernels below 257) and of 257.
The Zipf bias gives experts of more than 16 pairs, so further tiles of one expert occur."""
import numpy as np
import pytest

import maplemoe as M
from helpers import SEED, HostLayer, normed_hidden

pytestmark = pytest.mark.gpu
L = 30


@pytest.fixture(scope="module")
def layer():
    lib = M.lib()
    M.check(lib.mmoe_init(2048), "mmoe_init")
    hl = HostLayer(SEED, L)
    M.register_layer(L, hl.blk, hl.router)
    hl.bias = M.zipf_bias(SEED, 1.1)
    yield hl
    M.check(lib.mmoe_set_bias(L, None), "bias off")


ITEMS = (("GU_I32", 1024, np.int32), ("ACT", 512, np.float32), ("QA", 512, np.int8), ("QSA", 1, np.float32), ("QSUMA", 1, np.int32),
         ("DN_I32", 2048, np.int32), ("DOWN", 2048, np.float32), ("UTOK", 1, np.int32), ("UW", 1, np.float32), ("TP", 1, np.int32),
         ("SP", 1, np.int32))


@pytest.mark.parametrize("zipf", [0, 1])
@pytest.mark.parametrize("nb,order", [(2, 0), (3, 0), (3, 1), (4, 0), (6, 0), (7, 0), (20, 1), (31, 0), (32, 0), (33, 0), (239, 0), (240, 0), (359, 0), (360, 0)])
def test_split_matches_three_kernels(layer, nb, order, zipf):
    lib = M.lib()
    M.check(lib.mmoe_set_bias(L, M.ptr(layer.bias) if zipf else None), "bias")
    x, hn = normed_hidden(SEED, 5200 + nb, nb)
    out = {}
    M.check(lib.mmoe_set_debug(1), "debug on")
    try:
        for fused in (0, 1):
            M.check(lib.mmoe_set_expert_path(fused), "expert path"); M.check(lib.mmoe_set_decode_path(fused), "decode path")
            xg = x.copy()
            M.check(lib.mmoe_moe(L, M.ptr(hn), nb, M.ptr(xg), order), "mmoe_moe")
            plan = M.read_plan()
            out[fused] = [xg] + [M.read(n, (nb * 8, k), t) for n, k, t in ITEMS] + [plan["ue"], plan["ustart"], np.array([plan["nu"], plan["np"]])]
        if zipf and nb >= 20:
            assert np.diff(out[1][-2]).max() > 16
        for name, a, b in zip(["x"] + [i[0] for i in ITEMS] + ["ue", "ustart", "nu np"], out[0], out[1]):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), f"{name} differs"
    finally:
        M.check(lib.mmoe_set_debug(0), "debug off")
        M.check(lib.mmoe_set_expert_path(1), "expert path"); M.check(lib.mmoe_set_decode_path(1), "decode path")


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("nb", [2, 3, 8, 32])
def test_split_infinite_inputs(layer, nb, order):
    """tokens with infinite values beside ordinary ones: every token's x as from a call of its own (the one-token decode
    kernels), bit for bit"""
    lib = M.lib()
    M.check(lib.mmoe_set_bias(L, None), "bias")
    x, hn = normed_hidden(SEED, 5250 + nb, nb)
    hn[0] = np.inf
    hn[nb // 2, 100] = -np.inf
    hn[-1, 2047] = np.inf
    xg = x.copy()
    M.check(lib.mmoe_moe(L, M.ptr(hn), nb, M.ptr(xg), order), "mmoe_moe")
    for b in range(nb):
        h, want = hn[b:b + 1].copy(), x[b:b + 1].copy()
        M.check(lib.mmoe_moe(L, M.ptr(h), 1, M.ptr(want), order), "mmoe_moe")
        assert ((xg[b].view(np.int32) == want[0].view(np.int32)) | (np.isnan(xg[b]) & np.isnan(want[0]))).all(), b


@pytest.fixture(scope="module")
def slots(layer):
    lib = M.lib()
    M.check(lib.gpux_init(1, 256), "gpux_init")
    for s in range(256):
        lib.gpux_upload(0, s, *[M.ptr(a) for a in M.expert_views(layer.blk, s)])


@pytest.mark.parametrize("sizes", [[1], [1] * 24, [17] + [1] * 23, [2] * 48, [17] + [2] * 47, [1] * 192, [17, 16] + [1] * 190, [17] + [1] * 255])
def test_split_host_grouping(slots, sizes):
    """runs of the given lengths (17 pairs are two tiles) over 40 tokens through gpux_begin_multi"""
    lib = M.lib()
    nu, np_, nb = len(sizes), sum(sizes), 40
    _, hn = normed_hidden(SEED, 5300, nb)
    rng = np.random.default_rng(nu)
    sl = rng.permutation(256)[:nu].astype(np.int32)
    ps = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    pt = np.concatenate([np.sort(rng.permutation(nb)[:k]) for k in sizes]).astype(np.int32)
    out = {}
    try:
        for fused in (0, 1):
            M.check(lib.mmoe_set_expert_path(fused), "expert path")
            h = lib.gpux_begin_multi(0, M.ptr(hn), nb, nu, M.ptr(sl), M.ptr(ps), M.ptr(pt))
            assert h, lib.mmoe_last_error()
            out[fused] = np.full((np_, 2048), np.nan, np.float32)
            lib.gpux_end_multi(h, M.ptr(out[fused]), np_)
    finally:
        M.check(lib.mmoe_set_expert_path(1), "expert path")
    assert np.isfinite(out[0]).all() and np.array_equal(out[0].view(np.int32), out[1].view(np.int32))
