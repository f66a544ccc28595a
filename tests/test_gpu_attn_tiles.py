"""gfull_attn at the edges of its row tiles (4 tokens) and position blocks (16), against the oracle, bit for bit: chunks of 1 to
33 tokens whose first and last positions fall on, before and after a block, windows just inside and just past the 576
positions that one workgroup holds on chip (k_att_local; longer ones take the separate kernels), the window's own start
inside a block, and a context length that is no multiple of 16. Positions before the chunk are zero on both sides."""
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
