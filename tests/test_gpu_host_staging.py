"""Host data through the library's pinned blocks: gfull_moe calls queued one after the other (more than the ring of table
blocks holds) against the same calls with a wait after each; and the keys and values that gfull_read hands out when
mmoe_gfull_stack has copied them beside its work, against the ones gfull_read copies itself, over two chunks of
different size, a chunk whose copies nobody read, a repeated stack and a partial one, the ones of a chunk left where they
were handed out while the next chunk runs, and a stack and a gpux call that their caller captures and replays."""
import ctypes as C

import numpy as np
import pytest

import maplemoe as M
import pyoracle as O
from helpers import SEED, HostLayer
from test_gpu_attn import CTX, MAXTOK, gfull_model  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu
H, NL = 2048, 4


@pytest.fixture(scope="module")
def model(gfull_model):  # noqa: F811
    lib, _, post, routers, cs, norms, router_all = gfull_model
    M.check(lib.gfull_init(CTX, MAXTOK, O.WIN, M.ptr(norms), M.ptr(router_all), M.ptr(cs)), "gfull_init")
    rids = []
    for L in range(NL):
        hl = HostLayer(SEED, L % 2)
        rids.append(M.register_layer(L, hl.blk, routers[L % 2], post[L % 2]))
    return lib, rids


def test_queued_groupings(model):
    lib, rids = model
    rng = np.random.default_rng(SEED + 80)
    nb, calls = 24, []
    for k in range(10):
        top = np.argsort(rng.random((nb, 256)), 1)[:, :8].astype(np.int32)
        g = O.group(top, rng.random((nb, 8)).astype(np.float32))
        calls.append((g, M.block_loc(0, list(g["ue"])), np.array([rids[k % NL], -1, -1, -1], np.int32), np.ascontiguousarray(g["tp"])))
    x0 = rng.standard_normal((nb, H)).astype(np.float32)
    out = []
    for wait in (True, False):
        lib.gfull_begin(M.ptr(x0), nb, 0)
        assert lib.mmoe_gfull_post_norm(0, None) == 0    # the calls' input: hn of the chunk
        for g, loc, regs, tp in calls:
            lib.gfull_moe(g["nu"], M.ptr(loc), M.ptr(regs), M.ptr(g["ustart"]), M.ptr(g["utok"]), M.ptr(g["uw"]), M.ptr(tp))
            if wait:
                M.check(lib.mmoe_sync(), "sync")
        x = np.empty((nb, H), np.float32)
        lib.gfull_read(M.ptr(x), None)
        out.append(x)
    assert np.array_equal(out[0].view(np.int32), out[1].view(np.int32)) and not np.array_equal(out[0], x0)


def held_kv(lib, nb):
    """the chunk's keys and values where gfull_read hands them out"""
    p = C.c_void_p()
    lib.gfull_read(None, C.addressof(p))
    a = np.ctypeslib.as_array((C.c_uint16 * (24 * MAXTOK * 1024)).from_address(p.value)).reshape(24, MAXTOK, 1024)
    return a[:NL, :nb]


def read_kv(lib, nb):
    return held_kv(lib, nb).copy()


def test_kv_copied_beside_the_stack(model):
    lib, _ = model
    rng = np.random.default_rng(SEED + 81)
    chunks = [(0, 200), (200, 37), (237, 256)]
    xs = [rng.standard_normal((nb, H)).astype(np.float32) for _, nb in chunks]

    def run(read, stacks):
        got = []
        for (pos, nb), x in zip(chunks, xs):
            lib.gfull_begin(M.ptr(x), nb, pos)
            for L0, nl in stacks:
                M.check(lib.mmoe_gfull_stack(L0, nl), "stack")
            if read(nb):
                got.append(read_kv(lib, nb))
        return got

    lib.gfull_read(None, None)                                   # not asked for: gfull_read copies it all
    lib.gfull_begin(M.ptr(xs[0]), 200, 0)
    want = []
    for (pos, nb), x in zip(chunks, xs):
        lib.gfull_begin(M.ptr(x), nb, pos)
        M.check(lib.mmoe_gfull_stack(0, NL), "stack")
        lib.gfull_read(None, None)
        want.append(read_kv(lib, nb))
        lib.gfull_read(None, None)
    for name, read, stacks in (("beside", lambda nb: True, [(0, NL)]), ("unread chunk", lambda nb: nb != 37, [(0, NL)]),
                               ("in parts", lambda nb: True, [(0, 1), (1, 3)])):
        got = run(read, stacks)
        ref = [w for w, (_, nb) in zip(want, chunks) if read(nb)]
        assert all(np.array_equal(a, b) for a, b in zip(got, ref)), name
    # the same chunk twice (the second stack starts from the first one's hidden state), read once
    lib.gfull_begin(M.ptr(xs[0]), 200, 0)
    M.check(lib.mmoe_gfull_stack(0, NL), "stack"); M.check(lib.mmoe_gfull_stack(0, NL), "stack")
    twice = read_kv(lib, 200)
    lib.gfull_read(None, None)
    lib.gfull_begin(M.ptr(xs[0]), 200, 0)
    M.check(lib.mmoe_gfull_stack(0, NL), "stack"); M.check(lib.mmoe_gfull_stack(0, NL), "stack")
    assert np.array_equal(twice, read_kv(lib, 200)) and not np.array_equal(twice, want[0])


def test_kv_held_over_the_next_chunks(model):
    """what gfull_read handed out stays as it is until the next gfull_read that asks for it: over the next chunk's stack, over
    further chunks that nobody reads, over a read of the hidden state alone, and over a rejected chunk"""
    lib, _ = model
    wait = C.CDLL("libamdhip64.so").hipDeviceSynchronize   # for the copies too
    rng = np.random.default_rng(SEED + 82)
    xs = [rng.standard_normal((nb, H)).astype(np.float32) for nb in (200, 56, 200, 200)]
    pos, held, kept = 0, None, None

    def chunk(x):
        lib.gfull_begin(M.ptr(x), len(x), pos)
        M.check(lib.mmoe_gfull_stack(0, NL), "stack")

    for x in xs + xs[:2]:
        pos = 0 if pos + len(x) > CTX else pos
        chunk(x)
        if held is not None:
            assert wait() == 0 and np.array_equal(held, kept)
            chunk(x)                                  # once more, unread
            lib.gfull_begin(M.ptr(x), 0, pos)         # rejected
            assert wait() == 0 and np.array_equal(held, kept)
            chunk(x)
            lib.gfull_read(None, None)
            assert np.array_equal(held, kept)
        now = held_kv(lib, len(x))
        assert held is None or np.array_equal(held, kept)
        held, kept = now, now.copy()
        assert kept.any()
        pos += len(x)


@pytest.mark.parametrize("nb", [3, 8, 9])
def test_work_input_after_gpre_moe(model, nb):
    """the call's rows are in the work input (mmoe_read) whichever way they reached the card"""
    lib, rids = model
    rng = np.random.default_rng(SEED + 83 + nb)
    g = O.group(np.argsort(rng.random((nb, 256)), 1)[:, :8].astype(np.int32), rng.random((nb, 8)).astype(np.float32))
    x = rng.standard_normal((nb, H)).astype(np.float32)
    y, regs = np.empty_like(x), np.array([rids[0], -1, -1, -1], np.int32)
    loc, tp = M.block_loc(0, list(g["ue"])), np.ascontiguousarray(g["tp"])
    assert lib.gpre_moe(M.ptr(x), nb, g["nu"], M.ptr(loc), M.ptr(regs), None, M.ptr(g["ustart"]), M.ptr(g["utok"]), M.ptr(g["uw"]),
                        M.ptr(tp), M.ptr(y)) >= 0
    assert np.array_equal(M.read("HN", (nb, H), np.float32).view(np.int32), x.view(np.int32))


@pytest.mark.parametrize("nb", [6, 40])
def test_grouping_under_capture(model, nb):
    """a captured gfull_moe call, replayed with eager calls of other groupings (more than the ring holds) in between"""
    lib, rids = model
    hip = C.CDLL("libamdhip64.so")
    rng = np.random.default_rng(SEED + 90 + nb)
    calls = []
    for k in range(6):
        g = O.group(np.argsort(rng.random((nb, 256)), 1)[:, :8].astype(np.int32), rng.random((nb, 8)).astype(np.float32))
        calls.append((g, M.block_loc(0, list(g["ue"])), np.array([rids[k % NL], -1, -1, -1], np.int32), np.ascontiguousarray(g["tp"])))
    x0 = rng.standard_normal((nb, H)).astype(np.float32)

    def call(k):
        g, loc, regs, tp = calls[k]
        lib.gfull_moe(g["nu"], M.ptr(loc), M.ptr(regs), M.ptr(g["ustart"]), M.ptr(g["utok"]), M.ptr(g["uw"]), M.ptr(tp))

    def read():
        x = np.empty((nb, H), np.float32)
        lib.gfull_read(M.ptr(x), None)
        return x

    lib.gfull_begin(M.ptr(x0), nb, 0)
    assert lib.mmoe_gfull_post_norm(0, None) == 0
    for k in (*range(6), 0):
        call(k)
    want = read()
    stream, graph, ex = C.c_void_p(lib.mmoe_stream()), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    call(0)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    try:
        for _ in range(3):
            lib.gfull_begin(M.ptr(x0), nb, 0)
            assert lib.mmoe_gfull_post_norm(0, None) == 0
            for k in range(6):
                call(k)
            assert hip.hipGraphLaunch(ex, stream) == 0
            assert np.array_equal(read().view(np.int32), want.view(np.int32))
    finally:
        M.check(lib.mmoe_sync(), "sync")
        hip.hipGraphExecDestroy(ex); hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("mode", [0, 1])   # global, thread-local
@pytest.mark.parametrize("nb", [5, 200])
def test_stack_under_capture(model, nb, mode):
    """mmoe_gfull_stack captured by its caller while the copies of another chunk are under way, replayed with eager chunks in
    between: hidden state, keys and values of every replay as the eager call's"""
    lib, _ = model
    hip = C.CDLL("libamdhip64.so")
    rng = np.random.default_rng(SEED + 95 + nb)
    x0, x1 = (rng.standard_normal((n, H)).astype(np.float32) for n in (nb, 256))

    def chunk(x, pos, stack):
        lib.gfull_begin(M.ptr(x), len(x), pos)
        stack()

    def eager():
        M.check(lib.mmoe_gfull_stack(0, NL), "stack")

    def read():
        x = np.empty((nb, H), np.float32)
        lib.gfull_read(M.ptr(x), None)
        return x.view(np.int32), read_kv(lib, nb)

    chunk(x0, 0, eager)
    want = read()
    chunk(x1, 300, eager)
    stream, graph, ex = C.c_void_p(lib.mmoe_stream()), C.c_void_p(), C.c_void_p()
    lib.gfull_begin(M.ptr(x0), nb, 0)
    assert hip.hipStreamBeginCapture(stream, mode) == 0
    eager()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    try:
        for _ in range(3):
            chunk(x0, 0, lambda: hip.hipGraphLaunch(ex, stream))
            got = read()
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
            chunk(x1, 300, eager)
    finally:
        M.check(lib.mmoe_sync(), "sync")
        hip.hipGraphExecDestroy(ex); hip.hipGraphDestroy(graph)


def test_gpux_under_capture(model):
    """gpux_begin captured by its caller, replayed with other values in its input array and eager calls in between: gpux_end
    after a replay gives the replay's outputs"""
    lib, _ = model
    hip = C.CDLL("libamdhip64.so")
    M.check(lib.gpux_init(1, 8), "gpux_init")
    hl = HostLayer(SEED, 0)
    for s in range(8):
        lib.gpux_upload(0, s, *[M.ptr(a) for a in M.expert_views(hl.blk, 11 * s)])
    rng = np.random.default_rng(SEED + 99)
    xs = rng.standard_normal((3, H)).astype(np.float32)
    slots, few = np.arange(8, dtype=np.int32), np.array([5, 2], np.int32)

    def end(h, n):
        out = np.full((n, H), np.nan, np.float32)
        lib.gpux_end(h, M.ptr(out), n)
        return out.view(np.int32)

    want = [end(lib.gpux_begin(0, M.ptr(x), 8, M.ptr(slots)), 8) for x in xs]
    other = end(lib.gpux_begin(0, M.ptr(xs[0]), 2, M.ptr(few)), 2)
    x = xs[0].copy()                                             # the captured call's input
    stream, graph, ex = C.c_void_p(lib.mmoe_stream()), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    h = lib.gpux_begin(0, M.ptr(x), 8, M.ptr(slots))
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert h, lib.mmoe_last_error()
    assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    try:
        for k in (0, 1, 2, 1):
            x[:] = xs[k]
            assert hip.hipGraphLaunch(ex, stream) == 0
            assert np.array_equal(end(h, 8), want[k]), f"replay {k}"
            assert np.array_equal(end(lib.gpux_begin(0, M.ptr(xs[0]), 2, M.ptr(few)), 2), other)
            assert np.array_equal(end(lib.gpux_begin(0, M.ptr(xs[0]), 8, M.ptr(slots)), 8), want[0])
    finally:
        M.check(lib.mmoe_sync(), "sync")
        hip.hipGraphExecDestroy(ex); hip.hipGraphDestroy(graph)


def test_grouping_without_pairs(model):
    """a grouping whose experts have no pairs runs and changes nothing for the calls after it; one that starts below 0 is
    refused"""
    lib, _ = model
    M.check(lib.gpux_init(1, 2), "gpux_init")
    hl = HostLayer(SEED, 0)
    for s in range(2):
        lib.gpux_upload(0, s, *[M.ptr(a) for a in M.expert_views(hl.blk, s)])
    x = np.random.default_rng(SEED + 98).standard_normal((2, H)).astype(np.float32)
    slots, tok = np.array([0, 1], np.int32), np.zeros(2, np.int32)

    def call(*start):
        out, us = np.zeros((2, H), np.float32), np.array(start, np.int32)
        h = lib.gpux_begin_multi(0, M.ptr(x), 2, 2, M.ptr(slots), M.ptr(us), M.ptr(tok))
        if h:
            lib.gpux_end_multi(h, M.ptr(out), 2)
        return out if h else None

    want = call(0, 1, 2)
    assert want.any() and call(2, 2, 2) is not None
    assert call(-1, 1, 2) is None and b"ustart[0]" in lib.mmoe_last_error()
    assert np.array_equal(call(0, 1, 2).view(np.int32), want.view(np.int32))


def test_smaller_setup_drops_the_chunk(model, gfull_model):  # noqa: F811
    """a chunk begun under a larger set-up is no chunk of a smaller one: the calls that would use it say so"""
    lib, _ = model
    _, _, _, _, cs, norms, router_all = gfull_model
    x = np.random.default_rng(SEED + 97).standard_normal((200, H)).astype(np.float32)

    def init(ctx, maxtok):
        M.check(lib.gfull_init(ctx, maxtok, O.WIN, M.ptr(norms), M.ptr(router_all), M.ptr(cs)), "gfull_init")

    try:
        for nb, pos, ctx, maxtok in ((200, 0, CTX, 64), (20, 300, 256, 64)):
            init(CTX, MAXTOK)
            lib.gfull_begin(M.ptr(x), nb, pos)
            init(ctx, maxtok)
            assert lib.gfull_attn(0, 0, None) < 0 and lib.mmoe_gfull_stack(0, 1) != 0
            lib.gfull_begin(M.ptr(x), 20, 0)
            assert lib.gfull_attn(0, 0, None) >= 0, lib.mmoe_last_error()
    finally:
        init(CTX, MAXTOK)
