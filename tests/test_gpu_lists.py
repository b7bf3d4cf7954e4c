"""The lists that a step's layers share (the prefill's rows and work items, the
front's rows, the shared-prefix pass's items) are uploaded once and told apart
by value. Each call that changes what they are made of - lengths, ids, order,
positions, another kind of call on the same buffers - gets its own: a context
that runs a mixed sequence of calls equals a fresh context per call, bit for
bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def nda():
    import ndattn
    return ndattn


NH, QK, VD, W, LAYERS = 8, 64, 64, 256, 2


def context(max_seqs):
    N = nda()
    return N.Context(LAYERS, NH, NH, QK, VD, W, kv_dtype=N.KV_F16, max_seqs=max_seqs)


def data(seed, rows):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((rows, NH, d)).astype(np.float32) for d in (QK, QK, VD)]


def chunk(ctx, layer, lens, ids, seed):
    N = nda()
    q, k, v = (N.DevBuf.from_array(a) for a in data(seed + layer, int(sum(lens))))
    out = N.DevBuf(int(sum(lens)) * NH * VD * 4)
    ctx.prefill(layer, np.asarray(lens, np.uint32), q, k, v, out, seq_ids=ids)
    ctx.sync()
    return out.to_array(np.uint32, (int(sum(lens)), NH, VD))


# (lens, ids): the same totals in another split, another order, other ids,
# with a sequence left out, then the first again
CALLS = [([5, 40, 3], [0, 1, 2]), ([5, 40, 3], [0, 1, 2]), ([40, 5, 3], [0, 1, 2]), ([5, 40, 3], [1, 0, 2]),
         ([5, 40, 3], [3, 1, 2]), ([48], [0]), ([24, 0, 24], [0, 1, 2]), ([5, 40, 3], [0, 1, 2])]


@pytest.mark.parametrize("between", ["nothing", "append", "advance"])
def test_prefill_lists(between):
    N = nda()
    one = context(4)
    done = []           # (kind, args) so far, replayed in the fresh contexts
    for n, (lens, ids) in enumerate(CALLS):
        got = [chunk(one, layer, lens, ids, 10 * n) for layer in range(LAYERS)]
        fresh = context(4)
        for ids2, m in done:
            fresh.advance(len(ids2), ids2, m)
        for layer in range(LAYERS):
            # the positions before a sequence's own chunk were stored by the
            # shared context's earlier calls: bring them over
            for b in range(4):
                pos = one.seq_state(b)[0]
                if pos and layer == 0:
                    for li in range(LAYERS):
                        k, v, _, _ = one.kv_read(li, b, 0, pos)
                        fresh.kv_write(li, b, 0, k, v)
            want = chunk(fresh, layer, lens, ids, 10 * n)
            assert np.array_equal(got[layer], want), (n, layer)
        fresh.close()
        if between == "append":     # the row staging goes to another call
            k, v = (N.DevBuf.from_array(a) for a in data(900 + n, 2)[1:])
            one.kv_append(0, 2, k, v, seq_ids=[2, 0])
            one.kv_append(1, 2, k, v, seq_ids=[2, 0])
        elif between == "advance" and n % 2:
            one.advance(len([i for i, m in zip(ids, lens) if m]), [i for i, m in zip(ids, lens) if m], 1)
            done.append(([i for i, m in zip(ids, lens) if m], 1))
    one.close()


def ops(rng, groups):
    """A call of each kind on other sequences, lengths and positions than the
    last of its kind, or on the same again."""
    kept = {}
    for _ in range(60):
        kind = rng.choice(["front", "prefill", "step", "step", "advance"])
        if kind in kept and rng.random() < 0.4:
            yield kept[kind]
            continue
        if kind == "step":
            g = groups[rng.integers(len(groups))]
            what = (kind, [int(x) for x in (g if rng.random() < 0.5 else rng.permutation(g))], None)
        else:
            ids = [int(x) for x in rng.permutation(groups[rng.integers(len(groups))])[:rng.integers(1, 5)]]
            if kind == "front" and rng.random() < 0.3:
                what = (kind, ids, None)
            else:
                what = (kind, ids, [int(x) for x in rng.integers(0 if len(ids) > 1 else 1, 4, len(ids))])
                what[2][0] = max(1, what[2][0])
        kept[kind] = what
        yield what


@pytest.mark.parametrize("streams", [1, 2])
def test_lists_of_every_kind(streams):
    """Fronts, prefills and decode steps over two shared prefixes of different
    lengths (128 sequences each, which take the shared-prefix pass) in any
    order, each over two layers, from one stream or two in turn: outputs and
    histories equal those of a context whose every call is preceded by one of
    each kind on a spare sequence, so that no list of it is ever held."""
    N = nda()
    taps, spare, per = 3, 256, 128
    rng = np.random.default_rng(5)
    w = [(rng.standard_normal((taps, NH * d)) * 0.5).astype(np.float32) for d in (QK, QK, VD)]
    norms = [(rng.standard_normal(QK) * 0.25).astype(np.float32) for _ in range(2)]
    ctxs = []
    for _ in range(2):
        c = N.Context(LAYERS, NH, NH, QK, VD, W, kv_dtype=N.KV_F16, max_seqs=spare + 1)
        c.front_init(taps, 10000.0)
        for li in range(LAYERS):
            c.front_weights(li, *w, *norms)
        for g, npre in enumerate((64, 110)):
            c.seq_set_pos(g * per, npre)
            c.kv_fill_normal(1, seed=g, seq_ids=[g * per])
            pid = c.prefix_build(g * per)
            for b in range(g * per, (g + 1) * per):
                c.seq_attach(b, pid)
        ctxs.append(c)
    st = [N.vp() for _ in range(streams)]
    if streams > 1:
        for s in st:
            N._check(N.lib().nda_stream_create(N.C.byref(s)))
    one = [N.DevBuf.from_array(a) for a in data(1, 1)]
    dump = [N.DevBuf(NH * VD * 4) for _ in range(3)]
    for n, (kind, ids, m) in enumerate(ops(rng, [range(per), range(per, 2 * per)])):
        if kind == "advance":
            for c in ctxs:
                c.advance(len(ids), ids, 1, stream=st[n % streams])
            continue
        rows = len(ids) if m is None else sum(m)
        for layer in range(LAYERS):
            x = [N.DevBuf.from_array(a) for a in data(100 * n + layer, rows)]
            got = []
            for c in ctxs:
                s = st[n % streams] if c is ctxs[0] else None
                if c is ctxs[1]:
                    c.front(layer, 1, *one, *dump, seq_ids=[spare])
                    c.prefill(layer, [1], *one, dump[0], seq_ids=[spare])
                y = [N.DevBuf(rows * NH * d * 4) for d in (QK, QK, VD)]
                if kind == "front":
                    c.front(layer, len(ids), *x, *y, n_tokens=m, seq_ids=ids, stream=s)
                elif kind == "prefill":
                    c.prefill(layer, np.asarray(m, np.uint32), *x, y[0], seq_ids=ids, stream=s)
                else:
                    c.step(layer, len(ids), *x, y[0], seq_ids=ids, stream=s)
                got.append(y)
            for c in ctxs:
                c.sync()
            N.device_sync()
            for a, b in list(zip(*got))[:3 if kind == "front" else 1]:
                a, b = (t.to_array(np.uint32, (rows, NH * QK)) for t in (a, b))
                assert np.array_equal(a, b), (n, kind, layer)
    for b in range(0, 2 * per, 9):
        assert np.array_equal(*(c.front_hist(b).view(np.uint32) for c in ctxs)), b
    for c in ctxs:
        c.close()
    if streams > 1:
        for s in st:
            N._check(N.lib().nda_stream_destroy(s))


@pytest.mark.parametrize("kv,nh,nkv,qk,n", [("int8", 12, 2, 48, 40), ("int8", 12, 2, 48, 700), ("f16", 8, 8, 64, 20)])
def test_captured_steps(kv, nh, nkv, qk, n):
    """nda_step and nda_decode of sequences 0..n-1 in a graph (700 sequences:
    the launch that goes longest row first outside of one): every replay,
    between eager calls with listed ids and other row counts, equals the
    eager result."""
    N = nda()
    hip = N.C.CDLL("libamdhip64.so")

    def ok(rc):
        assert rc == 0, rc

    st, graph, ex = N.vp(), N.vp(), N.vp()
    N._check(N.lib().nda_stream_create(N.C.byref(st)))
    ctx = N.Context(1, nh, nkv, qk, VD, 320, kv_dtype=N.KV_F16 if kv == "f16" else N.KV_INT8, max_seqs=n)
    for b in range(n):
        ctx.seq_set_pos(b, (37 * b) % 300)
    ctx.kv_fill_normal(n, seed=3, stream=st)
    rng = np.random.default_rng(n)
    q, k, v = ([N.DevBuf.from_array(rng.standard_normal((n, h, d)).astype(np.float32)) for _ in range(2)]
               for h, d in ((nh, qk), (nkv, qk), (nkv, VD)))
    outs = [N.DevBuf(n * nh * VD * 4) for _ in range(3)]

    def calls(o):
        ctx.step(0, n, q[0], k[0], v[0], outs[o], stream=st)
        ctx.decode(0, n, q[1], outs[o + 1], stream=st)

    calls(0)
    ctx.sync(st)
    want = [outs[o].to_array(np.uint32, (n, nh, VD)) for o in (0, 1)]
    ok(hip.hipStreamBeginCapture(st, 2))
    calls(0)
    ok(hip.hipStreamEndCapture(st, N.C.byref(graph)))
    ok(hip.hipGraphInstantiate(N.C.byref(ex), graph, None, None, N.C.c_size_t(0)))
    for rep in range(4):
        ids = [int(x) for x in rng.permutation(n)[:n // (rep + 1)]]
        ctx.decode(0, len(ids), q[rep % 2], outs[2], seq_ids=ids, stream=st)
        ctx.sync(st)
        listed = outs[2].to_array(np.uint32, (len(ids), nh, VD))
        for o in (0, 1):
            outs[o].upload(np.zeros((n, nh, VD), np.float32))
        ok(hip.hipGraphLaunch(ex, st))
        ctx.sync(st)
        for o in (0, 1):
            assert np.array_equal(outs[o].to_array(np.uint32, (n, nh, VD)), want[o]), (rep, o)
        ctx.decode(0, len(ids), q[rep % 2], outs[2], seq_ids=ids, stream=st)
        ctx.sync(st)
        assert np.array_equal(outs[2].to_array(np.uint32, (len(ids), nh, VD)), listed), rep
    ok(hip.hipGraphExecDestroy(ex))
    ok(hip.hipGraphDestroy(graph))
    ctx.close()
    N._check(N.lib().nda_stream_destroy(st))
