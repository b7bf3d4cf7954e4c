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
