"""Walks on list tables (fw_table_walk.hip) against the CPU oracle, bit for bit: lists whose lengths sit at the edges of
the tables' shapes (quartets, the lanes of a group, groups, sequences), biases that are zero, close to even and far from
even, path rows of every alignment.  The tables are made when a call's walkers would read the edge array several times over,
so the first call on a graph is a large one and later, smaller calls walk on what it made."""
import numpy as np
import pytest

import fw_oracle_binding as _oracle

pytestmark = pytest.mark.gpu

V = 24000


def _lists(kind):
    """A directed graph with lists of every interesting length at every alignment; neighbours ascending, weights of `kind`."""
    rng = np.random.RandomState(3)
    deg = np.full(V, 3, dtype=np.int64)
    lengths = list(range(0, 70)) + list(range(122, 134)) + list(range(250, 262)) + list(range(508, 518)) + \
        list(range(764, 772)) + list(range(1016, 1034)) + list(range(1272, 1290)) + list(range(2040, 2056)) + \
        [3071, 3072, 3073, 4097, 8191, 16383, 16384, 16385, 20001]
    at = rng.permutation(V)[:len(lengths)]
    deg[at] = lengths
    xadj = np.zeros(V + 1, dtype=np.uint32)
    np.cumsum(deg, out=xadj[1:])
    E = int(xadj[-1])
    # half of the edges lead back to the listed vertices, so that walks meet them again and again
    adj = np.where(rng.random_sample(E) < 0.5, at[rng.randint(0, len(at), size=E)], rng.randint(0, V, size=E)).astype(np.int32)
    for v in range(V):
        adj[xadj[v]:xadj[v + 1]].sort()
    if kind == "even":
        w = (1.0 + 99.0 * rng.random_sample(E)).astype(np.float32)
    else:
        w = np.exp(rng.normal(0.0, 3.0, size=E)).astype(np.float32)
        w[rng.random_sample(E) < 0.3] = 0.0
        for v in at[::17]:
            w[xadj[v]:xadj[v + 1]] = 0.0
    return (xadj, adj, w), at


@pytest.mark.parametrize("kind", ["even", "uneven"])
@pytest.mark.parametrize("wg,thr", [(512, 16384), (256, 1024), (1024, 2000), (512, 1 << 30)])
def test_walks_on_tables(gpu, kind, wg, thr):
    csr, at = _lists(kind)
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(wg)
    try:
        cases = [(dict(app=gpu.APP_DEEPWALK, max_depth=21), 70000)]
        for n, depth in ((1, 81), (63, 2), (65, 15), (1000, 16), (777, 17), (4001, 33), (3, 1), (129, 100)):
            cases.append((dict(app=gpu.APP_DEEPWALK, max_depth=depth), n))
        cases.append((dict(app=gpu.APP_PPR, max_depth=50, tp=0.1), 3000))
        for p, q in ((2.0, 0.5), (0.25, 4.0), (4.0, 0.25), (1.0, 1.0), (0.1, 1.0)):
            cases.append((dict(app=gpu.APP_NODE2VEC, max_depth=18, p=p, q=q), 2000))
        for i, (kw, n) in enumerate(cases):
            p = gpu.default_params(wg_threads=wg, hub_threshold=thr, seed=100 + i, walker_base=i, **kw)
            starts = np.where(rng.random_sample(n) < 0.8, at[rng.randint(0, len(at), size=n)], rng.randint(0, V, size=n)).astype(np.int32)
            if n > 100:
                starts[5] = -1
                starts[7] = V
            ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(p), starts)
            paths, st = g.walk(p, starts)
            bad = np.nonzero((paths != ref).any(axis=1))[0]
            assert len(bad) == 0, (kw, n, bad[0], paths[bad[0]], ref[bad[0]])
            assert (st.steps, st.sampled_edges) == (steps, edges), (kw, n)
            if i == 0:
                assert st.launches >= 4  # the tables were made
            again, st2 = g.walk_batch(p, starts, batch_size=max(1, n // 3))
            assert (again == ref).all() and (st2.steps, st2.sampled_edges) == (steps, edges), (kw, n)
    finally:
        g.destroy()
