"""Walks on list tables (fw_table_walk.hip) against the CPU oracle, bit for bit: lists whose lengths sit at the edges of
the tables' shapes (quartets, the lanes of a group, groups, sequences), biases that are zero, close to even and far from
even, path rows of every alignment.  The tables are made when a call's walkers would read the edge array several times over,
so the first call on a graph is a large one and later, smaller calls walk on what it made."""
import ctypes as C

import numpy as np
import pytest
import torch

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


def _padded(x):
    return torch.from_numpy(np.concatenate([x, np.zeros(4, dtype=x.dtype)])).cuda()


def _adopt(gpu, xadj, adj, w):
    """A graph over arrays that the caller keeps, and those arrays."""
    arrays = _padded(xadj.view(np.int32)), _padded(adj), _padded(w)
    torch.cuda.synchronize()
    h = C.c_void_p()
    gpu.check(gpu.lib().fw_graph_adopt_device(len(xadj) - 1, len(adj), *[C.c_void_p(x.data_ptr()) for x in arrays], None, 0, C.byref(h)))
    return gpu.Graph(h), arrays


def _fill_memory(gpu, leave):
    """Takes device memory until at most `leave` bytes are free; returns the buffers."""
    held = []
    for chunk in (16 << 30, 1 << 30, 32 << 20):
        while torch.cuda.mem_get_info()[0] > leave + chunk:
            held.append(gpu.DeviceBuffer(chunk))
    if torch.cuda.mem_get_info()[0] > leave:
        held.append(gpu.DeviceBuffer(32 << 20))
    return held


def test_batches_come_before_tables(gpu):
    """fw_walk_batch: tables give way to the path matrices of the call, those of earlier calls too, and to the parking lists of a later one."""
    g = gpu.Graph.rmat(20, 16, a=0.25, b=0.25, c=0.25, symmetrise=True, seed=3)
    n = 2500000
    starts = np.random.RandomState(2).randint(0, g.V, size=n).astype(np.int32)
    big = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=81, seed=4)  # 820 MB
    held = []
    try:
        g.limit_tables(0)
        ref, st = g.walk(big, starts)
        g.limit_tables((1 << 64) - 1)
        for tables in (False, True):  # whether the graph has some when the batch comes
            if tables:
                for _ in range(40):
                    g.walk(big, starts[:70000])
                assert g.engine()[0] == gpu.ENGINE_TABLES
            assert (g.engine()[2] > 300 << 20) == tables
            # 820 MB fit beside 900, but not beside 500 and what the runtime holds of freed memory without counting it as free (130 MB seen)
            held = _fill_memory(gpu, 900 << 20 if not tables else 500 << 20)
            paths, st2 = g.walk_batch(big, starts, batch_size=n)
            assert g.engine()[0] == gpu.ENGINE_STREAM and g.engine()[2] == 0
            assert (paths == ref).all() and st2.steps == st.steps
            while held:
                held.pop().free()
            g.destroy()  # (with the batch's buffers)
            g = gpu.Graph.rmat(20, 16, a=0.25, b=0.25, c=0.25, symmetrise=True, seed=3)
        for _ in range(40):
            g.walk(big, starts[:70000])
        assert g.engine()[0] == gpu.ENGINE_TABLES
        short = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=5, seed=4, park_threshold=16)
        held = _fill_memory(gpu, 300 << 20)  # (the parking index takes some 20 MB and, where it fits, 270, the lists 200 and more)
        paths, _ = g.walk_batch(short, starts, batch_size=n)
        assert g.engine()[::2] == (gpu.ENGINE_PARK, 0)
        short.park_threshold = -1
        assert (paths == g.walk_batch(short, starts, batch_size=n)[0]).all()
    finally:
        for b in held:
            b.free()
        g.destroy()


def test_parking_lists_that_do_not_fit(gpu):
    """fw_walk_batch without room for its parking lists (more than 180 MB) walks without parking, and so does the next call."""
    g = gpu.Graph.rmat(20, 16, a=0.25, b=0.25, c=0.25, symmetrise=True, seed=3)  # (no list gets rows of its own)
    n = 2500000
    starts = np.random.RandomState(2).randint(0, g.V, size=n).astype(np.int32)
    p = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=5, seed=4, park_threshold=16)
    held = []
    try:
        ref, st = g.walk(p, starts)
        assert g.engine()[0] == gpu.ENGINE_PARK
        held = _fill_memory(gpu, 160 << 20)
        for _ in range(2):
            paths, st2 = g.walk_batch(p, starts, batch_size=n)
            assert g.engine()[0] == gpu.ENGINE_STREAM
            assert (paths == ref).all() and st2.steps == st.steps
        while held:
            held.pop().free()
        paths, _ = g.walk_batch(p, starts, batch_size=n)
        assert g.engine()[0] == gpu.ENGINE_PARK and (paths == ref).all()
    finally:
        for b in held:
            b.free()
        g.destroy()


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
            assert g.engine()[0] == gpu.ENGINE_TABLES
            assert (g.engine()[1] != 0) == (st.launches > 3)
            if i == 0:
                assert st.launches >= 4  # the tables were made
            again, st2 = g.walk_batch(p, starts, batch_size=max(1, n // 3))
            assert (again == ref).all() and (st2.steps, st2.sampled_edges) == (steps, edges), (kw, n)
    finally:
        g.destroy()


@pytest.mark.parametrize("wg,thr", [(512, 16384), (256, 1024)])
@pytest.mark.parametrize("n", [8192, 8193])
def test_wave_or_lane_per_walker(gpu, n, wg, thr):
    """Either side of the number of walkers up to which a wave walks each."""
    csr, at = _lists("uneven")
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(n)
    try:
        g.walk(gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21, wg_threads=wg, hub_threshold=thr), at[rng.randint(0, len(at), size=70000)].astype(np.int32))
        for kw in (dict(app=gpu.APP_DEEPWALK, max_depth=66), dict(app=gpu.APP_PPR, max_depth=20, tp=0.1), dict(app=gpu.APP_NODE2VEC, max_depth=9, p=0.25, q=4.0),
                   dict(app=gpu.APP_NODE2VEC, max_depth=9, p=2.0, q=0.5)):
            p = gpu.default_params(wg_threads=wg, hub_threshold=thr, seed=n, **kw)
            starts = at[rng.randint(0, len(at), size=n)].astype(np.int32)
            ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(p), starts)
            paths, st = g.walk(p, starts)
            assert g.engine()[0] == gpu.ENGINE_TABLES
            assert (paths == ref).all() and (st.steps, st.sampled_edges) == (steps, edges), kw
    finally:
        g.destroy()


@pytest.mark.parametrize("wg,thr", [(256, 16384), (512, 1 << 30)])
def test_sums_beyond_four_blocks(gpu, wg, thr):
    """Lists of 69 and 4297 groups: the sums of 64 groups are in registers, and behind them 64 blocks are looked at together."""
    V, hubs = 2000, (70001, 4400001)
    rng = np.random.RandomState(5)
    deg = np.full(V, 2, dtype=np.int64)
    deg[:2] = hubs
    xadj = np.zeros(V + 1, dtype=np.uint32)
    np.cumsum(deg, out=xadj[1:])
    adj = np.tile(np.array([0, 1], dtype=np.int32), int(xadj[-1]) // 2 + 1)[:int(xadj[-1])]  # every other vertex leads to the two
    for v in (0, 1):
        adj[xadj[v]:xadj[v + 1]] = np.sort(rng.randint(2, V, size=deg[v]))
    w = np.exp(rng.normal(0.0, 3.0, size=len(adj))).astype(np.float32)
    g = gpu.Graph.from_csr(xadj, adj, w)
    og = _oracle.Graph(xadj, adj, w)
    try:
        kw = dict(app=gpu.APP_DEEPWALK, wg_threads=wg, hub_threshold=thr)
        g.walk(gpu.default_params(max_depth=11, **kw), rng.randint(0, V, size=70000).astype(np.int32))
        starts = rng.randint(0, V, size=100).astype(np.int32)
        starts[:40] = np.arange(40) % 2
        p = gpu.default_params(max_depth=4, seed=9, **kw)
        ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(p), starts)
        paths, st = g.walk(p, starts)
        assert g.engine()[0] == gpu.ENGINE_TABLES
        assert (paths == ref).all() and (st.steps, st.sampled_edges) == (steps, edges)
    finally:
        g.destroy()


@pytest.mark.parametrize("kind", ["even", "uneven"])
def test_node2vec_on_hash_sets(gpu, kind):
    """The first call is long enough to pay for the sets (one walk of 100 steps counts as 0.4 ms of searches, 1.5 times 0.2 ms are asked
    for); the lists hold equal neighbours, and the longest have buckets that more than 16 neighbours fall into."""
    csr, at = _lists(kind)
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(7)
    try:
        warm = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21)
        g.walk(warm, at[rng.randint(0, len(at), size=70000)].astype(np.int32))
        for i, (p, q) in enumerate(((2.0, 0.5), (0.25, 4.0), (4.0, 0.25), (1.0, 1.0), (0.1, 1.0), (1.0, 3.0), (0.5, 0.25))):
            par = gpu.default_params(app=gpu.APP_NODE2VEC, max_depth=101, p=p, q=q, seed=50 + i)
            starts = at[rng.randint(0, len(at), size=400)].astype(np.int32)
            ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(par), starts)
            paths, st = g.walk(par, starts)
            bad = np.nonzero((paths != ref).any(axis=1))[0]
            assert len(bad) == 0, (p, q, bad[0], paths[bad[0]], ref[bad[0]])
            assert (st.steps, st.sampled_edges) == (steps, edges)
            assert st.launches == (5 if i < 2 else 3)  # the sets, then with the first return edge above the envelope their weights
    finally:
        g.destroy()


def test_weights_of_sets_have_to_be_earned(gpu):
    """Sets that are there are made again with their entries' weights only once the searches for the return edge have cost that: a small
    call with p < 1 searches the lists, a loop of them gets the weights."""
    csr, at = _lists("even")
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    starts = at[np.random.RandomState(3).randint(0, len(at), size=70000)].astype(np.int32)
    try:
        for _ in range(8):
            g.walk(gpu.default_params(app=gpu.APP_NODE2VEC, max_depth=21, seed=6, p=2.0, q=0.5), starts)
        sets = g.engine()
        par = gpu.default_params(app=gpu.APP_NODE2VEC, max_depth=21, seed=7, p=0.25, q=4.0)
        ref, _, _ = _oracle.walk(og, _oracle.from_walk_params(par), starts[:20])
        for i in range(20):
            paths, _ = g.walk(par, starts[:20])
            assert (paths == ref).all()
            if i == 0:
                assert g.engine() == sets
        assert g.engine()[2] > sets[2]
    finally:
        g.destroy()


def test_sets_of_a_long_list_have_to_be_earned(gpu):
    """A list of 3,000,000 entries takes its sets some 13 ms (it is read once per 8192 entries): a call whose searches cost 3 ms goes without
    them."""
    rng = np.random.RandomState(5)
    hub, vertices = 3000000, 20000
    xadj = np.full(vertices + 1, hub, dtype=np.uint32) + np.arange(-1, vertices, dtype=np.int64).astype(np.uint32)
    xadj[0] = 0
    adj = np.zeros(int(xadj[-1]), dtype=np.int32)
    adj[:hub] = np.sort(rng.randint(0, vertices, size=hub))
    w = (1.0 + 9.0 * rng.random_sample(len(adj))).astype(np.float32)
    g = gpu.Graph.from_csr(xadj, adj, w)
    try:
        starts = rng.randint(0, vertices, size=1000000).astype(np.int32)
        par = gpu.default_params(app=gpu.APP_NODE2VEC, max_depth=101, p=2.0, q=0.5, seed=3)
        paths, st = g.walk(par, starts)
        engine, made, _ = g.engine()
        assert engine == gpu.ENGINE_TABLES and made == 3  # the lists, without sets
        ref, _, _ = _oracle.walk(_oracle.Graph(xadj, adj, w), _oracle.from_walk_params(par), starts[:5])
        assert (paths[:5] == ref).all()
    finally:
        g.destroy()


def test_memory_of_tables(gpu):
    """fw_graph_limit_tables: what is above the bound is given back at once and not taken again, tables without room for sets, sets without
    room for their weights; the walks are the same."""
    csr, at = _lists("even")
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    starts = at[np.random.RandomState(3).randint(0, len(at), size=70000)].astype(np.int32)
    unlimited = (1 << 64) - 1

    def walk(engine, n=70000, **kw):
        par = gpu.default_params(max_depth=21, seed=6, **kw)
        ref, _, _ = _oracle.walk(og, _oracle.from_walk_params(par), starts[:3000])
        for _ in range(8 if kw["app"] == gpu.APP_NODE2VEC else 1):  # sets have to be earned by several calls
            paths, _ = g.walk(par, starts[:n])
            assert g.engine()[0] == engine
            assert (paths[:3000] == ref[:n]).all()
        return g.engine()[2]

    back = dict(app=gpu.APP_NODE2VEC, p=0.25, q=4.0)
    try:
        assert g.engine() == (gpu.ENGINE_NONE, 0, 0)
        held = walk(gpu.ENGINE_TABLES, app=gpu.APP_DEEPWALK)
        assert held > 8 * g.E
        g.limit_tables(held)
        assert g.engine()[2] == held
        assert walk(gpu.ENGINE_TABLES, **back) == held          # no room for sets: the lists are searched
        g.limit_tables(held + 9 * g.E + 70 * V)
        with_sets = walk(gpu.ENGINE_TABLES, **back)              # nor for their weights
        assert held + 8 * g.E <= with_sets <= held + 9 * g.E + 70 * V
        g.limit_tables(unlimited)
        assert walk(gpu.ENGINE_TABLES, **back) > with_sets
        g.limit_tables(held - 1)
        assert g.engine()[2] == 0
        for _ in range(20):
            assert walk(gpu.ENGINE_PARK, app=gpu.APP_DEEPWALK) == 0
        assert walk(gpu.ENGINE_STREAM, n=3000, app=gpu.APP_DEEPWALK) == 0
        g.limit_tables(unlimited)
        assert walk(gpu.ENGINE_TABLES, app=gpu.APP_DEEPWALK) == held
        g.limit_tables(0)
        assert walk(gpu.ENGINE_PARK, app=gpu.APP_DEEPWALK) == 0
    finally:
        g.destroy()


def test_modelled_traffic(gpu):
    """What the byte model charges: the making in the call that makes, by what it made, and per step the blocks that the application cannot do without: the record
    and a block of pairs (of neighbours), for node2vec a bucket of a hash set, or four blocks of a search."""
    (xadj, adj, w), at = _lists("even")
    lab = np.random.RandomState(1).randint(0, 3, size=len(adj)).astype(np.int32)
    g = gpu.Graph.from_csr(xadj, adj, w, lab)
    E, n = len(adj), 70000
    starts = at[np.random.RandomState(3).randint(0, len(at), size=n)].astype(np.int32)
    try:
        for app, reads, made in ((gpu.APP_DEEPWALK, 2, 8 * E + 4 * V), (gpu.APP_METAPATH, 2, 8 * E + 4 * V), (gpu.APP_NODE2VEC, 6, 4 * E + 16 * V)):
            par = gpu.default_params(app=app, max_depth=21, seed=6, schema=[0, 1, 2])
            for i in range(20):
                _, st = g.walk(par, starts)
                engine, launches, _ = g.engine()
                if engine == gpu.ENGINE_TABLES and app == gpu.APP_NODE2VEC and launches == 0 and i < 2:  # no sets yet
                    assert st.scattered_reads == reads * st.steps - 3 * n
                if launches != 0:
                    break
            assert launches != 0 and st.list_bytes == made
            _, st = g.walk(par, starts)
            assert g.engine()[:2] == (gpu.ENGINE_TABLES, 0) and st.list_bytes == 0
            assert st.record_bytes == 4 * n + 4 * n * 21
            if app == gpu.APP_NODE2VEC:
                assert st.scattered_reads == 3 * st.steps
            else:
                assert st.scattered_reads == reads * st.steps + n
    finally:
        g.destroy()


def test_kernel_times_leave_the_tables(gpu):
    """A call that asks for the split of its time walks on the tables that are there, like any other: nothing is made anew."""
    csr, at = _lists("even")
    g = gpu.Graph.from_csr(*csr)
    starts = at[np.random.RandomState(3).randint(0, len(at), size=70000)].astype(np.int32)
    try:
        for app in (gpu.APP_DEEPWALK, gpu.APP_NODE2VEC):
            par = gpu.default_params(app=app, max_depth=21, seed=6, p=0.25, q=4.0)
            for _ in range(8):  # sets have to be earned by several calls
                plain, _ = g.walk(par, starts)
            assert g.engine()[:2] == (gpu.ENGINE_TABLES, 0)
            par.time_kernels = 1
            paths, st = g.walk(par, starts)
            assert g.engine()[:2] == (gpu.ENGINE_TABLES, 0) and st.launches == 3
            assert st.hub_kernel_ms == 0.0 and st.walk_kernel_ms == st.kernel_ms > 0.0
            assert (paths == plain).all()
            paths, st = g.walk_batch(par, starts, batch_size=30000)
            assert g.engine()[:2] == (gpu.ENGINE_TABLES, 0)
            assert st.hub_kernel_ms == 0.0 and st.walk_kernel_ms == st.kernel_ms > 0.0
            assert (paths == plain).all()
    finally:
        g.destroy()


def test_calls_on_other_streams_and_threads(gpu):
    """Tables made in a call on one stream, sets on another, walked on from a third and from another thread."""
    import threading
    (xadj, adj, w), at = _lists("even")
    lab = np.random.RandomState(1).randint(0, 3, size=len(adj)).astype(np.int32)
    g = gpu.Graph.from_csr(xadj, adj, w, lab)
    og = _oracle.Graph(xadj, adj, w, lab)
    starts = at[np.random.RandomState(9).randint(0, len(at), size=70000)].astype(np.int32)
    d_starts = torch.from_numpy(starts).cuda()
    d_paths = torch.empty((70000, 21), dtype=torch.int32, device="cuda")
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    apps = [dict(app=gpu.APP_DEEPWALK), dict(app=gpu.APP_NODE2VEC, p=0.25, q=4.0), dict(app=gpu.APP_METAPATH, schema=[0, 1, 2])]
    refs = []
    for kw in apps:
        par = gpu.default_params(max_depth=21, seed=8, **kw)
        refs.append((par, _oracle.walk(og, _oracle.from_walk_params(par), starts[:5000])[0]))
    errors = []

    def walk(stream, par, ref):
        try:
            st = gpu.WalkStats()
            gpu.check(gpu.lib().fw_walk_device(g.handle, C.byref(par), C.c_void_p(d_starts.data_ptr()), 70000,
                                               C.c_void_p(d_paths.data_ptr()), C.c_void_p(stream.cuda_stream), C.byref(st)))
            assert (d_paths[:5000].cpu().numpy() == ref).all()
        except BaseException as e:  # noqa: B902
            errors.append(e)

    try:
        for i in range(24):
            par, ref = refs[i % 3]
            args = (streams[(i // 2) % 3], par, ref)
            if i % 4 == 3:
                t = threading.Thread(target=walk, args=args)
                t.start()
                t.join()
            else:
                walk(*args)
            assert not errors, (i, errors)
        assert g.engine()[:2] == (gpu.ENGINE_TABLES, 0)
    finally:
        g.destroy()


def test_changed_biases_on_adopted_arrays(gpu):
    """An adopted graph's owner may change the biases between calls: tables and the sets' weights are made anew."""
    csr, at = _lists("even")
    xadj, adj, w = csr
    g, (_, _, dw) = _adopt(gpu, xadj, adj, w)
    rng = np.random.RandomState(8)
    starts = at[rng.randint(0, len(at), size=70000)].astype(np.int32)
    try:
        for i in range(3):
            if i:
                w = np.roll(w, 17)
                dw.copy_(_padded(w))
                torch.cuda.synchronize()
            og = _oracle.Graph(xadj, adj, w)
            for p, q in ((0.25, 4.0), (2.0, 0.5)):
                par = gpu.default_params(app=gpu.APP_NODE2VEC, max_depth=21, p=p, q=q, seed=70 + i)
                ref, _, _ = _oracle.walk(og, _oracle.from_walk_params(par), starts)
                paths, st = g.walk(par, starts)
                assert st.launches >= 6 and g.engine()[:2] == (gpu.ENGINE_TABLES, st.launches - 3)  # tables and sets, or tables made anew
                assert (paths == ref).all()
    finally:
        g.destroy()


def test_small_calls_on_adopted_arrays(gpu):
    """Tables of an adopted graph last one call, so what earlier calls took without them does not pay for them: a loop of small
    calls streams its lists, however long it runs, also after a large call that made them."""
    csr, at = _lists("even")
    g, keep = _adopt(gpu, *csr)
    rng = np.random.RandomState(12)
    og = _oracle.Graph(*csr)
    try:
        for rounds in range(2):
            for i in range(150):
                par = gpu.default_params(app=gpu.APP_NODE2VEC if i % 3 == 0 else gpu.APP_DEEPWALK, max_depth=81, seed=i)
                starts = at[rng.randint(0, len(at), size=100)].astype(np.int32)
                paths, st = g.walk(par, starts)
                assert st.launches == 1, (rounds, i)
                if i % 50 == 0:
                    assert (paths == _oracle.walk(og, _oracle.from_walk_params(par), starts)[0]).all()
            par = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21, seed=5)
            starts = at[rng.randint(0, len(at), size=60000)].astype(np.int32)  # too few to park
            paths, st = g.walk(par, starts)
            assert st.launches == 6
            assert (paths == _oracle.walk(og, _oracle.from_walk_params(par), starts)[0]).all()
    finally:
        g.destroy()


@pytest.mark.parametrize("vertices,hub,n,length,engine", [(300000, 23000, 50000, 20, "STREAM"), (1000000, 100000, 70000, 15, "PARK"),
                                                          (1000000, 100000, 300000, 40, "TABLES"), (40000, 30, 500000, 80, "TABLES")])
def test_first_call_makes_tables_only_for_itself(gpu, vertices, hub, n, length, engine):
    """A first call that takes less without tables than making them takes (0.7 ms of its 0.9, 0.9 ms of its 1.0 in rounds of the
    parking pipeline) goes without; one that takes several times as much makes them, also where all lists are short (3 ms of walks, 0.3 of making)."""
    rng = np.random.RandomState(vertices)
    deg = np.full(vertices, 3, dtype=np.int64)
    deg[rng.permutation(vertices)[:2]] = hub
    xadj = np.zeros(vertices + 1, dtype=np.uint32)
    np.cumsum(deg, out=xadj[1:])
    adj = rng.randint(0, vertices, size=int(xadj[-1])).astype(np.int32)
    w = (1.0 + 99.0 * rng.random_sample(len(adj))).astype(np.float32)
    g = gpu.Graph.from_csr(xadj, adj, w)
    try:
        par = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=length + 1, seed=4)
        starts = rng.randint(0, vertices, size=n).astype(np.int32)
        paths, _ = g.walk(par, starts)
        assert g.engine()[0] == getattr(gpu, "ENGINE_" + engine)
        ref, _, _ = _oracle.walk(_oracle.Graph(xadj, adj, w), _oracle.from_walk_params(par), starts[:2000])
        assert (paths[:2000] == ref).all()
    finally:
        g.destroy()


def test_two_granularities_in_turn(gpu):
    """One set of tables per graph: calls of two granularities in turn replace it only after lists have been streamed for as long as
    making it takes, not in every call."""
    csr, at = _lists("even")
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(14)
    try:
        made = 0
        for i in range(60):
            par = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=81, seed=i, hub_threshold=(16384, 2000)[i & 1])
            starts = at[rng.randint(0, len(at), size=100)].astype(np.int32)
            paths, st = g.walk(par, starts)
            made += st.launches > 3
            assert (paths == _oracle.walk(og, _oracle.from_walk_params(par), starts)[0]).all(), i
        assert 1 <= made <= 15, made
    finally:
        g.destroy()


def test_changed_lists_on_adopted_arrays(gpu):
    """Other lists in the same arrays, longer and shorter ones and other neighbours: the regions are planned anew and the sets too."""
    (xadj, adj, w), at = _lists("even")
    g, (dx, da, dw) = _adopt(gpu, xadj, adj, w)
    rng = np.random.RandomState(13)
    try:
        for i in range(4):
            if i:
                deg = np.roll(np.diff(xadj.astype(np.int64)), 5 + i)[::-1]
                xadj = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32)
                adj = rng.randint(0, V, size=len(adj)).astype(np.int32)
                for v in range(V):
                    adj[xadj[v]:xadj[v + 1]].sort()
                for d, x in ((dx, xadj.view(np.int32)), (da, adj)):
                    d.copy_(_padded(x))
                torch.cuda.synchronize()
            og = _oracle.Graph(xadj, adj, w)
            starts = rng.randint(0, V, size=65000).astype(np.int32)  # too few to park
            starts[::2] = np.argsort(-np.diff(xadj.astype(np.int64)))[:64][rng.randint(0, 64, size=32500)]
            for app, p, q in ((gpu.APP_DEEPWALK, 1.0, 1.0), (gpu.APP_NODE2VEC, 0.25, 4.0), (gpu.APP_NODE2VEC, 2.0, 0.5)):
                par = gpu.default_params(app=app, max_depth=31, p=p, q=q, seed=90 + i)
                ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(par), starts)
                paths, st = g.walk(par, starts)
                assert st.launches >= 6 and g.engine()[0] == gpu.ENGINE_TABLES, (i, app, p)
                assert (paths == ref).all() and (st.steps, st.sampled_edges) == (steps, edges), (i, app, p)
    finally:
        g.destroy()


def test_biases_that_tables_cannot_hold(gpu):
    """A negative bias on an adopted graph (the upload of a host graph refuses it): the streaming kernels say what happens then, and
    later calls do not make tables in vain."""
    (xadj, adj, w), at = _lists("even")
    w = w.copy()
    w[np.random.RandomState(1).randint(0, len(w), size=50)] *= -1.0
    g, keep = _adopt(gpu, xadj, adj, w)
    starts = at[np.random.RandomState(2).randint(0, len(at), size=60000)].astype(np.int32)
    try:
        for i in range(3):
            par = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21, seed=5)
            paths, st = g.walk(par, starts)
            par.park_threshold = -1
            ref, _ = g.walk(par, starts)
            assert (paths == ref).all() and st.launches == 1
    finally:
        g.destroy()


@pytest.mark.parametrize("wg,thr", [(512, 16384), (256, 1024), (1024, 2000), (512, 1 << 30)])
def test_metapath_on_label_tables(gpu, wg, thr):
    """One label to as many as the tables hold, labels that no edge has, other values than 0 .. n; one more label than that
    leaves the tables aside."""
    (xadj, adj, _), at = _lists("even")
    rng = np.random.RandomState(wg + 1)
    values = np.array([7, -3, 0, 1 << 30, 5, 6, -(1 << 31), 11], dtype=np.int64)
    lab = values[np.minimum((rng.exponential(2.0, size=len(adj))).astype(np.int64), 7)].astype(np.int32)
    g = gpu.Graph.from_csr(xadj, adj, None, lab)
    og = _oracle.Graph(xadj, adj, None, lab)
    try:
        cases = [([7, -3, 0], 70000, 10), ([7], 4001, 17), ([-3, 7, 7, 5], 70000, 33), ([-3, 7, 7, 5], 1, 81), ([-3, 7, 7, 5], 777, 2),
                 ([7, -3, 0, 1 << 30, 5, 6, -(1 << 31), 11], 70000, 12), ([99, 7], 70000, 5), ([7, -3, 7, 99, 0], 70000, 9),
                 (list(values) + [99], 70000, 20)]
        for i, (schema, n, depth) in enumerate(cases):
            p = gpu.default_params(app=gpu.APP_METAPATH, max_depth=depth, schema=schema, wg_threads=wg, hub_threshold=thr,
                                   seed=300 + i, walker_base=i)
            starts = np.where(rng.random_sample(n) < 0.8, at[rng.randint(0, len(at), size=n)], rng.randint(0, V, size=n)).astype(np.int32)
            ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(p), starts)
            launches = set()
            for _ in range(20):  # the first calls with a schema may walk without tables
                paths, st = g.walk(p, starts)
                bad = np.nonzero((paths != ref).any(axis=1))[0]
                assert len(bad) == 0, (schema, n, bad[0], paths[bad[0]], ref[bad[0]])
                assert (st.steps, st.sampled_edges) == (steps, edges), (schema, n)
                launches.add(st.launches)
                if 6 in launches:
                    break
            assert (6 in launches) == (i not in (3, 4, 8)), (i, launches)  # made; there already (twice); too many labels
            again, st2 = g.walk_batch(p, starts, batch_size=max(1, n // 3))
            assert (again == ref).all() and (st2.steps, st2.sampled_edges) == (steps, edges), (schema, n)
    finally:
        g.destroy()


@pytest.mark.parametrize("grid,n,depth", [(1, 4097 + 64, 6), (1, 9001, 16), (2, 20000, 2), (3, 13001, 17)])
def test_short_rows_of_many_queries(gpu, grid, n, depth):
    """Rows of at most 16 entries: queries come 256 at a time while 1024 per workgroup are left, 64 at a time after that."""
    csr, at = _lists("even")
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(n)
    try:
        warm = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21)
        g.walk(warm, at[rng.randint(0, len(at), size=70000)].astype(np.int32))
        for app in (gpu.APP_DEEPWALK, gpu.APP_PPR):
            p = gpu.default_params(app=app, max_depth=depth, tp=0.3, seed=n, grid=grid)
            starts = rng.randint(0, V, size=n).astype(np.int32)
            ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(p), starts)
            paths, st = g.walk(p, starts)
            assert st.launches == 3
            bad = np.nonzero((paths != ref).any(axis=1))[0]
            assert len(bad) == 0, (app, bad[0], paths[bad[0]], ref[bad[0]])
            assert (st.steps, st.sampled_edges) == (steps, edges)
    finally:
        g.destroy()


@pytest.mark.parametrize("depth", [17, 31, 32, 33, 65, 100])
def test_rows_end_anywhere_in_a_line(gpu, depth):
    """Rows that begin and end at every place of a 64-byte line, walks of one entry to all of them, many that end together; nothing is
    stored before the matrix or behind it."""
    csr, at = _lists("uneven")
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(depth)
    n = 3001
    try:
        g.walk(gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21), at[rng.randint(0, len(at), size=70000)].astype(np.int32))
        starts = np.where(rng.random_sample(n) < 0.5, at[rng.randint(0, len(at), size=n)], rng.randint(0, V, size=n)).astype(np.int32)
        starts_dev = torch.from_numpy(starts).cuda()
        for app, tp, before in ((gpu.APP_PPR, 0.3, 0), (gpu.APP_PPR, 0.03, 7), (gpu.APP_DEEPWALK, 0.0, 5)):
            p = gpu.default_params(app=app, max_depth=depth, tp=tp, seed=depth, grid=2)
            ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(p), starts)
            room = torch.full((before + n * depth + 32,), 12345, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            st = gpu.WalkStats()
            gpu.check(gpu.lib().fw_walk_device(g.handle, C.byref(p), C.c_void_p(starts_dev.data_ptr()), n,
                                               C.c_void_p(room.data_ptr() + 4 * before), None, C.byref(st)))
            assert g.engine()[0] == gpu.ENGINE_TABLES
            out = room.cpu().numpy()
            paths = out[before:before + n * depth].reshape(n, depth)
            bad = np.nonzero((paths != ref).any(axis=1))[0]
            assert len(bad) == 0, (app, before, bad[0], paths[bad[0]], ref[bad[0]])
            assert (out[:before] == 12345).all() and (out[before + n * depth:] == 12345).all()
            assert (st.steps, st.sampled_edges) == (steps, edges)
    finally:
        g.destroy()


@pytest.mark.parametrize("depth", [17, 32, 33, 65])
def test_node2vec_rows_end_anywhere_in_a_line(gpu, depth):
    """As above for node2vec, whose walkers turn down proposals and come to the ends of their lines and rows at different times."""
    csr, at = _lists("uneven")
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(depth)
    n = 1501
    try:
        g.walk(gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21), at[rng.randint(0, len(at), size=70000)].astype(np.int32))
        starts = np.where(rng.random_sample(n) < 0.5, at[rng.randint(0, len(at), size=n)], rng.randint(0, V, size=n)).astype(np.int32)
        starts_dev = torch.from_numpy(starts).cuda()
        p = gpu.default_params(app=gpu.APP_NODE2VEC, max_depth=depth, p=2.0, q=0.5, seed=depth, grid=2)
        ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(p), starts)
        for before in (0, 7):
            room = torch.full((before + n * depth + 32,), 12345, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            st = gpu.WalkStats()
            gpu.check(gpu.lib().fw_walk_device(g.handle, C.byref(p), C.c_void_p(starts_dev.data_ptr()), n,
                                               C.c_void_p(room.data_ptr() + 4 * before), None, C.byref(st)))
            assert g.engine()[0] == gpu.ENGINE_TABLES and st.grid == 2
            out = room.cpu().numpy()
            paths = out[before:before + n * depth].reshape(n, depth)
            bad = np.nonzero((paths != ref).any(axis=1))[0]
            assert len(bad) == 0, (before, bad[0], paths[bad[0]], ref[bad[0]])
            assert (out[:before] == 12345).all() and (out[before + n * depth:] == 12345).all()
            assert (st.steps, st.sampled_edges) == (steps, edges)
    finally:
        g.destroy()


@pytest.mark.parametrize("two_groups", [False, True])
def test_node2vec_of_few_walkers_on_short_lists(gpu, two_groups):
    """Lists of one group: up to where a wave walks each follows from how many proposals are turned down (waves per SIMD: 4 without adjacency tests, 5 where
    some list has two groups, 6 for q < 1, 8 for q > 1); either side of it the oracle's walks."""
    simds = 4 * torch.cuda.get_device_properties(0).multi_processor_count
    rng = np.random.RandomState(8)
    deg = rng.randint(1, 100, size=4000)
    if two_groups:
        deg[17] = 1500
    xadj = np.zeros(len(deg) + 1, dtype=np.uint32)
    np.cumsum(deg, out=xadj[1:])
    adj = np.concatenate([np.sort(rng.randint(0, len(deg), size=d)) for d in deg]).astype(np.int32)
    w = (1.0 + 9.0 * rng.random_sample(len(adj))).astype(np.float32)
    g = gpu.Graph.from_csr(xadj, adj, w)
    og = _oracle.Graph(xadj, adj, w)
    try:
        for _ in range(30):
            g.walk(gpu.default_params(app=gpu.APP_NODE2VEC, max_depth=41), rng.randint(0, len(deg), size=70000).astype(np.int32))
        for p, q, waves in ((1.0, 1.0, 4 + two_groups), (0.25, 1.0, 4 + two_groups), (2.0, 0.5, 8 if two_groups else 6), (0.25, 4.0, 8)):
            for n in (waves * simds, waves * simds + 1):
                par = gpu.default_params(app=gpu.APP_NODE2VEC, max_depth=9, p=p, q=q, seed=n)
                starts = rng.randint(0, len(deg), size=n).astype(np.int32)
                ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(par), starts)
                paths, st = g.walk(par, starts)
                assert g.engine()[0] == gpu.ENGINE_TABLES
                assert (paths == ref).all() and (st.steps, st.sampled_edges) == (steps, edges), (p, q, n)
                assert (st.grid == (n + 3) // 4) == (n == waves * simds), (p, q, n, st.grid)
    finally:
        g.destroy()

# Calls of at most 8,192 walkers take a wave for each (fw_table_walk_wave), unless they give a grid: then a lane walks each.
def _compare(gpu, g, og, starts, p, what):
    ref, steps, edges = _oracle.walk(og, _oracle.from_walk_params(p), starts)
    paths, st = g.walk(p, starts)
    assert g.engine()[0] == gpu.ENGINE_TABLES, what
    bad = np.nonzero((paths != ref).any(axis=1))[0]
    assert len(bad) == 0, (what, bad[0], paths[bad[0]], ref[bad[0]])
    assert (st.steps, st.sampled_edges) == (steps, edges), what
    return st


@pytest.mark.parametrize("kind", ["even", "uneven"])
@pytest.mark.parametrize("wg,thr", [(512, 16384), (256, 1024), (1024, 2000), (512, 1 << 30)])
def test_lane_per_walker_with_few_walkers(gpu, kind, wg, thr):
    """The shapes of test_walks_on_tables that a wave per walker takes there, by the kernel of a lane per walker; with the grid left to the library, the other."""
    csr, at = _lists(kind)
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(wg)
    try:
        g.walk(gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21, wg_threads=wg, hub_threshold=thr), at[rng.randint(0, len(at), size=70000)].astype(np.int32))
        cases = [(dict(app=gpu.APP_DEEPWALK, max_depth=depth), n)
                 for n, depth in ((1, 81), (63, 2), (65, 15), (1000, 16), (777, 17), (4001, 33), (3, 1), (129, 100))]
        cases.append((dict(app=gpu.APP_PPR, max_depth=50, tp=0.1), 3000))
        for p, q in ((2.0, 0.5), (0.25, 4.0), (4.0, 0.25), (1.0, 1.0), (0.1, 1.0)):
            cases.append((dict(app=gpu.APP_NODE2VEC, max_depth=18, p=p, q=q), 2000))
        for i, (kw, n) in enumerate(cases):
            starts = np.where(rng.random_sample(n) < 0.8, at[rng.randint(0, len(at), size=n)], rng.randint(0, V, size=n)).astype(np.int32)
            if n > 100:
                starts[5] = -1
                starts[7] = V
            for grid in (2, 0):
                st = _compare(gpu, g, og, starts, gpu.default_params(wg_threads=wg, hub_threshold=thr, seed=100 + i, walker_base=i, grid=grid, **kw), (kw, n, grid))
                assert st.grid == (grid if grid else (n + 3) // 4)
    finally:
        g.destroy()


@pytest.mark.parametrize("kind", ["even", "uneven"])
@pytest.mark.parametrize("wg,thr", [(512, 16384), (1024, 2000)])
def test_node2vec_on_hash_sets_a_lane_per_walker(gpu, kind, wg, thr):
    """test_node2vec_on_hash_sets by the kernel of a lane per walker: buckets that overflow, sets with and without weights."""
    csr, at = _lists(kind)
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(7)
    try:
        g.walk(gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21, wg_threads=wg, hub_threshold=thr), at[rng.randint(0, len(at), size=70000)].astype(np.int32))
        for i, (p, q) in enumerate(((2.0, 0.5), (0.25, 4.0), (4.0, 0.25), (1.0, 1.0), (0.1, 1.0), (1.0, 3.0), (0.5, 0.25))):
            starts = at[rng.randint(0, len(at), size=400)].astype(np.int32)
            par = gpu.default_params(app=gpu.APP_NODE2VEC, max_depth=101, p=p, q=q, seed=50 + i, wg_threads=wg, hub_threshold=thr, grid=2)
            st = _compare(gpu, g, og, starts, par, (p, q))
            assert st.grid == 2
            assert st.launches == (5 if i < 2 else 3)  # as there
    finally:
        g.destroy()


def test_which_kernel_walks_on_tables(gpu):
    """A wave per walker up to as many walkers as there are waves resident (32 per compute unit), a lane for each beyond; MetaPath always the latter."""
    most = 32 * torch.cuda.get_device_properties(0).multi_processor_count
    csr, at = _lists("even")
    xadj, adj, w = csr
    g = gpu.Graph.from_csr(xadj, adj, w, np.random.RandomState(1).randint(0, 5, size=len(adj)).astype(np.int32))
    rng = np.random.RandomState(2)
    try:
        for kw in (dict(app=gpu.APP_DEEPWALK, max_depth=21), dict(app=gpu.APP_PPR, max_depth=21, tp=0.1), dict(app=gpu.APP_NODE2VEC, max_depth=21, p=2.0, q=0.5),
                   dict(app=gpu.APP_METAPATH, max_depth=21)):
            p = gpu.default_params(**kw)
            for _ in range(20):
                g.walk(p, at[rng.randint(0, len(at), size=70000)].astype(np.int32))
            for n in (most, most + 1):
                _, st = g.walk(p, at[rng.randint(0, len(at), size=n)].astype(np.int32))
                assert g.engine()[0] == gpu.ENGINE_TABLES
                assert (st.grid == (n + 3) // 4) == (n == most and kw["app"] != gpu.APP_METAPATH), (kw, n, st.grid)
    finally:
        g.destroy()


@pytest.mark.parametrize("few,side", [(14, "front"), (14, "back"), (14, "middle"), (5, "front"), (5, "back"), (5, "middle")])
@pytest.mark.parametrize("wg,thr", [(512, 16384), (256, 1024)])
def test_groups_with_a_lump(gpu, few, side, wg, thr):
    """Weights evenly spread over most lanes of a group, while the share of `few` of 64 lies in one of them.  Of five, no more than two lanes of a full group end beyond three
    blocks of where even weights would have them: it is searched from the guess on, the element up to six blocks off.  Of fourteen it is entered through its row."""
    V = 400
    rng = np.random.RandomState(8)
    deg = np.r_[rng.randint(60, 70, size=100), rng.randint(120, 260, size=100), rng.randint(500, 1100, size=196), [2500, 4096, 9001, 20000]]
    xadj = np.zeros(V + 1, dtype=np.uint32)
    np.cumsum(deg, out=xadj[1:])
    adj = np.concatenate([np.sort(rng.randint(0, V, size=d)) for d in deg]).astype(np.int32)
    w = (1.0 + 4.0 * rng.random_sample(len(adj))).astype(np.float32)
    for v in range(V):
        i = np.arange(xadj[v], xadj[v + 1])
        lane = ((i >> 2) - (int(xadj[v]) >> 2)) % 64  # of the group's quartets lane, lane + 64, ..
        lanes = min(64, len(i) // 4)
        poor_lanes = max(2, lanes * few // 64)
        lo = {"front": 0, "back": lanes - poor_lanes, "middle": (lanes - poor_lanes) // 2}[side]
        first = {"front": 0, "back": lanes - 1, "middle": lo + v % poor_lanes}[side]
        poor = (lane != first) & (lane >= lo) & (lane < lo + poor_lanes)
        w[i[poor]] = 0.001
        w[i[lane == first]] *= poor_lanes
    g = gpu.Graph.from_csr(xadj, adj, w)
    og = _oracle.Graph(xadj, adj, w)
    try:
        g.walk(gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21, wg_threads=wg, hub_threshold=thr), rng.randint(0, V, size=70000).astype(np.int32))
        for kw in (dict(app=gpu.APP_DEEPWALK, max_depth=20), dict(app=gpu.APP_PPR, max_depth=30, tp=0.1), dict(app=gpu.APP_NODE2VEC, max_depth=12, p=0.25, q=4.0)):
            for grid, n in ((2, 3000), (0, 3000), (0, 9000)):  # full waves of walkers, a wave per walker, a few walkers in each wave
                starts = rng.randint(0, V, size=n).astype(np.int32)
                st = _compare(gpu, g, og, starts, gpu.default_params(wg_threads=wg, hub_threshold=thr, seed=n, grid=grid, **kw), (few, side, kw, grid, n))
                assert st.grid == grid if grid else (st.grid == (n + 3) // 4) == (n == 3000)
    finally:
        g.destroy()


def _with_vertices(csr, more):
    """The graph and `more` vertices of one edge each into it: a block of the tables' regions each."""
    xadj, adj, w = csr
    rng = np.random.RandomState(5)
    n = len(xadj) - 1
    return (np.concatenate([xadj, (len(adj) + 1 + np.arange(more)).astype(np.uint32)]), np.concatenate([adj, rng.randint(0, n, size=more).astype(np.int32)]),
            np.concatenate([w, (1.0 + 4.0 * rng.random_sample(more)).astype(np.float32)]))


@pytest.mark.parametrize("kind", ["even", "uneven"])
@pytest.mark.parametrize("more,wg,thr", [(0, 512, 16384), (300000, 512, 16384), (300000, 1024, 2000)])
def test_lists_of_every_shape_in_regions_of_every_size(gpu, more, kind, wg, thr):
    """Rows of groups are read in one way up to 32 MiB of regions, or by waves of few walkers, and in another beyond that (300,000 vertices more are 38 MB)."""
    csr, at = _lists(kind)
    csr = _with_vertices(csr, more)
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(more + wg)
    try:
        p = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=21, wg_threads=wg, hub_threshold=thr)
        for _ in range(40):
            g.walk(p, at[rng.randint(0, len(at), size=70000)].astype(np.int32))
            if g.engine()[0] == gpu.ENGINE_TABLES:
                break
        assert (g.engine()[2] > 38000000) == (more != 0)
        cases = [dict(app=gpu.APP_DEEPWALK, max_depth=40), dict(app=gpu.APP_PPR, max_depth=40, tp=0.1), dict(app=gpu.APP_NODE2VEC, max_depth=20, p=2.0, q=0.5),
                 dict(app=gpu.APP_NODE2VEC, max_depth=20, p=0.1, q=1.0)]
        for i, kw in enumerate(cases):
            for grid, n in ((3, 4000), (0, 9001)):
                starts = np.where(rng.random_sample(n) < 0.8, at[rng.randint(0, len(at), size=n)], rng.randint(0, V + more, size=n)).astype(np.int32)
                st = _compare(gpu, g, og, starts, gpu.default_params(wg_threads=wg, hub_threshold=thr, seed=30 + i, walker_base=i, grid=grid, **kw), (kw, grid, n))
                assert st.grid == grid or (grid == 0 and st.grid != (n + 3) // 4)
    finally:
        g.destroy()


@pytest.mark.parametrize("kind", ["even", "uneven"])
@pytest.mark.parametrize("wg,thr", [(512, 16384), (1024, 2000)])
def test_lists_of_every_shape_in_gigabytes_of_regions(gpu, kind, wg, thr):
    """From 2 GiB of regions on (2^24 vertices more) and 2^19 walkers on, DeepWalk and node2vec do not keep blocks of pairs and read them by eight lanes: every row against calls of
    half as many walkers, which keep them (node2vec when it has its hash sets), some against the oracle.  PPR keeps them."""
    csr, at = _lists(kind)
    more = 1 << 24
    csr = _with_vertices(csr, more)
    g = gpu.Graph.from_csr(*csr)
    og = _oracle.Graph(*csr)
    rng = np.random.RandomState(wg)
    n = (1 << 19) + 333
    half = n // 2
    starts = np.where(rng.random_sample(n) < 0.8, at[rng.randint(0, len(at), size=n)], rng.randint(0, V + more, size=n)).astype(np.int32)
    try:
        p = gpu.default_params(app=gpu.APP_DEEPWALK, max_depth=41, wg_threads=wg, hub_threshold=thr)
        for _ in range(60):
            g.walk(p, starts)
            if g.engine()[0] == gpu.ENGINE_TABLES:
                break
        assert g.engine()[2] > 2 << 30
        for i, kw in enumerate((dict(app=gpu.APP_DEEPWALK, max_depth=20), dict(app=gpu.APP_DEEPWALK, max_depth=7), dict(app=gpu.APP_PPR, max_depth=30, tp=0.1),
                                dict(app=gpu.APP_NODE2VEC, max_depth=12, p=2.0, q=0.5), dict(app=gpu.APP_NODE2VEC, max_depth=12, p=0.1, q=4.0))):
            for grid in (0, 7):
                p = gpu.default_params(wg_threads=wg, hub_threshold=thr, seed=60 + i, grid=grid, **kw)
                paths, st = g.walk(p, starts)
                assert g.engine()[0] == gpu.ENGINE_TABLES and grid in (0, st.grid)
                steps = edges = 0
                for a, b in ((0, half), (half, n)):
                    p.walker_base = a
                    ref, s = g.walk(p, starts[a:b])
                    assert (paths[a:b] == ref).all(), (kw, grid, a)
                    steps, edges = steps + s.steps, edges + s.sampled_edges
                assert (st.steps, st.sampled_edges) == (steps, edges)
            for a in (0, half - 500, n - 1500):
                p.walker_base = a
                ref, _, _ = _oracle.walk(og, _oracle.from_walk_params(p), starts[a:a + 1500])
                assert (paths[a:a + 1500] == ref).all(), (kw, a)
    finally:
        g.destroy()
