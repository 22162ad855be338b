"""Batched part solves whose products are too large to share a launch: with a part's vertices near in
number their scatters share one, otherwise each follows its part's product.  Rows equal to the parts
solved one by one without the index."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["near", "apart"])
def test_scatter_routes(gpu_ctx, kind):
    import fastapsp_amd as fa
    from fastapsp_amd import synth
    side, K = 132, 34
    V = side * side
    u, v, w = synth.grid_graph(side, side, 0.10, 0.02, 1, 100, 3)
    if kind == "apart":
        name = np.random.default_rng(5).permutation(V)
        u, v = name[u], name[v]
    ro, col, w = synth.to_csr(V, u, v, w, False)
    with fa.Graph.from_csr(ro, col, w.astype(np.float32), K) as g:
        g.preCondition()
        n, off, b, _ = g.part_info()
        st2ed, gid = g.getMapping(), g.getGraphId()
    ed2st = np.empty_like(st2ed)
    ed2st[st2ed] = np.arange(V, dtype=np.int32)
    dg = gpu_ctx.upload_graph(ro, col, w)
    dg.set_partition(gid, st2ed, ed2st)
    ids = [1, 2, K]
    assert all((n[p] - b[p] + 127) // 128 * ((V + 127) // 128) >= 512 for p in ids)
    outs = [gpu_ctx.alloc((int(n[p]), V)) for p in ids]
    dg.subgraph_solve_batch([int(off[p]) for p in ids], [int(n[p]) for p in ids],
                            [int(b[p]) for p in ids], [o.ptr for o in outs], V)
    one = [gpu_ctx.alloc((int(n[p]), V)) for p in ids]
    for p, o, c in zip(ids, outs, one):
        dg.subgraph_solve(int(off[p]), int(n[p]), int(b[p]), c.ptr, V)
        gpu_ctx.sync()
        np.testing.assert_array_equal(o.get(), c.get())
    for o in outs + one:
        o.free()
    dg.close()
