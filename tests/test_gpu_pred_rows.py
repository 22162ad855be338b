"""Predecessor rows: each way the kernel reads in-neighbours (GPU), against the tight arcs themselves."""
import numpy as np
import pytest

import oracle_lib as O
from fastapsp_amd import INF, synth

pytestmark = pytest.mark.gpu


# Neighbours within a stretch of the row (read from LDS), just past its length,
# anywhere; 4, 6, 8 and more in-arcs; fewer vertices than a stretch; parallel
# arcs; odd row strides; one and many rows.
@pytest.mark.parametrize("V,span,degree", [(1, 0, 0), (3, 2, 3), (700, 40, 4), (1025, 1023, 6),
                                           (5000, 900, 4), (5000, 1200, 8), (9001, 9000, 5),
                                           (5000, 300, 12), (2048, 2047, 40)])
@pytest.mark.parametrize("nrows", [1, 37, 1500])
def test_pred_rows_valid_everywhere(gpu_ctx, V, span, degree, nrows):
    rng = np.random.default_rng(V + degree)
    to = np.repeat(np.arange(V), degree)
    frm = np.clip(to + rng.integers(-span, span + 1, to.size), 0, V - 1)
    keep = frm != to
    ro, col, w = synth.to_csr(V, frm[keep], to[keep], rng.integers(1, 30, to.size)[keep], True)
    if nrows * V > 8 << 20:
        nrows = (8 << 20) // V  # past the few-cells kernel all the same
    own = rng.integers(0, V, nrows).astype(np.int32)
    d = O.batched_sssp(own, ro, col, w)
    ld, ldp = V + 3, V + 1
    dist = np.full((nrows, ld), -5, np.int32)
    dist[:, :V] = d
    dg = gpu_ctx.upload_graph(ro, col, w)
    dd, do = gpu_ctx.to_device(dist), gpu_ctx.to_device(own)
    dp = gpu_ctx.to_device(np.full((nrows, ldp), -9, np.int32))
    dg.pred_rows(dd.ptr, ld, do.ptr, nrows, dp.ptr, ldp)
    got = dp.get()
    assert (got[:, V:] == -9).all()
    # the smallest in-neighbour that is tight
    want = np.full((nrows, V), V, np.int64)
    src = np.repeat(np.arange(V), np.diff(ro))
    for i in range(nrows):
        tight = (d[i, src].astype(np.int64) + w == d[i, col]) & (d[i, src] < INF)
        np.minimum.at(want[i], col[tight], src[tight])
        want[i, d[i] >= INF] = -1
        want[i, own[i]] = own[i]
    np.testing.assert_array_equal(got[:, :V], want)
    dg.close()
