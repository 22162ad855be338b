"""The coarse level of the boundary index (fastapsp_amd/csrc/hindex.hip): its host code, compiled as it
is against a host-only stand-in of the HIP runtime and CPU emulations of its kernels
(tests/cpp/hidx_host), under -fsanitize=address,undefined.  Rows equal to Dijkstra, with the level, with
its workspace refused, and on graphs that get none."""

import os
import shutil
import subprocess

import numpy as np
import pytest

import fastapsp_amd as fa
from fastapsp_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def graph(kind):
    if kind == "grid":
        u, v, w = synth.grid_graph(34, 34, 0.10, 0.02, 1, 100, 3)
        return (*synth.to_csr(1156, u, v, w, False), 33, True)
    if kind == "two grids":  # the second without an arc to the first
        u, v, w = synth.grid_graph(24, 24, 0.05, 0.0, 1, 50, 4)
        u, v, w = np.concatenate([u, u + 576]), np.concatenate([v, v + 576]), np.concatenate([w, w])
        return (*synth.to_csr(1152, u, v, w, False), 36, True)
    if kind == "few parts":
        u, v, w = synth.grid_graph(20, 20, 0.05, 0.02, 1, 50, 5)
        return (*synth.to_csr(400, u, v, w, False), 12, False)
    rng = np.random.default_rng(6)  # no locality: most boundary vertices would be a region's
    u, v = rng.integers(0, 160, 600), rng.integers(0, 160, 600)
    key = np.unique(np.minimum(u, v) * 160 + np.maximum(u, v))
    u, v = key // 160, key % 160
    u, v = u[u != v], v[u != v]
    return (*synth.to_csr(160, u, v, rng.integers(1, 9, u.size).astype(np.int32), False), 40, False)


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    tmp = tmp_path_factory.mktemp("hidx_host")
    csrc = os.path.join(ROOT, "fastapsp_amd", "csrc")
    cpp = os.path.join(ROOT, "tests", "cpp")
    src = open(os.path.join(csrc, "bindex.hip")).read()
    a, b = src.index("struct BidxPart {"), src.index("namespace fapk {")
    c = src.index("namespace fapi {\n\nnamespace {\n\nvoid free_bidx")
    (tmp / "bindex_host.inc").write_text(src[a:b] + '\n#include "emu_kernels.h"\n' + src[c:])
    src = open(os.path.join(csrc, "hindex.hip")).read()
    a, b = src.index("struct HidxRegion {"), src.index("namespace fapk {")
    c = src.index("namespace fapi {\n\nnamespace {")
    (tmp / "hindex_host.inc").write_text(src[a:b] + '\n#include "emu_coarse.h"\n' + src[c:])
    objs = []
    for name in ("tests/cpp/bidx_host/fw_emu.cpp", "fastapsp_amd/csrc/partition.cpp"):
        objs.append(str(tmp / os.path.basename(name)) + ".o")
        r = subprocess.run([gxx, "-std=c++17", "-O2", "-I" + os.path.join(ROOT, "include"), "-I" + csrc, "-c",
                            os.path.join(ROOT, name), "-o", objs[-1]], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-3000:]
    exe = str(tmp / "hidx_host")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                        "-fno-sanitize-recover=undefined", "-I" + os.path.join(cpp, "bidx_host", "mock"),
                        "-I" + os.path.join(cpp, "bidx_host"), "-I" + os.path.join(cpp, "hidx_host"),
                        "-I" + str(tmp), "-I" + os.path.join(ROOT, "include"), "-I" + csrc,
                        os.path.join(cpp, "hidx_host", "harness.cpp"), *objs, "-ldl", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


@pytest.mark.parametrize("kind", ["grid", "two grids", "few parts", "random"])
def test_rows_through_the_coarse_level(harness, tmp_path, kind):
    ro, col, wt, K, coarse = graph(kind)
    V = ro.size - 1
    with fa.Graph.from_csr(ro, col, wt.astype(np.float32), K) as g:
        g.preCondition()
        vn, vo, bn, _ = g.part_info()
        st2ed, gid = g.getMapping(), g.getGraphId()
    ed2st = np.empty(V, np.int32)
    ed2st[st2ed] = np.arange(V, dtype=np.int32)
    path = str(tmp_path / "graph.bin")
    with open(path, "wb") as f:
        np.array([V, len(col), K], np.int64).tofile(f)
        for a in (ro, col, wt, gid, st2ed, ed2st, vn, vo, bn):
            np.asarray(a, np.int32).tofile(f)
    r = subprocess.run([harness, path, str(int(coarse))], capture_output=True, text=True, timeout=600,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]
    assert "0 bad" in r.stdout and "runtime error" not in r.stderr, r.stdout + r.stderr
