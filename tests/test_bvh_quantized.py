"""The surface BVH's 8-bit child planes (64-byte nodes) on the host: the traversal source of the kernels
(naivetrace_amd/csrc/trace.hpp) compiled for the CPU by hipcc (tests/cpp/packed_traversal_check.cpp).
Decoded boxes contain the true ones with room to spare; the packed tree gives exactly the brute-force
closest hit and any-hit answer, and so does a plain descent of the tree's float planes.  Far from the
origin (x = -1e6, unit triangles, float spacing 1/16) the slab test cancels (as in the reference's
non-robust Embree mode); the packed tree, whose boxes are slightly larger, loses no more hits than the
float planes.  At 512 x 512 cells (the benchmark's heightfield size, 655k triangles) they still agree
exactly.  A "comb" of thin triangles whose boxes all contain an axis the triangles leave free, spaced so
that the binned SAH builds an unbalanced tree, drives rays along that axis through every node: the
deepest stacks reach past the LDS part of the traversal stack into its private spill area (kLdsStack
entries), and the results stay exact with no overflow.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "naivetrace_amd", "csrc")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    from naivetrace_amd import build
    exe = str(tmp_path_factory.mktemp("qbvh") / "packed_traversal_check")
    subprocess.run([build.hipcc(), "-O2", "-std=c++17", "-x", "hip", f"--offload-arch={build.ARCH}", "-Wno-unused-result",
                    os.path.join(ROOT, "tests", "cpp", "packed_traversal_check.cpp"), os.path.join(CSRC, "bvh_build.cpp"),
                    "-o", exe, "-lpthread"], check=True, capture_output=True)
    return exe


@pytest.mark.parametrize("grid,offset,exact", [(60, 0.0, True), (80, 5000.0, True), (8, -1e6, False), (512, 0.0, True)])
def test_quantized_bvh_matches_brute_force(checker, grid, offset, exact):
    rays = "16000" if grid >= 512 else "40000"
    r = subprocess.run([checker, str(grid), str(offset), rays], capture_output=True, text=True, timeout=300)
    print(r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
    f = r.stdout.split()
    val = lambda k: int(f[f.index(k) + 1])
    assert val("box_errors") == 0 and val("layout_errors") == 0
    assert val("hits") > 500
    if exact:
        for k in ("closest_diff", "prim_diff", "anyhit_diff", "full_closest_diff"):
            assert val(k) == 0, k
    else:
        assert val("closest_diff") <= val("full_closest_diff")
        assert val("anyhit_diff") <= val("full_closest_diff")
        assert val("closest_diff") < 0.01 * val("rays")


@pytest.mark.parametrize("teeth_k,rays", [(100, 300), (400, 300)])
def test_deep_tree_uses_stack_spill_exactly(checker, teeth_k, rays):
    r = subprocess.run([checker, str(teeth_k), "0", str(rays), "comb"], capture_output=True, text=True, timeout=300)
    print(r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
    f = r.stdout.split()
    val = lambda k: int(f[f.index(k) + 1])
    assert val("overflows") == 0
    assert val("max_stack") > val("lds_stack")  # the private spill area was used
    assert val("hits") > 50
    for k in ("closest_diff", "prim_diff", "anyhit_diff", "full_closest_diff"):
        assert val(k) == 0, k


@pytest.fixture(scope="module")
def watertight_checker(tmp_path_factory):
    from naivetrace_amd import build
    exe = str(tmp_path_factory.mktemp("wt") / "watertight_check")
    # Multiply-adds contracted as in the device build (-ffp-contract=fast-honor-pragmas), with FMA
    # instructions on the host, so the slab tests round the way the kernels' do.
    subprocess.run([build.hipcc(), "-O2", "-std=c++17", "-x", "hip", f"--offload-arch={build.ARCH}", "-Wno-unused-result",
                    "-ffp-contract=fast-honor-pragmas", "-Xarch_host", "-mfma",
                    os.path.join(ROOT, "tests", "cpp", "watertight_check.cpp"), os.path.join(CSRC, "bvh_build.cpp"),
                    "-o", exe, "-lpthread"], check=True, capture_output=True)
    return exe


@pytest.mark.parametrize("freq", [3, 12])
def test_rays_at_shared_edges_and_vertices_hit(watertight_checker, tmp_path, freq):
    """Rays aimed at the vertices and edge points of a closed icosphere from inside: the watertight
    triangle test and the packed traversal's slab tests (margins of the planes, distances widened by
    their rounding error) leave no gap, for closest-hit and any-hit queries and in a brute-force loop,
    and the closest hit is the loop's."""
    import numpy as np
    from naivetrace_amd import configs
    from test_gpu_trace import _edge_rays
    v, f = configs.icosphere(freq)
    v = (v * 3.7 + np.array([10.3, -2.1, 5.9])).astype(np.float32)
    c = v.mean(axis=0)
    org, d = _edge_rays(v, f, [c, c + [0.9, -0.4, 1.3], c + [-2.1, 1.7, 0.2]])
    path = tmp_path / "rays.bin"
    with open(path, "wb") as fo:
        np.array([len(v), len(f), len(org)], np.int32).tofile(fo)
        v.tofile(fo)
        f.astype(np.int32).tofile(fo)
        org.astype(np.float32).tofile(fo)
        d.astype(np.float32).tofile(fo)
    r = subprocess.run([watertight_checker, str(path)], capture_output=True, text=True, timeout=300)
    print(r.stdout.strip())
    assert r.returncode == 0, r.stderr
    f_ = r.stdout.split()
    assert int(f_[f_.index("rays") + 1]) == len(org)
    for k in ("packed", "anyhit", "brute", "distance"):
        assert int(f_[f_.index(k) + 2]) == 0, k
