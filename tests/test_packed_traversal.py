"""The packed traversal tree and its traversal code against brute force, on the host CPU
(tests/cpp/packed_traversal_check.cpp): layouts whose leaves hold one primitive to many nodes, a
single-leaf tree, a scene away from the origin, the benchmark heightfield's size, and combs whose
stacks reach past the LDS entries into the spill area.  Results are exact: the traversal only has to
reach every primitive the ray hits, and the primitive test decides."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "naivetrace_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    from naivetrace_amd import build
    exe = str(tmp_path_factory.mktemp("packed") / "packed_traversal_check")
    subprocess.run([build.hipcc(), "-O2", "-std=c++17", "-x", "hip", f"--offload-arch={build.ARCH}", "-Wno-unused-result",
                    os.path.join(ROOT, "tests", "cpp", "packed_traversal_check.cpp"), os.path.join(CSRC, "bvh_build.cpp"),
                    "-o", exe, "-lpthread"], check=True, capture_output=True)
    return exe


def run(program, *args):
    r = subprocess.run([program, *map(str, args)], capture_output=True, text=True, timeout=300)
    print(r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
    f = r.stdout.split()
    return lambda k: int(f[f.index(k) + 1])


@pytest.mark.parametrize("grid,offset,rays", [(1, 0.0, 2000), (2, 0.0, 5000), (7, 0.0, 20000), (60, 0.0, 40000), (80, 5000.0, 40000),
                                              (512, 0.0, 16000)])
def test_packed_traversal_matches_brute_force(program, grid, offset, rays):
    val = run(program, grid, offset, rays)
    assert val("box_errors") == 0 and val("layout_errors") == 0
    assert val("hits") > (10 if grid < 7 else 300)
    for k in ("closest_diff", "prim_diff", "anyhit_diff", "short_stack_diff"):
        assert val(k) == 0, k


def test_packed_traversal_spills_its_stack(program):
    val = run(program, 400, 0.0, 300, "comb")
    assert val("max_stack") > val("lds_stack")
    for k in ("closest_diff", "prim_diff", "anyhit_diff", "short_stack_diff"):
        assert val(k) == 0, k


def test_packed_traversal_with_spheres(program):
    """Sphere records (stored unpermuted, hit distances in FP64) among the triangles."""
    val = run(program, 60, 0.0, 40000, "spheres")
    assert val("box_errors") == 0 and val("layout_errors") == 0
    assert val("sphere_hits") > 50
    for k in ("closest_diff", "prim_diff", "anyhit_diff", "short_stack_diff"):
        assert val(k) == 0, k
