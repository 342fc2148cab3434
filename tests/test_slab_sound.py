"""The slab test of the silhouette search (geom.hpp) on the CPU, on trees that
tests/test_slab.py does not grow."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _counts(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-o", exe,
                           os.path.join(ROOT, "tests", "cpp", name + ".cpp")])
    return map(int, subprocess.check_output([exe]).split())


def test_leaves_without_edges(tmp_path):
    """Leaves that own no edges change their parents' boxes and centres, but not
    the radii: no edge of a cleared cone passes the silhouette predicate."""
    trials, clears, wrong = _counts(tmp_path, "slab_empty")
    assert wrong == 0
    assert clears > trials // 4


def test_tilted_leaves(tmp_path):
    """Merges take small angles from the arccos of a rounded cosine, so normals
    lie outside their cones by as much as 2e-3 after a few levels: no edge of a
    cleared cone passes the silhouette predicate even so."""
    trials, clears, wrong, excess = _counts(tmp_path, "slab_tilt")
    assert wrong == 0
    assert clears > trials // 20  # 20 in 220 are views from anywhere
    assert excess > 2000
