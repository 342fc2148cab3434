"""The slab test of the silhouette search (geom.hpp) on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_slab_never_clears_a_silhouette(tmp_path):
    """Cones of random patches (flat, curved, rough, near and far from the
    origin, single edges to 16), seen from random points: no edge of a cleared
    cone passes the silhouette predicate, with either orientation flag, and
    the test does clear a good part of what it sees."""
    exe = str(tmp_path / "slab_check")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-o", exe,
                           os.path.join(ROOT, "tests", "cpp", "slab_check.cpp")])
    trials, clears, wrong = map(int, subprocess.check_output([exe]).split())
    assert wrong == 0
    assert clears > trials // 3
