"""Which sources are built without machine LICM: those of the tree walks, whose registers it would fill with
constants, and not the brute force sum, whose loop over all triangles needs them there."""
import glob
import os

from lagrange_amd import build as B


def test_machine_licm():
    off = {f for f, flags in B.EXTRA_FLAGS.items() if "-disable-machine-licm" in flags}
    where = {}
    for src in glob.glob(os.path.join(B.HERE, "csrc", "*.hip")):
        text = open(src).read()
        for kernel in ("k_bruteforce(", "k_traverse(", "k_traverse_quad(", "k_point_bfs("):
            if "void " + kernel in text:
                where[kernel] = os.path.basename(src)
    assert where["k_bruteforce("] not in off
    assert off == {where[k] for k in where if k != "k_bruteforce("}
