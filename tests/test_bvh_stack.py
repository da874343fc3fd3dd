"""The rows of the device walk's stack (walk, node_step and leaf_step of
csrc/gbuffer_kernels.hip) replayed on the CPU over trees of up to the depth
bound, every box hit: the push writes without a guard, so no tree that the
builder accepts may reach past the array's last row."""
import re
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "neural_wavelet_prt_demo_amd" / "csrc"


def _constants():
    depth = int(re.search(r"constexpr int kBvhMaxDepth = (\d+);",
                          (CSRC / "kernels.hpp").read_text()).group(1))
    kernels = (CSRC / "gbuffer_kernels.hip").read_text()
    rows = re.search(r"constexpr int kStackRows = kBvhMaxDepth \+ (\d+);", kernels)
    # The statements replayed below.
    for line in ("stack[0] = kDone;", "stack[64 * sp] = second ? c0 : c1;", "sp += h0 & h1;",
                 "if (!(h0 | h1)) node = stack[64 * --sp];",
                 "if (last && !(ANY && hit)) node = stack[64 * --sp];"):
        assert line in kernels, line
    assert len(re.findall(r"__shared__ int stack_lds\[kStackRows \* 64\];", kernels)) == \
        len(re.findall(r"stack_lds\[", kernels))
    return depth, depth + int(rows.group(1))


def _comb(levels):
    """levels internal nodes in a chain, each with one leaf: (inner, leaf)."""
    tree = "leaf"
    for _ in range(levels):
        tree = (tree, "leaf")
    return tree


def _random_tree(rng, levels):
    if levels == 0 or rng.random() < 0.15:
        return "leaf"
    return (_random_tree(rng, levels - 1 if rng.random() < 0.7 else max(0, levels - 4)),
            _random_tree(rng, max(0, levels - 1 if rng.random() < 0.2 else levels - 6)))


def _highest_row(tree, hit, second):
    """The walk over `tree`; hit(child) and second() choose which boxes are
    hit and which child is next.  Returns the highest row written."""
    stack, sp, node, top = {0: "done"}, 1, tree, 0
    while node != "done":
        if node == "leaf":
            sp -= 1
            node = stack[sp]
            continue
        c0, c1 = node
        h0, h1 = hit(), hit()
        nxt = (not h0) or (h1 and second())
        stack[sp] = c0 if nxt else c1
        top = max(top, sp)
        sp += h0 and h1
        node = c1 if nxt else c0
        if not (h0 or h1):
            sp -= 1
            node = stack[sp]
    assert sp == 0
    return top


@pytest.mark.parametrize("inner_first", [True, False])
def test_comb_of_the_depth_bound_fits(inner_first):
    depth, rows = _constants()
    # inner child is c0, so `second` = not inner_first takes the leaf first
    assert _highest_row(_comb(depth), lambda: True, lambda: not inner_first) <= rows - 1
    assert _highest_row(_comb(depth), lambda: True, lambda: False) == rows - 1  # the last row
    assert _highest_row(_comb(depth + 1), lambda: True, lambda: False) == rows  # one past it


def test_random_trees_and_hits_fit():
    depth, rows = _constants()
    rng = np.random.default_rng(3)
    for trial in range(200):
        tree = (_random_tree(rng, depth - 1), _random_tree(rng, depth - 1))
        p = (1.0, 0.7, 0.3)[trial % 3]
        assert _highest_row(tree, lambda: bool(rng.random() < p),
                            lambda: bool(rng.random() < 0.5)) < rows
