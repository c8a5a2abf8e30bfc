"""CPU checks of the split GEMM's planner (neuralrs_amd/csrc/gemm_plan.hpp):
whatever it sends to a kernel, the kernel's 32-bit offsets can address."""
import pytest

import plan

pytestmark = pytest.mark.skipif(not plan.built(), reason="plan_query not built (run __graft_entry__.build())")


def largest_offset(ld, contiguous_k, rows, bk):
    """The largest byte offset of a staged tile's element from the tile's first
    one: `rows` rows of bk k values at leading dimension ld."""
    return 4 * ((rows - 1) * ld + bk - 1 if contiguous_k else (bk - 1) * ld + rows - 1)


def offsets(layout, m, n, k, tile):
    bm, bn, bk = tile
    a = largest_offset(m if layout == "TN" else k, layout != "TN", min(bm, m), bk)
    b = largest_offset(k if layout == "NT" else n, layout == "NT", min(bn, n), bk)
    return max(a, b)


# leading dimensions about every power of two where a tile's offsets may pass 2^31
EDGES = [(1 << e) + d for e in range(19, 28) for d in (-3, 0, 5)]


@pytest.mark.parametrize("layout", plan.LAYOUTS)
def test_the_products_of_the_gpu_tests_reach_their_tiles(layout):
    answers = plan.ask(*(("gemm", layout, *shape, 1, 0, 1, plan.CUS) for shape, _ in plan.TILES))
    for (shape, tile), answer in zip(plan.TILES, answers):
        assert answer.split()[:2] == [tile, "1"], (shape, answer)


def test_the_layers_of_the_gpu_tests_reach_their_tiles():
    answers = plan.ask(*(("conv", *shape, plan.CUS) for shape, _, _ in plan.CONV_TILES))
    for (shape, forward, backward), answer in zip(plan.CONV_TILES, answers):
        assert answer.split() == [forward, backward], (shape, answer)


@pytest.mark.parametrize("layout", plan.LAYOUTS)
def test_planned_tiles_are_addressable(layout):
    sizes = [(m, n, k) for big in EDGES for m, n, k in
             [(64, 64, big), (4096, 4096, big), (big, 64, 64), (64, big, 64), (big, 512, 512), (512, big, 512)]]
    answers = plan.ask(*(("gemm", layout, *s, 1, 0, 1, plan.CUS) for s in sizes))
    taken = 0
    for s, answer in zip(sizes, answers):
        if answer != "f32":
            taken += 1
            assert offsets(layout, *s, tuple(map(int, answer.split()[0].split("x")))) < 1 << 31, (s, answer)
    assert taken


@pytest.mark.parametrize("layout", plan.LAYOUTS)
def test_wide_matrices_keep_the_split_tiles(layout):
    """Rows of 2^21 floats and more still run the split GEMM, on the tiles that
    reach them."""
    wide = [(512, 2_500_000, 128), (64, 3_000_001, 65), (2_500_000, 512, 128), (100, 90, 4_000_000)]
    if layout == "NN":  # a k step of 16 rows reaches further
        wide.append((256, 20_000_000, 32))
    assert "f32" not in plan.ask(*(("gemm", layout, *s, 1, 0, 1, plan.CUS) for s in wide))


def test_short_reductions_of_aligned_rows_run_the_f32_kernel():
    """One k step of the f32 kernel, or two of which the split's second would be
    a partial one read value by value."""
    f32 = [("NN", 100, 50000, 32, 1), ("NT", 20860, 128, 52, 1), ("NT", 638, 404, 24, 23), ("TN", 2048, 640, 32, 1)]
    split = [("NN", 100, 50000, 64, 1), ("NT", 20860, 128, 64, 1), ("NT", 637, 404, 33, 23), ("TN", 20860, 128, 52, 1),
             ("NN", 4096, 4096, 32, 1), ("NN", 4000, 4000, 16, 1), ("TN", 2047, 641, 32, 1)]
    ask = lambda shapes: plan.ask(*(("gemm", *s, 0, 1, plan.CUS) for s in shapes))
    assert ask(f32) == ["f32"] * len(f32) and "f32" not in ask(split)


def test_shared_lhs_backward_groups_only_what_the_group_kernel_addresses():
    """Of 64 rows and 8.6 million columns, the rows of a gradient tile span 2^31
    bytes: the products have to run one after another."""
    sizes = [(rows, inner, cols) for rows in (64, 128, 4096) for inner in (64, 256) for cols in EDGES]
    answers = plan.ask(*(("shared", *s) for s in sizes))
    for (rows, inner, cols), answer in zip(sizes, answers):
        if answer == "1":
            assert offsets("NT", rows, inner, cols, (64, 64, 32)) < 1 << 31
            assert offsets("TN", inner, cols, rows, (64, 64, 32)) < 1 << 31
    assert plan.ask(("shared", 64, 64, 8_600_000)) == ["0"]
    assert plan.ask(("shared", 4096, 256, 256)) == ["1"]
