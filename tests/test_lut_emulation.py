"""CPU emulation of the first pass's cell table: every level of it against a
binary search over the range starts, both key widths, with and without a
window, with tables left, used up and never needed."""
from test_kernel_emulation import _build_and_run, gen_dir  # noqa: F401


def test_cell_table_finds_the_range_of_a_binary_search(gen_dir):  # noqa: F811
    out = _build_and_run(gen_dir, "lut_driver.cpp")
    assert out.count(" ok") == 16 and "bad 0" in out
