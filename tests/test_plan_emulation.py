"""CPU emulation of the register-resident plan kernel: every table it writes
against the general plan kernel's, over the forms a call can take (merged and
segmented first passes, later and last passes, few and many ks, both key
widths, bounds larger than the pass)."""
from test_kernel_emulation import _build_and_run, gen_dir  # noqa: F401


def test_register_plan_writes_what_the_general_plan_writes(gen_dir):  # noqa: F811
    out = _build_and_run(gen_dir, "plan_driver.cpp")
    assert out.count(" ok") == 12
