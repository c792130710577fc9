"""The number of the argument layouts follows kernel_args.h (CPU)."""
import os

from mgpu_old_amd import build


def test_number_follows_the_file():
    with open(os.path.join(build.CSRC, "kernel_args.h"), "rb") as f:
        text = f.read()
    assert build.args_layout() == build.args_layout(text) != 0
    assert build.args_layout(text.replace(b"uint32_t pad_;", b"uint32_t used;", 1)) != build.args_layout()
    assert build.args_layout(text + b"\n// a remark\n") == build.args_layout()
