"""Properties of the kernel sources that no single run of a kernel shows."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hestonexotics_amd", "csrc")


def test_path_kernels_compile_without_contraction():
    """Results are the same bits in every instance of a kernel (launch shape, split or persistent, one or two
    reduction kernels): no expression of kernels.hip may leave the fusing of a product to the
    compiler, whose choice changes with the code around it."""
    text = open(os.path.join(CSRC, "kernels.hip")).read()
    pragmas = [(m.start(), m.group(1)) for m in re.finditer(r"^#pragma clang fp contract\((\w+)\)", text, re.M)]
    assert [mode for _, mode in pragmas] == ["off"]
    assert pragmas[0][0] < text.index("namespace hexo {")
