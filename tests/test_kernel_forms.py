"""The forms of the transform kernels that the library holds are the ones its dispatch can reach: no more, no fewer."""
import os
import re

from __graft_entry__ import PKG_DIR


def _forms(kernel, ints):
    """Template arguments (the leading integers) of every instantiation of a kernel, from the library's symbol names."""
    with open(os.path.join(PKG_DIR, "libhemm.so"), "rb") as f:
        names = f.read()
    mangled = re.compile(b"%d%sI%s" % (len(kernel), kernel.encode(), b"L[ib]([0-9]+)E" * ints))
    return {tuple(int(x) for x in m) for m in mangled.findall(names)}


def test_row_passes():
    """Log2 of the rows (0: from the argument), points per thread, inverse."""
    points = {(4, 0), (8, 0), (16, 0), (4, 1), (8, 1)}
    assert _forms("ntt16_rows_kernel", 3) == {(lr,) + p for lr in (0, 8) for p in points}
