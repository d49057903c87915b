"""The forms of the transform kernels that the library holds are the ones its dispatch can reach: no more, no fewer."""
import os
import re

from __graft_entry__ import PKG_DIR


def _forms(kernel, ints):
    """Template arguments (the leading integers) of every instantiation of a kernel, from the library's symbol names."""
    with open(os.path.join(PKG_DIR, "libhemm.so"), "rb") as f:
        names = f.read()
    mangled = re.compile(b"%d%sI%s" % (len(kernel), kernel.encode(), b"L[ib](n?[0-9]+)E" * ints))
    return {tuple(int(x.replace(b"n", b"-")) for x in m) for m in mangled.findall(names)}


def _scratch():
    """Kernel (mangled name) -> bytes of scratch per lane, from the metadata of the library's kernels (MessagePack: a name, then its scratch)."""
    with open(os.path.join(PKG_DIR, "libhemm.so"), "rb") as f:
        held = f.read()
    entry = re.compile(b"\xa5\\.name(?:\xd9.|\xda..|[\xa0-\xbf])(_Z\\w+)\xbb\\.private_segment_fixed_size(\xcd..|\xcc.|[\x00-\x7f])", re.S)
    return {name.decode(): int.from_bytes(size[1:] or size, "big") for name, size in entry.findall(held)}


def test_scratch():
    """Registers spill in the sums whose launch bounds ask for more wavefronts than their registers allow, and in no other kernel."""
    scratch = _scratch()
    assert len(scratch) > 300
    may = re.compile("diagonal_sums_kernelI|hoisted_terms_(list_)?kernelILi2E")
    assert [name for name, size in scratch.items() if size and not may.search(name)] == []


def test_row_passes():
    """Log2 of the rows (0: from the argument), points per thread, inverse."""
    points = {(4, 0), (8, 0), (16, 0), (4, 1), (8, 1)}
    assert _forms("ntt16_rows_kernel", 3) == {(lr,) + p for lr in (0, 8) for p in points}
    # ... tail: sixteen points at 2^16 in plain passes alone, an encryption's (2) few limbs eight there at most
    assert {f for f in _forms("ntt16_rows_kernel", 4) if f[3] in (1, 3) and not f[2]} == {(lr, p, 0, t) for t in (1, 3) for lr, p in ((0, 4), (8, 4), (0, 8), (8, 8), (0, 16))}
    assert {f for f in _forms("ntt16_rows_kernel", 4) if f[3] == 2} == {(0, 4, 0, 2), (8, 4, 0, 2), (8, 8, 0, 2)}
    # what a decryption reads (the last argument, 2) is one or two limbs
    assert {f for f in _forms("ntt16_rows_kernel", 5) if f[4] == 2} == {(lr, 4, 1, 0, 2) for lr in (0, 8)}


def test_one_launch_transforms():
    """Log2 of the rows, points per thread, what is loaded resp. the tail: four points of 2^12 for few limbs, which an encryption's (tail 2)
    and a decryption's (load 2) always are."""
    assert {f[:2] for f in _forms("ntt_limb_inverse_kernel", 3)} == {(2, 8), (3, 8), (4, 4), (4, 8), (5, 8), (6, 16)}
    assert {f[:2] for f in _forms("ntt_limb_inverse_kernel", 3) if f[2] == 2} == {(2, 8), (3, 8), (4, 4)}
    assert {f[:2] for f in _forms("ntt_limb_forward_kernel", 4) if f[3] == 2} == {(2, 8), (3, 8), (4, 4)}


def test_column_passes():
    """Log2 of the rows, points per thread, slabs narrowed by two to this, inverse: whole slabs of few points only where they are fewer
    than the line of four and more than that of half slabs."""
    narrow = {(lr, 4, h, inv) for lr in (5, 6, 7, 8) for h in (1, 2) if h < 2 or lr < 7 for inv in (0, 1)}
    whole = {(lr, 16, 0, inv) for lr in (5, 6, 7, 8) for inv in (0, 1)} | {(7, 4, 0, 0), (8, 4, 0, 0), (8, 4, 0, 1)}
    assert _forms("ntt16_cols_kernel", 4) == narrow | whole


def test_converted_and_lifted_column_passes():
    """Log2 of the rows, points per thread, slabs narrowed by two to this (and the sources kept in registers)."""
    half = {(lr, p, 1) for lr in (5, 6, 7) for p in (4, 8)} | {(8, 4, 1)}
    whole = {(lr, 8, 0) for lr in (5, 6, 7, 8)}
    assert _forms("ntt16_cols_lifted_kernel", 3) == half | whole
    assert _forms("ntt16_cols_converted_kernel", 4) == {f + (k,) for f in half | whole | {(5, 4, 2), (6, 4, 2)} for k in (2, 5, 8)}


def test_column_slabs():
    """Sources kept in registers."""
    with open(os.path.join(PKG_DIR, "libhemm.so"), "rb") as f:
        assert set(re.findall(rb"25ntt16_slab_convert_kernelILi([0-9]+)E", f.read())) == {b"2", b"3", b"4", b"5"}


def test_embedding_rows():
    """Log2 of the rows, decoding, rows of a workgroup: eight for batches of messages, and a decoding is one."""
    two = {(lr, decode, 2) for lr in range(1, 8) for decode in (0, 1)}
    assert _forms("emb_rows_kernel", 3) == two | {(lr, 0, 8) for lr in range(3, 8)}
