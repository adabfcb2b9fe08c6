"""The level-ordered layout of ILU(0) factors (ks_ilu0_layout, host code): its steps, threads
and entries at the lines of its rule, what it leaves to the waiting rows, and its memory, which
stays a fixed multiple of the rows whatever the levels."""
import ctypes as C

import numpy as np
import pytest

from slepc_amd import matgen as M


class Layout(C.Structure):
    _fields_ = [("step", C.c_int), ("threads", C.c_int), ("entries", C.c_int), ("ring", C.c_int), ("bytes", C.c_int64)]


def layout(csr, lower):
    from slepc_amd import ks
    rp, ci = np.ascontiguousarray(csr[0], np.int32), np.ascontiguousarray(csr[1], np.int32)
    out = Layout()
    ks.check(ks.lib().ks_ilu0_layout(C.c_int(len(rp) - 1), rp.ctypes.data_as(C.c_void_p), ci.ctypes.data_as(C.c_void_p),
                                     C.c_int(lower), C.byref(out)), "ks_ilu0_layout")
    return out


def layered(widths, entries, far=False, seed=0):
    """A diagonally dominant matrix whose row p of level l of the forward solve needs up to
    `entries` rows of level l - 1, and whose upper part is the lower one turned around, so the
    backward solve has the same levels.  far: the last row needs row 0 too."""
    rng = np.random.default_rng(seed)
    start = np.concatenate([[0], np.cumsum(widths)])
    n = int(start[-1])
    i, j = [], []
    for l in range(1, len(widths)):
        p = np.arange(widths[l])
        for e in range(min(entries, widths[l - 1])):
            i.append(start[l] + p)
            j.append(start[l - 1] + (p + e * (1 + widths[l - 1] // 3)) % widths[l - 1])
    if far:
        i.append(np.array([n - 1]))
        j.append(np.array([0]))
    pairs = np.unique(np.stack([np.concatenate(i), np.concatenate(j)]), axis=1) if i else np.zeros((2, 0), int)
    rows = np.concatenate([pairs[0], n - 1 - pairs[0], np.arange(n)])
    cols = np.concatenate([pairs[1], n - 1 - pairs[1], np.arange(n)])
    vals = np.concatenate([rng.uniform(-1.0, 1.0, 2 * pairs.shape[1]), np.full(n, 10.0)])
    order = np.lexsort((cols, rows))
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int32)
    return rowptr, cols[order].astype(np.int32), vals[order]


CASES = [  # matrix, rows of a step (0: none), threads, entries
    (lambda: M.laplacian_1d(1), 1, 64, 2),
    (lambda: M.laplacian_1d(3000), 1, 64, 2),
    (lambda: layered([50] * 40, 2), 64, 64, 2),
    (lambda: layered([50] * 40, 4), 64, 64, 4),
    (lambda: layered([65] * 40, 2), 128, 128, 2),
    (lambda: layered([100] * 40, 3), 128, 128, 4),
    (lambda: layered([256] * 9, 2), 256, 256, 2),
    (lambda: layered([200] * 9, 4), 256, 256, 4),
    (lambda: layered([257] * 9, 1), 512, 512, 2),
    (lambda: layered([400] * 9, 4), 512, 512, 4),
    (lambda: layered([700] * 7, 2), 1024, 1024, 2),
    (lambda: layered([1500] * 7, 2), 1024, 1024, 2),      # two steps a level
    (lambda: layered([1500] * 7, 3), 512, 512, 4),        # three
    (lambda: layered([1000] + [3] * 1200, 2), 8, 64, 2),  # steps of 1024 would take 1,200 x 1024 slots
    (lambda: layered([100] * 80, 2, far=True), 128, 128, 4),  # 10,240 slots back: the longest ring
    (lambda: layered([200] * 80, 2, far=True), 0, 0, 0),  # 20,480 slots back: past the ring
    (lambda: layered([50] * 40, 5), 0, 0, 0),             # more entries a row than it takes
    (lambda: layered([9000] * 2, 1), 0, 0, 0),            # nine steps a level: the whole chip's work
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_layout_rule(i):
    make, step, threads, entries = CASES[i]
    csr = make()
    n = len(csr[0]) - 1
    for lower in (1, 0):
        L = layout(csr, lower)
        assert (L.step, L.threads, L.entries) == (step, threads, entries)
        assert L.bytes <= 304 * n and L.ring <= 16384
        if L.step:
            assert L.ring >= L.step and L.ring & (L.ring - 1) == 0


@pytest.mark.parametrize("n", [20000, 1000000])
def test_layout_memory_of_deep_levels(n):
    # a level a row: 304 bytes a row at most (four slots of two or four entries)
    csr = M.laplacian_1d(n)
    for lower in (1, 0):
        L = layout(csr, lower)
        assert L.step == 1 and L.bytes <= 304 * n
    csr = M.laplacian_2d(n // 10, 10)
    for lower in (1, 0):
        assert 0 < layout(csr, lower).bytes <= 304 * n


@pytest.mark.parametrize("rowptr,colidx", [([0, 1, 2], [1, 1]), ([0, 2, 3], [1, 0, 1]), ([0, 2, 3], [-1, 0, 1]),
                                           ([0, 2, 3], [0, 2, 1]), ([0, 0, 1], [1]), ([1, 2, 3], [0, 0, 1])])
def test_patterns_without_a_factorization_are_refused(rowptr, colidx):
    # no diagonal, decreasing, negative, past the last column, an empty row, rows that start past 0
    from slepc_amd import ks
    with pytest.raises(ks.KSError):
        layout((np.array(rowptr), np.array(colidx)), 1)
