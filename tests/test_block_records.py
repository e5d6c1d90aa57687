"""The block records' offsets (csrc/oal_records.h), compiled for the host: what a kernel forms from a record, base plus
32-bit offset, against the neighbour table it was made from, below and above the spans where one base, and one base
per layer, cease to reach."""
import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

from openaerolab_alpha_01_amd.geometry import build_neighbor_table

CSRC = Path(__file__).resolve().parent.parent / "openaerolab_alpha_01_amd" / "csrc"
ESIZE = {"f32": 4, "f64": 8, "16": 2}
NONE, ALL, LAYERS = 0, 1, 2


@pytest.fixture(scope="module")
def records(tmp_path_factory):
    d = tmp_path_factory.mktemp("records")
    (d / "r.cpp").write_text('''#include "oal_records.h"
extern "C" int fit(const int32_t* nt, uint32_t b, uint64_t es) { return oal::two_fit(nt, b, es); }
extern "C" int row_fits(int64_t nbx, uint64_t es) { return oal::row_fits(nbx, es); }
extern "C" int64_t row_offset(int dx, int dy, int64_t nbx, int64_t local, uint64_t es) { return oal::row_offset(dx, dy, nbx, local, es); }
extern "C" void offsets(const int32_t* nt, uint32_t b, int layers, uint32_t es, uint32_t* off, uint32_t* base) {
    oal::TwoRec r{};
    oal::two_offsets(nt, b, layers != 0, es, r);
    for (int k = 0; k < 27; ++k) off[k] = r.off[k];
    base[0] = r.base_z[0]; base[1] = r.base; base[2] = r.base_z[1];
}
''')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", str(CSRC), "-o", str(d / "r.so"), str(d / "r.cpp")],
                   check=True)
    lib = ctypes.CDLL(str(d / "r.so"))

    def row(nt, b, es):
        """(fit, block that each of the 27 offsets reaches) after checking that 32 bits hold every byte of it"""
        nt = np.ascontiguousarray(nt, dtype=np.int32)
        p = nt.ctypes.data_as(ctypes.c_void_p)
        f = lib.fit(p, ctypes.c_uint32(b), ctypes.c_uint64(es))
        if f == NONE:
            return f, None
        off, base = np.zeros(27, dtype=np.uint32), np.zeros(3, dtype=np.uint32)
        lib.offsets(p, ctypes.c_uint32(b), int(f == LAYERS), es, off.ctypes.data_as(ctypes.c_void_p),
                    base.ctypes.data_as(ctypes.c_void_p))
        blk = 27 * 4096 * es
        assert f == LAYERS or base[0] == base[1] == base[2]
        assert (off.astype(np.int64) + blk <= 2 ** 32).all() and (off % blk == 0).all()
        return f, np.repeat(base, 9).astype(np.int64) + off // blk
    row.lib = lib
    return row


def check(records, table, es, blocks):
    fits = set()
    for b in blocks:
        nt = table[b].astype(np.int64) - 1
        nt[13] = b
        f, reach = records(nt, b, es)
        fits.add(f)
        if f != NONE:
            here = nt >= 0
            assert (reach[here] == nt[here]).all(), (b, nt, reach)
            assert ((reach >= 0) & (reach < len(table))).all()   # absent neighbours: some block of the level
        span = nt[nt >= 0].max() - nt[nt >= 0].min() + 1
        assert (f == ALL) == (span * 27 * 4096 * es < 2 ** 32), (b, span, f)
    return fits


@pytest.mark.parametrize("form", list(ESIZE))
def test_wide_levels(records, form):
    """Levels whose block layers just fit two to 4 GiB and just do not: faces, edges and the inside."""
    es = ESIZE[form]
    most = (2 ** 32 - 1) // (27 * 4096 * es)          # blocks that 32 bits span: 9709 in FP32
    nbx = 60
    for nby, inside in ((most // 2 // nbx - 2, ALL), (most // 2 // nbx + 1, LAYERS)):
        nblk = (nbx, nby, 3)
        z, y, x = np.meshgrid(*(np.arange(n) for n in nblk[::-1]), indexing="ij")
        table = build_neighbor_table(np.stack([x.ravel(), y.ravel(), z.ravel()], 1) + 1, nblk)
        mid = nbx * nby + nbx * (nby // 2) + nbx // 2
        assert check(records, table, es, [mid]) == {inside}
        layer = nbx * nby
        edge = [0, nbx - 1, layer - 1, layer, layer + nbx - 1, 2 * layer - nbx, 2 * layer - 1, 3 * layer - 1]
        check(records, table, es, edge + list(range(layer + 5 * nbx - 3, layer + 5 * nbx + 3)))


@pytest.mark.parametrize("periodic", [(False, False, True), (True, True, True), (False, True, False)])
def test_wraps(records, periodic):
    """Wraps that span more than 4 GiB: of z by layers; of y, in a layer that alone is larger, not at all."""
    nblk = (26, 25, 16) if not periodic[1] else (100, 100, 3)
    z, y, x = np.meshgrid(*(np.arange(n) for n in nblk[::-1]), indexing="ij")
    table = build_neighbor_table(np.stack([x.ravel(), y.ravel(), z.ravel()], 1) + 1, nblk, periodic)
    rng = np.random.default_rng(1)
    blocks = set(rng.integers(0, len(table), 400).tolist()) | set(range(0, len(table), 97)) | {0, len(table) - 1}
    fits = check(records, table, 4, sorted(blocks))
    assert fits == ({ALL, LAYERS} if not periodic[1] else {LAYERS, NONE})


def test_any_order(records):
    """Rows in no order (octree levels and their ghosts), absent neighbours among them."""
    rng = np.random.default_rng(2)
    nb, seen = 30000, set()
    for i in range(3000):
        b = int(rng.integers(0, nb))
        spread = int(rng.choice([50, 4000, 9709, 9710, 30000]))
        at = rng.integers(0, nb, 3) if i % 2 else np.full(3, b)
        nt = np.clip(np.repeat(at, 9) + rng.integers(0, spread, 27) - spread // 2, 0, nb - 1)
        nt[9:18] = np.clip(b + rng.integers(0, spread, 9) - spread // 2, 0, nb - 1)
        nt[rng.random(27) < rng.choice([0.0, 0.3, 0.9])] = -1
        nt[13] = b
        f, reach = records(nt, b, 4)
        seen.add(f)
        if f != NONE:
            assert (reach[nt >= 0] == nt[nt >= 0]).all() and ((reach >= 0) & (reach < nb)).all()
        else:
            assert nt.max() - nt[nt >= 0].min() + 1 > 9709
    assert seen == {NONE, ALL, LAYERS}


@pytest.mark.parametrize("storage", list(ESIZE))
def test_rows_reached_by_signed_offsets(records, storage):
    """the regular one-plane forms keep the offset of a cell in the next row of blocks in 32 signed bits: every one
    of them is exact up to the longest row that counts as regular, and the next longer row has one that is not"""
    es = ESIZE[storage]
    fits = lambda n: bool(records.lib.row_fits(ctypes.c_int64(n), ctypes.c_uint64(es)))
    records.lib.row_offset.restype = ctypes.c_int64

    def exact(n):
        got = [records.lib.row_offset(dx, dy, ctypes.c_int64(n), ctypes.c_int64(c), ctypes.c_uint64(es))
               for dx in (-1, 0, 1) for dy in (-1, 0, 1) for c in (0, 4095)]
        assert got == [((dx + dy * n) * 27 * 4096 + c) * es for dx in (-1, 0, 1) for dy in (-1, 0, 1) for c in (0, 4095)]
        return all(np.int64(v).astype(np.int32) == v for v in got)

    last = max(n for n in range(1, 10000) if fits(n))
    assert last == {"f32": 4853, "f64": 2426, "16": 9707}[storage]
    assert all(fits(n) and exact(n) for n in (1, 2, 16, last // 2, last - 1, last))
    assert not any(fits(n) or exact(n) for n in (last + 2, 2 * last, 38836))
