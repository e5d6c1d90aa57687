"""The field download's chunks, slots and worker threads (csrc/oal_fields.h), compiled for the host with a stand-in
for the device: every cell arrives once and from its own chunk, a slot is written again only when it has been copied
out, errors end the call, and without pinned memory the chunks go through device memory."""
import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parent.parent / "openaerolab_alpha_01_amd" / "csrc"
SOURCE = '''#include "oal_fields.h"
#include <vector>
static double value(int a, size_t cell) { return 4.0 * cell + a; }
struct Dev {
    using error = int;
    bool pinned;
    int fail_issue, fail_wait, fail_direct;   // at this call, -1: never
    std::vector<std::vector<double>> mem;
    std::vector<std::pair<uint32_t, uint32_t>> due;
    long issued = 0, waited = 0, directs = 0, drained = 0;
    int reserve(uint32_t cells, int n) {
        if (!pinned) return 2;
        mem.assign(n, std::vector<double>(4 * (size_t)cells, -1.0));
        due.assign(n, {0, 0});
        return 0;
    }
    size_t slots() const { return mem.size(); }
    const double* slot(size_t i) const { return mem[i].data(); }
    int issue(size_t i, uint32_t c0, uint32_t n) {
        if (issued++ == fail_issue) return 719;
        std::fill(mem[i].begin(), mem[i].end(), -2.0);   // (what a copy still under way would read)
        due[i] = {c0, n};
        return 0;
    }
    int wait(size_t i) {
        if (waited++ == fail_wait) return 719;
        for (int a = 0; a < 4; ++a)
            for (uint32_t j = 0; j < due[i].second; ++j) mem[i][(size_t)a * due[i].second + j] = value(a, due[i].first + j);
        return 0;
    }
    int direct(uint32_t c0, uint32_t n, double* const (&dst)[4]) {
        if (directs++ == fail_direct) return 719;
        for (int a = 0; a < 4; ++a)
            for (uint32_t j = 0; dst[a] && j < n; ++j) dst[a][j] = value(a, (size_t)c0 + j);
        return 0;
    }
    void drain() { ++drained; }
};
extern "C" int run(uint64_t total, double* rho, double* u, int pinned, const int* fail, long* counts) {
    Dev d{pinned != 0, fail[0], fail[1], fail[2], {}, {}};
    const int e = oal::download_fields(d, total, rho, u);
    counts[0] = d.issued; counts[1] = d.directs; counts[2] = d.drained; counts[3] = (long)d.mem.size();
    return e;
}
'''


@pytest.fixture(scope="module")
def download(tmp_path_factory):
    d = tmp_path_factory.mktemp("fields")
    (d / "f.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-shared", "-fPIC", "-I", str(CSRC), "-o", str(d / "f.so"),
                    str(d / "f.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "f.so"))

    def run(total, rho=True, u=True, pinned=True, fail=(-1, -1, -1)):
        r = np.full(total, np.nan) if rho else None
        v = np.full((3, total), np.nan) if u else None
        counts = (ctypes.c_long * 4)()
        e = lib.run(ctypes.c_uint64(total), None if r is None else r.ctypes.data_as(ctypes.c_void_p),
                    None if v is None else v.ctypes.data_as(ctypes.c_void_p), int(pinned), (ctypes.c_int * 3)(*fail), counts)
        return e, r, v, list(counts)
    return run


def right(total, r, v):
    cell = 4.0 * np.arange(total)
    return (r is None or np.array_equal(r, cell)) and (v is None or all(np.array_equal(v[a], cell + a + 1) for a in range(3)))


# (chunks, slots) by the rule: a sixteenth of the cells, 4096 to 65536 of them; a quarter of the chunks and one, at most 12
TOTALS = {1: (1, 2), 4096: (1, 2), 4097: (2, 2), 13824: (4, 2), 65537: (16, 5), 131073: (16, 5), 409600: (16, 5),
          2 ** 20 + 1: (17, 6), 1204224: (19, 6), 2838528: (44, 12), 2949120: (45, 12)}


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("total", list(TOTALS))
def test_every_cell_once(download, total, pinned):
    for _ in range(3):
        e, r, v, (issued, directs, drained, slots) = download(total, pinned=pinned)
        chunks, want_slots = TOTALS[total]
        assert e == 0 and right(total, r, v) and drained == 0
        assert (issued, directs, slots) == ((chunks, 0, want_slots) if pinned else (0, chunks, 0))


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("rho,u", [(True, False), (False, True), (False, False)])
def test_one_field(download, rho, u, pinned):
    e, r, v, _ = download(300001, rho=rho, u=u, pinned=pinned)
    assert e == 0 and right(300001, r, v)


@pytest.mark.parametrize("total", [13824, 2838528])
@pytest.mark.parametrize("fail", [(0, -1, -1), (3, -1, -1), (-1, 0, -1), (-1, 2, -1), (-1, -1, 1)])
def test_errors_end_the_call(download, total, fail):
    e, r, v, (_, _, drained, _) = download(total, pinned=fail[2] < 0, fail=fail)
    assert e == 719 and drained == (1 if fail[2] < 0 else 0)
