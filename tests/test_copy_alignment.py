"""Copies at every alignment (include/gfd/wave_ops.h, vec_count / vec_offset):
entries whose two sides differ mod 16 and whose size is no multiple of 16 move
as 16-byte vectors that overlap at the entry's ends.

CPU: the cut itself, from the header, over all alignments and small sizes:
every vector inside the entry, every byte covered, every store but the first
and last aligned.  GPU: the batches built on it (page table, entry list, both
directions, tiles), byte-exact, with guard bytes around every entry."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import gfd_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GUARD = 0xA5

CUT = r"""
#include <cstdint>
#include <cstdio>
#include <vector>
#include "gfd/wave_ops.h"
int check(uint64_t n, uint32_t m, uint64_t nv) {
    std::vector<char> seen(n, 0);
    for (uint64_t v = 0; v < nv; v++) {
        const int32_t o = gfd::wave::vec_offset((int32_t)v, (int32_t)m, (int32_t)n);
        if (o < 0 || (uint64_t)o + 16 > n) return 1;
        if (v > 0 && v + 1 < gfd::wave::vec_count(n, m) && ((m + (uint64_t)o) & 15) != 0) return 2;
        for (int b = 0; b < 16; b++) seen[o + b] = 1;
    }
    for (char c : seen) if (!c) return 3;
    return 0;
}
int main() {
    for (uint64_t n = 16; n < 200; n++)
        for (uint32_t m = 0; m < 16; m++) {
            const uint64_t nv = gfd::wave::vec_count(n, m);
            int e = check(n, m, nv);
            if (!e) e = check(n, m, gfd::wave::vec_count(n, 15));  // the uniform batch's count
            if (e) { std::printf("n %llu m %u: %d\n", (unsigned long long)n, m, e); return 1; }
        }
    // the largest entry of a batch: offsets stay inside 31 bits
    const uint64_t big = (1ull << 29) - 1;
    for (uint32_t m = 0; m < 16; m++) {
        const int32_t last = (int32_t)gfd::wave::vec_count(big, 15) - 1;
        if (gfd::wave::vec_offset(last, (int32_t)m, (int32_t)big) != (int32_t)(big - 16)) return 2;
    }
    return 0;
}
"""


def test_vector_cut_covers_every_range(tmp_path):
    if shutil.which("hipcc") is None:
        pytest.skip("hipcc not available")
    src = tmp_path / "cut.hip"
    src.write_text(CUT)
    r = subprocess.run(["hipcc", "--cuda-host-only", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include"),
                        "-c", str(src), "-o", str(tmp_path / "cut.o")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run(["hipcc", str(tmp_path / "cut.o"), "-o", str(tmp_path / "cut")], capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(tmp_path / "cut")], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


# Every pair of alignments, sizes around the 16-byte edges, one and several
# passes of a wave; "one" repeats a single size (the uniform batch).
SIZES = {"mixed": [1, 2, 15, 16, 17, 31, 32, 33, 47, 63, 64, 100, 1000, 1023, 4096, 4111],
         "one-17": [17], "one-1000": [1000], "one-4096": [4096], "one-9": [9], "large": [65536 + 5, 262144 - 3]}


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", sorted(SIZES))
@pytest.mark.parametrize("to", ["hbm", "host"])
def test_entry_list_any_alignment(sizes, to):
    print("entry list, sizes %s to %s" % (sizes, to), flush=True)
    rng = np.random.default_rng(len(sizes))
    pairs = [(d, s) for d in range(16) for s in range(16)]
    n = len(pairs) if sizes != "large" else 24
    size = np.array([SIZES[sizes][i % len(SIZES[sizes])] for i in range(n)], np.uint64)
    room = (size + np.uint64(16 + 31)) // np.uint64(16) * np.uint64(16)  # a guard of 16 bytes or more behind each
    base = np.concatenate([[16], 16 + np.cumsum(room + np.uint64(16))]).astype(np.uint64)
    order = rng.permutation(len(pairs))[:n]
    d_off = base[:n] + np.array([pairs[i][0] for i in order], np.uint64)
    s_off = base[:n] + np.array([pairs[i][1] for i in order], np.uint64)
    total = int(base[n]) + 64
    data = rng.integers(0, 256, total, dtype=np.uint8)
    want = np.full(total, GUARD, np.uint8)
    for i in range(n):
        want[int(d_off[i]):int(d_off[i] + size[i])] = data[int(s_off[i]):int(s_off[i] + size[i])]
    host, dev = gfd_amd.HostBuffer(total), gfd_amd.DeviceBuffer(total)
    if to == "hbm":
        host.array[:] = data
        dev.fill(GUARD)
        src, dst = host.ptr, dev.ptr
    else:
        host.array[:] = GUARD
        dev.upload(data)
        src, dst = dev.ptr, host.ptr
    table = np.stack([np.uint64(dst) + d_off, np.uint64(src) + s_off, size], 1)
    t = gfd_amd.DeviceBuffer(table.nbytes)
    t.upload(table)
    gfd_amd.zero_copy_gather(t.ptr, n)
    gfd_amd.synchronize()
    got = dev.download() if to == "hbm" else host.array
    bad = np.nonzero(got != want)[0]
    assert bad.size == 0, "byte %d of %d" % (bad[0], total)


@pytest.mark.gpu
@pytest.mark.parametrize("size", [1, 15, 16, 17, 24, 1000, 1001, 3000])
@pytest.mark.parametrize("skew", [(0, 0), (3, 0), (0, 5), (7, 7), (1, 15)])
def test_tokens_any_alignment(size, skew):
    """Gather and offload through a page table; destination and source bases skewed."""
    n, (ds, ss) = 301, skew
    print("tokens size=%d skew=%s" % (size, skew), flush=True)
    rng = np.random.default_rng(size)
    host = gfd_amd.HostBuffer(n * (2 * size + 1) + 64)
    host.array[:] = rng.integers(0, 256, host.nbytes, dtype=np.uint8)
    off = ss + rng.permutation(n).astype(np.int64) * (2 * size + 1)
    want = np.stack([host.array[o:o + size] for o in off]).reshape(-1)
    table = gfd_amd.DeviceBuffer(8 * n)
    table.upload(np.uint64(host.ptr) + off.astype(np.uint64))
    dst = gfd_amd.DeviceBuffer(n * size + 64)
    dst.fill(GUARD)
    gfd_amd.zero_copy_gather_tokens(table.ptr, dst.ptr + ds, size, n)
    gfd_amd.synchronize()
    got = dst.download()
    assert (got[ds:ds + n * size] == want).all()
    assert (got[:ds] == GUARD).all() and (got[ds + n * size:] == GUARD).all()
    before = host.array.copy()
    for o in off:
        host.array[o:o + size] = 0
    gfd_amd.zero_copy_scatter_tokens(table.ptr, dst.ptr + ds, size, n)
    gfd_amd.synchronize()
    assert (host.array == before).all()


@pytest.mark.gpu
@pytest.mark.parametrize("size,skew,helpers", [(1000, (0, 0), 0), (1001, (0, 3), 0), (40, (5, 0), 3), (12, (1, 2), 0)])
def test_tiles_any_alignment(size, skew, helpers):
    """Tiles of a WarpSpecSession whose chunks are not 16-byte aligned."""
    n, (ds, ss) = 512, skew
    print("tiles size=%d skew=%s" % (size, skew), flush=True)
    host = gfd_amd.HostBuffer(n * size + 64)
    host.array[:] = np.random.default_rng(size).integers(0, 256, host.nbytes, dtype=np.uint8)
    dst = gfd_amd.DeviceBuffer(n * size + 64)
    dst.fill(GUARD)
    res, _ = gfd_amd.warp_spec_run(host.ptr + ss, dst.ptr + ds, n, size, 128, 32, num_blocks=2, helper_waves=helpers)
    assert res["error_bits"] == 0 and res["lists_done"] == 4
    got = dst.download()
    assert (got[ds:ds + n * size] == host.array[ss:ss + n * size]).all()
    assert (got[:ds] == GUARD).all() and (got[ds + n * size:] == GUARD).all()


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 2, 3, 63, 64, 65, 255, 511, 512, 513, 1025])
@pytest.mark.parametrize("signal", [False, True])
def test_entry_list_slices(count, signal):
    """Lists of at most 512 entries are cut into 1024 / count slices each, taken
    by the waves in strides; longer ones whole.  Sizes from 0 bytes (an empty
    entry) to some KiB, so that slices are empty, whole and partial."""
    print("slices count=%d signal=%d" % (count, signal), flush=True)
    rng = np.random.default_rng(count)
    size = rng.choice([0, 1, 16, 100, 1000, 16384, 30001], count).astype(np.uint64)
    size[0] = 5000
    start = np.concatenate([[0], np.cumsum(size + np.uint64(7))[:-1]]).astype(np.uint64)
    total = int(start[-1] + size[-1]) + 64
    host, dev = gfd_amd.HostBuffer(total), gfd_amd.DeviceBuffer(total)
    host.array[:] = rng.integers(0, 256, total, dtype=np.uint8)
    dev.fill(GUARD)
    want = np.full(total, GUARD, np.uint8)
    for o, n in zip(start.astype(int), size.astype(int)):
        want[o:o + n] = host.array[o:o + n]
    table = np.stack([np.uint64(dev.ptr) + start, np.uint64(host.ptr) + start, size], 1)
    t = gfd_amd.DeviceBuffer(table.nbytes)
    t.upload(table)
    if signal:
        word, counter = gfd_amd.HostBuffer(64, gfd_amd.HOST_COHERENT), gfd_amd.DeviceBuffer(64)
        counter.fill(0)
        word.array[:] = 0
        assert gfd_amd.lib().gfd_zero_copy_gather_signal(t.ptr, count, counter.ptr, word.ptr, 77, None) == 0
        gfd_amd.synchronize()
        assert int(word.array.view(np.uint64)[0]) == 77 and (counter.download()[:4] == 0).all()
    else:
        gfd_amd.zero_copy_gather(t.ptr, count)
        gfd_amd.synchronize()
    assert (dev.download() == want).all()
