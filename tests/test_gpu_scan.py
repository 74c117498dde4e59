"""The prefix sums of the counting sorts against numpy, on each side of every
switch of the launcher (one workgroup; block sums added up by the blocks; block
sums scanned by a launch), and their time where a small cutoff in a large box
or a large mesh takes them."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMALL, DIRECT = 4096, 2048 * 1024  # counts: one workgroup; blocks add the sums up


class Scan:
    def __init__(self, pkg):
        self.lib = pkg.lib()
        vp = ctypes.c_void_p
        self.lib.p3mk_queue_create.argtypes = [ctypes.POINTER(vp)]
        self.lib.p3mk_queue_destroy.argtypes, self.lib.p3mk_queue_destroy.restype = [vp], None
        self.lib.p3mk_queue_sync.argtypes = [vp]
        self.lib.p3mk_exclusive_scan.argtypes = [vp, ctypes.c_long, vp, vp, vp]
        self.q = vp()
        assert self.lib.p3mk_queue_create(ctypes.byref(self.q)) == 0

    def run(self, count, out, scratch):
        assert self.lib.p3mk_exclusive_scan(count.data_ptr(), count.numel(), out.data_ptr(), scratch.data_ptr(),
                                            self.q) == 0

    def sync(self):
        assert self.lib.p3mk_queue_sync(self.q) == 0

    def close(self):
        self.lib.p3mk_queue_destroy(self.q)


def buffers(m, count):
    """Counts, result and scratch of p3mk_scan_scratch_ints(m) ints, each but
    the counts with a guard word behind it."""
    import torch

    out = torch.full((m + 2,), -7, dtype=torch.int32, device="cuda")
    scratch = torch.full(((m + 1023) // 1024 + 2,), -7, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return count, out, scratch


@pytest.mark.parametrize("m", [1, 1023, 1025, SMALL - 1, SMALL, SMALL + 1, 100000, DIRECT - 1, DIRECT, DIRECT + 1,
                               DIRECT + 1024, 3 * DIRECT + 17])
def test_scan_vs_numpy(pkg, m):
    import torch

    scan = Scan(pkg)
    host = np.random.default_rng(m).integers(0, 5, m, dtype=np.int32)
    count, out, scratch = buffers(m, torch.tensor(host, device="cuda"))
    scan.run(count, out, scratch)
    scan.sync()
    got = out.cpu().numpy()
    assert got[0] == 0 and got[m + 1] == -7 and scratch[-1].item() == -7
    assert np.array_equal(got[1:m + 1], np.cumsum(host))
    scan.close()


def test_scan_time_is_linear(pkg):
    """Four times the counts take less than eight times as long at 2^28 (a
    cell grid of 322 cells per side): a scan that is quadratic in its blocks
    takes ten times as long."""
    import torch

    scan = Scan(pkg)
    best = {}
    for m in (1 << 26, 1 << 28):
        count, out, scratch = buffers(m, torch.ones(m, dtype=torch.int32, device="cuda"))
        times = []
        for _ in range(6):
            t = time.perf_counter()
            scan.run(count, out, scratch)
            scan.sync()
            times.append(time.perf_counter() - t)
        assert out[m].item() == m and out[m // 3].item() == m // 3
        best[m] = min(times)
        print("2^%d counts: %.0f us" % (m.bit_length() - 1, 1e6 * best[m]))
    assert best[1 << 28] < 8 * best[1 << 26]
    scan.close()
