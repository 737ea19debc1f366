"""Fields read back (lg_download_member): below, at and far above the size
that goes through the ring of pinned chunks (2^22 values; 12 chunks
of 2^18), for both precisions, members beyond the first and repeated reads, also
from several threads at once.  A read moves values and changes none: what was
uploaded (rounded to what the case holds) comes back to the bit."""
import threading

import numpy as np
import pytest

import lesgo_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,Nz,members", [
    (16, 16, 8, 2),        # far below the ring
    (256, 256, 61, 1),     # below: 258 * 256 * 63 values
    (256, 256, 63, 2),     # above: 65 levels, ragged; member 1's chunks cut differently
])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_download_returns_what_was_uploaded(nx, ny, Nz, members, precision):
    cfg = lesgo_amd.Config(nx, ny, Nz, precision=precision)
    c = lesgo_amd.Case(cfg, members=members)
    rng = np.random.default_rng(nx + Nz)
    want = {}
    for m in range(members):
        for f in ("u", "dudz"):
            a = rng.standard_normal(c.shape)
            if precision == "mixed":
                a = a.astype(np.float32).astype(np.float64)
            c.upload(f, a, member=m)
            want[f, m] = a
    for _ in range(2):
        for (f, m), a in want.items():
            assert np.array_equal(c.download(f, member=m), a), (f, m)

    bad = []

    def reader(key):
        for _ in range(3):
            if not np.array_equal(c.download(key[0], member=key[1]), want[key]):
                bad.append(key)

    th = [threading.Thread(target=reader, args=(k,)) for k in want]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
