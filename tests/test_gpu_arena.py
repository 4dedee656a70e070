"""An arena batch's writes and reads on the GPU (internal/gpu/batch.go:126-210):
every word arrives and no other changes, whichever way the move takes."""
import numpy as np
import pytest

import rkhip

pytestmark = pytest.mark.gpu

EDGE = 1 << 18  # words a kernel moves; more take the copy engine


@pytest.mark.parametrize("n", [1, 255, 256, 257, 5120, EDGE, EDGE + 1])
@pytest.mark.parametrize("off", [0, 3])
def test_words_arrive(n, off):
    rng = np.random.default_rng(n + off)
    words = rng.integers(0, 1 << 32, n, dtype=np.uint32).view(np.float32)  # any bits, NaNs among them
    fill = np.arange(n + 16, dtype=np.float32)
    with rkhip.Device(0) as dev:
        a = dev.arena(2 * n + 64, 4 * n + 64)
        for _ in range(2):  # the second batch takes the staging over again
            b = a.begin()
            b.write(0, fill)
            b.write(off, words)
            b.copy(off, n + 24, n)
            whole, copied = b.read(0, n + 16), b.read(n + 24, n)
            b.submit()
            want = fill.copy()
            want[off:off + n] = words
            assert np.array_equal(np.asarray(whole).view(np.uint32), want.view(np.uint32))
            assert np.array_equal(np.asarray(copied).view(np.uint32), words.view(np.uint32))
        a.free()
        assert dev.used == 0
