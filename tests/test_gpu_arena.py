"""An arena batch's writes and reads on the GPU (internal/gpu/batch.go:126-210):
every word arrives and no other changes, whichever way the move takes."""
import numpy as np
import pytest

import rkhip

pytestmark = pytest.mark.gpu

EDGE = 1 << 18  # words a kernel moves; more take the copy engine


@pytest.mark.parametrize("n", [1, 255, 256, 257, 4096, 4097, 5120, EDGE, EDGE + 1])
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


def test_a_single_move_takes_the_copy_engine():
    """A move that is all of a batch; a kernel moves the words of one among
    other operations, past what the runtime itself copies by a kernel."""
    n = 5000
    x = np.random.default_rng(2).normal(0, 1, n).astype(np.float32)
    with rkhip.Device(0) as dev:
        a = dev.arena(2 * n, 4 * n)

        def moves(record):
            dev.profile_start()
            try:
                b = a.begin()
                got = record(b)
                b.submit()
            finally:
                prof = dev.profile_stop()
            return prof.get("batch_move", (0, 0.0))[0], got

        assert moves(lambda b: b.write(0, x))[0] == 0
        k, got = moves(lambda b: b.read(0, n))
        assert k == 0 and np.array_equal(np.asarray(got), x)
        k, got = moves(lambda b: (b.write(n, 2 * x), b.copy(n, 0, n), b.read(0, n))[2])
        assert k == 2 and np.array_equal(np.asarray(got), 2 * x)
        k, got = moves(lambda b: (b.read(0, n), b.write(0, x), b.read(0, n)))
        assert k == 3 and np.array_equal(np.asarray(got[0]), 2 * x) and np.array_equal(np.asarray(got[2]), x)
        k, got = moves(lambda b: (b.write(0, 3 * x[:4096]), b.copy(0, n, n), b.read(n, 4096))[2])
        assert k == 0 and np.array_equal(np.asarray(got), 3 * x[:4096])
        b = a.begin()  # a held move that fails: nothing is delivered
        b.write(0, x)
        assert b.write(2 * n - 1, x) == -1
        with pytest.raises(rkhip.RKError):
            b.submit()
        b = a.begin()
        got = b.read(0, 4096)
        b.submit()
        a.free()
        assert dev.used == 0
