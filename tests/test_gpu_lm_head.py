"""The LM-head argmax of 1-8 rows against exact scores in numpy: both kernels
(dot2 for one and two rows, matrix cores beyond), tables at the edges of the 16-row
groups, of the two ways of sharing them and of the workgroup counts' steps, hidden sizes
with a padded last step and at and past the limits of the matrix-core kernel and of the
staged rows, the extreme values, ties, and what more rows cost."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(table, rows):
    import llm_accel
    vocab, hidden = table.shape
    wide = table.T.astype(np.float64)
    with llm_accel.Accelerator(llm_accel.Shape(vocab, hidden, 128, 1, hidden // 16, hidden // 16, 64,
                                               1e6)) as a:
        a.load_lm_head(table)
        a.upload(0, rows)
        for first, n in ((0, 8), (0, 3), (3, 5), (7, 1), (2, 2)):
            # below 2^53: exact in float64
            scores = rows[first:first + n].astype(np.float64) @ wide
            tokens, got = a.lm_head_argmax(0, first, n)
            assert tokens == [int(t) for t in scores.argmax(1)], f"rows {first}+{n}"
            assert got == [int(s) for s in scores.max(1)], f"rows {first}+{n}"


@pytest.mark.parametrize("vocab,hidden", [
    (1, 128), (15, 128), (16, 480), (17, 896), (1001, 2048), (32752, 128), (32753, 128),
    (33001, 256), (600, 2816), (600, 2944), (32770, 3840), (32770, 3968), (24580, 128),
    (24575, 256), (131077, 128), (32770, 4224)])
def test_tables(vocab, hidden):
    print(f"case vocab {vocab} hidden {hidden}", flush=True)
    rng = np.random.default_rng(vocab + hidden)
    table = rng.integers(-32768, 32768, size=(vocab, hidden)).astype(np.int16)
    rows = rng.integers(-32768, 32768, size=(8, hidden)).astype(np.int16)
    rows[1], rows[2], rows[6] = -32768, 32767, 0
    table[vocab // 2] = -32768
    _check(table, rows)


@pytest.mark.parametrize("vocab", [50, 40000])
def test_ties_take_the_first_index(vocab):
    rng = np.random.default_rng(vocab)
    table = rng.integers(-50, 50, size=(vocab, 256)).astype(np.int16)
    best = rng.integers(100, 200, size=256).astype(np.int16)
    rows = np.abs(rng.integers(1, 300, size=(8, 256))).astype(np.int16)
    for v in (vocab - 1, vocab // 2 + 5, vocab // 3):
        table[v] = best
    _check(table, rows)


def _fastest(f, n=15):
    best = 1e9
    for _ in range(n):
        t0 = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t0)
    return best


@pytest.mark.parametrize("vocab,hidden,rows,limit", [(100000, 2048, 2, 1.6), (60000, 4096, 2, 1.6),
                                                     (60000, 4096, 3, 3.5), (40000, 5120, 2, 2.5)])
def test_more_rows_than_one(vocab, hidden, rows, limit):
    """Both stream the table once: on large tables two staged rows take 1.1 times one
    row's time, two or three rows read from memory 1.2 to 2.2 times; with too few
    wavefronts in flight each was 2 to 5 times as long."""
    import llm_accel
    rng = np.random.default_rng(vocab)
    table = np.tile(rng.integers(-256, 256, size=(2000, hidden)).astype(np.int16), (vocab // 2000, 1))
    with llm_accel.Accelerator(llm_accel.Shape(vocab, hidden, 128, 1, hidden // 64, hidden // 64, 64,
                                               1e6)) as a:
        a.load_lm_head(table)
        a.upload(0, rng.integers(-2000, 2000, size=(8, hidden)).astype(np.int16))
        one, more = (_fastest(lambda: a.lm_head_argmax(0, 0, n)) for n in (1, rows))
    print(f"{vocab} x {hidden}: 1 row {one * 1e6:.0f} us, {rows} rows {more * 1e6:.0f}", flush=True)
    assert more < limit * one
