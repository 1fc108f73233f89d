"""The segment table of the streaming pass (host code): every macroparticle is
walked once, also where indexes come near 2^31."""
import numpy as np
import pytest

from cetasim_amd import capi

NCU = 256


def segments(counts, nwg=0, tile=0, room=1 << 24):
    c = np.array(counts, np.int64)
    n = capi.I64(room)
    begin, end = np.zeros(room, np.int64), np.zeros(room, np.int64)
    step, bunch, wg = (np.zeros(room, np.int32) for _ in range(3))
    capi.check(capi.load().cts_debug_layout(len(c), capi.i64ptr(c), nwg, tile, NCU, n, capi.i64ptr(begin),
                                            capi.i64ptr(end), capi.i32ptr(step), capi.i32ptr(bunch), capi.i32ptr(wg)))
    return [a[:n.value] for a in (begin, end, step, bunch, wg)]


def check_walk(counts, begin, end, step, bunch, wg):
    """Blocks of 256 from begin in steps of `step`, with the kernels' 32-bit
    offsets: none wraps, and each macroparticle is in exactly one block."""
    off = np.concatenate([[0], np.cumsum(np.array(counts, np.int64))])
    assert np.all(begin < end) and np.all(wg >= 0)
    assert np.all((begin >= off[bunch]) & (end <= off[bunch + 1]))
    length = end - begin
    assert np.all(step >= 256) and np.all(step % 256 == 0)
    assert np.all(length + step < 1 << 32)
    # strided segments of a bunch (step above a block): their first blocks
    # follow one another and there is one for every block within a step, or
    # for every block of the bunch
    for b in range(len(counts)):
        s = np.flatnonzero(bunch == b)
        nblk = -(-int(counts[b]) // 256)
        if np.all(step[s] == 256):
            assert begin[s[0]] == off[b] and end[s[-1]] == off[b + 1] and np.array_equal(begin[s[1:]], end[s[:-1]])
        else:
            assert np.all(step[s] == step[s[0]]) and np.all(end[s] == off[b + 1])
            assert len(s) == min(nblk, step[s[0]] // 256)
            assert np.array_equal(begin[s], off[b] + 256 * np.arange(len(s)))


@pytest.mark.parametrize("counts,nwg,tile", [
    ([20_001], 0, 0), ([100_000, 255, 257], 0, 0), ([9_000] * 480, 0, 0), ([5_000_000] * 3, 0, 0),
    ([5_000, 300], 7, 256), ([1 << 30], 2**31 - 1, 256),
    # more blocks than a stride of 32 bits holds
    ([1_200_000_000] * 2, 2**31 - 1, 256), ([1_200_000_000, 2_100_000_000, 1000], 1 << 24, 256)])
def test_every_macroparticle_once(counts, nwg, tile):
    check_walk(counts, *segments(counts, nwg, tile))


@pytest.mark.parametrize("n", [2**31 - 1, 2**31, 4_500_000_000])
def test_one_bunch_in_few_segments(n):
    """The default layout of one bunch: a segment per resident workgroup (a
    prologue and a reduction each), also beyond the strided layout's reach."""
    t = segments([n])
    check_walk([n], *t)
    assert len(t[0]) <= 1024


@pytest.mark.parametrize("counts", [[3000] * 8, [100, 70_000, 9], [9_001] * 90, [700, 3] * 60, [40_000] * 100,
                                    [80_000] * 60])
def test_reported_default_restores_it(counts):
    """The workgroups and tile that the default layout reports stand for it
    (here pieces and chunks: tile 0), and other counts of workgroups do not."""
    default = segments(counts)
    nwg = int(default[4].max()) + 1
    again, fewer = segments(counts, nwg, 0), segments(counts, nwg - 1, 0)
    assert all(np.array_equal(a, b) for a, b in zip(default, again))
    assert fewer[4].max() < nwg - 1
    check_walk(counts, *fewer)
