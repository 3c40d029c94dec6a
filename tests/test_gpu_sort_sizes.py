"""The radix sort where its shape changes: the one-workgroup sort's two
register sizes (4096 and 8192 keys), the 1024-, 4096- and 8192-key
tiles and their remainders, every number of passes with whole and partial last
digits, values and permutation, few distinct keys (stability), a workspace
shared by sorts of falling length, and the smallest workspace.  Bit for bit against numpy's stable sort."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 64, 65, 1024, 4095, 4096, 4097, 8191, 8192, 8193, 16385, 131073, 262143, 262144, 262145,
         (1 << 20) - 1, (1 << 20) + 1]


def _expect(keys, vals, begin, end):
    mask = np.uint64((1 << (end - begin)) - 1)
    order = np.argsort((keys.astype(np.uint64) >> np.uint64(begin)) & mask, kind="stable")
    return keys[order], (vals[order] if vals is not None else order.astype(np.uint32))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("begin,end,high", [(0, 32, 1 << 32), (0, 7, 128), (0, 15, 1 << 15), (3, 24, 1 << 32), (0, 24, 5)])
def test_sort_sizes(flip2, n, begin, end, high):
    rng = np.random.default_rng(n + 31 * end)
    keys = rng.integers(0, high, n, dtype=np.uint64).astype(np.uint32)
    for vals in (None, rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)):
        k, v = flip2.sort_pairs_u32(keys, vals, begin, end)
        ek, ev = _expect(keys, vals, begin, end)
        assert np.array_equal(k, ek) and np.array_equal(v, ev)


def test_workspace_covers_smaller_sorts(flip2):
    L = flip2.lib()
    for bits in (8, 24, 32):
        need = [L.flip2_sort_workspace_bytes(n, 0, bits) for n in SIZES]
        assert need == sorted(need)
    n = 300000
    ws_bytes = L.flip2_sort_workspace_bytes(n, 0, 24)
    ws = flip2.DeviceBuffer(ws_bytes)
    bufs = [flip2.DeviceBuffer(4 * n) for _ in range(4)]
    rng = np.random.default_rng(1)
    for m in (300000, 262143, 16385, 5000):
        keys = rng.integers(0, 1 << 24, m, dtype=np.uint64).astype(np.uint32)
        dk = flip2.DeviceBuffer.from_array(keys)
        flip2.check(L.flip2_sort_pairs_u32(dk.ptr, None, *(b.ptr for b in bufs), m, 0, 24, ws.ptr, ws_bytes, None))
        flip2.synchronize()
        ek, ev = _expect(keys, None, 0, 24)
        assert np.array_equal(bufs[0].to_array(np.uint32, m), ek)
        assert np.array_equal(bufs[1].to_array(np.uint32, m), ev)
    with pytest.raises(flip2.Flip2Error):
        flip2.check(L.flip2_sort_pairs_u32(dk.ptr, None, *(b.ptr for b in bufs), 5000, 0, 24, ws.ptr, 64, None))


@pytest.mark.parametrize("n", [8193, 16385, 131073, 262143])
def test_workspace_of_4096_key_tiles(flip2, n):
    """The smallest workspace the header states: below it a call is refused,
    with it sorts of the short tiles take the 4096-key ones."""
    L = flip2.lib()
    passes, end = 3, 24
    least = 4608 + 1024 * passes * ((n + 4095) // 4096)
    assert least < L.flip2_sort_workspace_bytes(n, 0, end)
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 1 << end, n, dtype=np.uint64).astype(np.uint32)
    dk, ws = flip2.DeviceBuffer.from_array(keys), flip2.DeviceBuffer(least)
    bufs = [flip2.DeviceBuffer(4 * n) for _ in range(4)]
    for ws_bytes in (least - 1, least):
        args = (dk.ptr, None, *(b.ptr for b in bufs), n, 0, end, ws.ptr, ws_bytes, None)
        if ws_bytes < least:
            with pytest.raises(flip2.Flip2Error):
                flip2.check(L.flip2_sort_pairs_u32(*args))
            continue
        for _ in range(2):  # the second call finds the first one's words in the workspace
            flip2.check(L.flip2_sort_pairs_u32(*args))
            flip2.synchronize()
            ek, ev = _expect(keys, None, 0, end)
            assert np.array_equal(bufs[0].to_array(np.uint32, n), ek)
            assert np.array_equal(bufs[1].to_array(np.uint32, n), ev)
