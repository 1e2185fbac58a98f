"""The tiles of the stream head and of the gather in the workspace layout
(host code only): finer tiles never take a call past the no-allocation array
that coarse ones keep within it."""
import ctypes

import pytest

from market_sim_amd import abi, ops


def _bytes(rows, open_rows, vocab, hidden, count, states=1, nnz=None):
    d = ops.DeviceBuffer
    nnz = count if nnz is None else nnz
    b = ops.DecodeTailBuffers(
        x=d(1 << 20, rows * hidden * 4), embedding=d(1 << 40, vocab * hidden * 2),
        row_state=d(1 << 31, rows * 4), state_offsets=d(1 << 32, (states + 1) * 4),
        state_tokens=d(1 << 33, nnz * 4), out_token=d(1 << 34, rows * 4),
        unrestricted_rows=d(1 << 35, open_rows * 4) if open_rows else d())
    a = ops.decode_tail_args(b, rows=rows, hidden=hidden, vocab=vocab, states=states, nnz=nnz,
                             max_count=count, unrestricted_count=open_rows, flags=abi.TAIL_NO_FUSED)
    n = ctypes.c_uint64()
    abi.check("bytes", abi.lib().mf_decode_tail_workspace_bytes(ctypes.byref(a), ctypes.byref(n)))
    return n.value


def test_finer_tiles_keep_within_the_no_alloc_array():
    most = abi.lib().mf_decode_tail_noalloc_max_bytes()
    record = 96
    # 43 coarse tiles of 192 tokens or 256 of 32: the finer ones where they fit
    few = _bytes(64, 8, 8192, 64, 16)
    assert few - _bytes(64, 7, 8192, 64, 16) >= 256 * record
    for open_rows in range(300, 1000, 50):
        n = _bytes(1000, open_rows, 8192, 64, 16)
        # what 192-token tiles take, and half a MiB for everything else
        coarse = open_rows * 43 * record + (1 << 20)
        assert n <= most or coarse > most - (1 << 19)


def test_gather_records_follow_the_mean_list():
    """97 rows whose states hold 266 ids on average and 2048 at most: tiles of
    16, 128 records a row; as many ids in every list: tiles of 64.  Records
    stay few (2^16), and a pack that fits the no-allocation array with tiles
    of 64 fits it with the finer ones."""
    record, most = 96, abi.lib().mf_decode_tail_noalloc_max_bytes()
    one = _bytes(97, 0, 50000, 960, 16, 300, 4800)   # one record a row
    per_row = [1 + round((_bytes(97, 0, 50000, 960, 2048, 300, nnz) - one) / (97 * record))
               for nnz in (79800, 300 * 2048)]       # (256-byte alignment is far below a row's record)
    assert per_row == [128, 32]
    for rows in (40, 100, 180, 250, 400):
        for longest in (2000, 10000, 40000):
            coarse = rows * (-(-longest // 64)) * record + rows * 8192 * 8 + (1 << 16)
            n = _bytes(rows, 0, 50000, 8192, longest, 300, 300 * 20)
            assert n <= coarse + (1 << 16) * record
            assert n <= most or coarse > most - (1 << 16)


@pytest.mark.parametrize("vocab", [1, 17, 192, 8192, 49152, 50021, 65537, 131072, 1000003])
def test_open_rows_have_records_for_every_tile(vocab):
    """At most 256 tokens per record, whatever the vocabulary."""
    per_row = _bytes(40, 33, vocab, 64, 1) - _bytes(40, 32, vocab, 64, 1)
    assert per_row >= (vocab + 255) // 256 * 96 - 256
