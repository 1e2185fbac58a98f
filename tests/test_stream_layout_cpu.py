"""The stream head's tiles in the workspace layout (host code only): finer
tiles of a small vocabulary never take a call past the no-allocation array
that coarse tiles keep within it."""
import ctypes

import pytest

from market_sim_amd import abi, ops


def _bytes(rows, open_rows, vocab, hidden, count):
    d = ops.DeviceBuffer
    b = ops.DecodeTailBuffers(
        x=d(1 << 20, rows * hidden * 4), embedding=d(1 << 30, vocab * hidden * 2),
        row_state=d(1 << 21, rows * 4), state_offsets=d(1 << 22, 8), state_tokens=d(1 << 23, count * 4),
        out_token=d(1 << 24, rows * 4), unrestricted_rows=d(1 << 25, open_rows * 4))
    a = ops.decode_tail_args(b, rows=rows, hidden=hidden, vocab=vocab, states=1, nnz=count,
                             max_count=count, unrestricted_count=open_rows)
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


@pytest.mark.parametrize("vocab", [1, 17, 192, 8192, 49152, 50021, 65537, 131072, 1000003])
def test_open_rows_have_records_for_every_tile(vocab):
    """At most 256 tokens per record, whatever the vocabulary."""
    per_row = _bytes(40, 33, vocab, 64, 1) - _bytes(40, 32, vocab, 64, 1)
    assert per_row >= (vocab + 255) // 256 * 96 - 256
