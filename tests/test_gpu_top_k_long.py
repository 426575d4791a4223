"""top_k of rows of more than 2^30 elements, whose positions do not fit a sort
word: the first words of the row's pieces, merged."""
import numpy as np
import pytest

from pjrtx_amd.hlo import Builder

pytestmark = pytest.mark.gpu

N = 2 ** 30 + 24  # two pieces of 2^29 elements and one of 24
PIECE = 2 ** 29


@pytest.mark.parametrize("dt", ["s8", "bf16"])
def test_top_k_past_2_30(client, dt):
    """Large values at the pieces' edges, ties across pieces (the earlier
    position first), and the row's many equal values for the rest."""
    at = np.array([0, 5, PIECE - 1, PIECE, PIECE + 7, 2 * PIECE - 1, 2 * PIECE, 2 * PIECE + 1, N - 1, 10 ** 6, 7 * 10 ** 8])
    val = np.array([3, 7, 7, 7, 5, 7, 7, 4, 7, 6, 2])
    x = np.zeros(N, np.int8 if dt == "s8" else np.uint16)  # bf16: as bits
    x[at] = val if dt == "s8" else (np.asarray(val, np.float32).view(np.uint32) >> 16)
    buf = client.buffer(x[None], dt)
    order = sorted(zip(-val, at))
    zeros = np.setdiff1d(np.arange(400), at)
    for k in (4, 50, 300):
        b = Builder()
        exe = client.compile(b.build(list(b.top_k(b.param((1, N), dt), k))))
        got_v, got_i = (o.to_numpy()[0] for o in exe.execute_buffers([buf]))
        want = np.concatenate([[a for _, a in order], zeros])[:k]
        np.testing.assert_array_equal(got_i, want)
        np.testing.assert_array_equal(got_v, x[want])
    buf.delete()
