"""The packed conduction operator (linear_op.hip) against the matrices of eight
explicit steps in FP64, on the CPU: what rounding to fp16 pairs may leave on its
entries, on a row's sum (constant profiles) and first moment (linear profiles),
and the units of the high halves that keep the matrix instruction exact."""
import ctypes
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "binarytpm_amd", "libbtpm.so")
N, B, L = 55, 8, 63           # nodes, steps per block, entries (nodes, surface values)
FRAG = 64 * 8
TILE, CHUNK = (0, 1, 1, 2, 2, 3), (0, 0, 1, 0, 1, 1)
RATES = [0.4998, 0.47366, 0.25, 0.126, 0.0634, 0.03, 0.015, 0.0047, 3e-4]


def packed(r, ntau):
    f = ctypes.CDLL(LIB)._ZN4btpm15linear_operatorEfiPDF16_
    f.argtypes, f.restype = [ctypes.c_float, ctypes.c_int, ctypes.c_void_p], None
    op = np.zeros(26 * FRAG + 128, np.float16)
    f(r, ntau, op.ctypes.data)
    return op


def entry(g, q):
    """Entry of slot q of lane group g (-1: none)."""
    if q < 2:
        return N + 2 * g + q
    node = 1 + 2 * g + q - 2 if q < 4 else 9 + 16 * (q // 4 - 1) + 4 * g + q % 4
    return node - 1 if node <= N else -1


def unpack(op, first, blocks):
    """hi, lo [row][entry] of the fragments from `first` on."""
    out = np.zeros((2, L, L))
    for b, (t, h) in enumerate(blocks):
        for half in range(2):
            v = op[(first + 2 * b + half) * FRAG:][:FRAG].astype(np.float64)
            for lane in range(64):
                row = entry((lane & 15) >> 2, 4 * t + (lane & 3))
                for j in range(8):
                    col = entry(lane >> 4, 8 * h + j)
                    if row >= 0 and col >= 0:
                        out[half, row, col] = v[lane * 8 + j]
                    else:
                        assert v[lane * 8 + j] == 0
    return out


def dense(r, steps, responses):
    r = float(np.float32(r))
    A = np.diag(np.full(N, 1 - 2 * r)) + np.diag(np.full(N - 1, r), 1) + np.diag(np.full(N - 1, r), -1)
    A[-1, -1] += r
    b = np.zeros(N)
    b[0] = r
    m = np.zeros((L, L))
    m[:N, :N] = np.linalg.matrix_power(A, steps)
    for k in range(steps):
        m[:N, N + k] = np.linalg.matrix_power(A, steps - 1 - k) @ b
    if responses:
        for s in range(B):
            m[N + s] = np.linalg.matrix_power(A, s + 1)[0] @ m[:N]
    return m


@pytest.mark.parametrize("steps", [8, 5, 1])
@pytest.mark.parametrize("r", RATES)
def test_operator(r, steps):
    op = packed(r, 640 + steps)
    own = op[26 * FRAG:].view(np.float32)[8:10].astype(np.float64)
    six = list(zip(TILE, CHUNK))
    for first, c, n, resp in ((0, own[0], B, True), (12, own[1], steps, False)):
        want = dense(r, n, resp)
        want[:N, :N] -= c * np.eye(N)
        hi, lo = unpack(op, first, six) / 32768.0
        check(hi, lo, want)
    want = dense(r, 0, True)
    want[:N] = 0.0
    check(*(unpack(op, 24, [(0, 0)]) / 32768.0), want)


def check(hi, lo, want):
    top = np.abs(want).max(1)
    unit = 2.0 ** (np.frexp(np.where(top > 0, top, 1.0))[1] - 15)
    assert np.array_equal(np.round(hi / unit[:, None]) * unit[:, None], hi)
    err = hi + lo - want
    # an entry of the largest binade leaves half a unit of its low half, 2^-10
    # units; those that make up for the others a few times that
    assert (np.abs(err).max(1) <= 2.0 ** -6 * unit).all()
    # the low halves left are below 2 units, so each is rounded by at most
    # 2^-11 units: the row's sum by one of them, the moment by two entries
    # within 8 nodes and one within 16
    assert (np.abs(err.sum(1)) <= 2.0 ** -11 * unit).all()
    at = np.r_[np.arange(1, N + 1), np.ones(B)]
    pos = np.r_[np.arange(1, N + 1), np.zeros(B)]
    assert (np.abs((err * (pos - at[:, None])).sum(1)) <= 2.0 ** -6 * unit).all()
