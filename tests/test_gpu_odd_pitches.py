"""Matrix products on operands whose rows do not lie one behind the other: rows that overlap (a pitch below the row's length), a single
row whose pitch is anything, rows in reverse order.  A tile over the edge of such an operand cannot rely on its pitch to tell rows
that exist from rows that do not; the sizes are tiles that hang over the rows, whole and partial last K-tiles.  Against the oracle."""
import ctypes as C

import numpy as np
import pytest

import kapy_hip as kh
from gpu_util import dev_zeros, dglobal, sync, to_dev, to_host

pytestmark = pytest.mark.gpu


def _check(ko, dt, M, N, K, a_pitch, b_pitch, out, tol, seed, **cfg):
    """lhs rows a_pitch elements apart, rhs columns b_pitch apart, both contiguous along K; guard words behind the result."""
    if kh.DTYPE_BYTES[dt] == 1:
        rng = np.random.default_rng(seed)
        codes = lambda n: rng.integers(0x20, 0x50, size=n).astype(np.uint8) | (rng.integers(0, 2, size=n).astype(np.uint8) << 7)  # noqa: E731
    else:
        codes = lambda n: ko.fill_normal(n, dt, seed, n % 7, 0.0, 0.5)  # noqa: E731
    a, b = codes((M - 1) * abs(a_pitch) + K), codes((N - 1) * abs(b_pitch) + K)
    a0, b0 = (M - 1) * max(-a_pitch, 0), (N - 1) * max(-b_pitch, 0)   # element (0, 0): the last row's place where rows run backwards
    want = np.zeros(M * N, np.float32 if out == kh.F32 else np.uint16)
    assert ko.lib().ko_matmul(C.byref(ko.mk_global(a, M, K, a_pitch, 1, dt, a0)), C.byref(ko.mk_global(b, K, N, 1, b_pitch, dt, b0)), None,
                              C.byref(ko.mk_global(want, M, N, N, 1, out)), kh.RN) == 0
    da, db, dd = to_dev(a), to_dev(b), dev_zeros(M * N + 64, kh.DTYPE_BYTES[out], fill=0x1234)
    kh.matmul(dglobal(da, M, K, a_pitch, 1, dt, a0), dglobal(db, K, N, 1, b_pitch, dt, b0), dglobal(dd, M, N, N, 1, out), **cfg)
    sync()
    got = to_host(dd, want.dtype)
    assert np.all(got[M * N:].view(np.uint32 if out == kh.F32 else np.uint16) == 0x1234)
    g, w = ko.decode(got[:M * N], out), ko.decode(want, out)
    assert np.all(np.isfinite(g)) and np.linalg.norm(g - w) <= tol * np.linalg.norm(w), (M, N, K, a_pitch, b_pitch, cfg)


@pytest.mark.parametrize("dt", [kh.F16, kh.BF16])
@pytest.mark.parametrize("M,N,K", [(200, 136, 128), (300, 264, 72), (129, 128, 320), (40, 72, 256)])
def test_16_bit_rows_that_overlap(ko, dt, M, N, K):
    for a_pitch, b_pitch in ((8, K), (K, 16), (24, 8)):
        for cfg in ({}, dict(tile=(256, 256, 64), stages=25), dict(tile=(128, 128, 64), stages=25)):
            _check(ko, dt, M, N, K, a_pitch, b_pitch, kh.F32, 1e-5, 81, **cfg)
    if K % 64 == 0:
        _check(ko, dt, M, N, K, 8, 16, kh.F32, 1e-5, 82, tile=(256, 128, 64))


@pytest.mark.parametrize("dt", [kh.F16, kh.BF16])
@pytest.mark.parametrize("N,K", [(136, 128), (129, 72), (264, 327)])
def test_16_bit_single_row_of_any_pitch(ko, dt, N, K):
    for pitch in (1, 3, 8):
        _check(ko, dt, 1, N, K, pitch, (K + 7) // 8 * 8, kh.F32, 1e-5, 83)


@pytest.mark.parametrize("M,N,K", [(200, 136, 256), (300, 264, 272), (513, 1000, 128), (640, 520, 384)])
def test_f8_rows_that_overlap(ko, M, N, K):
    for a_pitch, b_pitch in ((16, K), (K, 32), (48, 16)):
        for cfg in ({}, dict(tile=(256, 256, 128)), dict(tile=(128, 128, 128))):
            _check(ko, kh.F8E4M3, M, N, K, a_pitch, b_pitch, kh.F32, 1e-4, 84, **cfg)


@pytest.mark.parametrize("N,K", [(136, 144), (128, 272), (264, 128), (136, 512)])
def test_f8_single_row_of_any_pitch(ko, N, K):
    for pitch in (1, 3, 16):
        _check(ko, kh.F8E4M3, 1, N, K, pitch, K, kh.F32, 1e-4, 85)


@pytest.mark.parametrize("dt,M,N,K", [(kh.F8E4M3, 16, 128, 512), (kh.F8E4M3, 48, 136, 512), (kh.F8E4M3, 200, 136, 256), (kh.F8E4M3, 300, 520, 272), (kh.F8E4M3, 5, 48, 128),
                                      (kh.BF16, 200, 136, 128), (kh.F16, 300, 264, 72)])
def test_operand_rows_in_reverse_order(ko, dt, M, N, K):
    for a_pitch, b_pitch in ((-K, K), (K, -K - 16), (-K, -K)):
        _check(ko, dt, M, N, K, a_pitch, b_pitch, kh.F32, 1e-4 if kh.DTYPE_BYTES[dt] == 1 else 1e-5, 87)
    if kh.DTYPE_BYTES[dt] == 1:   # a split that is none is refused here as well
        with pytest.raises(kh.KapyError):
            _check(ko, dt, M, N, K, -K, K, kh.F32, 1e-4, 88, split_k=-1)


@pytest.mark.parametrize("out", [kh.F32, kh.F16])
@pytest.mark.parametrize("M,N,K,b_rm", [(1, 136, 128, False), (1, 264, 192, True), (40, 136, 64, False), (300, 264, 128, True), (300, 264, 128, False), (257, 520, 72, True)])
def test_results_of_any_row_pitch(ko, out, M, N, K, b_rm):
    """A single result row of any pitch, and result rows in reverse order: stored where they belong and nothing else touched."""
    a, b = ko.fill_normal(M * K, kh.F16, 86, 0, 0.0, 0.5), ko.fill_normal(K * N, kh.F16, 86, 1, 0.0, 0.5)
    b_str = (N, 1) if b_rm else (1, K)
    want = np.zeros(M * N, np.float32 if out == kh.F32 else np.uint16)
    assert ko.lib().ko_matmul(C.byref(ko.mk_global(a, M, K, K, 1, kh.F16)), C.byref(ko.mk_global(b, K, N, *b_str, kh.F16)), None,
                              C.byref(ko.mk_global(want, M, N, N, 1, out)), kh.RN) == 0
    da, db = to_dev(a), to_dev(b)
    for pitch in ((0, 8, -N) if M == 1 else (-N, -N - 8)):
        span = (M - 1) * -pitch if M > 1 else 0
        dd = dev_zeros(span + N + 512, kh.DTYPE_BYTES[out], fill=0x1234)
        kh.matmul(dglobal(da, M, K, K, 1, kh.F16), dglobal(db, K, N, *b_str, kh.F16), dglobal(dd, M, N, pitch, 1, out, dynamic_offset=span + 256))
        sync()
        got = to_host(dd, want.dtype)
        at = span + 256 + np.arange(M)[:, None] * pitch + np.arange(N)
        g, w = ko.decode(np.ascontiguousarray(got[at].ravel()), out), ko.decode(want, out)
        assert np.all(np.isfinite(g)) and np.linalg.norm(g - w) <= (1e-5 if out == kh.F32 else 1e-3) * np.linalg.norm(w), pitch
        rest = np.ones(got.size, bool)
        rest[at.ravel()] = False
        assert np.all(got[rest].view(np.uint32 if out == kh.F32 else np.uint16) == 0x1234), pitch
