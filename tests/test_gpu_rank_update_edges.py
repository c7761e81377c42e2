"""The rank-k updates of the integral and of the Hessian at the edges of their
geometry: rows of 1 column block of 8 waves, of one window (12 and 11 blocks) and
of two and three windows (up to 8 blocks) with a padded last block, single events,
chunks of up to 64 events with a ragged last one, and several chunks per workgroup.

Reference: numpy.  Both sides sum M terms in FP64, in different orders: the
difference from a sum is below M 2^-53 relative to the sum of magnitudes, with M up
to 33k 4e-12 in the worst case and its square root (2e-14) as it happens; 1e-12
relative to the largest element, as the other integral tests."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


def amplitudes(rng, M, W):
    return (rng.normal(size=(M, W)) + 1j * rng.normal(size=(M, W))) * np.linspace(0.4, 1.6, W)[None, :]


@pytest.mark.parametrize("waves,events", [(1, 1), (7, 63), (8, 64), (9, 65), (16, 7), (24, 129), (87, 55), (88, 57),
                                          (89, 111), (96, 8), (97, 56), (104, 64), (128, 65), (137, 64 * 256 * 2 + 9)])
def test_integral(gpu, waves, events):
    rng = np.random.default_rng(waves)
    a = amplitudes(rng, events, waves)
    w = rng.uniform(0.5, 2.0, size=events)
    assert H.rel_err(gpu.integral(a), a.T @ a.conj()) <= 1e-12
    ref = (a / w[:, None]).T @ a.conj() * (events / np.sum(1 / w))
    assert H.rel_err(gpu.integral(a, w), ref) <= 1e-12


@pytest.mark.parametrize("waves,events", [(1, 3), (9, 65), (88, 64 * 256 + 57), (96, 1000), (137, 300)])
def test_integral_of_rows_at_an_odd_double(gpu, waves, events):
    """Device arrays aligned to 8 bytes only give the bits of aligned ones."""
    rng = np.random.default_rng(waves)
    a = amplitudes(rng, events, waves)
    w = rng.uniform(0.5, 2.0, size=events)
    buf, odd, wbuf = gpu.DeviceBuffer(a.nbytes), gpu.DeviceBuffer(a.nbytes + 16), gpu.DeviceBuffer(w.nbytes)
    buf.upload(a)
    odd.upload(np.concatenate([[np.nan], a.view(np.float64).ravel(), [np.nan]]))
    wbuf.upload(w)
    for wt in (None, wbuf.address):
        ref = gpu.integral_device(buf.address, events, waves, wt)
        assert np.array_equal(gpu.integral_device(odd.address + 8, events, waves, wt), ref)
        if waves <= 128:
            assert np.array_equal(gpu.integral_device_noalloc(odd.address + 8, events, waves, wt), ref)


def hessian(A, nW, T, flat):
    """[P][P][3], [P], float of pwaLikelihood.cc:697-753 over P = rank 2 wmax amplitudes."""
    rank, wmax = T.shape[0], T.shape[2]
    W = sum(nW)
    sec = (np.arange(W) >= nW[0]).astype(int)
    at = np.where(sec, np.arange(W) - nW[0], np.arange(W))
    S = np.stack([np.stack([A[:, sec == s] @ T[r, s, :nW[s]] for s in range(2)]) for r in range(rank)])
    f = 2 / (np.sum(np.abs(S) ** 2, axis=(0, 1)) + flat ** 2)
    h = np.zeros((rank, 2, wmax, rank, 2, wmax, 3))
    ft = np.zeros((rank, 2, wmax), dtype=complex)
    d = [f[:, None] * S[r][sec].T * A.conj() for r in range(rank)]
    Q = (A * f[:, None]).T @ A.conj()
    for r in range(rank):
        ft[r, sec, at] = flat * f @ d[r]
        for q in range(rank):
            same = (sec[:, None] == sec[None, :]) & (r == q)
            for k, v in enumerate((d[r].real.T @ d[q].real - same * Q.real, d[r].real.T @ d[q].imag - same * Q.imag,
                                   d[r].imag.T @ d[q].imag - same * Q.real)):
                for i in range(W):
                    h[r, sec[i], at[i], q, sec, at, k] = v[i]
    P = rank * 2 * wmax
    return h.reshape(P, P, 3), ft, flat ** 2 * np.sum(f ** 2) - np.sum(f)


@pytest.mark.parametrize("nW,rank,events", [((0, 1), 1, 1), ((7, 0), 1, 63), ((3, 5), 2, 65), ((2, 3), 5, 40),
                                            ((8, 80), 1, 56), ((0, 96), 1, 300), ((1, 103), 1, 64),
                                            ((0, 136), 1, 129), ((13, 40), 3, 1000), ((5, 37), 4, 700), ((3, 36), 3, 130),
                                            ((8, 80), 2, 64 * 256 * 2 + 9)])
@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "mixed"])
def test_hessian(gpu, nW, rank, events, prec):
    rng = np.random.default_rng(sum(nW) + rank)
    A = amplitudes(rng, events, sum(nW))
    T = np.zeros((rank, 2, max(nW)), dtype=complex)
    for s in range(2):
        T[:, s, :nW[s]] = rng.normal(size=(rank, nW[s])) + 1j * rng.normal(size=(rank, nW[s]))
    if prec:  # the stored amplitudes; everything after them is FP64
        A = A.astype(np.complex64).astype(np.complex128)
    ctx = gpu.LikelihoodContext(0, prec)
    ctx.load(A, nW)
    flat = 0.7
    h, ft, hf = ctx.hessian(T, flat)
    rh, rft, rhf = hessian(A, nW, T, flat)
    assert H.rel_err(h, rh) <= 1e-12
    assert H.rel_err(ft, rft) <= 1e-12
    assert abs(hf - rhf) <= 1e-12 * abs(rhf) * 10  # a difference of two sums


def test_hessian_in_pieces(gpu):
    """An event list of more than 8 GiB of S (rank 100: 3216 bytes an event) is
    summed in pieces that add to each other.  Reference: the sum of two lists of
    one piece each."""
    rank, nW = 100, (1, 1)
    piece = (8 << 30) // (32 * rank + 16)
    N, first = piece + 300_001, piece - 100_003
    rng = np.random.default_rng(3)
    A = rng.normal(size=(N, 2)) + 1j * rng.normal(size=(N, 2))
    T = (rng.normal(size=(rank, 2, 1)) + 1j * rng.normal(size=(rank, 2, 1)))
    out = []
    for a in (A, A[:first], A[first:]):
        ctx = gpu.LikelihoodContext(0, 0)
        ctx.load(a, nW)
        out.append(ctx.hessian(T, 0.7))
        ctx.close()
    for whole, x, y in zip(*out):
        assert H.rel_err(whole, x + y) <= 1e-12
