"""Rounding error of the block transfers: no larger than that of a sum in so many
partial sums.

A chain of n additions leaves an error that grows with sqrt(n), so the number of
partial sums an element is formed in decides it.  Each case restates on the host a
sum in a stated number of partial sums (fused multiply-adds rounded to the
precision under test, computed in the next wider type), measures its error against
the same sum in extended precision, and asks of the GPU an error not above 1.06
times that: two estimates of one error over 1e4 and more results of two parts each
differ by 1% (one standard deviation) where the orders differ, and one chain
instead of two is 1.22 times and more above.
"""
import numpy as np
import pytest

import oracle
from helpers import gauss

pytestmark = pytest.mark.gpu
SLACK = 1.06
REAL = {0: np.float64, 1: np.float32}
WIDE = {0: np.longdouble, 1: np.float64}


def fma(prec, acc, a, b, sign=1):
    w = WIDE[prec]
    return (acc.astype(w) + sign * (a.astype(w) * b.astype(w))).astype(REAL[prec])


def cmac(prec, acc, a, b, conj_b=False):
    """acc + a b (or a conj(b)), real and imaginary part by two fused multiply-adds each."""
    s = -1 if conj_b else 1
    re, im = acc
    re = fma(prec, fma(prec, re, a.real, b.real), a.imag, b.imag, -s)
    im = fma(prec, fma(prec, im, a.imag, b.real), a.real, b.imag, s)
    return re, im


def add(x, y):
    return x[0] + y[0], x[1] + y[1]


def rms(got, want):
    d = got.astype(np.clongdouble) - want
    return float(np.sqrt((abs(d) ** 2).sum() / (abs(want) ** 2).sum()))


def block_rows(fd, blk, f):
    """[V, ..., Ef] as [block, row of a panel, ...] (row = block site, element)."""
    V, Ef = f.shape[0], f.shape[-1]
    cd = oracle.coarse_dims(fd, blk)
    mid = f.shape[1:-1]
    g = f.reshape(cd[3], blk[3], cd[2], blk[2], cd[1], blk[1], cd[0], blk[0], *mid, Ef)
    g = np.moveaxis(g, (0, 2, 4, 6), (0, 1, 2, 3))
    g = g.reshape(int(np.prod(cd)), int(np.prod(blk)), *mid, Ef)
    g = np.moveaxis(g, -1, 2)
    return g.reshape(g.shape[0], -1, *mid)


def promote_lanes(prec, nb):
    """Partial sums of an element: the lanes that share a row of a 64 KB tile."""
    if prec == 1 and nb <= 30:
        return 1
    return 2 if nb <= (59 if prec == 1 else 29) else 4


@pytest.mark.parametrize("nrhs", [1, 2, 5])
@pytest.mark.parametrize("prec,nb", [(0, 8), (0, 16), (0, 29), (0, 30), (0, 31), (0, 40),
                                     (0, 48), (0, 56), (1, 16), (1, 30), (1, 31), (1, 32),
                                     (1, 48), (1, 60), (1, 64)])
def test_promote_error(gpu, prec, nb, nrhs):
    print(f"[case] promote rounding nb={nb} nrhs={nrhs} prec={prec}", flush=True)
    fd, blk, Ef = (8, 4, 4, 4), (2, 2, 2, 2), 12
    Vf, Vc = int(np.prod(fd)), int(np.prod(oracle.coarse_dims(fd, blk)))
    ct = gpu.complex_dtype(prec)
    B = gauss(nb * Vf * Ef, 841).astype(ct).reshape(nb, Vf, Ef)
    c = gauss(Vc * nrhs * 2 * nb, 842).astype(ct).reshape(Vc, nrhs, 2, nb)
    agg = gpu.Aggregation(fd, blk, nb, Ef)
    agg.set_basis(gpu.DeviceBuffer.from_numpy(B.astype(np.complex128)))
    of = gpu.DeviceBuffer(Vf * nrhs * Ef * np.dtype(ct).itemsize)
    agg.promote(gpu.DeviceBuffer.from_numpy(c), of, prec, nrhs)
    gpu.synchronize()
    got = block_rows(fd, blk, of.to_numpy(ct, (Vf, nrhs, Ef)))          # [block][row][rhs]
    U = block_rows(fd, blk, B.transpose(1, 0, 2))                       # [block][row][nb]
    half = np.tile(np.arange(Ef) >= Ef // 2, int(np.prod(blk))).astype(int)
    C = c.transpose(0, 2, 1, 3)[:, half]                                # [block][row][rhs][nb]
    want = (C.astype(np.clongdouble) * U[:, :, None, :]).sum(-1)
    lanes = promote_lanes(prec, nb)
    per = -(-nb // lanes)
    sums = []
    for h in range(lanes):
        acc = (np.zeros(got.shape, REAL[prec]),) * 2
        for i in range(h * per, min(nb, h * per + per)):
            acc = cmac(prec, acc, C[..., i], U[:, :, None, i])
        sums.append(acc)
    while len(sums) > 1:
        sums = [add(sums[2 * q], sums[2 * q + 1]) for q in range(len(sums) // 2)]
    model = rms(sums[0][0] + 1j * sums[0][1], want)
    err = rms(got, want)
    print(f"error {err:.3e}, {lanes} partial sums on the host {model:.3e}", flush=True)
    assert err <= SLACK * model


def split(total, parts):
    """[lo, hi) of equal ranges, the last one shorter."""
    per = -(-total // parts)
    return [(lo, min(total, lo + per)) for lo in range(0, total, per)]


def in_order(terms):
    acc = terms[0]
    for t in terms[1:]:
        acc = add(acc, t)
    return acc


# fine lattice, block, elements per site
PROJECT = [((8, 8, 8, 4), (2, 1, 1, 1), 12), ((8, 8, 8, 2), (2, 2, 1, 1), 12),
           ((8, 8, 4, 4), (2, 2, 2, 2), 12), ((6, 6, 6, 6), (3, 3, 3, 3), 12),
           ((8, 8, 8, 8), (4, 4, 4, 4), 12), ((4, 4, 4, 2), (2, 2, 1, 1), 128),
           ((4, 4, 4, 4), (2, 2, 2, 2), 64)]


@pytest.mark.parametrize("nrhs", [1, 2, 5])
@pytest.mark.parametrize("prec,nb", [(0, 8), (0, 16), (0, 24), (0, 32), (0, 48), (1, 16), (1, 24),
                                     (1, 32), (1, 48), (1, 64)])
@pytest.mark.parametrize("fd,blk,Ef", PROJECT)
def test_project_error(gpu, fd, blk, Ef, prec, nb, nrhs):
    """Against a panel's rows dealt to 256 / nb groups (twice as many in FP32, which
    takes two columns a thread), the rows of a group and then the groups added in
    order, over as many row ranges as fill the chip (1024 / (blocks * chunks of four
    rhs), 64 rows at least), and the ranges added by 256 / (8 nb) threads each."""
    print(f"[case] project rounding fd={fd} blk={blk} Ef={Ef} nb={nb} nrhs={nrhs} prec={prec}",
          flush=True)
    Vf, Vc = int(np.prod(fd)), int(np.prod(oracle.coarse_dims(fd, blk)))
    ct = gpu.complex_dtype(prec)
    B = gauss(nb * Vf * Ef, 843).astype(ct).reshape(nb, Vf, Ef)
    f = gauss(Vf * nrhs * Ef, 844).astype(ct).reshape(Vf, nrhs, Ef)
    agg = gpu.Aggregation(fd, blk, nb, Ef)
    agg.set_basis(gpu.DeviceBuffer.from_numpy(B.astype(np.complex128)))
    oc = gpu.DeviceBuffer(Vc * nrhs * 2 * nb * np.dtype(ct).itemsize)
    agg.project(gpu.DeviceBuffer.from_numpy(f), oc, prec, nrhs)
    gpu.synchronize()
    got = oc.to_numpy(ct, (Vc, nrhs, 2, nb))
    U = block_rows(fd, blk, B.transpose(1, 0, 2))     # [block][row][nb]
    F = block_rows(fd, blk, f)                        # [block][row][rhs]
    rows = U.shape[1]
    sel = slice(0, max(1, 60000 // (nrhs * 2 * nb)))  # blocks compared
    U, F, got = U[sel], F[sel], got[sel]
    wgs = Vc * -(-nrhs // 4)
    S = max(1, min(-(-1024 // wgs), rows // 64)) if wgs < 1024 else 1
    G = 256 // nb * (2 if prec == 1 else 1)
    zg = max(1, 256 // (8 * nb))
    err, model = np.zeros(2), np.zeros(2)
    for k in range(2):
        mine = np.arange(rows) % Ef // (Ef // 2) == k
        want = np.einsum("bqi,bqr->bri", U[:, mine].conj().astype(np.clongdouble),
                         F[:, mine].astype(np.clongdouble))
        ranges = []
        for lo, hi in split(rows, S):
            groups = []
            for g in range(G):
                acc = (np.zeros(want.shape, REAL[prec]),) * 2
                for q in range(lo + g, hi, G):
                    if mine[q]:
                        acc = cmac(prec, acc, F[:, q, :, None], U[:, q, None, :], conj_b=True)
                groups.append(acc)
            ranges.append(in_order(groups))
        re, im = in_order([in_order(ranges[z::zg]) for z in range(min(zg, len(ranges)))])
        err[k], model[k] = rms(got[:, :, k], want), rms(re + 1j * im, want)
    print(f"error {err}, on the host {model}", flush=True)
    assert np.hypot(*err) <= SLACK * np.hypot(*model)
