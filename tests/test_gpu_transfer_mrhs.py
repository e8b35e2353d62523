"""Project and promote of several right-hand sides (the matrix-core form, and the
vector form in chunks of four where the dispatch keeps it) at the edges of its tiles:
basis widths around multiples of 16 and 4 (odd ones among them), 16-rhs column tiles
with remainders, blocks whose site count is no multiple of a wavefront's four or sixteen
sites, fields of a coarse level (element counts other than 12), masks, panels split over
workgroups, and fields at an address that is no multiple of 16 bytes.

Tolerances as in test_gpu_aggregation.py: relative L2 1e-13 in FP64 and 2e-6 in
FP32, where basis and inputs are rounded to 2^-24 and the sums are FP32.
"""
import ctypes

import numpy as np
import pytest

import oracle
from helpers import gauss, rel

pytestmark = pytest.mark.gpu

# fine lattice, block, nb, elements per site, nrhs
SHAPES = [
    ((4, 4, 4, 4), (4, 4, 4, 4), 16, 12, 12),   # one block, split over workgroups
    ((4, 4, 2, 4), (2, 2, 1, 2), 1, 12, 2),
    ((4, 2, 2, 4), (2, 2, 2, 2), 7, 12, 16),
    ((3, 3, 6, 3), (3, 3, 3, 3), 12, 12, 17),   # 81 sites a block, two column tiles
    ((6, 3, 3, 3), (3, 3, 3, 3), 20, 12, 3),
    ((8, 4, 4, 4), (4, 4, 4, 2), 24, 12, 5),
    ((4, 4, 4, 4), (2, 2, 2, 2), 17, 12, 33),
    ((4, 4, 4, 4), (4, 2, 2, 1), 33, 12, 4),
    ((4, 4, 2, 2), (2, 2, 2, 2), 48, 12, 12),
    ((4, 4, 4, 4), (2, 2, 2, 2), 56, 12, 7),
    ((4, 4, 4, 4), (2, 2, 2, 2), 16, 32, 12),   # a coarse level's field
    ((2, 2, 4, 2), (2, 2, 2, 2), 6, 6, 2),      # three elements per chirality
    ((2, 4, 2, 2), (2, 1, 2, 2), 10, 26, 19),
    ((16, 16, 8, 8), (2, 2, 2, 2), 8, 12, 2),   # 1024 blocks, no split
    ((6, 3, 3, 3), (3, 3, 3, 3), 5, 12, 8),     # at most 8 columns and 8 rhs, 81 sites
    ((4, 4, 4, 4), (2, 2, 4, 4), 8, 12, 9),
    ((16, 16, 8, 8), (4, 2, 2, 2), 56, 12, 5),  # eight wavefronts, the largest LDS of project
    # narrow bases, both sides of the rules that keep the vector form, in chunks of four
    ((4, 4, 4, 4), (2, 2, 2, 2), 4, 12, 9),
    ((6, 3, 3, 3), (3, 3, 3, 3), 3, 12, 9),
    ((3, 3, 3, 6), (3, 3, 3, 3), 4, 12, 17),
    ((12, 12, 12, 24), (3, 3, 3, 3), 2, 12, 7),   # 512 blocks, two chunks: no split
    ((12, 12, 12, 24), (3, 3, 3, 3), 4, 12, 10),
    ((16, 16, 16, 16), (4, 4, 4, 4), 1, 12, 13),
    ((8, 4, 4, 4), (2, 2, 2, 1), 32, 12, 3),      # split small blocks, few rhs
]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("fd,blk,nb,Ef,nrhs", SHAPES)
def test_transfers_match_oracle(gpu, fd, blk, nb, Ef, nrhs, prec):
    print(f"[case] fd={fd} blk={blk} nb={nb} Ef={Ef} nrhs={nrhs} prec={prec}", flush=True)
    Vf, Vc = int(np.prod(fd)), int(np.prod(oracle.coarse_dims(fd, blk)))
    dt = gpu.complex_dtype(prec)
    sz = np.dtype(dt).itemsize
    tol = 1e-13 if prec == 0 else 2e-6
    B = gauss(nb * Vf * Ef, 801).reshape(nb, Vf, Ef)
    agg = gpu.Aggregation(fd, blk, nb, Ef)
    agg.set_basis(gpu.DeviceBuffer.from_numpy(B))
    f = gauss(Vf * nrhs * Ef, 802).reshape(Vf, nrhs, Ef).astype(dt)
    c = gauss(Vc * nrhs * 2 * nb, 803).reshape(Vc, nrhs, 2 * nb).astype(dt)
    ref_c, ref_f = [], []
    for r in range(nrhs):
        ref_c.append(oracle.project_ef(fd, blk, nb, Ef, B, f[:, r].astype(np.complex128)))
        ref_f.append(oracle.promote_ef(fd, blk, nb, Ef, B, c[:, r].astype(np.complex128)))
    ref_c, ref_f = np.stack(ref_c, 1), np.stack(ref_f, 1)
    real = np.float64 if prec == 0 else np.float32
    for shift in (0, 8):  # the fields eight bytes into their buffers
        k = shift // np.dtype(real).itemsize
        pad = np.zeros(k, real)
        df = gpu.DeviceBuffer.from_numpy(np.concatenate([pad, f.ravel().view(real)]))
        dc = gpu.DeviceBuffer.from_numpy(np.concatenate([pad, c.ravel().view(real)]))
        oc = gpu.DeviceBuffer(Vc * nrhs * 2 * nb * sz)
        of = gpu.DeviceBuffer(f.size * sz + 2 * shift)
        of.zero()
        agg.project(df.ptr + shift, oc, prec, nrhs)
        agg.promote(dc.ptr + shift, of.ptr + shift, prec, nrhs)
        gpu.synchronize()
        got_c = oc.to_numpy(dt, ref_c.shape)
        raw = of.to_numpy(real, (2 * f.size + 2 * k,))
        got_f = raw[k:k + 2 * f.size].view(dt).reshape(ref_f.shape)
        for r in range(nrhs):
            assert rel(ref_c[:, r], got_c[:, r].astype(np.complex128)) < tol, (shift, r)
            assert rel(ref_f[:, r], got_f[:, r].astype(np.complex128)) < tol, (shift, r)
        assert not raw[:k].any() and not raw[k + 2 * f.size:].any()


@pytest.mark.parametrize("prec", [0, 1])
def test_masked_project_of_many_rhs(gpu, prec):
    """Inner and outer sites of each point on blocks with an odd extent."""
    fd, blk, nb, nrhs = (6, 4, 4, 3), (3, 2, 4, 3), 18, 18
    print(f"[case] masked fd={fd} blk={blk} nb={nb} nrhs={nrhs} prec={prec}", flush=True)
    Vf, Vc = int(np.prod(fd)), int(np.prod(oracle.coarse_dims(fd, blk)))
    dt = gpu.complex_dtype(prec)
    tol = 1e-13 if prec == 0 else 2e-6
    B = gauss(nb * Vf * 12, 811).reshape(nb, Vf, 12)
    agg = gpu.Aggregation(fd, blk, nb)
    agg.set_basis(gpu.DeviceBuffer.from_numpy(B))
    f = gauss(Vf * nrhs * 12, 812).reshape(Vf, nrhs, 12).astype(dt)
    df = gpu.DeviceBuffer.from_numpy(f)
    dc = gpu.DeviceBuffer(Vc * nrhs * 2 * nb * np.dtype(dt).itemsize)
    for point in range(9):
        for kind in (0, 1, 2):
            if kind == 2 and point == 8:
                continue  # no site is outside the self point
            agg.project_masked(df, dc, kind, point, prec, nrhs)
            gpu.synchronize()
            got = dc.to_numpy(dt, (Vc, nrhs, 2 * nb)).astype(np.complex128)
            for r in (0, 7, nrhs - 1):
                ref = oracle.project(fd, blk, nb, B, f[:, r].astype(np.complex128), kind=kind,
                                     point=point)
                assert rel(ref, got[:, r]) < tol, (point, kind, r)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("first,then", [(1, 4), (2, 3), (5, 8), (13, 16)])
def test_wider_projection_of_a_group_of_four_is_capturable(gpu, first, then, prec):
    """One block, so that its panel is split and the partial sums take a workspace:
    the one that a call of `first` rhs leaves serves `then` rhs under capture, where
    nothing can be allocated.  Every replay gives the eager result."""
    print(f"[case] capture first={first} then={then} prec={prec}", flush=True)
    fd, nb = (4, 4, 4, 4), 8
    Vf = int(np.prod(fd))
    dt = gpu.complex_dtype(prec)
    agg = gpu.Aggregation(fd, fd, nb)
    agg.set_basis(gpu.DeviceBuffer.from_numpy(gauss(nb * Vf * 12, 851)))
    df = gpu.DeviceBuffer.from_numpy(gauss(Vf * then * 12, 852).astype(dt))
    shape = (then, 2 * nb)
    want, got = (gpu.DeviceBuffer(then * 2 * nb * np.dtype(dt).itemsize) for _ in range(2))
    gpu.synchronize()
    hip, s = gpu.lib(), gpu.Stream()  # the HIP runtime is a dependency of the library
    agg.project(df, want, prec, first, stream=s)
    s.sync()
    graph, ex = ctypes.c_void_p(), ctypes.c_void_p()
    st = ctypes.c_void_p(s.handle)
    assert hip.hipStreamBeginCapture(st, 1) == 0  # thread-local mode
    try:
        agg.project(df, got, prec, then, stream=s)
    finally:
        end = hip.hipStreamEndCapture(st, ctypes.byref(graph))
    assert end == 0
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    try:
        for _ in range(3):
            got.zero()
            gpu.synchronize()
            assert hip.hipGraphLaunch(ex, st) == 0
            s.sync()
            agg.project(df, want, prec, then, stream=s)
            s.sync()
            assert np.array_equal(got.to_numpy(dt, shape), want.to_numpy(dt, shape))
    finally:
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(graph)
