"""Exact round trips through the tiled layout conversions: links (whole matrices or
32 x 32 tiles by N; both external layouts) and basis (48 or 192 panel rows a tile), at
sizes with partial tiles.  Values are moved, not computed: equality bit for bit (FP32
operators: equality with the rounded input)."""
import numpy as np
import pytest

import oracle
from helpers import gauss, rand_links

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("N", [2, 6, 14, 30, 32, 34, 48, 50, 64, 66])
def test_links_round_trip(gpu, N, prec):
    print(f"[case] links N={N} prec={prec}", flush=True)
    dims = (2, 1, 3, 2)
    V = int(np.prod(dims))
    links = rand_links(dims, N)
    op = gpu.CoarseOp(dims, N, prec)
    op.set_links(gpu.DeviceBuffer.from_numpy(links), gpu.LAYOUT_FLAT, invert=False)
    want = links.reshape(9, V, N, N)
    if prec == 1:
        want = want.astype(np.complex64).astype(np.complex128)
    out = gpu.DeviceBuffer(links.nbytes)
    op.get_links(out, gpu.LAYOUT_FLAT)
    gpu.synchronize()
    assert np.array_equal(out.to_numpy(np.complex128, want.shape), want)
    op.get_links(out, gpu.LAYOUT_SPLIT)
    gpu.synchronize()
    got = out.to_numpy(np.complex128, (9, V, 2, 2, N // 2, N // 2))
    split = want.reshape(9, V, 2, N // 2, 2, N // 2).transpose(0, 1, 2, 4, 3, 5)
    assert np.array_equal(got, split)


@pytest.mark.parametrize("disp_have", [1, -1])
@pytest.mark.parametrize("N", [2, 12, 32, 34, 48, 50])
def test_reconstructed_links(gpu, N, disp_have):
    """Links are conjugated and moved: equality bit for bit."""
    print(f"[case] reconstruct N={N} disp_have={disp_have}", flush=True)
    dims = (2, 5, 3, 2)
    V = int(np.prod(dims))
    links = rand_links(dims, N)
    op = gpu.CoarseOp(dims, N, gpu.F64)
    op.set_links(gpu.DeviceBuffer.from_numpy(links), gpu.LAYOUT_FLAT, invert=False)
    gpu.construct_remaining_links(op, disp_have)
    out = gpu.DeviceBuffer(links.nbytes)
    op.get_links(out, gpu.LAYOUT_FLAT)
    gpu.synchronize()
    want = oracle.construct_remaining_links(dims, N, links, disp_have).reshape(9, V, N, N)
    assert np.array_equal(out.to_numpy(np.complex128, want.shape), want)


@pytest.mark.parametrize("fd,blk,nb,Ef", [((2, 3, 1, 1), (1, 3, 1, 1), 1, 2),
                                          ((6, 3, 3, 3), (3, 3, 1, 3), 3, 26),
                                          ((4, 4, 2, 2), (2, 2, 2, 1), 4, 12),
                                          ((4, 4, 2, 2), (2, 2, 2, 1), 5, 12),
                                          ((4, 4, 2, 2), (2, 2, 2, 1), 17, 12),
                                          ((6, 3, 3, 3), (3, 3, 3, 3), 33, 26),
                                          ((4, 2, 2, 2), (2, 2, 1, 2), 64, 12)])
def test_basis_round_trip(gpu, fd, blk, nb, Ef):
    print(f"[case] basis fd={fd} blk={blk} nb={nb} Ef={Ef}", flush=True)
    Vf = int(np.prod(fd))
    B = gauss(nb * Vf * Ef, 821).reshape(nb, Vf, Ef)
    agg = gpu.Aggregation(fd, blk, nb, Ef)
    agg.set_basis(gpu.DeviceBuffer.from_numpy(B))
    out = gpu.DeviceBuffer(B.nbytes)
    agg.get_basis(out)
    gpu.synchronize()
    assert np.array_equal(out.to_numpy(np.complex128, B.shape), B)
    # the panels themselves: a projection reads them in their own order
    f = gauss(Vf * Ef, 822).reshape(Vf, Ef)
    Vc = int(np.prod(oracle.coarse_dims(fd, blk)))
    oc = gpu.DeviceBuffer(Vc * 2 * nb * 16)
    agg.project(gpu.DeviceBuffer.from_numpy(f), oc, 0, 1)
    gpu.synchronize()
    ref = oracle.project_ef(fd, blk, nb, Ef, B, f)
    got = oc.to_numpy(np.complex128, (Vc, 2 * nb))
    assert np.linalg.norm(got - ref) < 1e-13 * np.linalg.norm(ref)


def part(gpu, buf, first, shape):
    """Elements [first, ...) of a complex128 buffer."""
    out = np.empty(shape, np.complex128)
    gpu.call("mgc_memcpy_d2h", out.ctypes.data, buf.ptr + first * 16, out.nbytes, None)
    gpu.synchronize()
    return out


@pytest.mark.parametrize("N,dims,prec", [(34, (26, 26, 26, 27), 1), (50, (18, 18, 18, 20), 1),
                                         (2, (38, 37, 36, 37), 0), (2, (38, 37, 36, 37), 1)])
def test_links_round_trip_of_many_tiles(gpu, N, dims, prec):
    """More tiles than one launch has workgroups, or more than it may have work items
    (132 GB and 70 GB in all for the first two): the first, last and some sites between."""
    print(f"[case] many tiles N={N} dims={dims}", flush=True)
    V = int(np.prod(dims))
    buf = gpu.DeviceBuffer(9 * V * N * N * 16)
    gpu.random_gaussian(buf, 9 * V * N * N, gpu.F64, 5, 861)
    at = [(p, x) for p in (0, 4, 8) for x in (0, 1, V // 3, V // 2 + 1, V - 2)]
    want = [part(gpu, buf, (p * V + x) * N * N, (2, N, N)) for p, x in at]
    op = gpu.CoarseOp(dims, N, prec)
    op.set_links(buf, gpu.LAYOUT_FLAT, invert=False)
    buf.zero()
    op.get_links(buf, gpu.LAYOUT_FLAT)
    gpu.synchronize()
    for (p, x), w in zip(at, want):
        got = part(gpu, buf, (p * V + x) * N * N, (2, N, N))
        assert np.array_equal(got, w.astype(gpu.complex_dtype(prec)).astype(np.complex128)), (p, x)
    buf.close()
    op.close()


@pytest.mark.parametrize("dims,blk,nb,Ef", [((32, 16, 32, 32), (2, 2, 2, 1), 4, 12),
                                            ((64, 64, 32, 33), (2, 4, 1, 3), 1, 256)])
def test_basis_round_trip_of_many_tiles(gpu, dims, blk, nb, Ef):
    """As above (18 GB a copy): the import against the export."""
    print(f"[case] many tiles basis dims={dims} blk={blk} nb={nb} Ef={Ef}", flush=True)
    V = int(np.prod(dims))
    src, back = gpu.DeviceBuffer(nb * V * Ef * 16), gpu.DeviceBuffer(nb * V * Ef * 16)
    gpu.random_gaussian(src, nb * V * Ef, gpu.F64, 5, 862)
    agg = gpu.Aggregation(dims, blk, nb, Ef)
    agg.set_basis(src)
    agg.get_basis(back)
    gpu.synchronize()
    for i in (0, nb - 1):
        for x in (0, 1, V // 3, V // 2 + 1, V - 2):
            first = (i * V + x) * Ef
            assert np.array_equal(part(gpu, back, first, (2, Ef)), part(gpu, src, first, (2, Ef)))
    src.close()
    back.close()
    agg.close()
