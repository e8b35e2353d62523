"""The staged forms of the fine-operator apply against the plain one (a thread
reads its own records), bit for bit: they run the same per-thread arithmetic in
the same order.  Lattices with partial tiles and without the XCD-local order, the
rhs counts around each form's limits, and point masks that leave stages out."""
import numpy as np
import pytest

from helpers import gauss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dims", [(2, 3, 5, 3), (4, 4, 4, 4), (8, 8, 4, 8)])
@pytest.mark.parametrize("nrhs", [1, 2, 4, 5, 8, 9, 12, 17, 64, 129])
def test_forms_bit_equal(gpu, dims, nrhs, prec):
    print(f"[case] wilson forms dims={dims} nrhs={nrhs} prec={prec}", flush=True)
    V = int(np.prod(dims))
    dt = gpu.complex_dtype(prec)
    op = gpu.FineOp(dims, -0.1, 1.0)
    g = gpu.DeviceBuffer(4 * V * 9 * 16)
    gpu.random_gauge(g, dims)
    op.set_gauge(g)
    x = gauss(V * nrhs * 12, 831).astype(dt)
    din, dout = gpu.DeviceBuffer.from_numpy(x), gpu.DeviceBuffer(x.nbytes)
    calls = [lambda: op.M(din, dout, prec, nrhs), lambda: op.Mdag(din, dout, prec, nrhs),
             lambda: op.Mdiag(din, dout, prec, nrhs)]
    calls += [lambda p=p: op.Mdir(din, dout, p % 4, 1 if p < 4 else -1, prec, nrhs)
              for p in (0, 3, 6, 7)]
    for i, call in enumerate(calls):
        got = []
        for variant in (0, -1):
            gpu.call("mgc_fine_op_set_variant", variant)
            try:
                dout.zero()
                call()
                gpu.synchronize()
            finally:
                gpu.call("mgc_fine_op_set_variant", -1)
            got.append(dout.to_numpy(dt, x.shape))
        assert np.array_equal(got[0], got[1]), i
