"""The transforms that keep a limb in one workgroup's LDS: every ring degree
that has them, launches of one limb and on both sides of the launch sizes
where they take over, float64 and integer limbs (the 60-bit modulus) in one
launch, word for word against the oracle's NTT and back."""
import numpy as np
import pytest

from helpers import assert_equal_u64, make_params
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# logN: (polynomials, limbs) per launch
SIZES = {
    10: [(1, 1), (1, 5), (30, 4)],
    11: [(1, 1), (3, 5)],
    12: [(1, 1), (24, 4), (97, 1), (20, 5)],
    13: [(1, 2), (127, 1), (64, 2), (26, 5)],
    14: [(1, 2), (51, 5), (64, 4)],
}


@pytest.mark.parametrize("logn", list(SIZES))
def test_one_workgroup_transform(hip_lib, logn):
    q, p = make_params(logn, [60, 50, 50, 40, 50], [61])
    hip_lib.NewSchemeWithModuli(logn, q, p, 50, 64, 5)
    orc = O.Oracle(logn, q, p, h=64, seed=5)
    N = 1 << logn
    rng = np.random.default_rng(logn)
    try:
        for npoly, nrows in SIZES[logn]:
            print(f"[ntt] N=2^{logn}: {npoly} x {nrows} limbs", flush=True)
            x = np.stack([rng.integers(0, q[r], size=(npoly, N), dtype=np.uint64) for r in range(nrows)], axis=1)
            x[0, :, :] = (np.array(q[:nrows], dtype=np.uint64) - 1)[:, None]  # the largest words
            dev = hip_lib.device_upload(x)
            hip_lib.NttDevice(dev.ptr, npoly, nrows, 1)
            hip_lib.Synchronize()
            y = dev.download().reshape(npoly, nrows, N)
            for pi in range(npoly):
                for r in range(nrows):
                    want = orc.ntt(x[pi, r].copy(), r)
                    if not np.array_equal(y[pi, r], want):
                        assert_equal_u64(y[pi, r], want, f"NTT {npoly}x{nrows} poly {pi} limb {r}")
            hip_lib.NttDevice(dev.ptr, npoly, nrows, 0)
            hip_lib.Synchronize()
            back = dev.download().reshape(npoly, nrows, N)
            dev.free()
            assert_equal_u64(back, x, f"iNTT(NTT(x)) {npoly}x{nrows}")
    finally:
        orc.close()
        hip_lib.DeleteScheme()
