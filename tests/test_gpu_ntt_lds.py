"""The transforms that keep a limb in one workgroup's LDS: every ring degree
that has them, launches of one limb and on both sides of the launch sizes
where they take over, float64 and integer limbs (the 60-bit modulus) in one
launch, word for word against the oracle's NTT and back; and the fused
epilogues (ModDown, pair of rescales) of launches that run that way above
N = 2^11, through the linear transform and the polynomial they belong to."""
import numpy as np
import pytest

from helpers import assert_equal_u64, make_params, new_hip_scheme
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


# (logN, limbs): the key-switched giant groups divide by P in one launch of a
# transform a group and limb, from 97, 128 and 256 of them on in LDS
MODDOWNS = [(12, 5), (13, 6), (14, 12)]


@pytest.mark.parametrize("logn,limbs", MODDOWNS)
def test_one_workgroup_moddown(hip_lib, logn, limbs):
    """The giant groups' ModDown, whose forward transform ends in the epilogue
    that combines, and their decomposition, in a launch that runs in one
    workgroup's LDS a limb: the whole transform against the oracle's."""
    q, p = make_params(logn, [60, 50, 40, 55] + [45] * (limbs - 4), [61] * 4)
    slots, level, scale = 1 << (logn - 1), limbs - 1, float(1 << 40)
    new_hip_scheme(hip_lib, logn, q, p, 40, 64, 5, evaluator=False)
    orc = O.Oracle(logn, q, p, h=64, seed=5)
    rng = np.random.default_rng(logn)
    idx = sorted(rng.choice(slots, 32, replace=False).tolist())
    data = rng.uniform(-1, 1, (len(idx), slots)).astype(np.float32)
    vals = rng.uniform(-1, 1, slots).astype(np.float32)
    try:
        tid = hip_lib.GenerateLinearTransform(idx, data.reshape(-1), level, 2.0, "none")
        groups = hip_lib.lt_info(tid)["giant"] - 1  # one may have no rotation
        assert groups * limbs >= max(97, 1 << (logn - 6)), groups
        for ge in hip_lib.GetLinearTransformRotationKeys(tid):
            hip_lib.GenerateLinearTransformRotationKey(ge)
        print(f"[moddown] N=2^{logn}: {groups} groups of {limbs} limbs", flush=True)
        hip_lib.SetEncryptionCounter(0)
        ct = hip_lib.Encrypt(hip_lib.Encode(vals, level, 1 << 40))
        out = hip_lib.EvaluateLinearTransform(tid, ct)
        t = orc.lt_new(idx, data, level, 2.0)
        want, _ = orc.lt_eval(t, orc.encrypt(orc.encode(vals, level, scale), level, 0), level)
        orc.lt_free(t)
        assert_equal_u64(hip_lib.export_ciphertext(out), want, f"N=2^{logn} transform")
    finally:
        orc.close()
        hip_lib.DeleteScheme()


def test_one_workgroup_rescale_pair(hip_lib):
    """The degree-3 polynomial's scaled pair of rescales (an epilogue of its
    own) over 4 * 26 limbs of N = 2^12, in LDS."""
    logn, top, logscale = 12, 26, 45
    q, p = make_params(logn, [60] + [45] * top, [61] * 4)
    new_hip_scheme(hip_lib, logn, q, p, logscale, 64, 5, evaluator=False)
    orc = O.Oracle(logn, q, p, h=64, seed=5)
    scale = float(1 << logscale)
    c32 = np.asarray([0.047, 0.5, 0.24, -0.003], dtype=np.float32)
    vals = np.random.default_rng(6).uniform(-1, 1, 1 << (logn - 1)).astype(np.float32)
    try:
        hip_lib.GenerateRelinearizationKey()
        hip_lib.NewPolynomialEvaluator()
        hip_lib.SetEncryptionCounter(0)
        ct = hip_lib.Encrypt(hip_lib.Encode(vals, top, 1 << logscale))
        print(f"[pair] N=2^{logn}: {4 * top} limbs", flush=True)
        out = hip_lib.EvaluatePolynomial(ct, hip_lib.GenerateMonomial(c32.tolist()), 1 << logscale)
        ref = orc.encrypt(orc.encode(vals, top, scale), top, 0)
        want, _ = orc.eval_poly(ref, top, scale, c32.astype(np.float64), scale)
        assert_equal_u64(hip_lib.export_ciphertext(out), want, "polynomial")
    finally:
        orc.close()
        hip_lib.DeleteScheme()
