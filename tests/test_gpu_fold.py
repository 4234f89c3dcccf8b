"""RotateAddMany (a Linear's whole output fold: consecutive key switches that
share their transforms) against the oracle's rotate + add per step, word for
word, over the shapes where its kernels can go wrong: one and several special
moduli, a last digit of one modulus, digits from one to the unrolled kernel's
most (and one past it, which runs step by step), rings whose transforms take
the small and the large launches, rotations of every sign pattern, keys
generated here and loaded."""
import numpy as np
import pytest

from helpers import assert_equal_u64, make_params, new_hip_scheme
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# name: (logN, logq, logp, levels)
SHAPES = {
    "k1_dn5": (13, [60, 40, 40, 40, 40], [61], (4, 3, 0)),
    "k3_dn3": (13, [60] + [50] * 6, [61] * 3, (6, 5, 2)),
    "k8_dn1_dn4": (12, [60] + [50] * 25, [61] * 8, (25, 24, 7, 0)),
    "k2_dn8_dn9": (11, [55] + [45] * 16, [56] * 2, (16, 15, 14)),
    "k9": (11, [55] + [45] * 9, [56] * 9, (9,)),
    "n14": (14, [60] + [50] * 11, [61] * 4, (11,)),
}


@pytest.mark.parametrize("name", list(SHAPES))
def test_fold_matches_oracle(hip_lib, name):
    logn, logq, logp, levels = SHAPES[name]
    q, p = make_params(logn, logq, logp)
    slots = 1 << (logn - 1)
    scale = float(1 << 40)
    new_hip_scheme(hip_lib, logn, q, p, 40, 64, 31)
    orc = O.Oracle(logn, q, p, h=64, seed=31)
    rng = np.random.default_rng(3)
    try:
        for n, level in enumerate(levels):
            # the fold's halving amounts, then odd and negative ones (other sign patterns), one amount alone
            for j, amounts in enumerate(([slots // 2, slots // 4, slots // 8, slots // 16], [3, -1], [5])):
                print(f"[fold] {name} level {level} amounts {amounts}", flush=True)
                index = 8 * n + j
                vals = rng.uniform(-1, 1, slots).astype(np.float32)
                hip_lib.SetEncryptionCounter(index)
                pt = hip_lib.Encode(vals, level, int(scale))
                ct = hip_lib.Encrypt(pt)
                want = orc.encrypt(orc.encode(vals, level, scale), level, index)
                for a in amounts:
                    want = orc.add(want, orc.rotate(want, level, a), level)
                assert hip_lib.RotateAddMany(ct, amounts) == ct
                assert_equal_u64(hip_lib.export_ciphertext(ct), want, f"{name} level {level} fold {amounts}")
                hip_lib.DeletePlaintext(pt)
                hip_lib.DeleteCiphertext(ct)
    finally:
        orc.close()
        hip_lib.DeleteScheme()


def test_fold_full_size_equals_single_steps(hip_lib):
    """N = 2^16, 24 limbs, three digits: the fold of the 26-table lookup
    against RotateAdd step by step, once with generated and once with loaded
    keys (whose a halves are read)."""
    from helrm_amd import orion_host as oh
    params = oh.Params(16, [60] + [50] * 23, [61] * 8, 50, 192, seed=9)
    scheme = oh.Scheme(params, hip_lib)
    slots = params.get_slots()
    amounts = [slots >> i for i in range(1, 7)]
    vals = np.random.default_rng(4).uniform(-1, 1, slots)
    try:
        for loaded in (False, True):
            print(f"[fold] full size, loaded keys: {loaded}", flush=True)
            if loaded:
                for a in amounts[:3]:
                    g = pow(5, a, 4 * slots)
                    data, ptr = hip_lib.GenerateAndSerializeRotationKey(g)
                    hip_lib.FreeCArray(ptr)
                    hip_lib.LoadRotationKey(data, g)
            for level in (22, 7):
                ct = scheme.encrypt(scheme.encode(vals, level))
                ref = hip_lib.import_ciphertext(hip_lib.export_ciphertext(ct.ids[0]), level, float(1 << 50))
                ct.fold(amounts)
                for a in amounts:
                    hip_lib.RotateAdd(ref, a)
                assert_equal_u64(hip_lib.export_ciphertext(ct.ids[0]), hip_lib.export_ciphertext(ref), f"level {level}")
    finally:
        hip_lib.DeleteScheme()


def test_fold_refuses_and_leaves_input(hip_lib):
    q, p = make_params(11, [40, 30, 30], [41])
    new_hip_scheme(hip_lib, 11, q, p, 30, 64, 5)
    try:
        ct = hip_lib.Encrypt(hip_lib.Encode(np.ones(4, np.float32), 2, 1 << 30))
        before = hip_lib.export_ciphertext(ct)
        from helrm_amd.backend import HipError
        with pytest.raises(HipError, match="ciphertext not found"):
            hip_lib.RotateAddMany(ct + 100, [1, 2])
        assert hip_lib.RotateAddMany(ct, []) == ct
        for amounts, length in ((None, 2), (None, -1)):
            assert hip_lib.RotateAddMany.func(ct, amounts, length) == -1
        assert_equal_u64(hip_lib.export_ciphertext(ct), before, "empty fold")
    finally:
        hip_lib.DeleteScheme()
