"""The giant steps' key products, by digit count (each has its kernel up to
eight digits, a loop above), with keys generated here and loaded (a halves
read), and by number of groups: transforms with and without the unrotated
group, more groups than an accumulator holds.  Word for word against the
oracle's transform."""
import numpy as np
import pytest

from helpers import assert_equal_u64, make_params, new_hip_scheme
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (limbs, special moduli): 1, 2, 3, 4, 5, 6, 7, 8 and 9 digits at the top level
CHAINS = [(3, 3), (4, 2), (7, 3), (4, 1), (5, 1), (11, 2), (7, 1), (8, 1), (9, 1)]


@pytest.mark.parametrize("limbs,special", CHAINS)
def test_giant_steps_by_digits(hip_lib, limbs, special):
    logn, logscale = 10, 40
    q, p = make_params(logn, [60] + [45] * (limbs - 1), [61] * special)
    slots, level = 1 << (logn - 1), limbs - 1
    new_hip_scheme(hip_lib, logn, q, p, logscale, 64, 3, evaluator=False)
    orc = O.Oracle(logn, q, p, h=64, seed=3)
    rng = np.random.default_rng(limbs)
    vals = rng.uniform(-1, 1, slots).astype(np.float32)
    try:
        sets = ([0, 1, 3, 17, 40, 90], [5 + 16 * i for i in range(3, 25)])
        for n, idx in enumerate(sets):
            data = rng.uniform(-1, 1, (len(idx), slots)).astype(np.float32)
            tid = hip_lib.GenerateLinearTransform(list(idx), data.reshape(-1), level, 2.0, "none")
            t = orc.lt_new(list(idx), data, level, 2.0)
            want, _ = orc.lt_eval(t, orc.encrypt(orc.encode(vals, level, float(1 << logscale)), level, n), level)
            orc.lt_free(t)
            for loaded in (False, True):
                print(f"[giant] {limbs} limbs, {special} special, set {n}, loaded keys {loaded}", flush=True)
                for ge in hip_lib.GetLinearTransformRotationKeys(tid):
                    if loaded:
                        key, ptr = hip_lib.GenerateAndSerializeRotationKey(ge)
                        hip_lib.FreeCArray(ptr)
                        hip_lib.LoadRotationKey(key, ge)
                    else:
                        hip_lib.GenerateLinearTransformRotationKey(ge)
                hip_lib.SetEncryptionCounter(n)
                ct = hip_lib.Encrypt(hip_lib.Encode(vals, level, 1 << logscale))
                out = hip_lib.EvaluateLinearTransform(tid, ct)
                assert_equal_u64(hip_lib.export_ciphertext(out), want, f"set {n} loaded {loaded}")
            hip_lib.DeleteLinearTransform(tid)
    finally:
        orc.close()
        hip_lib.DeleteScheme()
