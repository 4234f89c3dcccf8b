"""One linear transform evaluated on ciphertexts of several levels: what it
keeps between calls (key and permutation tables, the stream keys of generated
keys) serves a level of fewer digits and a higher level after it, in either
order.  Word for word against the oracle's transform, with keys generated here
(their a halves regenerated from the stream keys)."""
import numpy as np
import pytest

from helpers import assert_equal_u64, make_params, new_hip_scheme
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (limbs, special moduli, levels): the unrolled giant products and the loop
# above eight digits; digit counts 4 -> 2, 6 -> 3 -> 1, 9 -> 8 -> 2
CHAINS = [(7, 2, (6, 3)), (11, 2, (10, 4, 1)), (17, 2, (16, 15, 3))]
# few scattered diagonals, and a dense block of 16 baby steps (packed diagonals)
SETS = {"scattered": [0, 1, 3, 17, 40, 90, 201], "dense16": list(range(256))}


@pytest.mark.parametrize("set_name", list(SETS))
@pytest.mark.parametrize("limbs,special,levels", CHAINS)
def test_transform_at_several_levels(hip_lib, limbs, special, levels, set_name):
    logn, logscale, idx = 10, 40, SETS[set_name]
    q, p = make_params(logn, [60] + [45] * (limbs - 1), [61] * special)
    slots, top = 1 << (logn - 1), limbs - 1
    new_hip_scheme(hip_lib, logn, q, p, logscale, 64, 3, evaluator=False)
    orc = O.Oracle(logn, q, p, h=64, seed=3)
    rng = np.random.default_rng(limbs)
    vals = rng.uniform(-1, 1, slots).astype(np.float32)
    data = rng.uniform(-1, 1, (len(idx), slots)).astype(np.float32)
    t = orc.lt_new(idx, data, top, 2.0)
    try:
        want = {}
        for n, level in enumerate(levels):
            want[level], _ = orc.lt_eval(t, orc.encrypt(orc.encode(vals, level, float(1 << logscale)), level, n), level)
        for order in (levels, levels[::-1]):
            # a transform of its own an order: the first call builds its tables
            tid = hip_lib.GenerateLinearTransform(idx, data.reshape(-1), top, 2.0, "none")
            if set_name == "dense16":
                info = hip_lib.lt_info(tid)
                assert info["baby"] == info["giant"] == 16
            for ge in hip_lib.GetLinearTransformRotationKeys(tid):
                hip_lib.GenerateLinearTransformRotationKey(ge)
            for level in order + order[:1]:
                print(f"[levels] {limbs} limbs, {special} special, {set_name}, order {order}: level {level}", flush=True)
                hip_lib.SetEncryptionCounter(levels.index(level))
                ct = hip_lib.Encrypt(hip_lib.Encode(vals, level, 1 << logscale))
                out = hip_lib.EvaluateLinearTransform(tid, ct)
                assert_equal_u64(hip_lib.export_ciphertext(out), want[level], f"order {order} level {level}")
            hip_lib.DeleteLinearTransform(tid)
    finally:
        orc.lt_free(t)
        orc.close()
        hip_lib.DeleteScheme()
