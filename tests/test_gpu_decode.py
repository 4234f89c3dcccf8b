"""The device decoder (multiword centred CRT, nearest double, special FFT in
two launches) against the oracle's float64 decoding, bit for bit, over every
table width of the CRT kernel, and the encoder's FFT at the smallest and
largest number of slots."""
import numpy as np
import pytest

from helpers import assert_equal_u64, make_params, new_hip_scheme
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# name: (logN, logq, levels); the levels reach 4, 8, 16, 24, 32 and more words
CHAINS = {
    "n10": (10, [60] + [50] * 44, (0, 1, 3, 4, 8, 9, 18, 19, 28, 29, 38, 39, 44)),
    "n11": (11, [55] + [45] * 6, (0, 3, 6)),
    "n13": (13, [60] + [40] * 4, (4,)),
    "n16": (16, [60] + [50] * 23, (22,)),
}


def coefficients(rng, n, Q):
    """Integers of every size a double can hold (few of them larger than the
    53 bits a double keeps end in zeros or ties), with the CRT's edges in front."""
    top = min(Q.bit_length() - 2, 900)
    out = []
    for i in range(n):
        bits = int(rng.integers(1, top + 1))
        v = int.from_bytes(rng.bytes((bits + 7) // 8), "little") >> (-bits % 8)
        if i % 5 == 0 and bits > 60:
            v = (v >> (bits - 55)) << (bits - 55)  # a tie at the rounding bit, or exact
            v += int(i % 3 == 0)                   # ... decided by the lowest bit
        out.append(v if i % 2 else -v)
    edges = [0, 1, -1, (1 << 53) + 1, -(1 << 53) - 1, (1 << 54) + 2, (1 << 54) + 6]
    if Q.bit_length() < 1000:
        edges += [Q // 2, Q // 2 - 1, Q // 2 + 1, -(Q // 2) + 1]
    else:
        edges += [1 << 899, -(1 << 899)]
    edges = [e for e in edges if abs(e) <= Q // 2 + 1]
    out[:len(edges)] = edges
    return out


@pytest.mark.parametrize("name", list(CHAINS))
def test_decode_bitexact(hip_lib, name):
    logn, logq, levels = CHAINS[name]
    q, p = make_params(logn, logq, [61])
    N = 1 << logn
    scale = float(1 << 40)
    new_hip_scheme(hip_lib, logn, q, p, 40, 64, 5, evaluator=False)
    orc = O.Oracle(logn, q, p, h=64, seed=5)
    rng = np.random.default_rng(8)
    try:
        for level in levels:
            print(f"[decode] {name} level {level}", flush=True)
            Q = 1
            for m in q[: level + 1]:
                Q *= int(m)
            coef = coefficients(rng, N, Q)
            rows = np.stack([orc.ntt(np.array([c % int(m) for c in coef], dtype=np.uint64), r)
                             for r, m in enumerate(q[: level + 1])])
            pt = hip_lib.import_plaintext(rows, level, scale)
            want = orc.decode_f64(rows, level, scale)
            got = hip_lib.decode_double(pt)
            np.testing.assert_array_equal(got.view(np.uint64), want.view(np.uint64))
            with np.errstate(over="ignore"):
                want32 = orc.decode(rows, level, scale)
            np.testing.assert_array_equal(np.asarray(hip_lib.Decode(pt), np.float32).view(np.uint32), want32.view(np.uint32))
            z = orc.decode_complex(rows, level, scale)
            dec = np.asarray(hip_lib.DecodeComplex(pt), np.float32)
            with np.errstate(over="ignore"):
                np.testing.assert_array_equal(dec[0::2], z.real.astype(np.float32))
                np.testing.assert_array_equal(dec[1::2], z.imag.astype(np.float32))
            hip_lib.DeletePlaintext(pt)
    finally:
        orc.close()
        hip_lib.DeleteScheme()


@pytest.mark.parametrize("logn", [10, 12, 16])
def test_encode_encrypt_sizes(hip_lib, logn):
    q, p = make_params(logn, [60, 50, 50], [61])
    slots = 1 << (logn - 1)
    new_hip_scheme(hip_lib, logn, q, p, 50, 192, 9, evaluator=False)
    orc = O.Oracle(logn, q, p, h=192, seed=9)
    rng = np.random.default_rng(2)
    try:
        for index, n in enumerate((1, 257, slots - 1, slots)):
            print(f"[encode] logn {logn} values {n}", flush=True)
            vals = rng.uniform(-4, 4, n).astype(np.float32)
            full = np.zeros(slots, np.float32)
            full[:n] = vals
            level = 2 - index % 3
            pt = hip_lib.Encode(vals, level, 1 << 50)
            want = orc.encode(full, level, float(1 << 50))
            assert_equal_u64(hip_lib.export_plaintext(pt), want, f"encode {n}")
            hip_lib.SetEncryptionCounter(index)
            ct = hip_lib.Encrypt(pt)
            assert_equal_u64(hip_lib.export_ciphertext(ct), orc.encrypt(want, level, index), f"encrypt {n}")
    finally:
        orc.close()
        hip_lib.DeleteScheme()


@pytest.mark.parametrize("h", [255, 256, 257, 700, 1024])
def test_encrypt_positions(hip_lib, h):
    """The ternary polynomial's positions travel with the launch up to 256 and
    through memory above, up to every place of the ring; one limb and several, a
    modulus of 61 bits in P."""
    q, p = make_params(10, [60, 50, 40, 55], [61, 61])
    new_hip_scheme(hip_lib, 10, q, p, 40, h, 4, evaluator=False)
    orc = O.Oracle(10, q, p, h=h, seed=4)
    rng = np.random.default_rng(h)
    try:
        for index, level in enumerate((3, 1, 0)):
            print(f"[encrypt] h {h} level {level}", flush=True)
            vals = rng.uniform(-1, 1, 512).astype(np.float32)
            hip_lib.SetEncryptionCounter(index)
            pt = hip_lib.Encode(vals, level, 1 << 40)
            ct = hip_lib.Encrypt(pt)
            want = orc.encode(vals, level, float(1 << 40))
            assert_equal_u64(hip_lib.export_ciphertext(ct), orc.encrypt(want, level, index), f"encrypt h {h} level {level}")
            dec = hip_lib.Decrypt(ct)
            got = hip_lib.decode_double(dec)
            ref = orc.decode_f64(hip_lib.export_plaintext(dec), level, float(1 << 40))
            np.testing.assert_array_equal(got.view(np.uint64), ref.view(np.uint64))
    finally:
        orc.close()
        hip_lib.DeleteScheme()
