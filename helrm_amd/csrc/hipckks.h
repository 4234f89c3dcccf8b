// hipckks.h -- internal declarations shared by the HIP kernels and the host
// runtime of the MI355X CKKS backend (not part of the C ABI; see
// include/helrm_hip.h for that).
//
// Data layout in HBM
//   * a polynomial is limb-major u64[rows][N]; every value is canonical in
//     [0, q) of its row's modulus;
//   * ciphertexts and plaintexts are in the NTT domain (bit-reversed
//     evaluation order, psi = g^((q-1)/2N) with g the smallest generator);
//   * a QP polynomial at level l has rows q_0..q_l then p_0..p_{K-1};
//   * linear-transform diagonals and Galois keys are stored pre-multiplied
//     by R = 2^64 mod q ("Montgomery form") so that a lazily accumulated
//     128-bit sum of products needs a single REDC per output word.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint64_t u64;
typedef int64_t i64;
typedef unsigned __int128 u128;

#define HCK_MAXMOD 96
#define HCK_MAXSRC 32

// Per-modulus constants (device table indexed by modulus index:
// 0..L-1 the Q chain, L..L+K-1 the P chain).
struct ModC {
  u64 q;
  u64 qinv;  // -q^-1 mod 2^64
  u64 r2;    // 2^128 mod q
  u64 rmod;  // 2^64 mod q
};

// Row -> modulus mapping for a batch of polynomials:
// rows [0, split) use moduli m0.., rows [split, n) use m1..;
// rows in [skip0, skip1) are left untouched.
struct RowMap {
  int n, split, m0, m1, skip0, skip1;
  __host__ __device__ int nact() const { return n - (skip1 - skip0); }
  __host__ __device__ int row(int r) const { return r < skip0 ? r : r + (skip1 - skip0); }
  __host__ __device__ int mod(int row) const { return row < split ? m0 + row : m1 + (row - split); }
};


#if defined(__HIP_DEVICE_COMPILE__) || defined(__HIPCC__)
// Words of a table that no kernel writes, at a wave-uniform index: read
// through the constant address space they are scalar loads also in a kernel
// that has stored before (where the compiler falls back to vector loads).
typedef const u64 __attribute__((address_space(4)))* cwords;
__device__ __forceinline__ cwords const_words(const void* p) { return (cwords)(uintptr_t)p; }
__device__ __forceinline__ u64 add_mod(u64 a, u64 b, u64 q) { u64 r = a + b; return r >= q ? r - q : r; }
__device__ __forceinline__ u64 sub_mod(u64 a, u64 b, u64 q) { return a >= b ? a - b : a + q - b; }
__device__ __forceinline__ u64 shoup_mul(u64 x, u64 w, u64 wp, u64 q) {
  u64 qh = __umul64hi(x, wp);
  u64 r = x * w - qh * q;
  return r >= q ? r - q : r;
}
// x >= m ? x - m : x, selecting on the borrow of the 64-bit subtraction
// (four VALU instructions; the compiler's own form adds a 64-bit compare).
__device__ __forceinline__ u64 csub_b(u64 x, u64 m) {
  uint32_t dl, dh;
  u64 b;
  asm("v_sub_co_u32_e64 %[dl], %[b], %[xl], %[ml]\n\t"
      "v_subb_co_u32_e64 %[dh], %[b], %[xh], %[mh], %[b]\n\t"
      "v_cndmask_b32_e64 %[dl], %[dl], %[xl], %[b]\n\t"
      "v_cndmask_b32_e64 %[dh], %[dh], %[xh], %[b]"
      : [dl] "=&v"(dl), [dh] "=&v"(dh), [b] "=&s"(b)
      : [xl] "v"((uint32_t)x), [xh] "v"((uint32_t)(x >> 32)), [ml] "v"((uint32_t)m), [mh] "v"((uint32_t)(m >> 32)));
  return ((u64)dh << 32) | dl;
}
// High 64 bits of y*p in six VALU instructions: the middle column
// yl*ph + yh*pl + hi(yl*pl) is summed with the carry-out of v_mad_u64_u32
// instead of being split into zero-extended halves.
__device__ __forceinline__ u64 mulhi64(u64 y, u64 p) {
  const uint32_t yl = (uint32_t)y, yh = (uint32_t)(y >> 32), pl = (uint32_t)p, ph = (uint32_t)(p >> 32);
  const u64 m1 = (u64)yl * ph + __umulhi(yl, pl);  // < 2^64
  u64 m2, c;
  asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(m2), "=s"(c) : "v"(yh), "v"(pl), "v"(m1));
  const u64 r = (u64)yh * ph + (m2 >> 32);  // < 2^64
  uint32_t rh;
  u64 c2;
  asm("v_addc_co_u32_e64 %0, %1, 0, %2, %3" : "=v"(rh), "=s"(c2) : "v"((uint32_t)(r >> 32)), "s"(c));
  return ((u64)rh << 32) | (uint32_t)r;
}
// Shoup product in [0, 2q) for any y < 2^64: y*w + floor(y*wp / 2^64) * nq
// mod 2^64 with nq = 2^64 - q, the low product added through the addend of
// v_mad_u64_u32 (no separate 64-bit subtraction).
__device__ __forceinline__ u64 shoup_lazy(u64 y, u64 w, u64 wp, u64 nq) {
  const u64 Q = mulhi64(y, wp);
  const u64 yw = y * w;
  u64 t, c;
  asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(t), "=s"(c) : "v"((uint32_t)Q), "s"((uint32_t)nq), "v"(yw));
  const uint32_t th = (uint32_t)(t >> 32) + (uint32_t)Q * (uint32_t)(nq >> 32) + (uint32_t)(Q >> 32) * (uint32_t)nq;
  return ((u64)th << 32) | (uint32_t)t;
}
// 128-bit lazy accumulator: (hi, lo) += a*b, keeping hi < q (needs q < 2^62).
__device__ __forceinline__ void mac_lazy(u64& lo, u64& hi, u64 a, u64 b, u64 q) {
  u64 plo = a * b, phi = __umul64hi(a, b);
  u64 nlo = lo + plo;
  hi = hi + phi + (nlo < lo ? 1 : 0);
  lo = nlo;
  hi = hi >= q ? hi - q : hi;
}
// Exact sum of up to 16 products of words below 2^62, in column form:
//   sum = s0 + s1*2^32 + (s2 + c0)*2^64 + c1*2^96
// s0 collects a0*b0, s1 collects a0*b1 + a1*b0, s2 collects a1*b1 (32-bit
// halves); c0 and c1 count the carries out of s0 and s1, taken from the
// carry-out of v_mad_u64_u32.  Seven VALU instructions per product (the
// carry reads sit three or more instructions after their writes).  s2 cannot
// overflow: a1, b1 < 2^30, so 16 products stay below 2^64.
struct Acc128 { u64 s0, s1, s2; uint32_t c0, c1; };
__device__ __forceinline__ void acc_zero(Acc128& A) { A.s0 = A.s1 = A.s2 = 0; A.c0 = A.c1 = 0; }
__device__ __forceinline__ void acc_mac(Acc128& A, u64 a, u64 b) {
  const uint32_t a0 = (uint32_t)a, a1 = (uint32_t)(a >> 32), b0 = (uint32_t)b, b1 = (uint32_t)(b >> 32);
  u64 ca, cb, cc, cd;
  // not volatile: a pure function of its operands, free to be scheduled
  asm(
      "v_mad_u64_u32 %[s0], %[ca], %[a0], %[b0], %[s0]\n\t"
      "v_mad_u64_u32 %[s1], %[cb], %[a0], %[b1], %[s1]\n\t"
      "v_mad_u64_u32 %[s1], %[cc], %[a1], %[b0], %[s1]\n\t"
      "v_mad_u64_u32 %[s2], %[cd], %[a1], %[b1], %[s2]\n\t"
      "v_addc_co_u32_e64 %[c0], %[cd], 0, %[c0], %[ca]\n\t"
      "v_addc_co_u32_e64 %[c1], %[cd], 0, %[c1], %[cb]\n\t"
      "v_addc_co_u32_e64 %[c1], %[cd], 0, %[c1], %[cc]"
      : [s0] "+v"(A.s0), [s1] "+v"(A.s1), [s2] "+v"(A.s2), [c0] "+v"(A.c0), [c1] "+v"(A.c1),
        [ca] "=&s"(ca), [cb] "=&s"(cb), [cc] "=&s"(cc), [cd] "=&s"(cd)
      : [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1));
}
// The same with b uniform across the wave (held in SGPRs: the constant of a
// basis conversion); each v_mad_u64_u32 reads one SGPR.
__device__ __forceinline__ void acc_mac_s(Acc128& A, u64 a, u64 b) {
  const uint32_t a0 = (uint32_t)a, a1 = (uint32_t)(a >> 32), b0 = (uint32_t)b, b1 = (uint32_t)(b >> 32);
  u64 ca, cb, cc, cd;
  asm("v_mad_u64_u32 %[s0], %[ca], %[b0], %[a0], %[s0]\n\t"
      "v_mad_u64_u32 %[s1], %[cb], %[b1], %[a0], %[s1]\n\t"
      "v_mad_u64_u32 %[s1], %[cc], %[b0], %[a1], %[s1]\n\t"
      "v_mad_u64_u32 %[s2], %[cd], %[b1], %[a1], %[s2]\n\t"
      "v_addc_co_u32_e64 %[c0], %[cd], 0, %[c0], %[ca]\n\t"
      "v_addc_co_u32_e64 %[c1], %[cd], 0, %[c1], %[cb]\n\t"
      "v_addc_co_u32_e64 %[c1], %[cd], 0, %[c1], %[cc]"
      : [s0] "+v"(A.s0), [s1] "+v"(A.s1), [s2] "+v"(A.s2), [c0] "+v"(A.c0), [c1] "+v"(A.c1),
        [ca] "=&s"(ca), [cb] "=&s"(cb), [cc] "=&s"(cc), [cd] "=&s"(cd)
      : [a0] "v"(a0), [a1] "v"(a1), [b0] "s"(b0), [b1] "s"(b1));
}
// Exact sum of at most 8 products of words below 2^61 (every modulus here is
// below 2^61).  Split at 32 bits the high halves are below 2^29, so a middle
// column of 4 products (8 terms below 2^61) and the top column of 8 products
// (below 2^58 each) cannot overflow: only the low column counts carries, and
// the middle column is kept in two halves (products 0-3 and 4-7).  5 VALU
// instructions per product instead of 7.
struct Acc61 { u64 s0, s1a, s1b, s2; uint32_t c0; };
__device__ __forceinline__ void acc61_zero(Acc61& A) { A.s0 = A.s1a = A.s1b = A.s2 = 0; A.c0 = 0; }
// the first product of an accumulator (and of its second middle half) sets
// the columns instead of adding to zeros; the accumulator starts from v * n,
// v at most 8 and n < 2^61 (below 2^32 in the middle column, which four
// products leave free)
__device__ __forceinline__ void acc61_first_s(Acc61& A, uint32_t v, u64 n, u64 a, u64 b) {
  const uint32_t a0 = (uint32_t)a, a1 = (uint32_t)(a >> 32), b0 = (uint32_t)b, b1 = (uint32_t)(b >> 32);
  u64 junk, ca;
  asm("v_mad_u64_u32 %[s0], %[j], %[n0], %[v], 0\n\t"
      "v_mad_u64_u32 %[s1], %[j], %[n1], %[v], 0\n\t"
      "v_mad_u64_u32 %[s0], %[ca], %[b0], %[a0], %[s0]\n\t"
      "v_mad_u64_u32 %[s1], %[j], %[b1], %[a0], %[s1]\n\t"
      "v_mad_u64_u32 %[s1], %[j], %[b0], %[a1], %[s1]\n\t"
      "v_mad_u64_u32 %[s2], %[j], %[b1], %[a1], 0\n\t"
      "v_cndmask_b32_e64 %[c0], 0, 1, %[ca]"
      : [s0] "=&v"(A.s0), [s1] "=&v"(A.s1a), [s2] "=&v"(A.s2), [c0] "=&v"(A.c0), [ca] "=&s"(ca), [j] "=&s"(junk)
      : [a0] "v"(a0), [a1] "v"(a1), [b0] "s"(b0), [b1] "s"(b1), [v] "v"(v), [n0] "s"((uint32_t)n), [n1] "s"((uint32_t)(n >> 32)));
}
__device__ __forceinline__ void acc61_first_half_s(Acc61& A, u64 a, u64 b) {
  const uint32_t a0 = (uint32_t)a, a1 = (uint32_t)(a >> 32), b0 = (uint32_t)b, b1 = (uint32_t)(b >> 32);
  u64 ca, junk;
  asm("v_mad_u64_u32 %[s0], %[ca], %[b0], %[a0], %[s0]\n\t"
      "v_mad_u64_u32 %[s1], %[j], %[b1], %[a0], 0\n\t"
      "v_mad_u64_u32 %[s1], %[j], %[b0], %[a1], %[s1]\n\t"
      "v_mad_u64_u32 %[s2], %[j], %[b1], %[a1], %[s2]\n\t"
      "v_addc_co_u32_e64 %[c0], %[j], 0, %[c0], %[ca]"
      : [s0] "+v"(A.s0), [s1] "=&v"(A.s1b), [s2] "+v"(A.s2), [c0] "+v"(A.c0), [ca] "=&s"(ca), [j] "=&s"(junk)
      : [a0] "v"(a0), [a1] "v"(a1), [b0] "s"(b0), [b1] "s"(b1));
}
template <int HALF>
__device__ __forceinline__ void acc61_mac_s(Acc61& A, u64 a, u64 b) {
  const uint32_t a0 = (uint32_t)a, a1 = (uint32_t)(a >> 32), b0 = (uint32_t)b, b1 = (uint32_t)(b >> 32);
  u64& s1 = HALF ? A.s1b : A.s1a;
  u64 ca, junk;
  asm("v_mad_u64_u32 %[s0], %[ca], %[b0], %[a0], %[s0]\n\t"
      "v_mad_u64_u32 %[s1], %[j], %[b1], %[a0], %[s1]\n\t"
      "v_mad_u64_u32 %[s1], %[j], %[b0], %[a1], %[s1]\n\t"
      "v_mad_u64_u32 %[s2], %[j], %[b1], %[a1], %[s2]\n\t"
      "v_addc_co_u32_e64 %[c0], %[j], 0, %[c0], %[ca]"
      : [s0] "+v"(A.s0), [s1] "+v"(s1), [s2] "+v"(A.s2), [c0] "+v"(A.c0), [ca] "=&s"(ca), [j] "=&s"(junk)
      : [a0] "v"(a0), [a1] "v"(a1), [b0] "s"(b0), [b1] "s"(b1));
}
__device__ __forceinline__ void acc61_value(const Acc61& A, u64& lo, u64& hi) {
  const u64 s1 = A.s1a + A.s1b;
  const u64 s1c = s1 < A.s1a ? 1 : 0;
  const u64 t = s1 << 32;
  lo = A.s0 + t;
  hi = A.s2 + A.c0 + (s1 >> 32) + (s1c << 32) + (lo < t ? 1 : 0);
}
// REDC(value of A) for an Acc61 whose value is below q * 2^64, a 32-bit word
// at a time on the columns as they are (21 VALU instructions; recombining the
// 128-bit value first takes 33):
//   m0 = s0 * qinv mod 2^32;  s1 = s1a + s1b + m0 q1 + (s0 + m0 q0) / 2^32
//   m1 = s1 * qinv mod 2^32;  r  = s2 + m1 q1 + (s1 + m1 q0) / 2^32
// with the carries out of s0 counted into s1's high word and those out of s1
// (kb, k1, kd, k3) into r's; r < 2q, then r >= q ? r - q : r.
__device__ __forceinline__ u64 acc61_redc(const Acc61& A, u64 q, u64 qinv) {
  const uint32_t q0 = (uint32_t)q, q1 = (uint32_t)(q >> 32), qi = (uint32_t)qinv;
  uint32_t m0, s1l, s1h, c0;
  u64 t, k0, kb, kc;
  asm("v_mul_lo_u32 %[m0], %[s0l], %[qi]\n\t"
      "v_add_co_u32_e64 %[s1l], %[kc], %[al], %[bl]\n\t"
      "v_mad_u64_u32 %[t], %[k0], %[m0], %[q0], %[s0]\n\t"
      "v_addc_co_u32_e64 %[s1h], %[kb], %[ah], %[bh], %[kc]\n\t"
      "v_addc_co_u32_e64 %[c0], %[kc], 0, %[c0i], %[k0]"
      : [m0] "=&v"(m0), [t] "=&v"(t), [s1l] "=&v"(s1l), [s1h] "=&v"(s1h), [c0] "=&v"(c0), [k0] "=&s"(k0), [kb] "=&s"(kb),
        [kc] "=&s"(kc)
      : [s0l] "v"((uint32_t)A.s0), [s0] "v"(A.s0), [c0i] "v"(A.c0), [al] "v"((uint32_t)A.s1a), [ah] "v"((uint32_t)(A.s1a >> 32)),
        [bl] "v"((uint32_t)A.s1b), [bh] "v"((uint32_t)(A.s1b >> 32)), [qi] "s"(qi), [q0] "s"(q0));
  u64 s1 = ((u64)s1h << 32) | s1l, k1, kd;
  asm("v_mad_u64_u32 %[s1], %[k1], %[m0], %[q1], %[s1]" : [s1] "+v"(s1), [k1] "=&s"(k1) : [m0] "v"(m0), [q1] "s"(q1));
  asm("v_add_co_u32_e64 %[s1l], %[kc], %[il], %[th]\n\t"
      "v_addc_co_u32_e64 %[s1h], %[kd], %[ih], %[c0], %[kc]"
      : [s1l] "=&v"(s1l), [s1h] "=&v"(s1h), [kc] "=&s"(kc), [kd] "=&s"(kd)
      : [il] "v"((uint32_t)s1), [ih] "v"((uint32_t)(s1 >> 32)), [th] "v"((uint32_t)(t >> 32)), [c0] "v"(c0));
  s1 = ((u64)s1h << 32) | s1l;
  uint32_t m1;
  u64 r = A.s2, k3, junk;
  asm("v_mul_lo_u32 %[m1], %[s1l], %[qi]\n\t"
      "v_mad_u64_u32 %[t], %[k3], %[m1], %[q0], %[s1]\n\t"
      "v_mad_u64_u32 %[r], %[j], %[m1], %[q1], %[r]"
      : [m1] "=&v"(m1), [t] "=&v"(t), [r] "+v"(r), [k3] "=&s"(k3), [j] "=&s"(junk)
      : [s1l] "v"(s1l), [s1] "v"(s1), [qi] "s"(qi), [q0] "s"(q0), [q1] "s"(q1));
  uint32_t rl, rh;
  asm("v_add_co_u32_e64 %[rl], %[j], %[il], %[th]\n\t"
      "v_addc_co_u32_e64 %[rh], %[j], %[ih], 0, %[j]\n\t"
      "v_addc_co_u32_e64 %[rh], %[j], %[rh], 0, %[kb]\n\t"
      "v_addc_co_u32_e64 %[rh], %[j], %[rh], 0, %[k1]\n\t"
      "v_addc_co_u32_e64 %[rh], %[j], %[rh], 0, %[kd]\n\t"
      "v_addc_co_u32_e64 %[rh], %[j], %[rh], 0, %[k3]"
      : [rl] "=&v"(rl), [rh] "=&v"(rh), [j] "=&s"(junk)
      : [il] "v"((uint32_t)r), [ih] "v"((uint32_t)(r >> 32)), [th] "v"((uint32_t)(t >> 32)), [kb] "s"(kb), [k1] "s"(k1),
        [kd] "s"(kd), [k3] "s"(k3));
  return csub_b(((u64)rh << 32) | rl, q);
}
// One destination word of a basis extension from at most 8 sources:
// REDC(sum_i y(i) * h[i] + v * n), y(i) < 2^61 (zero past the job's sources),
// h[i] < q the row's table words and n < q that of -S (Montgomery form, h
// read for all 8 i: the table holds spare words past its last row), v <= 8
// the overflow count: the sum is at most (2^64 - 8)(q - 1) + 8 (q - 1), so
// below q * 2^64 as the REDC needs.
template <class Y, class H>
__device__ __forceinline__ u64 bconv_word8(Y y, H h, uint32_t v, u64 n, u64 q, u64 qinv) {
  Acc61 A;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    if (i == 0) acc61_first_s(A, v, n, y(i), h[i]);
    else if (i < 4) acc61_mac_s<0>(A, y(i), h[i]);
    else if (i == 4) acc61_first_half_s(A, y(i), h[i]);
    else acc61_mac_s<1>(A, y(i), h[i]);
  }
  return acc61_redc(A, q, qinv);
}
// the 128-bit value (lo, hi) of an accumulator
__device__ __forceinline__ void acc_value(const Acc128& A, u64& lo, u64& hi) {
  const u64 t = A.s1 << 32;
  lo = A.s0 + t;
  hi = A.s2 + A.c0 + (A.s1 >> 32) + ((u64)A.c1 << 32) + (lo < t ? 1 : 0);
}
// Montgomery reduction of T = hi*2^64 + lo < q*2^64: returns T * 2^-64 mod q.
__device__ __forceinline__ u64 redc(u64 lo, u64 hi, u64 q, u64 qinv) {
  u64 m = lo * qinv;
  u64 t = hi + mulhi64(m, q) + (lo != 0 ? 1 : 0);
  return csub_b(t, q);
}
__device__ __forceinline__ u64 mont_mul(u64 a, u64 bR, u64 q, u64 qinv) {
  return redc(a * bR, __umul64hi(a, bR), q, qinv);
}
#endif
