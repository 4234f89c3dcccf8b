// kernels.hip -- gfx950 kernels of the CKKS backend.  Integer RNS arithmetic
// on the VALU (64-bit words, 128-bit lazy accumulation, one Montgomery REDC
// per output word); no MFMA: this is modular arithmetic, not a float
// contraction.  Every kernel is launched on the scheme's stream by the
// wrappers at the bottom of this file.
#include "hipckks.h"
#include "kernels.h"
#include <algorithm>
#include <cstddef>
#include <stdexcept>

// High word of a 128-bit sum of products of words < q < 2^62: after at most
// 16 products (plus one earlier fold) it is below 5q; bring it below q.
__device__ __forceinline__ u64 csub64(u64 x, u64 m) { return x >= m ? x - m : x; }
__device__ __forceinline__ u64 fold_hi4(u64 hi, u64 q) { return csub64(csub64(csub64(hi, q << 2), q << 1), q); }

// ---------------------------------------------------------------------------
// Element-wise kernels over (coefficient, row, batch)
// ---------------------------------------------------------------------------
__global__ void add_rows_kernel(u64* __restrict__ out, const u64* __restrict__ a, const u64* __restrict__ b,
                                size_t bstride, RowMap rm, const ModC* __restrict__ mods, int N, int sub) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int row = rm.row(blockIdx.y);
  u64 q = mods[rm.mod(row)].q;
  size_t o = (size_t)blockIdx.z * bstride + (size_t)row * N + x;
  out[o] = sub ? sub_mod(a[o], b[o], q) : add_mod(a[o], b[o], q);
}
void launch_add(u64* out, const u64* a, const u64* b, size_t bstride, int batch, RowMap rm, const ModC* mods, int N, bool sub, hipStream_t st) {
  if (rm.nact() <= 0 || batch <= 0) return;
  hipLaunchKernelGGL(add_rows_kernel, dim3(N / 256, rm.nact(), batch), dim3(256), 0, st, out, a, b, bstride, rm, mods, N, sub ? 1 : 0);
}

// out = in * c_row (per-row constant in Shoup form, indexed by modulus)
__global__ void mul_const_kernel(u64* __restrict__ out, size_t obstride, const u64* __restrict__ in, size_t bstride, RowMap rm,
                                 const u64* __restrict__ cw, const u64* __restrict__ cwp, const ModC* __restrict__ mods, int N) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int row = rm.row(blockIdx.y);
  int m = rm.mod(row);
  size_t o = (size_t)row * N + x;
  out[(size_t)blockIdx.z * obstride + o] = shoup_mul(in[(size_t)blockIdx.z * bstride + o], cw[m], cwp[m], mods[m].q);
}
void launch_mul_const(u64* out, size_t obstride, const u64* in, size_t bstride, int batch, RowMap rm, const u64* cw,
                      const u64* cwp, const ModC* mods, int N, hipStream_t st) {
  if (rm.nact() <= 0 || batch <= 0) return;
  hipLaunchKernelGGL(mul_const_kernel, dim3(N / 256, rm.nact(), batch), dim3(256), 0, st, out, obstride, in, bstride, rm, cw, cwp,
                     mods, N);
}

__global__ void mul_const_v_kernel(u64* __restrict__ out, const u64* __restrict__ in, size_t bstride, RowMap rm, RowConst c,
                                   const ModC* __restrict__ mods, int N) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int row = rm.row(blockIdx.y);
  const int m = rm.mod(row);
  const size_t o = (size_t)blockIdx.z * bstride + (size_t)row * N + x;
  out[o] = shoup_mul(in[o], c.w[m], c.wp[m], mods[m].q);
}
void launch_mul_const_v(u64* out, const u64* in, size_t bstride, int batch, RowMap rm, const RowConst& c, const ModC* mods,
                        int N, hipStream_t st) {
  if (rm.nact() <= 0 || batch <= 0) return;
  hipLaunchKernelGGL(mul_const_v_kernel, dim3(N / 256, rm.nact(), batch), dim3(256), 0, st, out, in, bstride, rm, c, mods, N);
}

// One thread per output dword of every (diagonal, row).  A packed row's
// dword d of chunk c holds bits [32 d, 32 d + 32) of the chunk's 64 fields:
// from field j = 32 d / 52 upward (and field j + 1 where field j ends inside
// the dword); a plain row's dwords are its words' halves.
__global__ __launch_bounds__(256) void pack_diags_kernel(uint32_t* __restrict__ dst, size_t dst_stride,
                                                        const u64* __restrict__ src, size_t src_stride,
                                                        const uint32_t* __restrict__ rowdesc, int N) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y, p = blockIdx.z;
  const uint32_t off = rowdesc[2 * k], bits = rowdesc[2 * k + 1];
  const u64* w = src + (size_t)p * src_stride + (size_t)k * N;
  uint32_t* o = dst + (size_t)p * dst_stride + off;
  if (bits == 0) {
    if (t < (size_t)2 * N) o[t] = (uint32_t)(w[t >> 1] >> (32 * (t & 1)));
    return;
  }
  if (t >= (size_t)(N / 64) * PK_CHUNK) return;
  const int c = (int)(t / PK_CHUNK), d = (int)(t % PK_CHUNK);
  const int bit0 = 32 * d, j = bit0 / PK_BITS, sh = bit0 - PK_BITS * j;
  const u64* wc = w + (size_t)c * 64;
  u64 v = wc[j] >> sh;
  if (sh + 32 > PK_BITS && j + 1 < 64) v |= wc[j + 1] << (PK_BITS - sh);
  o[t] = (uint32_t)v;
}
void launch_pack_diags(uint32_t* dst, size_t dst_stride, const u64* src, size_t src_stride, int np, const uint32_t* rowdesc,
                       int nrows, int N, hipStream_t st) {
  if (np <= 0 || nrows <= 0) return;
  hipLaunchKernelGGL(pack_diags_kernel, dim3((2 * N + 255) / 256, nrows, np), dim3(256), 0, st, dst, dst_stride, src, src_stride,
                     rowdesc, N);
}
// Word x of a packed row: chunk x / 64, field j = x % 64 at bit 52 j: its
// three dwords (the third only read when the field crosses two: shift > 12,
// never for the chunk's last field, whose index is clamped inside the chunk).
__device__ __forceinline__ u64 pk_field(const uint32_t* chunk, int j) {
  const int bit = PK_BITS * j, dw = bit >> 5, sh = bit & 31;
  const uint32_t d0 = chunk[dw], d1 = chunk[dw + 1], d2 = chunk[min(dw + 2, PK_CHUNK - 1)];
  return (u64)__builtin_amdgcn_alignbit(d1, d0, sh) |
         ((u64)(__builtin_amdgcn_alignbit(d2, d1, sh) & ((1u << (PK_BITS - 32)) - 1)) << 32);
}
__global__ __launch_bounds__(256) void unpack_diag_kernel(u64* __restrict__ dst, const uint32_t* __restrict__ src,
                                                         const uint32_t* __restrict__ rowdesc, int N) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
  const uint32_t off = rowdesc[2 * k], bits = rowdesc[2 * k + 1];
  const uint32_t* r = src + off;
  dst[(size_t)k * N + x] = bits ? pk_field(r + (size_t)(x >> 6) * PK_CHUNK, x & 63)
                                : ((u64)r[2 * (size_t)x + 1] << 32) | r[2 * (size_t)x];
}
void launch_unpack_diag(u64* dst, const uint32_t* src, const uint32_t* rowdesc, int nrows, int N, hipStream_t st) {
  hipLaunchKernelGGL(unpack_diag_kernel, dim3(N / 256, nrows, 1), dim3(256), 0, st, dst, src, rowdesc, N);
}

// One thread per word of the tensor product: both operands are read once,
// b is taken to Montgomery form in registers (b R = mont_mul(b, R^2)), and
// the three products are written together.
__global__ __launch_bounds__(256) void tensor_kernel(u64* __restrict__ d0, u64* __restrict__ d1, u64* __restrict__ d2,
                                                     const u64* __restrict__ a0, const u64* __restrict__ a1,
                                                     const u64* __restrict__ b0, const u64* __restrict__ b1,
                                                     const u64* __restrict__ pw, const u64* __restrict__ pwp,
                                                     const ModC* __restrict__ mods, int N) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  const ModC mc = mods[k];
  const size_t o = (size_t)k * N + x;
  const u64 b0R = mont_mul(b0[o], mc.r2, mc.q, mc.qinv), b1R = mont_mul(b1[o], mc.r2, mc.q, mc.qinv);
  const u64 va0 = a0[o], va1 = a1[o];
  u64 r0 = mont_mul(va0, b0R, mc.q, mc.qinv);
  u64 r1 = add_mod(mont_mul(va0, b1R, mc.q, mc.qinv), mont_mul(va1, b0R, mc.q, mc.qinv), mc.q);
  if (pw) {
    r0 = shoup_mul(r0, pw[k], pwp[k], mc.q);
    r1 = shoup_mul(r1, pw[k], pwp[k], mc.q);
  }
  d0[o] = r0;
  d1[o] = r1;
  d2[o] = mont_mul(va1, b1R, mc.q, mc.qinv);
}
void launch_tensor(u64* d0, u64* d1, u64* d2, const u64* a0, const u64* a1, const u64* b0, const u64* b1, int l,
                   const u64* pw, const u64* pwp, const ModC* mods, int N, hipStream_t st) {
  hipLaunchKernelGGL(tensor_kernel, dim3(N / 256, l + 1, 1), dim3(256), 0, st, d0, d1, d2, a0, a1, b0, b1, pw, pwp, mods, N);
}

// out = a * bR * R^-1 (b stored in Montgomery form), plus add (at out's stride)
// if given; with bmod, bR holds a row per modulus instead of one per row
__global__ void mont_mul_kernel(u64* out, const u64* __restrict__ a, size_t abstride,
                                const u64* __restrict__ bR, size_t bbstride, size_t obstride, RowMap rm,
                                const ModC* __restrict__ mods, int N, const u64* add, int bmod) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int row = rm.row(blockIdx.y), m = rm.mod(row);
  ModC mc = mods[m];
  u64 r = mont_mul(a[(size_t)blockIdx.z * abstride + (size_t)row * N + x],
                   bR[(size_t)blockIdx.z * bbstride + (size_t)(bmod ? m : row) * N + x], mc.q, mc.qinv);
  size_t o = (size_t)blockIdx.z * obstride + (size_t)row * N + x;
  out[o] = add ? add_mod(add[o], r, mc.q) : r;
}
void launch_mont_mul(u64* out, size_t obstride, const u64* a, size_t abstride, const u64* bR, size_t bbstride, int batch,
                     RowMap rm, const ModC* mods, int N, const u64* add, hipStream_t st, bool bmod) {
  if (rm.nact() <= 0 || batch <= 0) return;
  hipLaunchKernelGGL(mont_mul_kernel, dim3(N / 256, rm.nact(), batch), dim3(256), 0, st, out, a, abstride, bR, bbstride, obstride, rm, mods, N, add, bmod ? 1 : 0);
}

// out[row] = in[row] +- c.w[modulus of row] (a constant in every NTT slot)
__global__ void add_scalar_v_kernel(u64* __restrict__ out, const u64* __restrict__ in, RowMap rm, RowConst c,
                                    const ModC* __restrict__ mods, int N, int sub) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int row = rm.row(blockIdx.y);
  const int m = rm.mod(row);
  const u64 q = mods[m].q;
  const size_t o = (size_t)row * N + x;
  out[o] = sub ? sub_mod(in[o], c.w[m], q) : add_mod(in[o], c.w[m], q);
}
void launch_add_scalar_v(u64* out, const u64* in, RowMap rm, const RowConst& c, const ModC* mods, int N, bool sub,
                         hipStream_t st) {
  if (rm.nact() <= 0) return;
  hipLaunchKernelGGL(add_scalar_v_kernel, dim3(N / 256, rm.nact(), 1), dim3(256), 0, st, out, in, rm, c, mods, N, sub ? 1 : 0);
}

// v -> v*R mod q (to Montgomery form) or v*R^-1 (from), in place
__global__ void mont_convert_kernel(u64* __restrict__ data, size_t bstride, RowMap rm, const ModC* __restrict__ mods, int N, int to) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int row = rm.row(blockIdx.y);
  ModC mc = mods[rm.mod(row)];
  size_t o = (size_t)blockIdx.z * bstride + (size_t)row * N + x;
  u64 v = data[o];
  data[o] = to ? mont_mul(v, mc.r2, mc.q, mc.qinv) : redc(v, 0, mc.q, mc.qinv);
}
void launch_mont_convert(u64* data, size_t bstride, int batch, RowMap rm, const ModC* mods, int N, bool to, hipStream_t st) {
  if (rm.nact() <= 0 || batch <= 0) return;
  hipLaunchKernelGGL(mont_convert_kernel, dim3(N / 256, rm.nact(), batch), dim3(256), 0, st, data, bstride, rm, mods, N, to ? 1 : 0);
}


// Strided batched copy: dst[b][0..words) = src[b][0..words), 16 bytes per lane.
template <bool VEC>
__global__ __launch_bounds__(256) void copy_kernel(u64* __restrict__ dst, size_t dstride, const u64* __restrict__ src,
                                                   size_t sstride, size_t words) {
  const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 2;
  const u64* s = src + (size_t)blockIdx.y * sstride;
  u64* d = dst + (size_t)blockIdx.y * dstride;
  if (!VEC) {
    if (i < words) d[i] = s[i];
    if (i + 1 < words) d[i + 1] = s[i + 1];
  } else if (i + 1 < words) {
    const ulong2 v = *reinterpret_cast<const ulong2*>(s + i);
    *reinterpret_cast<ulong2*>(d + i) = v;
  } else if (i < words) {
    d[i] = s[i];
  }
}
void launch_copy(u64* dst, size_t dstride, const u64* src, size_t sstride, size_t words, int batch, hipStream_t st) {
  if (words == 0 || batch <= 0) return;
  const size_t blocks = (words + 511) / 512;
  const bool vec = (((uintptr_t)dst | (uintptr_t)src | (dstride * 8) | (sstride * 8)) & 15) == 0;
  if (vec) hipLaunchKernelGGL(copy_kernel<true>, dim3((unsigned)blocks, batch), dim3(256), 0, st, dst, dstride, src, sstride, words);
  else hipLaunchKernelGGL(copy_kernel<false>, dim3((unsigned)blocks, batch), dim3(256), 0, st, dst, dstride, src, sstride, words);
}

// ---------------------------------------------------------------------------
// RNS basis extension (exact, float64 overflow count as Lattigo ModUpExact):
//   y_i = x_i * (S/s_i)^-1 mod s_i;  v = (u64) sum_i (double)y_i/(double)s_i
//   out_t = sum_i y_i * (S/s_i mod t) - v*S mod t
// One thread per coefficient computes y and v once and produces a block of
// destination rows from them (read ns, write nd words); the row sum is
// exact in 128 bits (folded below 4t after every 16 products), then one
// Montgomery REDC removes the 2^64 the (S/s_i mod t) table carries.
// ---------------------------------------------------------------------------
// At most MAXS sources.  With MAXS == 8 every row takes 8 products: the
// sources past ns are zero and the table holds 8 spare words at its end, so
// a job of 7 sources runs the same straight-line code as one of 8.
// blockIdx.z selects (batch entry, job): all digits of a decomposition go
// in one launch.
template <int MAXS>
__global__ __launch_bounds__(256) void bconv_kernel(const u64* __restrict__ in, size_t in_bstride, BConvJobs jobs,
                                                    u64* __restrict__ out, size_t out_bstride,
                                                    const ModC* __restrict__ mods, int N) {
  const int b = blockIdx.z / jobs.n, d = blockIdx.z - b * jobs.n;
  const BConvJob& J = jobs.j[d];
  const BConvTable* __restrict__ tab = J.tab;
  const int ns = J.ns;
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const u64* inb = in + (size_t)b * in_bstride + (size_t)J.src_row * N;
  u64* outb = out + (size_t)b * out_bstride + J.out_off;
  const RowMap rm = J.rm;
  const int r0 = blockIdx.y * jobs.rows_per_block;
  const int r1 = min(r0 + jobs.rows_per_block, rm.nact());
  u64 y[MAXS];
  double vf = 0.0;
  // every source word in flight at once (rows past ns re-read row 0, unused)
#pragma unroll
  for (int i = 0; i < MAXS; i++) y[i] = inb[(size_t)(i < ns ? i : 0) * N + x];
  // the source constants are read without a branch per source (entries past
  // ns are zero and their terms are selected away), so that their scalar
  // loads are issued together instead of one round trip per source
#pragma unroll
  for (int i = 0; i < MAXS; i++) {
    const BConvSrc s = tab->src[i];
    const bool act = i < ns;
    const u64 yi = shoup_mul(y[i], s.hinv, s.hinvp, s.q);
    const double t = (double)yi / s.qd;
    y[i] = act ? yi : 0;
    vf += act ? t : 0.0;
  }
  const uint32_t v = J.force_v0 ? 0 : (uint32_t)(u64)vf;
  const u64* __restrict__ hat = tab->hat;
  const u64* __restrict__ nS = tab->nS;
  for (int r = r0; r < r1; r++) {
    const int row = rm.row(r);
    const int m = rm.mod(row);
    const ModC mc = mods[m];
    const u64* __restrict__ h = hat + (size_t)m * ns;
    // exact column sums of 16 products (words < 2^62), folded below q
    u64 res;
    if (MAXS <= 8) {
      res = bconv_word8([&](int i) { return y[i]; }, h, v, nS[m], mc.q, mc.qinv);
    } else {
      u128 acc = 0;
#pragma unroll
      for (int i0 = 0; i0 < MAXS; i0 += 16) {
        Acc128 A;
        acc_zero(A);
#pragma unroll
        for (int i = i0; i < i0 + 16 && i < MAXS; i++)
          if (i < ns) acc_mac_s(A, y[i], h[i]);
        if (i0 == 0) acc_mac_s(A, v, nS[m]);  // v < 2^6: nothing in the top column
        u64 lo, hi;
        acc_value(A, lo, hi);
        acc += ((u128)fold_hi4(hi, mc.q) << 64) | lo;
      }
      res = redc((u64)acc, fold_hi4((u64)(acc >> 64), mc.q), mc.q, mc.qinv);
    }
    outb[(size_t)row * N + x] = res;
  }
}
// The same extension for launches too small to fill the GPU one coefficient
// per thread (a single key switch: a few thousand waves, each running every
// destination row).  A workgroup takes 64 coefficients of one (batch entry,
// job): its four waves load the sources and compute y_i and y_i / s_i once
// (two sources each), share them through LDS, and each wave then produces
// every fourth destination row -- four times the waves for the same work.
// The overflow count sums y_i / s_i in source order, as the one-thread form.
constexpr int BCL_X = 64;
// launches of fewer one-coefficient-per-thread workgroups than this take the shared-source form
#ifndef BCL_MAX_BLOCKS
#define BCL_MAX_BLOCKS 2048
#endif
__global__ __launch_bounds__(256) void bconv_lds_kernel(const u64* __restrict__ in, size_t in_bstride, BConvJobs jobs,
                                                       u64* __restrict__ out, size_t out_bstride,
                                                       const ModC* __restrict__ mods, int N) {
  constexpr int MAXS = 8;
  const int b = blockIdx.z / jobs.n, d = blockIdx.z - b * jobs.n;
  const BConvJob& J = jobs.j[d];
  const BConvTable* __restrict__ tab = J.tab;
  const int ns = J.ns;
  // w is the wave's index: made wave-uniform for the compiler, so that the
  // row loop's table words and modulus constants are scalar loads (as
  // per-lane loads every row would wait on a memory round trip)
  const int lane = threadIdx.x & (BCL_X - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x / BCL_X);
  const int x = blockIdx.x * BCL_X + lane;
  const u64* inb = in + (size_t)b * in_bstride + (size_t)J.src_row * N;
  u64* outb = out + (size_t)b * out_bstride + J.out_off;
  const RowMap rm = J.rm;
  const int nrows = rm.nact();
  const bool flip = ((uint32_t)x * jobs.ginv & (uint32_t)(2 * N - 1)) >= (uint32_t)N;  // never with ginv = 0
  __shared__ u64 sy[MAXS][BCL_X];
  __shared__ double st[MAXS][BCL_X];
  // sources w and w + 4 of this coefficient
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int i = w + 4 * k;
    const BConvSrc s = tab->src[i];
    const bool act = i < ns;
    const u64 xi = inb[(size_t)(act ? i : 0) * N + x];
    u64 yi = shoup_mul(xi, s.hinv, s.hinvp, s.q);
    if (flip && yi) yi = s.q - yi;
    const double t = (double)yi / s.qd;
    sy[i][lane] = act ? yi : 0;
    st[i][lane] = act ? t : 0.0;
  }
  __syncthreads();
  u64 y[MAXS];
  double vf = 0.0;
#pragma unroll
  for (int i = 0; i < MAXS; i++) {
    y[i] = sy[i][lane];
    vf += st[i][lane];
  }
  const uint32_t v = J.force_v0 ? 0 : (uint32_t)(u64)vf;
  const u64* __restrict__ hat = tab->hat;
  const u64* __restrict__ nS = tab->nS;
  for (int r = w; r < nrows; r += 4) {
    const int row = rm.row(r);
    const int m = rm.mod(row);
    const ModC mc = mods[m];
    const u64* __restrict__ h = hat + (size_t)m * ns;
    const u64 e = bconv_word8([&](int i) { return y[i]; }, h, v, nS[m], mc.q, mc.qinv);
    outb[(size_t)row * N + x] = flip && e ? mc.q - e : e;
  }
}

static_assert(sizeof(BConvSrc) == 32 && offsetof(BConvTable, hat) == 32 * HCK_MAXSRC && offsetof(BConvTable, nS) == 32 * HCK_MAXSRC + 8 &&
                  sizeof(ModC) == 32 && offsetof(ModC, qinv) == 8, "tables read by word");
__device__ __forceinline__ BConvSrc bconv_src(cwords tab, int i) {
  return BConvSrc{tab[4 * i], tab[4 * i + 1], tab[4 * i + 2], __longlong_as_double((long long)tab[4 * i + 3])};
}
// From one key switch's product to the next one's digits (LinkArgs).  The
// ModDown of the first, the automorphism's sum and the ModUp of the second
// are all coefficient-wise, so one launch does them without a transform in
// between: a rotation chain then runs the inverse transform of the product's
// Q rows where it ran the forward transform of the ModDown's extension and
// the inverse transform of the sum, and six launches a step instead of
// eleven.  VALU-bound as the basis extensions it is made of (2 (l+1) + dn nqp
// rows of 8 products a coefficient).  Shape as bconv_lds_kernel: 64
// coefficients a workgroup, four waves; a wave computes every fourth row and
// the rows' source terms meet in LDS.  Its tables are read as constant words:
// behind its own stores the compiler read them as 90 vector loads a wave, a
// memory round trip a row (22.7 -> 20.4 us at 11 Q rows).  A fold step of 23 Q
// and 8 P rows at N = 2^16 takes 163 us with it against 181 by RotateAdd, with
// the two extensions and the transforms between them.
__global__ __launch_bounds__(256) void link_kernel(LinkArgs a) {
  extern __shared__ u64 sm[];
  const int lane = threadIdx.x & (BCL_X - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x / BCL_X);
  const int N = a.N, K = a.K, nq = a.l + 1, nqp = a.nqp;
  const int x = blockIdx.x * BCL_X + lane;
  const u64* x1 = a.x1 + x;
  u64* c1 = a.c1 + x;
  u64* digits = a.digits + x;
  const bool flip = ((uint32_t)x * a.ginv & (uint32_t)(2 * N - 1)) >= (uint32_t)N;
  // LDS: source terms (P rows: y and y / p of both polynomials, 8 slots each;
  // then the Q rows' y and y / q)
  const cwords pt = const_words(a.ptab);  // BConvTable: 4 words a source, then the pointers hat and nS
  const cwords phat = const_words((const void*)pt[4 * HCK_MAXSRC]), pnS = const_words((const void*)pt[4 * HCK_MAXSRC + 1]);
  const cwords mods = const_words(a.mods), pinv = const_words(a.pinv), pinvp = const_words(a.pinvp);
  for (int part = 0; part < 2; part++) {
    const u64* src = part ? x1 + (size_t)nq * N : a.x0p + x;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int i = w + 4 * k;
      const BConvSrc s = bconv_src(pt, i);
      const bool act = i < K;
      u64 yi = shoup_mul(src[(size_t)(act ? i : 0) * N], s.hinv, s.hinvp, s.q);
      if (flip && yi) yi = s.q - yi;
      const double t = (double)yi / s.qd;
      sm[(part * 16 + i) * BCL_X + lane] = act ? yi : 0;
      sm[(part * 16 + 8 + i) * BCL_X + lane] = act ? (u64)__double_as_longlong(t) : 0;
    }
  }
  __syncthreads();
  u64 y0[8], y1[8];
  double v0f = 0.0, v1f = 0.0;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    y1[i] = sm[(16 + i) * BCL_X + lane];
    v1f += __longlong_as_double((long long)sm[(24 + i) * BCL_X + lane]);
    y0[i] = sm[i * BCL_X + lane];
    v0f += __longlong_as_double((long long)sm[(8 + i) * BCL_X + lane]);
  }
  const uint32_t v1 = (uint32_t)(u64)v1f, v0 = (uint32_t)(u64)v0f;
  __syncthreads();
  // a row's words are loaded while the row before it is computed
  u64 zn = w < nq ? x1[(size_t)w * N] : 0, cn = w < nq ? c1[(size_t)w * N] : 0;
  for (int r = w; r < nq; r += 4) {
    const u64 q = mods[4 * r], qinv = mods[4 * r + 1];
    const cwords h = phat + (size_t)r * K;
    const u64 pi = pinv[r], pip = pinvp[r], n = pnS[r];
    const u64 z = zn, c = cn;
    const int rn = min(r + 4, nq - 1);
    zn = x1[(size_t)rn * N];
    cn = c1[(size_t)rn * N];
    const u64 e1 = bconv_word8([&](int i) { return y1[i]; }, h, v1, n, q, qinv);
    const u64 m = shoup_mul(flip ? add_mod(z, e1, q) : sub_mod(z, e1, q), pi, pip, q);
    const u64 s = add_mod(c, m, q);
    c1[(size_t)r * N] = s;
    const BConvSrc sd = bconv_src(const_words(a.dtab[r / K]), r % K);
    const u64 yi = shoup_mul(s, sd.hinv, sd.hinvp, sd.q);
    sm[r * BCL_X + lane] = yi;
    sm[(nq + r) * BCL_X + lane] = (u64)__double_as_longlong((double)yi / sd.qd);
    u64 e0 = bconv_word8([&](int i) { return y0[i]; }, h, v0, n, q, qinv);
    e0 = shoup_mul(e0, pi, pip, q);
    a.e0[(size_t)r * N + x] = flip || e0 == 0 ? e0 : q - e0;
  }
  __syncthreads();
  int first = w;  // this wave's first row of the digit: rows are dealt round robin over all digits
  for (int d = 0; d < a.dn; d++) {
    const int st0 = d * K, ns = min(st0 + K, nq) - st0, nrows = nqp - ns;
    const cwords dt = const_words(a.dtab[d]);
    const cwords dhat = const_words((const void*)dt[4 * HCK_MAXSRC]), dnS = const_words((const void*)dt[4 * HCK_MAXSRC + 1]);
    u64 y[8];
    double vf = 0.0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int r = st0 + (i < ns ? i : 0);
      const u64 yi = sm[r * BCL_X + lane];
      const double t = __longlong_as_double((long long)sm[(nq + r) * BCL_X + lane]);
      y[i] = i < ns ? yi : 0;
      vf += i < ns ? t : 0.0;
    }
    const uint32_t v = ns == 1 ? 0 : (uint32_t)(u64)vf;  // a digit of one modulus is spread without an overflow count
    int rr = first;
    for (; rr < nrows; rr += 4) {
      const int row = rr < st0 ? rr : rr + ns;
      const int m = row < nq ? row : a.L + row - nq;
      digits[((size_t)d * nqp + row) * N] =
          bconv_word8([&](int i) { return y[i]; }, dhat + (size_t)m * ns, v, dnS[m], mods[4 * m], mods[4 * m + 1]);
    }
    first = rr - nrows;
  }
}
size_t link_lds_bytes(int l) { return (size_t)std::max(4 * 8, 2 * (l + 1)) * BCL_X * 8; }
void launch_link(const LinkArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(link_kernel, dim3(a.N / BCL_X), dim3(256), link_lds_bytes(a.l), st, a);
}
void launch_bconv(const u64* in, size_t in_bstride, BConvJobs jobs, u64* out, size_t out_bstride, int batch,
                  const ModC* mods, int N, hipStream_t st) {
  if (jobs.n <= 0 || batch <= 0) return;
  int nrows = 0, nsmax = 0;
  for (int d = 0; d < jobs.n; d++) {
    nrows = std::max(nrows, jobs.j[d].rm.nact());
    nsmax = std::max(nsmax, jobs.j[d].ns);
  }
  if (nrows <= 0) return;
  // all destination rows in one thread unless that leaves too few workgroups
  const int cols = N / 256;
  // a launch of at most a few waves per SIMD: the shared-source form; also any
  // under an automorphism, which the other form knows nothing of
  const bool shared_ok = nsmax <= 8 && N % BCL_X == 0;
  if (jobs.ginv && !shared_ok) throw std::invalid_argument("basis extension under an automorphism: more than 8 sources");
  if (shared_ok && (jobs.ginv || (long)cols * batch * jobs.n < BCL_MAX_BLOCKS)) {
    hipLaunchKernelGGL(bconv_lds_kernel, dim3(N / BCL_X, 1, batch * jobs.n), dim3(256), 0, st, in, in_bstride, jobs, out,
                       out_bstride, mods, N);
    return;
  }
  int ny = 1;
  while (ny < nrows && (long)cols * batch * jobs.n * ny < 768) ny *= 2;
  jobs.rows_per_block = (nrows + ny - 1) / ny;
  ny = (nrows + jobs.rows_per_block - 1) / jobs.rows_per_block;
  dim3 grid(cols, ny, batch * jobs.n);
  if (nsmax <= 8)
    hipLaunchKernelGGL((bconv_kernel<8>), grid, dim3(256), 0, st, in, in_bstride, jobs, out, out_bstride, mods, N);
  else if (nsmax <= 16)
    hipLaunchKernelGGL((bconv_kernel<16>), grid, dim3(256), 0, st, in, in_bstride, jobs, out, out_bstride, mods, N);
  else
    hipLaunchKernelGGL((bconv_kernel<HCK_MAXSRC>), grid, dim3(256), 0, st, in, in_bstride, jobs, out, out_bstride, mods, N);
}
void launch_bconv(const u64* in, size_t in_bstride, int ns, const BConvTable* dtab, u64* out, size_t out_bstride, int batch,
                  const RowMap& rm, const ModC* mods, int N, hipStream_t st) {
  BConvJobs jobs{};
  jobs.n = 1;
  jobs.j[0] = BConvJob{dtab, 0, ns, 0, 0, rm, 0};
  launch_bconv(in, in_bstride, jobs, out, out_bstride, batch, mods, N, st);
}

__global__ void mul_i_kernel(u64* __restrict__ out, const u64* __restrict__ in, size_t bstride, RowMap rm,
                             const u64* __restrict__ iu, const u64* __restrict__ iup, const u64* __restrict__ niu,
                             const u64* __restrict__ niup, const ModC* __restrict__ mods, int N) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int row = rm.row(blockIdx.y), m = rm.mod(row);
  const size_t o = (size_t)blockIdx.z * bstride + (size_t)row * N + x;
  const bool lo = x < (N >> 1);
  out[o] = shoup_mul(in[o], lo ? iu[m] : niu[m], lo ? iup[m] : niup[m], mods[m].q);
}
void launch_mul_i(u64* out, const u64* in, size_t bstride, int batch, RowMap rm, const u64* iu, const u64* iup,
                  const u64* niu, const u64* niup, const ModC* mods, int N, hipStream_t st) {
  if (batch <= 0 || rm.nact() <= 0) return;
  hipLaunchKernelGGL(mul_i_kernel, dim3(N / 256, rm.nact(), batch), dim3(256), 0, st, out, in, bstride, rm, iu, iup, niu, niup,
                     mods, N);
}

// The counter PRNG of the key generator (see rand64 below).
__device__ __forceinline__ u64 mix64(u64 z) {
  z ^= z >> 30; z *= 0xbf58476d1ce4e5b9ULL;
  z ^= z >> 27; z *= 0x94d049bb133111ebULL;
  z ^= z >> 31; return z;
}
// Word (modulus index m, position x) of the a half of digit d of an
// evaluation key this library generated: a is sampled uniformly in the NTT
// domain, a[m][x] = floor(rand64(seed, stream_d, m*N + x) * q / 2^64), and
// kd = mix64(seed + G*(stream_d + 1)) is rand64's per-stream key, so the word
// is regenerated here instead of read (plain, not Montgomery form).
__device__ __forceinline__ u64 key_a_word(u64 kd, u64 ctr, u64 q) {
  return __umul64hi(mix64(kd ^ (ctr * 0xd1b54a32d192ed03ULL + 0x8cb92ba72f3d8dd7ULL)), q);
}

// ---------------------------------------------------------------------------
// Key inner product (gadget product) in QP, fused with the automorphism
// gather.  For output position i the thread reads every operand at
// src = perm[i]; inside an aligned block of 2^k outputs the sources form an
// aligned block of 2^k words, so the gathers stay coalesced.
//   mode 0: out = (sum_d dg_d*k0_d, sum_d dg_d*k1_d)                 (no perm)
//   mode 1: out = perm(sum dg*k0 + add0[Q rows], sum dg*k1)         (hoisted)
// Keys are in Montgomery form; the sum is accumulated lazily in 128 bits.
// With a.seeded the a halves (k1) are regenerated (key_a_word) instead of
// read: their products carry no factor R, so part 1 is multiplied by R
// after its REDC.  Launched for the naive transform's batches and for single
// key switches of more than HCK_KM1_DIG digits (keymac1_kernel below that).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void keymac_kernel(KeyMacArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y, b = blockIdx.z;
  const int N = a.N;
  const uint32_t* perm = a.perm ? a.perm[b] : a.perm1;
  const u64* key = a.key ? a.key[b] : a.key1;
  const int src = perm ? (int)perm[i] : i;
  const int kl = k <= a.l ? k : a.L + (k - a.l - 1);
  const ModC mc = a.mods[kl];
  const size_t db = (size_t)(a.digits_per_batch ? b : 0);
  const u64* dg = a.digits + db * a.dig_bstride;
  // the digit owning Q row k reads it from the decomposed polynomial itself
  const int own_d = (a.own && k <= a.l) ? k / a.K : -1;
  const u64* own = a.own ? a.own + db * a.own_bstride + (size_t)k * N : nullptr;
  const size_t kstride = (size_t)(a.L + a.K) * N;
  Acc128 A0, A1;
  acc_zero(A0); acc_zero(A1);
  const bool seeded = a.seeded && !a.key;
  for (int d = 0; d < a.dn; d++) {
    const u64 x = d == own_d ? own[src] : dg[((size_t)d * a.nqp + k) * N + src];
    const u64* kb = key + (size_t)d * 2 * kstride + (size_t)kl * N + src;
    acc_mac(A0, x, __builtin_nontemporal_load(&kb[0]));
    acc_mac(A1, x, seeded ? key_a_word(a.ka[d], (u64)kl * N + src, mc.q) : __builtin_nontemporal_load(&kb[kstride]));
  }
  u64 lo0, hi0, lo1, hi1;
  acc_value(A0, lo0, hi0);
  acc_value(A1, lo1, hi1);
  hi0 = fold_hi4(hi0, mc.q);
  hi1 = fold_hi4(hi1, mc.q);
  // add0 enters the high word (v*2^64 == v*R mod q), so the REDC below returns sum + add0
  if (a.add0 && k <= a.l) hi0 = add_mod(hi0, a.add0[(size_t)k * N + src], mc.q);
  const u64 add1 = (a.add1 && k <= a.l) ? a.add1[(size_t)k * N + src] : 0;
  if (!seeded) hi1 = add_mod(hi1, add1, mc.q);
  const size_t o = (size_t)b * a.out_bstride + (size_t)k * N + i;
  a.out0[o] = redc(lo0, hi0, mc.q, mc.qinv);
  const u64 r1 = redc(lo1, hi1, mc.q, mc.qinv);
  // regenerated a halves carry no R: the REDC left sum * R^-1, and add1 comes after the correction
  a.out1[o] = seeded ? add_mod(mont_mul(r1, mc.r2, mc.q, mc.qinv), add1, mc.q) : r1;
}
void launch_keymac(const KeyMacArgs& a, int batch, hipStream_t st) {
  if (batch <= 0) return;
  hipLaunchKernelGGL(keymac_kernel, dim3(a.N / 256, a.nqp, batch), dim3(256), 0, st, a);
}

// The key product of one key switch.  Bound by memory: DN digits unrolled, so
// that a word's 2 DN (3 DN with the a halves read) loads are in flight
// together, where keymac_kernel's loop waits for each digit's pair; at most 8
// products of words below q < 2^61 also need no folding of the sum's high
// word before the REDC.  Three digits, 31 rows of N = 2^16: 31 -> 24 us, 5.5 TB/s.
template <int DN, bool SEEDED, bool FOLD>
__global__ __launch_bounds__(256) void keymac1_kernel(KeyMac1Args a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y, N = a.N;
  const bool qrow = k <= a.l;
  const int src = a.perm ? (int)a.perm[i] : i;
  const int kl = qrow ? k : a.L + (k - a.l - 1);
  const ModC mc = a.mods[kl];
  const int own_d = qrow ? k / a.K : -1;
  const size_t kstride = (size_t)(a.L + a.K) * N, ro = (size_t)k * N;
  u64 x[DN], kb[DN], ka[DN];
#pragma unroll
  for (int d = 0; d < DN; d++) {
    const u64* dg = d == own_d ? a.own + ro : a.digits + (size_t)d * a.nqp * N + ro;
    const u64* key = a.key + (size_t)d * 2 * kstride + (size_t)kl * N + src;
    x[d] = dg[src];
    kb[d] = __builtin_nontemporal_load(key);
    if (!SEEDED) ka[d] = __builtin_nontemporal_load(key + kstride);
  }
  u64 add0 = 0, add1 = 0, c = 0;
  if (qrow) {
    if (FOLD) {
      u64 ci = a.c0[ro + i], cs = a.c0[ro + src];
      if (a.e0) {
        ci = add_mod(ci, a.e0[ro + i], mc.q);
        cs = add_mod(cs, a.e0[ro + src], mc.q);
      }
      c = add_mod(ci, cs, mc.q);
    } else {
      if (a.add0) add0 = a.add0[ro + src];
      if (a.add1) add1 = a.add1[ro + src];
    }
  }
  Acc128 A0, A1;
  acc_zero(A0); acc_zero(A1);
#pragma unroll
  for (int d = 0; d < DN; d++) {
    acc_mac(A0, x[d], kb[d]);
    acc_mac(A1, x[d], SEEDED ? key_a_word(a.ka[d], (u64)kl * N + src, mc.q) : ka[d]);
  }
  // at most 8 products of words below q < 2^61: the sum stays below q * 2^64
  u64 lo0, hi0, lo1, hi1;
  acc_value(A0, lo0, hi0);
  acc_value(A1, lo1, hi1);
  // add0 enters the high word (v*2^64 == v*R mod q), so the REDC returns sum + add0
  const u64 r0 = redc(lo0, add_mod(hi0, add0, mc.q), mc.q, mc.qinv);
  u64 r1;
  if (SEEDED) r1 = add_mod(mont_mul(redc(lo1, hi1, mc.q, mc.qinv), mc.r2, mc.q, mc.qinv), add1, mc.q);
  else r1 = redc(lo1, add_mod(hi1, add1, mc.q), mc.q, mc.qinv);
  if (FOLD && qrow) a.c0_out[ro + i] = add_mod(c, shoup_mul(r0, a.pinv[k], a.pinvp[k], mc.q), mc.q);
  else a.out0[ro + i] = r0;
  a.out1[ro + i] = r1;
}
template <int DN>
static void launch_keymac1_t(const KeyMac1Args& a, hipStream_t st) {
  if (DN < a.dn) {
    if constexpr (DN < HCK_KM1_DIG) launch_keymac1_t<DN + 1>(a, st);
    return;
  }
  const dim3 grid(a.N / 256, a.nqp), block(256);
  if (a.c0) {
    if (a.seeded) hipLaunchKernelGGL((keymac1_kernel<DN, true, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((keymac1_kernel<DN, false, true>), grid, block, 0, st, a);
  } else {
    if (a.seeded) hipLaunchKernelGGL((keymac1_kernel<DN, true, false>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((keymac1_kernel<DN, false, false>), grid, block, 0, st, a);
  }
}
void launch_keymac1(const KeyMac1Args& a, hipStream_t st) { launch_keymac1_t<1>(a, st); }

// Giant-step accumulation of the BSGS linear transform: for every QP row and
// output position i, sum over giant groups g of
//   [ sum_d dg_{g,d} * key_g[d] + T0_g ](perm_g[i])   (part 0)
//   [ sum_d dg_{g,d} * key_g[d] ](perm_g[i])           (part 1)
// plus the untransformed group (rotation 0) if present.  Everything folds
// into one lazy 128-bit accumulator per part: T0 is added to the high word
// (value*2^64 == value*R), so a single REDC finishes the row.
// running sum (lo, hi < q) += 128-bit column accumulator A, then A = 0
__device__ __forceinline__ void acc_flush(Acc128& A, u64& tlo, u64& thi, u64 q) {
  u64 lo, hi;
  acc_value(A, lo, hi);
  hi = fold_hi4(hi, q);
  tlo += lo;
  const u64 c = tlo < lo ? 1 : 0;
  thi = csub64(add_mod(thi, hi, q) + c, q);
  acc_zero(A);
}
__global__ __launch_bounds__(256) void giant_acc_kernel(GiantAccArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  const int N = a.N;
  const int kl = k <= a.l ? k : a.L + (k - a.l - 1);
  const ModC mc = a.mods[kl];
  const int own_d = (a.own && k <= a.l) ? k / a.K : -1;
  const size_t kstride = (size_t)(a.L + a.K) * N;
  Acc128 A0, A1;
  acc_zero(A0); acc_zero(A1);
  u64 tlo0 = 0, thi0 = 0, tlo1 = 0, thi1 = 0, t0 = 0;
  int cnt = 0;
  for (int g = 0; g < a.ng; g++) {
    if (cnt + a.dn > 16) {
      acc_flush(A0, tlo0, thi0, mc.q);
      acc_flush(A1, tlo1, thi1, mc.q);
      cnt = 0;
    }
    const uint32_t* perm = a.perm[g];
    const u64* key = a.key[g];
    const int src = (int)perm[i];
    const u64* dg = a.digits + (size_t)g * a.dig_bstride;
    const u64* own = a.own ? a.own + (size_t)g * a.own_bstride + (size_t)k * N : nullptr;
    const u64* ka = a.ka ? a.ka + (size_t)g * a.dn : nullptr;
    for (int d = 0; d < a.dn; d++) {
      const u64 x = d == own_d ? own[src] : dg[((size_t)d * a.nqp + k) * N + src];
      const u64* kb = key + (size_t)d * 2 * kstride + (size_t)kl * N + src;
      acc_mac(A0, x, __builtin_nontemporal_load(&kb[0]));
      acc_mac(A1, x, ka ? key_a_word(ka[d], (u64)kl * N + src, mc.q) : __builtin_nontemporal_load(&kb[kstride]));
    }
    cnt += a.dn;
    const u64* T0 = a.T + (size_t)a.tg[g] * a.T_gstride;
    t0 = add_mod(t0, T0[(size_t)k * N + src], mc.q);
  }
  acc_flush(A0, tlo0, thi0, mc.q);
  acc_flush(A1, tlo1, thi1, mc.q);
  // T0 terms enter the high word (v*2^64 == v*R mod q)
  thi0 = add_mod(thi0, t0, mc.q);
  u64 tz1 = 0;
  if (a.t_zero >= 0) {
    const u64* Tz = a.T + (size_t)a.t_zero * a.T_gstride;
    thi0 = add_mod(thi0, Tz[(size_t)k * N + i], mc.q);
    tz1 = Tz[a.T_pstride + (size_t)k * N + i];
  }
  const size_t o = (size_t)k * N + i;
  a.out0[o] = redc(tlo0, thi0, mc.q, mc.qinv);
  if (a.ka) {
    // regenerated a halves: the products' REDC lacks the factor R
    a.out1[o] = add_mod(mont_mul(redc(tlo1, thi1, mc.q, mc.qinv), mc.r2, mc.q, mc.qinv), tz1, mc.q);
  } else {
    a.out1[o] = redc(tlo1, add_mod(thi1, tz1, mc.q), mc.q, mc.qinv);
  }
}
// The same with the digit count known (up to HCK_KM1_DIG; longer
// decompositions take the loop above).  Bound by memory: the 2 DN + 1 words of
// a group (3 DN + 1 with the a halves read) are loaded together, behind the
// next group's source position, where the loop waits for each digit's pair.  31
// groups of 3 digits, 32 rows of N = 2^16: 800 -> 660 us, 5.5 TB/s over the
// b halves, digits and accumulators; 15 groups of 5 digits, 6 rows of 2^13:
// 17 -> 9 us.
template <int DN, bool SEEDED>
__global__ __launch_bounds__(256) void giant_acc_dn_kernel(GiantAccArgs a) {
  constexpr int PER = 16 / DN;  // groups per accumulator
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  const int N = a.N;
  const int kl = k <= a.l ? k : a.L + (k - a.l - 1);
  const ModC mc = a.mods[kl];
  const int own_d = (a.own && k <= a.l) ? k / a.K : -1;
  const size_t kstride = (size_t)(a.L + a.K) * N;
  Acc128 A0, A1;
  acc_zero(A0); acc_zero(A1);
  u64 tlo0 = 0, thi0 = 0, tlo1 = 0, thi1 = 0, t0 = 0;
  int next = (int)a.perm[0][i], cnt = 0;
  for (int g = 0; g < a.ng; g++) {
    const int src = next;
    next = (int)a.perm[min(g + 1, a.ng - 1)][i];
    const u64* dg = a.digits + (size_t)g * a.dig_bstride + (size_t)k * N + src;
    const u64* own = a.own ? a.own + (size_t)g * a.own_bstride + (size_t)k * N + src : nullptr;
    const u64* key = a.key[g] + (size_t)kl * N + src;
    u64 x[DN], kb[DN], ka[DN];
#pragma unroll
    for (int d = 0; d < DN; d++) {
      x[d] = *(d == own_d ? own : dg + (size_t)d * a.nqp * N);
      kb[d] = __builtin_nontemporal_load(key + (size_t)d * 2 * kstride);
      if (!SEEDED) ka[d] = __builtin_nontemporal_load(key + (size_t)d * 2 * kstride + kstride);
    }
    const u64 t = (a.T + (size_t)a.tg[g] * a.T_gstride)[(size_t)k * N + src];
    if (cnt == PER) {
      acc_flush(A0, tlo0, thi0, mc.q);
      acc_flush(A1, tlo1, thi1, mc.q);
      cnt = 0;
    }
    cnt++;
#pragma unroll
    for (int d = 0; d < DN; d++) {
      acc_mac(A0, x[d], kb[d]);
      acc_mac(A1, x[d], SEEDED ? key_a_word(a.ka[(size_t)g * DN + d], (u64)kl * N + src, mc.q) : ka[d]);
    }
    t0 = add_mod(t0, t, mc.q);
  }
  acc_flush(A0, tlo0, thi0, mc.q);
  acc_flush(A1, tlo1, thi1, mc.q);
  thi0 = add_mod(thi0, t0, mc.q);
  u64 tz1 = 0;
  if (a.t_zero >= 0) {
    const u64* Tz = a.T + (size_t)a.t_zero * a.T_gstride;
    thi0 = add_mod(thi0, Tz[(size_t)k * N + i], mc.q);
    tz1 = Tz[a.T_pstride + (size_t)k * N + i];
  }
  const size_t o = (size_t)k * N + i;
  a.out0[o] = redc(tlo0, thi0, mc.q, mc.qinv);
  if (SEEDED) a.out1[o] = add_mod(mont_mul(redc(tlo1, thi1, mc.q, mc.qinv), mc.r2, mc.q, mc.qinv), tz1, mc.q);
  else a.out1[o] = redc(tlo1, add_mod(thi1, tz1, mc.q), mc.q, mc.qinv);
}
template <int DN>
static bool launch_giant_acc_t(const GiantAccArgs& a, hipStream_t st) {
  if (DN < a.dn) {
    if constexpr (DN < HCK_KM1_DIG) return launch_giant_acc_t<DN + 1>(a, st);
    return false;
  }
  const dim3 grid(a.N / 256, a.nqp), block(256);
  if (a.ka) hipLaunchKernelGGL((giant_acc_dn_kernel<DN, true>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((giant_acc_dn_kernel<DN, false>), grid, block, 0, st, a);
  return true;
}
void launch_giant_acc(const GiantAccArgs& a, hipStream_t st) {
  if (a.ng > 0 && launch_giant_acc_t<1>(a, st)) return;
  hipLaunchKernelGGL(giant_acc_kernel, dim3(a.N / 256, a.nqp, 1), dim3(256), 0, st, a);
}

// ---------------------------------------------------------------------------
// Fused diagonal MAC of the BSGS linear transform.  One thread per (QP row,
// coefficient) holds the baby-step operands of its word in registers and
// streams every plaintext diagonal once, writing one accumulator pair per
// giant group:
//   T[g][p][k][x] = sum_{b in baby(g)} diag_{g,b}[k][x] * S_b[p][k][x]
// S_0 = P*c (Q rows only), S_b = hoisted rotation b (QP), computed in the
// prologue from the rotation's key and the decomposed input (the rotations
// are never written to or read from memory).  The next group's
// diagonals are loaded while the current group is multiplied (NB loads in
// flight per thread).  Products are summed exactly in 128 bits (16 products
// of words < 2^62 cannot overflow; the high word is folded below 4q after
// every 16), then one Montgomery REDC per word removes the 2^64 the
// diagonals carry.
// ---------------------------------------------------------------------------

// Plaintext index of baby b (chunk-relative) of group g: dense transforms
// (every group holds every baby of the chunk) store them group-major; the
// others use the index table, where an absent baby points at a zero plaintext.
template <bool DENSE>
__device__ __forceinline__ int mac_pidx(const DiagMacArgs& a, int g, int b) {
  if (DENSE) return g * a.nbaby + a.b0 + b;  // launched only when b0 + NB <= nbaby
  const int bb = a.b0 + b;
  return bb < a.nbaby ? a.gpi[(size_t)g * a.nbaby + bb] : a.zero_pidx;
}
// Diagonals are read exactly once per transform: non-temporal loads keep them
// from displacing reused data in L2 (measured 5 % faster on the full MAC).
// A later chunk of baby steps (ACC) also reads the group's accumulators
// written by the earlier chunks, together with its diagonals.
template <int NB, bool DENSE, bool ACC>
__device__ __forceinline__ void mac_load(const DiagMacArgs& a, const u64* dbase, int g, u64 (&d)[NB], u64 (&t)[2],
                                         const u64* Tb) {
#pragma unroll
  for (int b = 0; b < NB; b++) d[b] = __builtin_nontemporal_load(&dbase[(size_t)mac_pidx<DENSE>(a, g, b) * a.diag_stride]);
  if (ACC) {
    const u64* T = Tb + (size_t)g * a.T_gstride;
    t[0] = T[0];
    t[1] = T[a.T_pstride];
  }
}
template <int NB, bool ACC>
__device__ __forceinline__ void mac_group(const DiagMacArgs& a, const u64 (&d)[NB], const u64 (&t)[2], const u64 (&s0)[NB],
                                          const u64 (&s1)[NB], const ModC& mc, u64* T) {
  // exact column sums of 16 products; chunks of 16 are reduced to (lo, hi < q)
  u128 tot0 = 0, tot1 = 0;
#pragma unroll
  for (int c = 0; c < NB; c += 16) {
    Acc128 A0, A1;
    acc_zero(A0); acc_zero(A1);
#pragma unroll
    for (int b = c; b < c + 16 && b < NB; b++) {
      acc_mac(A0, d[b], s0[b]);
      acc_mac(A1, d[b], s1[b]);
    }
    u64 lo0, hi0, lo1, hi1;
    acc_value(A0, lo0, hi0);
    acc_value(A1, lo1, hi1);
    tot0 += ((u128)fold_hi4(hi0, mc.q) << 64) | lo0;
    tot1 += ((u128)fold_hi4(hi1, mc.q) << 64) | lo1;
  }
  // one chunk: hi < 4q was already folded below q
  u64 r0 = redc((u64)tot0, NB <= 16 ? (u64)(tot0 >> 64) : fold_hi4((u64)(tot0 >> 64), mc.q), mc.q, mc.qinv);
  u64 r1 = redc((u64)tot1, NB <= 16 ? (u64)(tot1 >> 64) : fold_hi4((u64)(tot1 >> 64), mc.q), mc.q, mc.qinv);
  if (ACC) { r0 = add_mod(r0, t[0], mc.q); r1 = add_mod(r1, t[1], mc.q); }
  __builtin_nontemporal_store(r0, &T[0]);
  __builtin_nontemporal_store(r1, &T[a.T_pstride]);
}

// One word of a hoisted baby rotation, keymac_kernel's arithmetic at (row k,
// position x): src = perm[x], sum_d digit_d[k][src] * key[d][p][kl][src]
// (+ P c0[k][src] in part 0), one REDC per part.
__device__ __forceinline__ void baby_rotation_at(const DiagMacArgs& a, int slot, int k, int kl, int x, const ModC& mc,
                                                 u64& r0, u64& r1) {
  const int N = a.N;
  const int src = (int)a.bperm[slot][x];
  const u64* key = a.bkey[slot];
  const u64* ka = a.bka ? a.bka + (size_t)slot * a.dn : nullptr;
  const int own_d = k <= a.l ? k / a.K : -1;
  const size_t kstride = (size_t)(a.L + a.K) * N;
  Acc128 A0, A1;
  acc_zero(A0); acc_zero(A1);
  for (int d = 0; d < a.dn; d++) {
    const u64 v = d == own_d ? a.own[(size_t)k * N + src] : a.digits[((size_t)d * a.nqp + k) * N + src];
    const u64* kb = key + (size_t)d * 2 * kstride + (size_t)kl * N + src;
    acc_mac(A0, v, __builtin_nontemporal_load(&kb[0]));
    acc_mac(A1, v, ka ? key_a_word(ka[d], (u64)kl * N + src, mc.q) : __builtin_nontemporal_load(&kb[kstride]));
  }
  u64 lo0, hi0, lo1, hi1;
  acc_value(A0, lo0, hi0);
  acc_value(A1, lo1, hi1);
  hi0 = fold_hi4(hi0, mc.q);
  hi1 = fold_hi4(hi1, mc.q);
  if (k <= a.l) hi0 = add_mod(hi0, a.pc[(size_t)k * N + src], mc.q);
  r0 = redc(lo0, hi0, mc.q, mc.qinv);
  r1 = redc(lo1, hi1, mc.q, mc.qinv);
  if (ka) r1 = mont_mul(r1, mc.r2, mc.q, mc.qinv);  // regenerated a halves carry no R
}

// The groups of a workgroup: a launch of few workgroups deals them out over
// blockIdx.z (each part computes the baby rotations for itself).
__device__ __forceinline__ int mac_g0(const DiagMacArgs& a) { return a.g0 + (int)blockIdx.z * a.gper; }
template <int NB, bool DENSE, bool ACC>
__global__ __launch_bounds__(256) void diag_mac_kernel(DiagMacArgs a) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  const int N = a.N;
  const int kl = k <= a.l ? k : a.L + (k - a.l - 1);
  const ModC mc = a.mods[kl];
  const int krow = k <= a.l ? k : a.lt_level + 1 + (k - a.l - 1);  // row inside a diagonal
  const u64* dbase = a.diag + (size_t)krow * N + x;
  u64 s0[NB], s1[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int bb = a.b0 + b;
    s0[b] = 0; s1[b] = 0;
    if (bb < a.nbaby) {
      if (a.baby_is_zero[bb]) {
        if (k <= a.l) { s0[b] = a.pc[(size_t)k * N + x]; s1[b] = a.pc[a.pc_pstride + (size_t)k * N + x]; }
      } else {
        baby_rotation_at(a, a.baby_slot[bb], k, kl, x, mc, s0[b], s1[b]);
      }
    }
  }
  // ping-pong: the next group's NB diagonals are in flight while a group is
  // multiplied.  The prefetches inside the loop are unconditional (the last
  // one or two groups are peeled off): a prefetch under a branch makes the
  // compiler wait for every outstanding load, the prefetch included, before
  // the current group's products.
  u64 dA[NB], dB[NB], tA[2], tB[2];
  u64* Tb = a.T + (size_t)k * N + x;
  int g = mac_g0(a);
  const int g1 = min(a.g1, g + a.gper);
  mac_load<NB, DENSE, ACC>(a, dbase, g, dA, tA, Tb);
  // (the scheduling barriers keep the machine scheduler from sinking the
  // prefetch below the products to save registers)
  for (; g + 2 < g1; g += 2) {
    mac_load<NB, DENSE, ACC>(a, dbase, g + 1, dB, tB, Tb);
    __builtin_amdgcn_sched_barrier(0);
    mac_group<NB, ACC>(a, dA, tA, s0, s1, mc, Tb + (size_t)g * a.T_gstride);
    mac_load<NB, DENSE, ACC>(a, dbase, g + 2, dA, tA, Tb);
    __builtin_amdgcn_sched_barrier(0);
    mac_group<NB, ACC>(a, dB, tB, s0, s1, mc, Tb + (size_t)(g + 1) * a.T_gstride);
  }
  if (g + 1 < g1) {
    mac_load<NB, DENSE, ACC>(a, dbase, g + 1, dB, tB, Tb);
    __builtin_amdgcn_sched_barrier(0);
    mac_group<NB, ACC>(a, dA, tA, s0, s1, mc, Tb + (size_t)g * a.T_gstride);
    mac_group<NB, ACC>(a, dB, tB, s0, s1, mc, Tb + (size_t)(g + 1) * a.T_gstride);
  } else {
    mac_group<NB, ACC>(a, dA, tA, s0, s1, mc, Tb + (size_t)g * a.T_gstride);
  }
}
// The dense 16-baby diagonal MAC over diagonals stored in the packed layout.
// Each wave fetches its 64 coefficients' chunk of 8 diagonals at a time
// (half a giant group) straight into LDS with global_load_lds_dwordx4 -- a
// packed row's chunk is 104 dwords (26 lanes x 16 B), a plain row's 128 (32
// lanes) -- the next half's while the current one is multiplied, so no
// registers are held by loads in flight, and unpacks its own word from LDS.
// A packed row reads 104 instead of 128 dwords per 64 words.
constexpr int MAC_HALF = 8, MAC_SLOT = 128;
typedef uint32_t MacLds[2][MAC_HALF][MAC_SLOT];  // one wave's two half-group buffers
// The group loop of one row (PK: stored packed).  Wait counts: vector memory
// operations complete in issue order; a half's 8 chunks are in LDS once at
// most the operations issued after them are outstanding: the next half's 8
// loads, plus the previous group's two accumulator stores when they came in
// between (first half of every group but the first).
template <bool PK>
__device__ __forceinline__ void mac_d16_rows(const DiagMacArgs& a, const u64 (&s0)[16], const u64 (&s1)[16], const ModC& mc,
                                             u64* Tb, const uint32_t* wbase, MacLds& lds, int lane) {
  constexpr int SLOT = PK ? PK_CHUNK : MAC_SLOT;  // dwords of one 64-word chunk
  const size_t ds = 2 * a.diag_stride;            // dwords from one diagonal to the next
  // half h = 2 g + i: diagonals 8 i .. 8 i + 7 of group g into buffer h & 1
  auto issue = [&](int h) {
    if (lane < SLOT / 4) {
      const uint32_t* src = wbase + (size_t)(h * MAC_HALF) * ds + 4 * lane;
#pragma unroll
      for (int b = 0; b < MAC_HALF; b++)
        __builtin_amdgcn_global_load_lds((const void*)(src + (size_t)b * ds),
                                         (__attribute__((address_space(3))) void*)&lds[h & 1][b][0], 16, 0, 0);
    }
  };
  const int g0 = mac_g0(a), g1 = min(a.g1, g0 + a.gper);
  issue(2 * g0);
  for (int g = g0; g < g1; g++) {
    Acc128 A0, A1;
    acc_zero(A0); acc_zero(A1);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int h = 2 * g + i;
      const bool more = i == 0 || g + 1 < g1;
      if (more) issue(h + 1);
      if (!more) __builtin_amdgcn_s_waitcnt((0x7 << 4) | (0xF << 8));                       // vmcnt(0)
      else if (i == 0 && g != g0) __builtin_amdgcn_s_waitcnt((0x7 << 4) | (0xF << 8) | 10);  // vmcnt(10)
      else __builtin_amdgcn_s_waitcnt((0x7 << 4) | (0xF << 8) | 8);                         // vmcnt(8)
#pragma unroll
      for (int b = 0; b < MAC_HALF; b++) {
        const uint32_t* c = &lds[h & 1][b][0];
        const u64 d = PK ? pk_field(c, lane) : ((u64)c[2 * lane + 1] << 32) | c[2 * lane];
        acc_mac(A0, d, s0[MAC_HALF * i + b]);
        acc_mac(A1, d, s1[MAC_HALF * i + b]);
      }
    }
    // 16 products of words < 2^62: the high word folded below q, one REDC
    u64 lo0, hi0, lo1, hi1;
    acc_value(A0, lo0, hi0);
    acc_value(A1, lo1, hi1);
    u64* T = Tb + (size_t)g * a.T_gstride;
    __builtin_nontemporal_store(redc(lo0, fold_hi4(hi0, mc.q), mc.q, mc.qinv), &T[0]);
    __builtin_nontemporal_store(redc(lo1, fold_hi4(hi1, mc.q), mc.q, mc.qinv), &T[a.T_pstride]);
  }
}
__global__ __launch_bounds__(256) void diag_mac_d16_kernel(DiagMacArgs a) {
  constexpr int NB = 16;
  __shared__ MacLds lds[4];
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  const int N = a.N;
  const int kl = k <= a.l ? k : a.L + (k - a.l - 1);
  const ModC mc = a.mods[kl];
  const int krow = k <= a.l ? k : a.lt_level + 1 + (k - a.l - 1);  // row inside a diagonal
  u64 s0[NB], s1[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    s0[b] = 0; s1[b] = 0;
    if (a.baby_is_zero[b]) {
      if (k <= a.l) { s0[b] = a.pc[(size_t)k * N + x]; s1[b] = a.pc[a.pc_pstride + (size_t)k * N + x]; }
    } else {
      baby_rotation_at(a, a.baby_slot[b], k, kl, x, mc, s0[b], s1[b]);
    }
  }
  u64* Tb = a.T + (size_t)k * N + x;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // this wave's chunk of the row: 64 coefficients from blockIdx.x * 256 + 64 w
  const uint32_t* rbase = reinterpret_cast<const uint32_t*>(a.diag) + a.pkrow[2 * krow];
  const size_t c = (size_t)blockIdx.x * 4 + w;
  if (a.pkrow[2 * krow + 1]) mac_d16_rows<true>(a, s0, s1, mc, Tb, rbase + c * PK_CHUNK, lds[w], lane);
  else mac_d16_rows<false>(a, s0, s1, mc, Tb, rbase + c * MAC_SLOT, lds[w], lane);
}
// Fewer workgroups than this (four on a CU) share out the giant groups, down to
// four a part.  N = 2^13, 10 rows: a wave a SIMD went through 26 groups one
// after the other, ten ragged tables 499 -> 436 us with four parts; N = 2^16
// fills the GPU with one.
constexpr long MAC_FILL = 1024;
void launch_diag_mac(const DiagMacArgs& args, hipStream_t st) {
  const int ng = args.g1 - args.g0;
  if (ng <= 0) return;
  DiagMacArgs a = args;
  int parts = 1;
  while ((long)(a.N / 256) * a.nqp * parts < MAC_FILL && ng >= 8 * parts) parts *= 2;
  a.gper = (ng + parts - 1) / parts;
  parts = (ng + a.gper - 1) / a.gper;
  if (a.pkrow) {
    // a transform stored packed (dense, 16 baby steps)
    hipLaunchKernelGGL(diag_mac_d16_kernel, dim3(a.N / 256, a.nqp, parts), dim3(256), 0, st, a);
    return;
  }
  dim3 grid(a.N / 256, a.nqp, parts);
  const bool dense = a.dense && a.nb_chunk == 16 && a.b0 + 16 <= a.nbaby;
  if (a.b0 == 0) {
    if (dense) hipLaunchKernelGGL((diag_mac_kernel<16, true, false>), grid, dim3(256), 0, st, a);
    else if (a.nb_chunk <= 8) hipLaunchKernelGGL((diag_mac_kernel<8, false, false>), grid, dim3(256), 0, st, a);
    else if (a.nb_chunk <= 16) hipLaunchKernelGGL((diag_mac_kernel<16, false, false>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((diag_mac_kernel<32, false, false>), grid, dim3(256), 0, st, a);
  } else {
    // later chunks of a transform with more than 32 baby steps accumulate
    if (a.nb_chunk <= 8) hipLaunchKernelGGL((diag_mac_kernel<8, false, true>), grid, dim3(256), 0, st, a);
    else if (a.nb_chunk <= 16) hipLaunchKernelGGL((diag_mac_kernel<16, false, true>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((diag_mac_kernel<32, false, true>), grid, dim3(256), 0, st, a);
  }
}

// RNS multiply-accumulate over a batch: out[r][x] = sum_p a[p][r][x] * b[p][r][x]
// mod q_r (canonical inputs and output).  Exact 128-bit column sums of 16
// products, then REDC and a Montgomery multiplication by R^2 mod q undo the
// 2^-64 of the REDC.
__global__ __launch_bounds__(256) void mulacc_kernel(const u64* __restrict__ a, const u64* __restrict__ b,
                                                     u64* __restrict__ out, int npoly, int nrows,
                                                     const ModC* __restrict__ mods, int N) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  const ModC mc = mods[r];
  const size_t pstride = (size_t)nrows * N, o = (size_t)r * N + x;
  Acc128 A;
  acc_zero(A);
  u64 tlo = 0, thi = 0;
  for (int p0 = 0; p0 < npoly; p0 += 16) {
    const int p1 = min(p0 + 16, npoly);
    for (int p = p0; p < p1; p++) acc_mac(A, a[(size_t)p * pstride + o], b[(size_t)p * pstride + o]);
    acc_flush(A, tlo, thi, mc.q);
  }
  out[o] = mont_mul(redc(tlo, thi, mc.q, mc.qinv), mc.r2, mc.q, mc.qinv);
}
void launch_mulacc(const u64* a, const u64* b, u64* out, int npoly, int nrows, const ModC* mods, int N, hipStream_t st) {
  if (npoly <= 0 || nrows <= 0) return;
  hipLaunchKernelGGL(mulacc_kernel, dim3(N / 256, nrows), dim3(256), 0, st, a, b, out, npoly, nrows, mods, N);
}

// ---------------------------------------------------------------------------
// Rescale helpers (DivRoundByLastModulus): u = iNTT(x_l) per polynomial;
// t_i = ((u + h) mod q_l - h) mod q_i for i < l; out_i = (x_i - NTT(t_i)) * q_l^-1
// ---------------------------------------------------------------------------
__global__ void rescale_spread_kernel(u64* __restrict__ t, const u64* __restrict__ u, int l, u64 half,
                                      const ModC* __restrict__ mods, int N) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int i = blockIdx.y, p = blockIdx.z;
  u64 ql = mods[l].q;
  u64 w = add_mod(u[(size_t)p * N + x], half, ql);
  ModC mc = mods[i];
  u64 wr = mont_mul(w, mc.rmod, mc.q, mc.qinv);  // w mod q_i
  u64 hr = mont_mul(half, mc.rmod, mc.q, mc.qinv);
  t[((size_t)p * l + i) * N + x] = sub_mod(wr, hr, mc.q);
}
void launch_rescale_spread(u64* t, const u64* u, int l, u64 half, const ModC* mods, int N, hipStream_t st) {
  hipLaunchKernelGGL(rescale_spread_kernel, dim3(N / 256, l, 2), dim3(256), 0, st, t, u, l, half, mods, N);
}

__global__ void rescale_pair_spread_kernel(u64* __restrict__ t, const u64* __restrict__ u, int l, u64 half, RescalePair rp,
                                           u64* __restrict__ ks, const ModC* __restrict__ mods, int N) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = blockIdx.y, b = blockIdx.z, g = b >> 1, p = b & 1;
  const u64 ql = mods[l].q;
  const u64 v = shoup_mul(u[(size_t)p * N + x], rp.kl[g], rp.klp[g], ql);
  const u64 w = add_mod(v, half, ql);
  const ModC mc = mods[i];
  const u64 wr = mont_mul(w, mc.rmod, mc.q, mc.qinv);  // w mod q_i
  const u64 hr = mont_mul(half, mc.rmod, mc.q, mc.qinv);
  t[((size_t)b * l + i) * N + x] = sub_mod(wr, hr, mc.q);
  if (x == 0 && p == 0) {
    ks[(size_t)(0 * 2 + g) * l + i] = rp.k[g][i];
    ks[(size_t)(1 * 2 + g) * l + i] = rp.kp[g][i];
    ks[(size_t)(2 * 2 + g) * l + i] = rp.c[g][i];
  }
}
void launch_rescale_pair_spread(u64* t, const u64* u, int l, u64 half, const RescalePair& rp, u64* ks, const ModC* mods,
                                int N, hipStream_t st) {
  hipLaunchKernelGGL(rescale_pair_spread_kernel, dim3(N / 256, l, 4), dim3(256), 0, st, t, u, l, half, rp, ks, mods, N);
}

// ModDown followed by a rescale, in the coefficient domain of the extension.
// ext[p] holds [x]_P extended to rows q_0..q_l (coefficient domain) and
// xl[p] row l of x (coefficient domain).  Row l of the ModDown result is
//   y = (xl - ext_l) * P^-1 mod q_l
// (the coefficients the rescale would get from the inverse NTT of that row),
// and the rescale subtracts t_i = ([y + half]_{q_l} - half) mod q_i; so that
// one forward NTT and one (P q_l)^-1 finish both steps, rows i < l become
//   ext_i + P * t_i mod q_i                (in place).
__global__ void moddown_rescale_spread_kernel(u64* __restrict__ ext, size_t e_bstride, const u64* __restrict__ xl,
                                              size_t x_bstride, int l, u64 half, u64 pinvl, u64 pinvlp,
                                              const u64* __restrict__ pmod_w, const u64* __restrict__ pmod_wp,
                                              const ModC* __restrict__ mods, int N) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = blockIdx.y, p = blockIdx.z;
  u64* e = ext + (size_t)p * e_bstride;
  const u64 ql = mods[l].q;
  const u64 y = shoup_mul(sub_mod(xl[(size_t)p * x_bstride + x], e[(size_t)l * N + x], ql), pinvl, pinvlp, ql);
  const u64 w = add_mod(y, half, ql);
  const ModC mc = mods[i];
  const u64 wr = mont_mul(w, mc.rmod, mc.q, mc.qinv);  // w mod q_i
  const u64 hr = mont_mul(half, mc.rmod, mc.q, mc.qinv);
  const u64 t = sub_mod(wr, hr, mc.q);
  u64* ei = e + (size_t)i * N + x;
  *ei = add_mod(*ei, shoup_mul(t, pmod_w[i], pmod_wp[i], mc.q), mc.q);
}
void launch_moddown_rescale_spread(u64* ext, size_t e_bstride, const u64* xl, size_t x_bstride, int l, u64 half, u64 pinvl,
                                   u64 pinvlp, const u64* pmod_w, const u64* pmod_wp, const ModC* mods, int N, int batch,
                                   hipStream_t st) {
  hipLaunchKernelGGL(moddown_rescale_spread_kernel, dim3(N / 256, l, batch), dim3(256), 0, st, ext, e_bstride, xl, x_bstride,
                     l, half, pinvl, pinvlp, pmod_w, pmod_wp, mods, N);
}

// ---------------------------------------------------------------------------
// Sampling (counter PRNG shared with the key/encryption specification):
//   rand64(seed, stream, ctr) = mix(mix(seed + G*(stream+1)) ^ (ctr*M1 + M2))
// ---------------------------------------------------------------------------
__device__ __forceinline__ u64 rand64(u64 seed, u64 stream, u64 ctr) {
  u64 k = mix64(seed + 0x9e3779b97f4a7c15ULL * (stream + 1));
  return mix64(k ^ (ctr * 0xd1b54a32d192ed03ULL + 0x8cb92ba72f3d8dd7ULL));
}
// uniform residues: row r (modulus m) coefficient x gets rand64(seed, stream, m*N + x) * q >> 64
__global__ void sample_uniform_kernel(u64* __restrict__ out, RowMap rm, u64 seed, u64 stream, const ModC* __restrict__ mods, int N) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int row = rm.row(blockIdx.y);
  int m = rm.mod(row);
  u64 r = rand64(seed, stream, (u64)m * N + x);
  out[(size_t)row * N + x] = __umul64hi(r, mods[m].q);
}
void launch_sample_uniform(u64* out, RowMap rm, u64 seed, u64 stream, const ModC* mods, int N, hipStream_t st) {
  hipLaunchKernelGGL(sample_uniform_kernel, dim3(N / 256, rm.nact(), 1), dim3(256), 0, st, out, rm, seed, stream, mods, N);
}
// centred binomial (eta = 21) error, the same integer reduced into every row
__global__ void sample_cbd_kernel(u64* __restrict__ out, RowMap rm, u64 seed, u64 stream, const ModC* __restrict__ mods, int N) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int row = rm.row(blockIdx.y);
  u64 q = mods[rm.mod(row)].q;
  u64 r = rand64(seed, stream, (u64)x);
  int e = __popcll(r & 0x1FFFFFULL) - __popcll((r >> 21) & 0x1FFFFFULL);
  out[(size_t)row * N + x] = e >= 0 ? (u64)e : q - (u64)(-e);
}
void launch_sample_cbd(u64* out, RowMap rm, u64 seed, u64 stream, const ModC* mods, int N, hipStream_t st) {
  hipLaunchKernelGGL(sample_cbd_kernel, dim3(N / 256, rm.nact(), 1), dim3(256), 0, st, out, rm, seed, stream, mods, N);
}
// small signed integers (int8, e.g. ternary) reduced into every row
__global__ void signed_rows_kernel(u64* __restrict__ out, RowMap rm, const int8_t* __restrict__ v, const ModC* __restrict__ mods, int N) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int row = rm.row(blockIdx.y);
  u64 q = mods[rm.mod(row)].q;
  int e = v[x];
  out[(size_t)row * N + x] = e >= 0 ? (u64)e : q - (u64)(-e);
}
void launch_signed_rows(u64* out, RowMap rm, const int8_t* v, const ModC* mods, int N, hipStream_t st) {
  hipLaunchKernelGGL(signed_rows_kernel, dim3(N / 256, rm.nact(), 1), dim3(256), 0, st, out, rm, v, mods, N);
}
// The polynomial with coefficient +1 at pos[i] / 2 for even pos[i], -1 for odd
// ones (distinct places) and 0 elsewhere, reduced into every row: 1024
// coefficients of a row a workgroup, gathered in LDS.  The positions come with
// the arguments (POS, an array of them) or from memory.
template <class POS>
__global__ __launch_bounds__(256) void ternary_rows_kernel(u64* __restrict__ out, RowMap rm, POS pos, int npos,
                                                          const ModC* __restrict__ mods, int N) {
  __shared__ int v[1024];
  const int base = blockIdx.x * 1024;
  for (int i = threadIdx.x; i < 1024; i += 256) v[i] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < npos; i += 256) {
    const uint32_t p = pos[i];
    const int x = (int)(p >> 1) - base;
    if (x >= 0 && x < 1024) v[x] = p & 1 ? -1 : 1;
  }
  __syncthreads();
  const int row = rm.row(blockIdx.y);
  const u64 q = mods[rm.mod(row)].q;
  for (int i = threadIdx.x; i < 1024; i += 256) out[(size_t)row * N + base + i] = v[i] < 0 ? q - 1 : (u64)v[i];
}
void launch_ternary_rows(u64* out, RowMap rm, const uint32_t* pos, int npos, const ModC* mods, int N, hipStream_t st) {
  hipLaunchKernelGGL(ternary_rows_kernel<const uint32_t*>, dim3(N / 1024, rm.nact(), 1), dim3(256), 0, st, out, rm, pos, npos,
                     mods, N);
}
void launch_ternary_rows(u64* out, RowMap rm, const TernaryPos& pos, int npos, const ModC* mods, int N, hipStream_t st) {
  hipLaunchKernelGGL(ternary_rows_kernel<TernaryPos>, dim3(N / 1024, rm.nact(), 1), dim3(256), 0, st, out, rm, pos, npos, mods,
                     N);
}
// The coefficients of a fresh encryption: part b of x = pk u, with rows
// q_0..q_l and p_0, plus its error e, divided by p_0 (Lattigo's ModDown from
// Q + {p_0}):
//   out_i = (x_i + e - ext_i) / p_0 mod q_i,  ext = x_{p_0} + e extended to q_i:
// one source, so y = x_{p_0} + e itself, less p_0 where its overflow count
// (u64)((double)y / (double)p_0) rounds to one.  One pass instead of two error
// launches, the extension and the combination, 45 us of 25 rows at N = 2^16;
// a thread takes every gridDim.y-th row, so that a coefficient's error and y
// are drawn a few times and not once a row.
__global__ __launch_bounds__(256) void encrypt_down_kernel(EncryptDownArgs a) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.z, N = a.N, nq = a.l + 1;
  const u64* in = a.x + (size_t)b * a.x_bstride + x;
  u64* out = a.out + (size_t)b * nq * N + x;
  const u64 p0 = a.mods[a.mp].q;
  const u64 r = rand64(a.seed, a.stream[b], (u64)x);
  const int e = __popcll(r & 0x1FFFFFULL) - __popcll((r >> 21) & 0x1FFFFFULL);
  const u64 y = add_mod(in[(size_t)nq * N], e >= 0 ? (u64)e : p0 - (u64)(-e), p0);
  const bool over = (u64)((double)y / (double)p0) != 0;
  for (int i = blockIdx.y; i < nq; i += gridDim.y) {
    const ModC mc = a.mods[i];
    const u64 xi = add_mod(in[(size_t)i * N], e >= 0 ? (u64)e : mc.q - (u64)(-e), mc.q);
    u64 ext = mont_mul(y, mc.rmod, mc.q, mc.qinv);  // y mod q_i
    if (over) ext = sub_mod(ext, mont_mul(p0, mc.rmod, mc.q, mc.qinv), mc.q);
    out[(size_t)i * N] = shoup_mul(sub_mod(xi, ext, mc.q), a.p0inv[i], a.p0invp[i], mc.q);
  }
}
void launch_encrypt_down(const EncryptDownArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(encrypt_down_kernel, dim3(a.N / 256, std::min(a.l + 1, 4), 2), dim3(256), 0, st, a);
}
// Galois-key body: b = -a*s' + e (+ P*s on own rows), in place on b; a, s', s in
// (a standard, sR/soR Montgomery), own rows [own0, own1) of the Q chain.
__global__ void gk_combine_kernel(u64* __restrict__ b, const u64* __restrict__ a, const u64* __restrict__ soR,
                                  const u64* __restrict__ sR, int own0, int own1, const u64* __restrict__ pmod,
                                  const ModC* __restrict__ mods, int N) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int m = blockIdx.y;
  ModC mc = mods[m];
  size_t o = (size_t)m * N + x;
  u64 v = sub_mod(b[o], mont_mul(a[o], soR[o], mc.q, mc.qinv), mc.q);
  if (m >= own0 && m < own1) v = add_mod(v, mont_mul(pmod[m], sR[o], mc.q, mc.qinv), mc.q);
  b[o] = v;
}
void launch_gk_combine(u64* b, const u64* a, const u64* soR, const u64* sR, int own0, int own1, const u64* pmod, int rows,
                       const ModC* mods, int N, hipStream_t st) {
  hipLaunchKernelGGL(gk_combine_kernel, dim3(N / 256, rows, 1), dim3(256), 0, st, b, a, soR, sR, own0, own1, pmod, mods, N);
}


// ---------------------------------------------------------------------------
// Integer VALU issue-rate probe: every lane runs iters x 8 independent
// instructions of one kind, so the launch is limited by VALU issue alone:
//   op 0: v_mad_u64_u32 (the 32 x 32 + 64 multiply-add the NTT butterflies,
//         key products and basis conversions are built from; its carry-out
//         goes to an SGPR pair that is never read)
//   op 1: v_add3_u32 (a plain full-rate 32-bit integer instruction)
// The faster of the two is the integer issue peak that VALU utilisation is
// quoted against.
// ---------------------------------------------------------------------------
template <int OP>
__global__ __launch_bounds__(256) void valu_probe_kernel(u64* __restrict__ out, uint32_t seed, int iters) {
  uint32_t a[8];
  u64 b[8];
#pragma unroll
  for (int i = 0; i < 8; i++) { a[i] = seed + threadIdx.x * 7u + (uint32_t)i; b[i] = (u64)a[i] * 0x12345ull; }
  const uint32_t c = seed | 1u;
  for (int it = 0; it < iters; it++) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (OP == 0) {
        u64 junk;
        asm volatile("v_mad_u64_u32 %0, %1, %2, %3, %0" : "+v"(b[i]), "=s"(junk) : "v"(a[i]), "v"(c));
      } else {
        asm volatile("v_add3_u32 %0, %0, %1, %1" : "+v"(a[i]) : "v"(c));
      }
    }
  }
  u64 s = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) s += a[i] + b[i];
  out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = s;
}
// Launch-latency probe: a kernel that does nothing (its store is never taken
// for the flags the host passes), to time a chain of dependent launches.
__global__ __launch_bounds__(256) void empty_probe_kernel(u64* out, int flag) {
  if (flag == 0x7fffffff && threadIdx.x == 0) out[blockIdx.x] = 1;
}
void launch_empty_probe(u64* out, int blocks, int flag, hipStream_t st) {
  hipLaunchKernelGGL(empty_probe_kernel, dim3(blocks), dim3(256), 0, st, out, flag);
}
void launch_valu_probe(int op, u64* out, int blocks, uint32_t seed, int iters, hipStream_t st) {
  if (op == 0) hipLaunchKernelGGL((valu_probe_kernel<0>), dim3(blocks), dim3(256), 0, st, out, seed, iters);
  else hipLaunchKernelGGL((valu_probe_kernel<1>), dim3(blocks), dim3(256), 0, st, out, seed, iters);
}
