// encoder.hip -- CKKS encoding on the device (Lattigo ckks.Encoder algorithm).
//
// A plaintext of `slots` = N/2 real values becomes N integer coefficients:
//   1. the values (fp32 as they cross the ABI, widened to float64) go through
//      the special inverse FFT over the rotation group 5^j mod 2N (DIF
//      butterflies len = slots .. 2, then bit reversal and division by slots);
//   2. real parts are coefficients [0, slots), imaginary parts [slots, N),
//      each scaled and rounded to a fixed-point integer (|v|*scale + 0.5
//      truncated below 2^64, exact mantissa * 2^e above);
//   3. the integer is reduced into every row of the plaintext's RNS basis.
// The forward NTT and the Montgomery conversion that follow are the library's
// own kernels.
//
// Decoding goes the other way: the centred CRT of each coefficient in multiword
// integers, the nearest double of it over the scale, and the special FFT.
//
// Every floating-point operation is the one of the scalar restatement, in the
// same order, with contraction into fused multiply-adds switched off, so the
// coefficients and the decoded values are bit-identical to a scalar float64
// evaluation of the algorithm.  The FFT's log2(slots) stages run in two
// launches through LDS: the stages inside aligned blocks of 256 values, and
// those across blocks on 8 columns of the (slots / 256) x 256 view.  At 2^15
// slots a launch a stage took 15 dependent launches for 512 KB of data.
#include "hipckks.h"
#include "kernels.h"

namespace {

constexpr int FFT_B = 256;   // values of a block (the stages len <= FFT_B)
constexpr int FFT_CW = 8;    // columns of a workgroup of the stages above: 64-byte rows, n / 256 <= 128 rows in 16 KB
struct FftArgs {
  double *re, *im;
  size_t pstride;
  int n, M;
  const int* rotgroup;
  const double *rre, *rim;
  // inverse: the column pass reads element k of plaintext p from
  // data[src * n + ((k + rot) mod n)], or 0 from nvals on; complex input: (re, im)
  // pairs at data[2k], data[2k + 1]
  const float* data;
  const EncodeSrc* src;  // nullptr: one plaintext, source 0 unrotated
  int nvals, complex_in;
  // forward: the column pass writes the real parts as float (mode 0) or double
  // (1), or (re, im) pairs of float (2)
  void* out;
  int mode;
};

// the twiddle of stage len, root j (conjugate for the inverse)
template <bool INV>
__device__ __forceinline__ double2 fft_root(const FftArgs& a, int len, int j) {
  const int lenq = len << 2, gap = a.M / lenq, r = a.rotgroup[j] & (lenq - 1);
  const int idx = (INV ? lenq - r : r) * gap;
  return make_double2(a.rre[idx], a.rim[idx]);
}
// one butterfly: forward (u, v) -> (u + w v, u - w v), inverse (u, v) ->
// (u + v, (u - v) w)
template <bool INV>
__device__ __forceinline__ void fft_butterfly(double2 w, double& ur, double& ui, double& vr, double& vi) {
#pragma clang fp contract(off)
  if (INV) {
    const double dr = ur - vr, di = ui - vi;
    ur = ur + vr;
    ui = ui + vi;
    vr = dr * w.x - di * w.y;
    vi = dr * w.y + di * w.x;
  } else {
    const double tr = vr * w.x - vi * w.y, ti = vr * w.y + vi * w.x;
    vr = ur - tr;
    vi = ui - ti;
    ur = ur + tr;
    ui = ui + ti;
  }
}

// Both kernels load every stage's twiddles (a table read behind another one)
// before the first stage: the stages wait for LDS only.  A launch of one
// plaintext has few workgroups, and the two reads a stage were most of its
// time: 2^15 slots, columns 13.5 -> 11.1 us, blocks 6.8 -> 3.8 us.

// stages len <= FFT_B of one block: 128 threads, a butterfly each per stage
template <bool INV>
__global__ __launch_bounds__(FFT_B / 2) void fft_block_kernel(FftArgs a) {
  constexpr int LB = 8;
  static_assert(FFT_B == 1 << LB, "stages of a block");
  __shared__ double sr[FFT_B], si[FFT_B];
  const int t = threadIdx.x, base = blockIdx.x * FFT_B;
  double* R = a.re + (size_t)blockIdx.y * a.pstride + base;
  double* I = a.im + (size_t)blockIdx.y * a.pstride + base;
  double2 w[LB];
#pragma unroll
  for (int s = 0; s < LB; s++) w[s] = fft_root<INV>(a, 2 << s, t & ((1 << s) - 1));
  for (int k = t; k < FFT_B; k += FFT_B / 2) { sr[k] = R[k]; si[k] = I[k]; }
#pragma unroll
  for (int q = 0; q < LB; q++) {
    const int s = INV ? LB - 1 - q : q, lenh = 1 << s;
    __syncthreads();
    const int j = t & (lenh - 1), k = 2 * (t - j) + j;
    fft_butterfly<INV>(w[s], sr[k], si[k], sr[k + lenh], si[k + lenh]);
  }
  __syncthreads();
  for (int k = t; k < FFT_B; k += FFT_B / 2) { R[k] = sr[k]; I[k] = si[k]; }
}

// stages len > FFT_B: FFT_CW columns of the (n / FFT_B) x FFT_B view, n / FFT_B = 2^LR rows
template <bool INV, int LR>
__global__ __launch_bounds__(256) void fft_col_kernel(FftArgs a) {
  constexpr int rows = 1 << LR, E = rows * FFT_CW, NB = (E / 2 + 255) / 256;  // NB: butterflies a thread and stage
  __shared__ double sr[E], si[E];
  const int col0 = blockIdx.x * FFT_CW;
  double* R = a.re + (size_t)blockIdx.y * a.pstride;
  double* I = a.im + (size_t)blockIdx.y * a.pstride;
  double2 w[LR][NB];
#pragma unroll
  for (int s = 0; s < LR; s++)
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int u = threadIdx.x + 256 * i, c = u % FFT_CW, jr = (u / FFT_CW) & ((1 << s) - 1);
      w[s][i] = fft_root<INV>(a, (2 << s) * FFT_B, jr * FFT_B + col0 + c);
    }
  for (int e = threadIdx.x; e < E; e += 256) {
    const int k = (e / FFT_CW) * FFT_B + col0 + e % FFT_CW;
    double v = 0.0, vi = 0.0;
    if (!INV) {
      v = R[k];
      vi = I[k];
    } else if (k < a.nvals) {
      if (a.complex_in) {
        v = (double)a.data[2 * (size_t)k];
        vi = (double)a.data[2 * (size_t)k + 1];
      } else {
        const EncodeSrc s = a.src ? a.src[blockIdx.y] : EncodeSrc{0, 0};
        v = (double)a.data[(size_t)s.src * a.n + ((k + s.rot) & (a.n - 1))];
      }
    }
    sr[e] = v;
    si[e] = vi;
  }
#pragma unroll
  for (int q = 0; q < LR; q++) {
    const int s = INV ? LR - 1 - q : q, rh = 1 << s;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int u = threadIdx.x + 256 * i;
      if (u < E / 2) {
        const int c = u % FFT_CW, b = u / FFT_CW, jr = b & (rh - 1);
        const int k = (2 * (b - jr) + jr) * FFT_CW + c, k2 = k + rh * FFT_CW;
        fft_butterfly<INV>(w[s][i], sr[k], si[k], sr[k2], si[k2]);
      }
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 256) {
    const int k = (e / FFT_CW) * FFT_B + col0 + e % FFT_CW;
    if (INV) {
      R[k] = sr[e];
      I[k] = si[e];
    } else if (a.mode == 0) {
      ((float*)a.out)[k] = (float)sr[e];
    } else if (a.mode == 1) {
      ((double*)a.out)[k] = sr[e];
    } else {
      ((float*)a.out)[2 * (size_t)k] = (float)sr[e];
      ((float*)a.out)[2 * (size_t)k + 1] = (float)si[e];
    }
  }
}
template <bool INV>
void launch_fft_col(const FftArgs& f, int np, hipStream_t st) {
  const dim3 grid(FFT_B / FFT_CW, np), block(256);
  switch (f.n / FFT_B) {
    case 2: hipLaunchKernelGGL((fft_col_kernel<INV, 1>), grid, block, 0, st, f); break;
    case 4: hipLaunchKernelGGL((fft_col_kernel<INV, 2>), grid, block, 0, st, f); break;
    case 8: hipLaunchKernelGGL((fft_col_kernel<INV, 3>), grid, block, 0, st, f); break;
    case 16: hipLaunchKernelGGL((fft_col_kernel<INV, 4>), grid, block, 0, st, f); break;
    case 32: hipLaunchKernelGGL((fft_col_kernel<INV, 5>), grid, block, 0, st, f); break;
    case 64: hipLaunchKernelGGL((fft_col_kernel<INV, 6>), grid, block, 0, st, f); break;
    default: hipLaunchKernelGGL((fft_col_kernel<INV, 7>), grid, block, 0, st, f); break;
  }
}

// fixed-point record of one coefficient (Lattigo SingleFloat64ToFixedPointCRT)
__device__ __forceinline__ void fixed_point(double value, double scale, u64& mag, u64& meta) {
#pragma clang fp contract(off)
  if (value == 0) { mag = 0; meta = 0; return; }
  u64 neg = 0;
  if (value < 0) { neg = 1; scale *= -1; }
  value *= scale;
  if (value >= 1.8446744073709552e+19) {
    int e;
    const double m = frexp(value, &e);
    mag = (u64)ldexp(m, 53);
    meta = neg | ((u64)(e - 53) << 8);
  } else {
    mag = (u64)(value + 0.5);
    meta = neg;
  }
}

__device__ __forceinline__ int brv_bits(int x, int bits) { return (int)(__brev((unsigned)x) >> (32 - bits)); }

// coefficient x of plaintext p: bit reversal, division by n, fixed point, residues in every row of rm
__global__ void encode_finish_kernel(u64* __restrict__ out, size_t out_pstride, RowMap rm, const double* __restrict__ re,
                                     const double* __restrict__ im, size_t pstride, int n, int logn, double scale,
                                     const ModC* __restrict__ mods, int N) {
#pragma clang fp contract(off)
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= N) return;
  const int p = blockIdx.y;
  const int i = x < n ? x : x - n;
  const int k = brv_bits(i, logn);
  const double v = (x < n ? re : im)[(size_t)p * pstride + k] / (double)n;
  u64 mag, meta;
  fixed_point(v, scale, mag, meta);
  const int neg = (int)(meta & 1), ex = (int)(meta >> 8);
  u64* o = out + (size_t)p * out_pstride;
  for (int a = 0; a < rm.nact(); a++) {
    const int row = rm.row(a);
    const ModC mc = mods[rm.mod(row)];
    u64 r = mont_mul(mag, mc.rmod, mc.q, mc.qinv);  // mag mod q
    for (int e = 0; e < ex; e++) r = add_mod(r, r, mc.q);
    if (neg && r) r = mc.q - r;
    o[(size_t)row * N + x] = r;
  }
}

// The coefficient x of a plaintext at its level: the centred CRT value
//   acc = sum_i y_i * (Q / q_i) - k Q,  y_i = x_i (Q / q_i)^-1 mod q_i,
// k = floor(sum_i y_i / q_i) in float64 (off by at most one, corrected), then
// Q - acc for acc >= floor(Q / 2), the nearest double of it (ties to even) over
// the scale, stored at its bit-reversed place of the FFT.  A workgroup takes 64
// coefficients: each of its four waves sums every fourth source in W words
// (2^(64 W) > 2^8 Q, in registers up to 32 words; W multiply-adds a source over
// wave-uniform table words), the first adds the four sums and finishes.  One
// thread a coefficient leaves a wave a SIMD at N = 2^16, each multiply-add
// waiting for the carry of the one before: 36 us at 23 limbs, 28 this way.
// Decrypt and Decode of 23 limbs there took 7.5 ms with this sum on the host
// (12 MB of residues fetched, 16 threads).
template <int W>
__global__ __launch_bounds__(256) void decode_crt_kernel(DecodeArgs d) {
#pragma clang fp contract(off)
  constexpr int UN = W <= 32 ? W : 1;
  __shared__ u64 part[3][W][64];
  __shared__ double pest[3][64];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = blockIdx.x * 64 + lane;
  const int N = d.N, n = N >> 1;
  u64 a[W];
#pragma unroll UN
  for (int w = 0; w < W; w++) a[w] = 0;
  double est = 0.0;
  u64 next = d.coef[(size_t)min(wv, d.nl - 1) * N + x];
  for (int i = wv; i < d.nl; i += 4) {
    const BConvSrc s = d.src[i];
    const u64 xi = next;
    next = d.coef[(size_t)min(i + 4, d.nl - 1) * N + x];  // in flight while row i is multiplied
    const u64 y = shoup_mul(xi, s.hinv, s.hinvp, s.q);
    est += (double)y / s.qd;
    const u64* h = d.hat + (size_t)i * W;
    u64 c = 0;
#pragma unroll UN
    for (int w = 0; w < W; w++) {
      const u128 t = (u128)h[w] * y + a[w] + c;
      a[w] = (u64)t;
      c = (u64)(t >> 64);
    }
  }
  if (wv) {
#pragma unroll UN
    for (int w = 0; w < W; w++) part[wv - 1][w][lane] = a[w];
    pest[wv - 1][lane] = est;
  }
  __syncthreads();
  if (wv) return;
  for (int p = 0; p < 3; p++) {
    u64 c = 0;
#pragma unroll UN
    for (int w = 0; w < W; w++) {
      const u128 t = (u128)a[w] + part[p][w][lane] + c;
      a[w] = (u64)t;
      c = (u64)(t >> 64);
    }
    est += pest[p][lane];
  }
  const u64* Q = d.hat + (size_t)d.nl * W;
  const u64* Qh = Q + W;
  const u64 k = (u64)est;
  u64 c = 0, br = 0;
#pragma unroll UN
  for (int w = 0; w < W; w++) {
    const u128 t = (u128)Q[w] * k + c;
    c = (u64)(t >> 64);
    const u128 s = (u128)a[w] - (u64)t - br;
    a[w] = (u64)s;
    br = (u64)(s >> 64) & 1;
  }
  // k one too large leaves acc - Q (negative), one too small acc + Q
  const u64 neg = 0 - (a[W - 1] >> 63);
  c = 0; br = 0;
#pragma unroll UN
  for (int w = 0; w < W; w++) {
    const u128 t = (u128)a[w] + (Q[w] & neg) + c;
    a[w] = (u64)t;
    c = (u64)(t >> 64);
    br = (u64)(((u128)a[w] - Q[w] - br) >> 64) & 1;
  }
  const u64 over = br - 1;  // all ones where acc >= Q
  u64 brh = 0;
  br = 0;
#pragma unroll UN
  for (int w = 0; w < W; w++) {
    const u128 t = (u128)a[w] - (Q[w] & over) - br;
    a[w] = (u64)t;
    br = (u64)(t >> 64) & 1;
    brh = (u64)(((u128)a[w] - Qh[w] - brh) >> 64) & 1;
  }
  const bool minus = brh == 0;
  br = 0;
#pragma unroll UN
  for (int w = 0; w < W; w++) {
    const u128 t = (u128)Q[w] - a[w] - br;
    br = (u64)(t >> 64) & 1;
    if (minus) a[w] = (u64)t;
  }
  // the top 64 bits, every bit below them in the last one
  u64 hi = 0, lo = 0, rest = 0;
  int top = -1;
#pragma unroll UN
  for (int w = W - 1; w >= 0; w--) {
    if (top < 0) {
      if (a[w]) { top = w; hi = a[w]; }
    } else if (w == top - 1) {
      lo = a[w];
    } else {
      rest |= a[w];
    }
  }
  double v;
  if (top <= 0) {
    v = (double)hi;
  } else {
    const int lz = __clzll((long long)hi);
    const u64 m = lz ? (hi << lz) | (lo >> (64 - lz)) : hi;
    const u64 low = lz ? lo << lz : lo;
    v = ldexp((double)(m | ((low | rest) ? 1 : 0)), 64 * top - lz);
  }
  if (minus) v = -v;
  v = v / d.scale;
  const int i = x < n ? x : x - n;
  (x < n ? d.re : d.im)[brv_bits(i, d.logn)] = v;
}

}  // namespace

void launch_encode_fft(u64* out, size_t out_pstride, RowMap rm, const float* data, const EncodeSrc* src, int np, int nvals,
                       double scale, double* re, double* im, size_t pstride, const int* rotgroup, const double* rre,
                       const double* rim, const ModC* mods, int logN, hipStream_t st, bool complex_in) {
  const int N = 1 << logN, n = N >> 1, logn = logN - 1;
  const int tpb = 256;
  const FftArgs f{re, im, pstride, n, 2 * N, rotgroup, rre, rim, data, src, nvals, complex_in ? 1 : 0, nullptr, 0};
  launch_fft_col<true>(f, np, st);
  hipLaunchKernelGGL(fft_block_kernel<true>, dim3(n / FFT_B, np), dim3(FFT_B / 2), 0, st, f);
  hipLaunchKernelGGL(encode_finish_kernel, dim3((N + tpb - 1) / tpb, np), dim3(tpb), 0, st, out, out_pstride, rm, re, im,
                     pstride, n, logn, scale, mods, N);
}

void launch_decode_fft(const DecodeArgs& d, int words, const int* rotgroup, const double* rre, const double* rim, void* out,
                       int mode, hipStream_t st) {
  const int n = d.N / 2;
  const dim3 grid(d.N / 64), block(256);
  switch (words) {
    case 4: hipLaunchKernelGGL(decode_crt_kernel<4>, grid, block, 0, st, d); break;
    case 8: hipLaunchKernelGGL(decode_crt_kernel<8>, grid, block, 0, st, d); break;
    case 12: hipLaunchKernelGGL(decode_crt_kernel<12>, grid, block, 0, st, d); break;
    case 16: hipLaunchKernelGGL(decode_crt_kernel<16>, grid, block, 0, st, d); break;
    case 20: hipLaunchKernelGGL(decode_crt_kernel<20>, grid, block, 0, st, d); break;
    case 24: hipLaunchKernelGGL(decode_crt_kernel<24>, grid, block, 0, st, d); break;
    case 28: hipLaunchKernelGGL(decode_crt_kernel<28>, grid, block, 0, st, d); break;
    case 32: hipLaunchKernelGGL(decode_crt_kernel<32>, grid, block, 0, st, d); break;
    default: hipLaunchKernelGGL(decode_crt_kernel<DECODE_MAXW>, grid, block, 0, st, d); break;
  }
  const FftArgs f{d.re, d.im, 0, n, 2 * d.N, rotgroup, rre, rim, nullptr, nullptr, 0, 0, out, mode};
  hipLaunchKernelGGL(fft_block_kernel<false>, dim3(n / FFT_B), dim3(FFT_B / 2), 0, st, f);
  launch_fft_col<false>(f, 1, st);
}
