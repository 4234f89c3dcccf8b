// kernels.h -- launch interface of kernels.hip (internal to the library).
#pragma once
#include "hipckks.h"

// Per-modulus constants of the float64 transform (moduli q <= FP_QMAX,
// fpntt.h); the other moduli leave the entry unused.
struct FpC {
  double q, qinv;  // q and fl(1/q)
  double cneg;     // 2^52 + q (canonical output of a negative residue)
  double ni, niq;  // N^-1 centred, and fl(N^-1 / q)
  double wn, wnq;  // the inverse transform's last twiddle times N^-1, centred, and fl(wn / q)
  double pad;
};
struct NttTables {
  const ModC* mods;
  // [mod][N][2]: (psi^brv(k), Shoup companion) and the same for psi^-1; for
  // a modulus q <= FP_QMAX the pair is (w, fl(w / q)) as float64 bits with
  // w = psi^brv(k) centred in (-q/2, q/2]
  const u64 *tw, *itw;
  const u64 *twr, *itwr;   // [mod][R][slots][P][2]: row-pass consecutive-round twiddles, lane-interleaved
  const u64 *ninv, *ninvp; // [mod]
  const FpC* fpc;          // [mod]
};
// N = R x C, R = 2^SA, C = 2^SB (the transform's column / row split)
void ntt_split(int logN, int* SA, int* SB);
// twiddle slots per lane of the row pass's consecutive round
int ntt_row_round_slots(int logN);

struct BConvSrc {
  u64 q, hinv, hinvp;  // source modulus, (S/s_i)^-1 mod s_i and its Shoup companion
  double qd;           // (double)q
};
struct BConvTable {
  BConvSrc src[HCK_MAXSRC];
  const u64* hat;  // [nmod][ns]   (S/s_i mod t) * R mod t  (Montgomery form)
  const u64* nS;   // [nmod]       (-S mod t) * R mod t
  int rows_per_block;
};

#define HCK_MAXDIG 16
struct KeyMacArgs {
  const u64* digits;       // [dn][nqp][N] (per batch if digits_per_batch)
  size_t dig_bstride;
  int digits_per_batch;
  const u64* const* key;   // per batch: [dnum][2][L+K][N] Montgomery form (nullptr: use key1)
  const uint32_t* const* perm;  // per batch (nullptr: use perm1)
  const u64* key1;         // single-batch key
  const uint32_t* perm1;   // single-batch permutation (nullptr: identity)
  const u64* add0;         // Q rows added to part 0 before the gather (mode 1)
  const u64* add1;         // Q rows added to part 1 the same way (nullptr: none)
  const u64* own;          // the decomposed polynomial (NTT, Q rows; per batch if digits_per_batch): a
  size_t own_bstride;      // digit's own rows are read from it (nullptr: from the digit buffer)
  u64 *out0, *out1;
  size_t out_bstride;
  const ModC* mods;
  int N, l, L, K, nqp, dn;
  // single-batch key generated by this library: its a halves are regenerated
  // from rand64's per-stream key of each digit instead of read
  int seeded;
  u64 ka[HCK_MAXDIG];
};

// One key switch's key product (keymac1_kernel): at most HCK_KM1_DIG digits,
// each with its own unrolled instantiation.  perm gathers every operand and
// so applies the automorphism to the outputs (nullptr: identity).
#define HCK_KM1_DIG 8
struct KeyMac1Args {
  const u64* digits;     // [dn][nqp][N]
  const u64* own;        // the decomposed polynomial (NTT, Q rows)
  const u64* key;        // [dnum][2][L+K][N], Montgomery form
  const uint32_t* perm;
  const u64 *add0, *add1;  // Q rows added to the parts (nullptr: none)
  u64 *out0, *out1;      // [nqp][N] each
  const ModC* mods;
  int N, l, L, K, nqp, dn;
  int seeded;            // the key's a halves are regenerated (ka) instead of read
  u64 ka[HCK_MAXDIG];
  // fold step (c0 set): out0's Q rows are not written; instead
  //   c0_out = c + perm(c) + P^-1 * (part 0),  c = c0 (+ e0)
  const u64 *c0, *e0;
  u64* c0_out;
  const u64 *pinv, *pinvp;
};

// From the product of one key switch to the digits of the next, in the
// coefficient domain (link_kernel): with z the coefficients of the QP
// polynomial x1 (level l) and M = (z - [z]_P) * P^-1 its ModDown,
//   c1 += M, every digit of c1 extended to its other QP rows,
// and from x0p, the P rows of a second QP polynomial, e0 = -[x0p]_P * P^-1 on
// the Q rows.  ginv: 0, or the inverse of the Galois element whose
// automorphism x0p and x1 already carry: ModDown rounds down, so at the
// positions where the automorphism changed the sign it is taken of the
// negated word and the result is negated.
struct LinkArgs {
  const u64* x1;                       // [nqp][N]
  const u64* x0p;                      // [K][N]
  u64* c1;                             // [l+1][N]
  u64* e0;                             // [l+1][N]
  u64* digits;                         // [dn][nqp][N]
  const struct BConvTable* ptab;       // P -> Q
  const struct BConvTable* dtab[HCK_MAXDIG];  // per digit
  const u64 *pinv, *pinvp;
  const ModC* mods;
  int N, l, L, K, nqp, dn;
  uint32_t ginv;
};
// LDS bytes of a link launch, at most LINK_LDS_MAX: its caller's limits, K <= 8
// and dn <= HCK_KM1_DIG, leave up to 64 Q rows, 64 KB
#define LINK_LDS_MAX 65536
size_t link_lds_bytes(int l);
void launch_link(const LinkArgs& a, hipStream_t st);

struct GiantAccArgs {
  const u64* digits;  // [ng][dn][nqp][N]
  size_t dig_bstride;
  const u64* const* key;       // [ng]
  const uint32_t* const* perm; // [ng]
  const int* tg;               // giant-group index into T per key-switched group
  int ng;
  const u64* own;              // [ng][l+1][N] decomposed polynomials (own digit rows), or nullptr
  size_t own_bstride;
  const u64* T;                // [ngroups][2][nqp][N]
  size_t T_gstride, T_pstride;
  int t_zero;                  // index of the rotation-0 group in T, or -1
  u64 *out0, *out1;            // QP accumulators [nqp][N]
  const ModC* mods;
  int N, l, L, K, nqp, dn;
  const u64* ka;               // [ng][dn] per-stream PRNG keys of the keys' a halves (regenerated), or nullptr (read)
};

// Diagonals of a dense 16-baby transform are stored packed: a row whose
// modulus is below 2^52 holds each run of 64 words (one wave's coefficients)
// as 52-bit fields in PK_CHUNK dwords (word j at bits [52 j, 52 j + 52));
// the other rows hold plain 64-bit words.  The row descriptor of row k is
// (dword offset of the row inside a diagonal, 52 or 0); rows and diagonals
// start on 16-byte boundaries.
#define PK_BITS 52
#define PK_CHUNK 104  // 64 * PK_BITS / 32
struct DiagMacArgs {
  const u64* diag;        // [np][lt_level+1+K][N] Montgomery form (packed: see pkrow)
  size_t diag_stride;     // u64 words from one diagonal to the next
  const u64* pc;          // P*c0, P*c1 : [2][l+1][N]
  size_t pc_pstride;
  const int* baby_is_zero;  // [nbaby]
  const int* baby_slot;     // [nbaby]
  const int* gpi;           // [ng][nbaby] plaintext index of baby b in group g (absent: a zero plaintext)
  int dense;                // every group holds every baby: index = g * nbaby + b
  int zero_pidx;            // index of the all-zero plaintext (babies past nbaby in a chunk use it)
  u64* T;                   // [ng][2][nqp][N]
  size_t T_gstride, T_pstride;
  const ModC* mods;
  int N, l, L, K, nqp, lt_level, ng, nbaby, b0, nb_chunk;
  int g0, g1;               // giant groups [g0, g1) of this launch
  // the hoisted baby rotations, computed in the kernel's prologue
  // (keymac_kernel's arithmetic per word)
  const u64* digits;              // [dn][nqp][N] decomposition of c1 (NTT)
  const u64* const* bkey;         // per baby slot: Galois key [dnum][2][L+K][N], Montgomery form
  const uint32_t* const* bperm;   // per baby slot: automorphism gather
  const u64* own;                 // c1 (Q rows, NTT): a digit's own rows
  int dn;
  const u64* bka;                 // [slot][dn] per-stream PRNG keys of the a halves (regenerated), or nullptr (read)
  const uint32_t* pkrow;          // packed layout: [row][2] descriptors, nullptr for plain [np][nqp][N]
  int gper;  // groups of a workgroup (set by the launch)
};

// In-place NTT (forward) / inverse NTT of rows rm of `batch` polynomials.
void launch_ntt(u64* data, size_t bstride, int batch, RowMap rm, int logN, bool forward, const NttTables& tw, hipStream_t st);
// Out-of-place: the transform of src's rows is written to the same rows of dst.
void launch_ntt(const u64* src, size_t sstride, u64* dst, size_t dstride, int batch, RowMap rm, int logN, bool forward,
                const NttTables& tw, hipStream_t st);
// NTT / inverse NTT of an explicit list of limbs: list is a device array of
// nlimbs {int64 word offset from data, int modulus index, int source: the
// limb is read `source` limbs (of N words) past its offset, 0 in place}.
void launch_ntt_list(u64* data, const void* list, int nlimbs, int logN, bool forward, const NttTables& tw, hipStream_t st);
// Forward NTT of the Q rows 0..l of ext (the extension of [x]_P to Q) fused
// with the ModDown combine: out[b][i][perm_inv^-1...] -- for every position p,
// out[b][i][perm_inv[p]] = (x[b][i][p] - NTT(ext)[b][i][p]) * P^-1 (+ add[b][i][p]
// for b < add_batches) (+ acc[b][i][perm_inv[p]] if acc, a buffer other than
// out); batch entries below x_from take x = 0; ext itself is left in an intermediate state.
void launch_ntt_moddown(u64* ext, size_t ext_bstride, int batch, int l, int logN, const u64* x, size_t x_bstride,
                        u64* out, size_t o_bstride, const u64* add, size_t a_bstride, int add_batches,
                        const uint32_t* perm_inv, const u64* pinv, const u64* pinvp, const NttTables& tw, hipStream_t st,
                        const u64* acc = nullptr, size_t c_bstride = 0, int x_from = 0);
// Two scaled rescales of one ciphertext x at level l (l output rows) in one
// forward transform: batch
// entry b = 2 g + p (p the part) ends in
//   out_g[p][i] = (K_g,i * x[p][i] - NTT(t[b])_i) * q_l^-1 (+ C_g,i if p == 0)
// with K and C per group and row in ks: ks[(0 * 2 + g) * l + i] = K_g,i,
// ks[(1 * 2 + g) * l + i] its Shoup companion, ks[(2 * 2 + g) * l + i] = C_g,i
// (rows i < l; every word read in the launch's stream order).
void launch_ntt_rescale_pair(u64* t, size_t t_bstride, int l, int logN, const u64* x, size_t x_bstride, u64* out0,
                             u64* out1, size_t o_bstride, const u64* ks, const u64* rsinv, const u64* rsinvp,
                             const NttTables& tw, hipStream_t st);
// dst[b][0..words) = src[b][0..words) for b < batch.
void launch_copy(u64* dst, size_t dstride, const u64* src, size_t sstride, size_t words, int batch, hipStream_t st);
void launch_add(u64* out, const u64* a, const u64* b, size_t bstride, int batch, RowMap rm, const ModC* mods, int N, bool sub, hipStream_t st);
void launch_mul_const(u64* out, size_t obstride, const u64* in, size_t bstride, int batch, RowMap rm, const u64* cw, const u64* cwp, const ModC* mods, int N, hipStream_t st);
// Packed diagonal storage: dst (packed layout, dst_stride dwords a
// diagonal) <- src (plain [np][nrows][N], src_stride words a diagonal), and
// back for one diagonal (dst plain [nrows][N]).
void launch_pack_diags(uint32_t* dst, size_t dst_stride, const u64* src, size_t src_stride, int np, const uint32_t* rowdesc,
                       int nrows, int N, hipStream_t st);
void launch_unpack_diag(u64* dst, const uint32_t* src, const uint32_t* rowdesc, int nrows, int N, hipStream_t st);
// Tensor product of two ciphertexts at level l (rows 0..l of each part):
// d0 = a0 b0, d1 = a0 b1 + a1 b0, d2 = a1 b1, every output (l + 1) x N words;
// with pw (P mod q and its Shoup companion per modulus) d0 and d1 come out
// multiplied by P, ready to be added to a key switch's QP result ahead of
// its ModDown.
void launch_tensor(u64* d0, u64* d1, u64* d2, const u64* a0, const u64* a1, const u64* b0, const u64* b1, int l,
                   const u64* pw, const u64* pwp, const ModC* mods, int N, hipStream_t st);
// Per-modulus constants passed by value in the kernel arguments (a scalar
// times a ciphertext, a scalar added to it): nothing to upload or to keep
// alive until the launch has run, so the host does not wait for the stream.
struct RowConst { u64 w[HCK_MAXMOD], wp[HCK_MAXMOD]; };
// out = in * c.w[modulus] (Shoup companion c.wp) on the rows of rm, batch entries bstride apart
void launch_mul_const_v(u64* out, const u64* in, size_t bstride, int batch, RowMap rm, const RowConst& c, const ModC* mods,
                        int N, hipStream_t st);
// out = in +- c.w[modulus] on the rows of rm (one polynomial)
void launch_add_scalar_v(u64* out, const u64* in, RowMap rm, const RowConst& c, const ModC* mods, int N, bool sub,
                         hipStream_t st);
void launch_mont_mul(u64* out, size_t obstride, const u64* a, size_t abstride, const u64* bR, size_t bbstride, int batch, RowMap rm, const ModC* mods, int N, const u64* add, hipStream_t st, bool bmod = false);
void launch_mont_convert(u64* data, size_t bstride, int batch, RowMap rm, const ModC* mods, int N, bool to, hipStream_t st);
// Basis extension of the ns source rows of `in` into the target rows rm of `out`.
// One source group of a batched basis extension (e.g. one digit of a
// decomposition): its table (device copy), source rows, destination rows.
struct BConvJob {
  const BConvTable* tab;
  int src_row, ns, force_v0, pad;
  RowMap rm;
  size_t out_off;  // word offset of the group's output inside a batch entry
};
#define HCK_MAXJOBS 16
// ginv: 0, or the inverse of a Galois element whose automorphism the source
// already carries (LinkArgs): at the positions whose sign it changed the
// extension is taken of the negated sources and negated (at most 8 sources a
// job: such a launch takes the shared-source form whatever its size).
struct BConvJobs { BConvJob j[HCK_MAXJOBS]; int n, rows_per_block; uint32_t ginv; };
// Basis extension of every job for every batch entry, in one launch.
void launch_bconv(const u64* in, size_t in_bstride, BConvJobs jobs, u64* out, size_t out_bstride, int batch,
                  const ModC* mods, int N, hipStream_t st);
// Single source group: the sources are rows [0, ns) of in.
void launch_bconv(const u64* in, size_t in_bstride, int ns, const BConvTable* dtab, u64* out, size_t out_bstride, int batch,
                  const RowMap& rm, const ModC* mods, int N, hipStream_t st);
void launch_keymac(const KeyMacArgs& a, int batch, hipStream_t st);
void launch_keymac1(const KeyMac1Args& a, hipStream_t st);
void launch_giant_acc(const GiantAccArgs& a, hipStream_t st);
void launch_diag_mac(const DiagMacArgs& a, hipStream_t st);
void launch_rescale_spread(u64* t, const u64* u, int l, u64 half, const ModC* mods, int N, hipStream_t st);
// The spread of two scaled rescales of one ciphertext (launch_ntt_rescale_pair):
// t[2 g + p][i] = ([K_g,l * u[p] + half]_{q_l} - half) mod q_i for rows i < l,
// u[p] the coefficients of row l of part p.  The launch also writes the
// per-row constants of the transform's epilogue (the ks layout above) to ks.
#define HCK_MAXQ 64
struct RescalePair {
  u64 kl[2], klp[2];                        // K_g mod q_l, Shoup companion
  u64 k[2][HCK_MAXQ], kp[2][HCK_MAXQ], c[2][HCK_MAXQ];  // per row i < l
};
void launch_rescale_pair_spread(u64* t, const u64* u, int l, u64 half, const RescalePair& rp, u64* ks, const ModC* mods,
                                int N, hipStream_t st);
// ModDown + rescale: rows i < l of the coefficient-domain extension ext become
// ext_i + P * t_i, t the rescale's spread of the ModDown result's row l
// ((xl - ext_l) * P^-1 mod q_l); ext and xl have `batch` entries.
void launch_moddown_rescale_spread(u64* ext, size_t e_bstride, const u64* xl, size_t x_bstride, int l, u64 half, u64 pinvl,
                                   u64 pinvlp, const u64* pmod_w, const u64* pmod_wp, const ModC* mods, int N, int batch,
                                   hipStream_t st);
void launch_sample_uniform(u64* out, RowMap rm, u64 seed, u64 stream, const ModC* mods, int N, hipStream_t st);
void launch_sample_cbd(u64* out, RowMap rm, u64 seed, u64 stream, const ModC* mods, int N, hipStream_t st);
void launch_signed_rows(u64* out, RowMap rm, const int8_t* v, const ModC* mods, int N, hipStream_t st);
// positions small enough to travel in the kernel arguments
struct TernaryPos {
  uint32_t p[256];
  __host__ __device__ uint32_t operator[](int i) const { return p[i]; }
};
void launch_ternary_rows(u64* out, RowMap rm, const uint32_t* pos, int npos, const ModC* mods, int N, hipStream_t st);
void launch_ternary_rows(u64* out, RowMap rm, const TernaryPos& pos, int npos, const ModC* mods, int N, hipStream_t st);
// x: [2][l + 2][N] coefficients (rows q_0..q_l, p_0), out: [2][l + 1][N]
struct EncryptDownArgs {
  const u64* x; size_t x_bstride;
  u64* out;
  const ModC* mods;
  const u64 *p0inv, *p0invp;  // [mod] p_0^-1 mod q and its Shoup companion
  u64 seed, stream[2];
  int N, l, mp;               // mp: index of p_0
};
void launch_encrypt_down(const EncryptDownArgs& a, hipStream_t st);
void launch_gk_combine(u64* b, const u64* a, const u64* soR, const u64* sR, int own0, int own1, const u64* pmod, int rows, const ModC* mods, int N, hipStream_t st);
// Device encoder (encoder.hip): plaintext p of a batch takes element k from
// data[src * slots + ((k + rot) mod slots)] (zero past nvals), runs the special
// inverse FFT in float64 (work buffers re/im, pstride words per plaintext),
// rounds to fixed point at `scale` and writes its residues to rows rm of
// out + p * out_pstride (coefficient domain; the caller applies the NTT).
struct EncodeSrc { int src, rot; };
void launch_encode_fft(u64* out, size_t out_pstride, RowMap rm, const float* data, const EncodeSrc* src, int np, int nvals,
                       double scale, double* re, double* im, size_t pstride, const int* rotgroup, const double* rre,
                       const double* rim, const ModC* mods, int logN, hipStream_t st, bool complex_in = false);
// Device decoder: coefficients coef[nl][N] (rows q_0 .. q_{nl-1}), tables of the
// level: src[i] (hinv of Q / q_i), hat [nl][W] words of Q / q_i, then Q and
// floor(Q / 2); W the multiple of 4 up to 32 that is not below `words`, or DECODE_MAXW
// (words of 2^8 Q; decode_words).  re / im are work buffers of N / 2 doubles;
// out takes the slots' real parts as float (mode 0) or double (1), or (re, im)
// pairs of float (2).
#define DECODE_MAXW 96
struct DecodeArgs {
  const u64* coef;
  int nl, N, logn;
  const BConvSrc* src;
  const u64* hat;
  double scale;
  double *re, *im;
};
inline int decode_words(int words) { return words <= 32 ? (words + 3) / 4 * 4 : DECODE_MAXW; }
void launch_decode_fft(const DecodeArgs& d, int words, const int* rotgroup, const double* rre, const double* rim, void* out,
                       int mode, hipStream_t st);
// multiplication by the imaginary unit (the monomial X^(N/2)) in the NTT domain:
// slot x < N/2 times iu[m], slot x >= N/2 times q - iu[m] (Shoup pairs iu / iup, niu / niup)
void launch_mul_i(u64* out, const u64* in, size_t bstride, int batch, RowMap rm, const u64* iu, const u64* iup,
                  const u64* niu, const u64* niup, const ModC* mods, int N, hipStream_t st);
// out[r][x] = sum_{p < npoly} a[p][r][x] * b[p][r][x] mod q_r, rows r < nrows of the modulus table
void launch_mulacc(const u64* a, const u64* b, u64* out, int npoly, int nrows, const ModC* mods, int N, hipStream_t st);
// Integer VALU issue-rate probe: `blocks` workgroups of 256 lanes, each lane
// iters x 8 independent instructions (op 0: v_mad_u64_u32, op 1: v_add3_u32);
// one word per lane written to out.
void launch_valu_probe(int op, u64* out, int blocks, uint32_t seed, int iters, hipStream_t st);
// an empty kernel over `blocks` workgroups (flag != 0x7fffffff: no store)
void launch_empty_probe(u64* out, int blocks, int flag, hipStream_t st);
