// Kernels of the FFT multiply: transform passes, the fused middle pass, the
// rounding/unpack pass and the carry resolve. See fft_device.h for the
// transform structure.
#pragma once
#include <type_traits>

#include "fft_device.h"

namespace bcg {

// One product of a batch.
struct MulDesc {
  const uint32_t *a;
  const uint32_t *b;
  uint32_t *c;
  const uint32_t *d;  // optional addend: c = a*b + d (low cl words)
  unsigned long long al, bl, cl, dl;
  int bits;
  int cbits;
  int gk = 0;  // batched group mode: words per group sum of this product's digits (0: none)
};

struct PassArgs {
  cd *data;                 // complex array of the pass (operand A / product)
  const cd *data_b;         // operand B spectrum array (middle pass)
  const uint32_t *wa;       // digits of A come from these words (pack passes)
  const uint32_t *wb;
  unsigned long long al, bl;
  long long *coef;          // unpack output: 2N rounded coefficients
  unsigned long long N;     // transform length
  unsigned long long M;     // pass column count (stride between rows)
  unsigned long long S;     // pass span L * M
  unsigned long long tw_mul;// 4N / S: converts e^{2 pi i / S} exponents to Omega exponents
  const cd *tl;             // e^{2 pi i t / L}, t < L/2
  Roots roots;
  int bits;                 // digit size
  int ntiles;
  unsigned int *margin;     // float bits of the worst |x - round(x)| (atomic max; zeroed by the packing pass)
  int margin_mask;          // slot (block & mask) * MARGIN_STRIDE; batched: mask + 1 slots per product
  double inv_n;
  int fast_round;           // every coefficient < 2^51: round with the 1.5 * 2^52 addition
  const MulDesc *desc;      // batched launch: product blockIdx.y, else nullptr
  int operand;              // batched first pass: 0 reads desc.a, 1 reads desc.b
  int coef_T;               // last pass: coefficient j at coef[(j % M) * 2L + j / M]
  uint32_t *ybuf;           // last pass, group mode: digits [C g, C g + C) summed into ybuf[g K .. g K + K)
  int ygK;                  // words per group sum (a multiple of 4: 16-byte stores)
  int pair;                 // forward passes of A and B in one launch: grid.y = 1 runs B (data_b, wb, bl)
  int pcount;               // batched forward passes of both operands: grid.y = 2 pcount, rows >= pcount run B
  int lower;                // packing pass of single products: every operand leaves the upper half empty
  unsigned long long ystride;  // batched group mode: group-sum words per product in ybuf
};

// Margin slots: a product spreads its atomics over up to MARGIN_SLOTS
// addresses MARGIN_STRIDE words apart (one 128-byte line each), so that its
// workgroups, which mostly end together, do not serialise on one address: with
// one word per product the atomics of 2048 waves on two products took longer
// than their unpacking pass (37 us against 19 us). The carry takes the
// maximum over the slots (margin_of_slots) to where the host reads it.
constexpr int MARGIN_SLOTS = 64;
constexpr int MARGIN_STRIDE = 32;

// Batched launches (desc != nullptr): product p = blockIdx.y owns the arrays
// data + p*N, data_b + p*N, coef + p*2N and margin_mask + 1 margin slots.
__device__ __forceinline__ void bind_product(PassArgs &a) {
  if (!a.desc) {
    if (a.pair && blockIdx.y == 1) {
      a.data = const_cast<cd *>(a.data_b);
      a.wa = a.wb;
      a.al = a.bl;
    }
    return;
  }
  unsigned long long p = blockIdx.y;
  if (a.pcount) {  // both operands in one launch: the upper half of grid.y runs B into data_b
    const bool opb = p >= (unsigned long long)a.pcount;
    if (opb) {
      p -= (unsigned long long)a.pcount;
      a.data = const_cast<cd *>(a.data_b);
    }
    a.operand = opb ? 1 : 0;
    a.data_b = nullptr;
  }
  const MulDesc &d = a.desc[p];
  a.wa = a.operand ? d.b : d.a;
  a.al = a.operand ? d.bl : d.al;
  a.wb = d.b;
  a.bl = d.bl;
  a.bits = d.bits;
  if (a.data) a.data += p * a.N;
  if (a.data_b) a.data_b += p * a.N;
  if (a.coef) a.coef += p * 2 * a.N;
  if (a.ybuf) a.ybuf += p * a.ystride;
  // both operands' packing rows clear the same slots
  if (a.margin) a.margin += p * (unsigned long long)(a.margin_mask + 1) * MARGIN_STRIDE;
}

// Tile order that keeps adjacent column tiles on one XCD at the same time:
// workgroup b runs on XCD b % 8, so tile = (b % 8) * (ntiles / 8) + b / 8.
__device__ __forceinline__ int tile_of_block(int ntiles) {
  int b = blockIdx.x;
  if (ntiles >= 64 && (ntiles & 7) == 0) return (b & 7) * (ntiles >> 3) + (b >> 3);
  return b;
}

// b-bit digit j of a little-endian word array (0 beyond the last word).
__device__ __forceinline__ double digit_at(const uint32_t *__restrict__ w, unsigned long long wl, unsigned long long j,
                                           int bits) {
  unsigned long long s = j * (unsigned long long)bits;
  unsigned long long wi = s >> 5;
  if (wi >= wl) return 0.0;
  unsigned sh = (unsigned)(s & 31);
  unsigned long long v = w[wi];
  if (wi + 1 < wl) v |= (unsigned long long)w[wi + 1] << 32;
  return (double)((v >> sh) & ((1ull << bits) - 1ull));
}

// Nearest integer of x clamped at 0, and the rounding distance into worst.
// Equals fft/convert.c's (uint64_t)(x + 0.5) whenever |x - round x| < 1/2
// (the multiply re-runs with smaller digits from 1/4 on). fast: |x| < 2^51,
// where adding 1.5 * 2^52 leaves round-to-nearest(x) in the low mantissa bits.
__device__ __forceinline__ long long round_coef(double x, bool fast, double &worst) {
  if (fast) {
    // no clamp at 0: a negative result means an error of at least 1/2 in a
    // non-negative coefficient, outside the regime the margin check trusts
    const double magic = 6755399441055744.0;  // 1.5 * 2^52
    const double y = x + magic;
    worst = fmax(worst, fabs(x - (y - magic)));
    return __double_as_longlong(y) - __double_as_longlong(magic);
  }
  worst = fmax(worst, fabs(x - rint(x)));
  const long long v = (long long)(x + 0.5);
  return v > 0 ? v : 0;
}

// Round one output point j = row * M + col, already multiplied by
// Omega^{-j} (f = w_j Omega^{-j}, unscaled), into coefficients c_j (real part)
// and c_{j+N} (imaginary part); returns the rounding margin. L is the pass
// length of the transposed layout (coef_T only).
__device__ __forceinline__ double round_store(const PassArgs &a, cd f, unsigned long long row,
                                              unsigned long long col, unsigned long long L) {
  double m = 0.0;
  const long long cr = round_coef(f.x * a.inv_n, a.fast_round, m);
  const long long ci = round_coef(f.y * a.inv_n, a.fast_round, m);
  if (a.coef_T) {
    // column-major [col][2L] (real part rows, then imaginary)
    a.coef[col * 2 * L + row] = cr;
    a.coef[col * 2 * L + L + row] = ci;
  } else {
    const unsigned long long j = row * a.M + col;
    a.coef[j] = cr;
    a.coef[j + a.N] = ci;
  }
  return m;
}

// Exact sum of C coefficients v[i] 2^{b i + pos0} (pos0 < 32) as K words
// (K >= the words the sum spans) into out[0..K) (LDS or global). pos0 and b
// are the same across the wave (callers derive them from the tile, never
// from the lane), so the shifts and the word emissions are scalar decisions.
template <int C>
__device__ __forceinline__ void group_sum_words(const unsigned long long (&v)[C], int pos0, int b, int K,
                                                uint32_t *out) {
  // 128-bit accumulator w3:w2:w1:w0; bit 0 is bit 32 k of the sum. Each term
  // v 2^pos (v < 2^51, pos < 32) spans three words and enters through one
  // add-with-carry chain.
  unsigned w0 = 0, w1 = 0, w2 = 0, w3 = 0;
  int pos = pos0, k = 0;
#pragma unroll
  for (int i = 0; i < C; i++) {
    if (pos >= 32) {
      out[k++] = w0;
      w0 = w1;
      w1 = w2;
      w2 = w3;
      w3 = 0;
      pos -= 32;
    }
    const unsigned long long lo = v[i] << pos;
    // v >> (64 - pos), 0 for pos = 0, without a select: (v >> 1) >> (63 - pos)
    const unsigned hi = (unsigned)((unsigned)(v[i] >> 33) >> (31 - pos));
    unsigned c0, c1, c2, c3;
    w0 = __builtin_addc(w0, (unsigned)lo, 0u, &c0);
    w1 = __builtin_addc(w1, (unsigned)(lo >> 32), c0, &c1);
    w2 = __builtin_addc(w2, hi, c1, &c2);
    w3 = __builtin_addc(w3, 0u, c2, &c3);
    pos += b;
  }
  for (; k < K; k++) {
    out[k] = w0;
    w0 = w1;
    w1 = w2;
    w2 = w3;
    w3 = 0;
  }
}

// Bit offset (j0 b) & 31 of a group's first digit j0 = t M + m0 (+ N): the
// same for every row t of a tile, since 32 | M b in the passes that sum groups.
__device__ __forceinline__ int group_pos0(const PassArgs &a, unsigned long long m0, int half) {
  return (int)(((m0 + (half ? a.N : 0ull)) * (unsigned long long)a.bits) & 31ull);
}

// Group sums of the last inverse pass (group mode). After the final stage the
// tile slot (row t, column c) holds the rounded coefficient pair (c_j, c_{j+N})
// of j = t M + m0 + c. For each row, the C real parts (digits j0 + [0, C),
// j0 = t M + m0) and the C imaginary parts (j0 + N + [0, C)) each give one
// exact sum sum_i c_i 2^{b i}, written shifted by (j0 b mod 32) as ygK
// little-endian words (ygK a multiple of 4, zero padded) at ybuf[(j0 / C)
// ygK ...]: the words from word floor(j0 b / 32) up. One thread per row; the
// words are assembled in the row's own LDS slots and leave as 16-byte stores.
template <int L, int C, int T = Tile<L, C>::T>
__device__ __forceinline__ void write_group_sums(const PassArgs &a, cd *lds, unsigned long long m0, int tid) {
  const int b = a.bits;
  const int K = a.ygK;
  for (int t = tid; t < L; t += T) {
    const int s0 = slot<C>(t, 0);  // the row's C slots are contiguous
    unsigned long long re[C], im[C];
#pragma unroll
    for (int i = 0; i < C; i++) {
      const longlong2 v = reinterpret_cast<const longlong2 *>(lds)[s0 + i];
      re[i] = (unsigned long long)v.x;
      im[i] = (unsigned long long)v.y;
    }
    uint32_t *lw = reinterpret_cast<uint32_t *>(lds + s0);
#pragma unroll
    for (int half = 0; half < 2; half++) {
      const unsigned long long j0 = (unsigned long long)t * a.M + m0 + (half ? a.N : 0ull);
      group_sum_words<C>(half ? im : re, group_pos0(a, m0, half), b, K, lw + half * K);
      uint4 *dst = reinterpret_cast<uint4 *>(a.ybuf + (j0 / C) * (unsigned long long)K);
      for (int q = 0; q < K / 4; q++)
        dst[q] = make_uint4(lw[half * K + 4 * q], lw[half * K + 4 * q + 1], lw[half * K + 4 * q + 2],
                            lw[half * K + 4 * q + 3]);
    }
  }
}

// The same for one half (0: real parts, digits j0 + [0, C); 1: imaginary
// parts, j0 + N + [0, C)) from 8-byte coefficient slots.
template <int L, int C>
__device__ __forceinline__ void write_group_half(const PassArgs &a, long long *lc, unsigned long long m0, int tid,
                                                 int half) {
  using TC = Tile<L, C>;
  const int b = a.bits;
  const int K = a.ygK;
  for (int t = tid; t < L; t += TC::T) {
    const int s0 = slot<C>(t, 0);  // the row's C slots are contiguous
    unsigned long long v[C];
#pragma unroll
    for (int i = 0; i < C; i++) v[i] = (unsigned long long)lc[s0 + i];
    uint32_t *lw = reinterpret_cast<uint32_t *>(lc + s0);
    const unsigned long long j0 = (unsigned long long)t * a.M + m0 + (half ? a.N : 0ull);
    group_sum_words<C>(v, group_pos0(a, m0, half), b, K, lw);
    uint4 *dst = reinterpret_cast<uint4 *>(a.ybuf + (j0 / C) * (unsigned long long)K);
    for (int q = 0; q < K / 4; q++) dst[q] = make_uint4(lw[4 * q], lw[4 * q + 1], lw[4 * q + 2], lw[4 * q + 3]);
  }
}

// Wave-level max then one atomic per wave, into slot (blockIdx.x & mask).
__device__ __forceinline__ void margin_reduce(unsigned int *m, double d, int mask = 0) {
  float f = (float)d;
  for (int off = 32; off > 0; off >>= 1) f = fmaxf(f, __shfl_xor(f, off, 64));
  if ((threadIdx.x & 63) == 0) atomicMax(m + (blockIdx.x & mask) * MARGIN_STRIDE, __float_as_uint(f));
}

// The packing pass of a product zeroes its margin slots (the unpacking pass,
// later on the same stream, raises them): a fill kernel of its own is a launch.
__device__ __forceinline__ void margin_clear(const PassArgs &a) {
  if (blockIdx.x != 0) return;
  for (int i = threadIdx.x; i <= a.margin_mask; i += blockDim.x) a.margin[i * MARGIN_STRIDE] = 0u;
}

// First wave: the largest of the mask + 1 slots, on every lane.
__device__ __forceinline__ unsigned margin_of_slots(const unsigned int *m, int mask = MARGIN_SLOTS - 1) {
  unsigned v = m[(threadIdx.x & mask) * MARGIN_STRIDE];  // non-negative floats order like their bit patterns
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

// What the host reads after a call, in host memory the kernels write: the worst
// rounding distance (float bits), whether a carry block's carry-in is still open
// (see k_carry_groups), 1 + the index of the highest nonzero word (see
// k_top_nonzero, k_addsub) and the order of a difference's operands.
struct HostResult {
  unsigned margin;
  unsigned open_carry;
  unsigned long long top;
  unsigned long long exp;      // k_rcp_small: the result's exponent (top: its length, swapped: its sign)
  unsigned swapped;
  unsigned set_margin[64];     // k_margin_out: of a deferral scope's products
  unsigned seq;                // number of the last launch whose results are in (host_done)
};
__device__ __forceinline__ void host_store(unsigned *p, unsigned v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Everything this thread left for the host, and what earlier launches on the
// stream left, is in host memory (host_wait).
__device__ __forceinline__ void host_done(HostResult *h, unsigned seq) {
  __threadfence_system();
  host_store(&h->seq, seq);
}

// ------------------------------------------------------------ forward pass

// Length-L DIF down C adjacent columns of one span; stage 0 loads straight from
// global (or from words when PACK), the rest run in LDS; the store multiplies
// row r (frequency k) by the pass twiddle e^{2 pi i m k / S}.
// Tiles of two radix-16 stages (L = 256): stage 1 runs in registers too, and
// the transpose between the stages goes through LDS one half (real parts,
// then imaginary parts) at a time, so a tile needs half the LDS and twice as
// many waves fit on a CU.
template <int L, int C>
struct SplitTile {
  static constexpr bool ON = Tile<L, C>::NST2 == 2 && Tile<L, C>::FIRSTB == 4;
  static constexpr int BYTES = Tile<L, C>::LDS_ELEMS * (ON ? 8 : 16);
};

// Rows r0 + 16 t (t < 16) of column c in x become rows 16 r0 + t in y, one
// double plane at a time through ld (barrier-separated; ends with a barrier).
template <int C>
__device__ __forceinline__ void split_transpose(double *ld, const cd (&x)[16], cd (&y)[16], int r0, int c,
                                                bool to_blocks) {
#pragma unroll
  for (int plane = 0; plane < 2; plane++) {
#pragma unroll
    for (int t = 0; t < 16; t++) {
      const int row = to_blocks ? r0 + 16 * t : 16 * r0 + t;
      ld[slot<C>(row, c)] = plane ? x[t].y : x[t].x;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 16; t++) {
      const int row = to_blocks ? 16 * r0 + t : r0 + 16 * t;
      if (plane)
        y[t].y = ld[slot<C>(row, c)];
      else
        y[t].x = ld[slot<C>(row, c)];
    }
    __syncthreads();
  }
}

// Buffer resource over `words` 32-bit words at p: loads at byte offsets at or
// beyond 4 * words return 0 (the resource's range check). The record count is
// a 32-bit byte count; larger arrays are only ever read below 2^32 bytes.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t word_rsrc(const uint32_t *p, unsigned long long words) {
  const unsigned bytes = words >= 0x3fffffffull ? 0xfffffffcu : (unsigned)(words * 4ull);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(p), (short)0, (int)bytes, 0x00020000);
}

// Digits of the packing pass, read straight from the operand words. Lane
// (r0, c) takes column m = m0 + c of rows r0 + h L/16 (h < 16) in both halves:
// digit j = row M + m (+ N) starts at bit j b, that is at bit (m b) & 31 of
// word row (M b / 32) + (m b >> 5) (+ N b / 32), as M b and N b are multiples
// of 32. Words at or beyond al read as 0 through the range check. When b does
// not divide 32 a digit may straddle two words; the second comes from a
// resource based one word higher, so every load is one whole dword either in
// or out of range.
struct PackDigits {
  __amdgpu_buffer_rsrc_t w0, w1, u0, u1;
  unsigned off;   // byte offset of the lane's word in row r0
  unsigned step;  // bytes between rows r0 + h L/E and r0 + (h + 1) L/E
  unsigned sh, bits;
  bool upper;     // the upper half (digits N ..) holds words
  bool one;       // b divides 32: a digit never straddles two words

  template <int L, int E = 16>
  __device__ __forceinline__ void init(const PassArgs &a, int r0, unsigned long long m) {
    bits = (unsigned)a.bits;
    const unsigned long long row_w = (a.M * bits) >> 5, half_w = (a.N * bits) >> 5, mb = m * bits;
    const unsigned long long al = a.al;
    w0 = word_rsrc(a.wa, al);
    w1 = word_rsrc(a.wa + 1, al ? al - 1 : 0);
    // an empty upper half gets empty resources: its loads return 0 without a
    // memory access, and both halves' loads issue together
    upper = half_w < al;
    u0 = word_rsrc(upper ? a.wa + half_w : a.wa, upper ? al - half_w : 0);
    u1 = word_rsrc(upper ? a.wa + half_w + 1 : a.wa, upper ? al - half_w - 1 : 0);
    off = (unsigned)(((unsigned long long)r0 * row_w + (mb >> 5)) * 4ull);
    step = (unsigned)(row_w * (unsigned long long)(L / E) * 4ull);
    sh = (unsigned)(mb & 31ull);
    one = (bits & (bits - 1u)) == 0u;  // b <= 32 divides 32
  }

  // Lower-half digits only (launches whose operands all leave the upper half
  // empty).
  template <int E>
  __device__ __forceinline__ void load_lower(unsigned (&d)[E]) const {
    unsigned lo[E];
#pragma unroll
    for (int h = 0; h < E; h++) lo[h] = __builtin_amdgcn_raw_buffer_load_b32(w0, off + (unsigned)h * step, 0, 0);
    if (one) {
#pragma unroll
      for (int h = 0; h < E; h++) d[h] = __builtin_amdgcn_ubfe(lo[h], sh, bits);
    } else {
      unsigned hi[E];
#pragma unroll
      for (int h = 0; h < E; h++) hi[h] = __builtin_amdgcn_raw_buffer_load_b32(w1, off + (unsigned)h * step, 0, 0);
#pragma unroll
      for (int h = 0; h < E; h++) d[h] = __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(hi[h], lo[h], sh), 0, bits);
    }
  }

  // Lower-half digits into d, upper-half digits into e (0 when empty); every
  // load is issued before the first is used.
  template <int E>
  __device__ __forceinline__ void load(unsigned (&d)[E], unsigned (&e)[E]) const {
    unsigned lo[E], ulo[E];
#pragma unroll
    for (int h = 0; h < E; h++) {
      lo[h] = __builtin_amdgcn_raw_buffer_load_b32(w0, off + (unsigned)h * step, 0, 0);
      ulo[h] = __builtin_amdgcn_raw_buffer_load_b32(u0, off + (unsigned)h * step, 0, 0);
    }
    if (one) {
#pragma unroll
      for (int h = 0; h < E; h++) {
        d[h] = __builtin_amdgcn_ubfe(lo[h], sh, bits);
        e[h] = __builtin_amdgcn_ubfe(ulo[h], sh, bits);
      }
    } else {
      unsigned hi[E], uhi[E];
#pragma unroll
      for (int h = 0; h < E; h++) {
        hi[h] = __builtin_amdgcn_raw_buffer_load_b32(w1, off + (unsigned)h * step, 0, 0);
        uhi[h] = __builtin_amdgcn_raw_buffer_load_b32(u1, off + (unsigned)h * step, 0, 0);
      }
#pragma unroll
      for (int h = 0; h < E; h++) {
        d[h] = __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(hi[h], lo[h], sh), 0, bits);
        e[h] = __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(uhi[h], ulo[h], sh), 0, bits);
      }
    }
  }
};

// Streaming loads and stores of the sixteen rows K r0 + S t (t < 16) of column
// m0 + c, rows M points apart, for lane (r0, c) of a C-column tile: one lane
// base address, plus the row step S t M, which is the same across the wave
// (scalar registers), so each access costs one address addition and the
// sixteen accesses hold no per-row address registers.
template <int K, int S, bool PLAIN = false>
__device__ __forceinline__ void load_rows16(const cd *base, cd (&v)[16], int r0, int c, unsigned long long m0,
                                            unsigned long long M) {
  const cd *lb = base + (unsigned long long)(K * r0) * M + m0 + c;
#pragma unroll
  for (int t = 0; t < 16; t++) v[t] = ld_pol<PLAIN>(lb + (unsigned long long)(S * t) * M);
}

template <int K, int S, bool PLAIN = false>
__device__ __forceinline__ void store_rows16(cd *base, const cd (&v)[16], int r0, int c, unsigned long long m0,
                                             unsigned long long M) {
  cd *lb = base + (unsigned long long)(K * r0) * M + m0 + c;
#pragma unroll
  for (int t = 0; t < 16; t++) st_pol<PLAIN>(lb + (unsigned long long)(S * t) * M, v[t]);
}

// LOWER (packing pass): every operand of the launch leaves the upper digit
// half empty, so a_{j+N} = 0 and the weighted point is a_j w exactly. The packing of
// split 8-column tiles is held to the 128 registers of four waves (130 without, no spill).
template <int L, int C, bool PACK, int CACHE = 0, bool LOWER = false>
__global__ __launch_bounds__((Tile<L, C>::T))
__attribute__((amdgpu_waves_per_eu((PACK && !LOWER && C == 8 && SplitTile<L, C>::ON) ? 4 : 1, 8))) void k_fwd(PassArgs a) {
  using TC = Tile<L, C>;
  using ST = SplitTile<L, C>;
  using Walk = std::conditional_t<!PACK && CACHE == 0, Walk16Fine, Walk16>;
  bind_product(a);
  // the split transpose pays off where compute dominates (the packing pass);
  // the strided pass keeps the full tile (measured faster at fewer waves)
  constexpr bool SPLIT = ST::ON && PACK;
  constexpr int TILE_BYTES = SPLIT ? ST::BYTES : Tile<L, C>::LDS_ELEMS * 16;
  __shared__ __align__(16) unsigned char lds_raw[TILE_BYTES];
  cd *lds = reinterpret_cast<cd *>(lds_raw);
  const int tid = threadIdx.x;
  const int tile = tile_of_block(a.ntiles);
  const unsigned long long tpb = a.M / C;
  const unsigned long long ob = (unsigned)tile / (unsigned)tpb;  // tpb < 2^31
  const unsigned long long m0 = ((unsigned)tile % (unsigned)tpb) * (unsigned long long)C;
  cd *base = a.data + ob * a.S;
  constexpr int RB0 = TC::FIRSTB;
  constexpr int R0 = 1 << RB0;
  constexpr int PER0 = TC::EPT / R0;
  constexpr int SUB0 = L / R0;
  // Thread tid owns column c = tid % C and rows r0 + h * L/16, r0 = tid / C,
  // h = 0..15 (T = L*C/16): row r0 + h*L/16 has frequency 16 brev(r0) + brev4(h).
  const int c = tid % C;
  const int r0 = tid / C;
  const unsigned long long m = m0 + c;
  // PACK: digit pairs (a_j, a_{j+N}) of rows r0 + h L/16 and the right-angle
  // weight Omega^{row M + m} = Omega^{r0 M + m} e^{2 pi i h / 64}
  if constexpr (PACK) {
    if (a.margin) margin_clear(a);
  }
  unsigned dre[PACK ? 16 : 1], dim_[PACK ? 16 : 1];
  cd wpack = make_double2(1.0, 0.0);
  cd tb0[4];  // split tile: stage-0 level twiddles, loaded ahead of the digits
  if constexpr (SPLIT) level_bases<4>(a.tl, r0, 1, tb0);
  if constexpr (PACK) {
    PackDigits pd;
    pd.template init<L>(a, r0, m);
    if constexpr (LOWER)
      pd.load_lower(dre);
    else
      pd.load(dre, dim_);
    wpack = omega_direct(a.roots, (unsigned long long)r0 * a.M + m);
  }
  if constexpr (SPLIT) {
    // PER0 = 1, SUB0 = 16: rows r0 + 16 t, then rows 16 r0 + t after the transpose
    cd x[16], y[16];
#pragma unroll
    for (int t = 0; t < 16; t++) {
      if constexpr (PACK && LOWER) {
        const cd w = cmul(wpack, w64(t));
        const double r = (double)dre[t];
        x[t] = make_double2(r * w.x, r * w.y);
      } else if constexpr (PACK) {
        // (a_j + i a_{j+N}) w (a_{j+N} = 0 throughout when the upper half is empty)
        x[t] = cmul(make_double2((double)dre[t], (double)dim_[t]), cmul(wpack, w64(t)));
      } else {
        x[t] = ld_nt(&base[(unsigned long long)(r0 + 16 * t) * a.M + m]);
      }
    }
    const cd t1[3] = {a.tl[r0 + 16], a.tl[r0 + 32], a.tl[r0 + 48]};
    levels4_fine<false>(x, tb0, t1, a.tl[2 * (r0 + 16)]);
    split_transpose<C>(reinterpret_cast<double *>(lds_raw), x, y, r0, c, false);
    dif_levels_q0<4>(y);
    // row 16 r0 + t has frequency 16 brev4(t) + brev4(r0)
    Walk16 w;
    if (a.M > 1) w.template init_shared<C>(a.roots, a.tw_mul * m * brev((unsigned)r0, 4), a.tw_mul * m * 16ull);
    if (a.M > 1) {
#pragma unroll
      for (int t = 0; t < 16; t++) y[t] = cmul(y[t], w.at(t));
    }
    store_rows16<16, 1>(base, y, r0, c, m0, a.M);
    return;
  }
#pragma unroll
  for (int i = 0; i < PER0; i++) {
    int q = r0 + i * (TC::T / C);
    cd x[R0];
#pragma unroll
    for (int t = 0; t < R0; t++) {
      unsigned long long row = (unsigned long long)(q + t * SUB0);
      if constexpr (PACK && LOWER) {
        const int h = i + t * PER0;
        const cd w = cmul(wpack, w64(h));
        x[t] = make_double2((double)dre[h] * w.x, (double)dre[h] * w.y);
      } else if constexpr (PACK) {
        const int h = i + t * PER0;
        x[t] = cmul(make_double2((double)dre[h], (double)dim_[h]), cmul(wpack, w64(h)));
      } else {
        x[t] = ld_pol<(CACHE & 1) != 0>(&base[row * a.M + m]);
      }
    }
    first_stage<L, RB0, false>(x, a.tl, q);
#pragma unroll
    for (int t = 0; t < R0; t++) lds[slot<C>(q + t * SUB0, c)] = x[t];
  }
  __syncthreads();
  forward_rest<L, C>(lds, a.tl, tid);
  // pass twiddle e^{2 pi i m k / S} = Omega^{tw_mul m k}
  Walk w;
  if (a.M > 1) w.template init_shared<C>(a.roots, a.tw_mul * m * 16ull * brev((unsigned)r0, TC::LOG - 4), a.tw_mul * m);
#pragma unroll
  for (int h = 0; h < 16; h++) {
    const int row = r0 + h * (L / 16);
    cd v = lds[slot<C>(row, c)];
    if (a.M > 1) v = cmul(v, w.at(h));
    st_pol<(CACHE & 2) != 0>(&base[(unsigned long long)row * a.M + m], v);
  }
}

// ------------------------------------------------------------ inverse pass

// Mirror of k_fwd: staged load with the conjugate pass twiddle, DIT stages in
// LDS, stage 0 stores straight to global, or rounds to coefficients: MODE 0
// stores points, MODE 1 writes the 2N coefficients, MODE 2 their group sums
// (a.ybuf). The two unpacking modes are separate kernels, so the group mode
// is not held to the registers of the coefficient stores.
// The unpacking pass of a split tile is held to 168 VGPRs (three waves per
// SIMD; measured faster than two waves without the two spilled registers).
template <int L, int C, int MODE, int CACHE = 0>
__global__ __launch_bounds__((Tile<L, C>::T))
__attribute__((amdgpu_waves_per_eu((MODE == 1 && SplitTile<L, C>::ON && C >= 8) ? 3 : 1, 8))) void k_inv(PassArgs a) {
  constexpr bool UNPACK = MODE != 0;
  constexpr bool GROUPS = MODE == 2;
  using TC = Tile<L, C>;
  using ST = SplitTile<L, C>;
  using Walk = std::conditional_t<!UNPACK && CACHE == 0, Walk16Fine, Walk16>;
  bind_product(a);
  __shared__ __align__(16) unsigned char lds_raw[ST::BYTES];
  cd *lds = reinterpret_cast<cd *>(lds_raw);
  const int tid = threadIdx.x;
  const int tile = tile_of_block(a.ntiles);
  const unsigned long long tpb = a.M / C;
  const unsigned long long ob = (unsigned)tile / (unsigned)tpb;  // tpb < 2^31
  const unsigned long long m0 = ((unsigned)tile % (unsigned)tpb) * (unsigned long long)C;
  cd *base = a.data + ob * a.S;
  const int c = tid % C;
  const int r0 = tid / C;
  const unsigned long long m = m0 + c;
  if constexpr (ST::ON) {
    // rows 16 r0 + t (frequency 16 brev4(t) + brev4(r0)) with the conjugate
    // pass twiddle, stage 1 in registers, transpose to rows r0 + 16 t, stage 0
    cd x[16], y[16], tb0[4];
    load_rows16<16, 1, (CACHE & 1) != 0>(base, y, r0, c, m0, a.M);
    Walk w;
    if (a.M > 1) {
      w.template init_shared<C>(a.roots, a.tw_mul * m * brev((unsigned)r0, 4), a.tw_mul * m * 16ull);
#pragma unroll
      for (int t = 0; t < 16; t++) y[t] = cmulc(y[t], w.at(t));
    }
    dit_levels_q0<4>(y);
    // stage-0 level twiddles, loaded while the transpose runs
    level_bases<4>(a.tl, r0, 1, tb0);
    double *ld = reinterpret_cast<double *>(lds_raw);
    split_transpose<C>(ld, y, x, r0, c, true);
    if constexpr (MODE != 1) {  // storing coefficients leaves no registers for them
      const cd t1[3] = {a.tl[r0 + 16], a.tl[r0 + 32], a.tl[r0 + 48]};
      levels4_fine<true>(x, tb0, t1, a.tl[2 * (r0 + 16)]);
    } else {
      dit_levels<4>(x, tb0);
    }
    if constexpr (!UNPACK) {
      store_rows16<1, 16, (CACHE & 2) != 0>(base, x, r0, c, m0, a.M);
    } else {
      double worst = 0.0;
      const cd wun = omega_direct(a.roots, (unsigned long long)r0 * a.M + m);
      if constexpr (GROUPS) {
        // group mode (coefficients below 2^51): the real coefficients, then
        // the imaginary ones, each summed per row from LDS
        long long *lc = reinterpret_cast<long long *>(lds_raw);
        long long ci[16];
#pragma unroll
        for (int t = 0; t < 16; t++) {
          const cd f = cmulc(x[t], cmul(wun, w64(t)));
          lc[slot<C>(r0 + 16 * t, c)] = round_coef(f.x * a.inv_n, true, worst);
          ci[t] = round_coef(f.y * a.inv_n, true, worst);
        }
        __syncthreads();
        write_group_half<L, C>(a, lc, m0, tid, 0);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 16; t++) lc[slot<C>(r0 + 16 * t, c)] = ci[t];
        __syncthreads();
        write_group_half<L, C>(a, lc, m0, tid, 1);
      } else {
#pragma unroll
        for (int t = 0; t < 16; t++)
          worst = fmax(worst, round_store(a, cmulc(x[t], cmul(wun, w64(t))), (unsigned long long)(r0 + 16 * t), m, L));
      }
      margin_reduce(a.margin, worst, a.margin_mask);
    }
    return;
  }
  // all sixteen loads in flight first, then the conjugate pass twiddle
  // (rows r0 + h * L/16 as in k_fwd) on the way into LDS
  cd xs[16];
  load_rows16<1, L / 16, (CACHE & 1) != 0>(base, xs, r0, c, m0, a.M);
  Walk w;
  if (a.M > 1) w.template init_shared<C>(a.roots, a.tw_mul * m * 16ull * brev((unsigned)r0, TC::LOG - 4), a.tw_mul * m);
#pragma unroll
  for (int h = 0; h < 16; h++) {
    const int row = r0 + h * (L / 16);
    lds[slot<C>(row, c)] = (a.M > 1) ? cmulc(xs[h], w.at(h)) : xs[h];
  }
  __syncthreads();
  inverse_front<L, C>(lds, a.tl, tid);
  constexpr int RB0 = TC::FIRSTB;
  constexpr int R0 = 1 << RB0;
  constexpr int PER0 = TC::EPT / R0;
  constexpr int SUB0 = L / R0;
  double worst = 0.0;
  cd wun = make_double2(1.0, 0.0);
  if (UNPACK) wun = omega_direct(a.roots, (unsigned long long)r0 * a.M + m);
  constexpr bool groups = GROUPS;
#pragma unroll
  for (int i = 0; i < PER0; i++) {
    int q = r0 + i * (TC::T / C);
    cd x[R0];
#pragma unroll
    for (int t = 0; t < R0; t++) x[t] = lds[slot<C>(q + t * SUB0, c)];
    first_stage<L, RB0, true>(x, a.tl, q);
#pragma unroll
    for (int t = 0; t < R0; t++) {
      unsigned long long row = (unsigned long long)(q + t * SUB0);
      if constexpr (UNPACK) {
        const int h = i + t * PER0;
        const cd f = cmulc(x[t], cmul(wun, w64(h)));
        if (groups) {
          // in place: this thread alone reads and writes these slots in the final stage
          // group mode implies coefficients below 2^51
          const long long cr = round_coef(f.x * a.inv_n, true, worst);
          const long long ci = round_coef(f.y * a.inv_n, true, worst);
          reinterpret_cast<longlong2 *>(lds)[slot<C>(q + t * SUB0, c)] = make_longlong2(cr, ci);
        } else {
          worst = fmax(worst, round_store(a, f, row, m, L));
        }
      } else {
        st_pol<(CACHE & 2) != 0>(&base[row * a.M + m], x[t]);
      }
    }
  }
  if constexpr (UNPACK) {
    if constexpr (groups) {
      __syncthreads();
      write_group_sums<L, C>(a, lds, m0, tid);
    }
    margin_reduce(a.margin, worst, a.margin_mask);
  }
}

// ------------------------------------- packing and unpacking, few tiles
//
// The packing pass of k_fwd and the unpacking pass of k_inv with eight columns and
// eight points per thread on the row stages, a column's L points in LDS of its
// own: the same tiles in twice the waves. For launches that leave SIMDs idle, which
// are bound by a workgroup's chain of loads and instructions (see launch_impl.h);
// where the waves are enough, sixteen points per thread spend fewer instructions on
// twiddles.
template <int L>
struct Strip {
  using RC = Row<L, 8>;
  static constexpr int C = 8;
  // neighbouring columns' points half the banks apart, neighbouring rows one after
  // the other: eight rows of eight columns, a wave, meet each bank equally often
  static constexpr int COL = RC::LDS_ELEMS + (24 - RC::LDS_ELEMS % 16) % 16;
  static_assert(COL * C >= L * C + L * C / 16, "the coefficients of the tile fit");
};

// Walk16Fine for the eight rows 8 r0 + t: Omega^{u0 + brev3(t) du}. With it and stages
// without twiddle products the rounding distances of 300007 by 41003 words are 0.996 of
// those of the sixteen-point kernels (root mean square), 1.039 with Walk16's products;
// 53.5 -> 53.7 us.
struct Walk8 {
  Roots r;
  unsigned long long u0, du;
  cd g2, g4, g6, p;
  template <int C>
  __device__ __forceinline__ void init_shared(const Roots &roots, unsigned long long u, unsigned long long d) {
    static_assert(4 * C <= 64, "four lanes of a wave share a column");
    r = roots;
    u0 = u;
    du = d;
    const int lane = threadIdx.x & 63;
    const int src0 = (lane % C) + (lane / (4 * C)) * (4 * C);
    const cd mine = omega_direct(roots, d * (2 * ((lane / C) & 3)));
    g2 = make_double2(__shfl(mine.x, src0 + C, 64), __shfl(mine.y, src0 + C, 64));
    g4 = make_double2(__shfl(mine.x, src0 + 2 * C, 64), __shfl(mine.y, src0 + 2 * C, 64));
    g6 = make_double2(__shfl(mine.x, src0 + 3 * C, 64), __shfl(mine.y, src0 + 3 * C, 64));
  }
  // i = 0..7 in increasing order; brev3(i): 0 4 2 6 1 5 3 7
  __device__ __forceinline__ cd at(int i) {
    if ((i & 3) == 0) p = omega_direct(r, u0 + (i >> 2) * du);
    switch (i & 3) {
      case 1: return cmul(p, g4);
      case 2: return cmul(p, g2);
      case 3: return cmul(p, g6);
      default: return p;
    }
  }
};

template <int L, bool LOWER>
__global__ __launch_bounds__(L) void k_fwd8(PassArgs a) {
  using SC = Strip<L>;
  constexpr int C = SC::C, E = 8, LOG = SC::RC::LOG;
  bind_product(a);
  __shared__ cd lds[SC::COL * C];
  const int tid = threadIdx.x;
  const int tile = tile_of_block(a.ntiles);
  const unsigned long long tpb = a.M / C;
  const unsigned long long ob = (unsigned)tile / (unsigned)tpb;  // tpb < 2^31
  const int c = tid % C, r0 = tid / C;
  const unsigned long long m = ((unsigned)tile % (unsigned)tpb) * (unsigned long long)C + c;
  cd *base = a.data + ob * a.S + m;
  cd x[E], y[E];
  if (a.margin) margin_clear(a);
  unsigned dre[E], dim_[E];
  PackDigits pd;
  pd.template init<L, E>(a, r0, m);
  if constexpr (LOWER)
    pd.load_lower(dre);
  else
    pd.load(dre, dim_);
  // right-angle weight of row r0 + h L/8: Omega^{r0 M + m} e^{2 pi i h / 32}
  const cd wpack = omega_direct(a.roots, (unsigned long long)r0 * a.M + m);
#pragma unroll
  for (int h = 0; h < E; h++) {
    const cd w = cmul(wpack, w64(2 * h));
    if constexpr (LOWER)
      x[h] = make_double2((double)dre[h] * w.x, (double)dre[h] * w.y);
    else
      x[h] = cmul(make_double2((double)dre[h], (double)dim_[h]), w);
  }
  row_forward<L, E, true>(x, y, lds + c * SC::COL, a.tl, r0);
  // row 8 r0 + t has frequency (L / 8) brev3(t) + brev(r0)
  Walk8 w;
  w.template init_shared<C>(a.roots, a.tw_mul * m * brev((unsigned)r0, LOG - 3), a.tw_mul * m * (L / E));
#pragma unroll
  for (int t = 0; t < E; t++) st_pol<false>(&base[(unsigned long long)(E * r0 + t) * a.M], cmul(y[t], w.at(t)));
}

// GROUPS: group sums (k_inv's MODE 2), else coefficients.
template <int L, bool GROUPS>
__global__ __launch_bounds__(L) void k_inv8(PassArgs a) {
  using SC = Strip<L>;
  constexpr int C = SC::C, E = 8, LOG = SC::RC::LOG;
  bind_product(a);
  __shared__ cd lds[SC::COL * C];
  const int tid = threadIdx.x;
  const int tile = tile_of_block(a.ntiles);
  const unsigned long long tpb = a.M / C;
  const unsigned long long ob = (unsigned)tile / (unsigned)tpb;  // tpb < 2^31
  const unsigned long long m0 = ((unsigned)tile % (unsigned)tpb) * (unsigned long long)C;
  const int c = tid % C, r0 = tid / C;
  const unsigned long long m = m0 + c;
  cd *base = a.data + ob * a.S + m;
  cd x[E], y[E];
#pragma unroll
  for (int t = 0; t < E; t++) y[t] = ld_nt(&base[(unsigned long long)(E * r0 + t) * a.M]);
  Walk8 w;
  w.template init_shared<C>(a.roots, a.tw_mul * m * brev((unsigned)r0, LOG - 3), a.tw_mul * m * (L / E));
#pragma unroll
  for (int t = 0; t < E; t++) y[t] = cmulc(y[t], w.at(t));
  row_inverse<L, E, true>(y, x, lds + c * SC::COL, a.tl, r0);
  double worst = 0.0;
  const cd wun = omega_direct(a.roots, (unsigned long long)r0 * a.M + m);
  if constexpr (GROUPS) __syncthreads();  // the points are read: the tile takes the coefficients
#pragma unroll
  for (int h = 0; h < E; h++) {
    const int row = r0 + h * (L / E);
    const cd f = cmulc(x[h], cmul(wun, w64(2 * h)));
    if constexpr (GROUPS) {
      // group mode implies coefficients below 2^51
      const long long cr = round_coef(f.x * a.inv_n, true, worst);
      const long long ci = round_coef(f.y * a.inv_n, true, worst);
      reinterpret_cast<longlong2 *>(lds)[slot<C>(row, c)] = make_longlong2(cr, ci);
    } else {
      worst = fmax(worst, round_store(a, f, (unsigned long long)row, m, L));
    }
  }
  if constexpr (GROUPS) {
    __syncthreads();
    write_group_sums<L, C, L>(a, lds, m0, tid);
  }
  margin_reduce(a.margin, worst, a.margin_mask);
}

// ------------------------------------------------------------- middle pass

// Points per thread of a middle pass: a block of a power of two shares its CU
// with enough others for sixteen to pay (2^26 points in blocks of 1024, whole
// product: 2.50 ms against 2.54 ms with eight; equal below 2^23 points).
constexpr int mid_points(int L) { return L % 3 != 0 && L >= 256 ? 16 : 8; }

// Middle pass of a multi-pass plan (in place into a.data): last forward pass of
// A (and B), pointwise product (or square), first inverse pass of one contiguous
// block of L points (see Row). BPW blocks per workgroup, each with its own LDS
// tile: short blocks have fewer threads than a wave, or a part of one left over.
// With eight points a thread B's are loaded together with A's, so they arrive
// under A's stages (not with 1024 threads, whose 128 registers would spill).
// Bound by HBM where many blocks are in flight (5.4 TB/s at 2^26 points); 6144
// points on 64 workgroups 33 -> 22 us against 24 points a thread.
template <int L, bool SQUARE, int BPW = 1, int CACHE = 0>
__global__ __launch_bounds__((Row<L, mid_points(L)>::T * BPW)) void k_mid(PassArgs a) {
  constexpr int E = mid_points(L);
  using RC = Row<L, E>;
  bind_product(a);
  __shared__ cd lds_all[RC::LDS_ELEMS * BPW];
  const int sub = BPW > 1 ? (int)threadIdx.x / RC::T : 0;
  const int tid = BPW > 1 ? (int)threadIdx.x % RC::T : (int)threadIdx.x;
  cd *lds = lds_all + sub * RC::LDS_ELEMS;
  const unsigned long long j0 = ((unsigned long long)blockIdx.x * BPW + sub) * L + tid;
  cd x[E], xa[RC::XR];
#pragma unroll
  for (int h = 0; h < E; h++) x[h] = ld_pol<(CACHE & 1) != 0>(&a.data[j0 + h * RC::T]);
  if constexpr (!SQUARE) {
    cd y[E], xb[RC::XR];
    constexpr bool EARLY = E == 8 && RC::T * BPW < 1024;
    auto load_b = [&] {
#pragma unroll
      for (int h = 0; h < E; h++) y[h] = ld_pol<(CACHE & 1) != 0>(&a.data_b[j0 + h * RC::T]);
    };
    if constexpr (EARLY) load_b();
    row_forward<L, E>(x, xa, lds, a.tl, tid);
    if constexpr (!EARLY) load_b();
    __syncthreads();
    row_forward<L, E>(y, xb, lds, a.tl, tid);
#pragma unroll
    for (int i = 0; i < RC::XR; i++) xa[i] = cmul(xa[i], xb[i]);
  } else {
    row_forward<L, E>(x, xa, lds, a.tl, tid);
#pragma unroll
    for (int i = 0; i < RC::XR; i++) xa[i] = cmul(xa[i], xa[i]);
  }
  row_inverse<L, E>(xa, x, lds, a.tl, tid);
#pragma unroll
  for (int h = 0; h < E; h++) st_pol<(CACHE & 2) != 0>(&a.data[j0 + h * RC::T], x[h]);
}

// Innermost pass of a transform that stands alone: one contiguous block of L points
// in place, forward or inverse, BPW blocks per workgroup as in k_mid. The
// innermost stage holds neighbouring points per thread, so global memory is reached
// through one more turn in LDS, at points tid + h T. Bound by the chain of one
// workgroup where each CU has one: 256 blocks of 4096 points 13 us (14 us with sixteen
// points a thread; 6.5 us at the rate of a copy). Powers of two take no twiddle that is a
// product: root mean square error against 80-bit sums at 4096 points 2.33e-16 of the
// spectrum's, 2.58e-16 with products (2.54e-16 with sixteen points a thread), in the same
// time. Lengths 3 * 2^k gain nothing so.
template <int L, bool INV, int BPW = 1>
__global__ __launch_bounds__((Row<L, 8>::T * BPW)) void k_row(PassArgs a) {
  constexpr int E = 8;
  using RC = Row<L, E>;
  __shared__ cd lds_all[RC::LDS_ELEMS * BPW];
  const int sub = BPW > 1 ? (int)threadIdx.x / RC::T : 0;
  const int tid = BPW > 1 ? (int)threadIdx.x % RC::T : (int)threadIdx.x;
  cd *lds = lds_all + sub * RC::LDS_ELEMS;
  cd *base = a.data + ((unsigned long long)blockIdx.x * BPW + sub) * L + tid;
  cd x[E], xr[RC::XR];
#pragma unroll
  for (int h = 0; h < E; h++) x[h] = ld_nt(&base[h * RC::T]);
  if constexpr (INV) {
#pragma unroll
    for (int h = 0; h < E; h++) lds[RC::template slot<RC::T>(tid, h)] = x[h];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RC::XR; i++) xr[i] = row_has<L, E>(tid, i) ? lds[row_at<L, E>(tid, i)] : make_double2(0.0, 0.0);
    row_inverse<L, E, !RC::THREE>(xr, x, lds, a.tl, tid);
  } else {
    row_forward<L, E, !RC::THREE>(x, xr, lds, a.tl, tid);
#pragma unroll
    for (int i = 0; i < RC::XR; i++)
      if (row_has<L, E>(tid, i)) lds[row_at<L, E>(tid, i)] = xr[i];
    __syncthreads();
#pragma unroll
    for (int h = 0; h < E; h++) x[h] = lds[RC::template slot<RC::T>(tid, h)];
  }
#pragma unroll
  for (int h = 0; h < E; h++) base[h * RC::T] = x[h];
}

// ------------------------------------------------------------ carry resolve

// Carry functions of single-bit carry chains: bit0 = carry out for carry in 0,
// bit1 = carry out for carry in 1. compose(f, g) applies f first, then g.
__device__ __forceinline__ unsigned carry_compose(unsigned f, unsigned g) {
  unsigned h0 = (f & 1u) ? (g >> 1) & 1u : g & 1u;
  unsigned h1 = (f & 2u) ? (g >> 1) & 1u : g & 1u;
  return h0 | (h1 << 1);
}


// Product words from rounded coefficients: value = sum_j c_j 2^{b j}.
// Word w collects P_w = sum_j piece(c_j 2^{bj}, word w) (< 2^37); then
// v_w = lo32(P_w) + hi(P_{w-1}) and a carry chain of single bits resolves v.
// Each thread owns CWPT consecutive words; a block owns CWPT * CT words.
constexpr int CWPT = 4;
constexpr int CT = 256;

struct CarryArgs {
  const MulDesc *desc;       // batched: product blockIdx.y, else nullptr
  unsigned long long coef_stride;  // batched: coefficients per product (2N)
  const long long *coef;
  unsigned long long ncoef;
  int bits;
  int cbits;                 // every coefficient < 2^cbits (cbits <= 63)
  uint32_t *out;
  unsigned long long CL;
  unsigned char *blk_fn;     // per block: bit0 = carry out if carry in 0, bit1 = if carry in 1
  unsigned long long nblk;
  const uint32_t *add;       // optional addend words (value += add), addl words
  unsigned long long addl;
  int coef_T;                // coefficient j at coef[(j % cM) * crows + j / cM]
  unsigned cM, crows;
  unsigned lds_slots;        // int64 slots of dynamic LDS per block (coefficient window)
  const uint32_t *ybuf;      // group mode: group sums instead of coefficients (ncoef digits in all)
  int gC, gK, gKs;           // digits per group, words per group sum, group stride (words)
  long long ng;              // groups: ncoef / gC
  unsigned wpb;              // words per carry block
  unsigned long long ystride;  // batched group mode: group-sum words per product
  HostResult *host;            // nullptr, or where block 0 leaves the margin and open blocks their flag
  const unsigned int *margin;  // margin slots of the product (with host or margin_out)
  int margin_mask;             // one less than their number
  unsigned int *margin_out;    // batched: product p's margin goes to margin_out[p]
};

__device__ __forceinline__ long long coef_at(const CarryArgs &a, long long j) {
  if (!a.coef_T) return a.coef[j];
  unsigned jj = (unsigned)j;
  return a.coef[(unsigned long long)(jj % a.cM) * a.crows + jj / a.cM];
}

__device__ __forceinline__ void word_partials(const CarryArgs &a, long long wfirst, unsigned long long (&P)[CWPT + 1]) {
  // words wfirst-1 .. wfirst+CWPT-1 -> P[0..CWPT]
#pragma unroll
  for (int k = 0; k <= CWPT; k++) P[k] = 0;
  long long lo_bit = 32 * (wfirst - 1) - a.cbits + 1;
  long long jlo = lo_bit <= 0 ? 0 : (lo_bit + a.bits - 1) / a.bits;
  long long hi_bit = 32 * (wfirst + CWPT) - 1;
  long long jhi = hi_bit / a.bits;
  if (jhi >= (long long)a.ncoef) jhi = (long long)a.ncoef - 1;
  for (long long j = jlo; j <= jhi; j++) {
    unsigned long long c = (unsigned long long)coef_at(a, j);
    if (!c) continue;
    long long shift = (long long)a.bits * j - 32 * (wfirst - 1);
#pragma unroll
    for (int k = 0; k <= CWPT; k++) {
      long long sh = shift - 32 * k;
      unsigned long long piece;
      if (sh >= 0)
        piece = sh < 32 ? (unsigned long long)(uint32_t)(c << sh) : 0ull;
      else
        piece = -sh < 64 ? (unsigned long long)(uint32_t)(c >> (-sh)) : 0ull;
      P[k] += piece;
    }
  }
  if (a.add) {
#pragma unroll
    for (int k = 0; k <= CWPT; k++) {
      long long w = wfirst - 1 + k;
      if (w >= 0 && w < (long long)a.addl) P[k] += a.add[w];
    }
  }
}

// Batched carries: product p's coefficients at coef + p * coef_stride, its
// block functions at blk_fn + p * nblk, its words and sizes from desc[p].
__device__ __forceinline__ void bind_carry(CarryArgs &a, unsigned long long p) {
  if (!a.desc) return;
  const MulDesc &d = a.desc[p];
  if (a.coef) a.coef += p * a.coef_stride;
  if (a.ybuf) {
    a.ybuf += p * a.ystride;
    a.gK = d.gk;
  }
  a.bits = d.bits;
  a.cbits = d.cbits;
  a.out = d.c;
  a.CL = d.cl;
  a.add = d.d;
  a.addl = d.dl;
  if (a.margin) a.margin += p * (unsigned long long)(a.margin_mask + 1) * MARGIN_STRIDE;
  if (a.margin_out) a.margin_out += p;
  a.blk_fn += p * a.nblk;
  a.nblk = (d.cl + a.wpb - 1) / a.wpb;
}

// Coefficient window of one carry block in LDS: words [W0 - 2, W0 + CT*CWPT) need
// coefficients j with b j in (32 (W0-2) - cbits, 32 (W0 + CT*CWPT)); the
// window is sized per launch (dynamic LDS) from the smallest digit size.
// 0 (no staging: coefficients are read from global memory) when the window
// would exceed CARRY_LDS_MAX slots (digit sizes below 4 bits).
constexpr unsigned CARRY_LDS_MAX = 8256;
__host__ __device__ inline unsigned carry_slots(int bits, int cbits) {
  unsigned n = (unsigned)((32ull * CT * CWPT + (unsigned long long)cbits + 96) / (unsigned long long)bits + 4);
  return n <= CARRY_LDS_MAX ? n : 0u;
}

// floor(x / b) for 0 <= x < 2^40 through a double reciprocal plus one fix-up.
__device__ __forceinline__ long long div_small(long long x, int b, double inv_b) {
  long long q = (long long)((double)x * inv_b);
  if ((q + 1) * b <= x) q++;
  if (q * b > x) q--;
  return q;
}

constexpr int CARRY_GCOV = 4;  // most group sums covering one word

// x / b for 0 <= x < 2^24 and 1 <= b <= 64 through the float reciprocal,
// corrected to the exact floor.
__device__ __forceinline__ int fdiv_small(int x, int b, float inv_b) {
  int q = (int)((float)x * inv_b);
  if (q * b > x) q--;
  else if ((q + 1) * b <= x) q++;
  return q;
}

// P_w of a block word from the staged window win[0..cnt) (coefficient jbase +
// i at win[i]) in block-relative 32-bit arithmetic: x = 32 (w - W0) + D is the
// word's lowest bit above bit b jbase (D = 32 W0 - b jbase, small), so every
// numerator stays far below 2^24 and the float-reciprocal division is exact.
__device__ __forceinline__ unsigned long long partial_rel(const long long *win, int cnt, int bits, int cbits,
                                                          float inv_b, int x) {
  const int lo = x - cbits + 1;
  const int ilo = lo <= 0 ? 0 : fdiv_small(lo + bits - 1, bits, inv_b);
  int ihi = x + 31 < 0 ? -1 : fdiv_small(x + 31, bits, inv_b);
  if (ihi >= cnt) ihi = cnt - 1;
  unsigned long long P = 0;
  int sh = bits * ilo - x;  // in (-cbits, 32)
  for (int i = ilo; i <= ihi; i++, sh += bits) {
    const unsigned long long c = (unsigned long long)win[i];
    P += (unsigned long long)(uint32_t)(sh >= 0 ? c << sh : c >> -sh);
  }
  return P;
}

// The carry into a block of words: v_w = lo(P_w) + hi(P_{w-1}) < 2^33 carries
// v >> 32 out of word w = W0 - 1 whatever comes into it, unless its low word is
// all ones (a chance of 2^-32 for ordinary digits): then the carry-in is open, the
// block is written as for 0 and marked (bit 2 of its function) for
// k_carry_ripple. So almost every block finishes by itself, from two words of its
// predecessor's range; scanning all blocks' functions in a second kernel and
// incrementing in a third cost 6 to 10 us per product.
struct BlockCarry {
  unsigned cin;   // carry into the block's first word (0 when open)
  unsigned open;
};
__device__ __forceinline__ BlockCarry block_carry(unsigned long long Pm1, unsigned long long Pm2) {
  const unsigned long long v = (Pm1 & 0xffffffffull) + (Pm2 >> 32);
  BlockCarry c;
  c.open = (unsigned)v == 0xffffffffu ? 1u : 0u;
  c.cin = (unsigned)(v >> 32);
  return c;
}

// A block's function and mark, and the host's flag when its carry-in is open.
__device__ __forceinline__ void carry_publish(const CarryArgs &a, unsigned fn, const BlockCarry &c) {
  a.blk_fn[blockIdx.x] = (unsigned char)(fn | (c.open << 2));
  if (c.open && a.host) host_store(&a.host->open_carry, 1u);
}

// First wave of a product's block 0: its margin to where the host reads it.
__device__ __forceinline__ void carry_margin(const CarryArgs &a) {
  if (!a.host && !a.margin_out) return;
  const unsigned m = margin_of_slots(a.margin, a.margin_mask);
  if (threadIdx.x != 0) return;
  if (a.host) host_store(&a.host->margin, m);
  else *a.margin_out = m;
}

// Words of one block from coefficients: P_w (< 2^37) per word, v_w = lo(P_w) +
// hi(P_{w-1}), a wave-shuffle scan of per-thread carry functions, words
// written for the block's carry-in, its function and mark saved for k_carry_ripple.
// The coefficient window is staged into LDS with eight loads in flight per
// thread; each thread's word w-1 partial comes from its left neighbour.
static __global__ __launch_bounds__(CT) void k_carry_local(CarryArgs a) {
  extern __shared__ long long cl[];
  __shared__ unsigned wave_fn[CT / 64];
  __shared__ BlockCarry bc;
  const int tid = threadIdx.x;
  bind_carry(a, blockIdx.y);
  if (blockIdx.x >= a.nblk) return;
  const long long W0 = (long long)blockIdx.x * CT * CWPT;
  const long long wfirst = W0 + (long long)tid * CWPT;
  const double inv_b = 1.0 / (double)a.bits;
  long long lo_bit = 32 * (W0 - 2) - a.cbits + 1;
  long long jbase = lo_bit <= 0 ? 0 : div_small(lo_bit + a.bits - 1, a.bits, inv_b);
  long long jend = div_small(32 * (W0 + (long long)CT * CWPT) - 1, a.bits, inv_b);  // inclusive
  if (jend >= (long long)a.ncoef) jend = (long long)a.ncoef - 1;
  const long long cnt = jend >= jbase ? jend - jbase + 1 : 0;
  const bool staged = cnt <= (long long)a.lds_slots;
  if (staged) {
    for (long long t0 = 0; t0 < cnt; t0 += 8 * CT) {
      long long r[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const long long t = t0 + u * CT + tid;
        r[u] = t < cnt ? coef_at(a, jbase + t) : 0;
      }
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const long long t = t0 + u * CT + tid;
        if (t < cnt) cl[t] = r[u];
      }
    }
  }
  __syncthreads();
  unsigned long long P[CWPT + 1], Pm2 = 0;  // Pm2: word W0 - 2 (thread 0)
  if (staged) {
    const int lane = tid & 63;
    const int D = (int)(32 * W0 - (long long)a.bits * jbase);
    const float inv_bf = 1.0f / (float)a.bits;
    const int cnti = (int)cnt, x0 = 32 * tid * CWPT + D;  // lowest bit of word wfirst
#pragma unroll
    for (int k = 1; k <= CWPT; k++) {
      long long w = wfirst - 1 + k;
      P[k] = (w < (long long)a.CL) ? partial_rel(cl, cnti, a.bits, a.cbits, inv_bf, x0 + 32 * (k - 1)) : 0ull;
    }
    // word wfirst-1 is the left neighbour's last word
    unsigned long long left = __shfl_up(P[CWPT], 1, 64);
    if (lane == 0)
      left = (wfirst >= 1 && wfirst - 1 < (long long)a.CL) ? partial_rel(cl, cnti, a.bits, a.cbits, inv_bf, x0 - 32)
                                                          : 0ull;
    P[0] = left;
    if (tid == 0 && W0) Pm2 = partial_rel(cl, cnti, a.bits, a.cbits, inv_bf, x0 - 64);
    if (a.add) {
#pragma unroll
      for (int k = 0; k <= CWPT; k++) {
        long long w = wfirst - 1 + k;
        if (w >= 0 && w < (long long)a.addl && w < (long long)a.CL) P[k] += a.add[w];
      }
      if (tid == 0 && W0 && W0 - 2 < (long long)a.addl) Pm2 += a.add[W0 - 2];
    }
  } else {
    if (tid == 0 && W0) {
      word_partials(a, W0 - 1, P);
      Pm2 = P[0];
    }
    if (wfirst < (long long)a.CL)
      word_partials(a, wfirst, P);
    else
      for (int k = 0; k <= CWPT; k++) P[k] = 0;
  }
  if (wfirst == 0) P[0] = 0;
  if (tid == 0) bc = block_carry(P[0], Pm2);
  unsigned long long v[CWPT];
#pragma unroll
  for (int k = 0; k < CWPT; k++) v[k] = (P[k + 1] & 0xffffffffull) + (P[k] >> 32);
  unsigned f0 = 0, f1 = 1;
#pragma unroll
  for (int k = 0; k < CWPT; k++) {
    f0 = (unsigned)((v[k] + f0) >> 32);
    f1 = (unsigned)((v[k] + f1) >> 32);
  }
  const unsigned f = f0 | (f1 << 1);
  // inclusive scan of carry functions within the wave, then across waves
  const int lane = tid & 63, wave = tid >> 6;
  unsigned inc = f;
  for (int off = 1; off < 64; off <<= 1) {
    unsigned gq = __shfl_up(inc, off, 64);
    if (lane >= off) inc = carry_compose(gq, inc);
  }
  unsigned excl = __shfl_up(inc, 1, 64);
  if (lane == 0) excl = 2u;
  if (lane == 63) wave_fn[wave] = inc;
  __syncthreads();
  unsigned pre = 2u;
  for (int w = 0; w < wave; w++) pre = carry_compose(pre, wave_fn[w]);
  if (tid == 0) {
    unsigned tot = 2u;
    for (int w = 0; w < CT / 64; w++) tot = carry_compose(tot, wave_fn[w]);
    carry_publish(a, tot, bc);
  }
  if (blockIdx.x == 0 && tid < 64) carry_margin(a);
  unsigned cin = (carry_compose(pre, excl) >> bc.cin) & 1u;
  uint32_t o[CWPT];
#pragma unroll
  for (int k = 0; k < CWPT; k++) {
    unsigned long long sum = v[k] + cin;
    o[k] = (uint32_t)sum;
    cin = (unsigned)(sum >> 32);
  }
  if (wfirst + CWPT <= (long long)a.CL && ((reinterpret_cast<uintptr_t>(a.out + wfirst) & 15) == 0)) {
    *reinterpret_cast<uint4 *>(a.out + wfirst) = make_uint4(o[0], o[1], o[2], o[3]);
  } else {
#pragma unroll
    for (int k = 0; k < CWPT; k++)
      if (wfirst + k < (long long)a.CL) a.out[wfirst + k] = o[k];
  }
}

// Carry resolve from group sums (see write_group_sums): group g (digits
// [G g, G g + G)) covers words W_g .. W_g + K - 1, W_g = floor(G b g / 32),
// and at most CARRY_GCOV groups cover one word. A block owns GCT * GWPT
// words; the group sums under them are staged in LDS with 16-byte loads;
// each thread walks its GWPT + 1 words (the first is its left neighbour's
// last) with a running group index, forms P_w, v_w = lo(P_w) + hi(P_{w-1})
// and the carry-function scan of k_carry_local.
constexpr int GCT = 256;
constexpr int GWPT = 8;  // 2048-word blocks: 17 KB of staged groups, nine blocks per CU
template <int GCOV>  // group sums that can cover one word (<= CARRY_GCOV)
static __global__ __launch_bounds__(GCT) void k_carry_groups(CarryArgs a) {
  extern __shared__ uint32_t gl_w[];
  __shared__ unsigned wave_fn[GCT / 64];
  __shared__ BlockCarry bc;
  bind_carry(a, blockIdx.y);  // batched: product blockIdx.y
  if ((unsigned long long)blockIdx.x >= a.nblk) return;
  const int tid = threadIdx.x;
  const long long W0 = (long long)blockIdx.x * GCT * GWPT;
  const int gb = a.gC * a.bits;  // bits per group, >= 32
  const double inv_gb = 1.0 / (double)gb;
  const long long ng = a.ng;
  long long g_first = W0 == 0 ? 0 : div_small(32 * (W0 - 2) + 31, gb, inv_gb) - (CARRY_GCOV - 1);
  if (g_first < 0) g_first = 0;
  long long g_last = div_small(32 * (W0 + (long long)GCT * GWPT - 1) + 31, gb, inv_gb);
  if (g_last >= ng) g_last = ng - 1;
  // LDS word i lives at i + i / 32: threads read words GWPT apart, and the pad
  // keeps those reads on distinct banks
  {
    const int nvec = g_last >= g_first ? (int)((g_last - g_first + 1) * a.gKs / 4) : 0;
    const uint4 *src = reinterpret_cast<const uint4 *>(a.ybuf + g_first * a.gKs);
    for (int t0 = 0; t0 < nvec; t0 += 8 * GCT) {
      uint4 r[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int t = t0 + u * GCT + tid;
        r[u] = t < nvec ? src[t] : make_uint4(0u, 0u, 0u, 0u);
      }
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int t = t0 + u * GCT + tid;
        if (t < nvec) {
          const unsigned i = (unsigned)(4 * t), pi = i + (i >> 5);  // 4 words never straddle a pad
          gl_w[pi] = r[u].x;
          gl_w[pi + 1] = r[u].y;
          gl_w[pi + 2] = r[u].z;
          gl_w[pi + 3] = r[u].w;
        }
      }
    }
  }
  __syncthreads();
  const long long wfirst = W0 + (long long)tid * GWPT;
  // Block-relative 32-bit arithmetic: staged group gl (group g_first + gl)
  // starts at bit B0 + gl gb, B0 = g_first gb, i.e. in block word
  // D + ((r0 + gl gb) >> 5), r0 = B0 & 31, D = (B0 >> 5) - W0 (<= 0).
  const unsigned long long B0 = (unsigned long long)g_first * (unsigned long long)gb;
  const int r0 = (int)(B0 & 31ull);
  const int D = (int)((long long)(B0 >> 5) - W0);
  const int ngl = (int)(g_last - g_first + 1);
  // words below lim (relative) exist: w < CL
  const long long lim64 = (long long)a.CL - W0;
  const int lim = lim64 > (1 << 30) ? (1 << 30) : (int)lim64;
  const int wmin = W0 == 0 ? 0 : -1;  // word W0 - 1 exists unless W0 = 0
  unsigned long long P[GWPT + 1], Pm2 = 0;  // Pm2: word W0 - 2 (thread 0)
  if (tid == 0 && W0) {
    const int num = 32 * (-2 - D) + 31 - r0;
    const int gh = num < 0 ? -1 : min((int)((unsigned)num / (unsigned)gb), ngl - 1);
#pragma unroll
    for (int t = 0; t < GCOV; t++) {
      const int off = -2 - (((r0 + (gh - t) * gb) >> 5) + D);
      if (gh - t >= 0 && off < a.gK) {
        const unsigned i = (unsigned)((gh - t) * a.gKs + off);
        Pm2 += gl_w[i + (i >> 5)];
      }
    }
    if (a.add && W0 - 2 < (long long)a.addl) Pm2 += a.add[W0 - 2];
  }
  if ((gb & 31) == 0) {
    // Word-aligned group starts (G b a multiple of 32, e.g. b even): group gl
    // starts at block word D + gl Q, so word wl = D + gh Q + o takes word
    // o + t Q of group gh - t, at LDS index ih - t (gKs - Q), ih = gh gKs + o;
    // all advance by one per word. A term counts where its group is staged:
    // none below the first, and none past the last group of the product, which an
    // output longer than the digits (AL + BL + 1 words at a full class, a long
    // addend) goes beyond. o < Q < K, so term 0 needs no more than that.
    const int Q = gb >> 5, dg = a.gKs - Q;
    const unsigned staged = ngl > 0 ? (unsigned)ngl : 0u;
    int wl = tid * GWPT - 1;
    const int x0 = wl - D;  // >= -1
    int gh = x0 < 0 ? -1 : (int)((unsigned)x0 / (unsigned)Q);
    int o = x0 - gh * Q;
    int ih = gh * a.gKs + o;
#pragma unroll
    for (int k = 0; k <= GWPT; k++, wl++) {
      if (k > 0) {
        const bool wrap = o + 1 == Q;
        o = wrap ? 0 : o + 1;
        gh += wrap ? 1 : 0;
        ih += wrap ? 1 + dg : 1;
      }
      unsigned long long p = 0;
#pragma unroll
      for (int t = 0; t < GCOV; t++) {
        const bool ok = (unsigned)(gh - t) < staged && (t == 0 || o + t * Q < a.gK);
        const unsigned i = ok ? (unsigned)(ih - t * dg) : 0u;
        const unsigned x = gl_w[i + (i >> 5)];
        p += ok ? x : 0u;
      }
      P[k] = (wl >= wmin && wl < lim) ? p : 0ull;
    }
  } else {
    // running group: gl = last staged group starting at or before word wl (-1: none)
    int wl = tid * GWPT - 1;
    const int num = 32 * (wl - D) + 31 - r0;
    int gl = num < 0 ? -1 : (int)((unsigned)num / (unsigned)gb);
    if (gl > ngl - 1) gl = ngl - 1;
    int Wt[GCOV];  // Wt[t]: first block word of group gl - t
#pragma unroll
    for (int t = 0; t < GCOV; t++) Wt[t] = ((r0 + (gl - t) * gb) >> 5) + D;
    int wnext = ((r0 + (gl + 1) * gb) >> 5) + D;  // first word of group gl + 1
#pragma unroll
    for (int k = 0; k <= GWPT; k++, wl++) {
      if (k > 0 && gl + 1 < ngl && wnext <= wl) {
        gl++;
#pragma unroll
        for (int t = GCOV - 1; t > 0; t--) Wt[t] = Wt[t - 1];
        Wt[0] = wnext;
        wnext = ((r0 + (gl + 1) * gb) >> 5) + D;
      }
      // branch-free: out-of-range terms read slot 0 and count as 0
      unsigned long long p = 0;
#pragma unroll
      for (int t = 0; t < GCOV; t++) {
        const int off = wl - Wt[t];
        const bool ok = gl - t >= 0 && off < a.gK;
        const unsigned i = ok ? (unsigned)((gl - t) * a.gKs + off) : 0u;
        const unsigned x = gl_w[i + (i >> 5)];
        p += ok ? x : 0u;
      }
      P[k] = (wl >= wmin && wl < lim) ? p : 0ull;
    }
  }
  if (a.add) {  // the addend's words, where they exist
#pragma unroll
    for (int k = 0; k <= GWPT; k++) {
      const long long w = wfirst - 1 + k;
      if (w >= 0 && w < (long long)a.CL && w < (long long)a.addl) P[k] += a.add[w];
    }
  }
  if (wfirst == 0) P[0] = 0;
  if (tid == 0) bc = block_carry(P[0], Pm2);
  unsigned long long v[GWPT];
#pragma unroll
  for (int k = 0; k < GWPT; k++) v[k] = (P[k + 1] & 0xffffffffull) + (P[k] >> 32);
  unsigned f0 = 0, f1 = 1;
#pragma unroll
  for (int k = 0; k < GWPT; k++) {
    f0 = (unsigned)((v[k] + f0) >> 32);
    f1 = (unsigned)((v[k] + f1) >> 32);
  }
  const unsigned f = f0 | (f1 << 1);
  const int lane = tid & 63, wave = tid >> 6;
  unsigned inc = f;
  for (int off = 1; off < 64; off <<= 1) {
    unsigned gq = __shfl_up(inc, off, 64);
    if (lane >= off) inc = carry_compose(gq, inc);
  }
  unsigned excl = __shfl_up(inc, 1, 64);
  if (lane == 0) excl = 2u;
  if (lane == 63) wave_fn[wave] = inc;
  __syncthreads();
  unsigned pre = 2u;
  for (int q = 0; q < wave; q++) pre = carry_compose(pre, wave_fn[q]);
  if (tid == 0) {
    unsigned tot = 2u;
    for (int q = 0; q < GCT / 64; q++) tot = carry_compose(tot, wave_fn[q]);
    carry_publish(a, tot, bc);
  }
  if (blockIdx.x == 0 && tid < 64) carry_margin(a);
  unsigned cin = (carry_compose(pre, excl) >> bc.cin) & 1u;
  uint32_t o[GWPT];
#pragma unroll
  for (int k = 0; k < GWPT; k++) {
    unsigned long long sum = v[k] + cin;
    o[k] = (uint32_t)sum;
    cin = (unsigned)(sum >> 32);
  }
  if (wfirst + GWPT <= (long long)a.CL && ((reinterpret_cast<uintptr_t>(a.out + wfirst) & 15) == 0)) {
    uint4 *dst = reinterpret_cast<uint4 *>(a.out + wfirst);
#pragma unroll
    for (int q = 0; q < GWPT / 4; q++) dst[q] = make_uint4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
  } else {
#pragma unroll
    for (int k = 0; k < GWPT; k++)
      if (wfirst + k < (long long)a.CL) a.out[wfirst + k] = o[k];
  }
}

// The blocks whose carry-in the block itself left open (bit 2 of its function):
// their carry-in is what the nearest lower block that does not propagate hands
// on. Each workgroup looks at RIPPLE_BLOCKS functions and is done when none of
// them is marked; otherwise it walks down to the carry into its first block,
// then up through its blocks, and adds the carry where it is 1: a block of
// 0xffffffff words (one that propagates) is cleared, in any other the words up
// to the first other one are cleared and that one takes the +1.
constexpr int RIPPLE_BLOCKS = 256;
static __global__ __launch_bounds__(RIPPLE_BLOCKS) void k_carry_ripple(CarryArgs a) {
  __shared__ unsigned char fn[RIPPLE_BLOCKS];
  __shared__ int near;
  __shared__ unsigned long long first;
  const int tid = threadIdx.x;
  bind_carry(a, blockIdx.y);
  const unsigned long long b0 = (unsigned long long)blockIdx.x * RIPPLE_BLOCKS;
  if (b0 >= a.nblk) return;
  const int n = (int)(a.nblk - b0 < RIPPLE_BLOCKS ? a.nblk - b0 : RIPPLE_BLOCKS);
  const unsigned f = tid < n ? a.blk_fn[b0 + tid] : 0u;
  fn[tid] = (unsigned char)f;
  if (!__syncthreads_or((int)(f & 4u))) return;
  // carry into block b0: the nearest block below whose function is constant
  unsigned c = 0;
  for (unsigned long long hi = b0; hi > 0;) {
    const unsigned long long lo = hi > RIPPLE_BLOCKS ? hi - RIPPLE_BLOCKS : 0;
    if (tid == 0) near = -1;
    __syncthreads();
    const unsigned g = lo + tid < hi ? a.blk_fn[lo + tid] & 3u : 2u;
    if (g != 2u) atomicMax(&near, tid);
    __syncthreads();
    const int k = near;
    __syncthreads();
    if (k >= 0) {
      c = a.blk_fn[lo + k] & 1u;
      break;
    }
    hi = lo;
  }
  for (int k = 0; k < n; k++) {  // uniform across the workgroup
    const unsigned g = fn[k];
    if ((g & 4u) && c) {
      const unsigned long long w0 = (b0 + k) * a.wpb;
      const unsigned long long w1 = w0 + a.wpb < a.CL ? w0 + a.wpb : a.CL;
      if ((g & 3u) == 2u) {
        for (unsigned long long w = w0 + tid; w < w1; w += RIPPLE_BLOCKS) a.out[w] = 0u;
      } else {
        if (tid == 0) first = w1;
        __syncthreads();
        for (unsigned long long w = w0 + tid; w < w1; w += RIPPLE_BLOCKS)
          if (a.out[w] != 0xffffffffu) {
            atomicMin(&first, w);
            break;
          }
        __syncthreads();
        const unsigned long long fw = first;
        for (unsigned long long w = w0 + tid; w < fw; w += RIPPLE_BLOCKS) a.out[w] = 0u;
        if (tid == 0 && fw < w1) a.out[fw] += 1u;
        __syncthreads();
      }
    }
    c = (g >> c) & 1u;
  }
}

// Margins of whole slot sets to the host, one per workgroup: of a product ahead
// of its carry (products in place), of the products of a deferral scope.
static __global__ __launch_bounds__(64) void k_margin_out(const unsigned int *m, unsigned *host) {
  const unsigned v = margin_of_slots(m + (size_t)blockIdx.x * MARGIN_SLOTS * MARGIN_STRIDE);
  if (threadIdx.x == 0) host_store(host + blockIdx.x, v);
}

// --------------------------------------------------------------- utilities

static __global__ void k_zero_u32(unsigned int *p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

static __global__ void k_fill_u32(uint32_t *p, unsigned long long n, uint32_t v) {
  unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long st = (unsigned long long)gridDim.x * blockDim.x;
  for (; i < n; i += st) p[i] = v;
}

}  // namespace bcg

namespace bcg {

// ------------------------------------------- one-workgroup products (batched)


// P_w for one word from coefficients held in LDS (see word_partials).
__device__ __forceinline__ unsigned long long word_partial_lds(const long long *coef, long long ncoef, int bits,
                                                               int cbits, long long w) {
  if (w < 0) return 0ull;
  long long lo_bit = 32 * w - cbits + 1;
  long long jlo = lo_bit <= 0 ? 0 : (lo_bit + bits - 1) / bits;
  long long jhi = (32 * w + 31) / bits;
  if (jhi >= ncoef) jhi = ncoef - 1;
  unsigned long long P = 0;
  for (long long j = jlo; j <= jhi; j++) {
    unsigned long long c = (unsigned long long)coef[j];
    long long sh = (long long)bits * j - 32 * w;
    if (sh >= 0)
      P += (unsigned long long)(uint32_t)(c << sh);
    else if (-sh < 64)
      P += (unsigned long long)(uint32_t)(c >> (-sh));
  }
  return P;
}

// Words out[0..CL) = (sum_j coef[j] 2^{bits j}) mod 2^{32 CL}, coefficients in
// LDS, carries resolved with a workgroup scan of carry functions; 64-bit word
// indices, every word's partial computed twice (for output lengths of 2^19
// words and more: a short product with a long addend).
template <int T>
__device__ void wg_carry_wide(const long long *coef, long long ncoef, int bits, int cbits, uint32_t *out, long long CL,
                         const uint32_t *add, long long addl, int tid) {
  __shared__ unsigned wave_fn[T / 64 + 1];
  const long long per = (CL + T - 1) / T;
  const long long w0 = (long long)tid * per;
  long long w1 = w0 + per;
  if (w1 > CL) w1 = CL;
  // this thread's carry function over words [w0, w1)
  unsigned f = 2u;  // identity
  {
    unsigned long long prev = word_partial_lds(coef, ncoef, bits, cbits, w0 - 1);
    if (add && w0 >= 1 && w0 - 1 < addl) prev += add[w0 - 1];
    unsigned c0 = 0, c1 = 1;
    for (long long w = w0; w < w1; w++) {
      unsigned long long P = word_partial_lds(coef, ncoef, bits, cbits, w);
      if (add && w < addl) P += add[w];
      unsigned long long v = (P & 0xffffffffull) + (prev >> 32);
      c0 = (unsigned)((v + c0) >> 32);
      c1 = (unsigned)((v + c1) >> 32);
      prev = P;
    }
    if (w0 < w1) f = c0 | (c1 << 1);
  }
  // inclusive scan within the wave
  const int lane = tid & 63, wave = tid >> 6;
  unsigned inc = f;
  for (int off = 1; off < 64; off <<= 1) {
    unsigned g = __shfl_up(inc, off, 64);
    if (lane >= off) inc = carry_compose(g, inc);
  }
  unsigned excl = __shfl_up(inc, 1, 64);
  if (lane == 0) excl = 2u;
  if (lane == 63) wave_fn[wave] = inc;
  __syncthreads();
  unsigned pre = 2u;
  for (int w = 0; w < wave; w++) pre = carry_compose(pre, wave_fn[w]);
  unsigned cin = carry_compose(pre, excl) & 1u;  // carry into word w0 (block carry-in is 0)
  // write the words
  unsigned long long prev = word_partial_lds(coef, ncoef, bits, cbits, w0 - 1);
  if (add && w0 >= 1 && w0 - 1 < addl) prev += add[w0 - 1];
  for (long long w = w0; w < w1; w++) {
    unsigned long long P = word_partial_lds(coef, ncoef, bits, cbits, w);
    if (add && w < addl) P += add[w];
    unsigned long long v = (P & 0xffffffffull) + (prev >> 32) + cin;
    out[w] = (uint32_t)v;
    cin = (unsigned)(v >> 32);
    prev = P;
  }
}

// P_w for word w < 2^19 from the coefficients in LDS, 32-bit index arithmetic:
// coefficient j (below 2^cbits) sits at bit b j, so words take j in
// [ceil((32 w - cbits + 1) / b), floor((32 w + 31) / b)].
__device__ __forceinline__ unsigned long long word_partial32(const long long *coef, int ncoef, int bits, int cbits,
                                                             float inv_b, int w) {
  if (w < 0) return 0ull;
  const int lo_bit = 32 * w - cbits + 1;
  const int jlo = lo_bit <= 0 ? 0 : fdiv_small(lo_bit + bits - 1, bits, inv_b);
  int jhi = fdiv_small(32 * w + 31, bits, inv_b);
  if (jhi >= ncoef) jhi = ncoef - 1;
  unsigned long long P = 0;
  int sh = bits * jlo - 32 * w;  // in (-cbits, 32)
  for (int j = jlo; j <= jhi; j++, sh += bits) {
    const unsigned long long c = (unsigned long long)coef[j];
    P += (unsigned long long)(uint32_t)(sh >= 0 ? c << sh : c >> -sh);
  }
  return P;
}

// Words out[0..CL) = (sum_j coef[j] 2^{bits j} + add) mod 2^{32 CL}, coefficients
// in LDS. Each thread takes CL / T consecutive words and writes them as for a
// carry-in of 0, computing every word's partial once, while it tracks its
// carry outs for carry-ins 0 and 1; a workgroup scan of those carry functions
// gives each thread its carry-in, and a carry-in of 1 then ripples through the
// thread's leading all-ones words.
template <int T>
__device__ void wg_carry(const long long *coef, long long ncoef, int bits, int cbits, uint32_t *out, long long CL,
                         const uint32_t *add, long long addl, int tid) {
  if (CL >= (1ll << 19) || ncoef >= (1ll << 30)) {  // 32 w + 31 < 2^24 below
    wg_carry_wide<T>(coef, ncoef, bits, cbits, out, CL, add, addl, tid);
    return;
  }
  __shared__ unsigned wave_fn[T / 64 + 1];
  const int cl = (int)CL, nc = (int)ncoef;
  const float inv_b = 1.0f / (float)bits;
  const int per = (cl + T - 1) / T;
  const int w0 = tid * per;
  const int w1 = w0 + per < cl ? w0 + per : cl;
  unsigned f = 2u;  // identity
  {
    unsigned long long prev = word_partial32(coef, nc, bits, cbits, inv_b, w0 - 1);
    if (add && w0 >= 1 && w0 - 1 < addl) prev += add[w0 - 1];
    unsigned c0 = 0, c1 = 1;
    for (int w = w0; w < w1; w++) {
      unsigned long long P = word_partial32(coef, nc, bits, cbits, inv_b, w);
      if (add && w < addl) P += add[w];
      const unsigned long long v = (P & 0xffffffffull) + (prev >> 32);
      const unsigned long long s0 = v + c0;
      out[w] = (uint32_t)s0;
      c0 = (unsigned)(s0 >> 32);
      c1 = (unsigned)((v + c1) >> 32);
      prev = P;
    }
    if (w0 < w1) f = c0 | (c1 << 1);
  }
  // inclusive scan within the wave
  const int lane = tid & 63, wave = tid >> 6;
  unsigned inc = f;
  for (int off = 1; off < 64; off <<= 1) {
    unsigned g = __shfl_up(inc, off, 64);
    if (lane >= off) inc = carry_compose(g, inc);
  }
  unsigned excl = __shfl_up(inc, 1, 64);
  if (lane == 0) excl = 2u;
  if (lane == 63) wave_fn[wave] = inc;
  __syncthreads();
  unsigned pre = 2u;
  for (int w = 0; w < wave; w++) pre = carry_compose(pre, wave_fn[w]);
  const unsigned cin = carry_compose(pre, excl) & 1u;  // carry into word w0 (block carry-in is 0)
  if (cin) {
    for (int w = w0; w < w1; w++) {
      const uint32_t x = out[w] + 1u;
      out[w] = x;
      if (x) break;
    }
  }
}

// All products of one transform length class L (one-pass plans: N = L).
struct ClassArgs {
  const MulDesc *desc;    // nullptr: the single product `one`
  Roots roots;
  const cd *tl;
  unsigned int *margins;  // per product, float bits of the worst rounding distance
  int clear;              // a set of MARGIN_SLOTS slots: clear the others
  MulDesc one;            // a single product travels in the launch itself
};

// Values the same in every lane, held in scalar registers.
__device__ __forceinline__ unsigned long long uniform64(unsigned long long v) {
  return (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v) |
         (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32)) << 32;
}
template <class T>
__device__ __forceinline__ T *uniform_ptr(T *p) {
  return reinterpret_cast<T *>(uniform64(reinterpret_cast<unsigned long long>(p)));
}

// A product's descriptor, the same for the whole workgroup. The compiler reads
// it with vector loads (the kernel stores to global memory between products),
// and a buffer resource made of vector registers costs a loop per load.
__device__ __forceinline__ MulDesc uniform_desc(const MulDesc &m) {
  MulDesc d;
  d.a = uniform_ptr(m.a);
  d.b = uniform_ptr(m.b);
  d.c = uniform_ptr(m.c);
  d.d = uniform_ptr(m.d);
  d.al = uniform64(m.al);
  d.bl = uniform64(m.bl);
  d.cl = uniform64(m.cl);
  d.dl = uniform64(m.dl);
  d.bits = __builtin_amdgcn_readfirstlane(m.bits);
  d.cbits = __builtin_amdgcn_readfirstlane(m.cbits);
  return d;
}

// Digits tid + h T of an operand (h < 8) into lo, digits tid + h T + L into up
// (zero beyond the operand). For 32 | T a lane's digits sit a whole number of
// words apart, so one bit offset and one byte offset serve all sixteen, read
// with range-checked buffer loads as in PackDigits; shorter rows go digit by
// digit.
template <int L>
__device__ __forceinline__ void row_digits(const uint32_t *w, unsigned long long wl, int bits, int tid,
                                           unsigned (&lo)[8], unsigned (&up)[8]) {
  constexpr int T = Row<L>::T;
  if constexpr (T % 32 == 0) {
    const unsigned b = (unsigned)bits, bit = (unsigned)tid * b;
    const unsigned step = (unsigned)(T / 32) * b * 4u;  // bytes between digits j and j + T
    const unsigned off = (bit >> 5) * 4u, sh = bit & 31u;
    const __amdgpu_buffer_rsrc_t w0 = word_rsrc(w, wl), w1 = word_rsrc(w + 1, wl - 1);
#pragma unroll
    for (int h = 0; h < 8; h++) {
      lo[h] = __builtin_amdgcn_raw_buffer_load_b32(w0, off + (unsigned)h * step, 0, 0);
      up[h] = __builtin_amdgcn_raw_buffer_load_b32(w0, off + (unsigned)(h + 8) * step, 0, 0);
    }
    if ((b & (b - 1u)) == 0u) {  // b <= 32 divides 32: no digit straddles two words
#pragma unroll
      for (int h = 0; h < 8; h++) {
        lo[h] = __builtin_amdgcn_ubfe(lo[h], sh, b);
        up[h] = __builtin_amdgcn_ubfe(up[h], sh, b);
      }
    } else {
      unsigned lo1[8], up1[8];
#pragma unroll
      for (int h = 0; h < 8; h++) {
        lo1[h] = __builtin_amdgcn_raw_buffer_load_b32(w1, off + (unsigned)h * step, 0, 0);
        up1[h] = __builtin_amdgcn_raw_buffer_load_b32(w1, off + (unsigned)(h + 8) * step, 0, 0);
      }
#pragma unroll
      for (int h = 0; h < 8; h++) {
        lo[h] = __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(lo1[h], lo[h], sh), 0, b);
        up[h] = __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(up1[h], up[h], sh), 0, b);
      }
    }
  } else {
#pragma unroll
    for (int h = 0; h < 8; h++) {
      lo[h] = (unsigned)digit_at(w, wl, (unsigned long long)(tid + h * T), bits);
      up[h] = (unsigned)digit_at(w, wl, (unsigned long long)(tid + h * T + L), bits);
    }
  }
}

// One workgroup per product of a length class runs it whole: pack, forward,
// pointwise, inverse, rounding and the carry resolve, with the coefficients
// never leaving LDS. Row tid + h T has the right-angle weight
// Omega^{tid} e^{2 pi i h / 32} (T = L / 8, N = L): one computed point and
// eight constants per thread. Bound by LDS exchanges and FP64 issue, with one
// (8192 points) to sixteen workgroups on a CU. Workgroups that loop over the
// class's products had the loop's constants and twiddles hoisted into 50 more
// registers; the products of a class cost the same, so the dispatcher
// balances them as well.
template <int L>
__global__ __launch_bounds__((Row<L>::T)) void k_mul1(ClassArgs ca) {
  using RC = Row<L>;
  __shared__ cd lds[RC::LDS_ELEMS];
  __shared__ float wmax[(RC::T + 63) / 64];
  const int tid = threadIdx.x, idx = blockIdx.x;
  const MulDesc d = ca.desc ? uniform_desc(ca.desc[idx]) : ca.one;
  cd wt = omega_direct(ca.roots, (unsigned long long)tid);
  const bool square = d.a == d.b && d.al == d.bl;
  cd x[8], xa[RC::XR];
  unsigned lo[8], up[8];
  row_digits<L>(d.a, d.al, d.bits, tid, lo, up);
#pragma unroll
  for (int h = 0; h < 8; h++) x[h] = cmul(make_double2((double)lo[h], (double)up[h]), cmul(wt, w64(2 * h)));
  if (square) {
    row_forward<L, 8>(x, xa, lds, ca.tl, tid);
#pragma unroll
    for (int i = 0; i < RC::XR; i++) xa[i] = cmul(xa[i], xa[i]);
  } else {
    cd xb[RC::XR];
    row_digits<L>(d.b, d.bl, d.bits, tid, lo, up);  // arrive under A's stages
    row_forward<L, 8>(x, xa, lds, ca.tl, tid);
    asm volatile("" : "+v"(wt.x), "+v"(wt.y));
#pragma unroll
    for (int h = 0; h < 8; h++) x[h] = cmul(make_double2((double)lo[h], (double)up[h]), cmul(wt, w64(2 * h)));
    __syncthreads();
    row_forward<L, 8>(x, xb, lds, ca.tl, tid);
#pragma unroll
    for (int i = 0; i < RC::XR; i++) xa[i] = cmul(xa[i], xb[i]);
  }
  row_inverse<L, 8>(xa, x, lds, ca.tl, tid);
  __syncthreads();  // LDS now becomes the coefficient array
  long long *coef = (long long *)lds;
  const double inv_n = 1.0 / (double)L;
  double worst = 0.0;
  const bool fast = d.cbits <= 51;
  asm volatile("" : "+v"(wt.x), "+v"(wt.y));
#pragma unroll
  for (int h = 0; h < 8; h++) {
    const int j = tid + h * RC::T;
    const cd f = cmulc(x[h], cmul(wt, w64(2 * h)));
    coef[j] = round_coef(f.x * inv_n, fast, worst);
    coef[j + L] = round_coef(f.y * inv_n, fast, worst);
  }
  float far = (float)worst;
  for (int off = 32; off > 0; off >>= 1) far = fmaxf(far, __shfl_xor(far, off, 64));
  if ((tid & 63) == 0) wmax[tid >> 6] = far;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < (RC::T + 63) / 64; w++) far = fmaxf(far, wmax[w]);
    host_store(ca.margins + idx, __float_as_uint(far));
  }
  if (ca.clear)
    for (int i = 1 + tid; i < MARGIN_SLOTS; i += RC::T) ca.margins[i * MARGIN_STRIDE] = 0u;
  wg_carry<RC::T>(coef, 2 * L, d.bits, d.cbits, d.c, (long long)d.cl, d.d, (long long)d.dl, tid);
}

}  // namespace bcg

namespace bcg {

// out[w] = low word of val(w) + carries for w < n (val < 2^32 + 2^31, carry-in
// cin), each of the workgroup's T threads a run of consecutive words; returns 1 +
// the highest nonzero index (0: none), the same in every thread. What val reads
// may be overwritten only after the return.
template <int T, class F>
__device__ long long wg_carry_words(uint32_t *out, long long n, unsigned cin, F val) {
  constexpr int W = T / 64;
  __shared__ unsigned fn[W];
  __shared__ long long tops[W];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long long per = (n + T - 1) / T, w0 = tid * per, w1 = w0 + per < n ? w0 + per : n;
  unsigned c0 = 0, c1 = 1;
  for (long long w = w0; w < w1; w++) {
    const unsigned long long v = val(w);
    c0 = (unsigned)((v + c0) >> 32);
    c1 = (unsigned)((v + c1) >> 32);
  }
  unsigned inc = w0 < w1 ? c0 | (c1 << 1) : 2u;
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned g1 = __shfl_up(inc, off, 64);
    if (lane >= off) inc = carry_compose(g1, inc);
  }
  unsigned excl = __shfl_up(inc, 1, 64);
  if (lane == 0) excl = 2u;
  if (lane == 63) fn[wave] = inc;
  __syncthreads();
  unsigned pre = 2u;
  for (int w = 0; w < wave; w++) pre = carry_compose(pre, fn[w]);
  unsigned c = (carry_compose(pre, excl) >> cin) & 1u;
  long long top = 0;
  for (long long w = w0; w < w1; w++) {
    const unsigned long long v = val(w) + c;
    c = (unsigned)(v >> 32);
    out[w] = (uint32_t)v;
    if ((uint32_t)v) top = w + 1;
  }
  for (int off = 32; off > 0; off >>= 1) {
    const long long o = __shfl_xor(top, off, 64);
    top = o > top ? o : top;
  }
  if (lane == 0) tops[wave] = top;
  __syncthreads();
  for (int w = 0; w < W; w++) top = tops[w] > top ? tops[w] : top;
  __syncthreads();
  return top;
}

// Schoolbook product (+ addend) of one workgroup from operands a, b (in LDS, or
// in global memory): thread w sums column w of 32x32-bit products, low and high
// halves apart, and the carry chain is a scan over the threads. One thread
// walking the chain was 5 of 8 us at 43 words.
template <int T>
__device__ void wg_basecase(uint32_t *C, unsigned long long CL, const uint32_t *a, int al, const uint32_t *b, int bl,
                            const uint32_t *D, unsigned long long DL, unsigned long long *lo,
                            unsigned long long *hi) {
  const int W = al + bl;
  for (int w = threadIdx.x; w < W; w += T) {
    const int i0 = w >= bl ? w - bl + 1 : 0, i1 = w < al ? w : al - 1;
    unsigned long long l = 0, h = 0;
#pragma unroll 4
    for (int i = i0; i <= i1; i++) {
      const unsigned long long pr = (unsigned long long)a[i] * b[w - i];
      l += pr & 0xffffffffull;
      h += pr >> 32;
    }
    lo[w] = l;
    hi[w] = h;
  }
  __syncthreads();
  auto P = [&](long long w) {
    unsigned long long v = w >= 0 && w < W ? lo[w] : 0ull;
    if (w >= 1 && w - 1 < W) v += hi[w - 1];
    if (D && w >= 0 && (unsigned long long)w < DL) v += D[w];
    return v;
  };
  wg_carry_words<T>(C, (long long)CL, 0u,
                    [&](long long w) { return (P(w) & 0xffffffffull) + (P(w - 1) >> 32); });
}

// Batched schoolbook products (AL + BL < 100 words): one wave per product.
static __global__ __launch_bounds__(64) void k_basecase_batch(const MulDesc *desc, int count) {
  __shared__ unsigned long long lo[128], hi[128];
  __shared__ uint32_t ab[128];
  const int p = blockIdx.x;
  if (p >= count) return;
  const MulDesc d = desc[p];
  const int al = (int)d.al, bl = (int)d.bl;
  for (int i = threadIdx.x; i < al + bl; i += 64) ab[i] = i < al ? d.a[i] : d.b[i - al];
  __syncthreads();
  wg_basecase<64>(d.c, d.cl, ab, al, ab + al, bl, d.d, d.dl, lo, hi);
}

// One schoolbook product. STAGE: the operands go through LDS (al + bl <=
// BASECASE_STAGE), so C may be A or B.
constexpr int BASECASE_STAGE = 1024;
template <int T, bool STAGE>
__global__ __launch_bounds__(T) void k_basecase(const uint32_t *A, int al, const uint32_t *B, int bl, uint32_t *C,
                                                unsigned long long CL, const uint32_t *D, unsigned long long DL) {
  extern __shared__ unsigned long long dyn[];
  unsigned long long *lo = dyn, *hi = dyn + (al + bl);
  if constexpr (STAGE) {
    uint32_t *ab = reinterpret_cast<uint32_t *>(dyn + 2 * (al + bl));
    for (int i = threadIdx.x; i < al + bl; i += T) ab[i] = i < al ? A[i] : B[i - al];
    __syncthreads();
    wg_basecase<T>(C, CL, ab, al, ab + al, bl, D, DL, lo, hi);
  } else {
    wg_basecase<T>(C, CL, A, al, B, bl, D, DL, lo, hi);
  }
}

// k_mul1 with twice the threads: one half transforms A, the other B, each in a tile
// of its own; they exchange the transforms, both run the inverse and round half of
// the points, and all carry. The same operations on the same values as k_mul1.
// For a product alone on its CU, where one wave per SIMD waits for its own chain: 300
// by 300 words 23.4 -> 21.0 us, 600 26.1 -> 24.7, 1000 by 777 25.6 -> 24.7 us a call.
// From 3072 points a half fills the SIMDs and the barriers of 1024 threads cost more
// (2000 words 29.7 -> 31.0 us), and where workgroups share a CU the second inverse is
// work for nothing (4096 products of a batch 631 -> 637 us).
template <int L>
constexpr bool has_mul2() {
  return Row<L>::T % 64 == 0 && Row<L>::T <= 256;
}

template <int L>
__global__ __launch_bounds__((2 * Row<L>::T)) void k_mul2(ClassArgs ca) {
  using RC = Row<L>;
  constexpr int T = RC::T, XR = RC::XR;
  __shared__ cd tiles[2][RC::LDS_ELEMS];
  __shared__ float wmax[2 * T / 64];
  const int idx = blockIdx.x, tid = (int)threadIdx.x % T;
  const int half = __builtin_amdgcn_readfirstlane((int)threadIdx.x / T);  // whole waves
  const MulDesc d = ca.desc ? uniform_desc(ca.desc[idx]) : ca.one;
  cd *lds = tiles[half];
  cd wt = omega_direct(ca.roots, (unsigned long long)tid);
  cd x[8], xa[XR], xo[XR];
  unsigned lo[8], up[8];
  row_digits<L>(half ? d.b : d.a, half ? d.bl : d.al, d.bits, tid, lo, up);
#pragma unroll
  for (int h = 0; h < 8; h++) x[h] = cmul(make_double2((double)lo[h], (double)up[h]), cmul(wt, w64(2 * h)));
  row_forward<L, 8>(x, xa, lds, ca.tl, tid);
#pragma unroll
  for (int i = 0; i < XR; i++)
    if (row_has<L, 8>(tid, i)) lds[row_at<L, 8>(tid, i)] = xa[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < XR; i++)
    xo[i] = row_has<L, 8>(tid, i) ? tiles[half ^ 1][row_at<L, 8>(tid, i)] : make_double2(0.0, 0.0);
#pragma unroll
  for (int i = 0; i < XR; i++) xa[i] = half ? cmul(xo[i], xa[i]) : cmul(xa[i], xo[i]);
  __syncthreads();  // the other half has read this tile
  row_inverse<L, 8>(xa, x, lds, ca.tl, tid);
  __syncthreads();  // the first tile now becomes the coefficient array
  long long *coef = (long long *)tiles[0];
  const double inv_n = 1.0 / (double)L;
  double worst = 0.0;
  const bool fast = d.cbits <= 51;
  asm volatile("" : "+v"(wt.x), "+v"(wt.y));
  auto round = [&](int h) {
    const int j = tid + h * T;
    const cd f = cmulc(x[h], cmul(wt, w64(2 * h)));
    coef[j] = round_coef(f.x * inv_n, fast, worst);
    coef[j + L] = round_coef(f.y * inv_n, fast, worst);
  };
  if (half) {
#pragma unroll
    for (int h = 4; h < 8; h++) round(h);
  } else {
#pragma unroll
    for (int h = 0; h < 4; h++) round(h);
  }
  float far = (float)worst;
  for (int off = 32; off > 0; off >>= 1) far = fmaxf(far, __shfl_xor(far, off, 64));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = far;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 2 * T / 64; w++) far = fmaxf(far, wmax[w]);
    host_store(ca.margins + idx, __float_as_uint(far));
  }
  if (ca.clear)
    for (int i = 1 + (int)threadIdx.x; i < MARGIN_SLOTS; i += 2 * T) ca.margins[i * MARGIN_STRIDE] = 0u;
  wg_carry<2 * T>(coef, 2 * L, d.bits, d.cbits, d.c, (long long)d.cl, d.d, (long long)d.dl, (int)threadIdx.x);
}

}  // namespace bcg
