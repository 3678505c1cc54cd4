// FP64 contractions held by single waves, operands straight from memory.
//
// v_mfma_f64_16x16x4f64 takes 64 cycles per SIMD on gfx950 (78.6 TFLOP/s over
// the chip), so a wave with TM x TN accumulator tiles needs only
// 32 (TM + TN) / (TM TN) bytes per clock and CU of operands: within what L1
// delivers without any staging in LDS.  A wave therefore loads its operands
// into registers itself, one chunk of 8 k ahead of the MFMAs that use them;
// there is no LDS, no barrier, and waves do not wait for each other.
//
// Operand forms, per chunk of 8 k (lane l: i = l % 16, g = l / 16; the MFMA's
// step s = 0, 1 takes k = 2 g + s, on both operands alike):
//   K-contiguous   -- one 16-byte load per tile: k = 2g, 2g + 1 of the lane's row
//   row-contiguous -- two 16-byte loads per pair of tiles: the lane's two rows
//                     at k = 2g and at k = 2g + 1
// Tiles 2P and 2P + 1 interleave their rows (32 P + 2 i + e), so both forms
// give the same row order and two neighbouring columns leave in one 16-byte
// store; an odd last tile has rows 16 t + i.
//
// All extents are multiples of 8 (the walk pads its arrays with zeros), so
// there is no K tail; rows past the extent repeat the last valid one and are
// not stored.
#pragma once
#include <hip/hip_runtime.h>

namespace pamd {

typedef double wg_d4 __attribute__((ext_vector_type(4)));
typedef double wg_d2 __attribute__((ext_vector_type(2)));

// One run of a contraction (wave-uniform): nout x nk chunks; the operands of
// outer step u start at A + u aos, B + u bos.  Strides in elements; ak == 1
// means K-contiguous rows, otherwise the rows are contiguous (ar == 1).
struct WSeg {
  const double *A, *B;
  long long ar, ak, br, bk, aos, bos;
  int nk, nout;
};

// row of MFMA row / column index r of tile t, of T tiles
template <int T>
__device__ __forceinline__ int wg_row(int t, int r) {
  return t < (T & ~1) ? 32 * (t >> 1) + 2 * r + (t & 1) : 16 * t + r;
}

// per-lane byte offsets of one operand's loads
template <int T>
__device__ __forceinline__ void wg_offsets(int r0, int R, long long rs, long long ks, bool kc, int lane,
                                           unsigned (&off)[T]) {
  const int i = lane & 15, g = lane >> 4;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    if (kc) {
      const int r = min(r0 + wg_row<T>(t, i), R - 1);
      off[t] = (unsigned)r * (unsigned)(rs * 8) + (unsigned)(16 * g);
    } else {
      // the pair's two tiles share the offset of the first
      const int te = t < (T & ~1) ? (t & ~1) : t;
      const int r = min(r0 + wg_row<T>(te, i), t < (T & ~1) ? R - 2 : R - 1);
      off[t] = (unsigned)r * 8u + (unsigned)(2 * g) * (unsigned)(ks * 8);
    }
  }
}

// Buffer loads: the address is a scalar base plus a 32-bit lane offset plus a
// scalar offset, so a chunk's loads need no vector address arithmetic.
template <int T>
__device__ __forceinline__ void wg_load(const char *p, int ks8, bool kc, const unsigned (&off)[T],
                                        wg_d2 (&x)[T]) {
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, -1, 0x00027000);
  if (kc) {
#pragma unroll
    for (int t = 0; t < T; ++t)
      x[t] = __builtin_bit_cast(wg_d2, __builtin_amdgcn_raw_buffer_load_b128(r, off[t], 0, 0));
  } else {
#pragma unroll
    for (int t = 0; t < (T & ~1); t += 2) {
      x[t] = __builtin_bit_cast(wg_d2, __builtin_amdgcn_raw_buffer_load_b128(r, off[t], 0, 0));
      x[t + 1] = __builtin_bit_cast(wg_d2, __builtin_amdgcn_raw_buffer_load_b128(r, off[t], ks8, 0));
    }
    if (T & 1) {
      x[T - 1][0] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off[T - 1], 0, 0));
      x[T - 1][1] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off[T - 1], ks8, 0));
    }
  }
}

// operand of tile t at step s of a loaded chunk
template <int T>
__device__ __forceinline__ double wg_get(const wg_d2 (&x)[T], bool kc, int t, int s) {
  return (kc || t >= (T & ~1)) ? x[t][s] : x[(t & ~1) + s][t & 1];
}

template <int TM, int TN>
__device__ __forceinline__ void wg_mma(const wg_d2 (&a)[TM], const wg_d2 (&b)[TN], bool akc, bool bkc,
                                       wg_d4 (&acc)[TM][TN]) {
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int x = 0; x < TM; ++x)
#pragma unroll
      for (int y = 0; y < TN; ++y)
        acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(wg_get<TM>(a, akc, x, s), wg_get<TN>(b, bkc, y, s),
                                                         acc[x][y], 0, 0, 0);
}

// chunks in registers: two loads ahead where 256 registers hold three chunks
// beside the accumulators, else one
constexpr int wg_buffers(int tm, int tn) { return 8 * tm * tn + 12 * (tm + tn) + 40 <= 256 ? 3 : 2; }

// acc += sum over the runs that gen yields.  AKC, BKC: whether the operand is
// K-contiguous, in every run.  (Choosing per run would put two copies of the
// MFMAs into the loop, and the compiler then spills.)
// gen.next(WSeg &) is wave-uniform and false at the end; chunks: the number of
// chunks of all its runs.
template <int TM, int TN, bool AKC, bool BKC, class Gen>
__device__ __forceinline__ void wg_accumulate(Gen &gen, int chunks, int m0, int M, int n0, int N,
                                              int lane, wg_d4 (&acc)[TM][TN]) {
  WSeg s;
  if (!gen.next(s)) return;
  unsigned oa[TM], ob[TN];
  const char *pa, *pb, *a0, *b0;
  long long ak8, bk8;
  int kl, ol;
  auto begin = [&]() {
    wg_offsets<TM>(m0, M, s.ar, s.ak, AKC, lane, oa);
    wg_offsets<TN>(n0, N, s.br, s.bk, BKC, lane, ob);
    ak8 = s.ak * 8;
    bk8 = s.bk * 8;
    a0 = pa = (const char *)s.A;
    b0 = pb = (const char *)s.B;
    kl = s.nk;
    ol = s.nout;
  };
  begin();
  constexpr int NB = wg_buffers(TM, TN);
  wg_d2 a[NB][TM], b[NB][TN];
  // loads the current chunk and moves on (after the last one the addresses
  // stay where they are)
  auto fetch = [&](int q) {
    wg_load<TM>(pa, (int)ak8, AKC, oa, a[q]);
    wg_load<TN>(pb, (int)bk8, BKC, ob, b[q]);
    if (--kl > 0) {
      pa += 8 * ak8;
      pb += 8 * bk8;
    } else if (--ol > 0) {
      a0 += s.aos * 8;
      b0 += s.bos * 8;
      pa = a0;
      pb = b0;
      kl = s.nk;
    } else if (gen.next(s)) {
      begin();
    } else {
      kl = ol = 1;
    }
  };
  auto mma = [&](int q) { wg_mma<TM, TN>(a[q], b[q], AKC, BKC, acc); };
  // NB chunks per iteration and one exit: the accumulators keep their registers
  // (a copy of them per iteration otherwise).  A fetch past the last chunk reads
  // that chunk again and is not used.
#pragma unroll
  for (int q = 0; q < NB - 1; ++q) fetch(q);
  const int full = (chunks - 1) / NB, rest = chunks - full * NB;
  for (int p = full; p > 0; --p) {
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      fetch((q + NB - 1) % NB);
      mma(q);
    }
  }
  if (rest == NB) fetch(NB - 1);
#pragma unroll
  for (int q = 0; q < NB; ++q)
    if (q < rest) mma(q);
}

// f(element of C, x, y, r) for the columns of the pair of tiles y, y + 1 of tile
// row x that lie in C (rows < M, columns < N, even), f1 for an odd last tile's
template <int TM, int TN, class F, class F1>
__device__ __forceinline__ void wg_each(double *C, long long rs, int m0, int M, int n0, int N, int lane, int x,
                                        F &&f, F1 &&f1) {
  const int i = lane & 15, g = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = m0 + wg_row<TM>(x, 4 * r + g);
    if (row >= M) continue;
    double *c = C + row * rs;
#pragma unroll
    for (int y = 0; y < (TN & ~1); y += 2) {
      const int col = n0 + 16 * y + 2 * i;
      if (col < N) f((wg_d2 *)(c + col), y, r);
    }
    if (TN & 1) {
      const int col = n0 + 16 * (TN - 1) + i;
      if (col < N) f1(c + col, TN - 1, r);
    }
  }
}

template <int TM, int TN>
__device__ __forceinline__ void wg_zero(wg_d4 (&acc)[TM][TN]) {
#pragma unroll
  for (int x = 0; x < TM; ++x)
#pragma unroll
    for (int y = 0; y < TN; ++y) acc[x][y] = wg_d4{0.0, 0.0, 0.0, 0.0};
}

// c = tile row x of C
template <int TM, int TN>
__device__ __forceinline__ void wg_read(double *C, long long rs, int m0, int M, int n0, int N, int lane, int x,
                                        wg_d4 (&c)[TN]) {
#pragma unroll
  for (int y = 0; y < TN; ++y) c[y] = wg_d4{0.0, 0.0, 0.0, 0.0};
  wg_each<TM, TN>(
      C, rs, m0, M, n0, N, lane, x,
      [&](wg_d2 *p, int y, int r) {
        const wg_d2 v = *p;
        c[y][r] = v[0];
        c[y + 1][r] = v[1];
      },
      [&](double *p, int y, int r) { c[y][r] = *p; });
}

// tile row x of C = c
template <int TM, int TN>
__device__ __forceinline__ void wg_write(double *C, long long rs, int m0, int M, int n0, int N, int lane, int x,
                                         const wg_d4 (&c)[TN]) {
  wg_each<TM, TN>(
      C, rs, m0, M, n0, N, lane, x, [&](wg_d2 *p, int y, int r) { *p = wg_d2{c[y][r], c[y + 1][r]}; },
      [&](double *p, int y, int r) { *p = c[y][r]; });
}

// C = acc, or C += acc: the reads of a tile row are all issued, and the row
// before is written, ahead of their use (one by one, each read would wait
// behind a write)
template <int TM, int TN>
__device__ __forceinline__ void wg_store(double *C, long long rs, int m0, int M, int n0, int N, int lane,
                                         bool add, const wg_d4 (&acc)[TM][TN]) {
  if (!add) {
#pragma unroll
    for (int x = 0; x < TM; ++x) wg_write<TM, TN>(C, rs, m0, M, n0, N, lane, x, acc[x]);
    return;
  }
  wg_d4 c[2][TN];
  wg_read<TM, TN>(C, rs, m0, M, n0, N, lane, 0, c[0]);
#pragma unroll
  for (int x = 0; x < TM; ++x) {
    if (x + 1 < TM) wg_read<TM, TN>(C, rs, m0, M, n0, N, lane, x + 1, c[(x + 1) & 1]);
#pragma unroll
    for (int y = 0; y < TN; ++y) c[x & 1][y] += acc[x][y];
    wg_write<TM, TN>(C, rs, m0, M, n0, N, lane, x, c[x & 1]);
  }
}

}  // namespace pamd
