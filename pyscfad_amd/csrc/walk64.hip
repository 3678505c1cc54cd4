// Kernels of the batched FP64 walk (walk64.h).
//
// Measured on one MI355X against the one-triple walk (25 launches and two
// streams per triple): E(T) + VJP o4/v16 4.5 -> 0.35 ms, o8/v40 40.4 -> 1.19 ms,
// o11/v77 160 -> 16.0 ms, o16/v160 1123 -> 490 ms; energy o5/v19 1.34 -> 0.096 ms;
// pair energies o16/v160 189 -> 118 ms.  Small sizes were bound by launches, odd
// ones by the register-staged engine, o16/v160 by short contractions (K = v) on
// padded tiles.  At o16/v160 the contractions now run at 61-64 TFLOP/s of their
// unpadded work (a large rocBLAS product: 72.6; the FP64 MFMA rate at the clock it
// holds there, 2.2 GHz: 72), W build 5 x 2 tiles, VT's adjoint 5 x 3 and TB's 5 x 4
// (11 column tiles padded to 12).
#include <algorithm>
#include "engine_staging.h"
#include "vr_layout.h"
#include "walk64.h"
#include "wave_gemm.h"

namespace pamd {

// ---------------------------------------------------------------------------
// padded inputs
// ---------------------------------------------------------------------------
// VT: a 32 x 32 tile (q, k) of one (x, p) per workgroup.  Full ovvv rows run
// along q, VT rows along k, so the tile is turned in LDS; packed ovvv and the
// t2 part are read along whichever index is contiguous.
__device__ __forceinline__ void prep_vt(const WalkDims &d, const double *__restrict__ ovvv, int packed,
                                        const double *__restrict__ t2, double *__restrict__ VT, int bq, int bk,
                                        int bz, int nz, double (*tile)[33]) {
  const int o = d.o, v = d.v, vp = d.vp, up = d.up;
  const int q0 = bq * 32, k0 = bk * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const size_t npair = (size_t)v * (v + 1) / 2;
  for (int xp = bz; xp < o * vp; xp += nz) {
    const int x = xp / vp, p = xp - x * vp;
    // tile[k][q], lanes along q
    for (int r = ty; r < 32; r += 8) {
      const int k = k0 + r, q = q0 + tx;
      double val = 0.0;
      if (p < v && q < v && k < v + o) {
        if (k >= v) {
          val = t2[(((size_t)x * o + (k - v)) * v + p) * v + q];
        } else if (!packed) {
          val = ovvv[(((size_t)x * v + p) * v + k) * v + q];
        } else if (q <= k) {
          val = ovvv[((size_t)x * v + p) * npair + (size_t)k * (k + 1) / 2 + q];
        }
      }
      tile[r][tx] = val;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
      const int q = q0 + r, k = k0 + tx;
      if (q < vp && k < up) {
        double val = tile[tx][r];
        if (packed && p < v && q < v && k < v && q > k)
          val = ovvv[((size_t)x * v + p) * npair + (size_t)q * (q + 1) / 2 + k];
        VT[((size_t)x * vp + p) * d.sp + (size_t)q * up + k] = val;
      }
    }
    __syncthreads();
  }
}

// TB (turned: TBt[z][y][k][r] = TB[z][y][r][k])
__device__ __forceinline__ void prep_tb(const WalkDims &d, const double *__restrict__ t2,
                                        const double *__restrict__ ovoo, double *__restrict__ out, bool turned,
                                        unsigned blk, unsigned nblk) {
  const int o = d.o, v = d.v, vp = d.vp, up = d.up;
  const size_t total = (size_t)o * o * vp * up;
  const int fast = turned ? vp : up, slow = turned ? up : vp;
  for (size_t t = (size_t)blk * 256 + threadIdx.x; t < total; t += (size_t)nblk * 256) {
    const int x = (int)(t % fast);
    const size_t u = t / fast, zy = u / slow;
    const int y = (int)(u % slow);
    const int k = turned ? y : x, r = turned ? x : y;
    double val = 0.0;
    if (r < v && k < v)
      val = t2[(zy * v + r) * v + k];
    else if (r < v && k < v + o)
      val = -ovoo[(((zy / o) * v + r) * o + (k - v)) * o + zy % o];
    out[t] = val;
  }
}

// OVS[x][y][p][q] = ovov[x,p,y,q] + ovov[y,q,x,p], or (amp) T2S[x][y][p][q] =
// t2[x,y,p,q] + t2[y,x,q,p]: the transposed term goes through LDS.
__device__ __forceinline__ void prep_sym(const WalkDims &d, const double *__restrict__ ovov,
                                         const double *__restrict__ t2, double *__restrict__ dst, bool amp,
                                         int ntile, int blk, double (*tile)[33]) {
  const int o = d.o, v = d.v, vp = d.vp;
  const int xy = blk / (ntile * ntile), tl = blk - xy * ntile * ntile;
  const int x = xy / o, y = xy % o;
  const int p0 = (tl / ntile) * 32, q0 = (tl % ntile) * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  auto src = [&](int xx, int pp, int yy, int qq) {
    return amp ? t2[(((size_t)xx * o + yy) * v + pp) * v + qq]
               : ovov[(((size_t)xx * v + pp) * o + yy) * v + qq];
  };
  for (int r = ty; r < 32; r += 8) {
    const int q = q0 + r, p = p0 + tx;
    tile[r][tx] = (q < v && p < v) ? src(y, q, x, p) : 0.0;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int p = p0 + r, q = q0 + tx;
    if (p >= vp || q >= vp) continue;
    const double a = (p < v && q < v) ? src(x, p, y, q) + tile[tx][r] : 0.0;
    dst[((size_t)xy * vp + p) * vp + q] = a;
  }
}

__device__ __forceinline__ void prep_small(const WalkDims &d, const double *mo, const double *t1,
                                           const double *fvo, double *t1p, double *fvop, double *mop, int t) {
  const int o = d.o, v = d.v, vp = d.vp;
  if (t < o * vp) {
    const int i = t / vp, a = t - i * vp;
    t1p[t] = a < v ? t1[(size_t)i * v + a] : 0.0;
    // fvo is (v, o): the padding is one block at its end
    if (fvo) fvop[t] = t < v * o ? fvo[t] : 0.0;
  }
  // padded orbitals repeat the last energy: any denominator that is not zero
  if (t < o + vp) mop[t] = mo[min(t, o + v - 1)];
}

// the triples of pair t = i o + j, in closed form: the triples before (i, j, j)
__device__ __forceinline__ void prep_triples(int o, int shard, int nshards, const WalkBatches &wb, int *tri, int t) {
  const int i = t / o, j = t % o;
  if (j < i) return;
  // triples with first index < i: sum_{x<i} ((o-x)(o-x+1)/2 - 1)
  auto cum = [](long long n) { return n * (n + 1) * (n + 2) / 6; };  // sum_{y<=n} y(y+1)/2
  long long w = cum(o) - cum(o - i) - i;
  // same i, second index < j: sum_{y=i}^{j-1} (o - y), less (i, i, i)
  w += (long long)(j - i) * o - ((long long)j * (j - 1) / 2 - (long long)i * (i - 1) / 2);
  if (j > i) w -= 1;
  for (int k = (i == j ? j + 1 : j); k < o; ++k, ++w)
    if (w % nshards == shard) {
      const long long t = w / nshards, run = t / kWalkRun;
      tri[run % wb.count * wb.cap + run / wb.count * kWalkRun + t % kWalkRun] = i | (j << 10) | (k << 20);
    }
}

__device__ __forceinline__ void prep_pairs(int o, int *tri, int t) {
  const int j = t / o, k = t % o;
  if (k < j) return;
  int *p = tri + (size_t)(j * o - j * (j - 1) / 2 + k - j) * o;
  for (int l = 0; l < o; ++l) p[l] = l | (j << 10) | (k << 20);
}

// The pieces do not depend on each other: a workgroup's number says which it
// works on.  (Eight launches at o4/v16, each 3 us of a call that takes 100.)
__global__ __launch_bounds__(256) void k_walk_prep(WalkPrep A) {
  __shared__ double tile[32][33];
  const WalkDims &d = A.d;
  unsigned blk = blockIdx.x;
  if (blk < A.blocks[0]) {
    const unsigned nq = (d.vp + 31) / 32, nk = (d.up + 31) / 32, r = blk / nq;
    prep_vt(d, A.ovvv, A.packed, A.t2, A.VT, (int)(blk - r * nq), (int)(r % nk), (int)(r / nk),
            (int)(A.blocks[0] / (nq * nk)), tile);
    return;
  }
  blk -= A.blocks[0];
  if (blk < A.blocks[1]) {  // TBt, and with an adjoint TB
    const unsigned n = A.TB ? A.blocks[1] / 2 : A.blocks[1];
    const bool turned = blk < n;
    prep_tb(d, A.t2, A.ovoo, turned ? A.TBt : A.TB, turned, turned ? blk : blk - n, n);
    return;
  }
  blk -= A.blocks[1];
  if (blk < A.blocks[2]) {
    const unsigned n = A.blocks[2] / 2;
    const bool amp = blk >= n;
    prep_sym(d, A.ovov, A.t2, amp ? A.T2S : A.OVS, amp, (d.vp + 31) / 32, (int)(amp ? blk - n : blk), tile);
    return;
  }
  blk -= A.blocks[2];
  const int o = d.o, ns = o * d.vp + d.vp + o;
  long long t = (long long)blk * 256 + threadIdx.x;
  if (t < ns) {
    prep_small(d, A.mo, A.t1, A.fvo, A.t1p, A.fvop, A.mop, (int)t);
    return;
  }
  t -= ns;
  if (t < A.norb) {
    put_orbit(t, A.orb);
    return;
  }
  t -= A.norb;
  if (t < o * o) {
    if (A.pairs)
      prep_pairs(o, A.tri, (int)t);
    else
      prep_triples(o, A.shard, A.nshards, A.wb, A.tri, (int)t);
    return;
  }
  t -= o * o;
#pragma unroll
  for (int z = 0; z < 2; ++z) {
    if (t < (long long)A.nzero[z]) {
      A.zero[z][t] = 0.0;
      return;
    }
    t -= (long long)A.nzero[z];
  }
}

hipError_t launch_walk_prep(WalkPrep a, hipStream_t s) {
  const WalkDims &d = a.d;
  const unsigned nq = (d.vp + 31) / 32, nk = (d.up + 31) / 32;
  const size_t ntb = (size_t)d.o * d.o * d.vp * d.up;
  a.blocks[0] = a.VT ? nq * nk * (unsigned)std::min(d.o * d.vp, 65535) : 0;
  a.blocks[1] = a.TBt ? (unsigned)std::min<size_t>((ntb + 255) / 256, 262144) * (a.TB ? 2 : 1) : 0;
  a.blocks[2] = 2u * (unsigned)(d.o * d.o) * nq * nq;
  const long long rest = (long long)d.o * d.vp + d.vp + d.o + a.norb + (long long)d.o * d.o +
                         (long long)(a.nzero[0] + a.nzero[1]);
  a.blocks[3] = (unsigned)((rest + 255) / 256);
  const long long total = (long long)a.blocks[0] + a.blocks[1] + a.blocks[2] + a.blocks[3];
  if (total >= (1LL << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_walk_prep, dim3((unsigned)total), dim3(256), 0, s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// contractions: one wave per TM x TN block of 16 x 16 tiles, four consecutive
// blocks (the same rows, neighbouring columns where there are several) per
// workgroup
// ---------------------------------------------------------------------------
struct WalkTile {
  int batch, fixed, m0, n0;
  bool ok;
};

// work item -> (batch, fixed index, row block, column block), columns fastest
template <int TM, int TN>
__device__ __forceinline__ WalkTile walk_tile(int nfix, int M, int N, long long total) {
  const int nm = (M + 16 * TM - 1) / (16 * TM), nn = (N + 16 * TN - 1) / (16 * TN);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int w = xcd_remap(blockIdx.x, gridDim.x) * 4 + wave;
  WalkTile t;
  t.ok = w < total;
  t.n0 = (w % nn) * 16 * TN;
  w /= nn;
  t.m0 = (w % nm) * 16 * TM;
  w /= nm;
  t.fixed = w % nfix;
  t.batch = w / nfix;
  return t;
}

struct WalkArgs {
  WalkDims d;
  const double *VT, *TB;
  double *W, *out;
  const int *tri;
  int nb, S;
};

__device__ __forceinline__ void walk_ijk(const int *tri, int b, int &i, int &j, int &k) {
  const int t = tri[b];
  i = t & 1023;
  j = (t >> 10) & 1023;
  k = t >> 20;
}

// W build, pass 0 at fixed b (rows a, columns c): the two products whose TB factor
// is over c (form 0), then the two over a (form 1); pass 1 at fixed a (rows b,
// columns c): the two over b, added (form 2).  VT is K-contiguous, and TB is read
// from its transpose, row-contiguous: 16 lanes of a K-contiguous load lie in 16
// rows, and L1 takes the 64 lanes one by one (64 accesses of a 1 KB load, against
// 16).  With both operands K-contiguous that, not the MFMAs, bound 5 x 2 tiles
// (51 TFLOP/s at o16/v160).
template <int FORM>
struct GenW {
  const double *VT, *TBt;
  long long vp, up, sp, o, x;
  int i, j, k, q;
  __device__ __forceinline__ const double *V(int y) const { return VT + y * vp * sp; }
  __device__ __forceinline__ const double *T(int z, int y) const { return TBt + (z * o + y) * vp * up; }
  __device__ __forceinline__ bool next(WSeg &s) {
    if (q >= 2) return false;
    s.nk = (int)(up >> 3);
    s.nout = 1;
    s.aos = s.bos = 0;
    const double *tb, *v;
    long long vs = up;
    if (FORM == 0) {  // VT[i][a][b] TB[k,j][c], VT[j][b][a] TB[k,i][c]
      v = q == 0 ? V(i) + x * up : V(j) + x * sp;
      if (q == 0) vs = sp;
      tb = q == 0 ? T(k, j) : T(k, i);
    } else if (FORM == 1) {  // TB[i,k][a] VT[j][b][c], TB[i,j][a] VT[k][c][b]
      v = q == 0 ? V(j) + x * sp : V(k) + x * up;
      if (q == 1) vs = sp;
      tb = q == 0 ? T(i, k) : T(i, j);
    } else {  // TB[j,k][b] VT[i][a][c], TB[j,i][b] VT[k][c][a]
      v = q == 0 ? V(i) + x * sp : V(k) + x * up;
      if (q == 1) vs = sp;
      tb = q == 0 ? T(j, k) : T(j, i);
    }
    (FORM == 0 ? s.A : s.B) = v;
    (FORM == 0 ? s.ar : s.br) = vs;
    (FORM == 0 ? s.ak : s.bk) = 1;
    (FORM == 0 ? s.B : s.A) = tb;
    (FORM == 0 ? s.br : s.ar) = 1;
    (FORM == 0 ? s.bk : s.ak) = vp;
    ++q;
    return true;
  }
};

template <int TM, int TN, int PASS>
__global__ __launch_bounds__(256, 2) void k_walk_w(WalkArgs A, long long total) {
  const int vp = A.d.vp;
  const WalkTile t = walk_tile<TM, TN>(vp, vp, vp, total);
  if (!t.ok) return;
  const int lane = threadIdx.x & 63;
  int i, j, k;
  walk_ijk(A.tri, t.batch, i, j, k);
  const long long up = A.d.up, sp = A.d.sp, o = A.d.o;
  const long long v2 = A.d.ws, rs = PASS == 0 ? v2 : vp;
  double *C = A.W + t.batch * v2 * vp + t.fixed * (PASS == 0 ? vp : v2);
  const int chunks = 2 * (int)(up >> 3);
  wg_d4 acc[TM][TN];
  wg_zero<TM, TN>(acc);
  if (PASS == 0) {
    GenW<0> g0{A.VT, A.TB, vp, up, sp, o, t.fixed, i, j, k, 0};
    wg_accumulate<TM, TN, true, false>(g0, chunks, t.m0, vp, t.n0, vp, lane, acc);
    GenW<1> g1{A.VT, A.TB, vp, up, sp, o, t.fixed, i, j, k, 0};
    wg_accumulate<TM, TN, false, true>(g1, chunks, t.m0, vp, t.n0, vp, lane, acc);
  } else {
    GenW<2> g{A.VT, A.TB, vp, up, sp, o, t.fixed, i, j, k, 0};
    wg_accumulate<TM, TN, false, true>(g, chunks, t.m0, vp, t.n0, vp, lane, acc);
  }
  wg_store<TM, TN>(C, rs, t.m0, vp, t.n0, vp, lane, PASS == 1, acc);
}

// Adjoint of VT[x]: the batch's triples that hold x, in order.  Pass 0: x = i
// and x = j, at a fixed first virtual index p of VTb[x][p][q], rows q; pass 1:
// x = k, at a fixed second index q, rows p (= c, the contiguous index of Wbar).
// Per triple two runs over one virtual index, h = 0 and 1; in pass 0 the first
// has Wbar K-contiguous and the second row-contiguous.
struct GenVT {
  const double *W, *TB;
  const int *ent;  // LDS: slot | second << 31 of every run pair
  const int *tri;
  long long vp, up, v2, o, x;
  int n, e, h, step, pass;  // step 1: both runs of an entry, 2: run h only
  __device__ __forceinline__ const double *T(int z, int y) const { return TB + (z * o + y) * vp * up; }
  __device__ __forceinline__ bool next(WSeg &s) {
    if (e >= n) return false;
    const int en = __builtin_amdgcn_readfirstlane(ent[e]);
    const int slot = en & 0x7fffffff;
    const bool second = en < 0;
    int i, j, k;
    walk_ijk(tri, slot, i, j, k);
    const double *w = W + slot * v2 * vp;
    s.br = 1;
    s.bk = up;
    s.nk = (int)(vp >> 3);
    s.nout = 1;
    s.aos = s.bos = 0;
    if (pass == 0) {
      if (!second) {  // x = i, fixed a
        s.A = w + x * v2;
        s.ar = h ? 1 : vp;
        s.ak = h ? vp : 1;
        s.B = h ? T(j, k) : T(k, j);
      } else {  // x = j, fixed b
        s.A = w + x * vp;
        s.ar = h ? 1 : v2;
        s.ak = h ? v2 : 1;
        s.B = h ? T(i, k) : T(k, i);
      }
    } else {  // x = k, rows c: fixed a, K = b; then fixed b, K = a
      s.A = w + x * (h ? vp : v2);
      s.ar = 1;
      s.ak = h ? v2 : vp;
      s.B = h ? T(i, j) : T(j, i);
    }
    if (step == 2 || h) ++e;
    if (step == 1) h ^= 1;
    return true;
  }
};

template <int TM, int TN, int PASS>
__global__ __launch_bounds__(256, 2) void k_walk_vtb(WalkArgs A, long long total, int first) {
  __shared__ int ents[4][2 * kWalkMaxBatch];
  const int vp = A.d.vp, up = A.d.up;
  // each XCD takes an eighth of the fixed index for every x, the x with the
  // most triples first
  WalkTile t = walk_tile<TM, TN>(vp >> 3, vp, up, total);
  if (!t.ok) return;
  t.fixed += t.batch / A.d.o * (vp >> 3);
  t.batch = PASS == 0 ? t.batch % A.d.o : A.d.o - 1 - t.batch % A.d.o;
  const int lane = threadIdx.x & 63;
  int *ent = ents[threadIdx.x >> 6];
  const int x = t.batch;
  int n = 0;
  for (int b0 = 0; b0 < A.nb; b0 += 64) {
    const int b = b0 + lane;
    const int w = b < A.nb ? A.tri[b] : -1;
    const int i = w & 1023, j = (w >> 10) & 1023, k = w >> 20;
    const bool m0 = w >= 0 && (PASS == 0 ? i == x : k == x), m1 = w >= 0 && PASS == 0 && j == x;
    const unsigned long long lo = (1ULL << lane) - 1;
    const unsigned long long c0 = __ballot(m0), c1 = __ballot(m1);
    if (m0) ent[n + __popcll(c0 & lo)] = b;
    n += __popcll(c0);
    if (m1) ent[n + __popcll(c1 & lo)] = b | (1 << 31);
    n += __popcll(c1);
  }
  n = __builtin_amdgcn_readfirstlane(n);
  if (n == 0 && !(PASS == 0 && first)) return;
  __builtin_amdgcn_wave_barrier();
  const long long rs = PASS == 0 ? up : A.d.sp;
  double *C = A.out + x * vp * A.d.sp + t.fixed * (PASS == 0 ? A.d.sp : up);
  wg_d4 acc[TM][TN];
  wg_zero<TM, TN>(acc);
  const int chunks = n * (vp >> 3);
  if (PASS == 0) {
    GenVT g0{A.W, A.TB, ent, A.tri, vp, up, A.d.ws, A.d.o, t.fixed, n, 0, 0, 2, 0};
    wg_accumulate<TM, TN, true, false>(g0, chunks, t.m0, vp, t.n0, up, lane, acc);
    GenVT g1{A.W, A.TB, ent, A.tri, vp, up, A.d.ws, A.d.o, t.fixed, n, 0, 1, 2, 0};
    wg_accumulate<TM, TN, false, false>(g1, chunks, t.m0, vp, t.n0, up, lane, acc);
  } else {
    GenVT g{A.W, A.TB, ent, A.tri, vp, up, A.d.ws, A.d.o, t.fixed, n, 0, 0, 1, 1};
    wg_accumulate<TM, TN, false, false>(g, 2 * chunks, t.m0, vp, t.n0, up, lane, acc);
  }
  wg_store<TM, TN>(C, rs, t.m0, vp, t.n0, up, lane, PASS == 1 || !first, acc);
}

// Adjoint of TB, per triple and piece: rows over one virtual index of Wbar, K
// over the other two (outer, inner), a part of the outer one per work item.
struct GenTB {
  WSeg s0;
  bool more;
  __device__ __forceinline__ bool next(WSeg &s) {
    s = s0;
    const bool m = more;
    more = false;
    return m;
  }
};

template <int TM, int TN, int RC>
__global__ __launch_bounds__(256, 2) void k_walk_tbb(WalkArgs A, long long total) {
  const long long vp = A.d.vp, up = A.d.up, v2 = A.d.ws, sp_ = A.d.sp;
  // work: triple, then (piece of this form, part), rows, columns
  constexpr int NP = RC ? 2 : 4;
  const WalkTile t = walk_tile<TM, TN>(NP * A.S, (int)vp, (int)up, total);
  if (!t.ok) return;
  const int lane = threadIdx.x & 63;
  const int pc = t.fixed / A.S, sp = t.fixed - pc * A.S;
  const int pr = RC ? 2 * pc : (pc < 2 ? 2 * pc + 1 : pc + 2);  // 0, 2 / 1, 3, 4, 5
  int i, j, k;
  walk_ijk(A.tri, t.batch, i, j, k);
  const int per = ((int)vp + A.S - 1) / A.S;
  const int u0 = sp * per, u1 = min((int)vp, u0 + per);
  const double *w = A.W + t.batch * v2 * vp;
  WSeg s;
  s.br = 1;
  s.nk = (int)(vp >> 3);
  s.nout = u1 - u0;
  const int x = pr < 2 ? i : (pr < 4 ? j : k);
  s.B = A.VT + x * vp * sp_;
  switch (pr) {
    case 0:  // rows c, K = (a, b), VT[i][a][b]
      s.A = w; s.ar = 1; s.ak = vp; s.aos = v2; s.bk = up; s.bos = sp_;
      break;
    case 2:  // rows c, K = (b, a), VT[j][b][a]
      s.A = w; s.ar = 1; s.ak = v2; s.aos = vp; s.bk = up; s.bos = sp_;
      break;
    case 1:  // rows b, K = (a, c), VT[i][a][c]
      s.A = w; s.ar = vp; s.ak = 1; s.aos = v2; s.bk = up; s.bos = sp_;
      break;
    case 3:  // rows a, K = (b, c), VT[j][b][c]
      s.A = w; s.ar = v2; s.ak = 1; s.aos = vp; s.bk = up; s.bos = sp_;
      break;
    case 4:  // rows b, K = (a, c), VT[k][c][a]
      s.A = w; s.ar = vp; s.ak = 1; s.aos = v2; s.bk = sp_; s.bos = up;
      break;
    default:  // rows a, K = (b, c), VT[k][c][b]
      s.A = w; s.ar = v2; s.ak = 1; s.aos = vp; s.bk = sp_; s.bos = up;
      break;
  }
  s.A += u0 * s.aos;
  s.B += u0 * s.bos;
  GenTB g{s, u1 > u0};
  double *C = A.out + (((size_t)t.batch * 6 + pr) * A.S + sp) * vp * up;
  wg_d4 acc[TM][TN];
  wg_zero<TM, TN>(acc);
  wg_accumulate<TM, TN, !RC, false>(g, s.nk * s.nout, t.m0, (int)vp, t.n0, (int)up, lane, acc);
  wg_store<TM, TN>(C, up, t.m0, (int)vp, t.n0, (int)up, lane, false, acc);
}

// Block shape for nprod M x N products: the work of the busiest SIMD (blocks
// per SIMD, rounded up, times their tiles), weighted by what L1 takes to feed it:
// (TM + TN) / (TM TN) loads per MFMA pair, free up to 0.8 (measured at o16/v160
// and o8/v40: 5 x 2 and 3 x 3 tiles run at the rate of 5 x 3, 3 x 1 at half of
// it).  most: tiles that a wave of that kernel holds at two waves per SIMD.
struct WalkShape {
  int tm, tn;
};
constexpr WalkShape kWalkShapes[] = {{5, 4}, {4, 4}, {5, 3}, {5, 2}, {4, 3}, {3, 3}, {4, 2},
                                     {3, 2}, {2, 2}, {3, 1}, {2, 1}, {1, 1}};
static WalkShape walk_shape(long long nprod, int M, int N, int most) {
  WalkShape best = {1, 1};
  double cost = 1e300;
  for (const WalkShape &w : kWalkShapes) {
    if (w.tm * w.tn > most) continue;
    const long long blocks = nprod * ((M + 16 * w.tm - 1) / (16 * w.tm)) * ((N + 16 * w.tn - 1) / (16 * w.tn));
    const double rounds = (double)((blocks + 1023) / 1024);
    const double loads = (double)(w.tm + w.tn) / (w.tm * w.tn);
    const double c = rounds * w.tm * w.tn * std::max(1.0, 1.25 * loads);
    if (c < cost) {
      cost = c;
      best = w;
    }
  }
  return best;
}

#define WALK_SHAPES(X) \
  X(5, 4) X(4, 4) X(5, 3) X(5, 2) X(4, 3) X(3, 3) X(4, 2) X(3, 2) X(2, 2) X(3, 1) X(2, 1) X(1, 1)

template <class F>
static hipError_t walk_launch(long long nprod, int M, int N, int most, F &&f) {
  const WalkShape w = walk_shape(nprod, M, N, most);
  const long long total = nprod * ((M + 16 * w.tm - 1) / (16 * w.tm)) * ((N + 16 * w.tn - 1) / (16 * w.tn));
  if (total > (1LL << 31) - 8) return hipErrorInvalidValue;
  f(w, total, dim3((unsigned)((total + 3) / 4)));
  return hipGetLastError();
}

hipError_t launch_walk_w(const WalkDims &d, const double *VT, const double *TBt, double *W, const int *tri,
                         int nb, hipStream_t s) {
  WalkArgs A{d, VT, TBt, W, nullptr, tri, nb, 1};
  const long long nprod = (long long)nb * d.vp;
  return walk_launch(nprod, d.vp, d.vp, 20, [&](WalkShape w, long long total, dim3 grid) {
#define X(TM, TN)                                                                          \
  if (w.tm == TM && w.tn == TN) {                                                          \
    hipLaunchKernelGGL((k_walk_w<TM, TN, 0>), grid, dim3(256), 0, s, A, total);            \
    hipLaunchKernelGGL((k_walk_w<TM, TN, 1>), grid, dim3(256), 0, s, A, total);            \
  }
    WALK_SHAPES(X)
#undef X
  });
}

hipError_t launch_walk_vtb(const WalkDims &d, const double *Wb, const double *TB, double *VTb,
                           const int *tri, int nb, bool first, hipStream_t s) {
  if (nb > kWalkMaxBatch) return hipErrorInvalidValue;
  WalkArgs A{d, nullptr, TB, const_cast<double *>(Wb), VTb, tri, nb, 1};
  const long long nprod = (long long)d.o * d.vp;
  return walk_launch(nprod, d.vp, d.up, 16, [&](WalkShape w, long long total, dim3 grid) {
#define X(TM, TN)                                                                               \
  if (w.tm == TM && w.tn == TN) {                                                               \
    hipLaunchKernelGGL((k_walk_vtb<TM, TN, 0>), grid, dim3(256), 0, s, A, total, first ? 1 : 0); \
    hipLaunchKernelGGL((k_walk_vtb<TM, TN, 1>), grid, dim3(256), 0, s, A, total, 0);             \
  }
    WALK_SHAPES(X)
#undef X
  });
}

hipError_t launch_walk_tbb(const WalkDims &d, const double *Wb, const double *VT, double *part,
                           const int *tri, int nb, int S, hipStream_t s) {
  WalkArgs A{d, VT, nullptr, const_cast<double *>(Wb), part, tri, nb, S};
  hipError_t e = walk_launch(2LL * nb * S, d.vp, d.up, 20, [&](WalkShape w, long long total, dim3 grid) {
#define X(TM, TN)              \
  if (w.tm == TM && w.tn == TN) \
    hipLaunchKernelGGL((k_walk_tbb<TM, TN, 1>), grid, dim3(256), 0, s, A, total);
    WALK_SHAPES(X)
#undef X
  });
  if (e != hipSuccess) return e;
  return walk_launch(4LL * nb * S, d.vp, d.up, 20, [&](WalkShape w, long long total, dim3 grid) {
#define X(TM, TN)              \
  if (w.tm == TM && w.tn == TN) \
    hipLaunchKernelGGL((k_walk_tbb<TM, TN, 0>), grid, dim3(256), 0, s, A, total);
    WALK_SHAPES(X)
#undef X
  });
}

// ---------------------------------------------------------------------------
// V-bar reductions of a batch (the blocks are listed at k_vr, which a single
// triple uses: there the sums must be split to fill the GPU).  Vbar is read
// twice and little else, so the work is in not adding barriers and idle lanes to
// that: one wave owns one a and walks the rows b, its sums over b stay in
// registers, and rows of at most 64 (32) elements run two (four) to a wave, two
// elements to a lane.  k_vr spends most of its time in the LDS combines of eight
// waves that see v / 8 rows each.  Measured, o11/v77, 140 triples: 1380 -> 420 us.
// ---------------------------------------------------------------------------
typedef double vr_d2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double vr_wave_sum(double x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}

// sums of four values over G lanes; lane G / 4 q of them ends up with value q
template <int G>
__device__ __forceinline__ double group_sum4(double v0, double v1, double v2, double v3) {
  const int lane = threadIdx.x & 63;
  const bool hi = (lane & (G / 2)) != 0, mid = (lane & (G / 4)) != 0;
  double x = hi ? v2 : v0, y = hi ? v3 : v1;
  x += __shfl_xor(hi ? v0 : v2, G / 2, 64);
  y += __shfl_xor(hi ? v1 : v3, G / 2, 64);
  double z = mid ? y : x;
  z += __shfl_xor(mid ? x : y, G / 4, 64);
#pragma unroll
  for (int off = G / 8; off > 0; off >>= 1) z += __shfl_xor(z, off, 64);
  return z;
}

// G lanes per row, Q pairs of columns per lane; all extents multiples of 8
template <int G, int Q, bool FVO>
__device__ __forceinline__ void vr_rows(const VRArgs &A, double *R, const double *Vb, int i, int j, int k, int a) {
  constexpr int RP = 64 / G, U = Q > 2 ? 2 : (8 / RP < 4 ? 8 / RP : 4);
  const int lane = threadIdx.x & 63, row = lane / G, l = lane % G;
  const int o = A.o, v = A.v;
  const size_t vv = (size_t)v * v;
  auto pair = [&](const double *arr, int x, int y) { return arr + ((size_t)x * o + y) * vv; };
  vr_d2 c1[Q], c2[Q], c3[Q], c4[FVO ? Q : 1], r3[Q], pk[Q], fk[Q], r4[FVO ? Q : 1];
  int c[Q];
  bool ok[Q];
  const vr_d2 zero = {0.0, 0.0};
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int at = 2 * (l + G * q);
    ok[q] = at < v;
    c[q] = ok[q] ? at : v - 2;  // (lanes past the row read its end, times zero)
    c1[q] = ok[q] ? *(const vr_d2 *)(A.t1 + (size_t)k * v + c[q]) : zero;
    c2[q] = ok[q] ? *(const vr_d2 *)(pair(A.ovs, i, k) + (size_t)a * v + c[q]) : zero;
    c3[q] = ok[q] ? *(const vr_d2 *)(pair(A.t2s, i, k) + (size_t)a * v + c[q]) : zero;
    if (FVO) c4[q] = ok[q] ? vr_d2{A.fvo[(size_t)c[q] * o + k], A.fvo[(size_t)(c[q] + 1) * o + k]} : zero;
    r3[q] = pk[q] = fk[q] = zero;
    if (FVO) r4[q] = zero;
  }
  const double *sij = pair(A.ovs, i, j) + (size_t)a * v, *tij = pair(A.t2s, i, j) + (size_t)a * v;
  const double *sjk = pair(A.ovs, j, k), *tjk = pair(A.t2s, j, k), *x0 = Vb + (size_t)a * vv;
  double t1i = 0.0, fvoi = 0.0;
  for (int b0 = 0; b0 < v; b0 += RP * U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int b = b0 + u * RP + row;
      const double t1j = A.t1[(size_t)j * v + b], S1 = sij[b], T1 = tij[b];
      const double fj = FVO ? A.fvo[(size_t)b * o + j] : 0.0;
      double sr1 = 0.0, sr2 = 0.0, spj = 0.0, sfj = 0.0;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const size_t at = (size_t)b * v + c[q];
        const vr_d2 x = *(const vr_d2 *)(x0 + at);
        vr_d2 s = *(const vr_d2 *)(sjk + at), t = *(const vr_d2 *)(tjk + at);
        s = ok[q] ? s : zero;
        t = ok[q] ? t : zero;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          sr1 = fma(x[e], c1[q][e], sr1);
          spj = fma(x[e], c2[q][e], spj);
          sfj = fma(x[e], c3[q][e], sfj);
          r3[q][e] = fma(x[e], t1j, r3[q][e]);
          pk[q][e] = fma(x[e], S1, pk[q][e]);
          fk[q][e] = fma(x[e], T1, fk[q][e]);
          t1i = fma(x[e], s[e], t1i);
          fvoi = fma(x[e], t[e], fvoi);
          if (FVO) {
            sr2 = fma(x[e], c4[q][e], sr2);
            r4[q][e] = fma(x[e], fj, r4[q][e]);
          }
        }
      }
      const double z = group_sum4<G>(sr1, sr2, spj, sfj);
      if (l % (G / 4) == 0) {
        const int q = l / (G / 4);
        if (FVO || q != 1) R[(size_t)(q < 2 ? q : q + 6) * vv + (size_t)a * v + b] = z;
      }
    }
  }
  // the rows of a wave's RP groups
  auto across = [&](double x) {
#pragma unroll
    for (int off = 32; off >= G; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
  };
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    auto put2 = [&](int blk, const vr_d2 &s) {
      const vr_d2 x = {across(s[0]), across(s[1])};
      if (row == 0 && ok[q]) *(vr_d2 *)(R + (size_t)blk * vv + (size_t)a * v + c[q]) = x;
    };
    put2(2, r3[q]);
    if (FVO) put2(3, r4[q]);
    put2(6, pk[q]);
    put2(7, fk[q]);
  }
  t1i = vr_wave_sum(t1i);
  fvoi = vr_wave_sum(fvoi);
  if (lane == 0) {
    R[10 * vv + a] = t1i;
    R[10 * vv + v + a] = fvoi;
  }
}

// grid (row blocks: four a each; then sums over a: 256 positions (b, c) each), triples
template <int G, int Q, bool FVO>
__global__ __launch_bounds__(256) void k_walk_vr(VRArgs A) {
  const int v = A.v, o = A.o, nrow = (v + 3) / 4;
  const size_t vv = (size_t)v * v;
  int i, j, k;
  walk_ijk(A.tri, blockIdx.y, i, j, k);
  const double *Vb = A.Vb + (size_t)blockIdx.y * vv * v;
  double *R = A.R + (size_t)blockIdx.y * A.r_stride;
  if ((int)blockIdx.x < nrow) {
    const int a = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    vr_rows<G, Q, FVO>(A, R, Vb, i, j, k, a);  // (v is a multiple of 8: a < v)
    return;
  }
  const size_t t = (size_t)(blockIdx.x - nrow) * 256 + threadIdx.x;
  if (t >= vv) return;
  const double *x = Vb + t, *t1 = A.t1 + (size_t)i * v;
  double r5 = 0.0, r6 = 0.0;
#pragma unroll 8
  for (int a = 0; a < v; ++a) {
    const double y = x[a * vv];
    r5 = fma(y, t1[a], r5);
    if (FVO) r6 = fma(y, A.fvo[(size_t)a * o + i], r6);
  }
  R[4 * vv + t] = r5;
  if (FVO) R[5 * vv + t] = r6;
}

hipError_t launch_walk_vr(const VRArgs &a, hipStream_t s) {
  if (a.v > 512) return launch_vr(a, s);
  const size_t vv = (size_t)a.v * a.v;
  const dim3 grid((unsigned)((a.v + 3) / 4 + (vv + 255) / 256), a.nb), block(256);
#define WALK_VR(G, Q)                                                      \
  if (a.has_fvo)                                                           \
    hipLaunchKernelGGL((k_walk_vr<G, Q, true>), grid, block, 0, s, a);     \
  else                                                                     \
    hipLaunchKernelGGL((k_walk_vr<G, Q, false>), grid, block, 0, s, a)
  if (a.v <= 32) {
    WALK_VR(16, 1);
  } else if (a.v <= 64) {
    WALK_VR(32, 1);
  } else if (a.v <= 128) {
    WALK_VR(64, 1);
  } else if (a.v <= 256) {
    WALK_VR(64, 2);
  } else {
    WALK_VR(64, 4);
  }
#undef WALK_VR
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// gather
// ---------------------------------------------------------------------------
// more than one column block (v > 512): their parts of blocks 0, 1, 8, 9 and of
// the two vectors, in place (fixed order)
__global__ __launch_bounds__(256) void k_walk_vrsum(int v, double *R, size_t r_stride, int has_fvo) {
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (size_t)v * v) return;
  double *r = R + blockIdx.y * r_stride;
  r[t] = vr_csum(r, v, 0, t);
  if (has_fvo) vr_cpart(r, v, 0, 1)[t] = vr_csum(r, v, 1, t);
  vr_cpart(r, v, 0, 8)[t] = vr_csum(r, v, 8, t);
  vr_cpart(r, v, 0, 9)[t] = vr_csum(r, v, 9, t);
  if (t < (size_t)v)
    for (int q = 0; q < 2; ++q) {
      double x = 0.0;
      for (int cb = 0; cb < vr_col_blocks(v); ++cb) x += vr_part_vec(r, v, cb * kVRS, q)[t];
      vr_part_vec(r, v, 0, q)[t] = x;
    }
}

// column sums of a triple's blocks: vec[b] = {for t1[k], t1[j], t1[i], fvo[k],
// fvo[j], fvo[i]}, 64 columns per workgroup, the four waves splitting the rows
__device__ __forceinline__ void walk_cols(int v, const double *R, size_t r_stride, double *vec, int bx, int by,
                                          double (*red)[4][64]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = bx * 64 + lane;
  const double *r = R + by * r_stride;
  const size_t vv = (size_t)v * v;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  constexpr int blk[4] = {6, 8, 7, 9};
  if (c < v)
    for (int a = wave; a < v; a += 4)
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] += r[blk[q] * vv + (size_t)a * v + c];
#pragma unroll
  for (int q = 0; q < 4; ++q) red[q][wave][lane] = s[q];
  __syncthreads();
  if (wave == 0 && c < v) {
    double *d = vec + (size_t)by * 6 * v;
    constexpr int to[4] = {0, 1, 3, 4};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      d[(size_t)to[q] * v + c] = red[q][0][lane] + red[q][1][lane] + red[q][2][lane] + red[q][3][lane];
    d[2 * (size_t)v + c] = vr_part_vec(const_cast<double *>(r), v, 0, 0)[c];
    d[5 * (size_t)v + c] = vr_part_vec(const_cast<double *>(r), v, 0, 1)[c];
  }
}

// t1_bar and fvo_bar of occupied orbital blockIdx.y from the batch's vectors: 64
// columns per workgroup, the four waves splitting the triples
__global__ __launch_bounds__(256) void k_walk_t1(WalkGather G) {
  __shared__ double red[2][4][64];
  const int v = G.d.v, vp = G.d.vp, o = G.d.o, x = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = blockIdx.x * 64 + lane;
  double st = 0.0, sf = 0.0;
  if (c < v)
#pragma unroll 4
    for (int b = wave; b < G.nb; b += 4) {
      const int w = G.tri[b];
      const int i = w & 1023, j = (w >> 10) & 1023, k = w >> 20;
      const double *d = G.vec + (size_t)b * 6 * vp + c;
      if (k == x) st += d[0], sf += d[3 * (size_t)vp];
      if (j == x) st += d[(size_t)vp], sf += d[4 * (size_t)vp];
      if (i == x) st += d[2 * (size_t)vp], sf += d[5 * (size_t)vp];
    }
  red[0][wave][lane] = st;
  red[1][wave][lane] = sf;
  __syncthreads();
  if (wave != 0 || c >= v) return;
  st = (red[0][0][lane] + red[0][1][lane]) + (red[0][2][lane] + red[0][3][lane]);
  sf = (red[1][0][lane] + red[1][1][lane]) + (red[1][2][lane] + red[1][3][lane]);
  double *t = G.t1_bar + (size_t)x * v + c, *f = G.fvo_bar + (size_t)c * o + x;
  *t = 0.5 * st + (G.first ? 0.0 : *t);
  *f = 0.5 * sf + (G.first ? 0.0 : *f);
}

// t2_bar[x,y], ovov_bar[x,.,y,.] and ovoo_bar[x,.,.,y]: a workgroup holds 256
// positions (p, k) of one pair (x, y) and walks the batch's triples that write
// to it, so every position is summed by one thread in a fixed order.
__device__ __forceinline__ void walk_gather(const WalkGather &G, int nblk, int blk, int *list, int *cnt) {
  const int o = G.d.o, v = G.d.v, vp = G.d.vp, up = G.d.up;
  const int xy = blk / nblk, x = xy / o, y = xy - x * o;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // slots that write to (x, y), with the mask of their pieces
  static_assert(kWalkMaxBatch <= 256, "one slot per thread");
  int mask = 0;
  if ((int)threadIdx.x < G.nb) {
    const int w = G.tri[threadIdx.x];
    const int i = w & 1023, j = (w >> 10) & 1023, k = w >> 20;
    mask = (x == k && y == j ? 1 : 0) | (x == j && y == k ? 2 : 0) | (x == k && y == i ? 4 : 0) |
           (x == i && y == k ? 8 : 0) | (x == j && y == i ? 16 : 0) | (x == i && y == j ? 32 : 0);
  }
  const unsigned long long m = __ballot(mask != 0);
  if (lane == 0) cnt[wave] = __popcll(m);
  __syncthreads();
  int at = 0, n = 0;
  for (int w = 0; w < 4; ++w) {
    if (w < wave) at += cnt[w];
    n += cnt[w];
  }
  if (mask) list[at + __popcll(m & ((1ULL << lane) - 1))] = threadIdx.x | (mask << 16);
  __syncthreads();
  const int t = (blk - xy * nblk) * 256 + threadIdx.x;
  if (t >= vp * up) return;
  const int p = t / up, k = t - p * up;
  if (p >= v || k >= v + o) return;
  const size_t vv = (size_t)vp * vp, slab = (size_t)vp * up;
  const size_t pq = (size_t)p * vp + k, qp = (size_t)k * vp + p;
  double s = 0.0, r = 0.0;
  for (int e = 0; e < n; ++e) {
    const int b = list[e] & 0xffff, mk = list[e] >> 16;
    const double *R = G.R + b * G.r_stride;
    for (int pr = 0; pr < 6; ++pr) {
      if (!((mk >> pr) & 1)) continue;
      const double *q = G.part + ((size_t)b * 6 + pr) * G.S * slab + t;
      for (int sp = 0; sp < G.S; ++sp) s += q[sp * slab];
      if (k < v) {
        // R5, R5, R3, R3, R1, R1 over (b,c), (a,c), (a,b), transposed for even pieces
        const size_t at_ = (pr & 1) ? pq : qp;
        const size_t rb = (size_t)(pr < 2 ? 4 : (pr < 4 ? 2 : 0)) * vv;
        r += R[rb + at_];
        if (G.has_fvo) s += 0.5 * R[rb + vv + at_];
      }
    }
  }
  if (k < v) {
    double *t2 = G.t2_bar + ((size_t)xy * v + p) * v + k;
    double *ov = G.ovov_bar + (((size_t)x * v + p) * o + y) * v + k;
    *t2 = s + (G.first ? 0.0 : *t2);
    *ov = 0.5 * r + (G.first ? 0.0 : *ov);
  } else {
    double *oo = G.ovoo_bar + (((size_t)x * v + p) * o + (k - v)) * o + y;
    *oo = (G.first ? 0.0 : *oo) - s;
  }
}

// tri_e of the triple in slot b, by one wave
__device__ __forceinline__ void walk_energy(const int *tri, int o, const double *part_t, int G, double *tri_e,
                                            int b) {
  const int lane = threadIdx.x & 63;
  const double *p = part_t + (size_t)b * G;
  double s = 0.0;
  for (int r = lane; r < G; r += 64) s += p[r];
  s = vr_wave_sum(s);
  const int w = tri[b];
  if (lane == 0) tri_e[((size_t)(w & 1023) * o + ((w >> 10) & 1023)) * o + (w >> 20)] = s;
}

__global__ __launch_bounds__(64) void k_walk_energies(const int *tri, int o, const double *part_t, int G,
                                                      double *tri_e) {
  walk_energy(tri, o, part_t, G, tri_e, blockIdx.x);
}

hipError_t launch_walk_energies(const int *tri, int nb, int o, const double *part_t, int G, double *tri_e,
                                hipStream_t s) {
  if (nb > 0) hipLaunchKernelGGL(k_walk_energies, dim3(nb), dim3(64), 0, s, tri, o, part_t, G, tri_e);
  return hipGetLastError();
}

// One launch: the column sums (ncol workgroups), the gather (o^2 nblk) and the
// triple energies (four to a workgroup).
__global__ __launch_bounds__(256) void k_walk_gather(WalkGather G, int ncol, int nblk) {
  __shared__ double red[4][4][64];
  __shared__ int list[kWalkMaxBatch];
  __shared__ int cnt[4];
  int blk = blockIdx.x;
  if (blk < ncol) {
    const int n = (G.d.vp + 63) / 64;
    walk_cols(G.d.vp, G.R, G.r_stride, G.vec, blk % n, blk / n, red);
    return;
  }
  blk -= ncol;
  if (blk < nblk * G.d.o * G.d.o) {
    walk_gather(G, nblk, blk, list, cnt);
    return;
  }
  const int b = (blk - nblk * G.d.o * G.d.o) * 4 + (threadIdx.x >> 6);
  if (b < G.nb) walk_energy(G.tri, G.d.o, G.part_t, G.G, G.tri_e, b);
}

hipError_t launch_walk_gather(const WalkGather &g, hipStream_t s) {
  const int v = g.d.vp, o = g.d.o;
  if (g.nb > kWalkMaxBatch) return hipErrorInvalidValue;
  if (g.nb > 0 && vr_col_blocks(v) > 1)
    hipLaunchKernelGGL(k_walk_vrsum, dim3((v * v + 255) / 256, g.nb), dim3(256), 0, s, v,
                       const_cast<double *>(g.R), g.r_stride, g.has_fvo);
  const int ncol = (v + 63) / 64 * g.nb, nblk = (v * g.d.up + 255) / 256;
  const long long total = ncol + (long long)nblk * o * o + (g.tri_e ? (g.nb + 3) / 4 : 0);
  if (total >= (1LL << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_walk_gather, dim3((unsigned)total), dim3(256), 0, s, g, ncol, nblk);
  hipLaunchKernelGGL(k_walk_t1, dim3((g.d.v + 63) / 64, o), dim3(256), 0, s, g);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// projected walk
// ---------------------------------------------------------------------------
struct WalkUpload {
  double v[256];
};
__global__ void k_walk_upload(WalkUpload u, int n, double *dst) {
  if ((int)threadIdx.x < n) dst[threadIdx.x] = u.v[threadIdx.x];
}

hipError_t launch_walk_upload(const double *src, size_t n, double *dst, hipStream_t s) {
  for (size_t at = 0; at < n; at += 256) {
    WalkUpload u;
    const int m = (int)std::min<size_t>(256, n - at);
    for (int q = 0; q < m; ++q) u.v[q] = src[at + q];
    hipLaunchKernelGGL(k_walk_upload, dim3(1), dim3(256), 0, s, u, m, dst + at);
  }
  return hipGetLastError();
}

// sum over the workgroup's 256 threads, in a fixed order, on thread 0
__device__ __forceinline__ double walk_block_sum(double x, double *red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(256) void k_walk_pair_energies(const double *part_t, int G, const int *tri, int o,
                                                            double *pair_e) {
  __shared__ double red[4];
  double s = 0.0;
  for (int r = threadIdx.x; r < G; r += 256) s += part_t[(size_t)blockIdx.x * G + r];
  s = walk_block_sum(s, red);
  const int w = tri[(size_t)blockIdx.x * o];
  if (threadIdx.x == 0) pair_e[((w >> 10) & 1023) * o + (w >> 20)] = s;
}

hipError_t launch_walk_pair_energies(const double *part_t, int G, const int *tri, int np, int o,
                                     double *pair_e, hipStream_t s) {
  hipLaunchKernelGGL(k_walk_pair_energies, dim3(np), dim3(256), 0, s, part_t, G, tri, o, pair_e);
  return hipGetLastError();
}

// one workgroup per (l, f)
__global__ __launch_bounds__(256) void k_walk_ulo(const double *part_u, int G, double ebar, const int *tri, int np,
                                                  int o, int first, double *ulo_bar) {
  __shared__ double red[4];
  const int l = blockIdx.x, f = blockIdx.y;
  double s = 0.0;
  for (int t = threadIdx.x; t < np * G; t += 256) {
    const int p = t / G, g = t - p * G, w = tri[(size_t)p * o];
    const double x = part_u[(((size_t)p * o + l) * G + g) * kMaxFrag + f];
    s += x * (((w >> 10) & 1023) == (w >> 20) ? 1.0 : 2.0);
  }
  s = walk_block_sum(s, red);
  if (threadIdx.x == 0) {
    double *d = ulo_bar + (size_t)f * o + l;
    *d = ebar * s / 3.0 + (first ? 0.0 : *d);
  }
}

hipError_t launch_walk_ulo(const double *part_u, int G, int nfrag, double ebar, const int *tri, int np, int o,
                           bool first, double *ulo_bar, hipStream_t s) {
  hipLaunchKernelGGL(k_walk_ulo, dim3(o, nfrag), dim3(256), 0, s, part_u, G, ebar, tri, np, o, first ? 1 : 0,
                     ulo_bar);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// exit
// ---------------------------------------------------------------------------
// ovvv_bar[x,p,f,q] = VTb[x][p][q][f], or packed g[f,q] + g[q,f] (q < f), g[f,f]:
// a 32 x 32 tile (f, q) of one (x, p) per workgroup, turned in LDS
__device__ __forceinline__ void fold_ovvv(const WalkDims &d, const double *__restrict__ VTb, int packed,
                                          double *__restrict__ out, int bf, int bq, int bz, int nz,
                                          double (*tile)[33]) {
  const int f0 = bf * 32, q0 = bq * 32, v = d.v, vp = d.vp, up = d.up;
  if (packed && q0 > f0) return;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const size_t npair = (size_t)v * (v + 1) / 2;
  for (int xp = bz; xp < d.o * v; xp += nz) {
    const double *g = VTb + ((size_t)(xp / v) * vp + xp % v) * d.sp;
    for (int r = ty; r < 32; r += 8) {
      const int q = q0 + r, f = f0 + tx;
      tile[r][tx] = (q < v && f < v) ? g[(size_t)q * up + f] : 0.0;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
      const int f = f0 + r, q = q0 + tx;
      if (f >= v || q >= v) continue;
      if (!packed)
        out[((size_t)xp * v + f) * v + q] = tile[tx][r];
      else if (q <= f)
        out[xp * npair + (size_t)f * (f + 1) / 2 + q] = tile[tx][r] + (q < f ? g[(size_t)f * up + q] : 0.0);
    }
    __syncthreads();
  }
}

// t2_bar[x,m,p,q] += VTb[x][p][q][v + m], one (x, p) and 32 (m, q) per workgroup
__device__ __forceinline__ void fold_t2(const WalkDims &d, const double *__restrict__ VTb,
                                        double *__restrict__ t2_bar, int bq, int bm, int bz, int nz,
                                        double (*tile)[33]) {
  const int q0 = bq * 32, m0 = bm * 32, o = d.o, v = d.v, vp = d.vp, up = d.up;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int xp = bz; xp < o * v; xp += nz) {
    const int x = xp / v, p = xp - x * v;
    const double *g = VTb + ((size_t)x * vp + p) * d.sp + v;
    for (int r = ty; r < 32; r += 8)
      tile[r][tx] = (q0 + r < v && m0 + tx < o) ? g[(size_t)(q0 + r) * up + m0 + tx] : 0.0;
    __syncthreads();
    for (int r = ty; r < 32; r += 8)
      if (m0 + r < o && q0 + tx < v)
        t2_bar[(((size_t)x * o + m0 + r) * v + p) * v + q0 + tx] += tile[tx][r];
    __syncthreads();
  }
}

// column sums of part_mo: kWalkMoParts row ranges, then those in order
__device__ __forceinline__ void fold_mo(const double *part, int rows, int cols, double *part2, int c, int y) {
  if (c >= cols) return;
  const int per = (rows + kWalkMoParts - 1) / kWalkMoParts;
  double s = 0.0;
  for (int r = y * per; r < min(rows, (y + 1) * per); ++r) s += part[(size_t)r * cols + c];
  part2[(size_t)y * cols + c] = s;
}

// the three in one launch: n0 workgroups of fold_ovvv, n1 of fold_t2, then fold_mo
__global__ __launch_bounds__(256) void k_walk_finish(WalkDims d, const double *__restrict__ VTb, int packed,
                                                     double *__restrict__ ovvv_bar, double *__restrict__ t2_bar,
                                                     const double *part_mo, int rows, double *part2, unsigned n0,
                                                     unsigned n1, int nz) {
  __shared__ double tile[32][33];
  const unsigned nt = (d.v + 31) / 32, nm = (d.o + 31) / 32;
  unsigned blk = blockIdx.x;
  if (blk < n0) {
    const unsigned r = blk / nt;
    fold_ovvv(d, VTb, packed, ovvv_bar, (int)(blk - r * nt), (int)(r % nt), (int)(r / nt), nz, tile);
    return;
  }
  blk -= n0;
  if (blk < n1) {
    const unsigned r = blk / nt;
    fold_t2(d, VTb, t2_bar, (int)(blk - r * nt), (int)(r % nm), (int)(r / nm), nz, tile);
    return;
  }
  blk -= n1;
  const int cols = d.o + d.vp, nc = (cols + 63) / 64;
  fold_mo(part_mo, rows, cols, part2, (int)(blk % nc) * 64 + (threadIdx.x & 63),
          (int)(blk / nc) * 4 + (threadIdx.x >> 6));
}

hipError_t launch_walk_finish(const WalkDims &d, const double *VTb, int packed, double *ovvv_bar,
                              double *t2_bar, const double *part_mo, int rows, double *part2,
                              double *mo_bar, hipStream_t s) {
  const unsigned nt = (d.v + 31) / 32, nm = (d.o + 31) / 32;
  const unsigned nz = (unsigned)std::min(d.o * d.v, 65535);
  static_assert(kWalkMoParts % 4 == 0, "four row ranges per workgroup");
  const unsigned n0 = nt * nt * nz, n1 = nt * nm * nz, n2 = (d.o + d.vp + 63) / 64 * (kWalkMoParts / 4);
  if ((long long)nt * (nt + nm) * nz + n2 >= (1LL << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_walk_finish, dim3(n0 + n1 + n2), dim3(256), 0, s, d, VTb, packed, ovvv_bar, t2_bar, part_mo,
                     rows, part2, n0, n1, (int)nz);
  return launch_reduce_rows(part2, kWalkMoParts, d.o + d.v, d.o + d.vp, mo_bar, 0, s);
}

}  // namespace pamd
