// Epilogue of the batched FP64 walk: V, Z = r3(W + V), 1/D, the energy and the
// adjoint's seeds of many triples per launch (walk64.h; the algorithm of
// ccsd_t_vjp.c:42-117, one occupied triple per grid row).
//
// A workgroup takes one orbit of 8 x 8 x 8 virtual tiles {(A, B, C) and its
// permutations}, A >= B >= C.  Thread (al, be, ga) owns the six images of the
// position a = (A, al), b = (B, be), c = (C, ga): abc, acb, bac, bca, cab, cba, each
// in its own tile.  The six sit in LDS for the turn only; everything after is
// in registers:
//   * r3 of all six from two sums (even and odd permutations),
//   * one denominator and one reciprocal for the six (D is symmetric),
//   * one dE/d(e_virtual) reduction per orbit instead of one per tile,
//   * Wbar and Vbar go back into the thread's own LDS slots and leave in rows.
// (One element per thread and tile instead needs five further LDS reads per
// element of W and of W + V, six reciprocals and six reductions.)  The pair
// blocks of the V terms, 18 of 8 x 8, are staged in LDS too: read from global
// memory per element they were 36 loads per thread and orbit against 6 of W.
// Where tiles coincide (A == B, B == C) only the threads with al >= be, be >= ga
// work; an image that coincides with another counts once.
// Loads of the next orbit are in flight during the arithmetic of the current
// one.  Bound by memory: W read, Wbar and Vbar written.  Measured at v = 160, against
// one element per thread: energies of 200 triples 4.6 -> 2.1 ms (3.1 TB/s), with
// the seeds of 114 triples 6.9 -> 3.5 ms (3.2 TB/s).
#include <algorithm>
#include "bf16_split.h"
#include "engine_staging.h"
#include "walk64.h"

namespace pamd {

namespace {

constexpr int kT3 = 512, kSRow = 9, kSBlk = 8 * kSRow;

// distinct tiles of an orbit by equality pattern (A == B) + 2 (B == C): ranges of
// tile p (0 A, 1 B, 2 C), and the tile of each image
struct WalkOrbit {
  int np;
  int sel[6][3];
  int tile[6];
};
__constant__ WalkOrbit kWalkOrbit[4] = {
    {6, {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}}, {0, 1, 2, 3, 4, 5}},
    {3, {{0, 0, 2}, {0, 2, 0}, {2, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, {0, 1, 0, 1, 2, 2}},
    {3, {{0, 1, 1}, {1, 0, 1}, {1, 1, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, {0, 0, 1, 2, 1, 2}},
    {1, {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, {0, 0, 0, 0, 0, 0}},
};

typedef const __attribute__((address_space(4))) unsigned long long *EntryPtr;

// table entry of an orbit: its three tile indices and the pattern, 16 bits each,
// picked by shifts (an array indexed at run time would live in scratch memory)
struct OrbitPos {
  unsigned long long e;
  __device__ __forceinline__ int val(int r) const { return (int)((e >> (16 * r)) & 0xffff); }
  __device__ __forceinline__ int pat() const { return (int)(e >> 48); }
};
__device__ __forceinline__ OrbitPos orbit_at(const unsigned short *tab, long long q) {
  return {((EntryPtr)tab)[q]};
}

// range r (0 A, 1 B, 2 C) of axis x of distinct tile p, and tile of image m; SIX:
// all six tiles are distinct (nearly every orbit), so both are constants
template <bool SIX>
struct Pattern {
  int pat;
  static constexpr int kSel[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
  __device__ __forceinline__ int np() const { return SIX ? 6 : kWalkOrbit[pat].np; }
  __device__ __forceinline__ int sel(int p, int x) const { return SIX ? kSel[p][x] : kWalkOrbit[pat].sel[p][x]; }
  __device__ __forceinline__ int tile(int m) const { return SIX ? m : kWalkOrbit[pat].tile[m]; }
};

// images: abc, acb, bac, bca, cab, cba; even permutations 0, 3, 4
__device__ __forceinline__ void r3_six(const double (&x)[6], double (&z)[6]) {
  const double ev = x[0] + x[3] + x[4], od = x[1] + x[2] + x[5];
  const double e = ev - 2.0 * od, o = od - 2.0 * ev;
  z[0] = fma(3.0, x[0], e);
  z[3] = fma(3.0, x[3], e);
  z[4] = fma(3.0, x[4], e);
  z[1] = fma(3.0, x[1], o);
  z[2] = fma(3.0, x[2], o);
  z[5] = fma(3.0, x[5], o);
}

// LDS slot of tile position 64 a + 8 b + c: the low five bits swizzled by a, so
// that all six permuted patterns spread over the banks
__device__ __forceinline__ int slot_of(int a, int b, int c) {
  return ((a << 6) | (b << 3) | c) ^ (a | ((a & 3) << 3));
}

__device__ __forceinline__ double wave_sum64(double x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}

// Element (row, column) of an 8 x 8 block at a uniform address: lane offset
// (lane / 8) v + lane % 8, the same for W, Vbar and the pair blocks (the wave is
// the block's slab of W), so an access takes no vector address arithmetic.
typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double ld64(const double *p, unsigned off8) {
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, -1, 0x00027000);
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off8, 0, 0));
}
__device__ __forceinline__ void st64(double *p, unsigned off8, double x) {
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, -1, 0x00027000);
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2_t, x), r, off8, 0, 0);
}
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// occupied index x (0 i, 1 j, 2 k) of a packed triple
__device__ __forceinline__ int occ_of(int t, int x) { return (t >> (10 * x)) & 1023; }

template <bool FVO>
struct Staged {
  double s[FVO ? 6 : 3], t[FVO ? 2 : 1];
};

}  // namespace

// The staged values of one orbit: wave w takes blocks w, w + 8, w + 16 of the 18
// (ij, ik, jk of AB, BA, AC, CA, BC, CB), waves 0 to 2 also the 24 singles of an
// occupied orbital.  off8: the lane's offset in a block.
template <bool FVO>
__device__ __forceinline__ void stage_load(const OrbitArgs &A, int t, const OrbitPos &o, unsigned off8,
                                           Staged<FVO> &st) {
  const int wave = wave_id(), lane = threadIdx.x & 63, v = A.v;
  const long long vv = (long long)v * v;
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    const int blk = wave + 8 * u;
    if (blk < 18) {
      // (picked by shifts throughout: no branches, no indexed arrays)
      const int which = blk / 6, pr = blk - which * 6;
      // ranges of AB, BA, AC, CA, BC, CB; pairs (i, j), (i, k), (j, k)
      const int row = o.val((0x984 >> (2 * pr)) & 3), col = o.val((0x621 >> (2 * pr)) & 3);
      const int x = occ_of(t, which >> 1), y = occ_of(t, which == 0 ? 1 : 2);
      const long long at = ((long long)x * A.o + y) * vv + (long long)row * 8 * v + col * 8;
      st.s[u] = ld64(A.ovs + at, off8);
      if (FVO) st.s[3 + u] = ld64(A.t2s + at, off8);
    }
  }
  if (wave < 3 && lane < 24) {
    const unsigned idx = o.val(lane >> 3) * 8 + (lane & 7);
    const int x = occ_of(t, wave);
    st.t[0] = ld64(A.t1 + (long long)x * v, idx * 8);
    if (FVO) st.t[1] = ld64(A.fvo + x, idx * 8 * (unsigned)A.o);
  }
}

template <bool FVO>
struct StageLds {
  double S[FVO ? 36 : 18][kSBlk];  // [which * 6 + pair block][row * 9 + col]
  double t[FVO ? 2 : 1][3][24];
};

template <bool FVO>
__device__ __forceinline__ void stage_store(const Staged<FVO> &st, StageLds<FVO> &L) {
  const int wave = wave_id(), lane = threadIdx.x & 63;
  const int at = (lane >> 3) * kSRow + (lane & 7);
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    const int blk = wave + 8 * u;
    if (blk < 18) {
      L.S[blk][at] = st.s[u];
      if (FVO) L.S[18 + blk][at] = st.s[3 + u];
    }
  }
  if (wave < 3 && lane < 24) {
    L.t[0][wave][lane] = st.t[0];
    if (FVO) L.t[1][wave][lane] = st.t[1];
  }
}

// V of the six images: sum over (ij, k), (ik, j), (jk, i)
template <bool FVO>
__device__ __forceinline__ void v_six(const StageLds<FVO> &L, int al, int be, int ga, double (&x)[6]) {
#pragma unroll
  for (int q = 0; q < 6; ++q) x[q] = 0.0;
#pragma unroll
  for (int h = 0; h < (FVO ? 2 : 1); ++h) {
    const int at[6] = {al * kSRow + be, be * kSRow + al, al * kSRow + ga,
                       ga * kSRow + al, be * kSRow + ga, ga * kSRow + be};
    // pair w with the third index's single t (ij: k, ik: j, jk: i); image m takes
    // pair block (x, y), (x, z) or (y, z) and the single of the position left
    constexpr int blk[3][6] = {{0, 2, 1, 4, 3, 5}, {2, 0, 4, 1, 5, 3}, {4, 5, 2, 3, 0, 1}};
    constexpr int sgl[3][6] = {{2, 1, 2, 0, 1, 0}, {1, 2, 0, 2, 0, 1}, {0, 0, 1, 1, 2, 2}};
#pragma unroll
    for (int w = 0; w < 3; ++w) {
      const double t[3] = {L.t[h][2 - w][al], L.t[h][2 - w][8 + be], L.t[h][2 - w][16 + ga]};
      double s[6];
#pragma unroll
      for (int p = 0; p < 6; ++p) s[p] = L.S[18 * h + 6 * w + p][at[p]];
#pragma unroll
      for (int m = 0; m < 6; ++m) x[m] = fma(s[blk[w][m]], t[sgl[w][m]], x[m]);
      // one pair's nine values at a time: all 27 in flight would spill
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// 1/D: hardware estimate and two Newton steps (D <= -(HOMO-LUMO gap) < 0)
__device__ __forceinline__ double recip(double D) {
  double r = __builtin_amdgcn_rcp(D);
  r = fma(r, fma(-D, r, 1.0), r);
  return fma(r, fma(-D, r, 1.0), r);
}

// W of the orbit's tiles at the thread's row position (slots past the distinct
// ones repeat tile 0 and are not used); a tile's slab of the wave starts at tile_at
template <bool SIX>
__device__ __forceinline__ long long tile_at(const OrbitPos &o, const Pattern<SIX> &pt, int p, long long slab, int v) {
  return (long long)(o.val(pt.sel(p, 0)) * 8 + wave_id()) * slab + (long long)o.val(pt.sel(p, 1)) * 8 * v +
         o.val(pt.sel(p, 2)) * 8;
}
__device__ __forceinline__ void w_load(const double *W, long long ws, int v, const OrbitPos &o, unsigned off8,
                                       double (&w)[6]) {
  if (o.pat() == 0) {
#pragma unroll
    for (int p = 0; p < 6; ++p) w[p] = ld64(W + tile_at(o, Pattern<true>{0}, p, ws, v), off8);
  } else {
#pragma unroll
    for (int p = 0; p < 6; ++p) w[p] = ld64(W + tile_at(o, Pattern<false>{o.pat()}, p, ws, v), off8);
  }
}

struct VirSums {
  double stg[8][17];  // per wave: c sums, b sums, a sum of the orbit
};

// adds the orbit's sums of -d over two of the three axes into vir (LDS, one
// entry per virtual orbital): first half before a barrier, second after it
__device__ __forceinline__ void vir_stage(double d, VirSums &S) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double sc = d;  // over be
  sc += __shfl_xor(sc, 8, 64);
  sc += __shfl_xor(sc, 16, 64);
  sc += __shfl_xor(sc, 32, 64);
  double sb = d;  // over ga
  sb += __shfl_xor(sb, 1, 64);
  sb += __shfl_xor(sb, 2, 64);
  sb += __shfl_xor(sb, 4, 64);
  double sa = sb;
  sa += __shfl_xor(sa, 8, 64);
  sa += __shfl_xor(sa, 16, 64);
  sa += __shfl_xor(sa, 32, 64);
  if (lane < 8) S.stg[wave][lane] = sc;
  if ((lane & 7) == 0) S.stg[wave][8 + (lane >> 3)] = sb;
  if (lane == 0) S.stg[wave][16] = sa;
}
__device__ __forceinline__ void vir_add(const VirSums &S, const OrbitPos &o, double *vir) {
  const int tid = threadIdx.x;
  if (tid >= 24) return;
  const int r = tid >> 3, off = tid & 7;
  const int v0 = o.val(0), v1 = o.val(1), v2 = o.val(2);
  const int mine = r == 0 ? v0 : r == 1 ? v1 : v2;
  if ((r > 0 && mine == v0) || (r > 1 && mine == v1)) return;  // the first range of a tile owns it
  double sum = 0.0;
  if (v0 == mine) sum += S.stg[off][16];
  if (v1 == mine)
    for (int w = 0; w < 8; ++w) sum += S.stg[w][8 + off];
  if (v2 == mine)
    for (int w = 0; w < 8; ++w) sum += S.stg[w][off];
  vir[mine * 8 + off] -= sum;
}

// block sum over 512 threads in wave order, on every thread
__device__ __forceinline__ double block_sum512(double x, double *red) {
  x = wave_sum64(x);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < 8; ++w) s += red[w];
  return s;
}

// weight of a thread's six images in sums over the orbit; 0: not its owner
__device__ __forceinline__ double image_weight(int pat, int al, int be, int ga) {
  const bool ab = pat & 1, bc = pat & 2;
  if ((ab && al < be) || (bc && be < ga)) return 0.0;
  const bool e1 = ab && al == be, e2 = bc && be == ga;
  return e1 && e2 ? 1.0 / 6.0 : (e1 || e2 ? 0.5 : 1.0);
}

// Energy (VJP false), or energy and seeds.  Grid (G, triples).  PL: Wbar leaves as
// three bf16 planes (split-BF16x3; one triple), W is kept.
template <bool VJP, bool FVO, bool PL>
__global__ __launch_bounds__(512, 4) void k_walk_orbit(OrbitArgs A) {
  __shared__ double Ws[6][kT3];
  __shared__ double Vs[VJP ? 6 : 1][VJP ? kT3 : 1];
  __shared__ StageLds<FVO> L;
  __shared__ VirSums S;
  __shared__ double red[8];
  extern __shared__ double vir[];
  const int tid = threadIdx.x;
  const int al = wave_id(), be = (tid >> 3) & 7, ga = tid & 7;
  const unsigned off8 = (unsigned)(be * A.v + ga) * 8;
  const int v = A.v, t = A.tri[blockIdx.y];
  const int i = occ_of(t, 0), j = occ_of(t, 1), k = occ_of(t, 2);
  double g = A.ebar * (i == j || j == k ? 1.0 : 2.0);
  if (A.wt) g *= (A.wt[i] + A.wt[j] + A.wt[k]) / 3.0;
  double *W = A.W + (size_t)blockIdx.y * v * A.ws;
  double *Vb = VJP ? A.Vb + (size_t)blockIdx.y * v * v * v : nullptr;
  const double eo = A.mo[i] + A.mo[j] + A.mo[k];
  const double *ev = A.mo + A.o;
  if (VJP)
    for (int x = tid; x < v; x += 512) vir[x] = 0.0;
  const int own = slot_of(al, be, ga);
  const int img[6] = {own, slot_of(al, ga, be), slot_of(be, al, ga),
                      slot_of(be, ga, al), slot_of(ga, al, be), slot_of(ga, be, al)};
  double esum = 0.0, osum = 0.0;
  const long long first = xcd_remap(blockIdx.x, gridDim.x);
  double wn[6];
  Staged<FVO> sn;
  OrbitPos o;
  if (first < A.norb) {
    o = orbit_at(A.tab, first);
    w_load(W, A.ws, v, o, off8, wn);
    stage_load<FVO>(A, t, o, off8, sn);
  }
  for (long long q = first; q < A.norb; q += gridDim.x) {
    const OrbitPos oc = o;
#pragma unroll
    for (int p = 0; p < 6; ++p) Ws[p][own] = wn[p];
    stage_store<FVO>(sn, L);
    const double D = eo - ev[oc.val(0) * 8 + al] - ev[oc.val(1) * 8 + be] - ev[oc.val(2) * 8 + ga];
    __syncthreads();
    if (q + gridDim.x < A.norb) {
      o = orbit_at(A.tab, q + gridDim.x);
      w_load(W, A.ws, v, o, off8, wn);
      stage_load<FVO>(A, t, o, off8, sn);
    }
    auto body = [&](auto pt) {
      const double wt = pt.pat == 0 ? 1.0 : image_weight(pt.pat, al, be, ga);
      double d = 0.0;
      if (pt.pat == 0 || wt != 0.0) {
        double w[6], x[6], z[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) w[m] = Ws[pt.tile(m)][img[m]];
        v_six<FVO>(L, al, be, ga, x);
#pragma unroll
        for (int m = 0; m < 6; ++m) x[m] = fma(0.5, x[m], w[m]);
        r3_six(x, z);
        const double rD = recip(D);
        double wz = 0.0;
#pragma unroll
        for (int m = 0; m < 6; ++m) wz = fma(w[m], z[m], wz);
        wz *= wt * rD;
        esum += wz;
        if (VJP) {
          r3_six(w, x);
          const double gr = g * rD;
#pragma unroll
          for (int m = 0; m < 6; ++m) {
            const double vb = gr * x[m];
            Ws[pt.tile(m)][img[m]] = fma(gr, z[m], vb);
            Vs[pt.tile(m)][img[m]] = vb;
          }
          d = -g * wz * rD;
          osum += d;
        }
      }
      if (VJP) vir_stage(d, S);
      __syncthreads();
      if (VJP) {
#pragma unroll
        for (int p = 0; p < 6; ++p) {
          if (p >= pt.np()) continue;
          const long long at = tile_at(oc, pt, p, (long long)v * v, v);
          if (PL)
            put3(A.Wb3, (long long)v * v * v, at + off8 / 8, Ws[p][own]);
          else
            st64(W + tile_at(oc, pt, p, A.ws, v), off8, Ws[p][own]);
          st64(Vb + at, off8, Vs[p][own]);
        }
      }
    };
    if (oc.pat() == 0)
      body(Pattern<true>{0});
    else
      body(Pattern<false>{oc.pat()});
    if (VJP) {
      vir_add(S, oc, vir);
      __syncthreads();
    }
  }
  const size_t rw = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
  const double et = block_sum512(esum, red);
  if (tid == 0) A.part_t[rw] = et;
  if (VJP) {
    const double ot = block_sum512(osum, red);
    double *pm = A.part_mo + rw * (A.o + v);
    for (int x = tid; x < v; x += 512) pm[A.o + x] += vir[x];
    if (tid == 0) {
      pm[i] += ot;
      pm[j] += ot;
      pm[k] += ot;
    }
  }
}

// Projector sums of a batch of pairs, grid (G, pairs): acc[f][0 / 1][orbit][image]
// [thread] = sum_l u_f[l] W_ljk, sum_l u_f[l] Z_ljk / D_ljk of the thread's images,
// in registers over l, two fragment orbitals at a time; part_t gets the pair's
// sum_f <A_f, B_f>.  The next triple's W is in flight during the current one's
// arithmetic.
template <bool FVO, int NF>
__global__ __launch_bounds__(512, 2) void k_walk_acc(OrbitArgs A, int f0) {
  __shared__ double Ws[6][kT3];
  __shared__ StageLds<FVO> L;
  __shared__ double red[8];
  const int tid = threadIdx.x;
  const int al = wave_id(), be = (tid >> 3) & 7, ga = tid & 7;
  const unsigned off8 = (unsigned)(be * A.v + ga) * 8;
  const int v = A.v, no = A.o;
  const int *tri = A.tri + (size_t)blockIdx.y * no;
  const double *W = A.W + (size_t)blockIdx.y * no * v * A.ws;
  const size_t wblk = (size_t)v * A.ws, ablk = (size_t)A.norb * 6 * kT3;
  double *acc = A.accA + ((size_t)blockIdx.y * A.nfrag + f0) * 2 * ablk;
  const double *ev = A.mo + no;
  const int own = slot_of(al, be, ga);
  const int img[6] = {own, slot_of(al, ga, be), slot_of(be, al, ga),
                      slot_of(be, ga, al), slot_of(ga, al, be), slot_of(ga, be, al)};
  double esum = 0.0;
  for (long long q = xcd_remap(blockIdx.x, gridDim.x); q < A.norb; q += gridDim.x) {
    const OrbitPos o = orbit_at(A.tab, q);
    const double wt = image_weight(o.pat(), al, be, ga);
    const double ed = ev[o.val(0) * 8 + al] + ev[o.val(1) * 8 + be] + ev[o.val(2) * 8 + ga];
    double a[NF][6], b[NF][6];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int m = 0; m < 6; ++m) a[f][m] = b[f][m] = 0.0;
    double wn[6];
    Staged<FVO> sn;
    w_load(W, A.ws, v, o, off8, wn);
    int t = tri[0];
    stage_load<FVO>(A, t, o, off8, sn);
    for (int l = 0; l < no; ++l) {
      const double eo = A.mo[occ_of(t, 0)] + A.mo[occ_of(t, 1)] + A.mo[occ_of(t, 2)];
#pragma unroll
      for (int p = 0; p < 6; ++p) Ws[p][own] = wn[p];
      stage_store<FVO>(sn, L);
      __syncthreads();
      if (l + 1 < no) {
        w_load(W + (l + 1) * wblk, A.ws, v, o, off8, wn);
        t = tri[l + 1];
        stage_load<FVO>(A, t, o, off8, sn);
      }
      auto body = [&](auto pt) {
        double w[6], x[6], z[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) w[m] = Ws[pt.tile(m)][img[m]];
        v_six<FVO>(L, al, be, ga, x);
#pragma unroll
        for (int m = 0; m < 6; ++m) x[m] = fma(0.5, x[m], w[m]);
        r3_six(x, z);
        const double rD = recip(eo - ed);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const double u = A.udev[(f0 + f) * no + l], ur = u * rD;
#pragma unroll
          for (int m = 0; m < 6; ++m) {
            a[f][m] = fma(u, w[m], a[f][m]);
            b[f][m] = fma(ur, z[m], b[f][m]);
          }
        }
      };
      if (o.pat() == 0)
        body(Pattern<true>{0});
      else if (wt != 0.0)
        body(Pattern<false>{o.pat()});
      __syncthreads();
    }
    double s = 0.0;
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int m = 0; m < 6; ++m) {
        s = fma(a[f][m], b[f][m], s);
        acc[(2 * f) * ablk + (q * 6 + m) * kT3 + tid] = a[f][m];
        acc[(2 * f + 1) * ablk + (q * 6 + m) * kT3 + tid] = b[f][m];
      }
    esum += wt * s;
  }
  const double et = block_sum512(esum, red);
  if (tid == 0) {
    double *e = A.part_t + (size_t)blockIdx.y * gridDim.x + blockIdx.x;
    *e = et + (f0 ? *e : 0.0);
  }
}

// Seeds of the projected energy, grid (G, triples (l, j, k)), from the pair's
// finished sums: Q = g sum_f u_f A_f, Wbar = g sum_f u_f B_f + r3(Q) / D, Vbar =
// r3(Q) / D, Dbar = -Q Z / D^2, and part_u[f] = <W, B_f> + <A_f, Z / D>.
// Two waves per SIMD: at four the 128 registers spill 24 (o10/v64, two fragment
// orbitals, 183 triples a launch: 877 us; 680 without spills; 819 with the next orbit's W in
// flight as in k_walk_orbit).
template <bool FVO>
__global__ __launch_bounds__(512, 2) void k_walk_proj(OrbitArgs A) {
  __shared__ double Ws[6][kT3];
  __shared__ double Vs[6][kT3];
  __shared__ StageLds<FVO> L;
  __shared__ VirSums S;
  __shared__ double red[8];
  extern __shared__ double vir[];
  const int tid = threadIdx.x;
  const int al = wave_id(), be = (tid >> 3) & 7, ga = tid & 7;
  const unsigned off8 = (unsigned)(be * A.v + ga) * 8;
  const int v = A.v, t = A.tri[blockIdx.y];
  const int i = occ_of(t, 0), j = occ_of(t, 1), k = occ_of(t, 2);
  const double g = A.ebar * (j == k ? 1.0 : 2.0) / 3.0;
  const size_t pair = blockIdx.y / A.o, ablk = (size_t)A.norb * 6 * kT3;
  const double *acc = A.accA + pair * A.nfrag * 2 * ablk;
  double *W = A.W + (size_t)blockIdx.y * v * A.ws;
  double *Vb = A.Vb + (size_t)blockIdx.y * v * v * v;
  const double eo = A.mo[i] + A.mo[j] + A.mo[k];
  const double *ev = A.mo + A.o;
  for (int x = tid; x < v; x += 512) vir[x] = 0.0;
  const int own = slot_of(al, be, ga);
  const int img[6] = {own, slot_of(al, ga, be), slot_of(be, al, ga),
                      slot_of(be, ga, al), slot_of(ga, al, be), slot_of(ga, be, al)};
  double osum = 0.0, udot[kMaxFrag];
#pragma unroll
  for (int f = 0; f < kMaxFrag; ++f) udot[f] = 0.0;
  for (long long q = xcd_remap(blockIdx.x, gridDim.x); q < A.norb; q += gridDim.x) {
    const OrbitPos o = orbit_at(A.tab, q);
    {
      double wn[6];
      Staged<FVO> sn;
      w_load(W, A.ws, v, o, off8, wn);
      stage_load<FVO>(A, t, o, off8, sn);
#pragma unroll
      for (int p = 0; p < 6; ++p) Ws[p][own] = wn[p];
      stage_store<FVO>(sn, L);
    }
    const double D = eo - ev[o.val(0) * 8 + al] - ev[o.val(1) * 8 + be] - ev[o.val(2) * 8 + ga];
    __syncthreads();
    auto body = [&](auto pt) {
      const double wt = pt.pat == 0 ? 1.0 : image_weight(pt.pat, al, be, ga);
      double d = 0.0;
      if (pt.pat == 0 || wt != 0.0) {
        double w[6], x[6], z[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) w[m] = Ws[pt.tile(m)][img[m]];
        v_six<FVO>(L, al, be, ga, x);
#pragma unroll
        for (int m = 0; m < 6; ++m) x[m] = fma(0.5, x[m], w[m]);
        r3_six(x, z);
        const double rD = recip(D);
        double Q[6], P[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) {
          z[m] *= rD;
          Q[m] = P[m] = 0.0;
        }
#pragma unroll
        for (int f = 0; f < kMaxFrag; ++f) {
          if (f >= A.nfrag) continue;
          const double u = g * A.udev[f * A.o + i];
          double s = 0.0;
#pragma unroll
          for (int m = 0; m < 6; ++m) {
            const double a = ld64(acc + (2 * f) * ablk + (q * 6 + m) * kT3, tid * 8);
            const double b = ld64(acc + (2 * f + 1) * ablk + (q * 6 + m) * kT3, tid * 8);
            Q[m] = fma(u, a, Q[m]);
            P[m] = fma(u, b, P[m]);
            s = fma(w[m], b, fma(a, z[m], s));
          }
          udot[f] = fma(wt, s, udot[f]);
          // one fragment orbital's twelve values at a time: more in flight spill
          __builtin_amdgcn_sched_barrier(0);
        }
        r3_six(Q, x);
        double qz = 0.0;
#pragma unroll
        for (int m = 0; m < 6; ++m) {
          const double vb = x[m] * rD;
          Ws[pt.tile(m)][img[m]] = P[m] + vb;
          Vs[pt.tile(m)][img[m]] = vb;
          qz = fma(Q[m], z[m], qz);
        }
        d = -wt * qz * rD;
        osum += d;
      }
      vir_stage(d, S);
      __syncthreads();
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        if (p >= pt.np()) continue;
        st64(W + tile_at(o, pt, p, A.ws, v), off8, Ws[p][own]);
        st64(Vb + tile_at(o, pt, p, (long long)v * v, v), off8, Vs[p][own]);
      }
    };
    if (o.pat() == 0)
      body(Pattern<true>{0});
    else
      body(Pattern<false>{o.pat()});
    vir_add(S, o, vir);
    __syncthreads();
  }
  const size_t rw = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
  const double ot = block_sum512(osum, red);
  for (int f = 0; f < A.nfrag; ++f) {
    double u = 0.0;
#pragma unroll
    for (int m = 0; m < kMaxFrag; ++m) u = m == f ? udot[m] : u;
    const double s = block_sum512(u, red);
    if (tid == 0) A.part_u[rw * kMaxFrag + f] = s;
  }
  double *pm = A.part_mo + rw * (A.o + v);
  for (int x = tid; x < v; x += 512) pm[A.o + x] += vir[x];
  if (tid == 0) {
    pm[i] += ot;
    pm[j] += ot;
    pm[k] += ot;
  }
}

hipError_t launch_walk_orbit(const OrbitArgs &a, int G, hipStream_t s) {
  const dim3 grid(G, a.nb), block(512);
  const size_t lds = a.vjp ? sizeof(double) * a.v : 0;
  if (a.vjp && a.Wb3 && a.nb != 1) return hipErrorInvalidValue;
  if (a.vjp && a.Wb3 && a.has_fvo)
    hipLaunchKernelGGL((k_walk_orbit<true, true, true>), grid, block, lds, s, a);
  else if (a.vjp && a.Wb3)
    hipLaunchKernelGGL((k_walk_orbit<true, false, true>), grid, block, lds, s, a);
  else if (a.vjp && a.has_fvo)
    hipLaunchKernelGGL((k_walk_orbit<true, true, false>), grid, block, lds, s, a);
  else if (a.vjp)
    hipLaunchKernelGGL((k_walk_orbit<true, false, false>), grid, block, lds, s, a);
  else if (a.has_fvo)
    hipLaunchKernelGGL((k_walk_orbit<false, true, false>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((k_walk_orbit<false, false, false>), grid, block, 0, s, a);
  return hipGetLastError();
}

hipError_t launch_walk_acc(const OrbitArgs &a, int G, int np, hipStream_t s) {
  const dim3 grid(G, np), block(512);
  for (int f = 0; f < a.nfrag; f += 2) {
    const bool two = f + 1 < a.nfrag;
    if (a.has_fvo && two)
      hipLaunchKernelGGL((k_walk_acc<true, 2>), grid, block, 0, s, a, f);
    else if (a.has_fvo)
      hipLaunchKernelGGL((k_walk_acc<true, 1>), grid, block, 0, s, a, f);
    else if (two)
      hipLaunchKernelGGL((k_walk_acc<false, 2>), grid, block, 0, s, a, f);
    else
      hipLaunchKernelGGL((k_walk_acc<false, 1>), grid, block, 0, s, a, f);
  }
  return hipGetLastError();
}

hipError_t launch_walk_proj(const OrbitArgs &a, int G, hipStream_t s) {
  const dim3 grid(G, a.nb), block(512);
  if (a.has_fvo)
    hipLaunchKernelGGL(k_walk_proj<true>, grid, block, sizeof(double) * a.v, s, a);
  else
    hipLaunchKernelGGL(k_walk_proj<false>, grid, block, sizeof(double) * a.v, s, a);
  return hipGetLastError();
}

}  // namespace pamd
