// The batched FP64 walk: many occupied triples per launch.
//
// Joined arrays.  The particle and the hole term of w_abc[ijk]
// (pyscfadlib/pyscfadlib/vjp/cc/ccsd_t.c:121-142) contract over f (virtual) and m
// (occupied) alike, so with
//   VT[x][p][q][f] = ovvv[x,p,f,q],  VT[x][p][q][v + m] = t2[x,m,p,q]
//   TB[z][y][r][f] = t2[z,y,r,f],    TB[z][y][r][v + m] = -ovoo[z,r,m,y]
// the twelve terms of W_ijk are six products over one index k < v + o:
//   W[a,b,c] = VT[i][a][b] TB[k,j][c] + VT[i][a][c] TB[j,k][b] + VT[j][b][a] TB[k,i][c]
//            + VT[j][b][c] TB[i,k][a] + VT[k][c][a] TB[j,i][b] + VT[k][c][b] TB[i,j][a],
// the adjoint of VT collects dE/d ovvv with the hole-term part of dE/d t2, and
// that of TB the particle-term part of dE/d t2 with dE/d ovoo.
//
// Padded space.  Virtual extents are padded to vp = 8 ceil(v / 8), the joined
// one to up = 8 ceil((v + o) / 8), with zeros: W and Wbar vanish there by
// themselves, every extent is a multiple of 8, rows are 16-byte aligned, and
// no kernel has a tail.
#pragma once
#include "ccsdt_common.h"

namespace pamd {

// triples per batch: the gather gives each slot of a batch to one of a workgroup's
// 256 threads, and the adjoint of VT keeps the batch's entries in LDS
constexpr int kWalkMaxBatch = 256;

// Slabs: VT[x][p] (vp x up) and W[a] (vp x vp) start an odd multiple of 256
// bytes apart (sp, ws elements).  L2 interleaves its 16 channels every 256
// bytes, and the walk reads 16 rows one slab apart at once: with vp = 160 a
// slab is a multiple of 4096 bytes, and all 16 rows would come from one channel.
struct WalkDims {
  int o, v, vp, up;
  long long sp, ws;
};
inline WalkDims walk_dims(int o, int v) {
  const int vp = (v + 7) / 8 * 8, up = (v + o + 7) / 8 * 8;
  auto odd = [](long long n) { return ((n + 31) / 32 | 1) * 32; };
  return {o, v, vp, up, odd((long long)vp * up), odd((long long)vp * vp)};
}
// 32-bit byte offsets within one occupied slab of VT
inline bool walk_dims_ok(const WalkDims &d) {
  return (d.vp + 8) * d.sp * 8 < (1LL << 32);
}

// Batches.  The call's triples (walk order i <= j <= k without i == j == k, every
// nshards-th from shard on) are cut into runs of 8, dealt to the batches in
// turn: a run shares i, j and so its slabs of VT, while every batch has about
// the same number of triples with each x, over which the adjoint of VT[x]
// sums.  (Batches of consecutive triples hold one i nearly throughout: that
// adjoint took 288 instead of 63 ms at o16/v160.)
constexpr int kWalkRun = 8;
struct WalkBatches {
  int cap;          // slots of a batch in the table (a multiple of 8)
  int count;        // batches
  long long n;      // triples
  int size(int b) const {
    const long long runs = (n + kWalkRun - 1) / kWalkRun;
    if (b >= runs) return 0;
    const long long mine = (runs - b + count - 1) / count, last = b + (mine - 1) * count;
    const long long cut = last == runs - 1 ? runs * kWalkRun - n : 0;
    return (int)(mine * kWalkRun - cut);
  }
};
inline WalkBatches walk_batches(long long n, int nb) {
  const long long runs = (n + kWalkRun - 1) / kWalkRun, per = nb / kWalkRun > 0 ? nb / kWalkRun : 1;
  const int count = (int)(runs > 0 ? (runs + per - 1) / per : 1);
  const int cap = (int)((runs + count - 1) / count) * kWalkRun;
  return {cap > 0 ? cap : kWalkRun, count, n};
}
// Everything a call prepares, in one launch: padded inputs (TBt[z][y][k][r] =
// TB[z][y][r][k]; VT null: only what the orbit epilogue and the V-bar reductions
// read), the orbit table, the triple table (tri[b cap + slot] = i | j << 10 |
// k << 20; pairs: slot p o + l is the triple (l, j, k) of the p-th pair j <= k, and
// nothing is left out) and two arrays to be zeroed.
struct WalkPrep {
  WalkDims d;
  const double *mo, *t1, *t2, *ovvv, *ovoo, *ovov, *fvo;
  double *VT, *TB, *TBt, *OVS, *T2S, *t1p, *fvop, *mop;
  unsigned short *orb;
  int *tri;
  double *zero[2];
  size_t nzero[2];
  long long norb;
  WalkBatches wb;
  int packed, shard, nshards, pairs;
  unsigned blocks[4];  // of VT, TB, the symmetrised blocks and the rest (set by the launcher)
};
hipError_t launch_walk_prep(WalkPrep a, hipStream_t s);

// W of nb triples (tri[0 .. nb)), each a block of vp ws elements
hipError_t launch_walk_w(const WalkDims &d, const double *VT, const double *TBt, double *W, const int *tri,
                         int nb, hipStream_t s);
// epilogue (OrbitArgs' batch fields, grid rows of G workgroups; walk64_orbit.hip):
// energies and, with vjp, Wbar (over W, or as bf16 planes when Wb3 is set), Vbar and
// the mo_energy_bar rows
hipError_t launch_walk_orbit(const OrbitArgs &a, int G, hipStream_t s);
// projected walk: the sums over l of np pairs into accA (walk_acc_doubles per
// pair and fragment orbital), their energies into part_t; then the seeds of all
// nb triples
inline size_t walk_acc_doubles(const WalkDims &d) {
  const size_t nt = d.vp / 8;
  return nt * (nt + 1) * (nt + 2) / 6 * 6 * 512 * 2;
}
hipError_t launch_walk_acc(const OrbitArgs &a, int G, int np, hipStream_t s);
hipError_t launch_walk_proj(const OrbitArgs &a, int G, hipStream_t s);
// VTb += dE/dVT of nb triples (Wb: their Wbar blocks); first: VTb is overwritten
hipError_t launch_walk_vtb(const WalkDims &d, const double *Wb, const double *TB, double *VTb,
                           const int *tri, int nb, bool first, hipStream_t s);
// part[b][pr][sp]: part sp of S of the vp x up block that triple b adds to TB's
// adjoint at [k,j], [j,k], [k,i], [i,k], [j,i], [i,j] (pr = 0 .. 5)
hipError_t launch_walk_tbb(const WalkDims &d, const double *Wb, const double *VT, double *part,
                           const int *tri, int nb, int S, hipStream_t s);

// V-bar reductions of a batch (VRArgs with tri set, parts = 1)
hipError_t launch_walk_vr(const VRArgs &a, hipStream_t s);

// gather of a batch into the cotangents (overwritten when first)
struct WalkGather {
  WalkDims d;
  const int *tri;
  int nb, S, G, has_fvo, first;
  const double *part;       // launch_walk_tbb
  const double *R;          // V-bar reductions, r_stride doubles per triple
  size_t r_stride;
  const double *part_t;     // [nb][G] energy sums of the orbit epilogue
  double *vec;              // scratch [nb][6][vp]
  double *t1_bar, *t2_bar, *ovoo_bar, *ovov_bar, *fvo_bar;
  double *tri_e;            // triple energies (null: not wanted)
};
hipError_t launch_walk_gather(const WalkGather &g, hipStream_t s);
// tri_e of nb triples from the orbit epilogue's G sums each
hipError_t launch_walk_energies(const int *tri, int nb, int o, const double *part_t, int G, double *tri_e,
                                hipStream_t s);

// dst[0 .. n) = src (host), through kernel arguments: no copy to wait for or to
// record in a captured graph
hipError_t launch_walk_upload(const double *src, size_t n, double *dst, hipStream_t s);
// pair_e[j o + k] of np pairs from their G part_t sums (launch_walk_acc)
hipError_t launch_walk_pair_energies(const double *part_t, int G, const int *tri, int np, int o,
                                     double *pair_e, hipStream_t s);
// ulo_bar[f][l] (+)= sum over np pairs of g_jk sum of the G part_u rows of (l, j, k)
hipError_t launch_walk_ulo(const double *part_u, int G, int nfrag, double ebar, const int *tri, int np, int o,
                           bool first, double *ulo_bar, hipStream_t s);

// at exit: ovvv_bar from VTb, its hole part added to t2_bar, and
// mo_energy_bar from the rows of part_mo (o + vp columns; part2: scratch of
// kWalkMoParts (o + vp))
constexpr int kWalkMoParts = 64;
hipError_t launch_walk_finish(const WalkDims &d, const double *VTb, int packed, double *ovvv_bar,
                              double *t2_bar, const double *part_mo, int rows, double *part2,
                              double *mo_bar, hipStream_t s);

}  // namespace pamd
