// Host driver and C ABI for the (T) energy and its adjoint.
//
// Walk: occupied triples i <= j <= k (i == j == k contributes nothing: X is then
// fully symmetric and r3(X) = 0).  Per triple:
//   1. W build -- three segmented MFMA GEMMs write W_ijk[a,b,c] (v^3):
//        pass C  (rows (a,b), cols c):  P1 + P3 + H5 + H6
//        pass B  (rows b, cols (a,c)):  P2 + P5 + H3 + H4
//        pass A  (rows a, cols (b,c)):  P4 + P6 + H1 + H2
//      (P1..P6 / H1..H6: the six joint permutations of the particle / hole
//      term of w_abc[ijk], pyscfadlib/pyscfadlib/vjp/cc/ccsd_t.c:121-142 with
//      the permutation tables of ccsd_t.c:74-96).
//   2. orbit epilogue: V, Z = r3(W + V), 1/D, energy; for the adjoint also
//      Wbar, Vbar and dE/d(mo_energy) (ccsd_t_vjp.c:42-117).
//   3. adjoint (ccsd_t_vjp.c:139-269 restated as large contractions):
//        ovvv_bar  -- 3 GEMMs into the Vp-layout accumulator (rows = pairs)
//        t2_bar    -- 6 split-K GEMMs (K = a virtual pair) + V-term pieces
//        ovoo_bar  -- 6 split-K GEMMs (hole terms)
//        t2_bar    -- 3 GEMMs for the hole-term t2 reads (T2m layout)
//        ovov_bar, t1_bar, fvo_bar -- Vbar contractions (k_vr_*) + gather.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <algorithm>
#include <climits>
#include <vector>
#include <atomic>
#include <chrono>
#include <mutex>
#include "ccsdt_common.h"
#include "gemm_desc.h"
#include "walk64.h"
#include "../../include/pyscfad_amd_ccsdt.h"
#include "../../include/pyscfad_amd_debug.h"

namespace pamd {

static const int kGmax = 1024;

// When set, GEMM launches are recorded instead of run and the other per-triple
// kernels are skipped (host-only descriptor inspection, no GPU work).  Per host
// thread, like every other piece of per-call state here.
static thread_local std::vector<GemmDesc> *g_record = nullptr;
// with it, when set: the launch that each recorded descriptor belongs to
static thread_local std::vector<int> *g_record_launch = nullptr;

// Sampled launch timing (pamd_profile_*): for one triple in g_prof_every, every
// launch is bracketed by hipEvents on its own stream; the events are read after
// the call has been queued completely.
// GEMM kinds: W build; adjoint to ovvv (Vpb), to t2 via split-K partials
// (particle), to ovoo (hole split-K partials), to t2 through T2mb (hole)
enum ProfKind {
  kProfWBuild = 0,
  kProfAdjOvvv,
  kProfAdjT2P,
  kProfAdjOvoo,
  kProfAdjT2H,
  kProfOrbit,
  kProfVR,
  kProfCombine,
  kProfNum
};
static const char *kProfNames[kProfNum] = {"gemm_wbuild", "gemm_adj_ovvv", "gemm_adj_t2p",
                                           "gemm_adj_ovoo", "gemm_adj_t2h", "orbit_epilogue",
                                           "vbar_reduce", "combine"};
struct ProfRec {
  int kind;
  hipEvent_t a, b;
  double flops, bytes;
};
struct ProfStat {
  long long launches;
  double ms, flops, bytes;
};
// The switches and the accumulated statistics are process-wide (read and reset
// through pamd_profile_*, the statistics under g_prof_mutex); whether the current
// triple is sampled, and its pending event records, belong to the calling thread,
// so concurrent calls from different host threads never see each other's state.
static std::atomic<int> g_prof_every{0};
static std::atomic<int> g_progress_every{0};  // report (to stderr) every N triples, after a stream sync
static thread_local bool g_prof_on = false;  // sampling the current triple
// set for the duration of a call that must not allocate: no event records then
static thread_local bool g_prof_blocked = false;
static thread_local std::vector<ProfRec> g_prof_recs;
static ProfStat g_prof_stat[kProfNum];
static std::mutex g_prof_mutex;

static hipError_t prof_begin(hipStream_t s, ProfRec &r, int kind, double flops, double bytes) {
  r.kind = kind;
  r.flops = flops;
  r.bytes = bytes;
  hipError_t e = hipEventCreate(&r.a);
  if (e != hipSuccess) return e;
  e = hipEventCreate(&r.b);
  if (e != hipSuccess) return e;
  return hipEventRecord(r.a, s);
}

static hipError_t prof_end(hipStream_t s, ProfRec &r) {
  hipError_t e = hipEventRecord(r.b, s);
  g_prof_recs.push_back(r);
  return e;
}

static hipError_t prof_collect() {
  hipError_t first = hipSuccess;
  for (ProfRec &r : g_prof_recs) {
    float ms = 0.f;
    hipError_t e = hipEventSynchronize(r.b);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, r.a, r.b);
    if (e == hipSuccess) {
      std::lock_guard<std::mutex> lock(g_prof_mutex);
      ProfStat &st = g_prof_stat[r.kind];
      st.launches += 1;
      st.ms += ms;
      st.flops += r.flops;
      st.bytes += r.bytes;
    } else if (first == hipSuccess) {
      first = e;
    }
    hipEventDestroy(r.a);
    hipEventDestroy(r.b);
  }
  g_prof_recs.clear();
  return first;
}

static double gemm_flops(const GemmDesc &d) {
  double k = 0;
  for (int q = 0; q < d.nseg; ++q) k += d.seg[q].L;
  return 2.0 * d.M * (double)d.N * k;
}

// timed launch wrapper for any kernel
template <class F>
static hipError_t timed(hipStream_t s, int kind, double flops, double bytes, F &&launch) {
  if (!g_prof_on || g_prof_blocked) return launch();
  ProfRec r;
  hipError_t e = prof_begin(s, r, kind, flops, bytes);
  if (e != hipSuccess) return e;
  e = launch();
  if (e != hipSuccess) return e;
  return prof_end(s, r);
}

static long long num_triples(int o) { return (long long)o * (o + 1) * (o + 2) / 6 - o; }

struct Layout {
  // extents the operand arrays are laid out with: (o, v), or with pad their
  // multiples of 8
  int pad, op, vp;
  size_t off_t1, off_fvo, off_mo, off_tab;
  size_t off_Vp, off_T2m, off_OOt, off_OVS, off_T2S, off_orb, off_W, off_tri, off_part_t, off_T2g, off_W8;
  int wbatch;  // W blocks of the energy walk's batched W build (1 with the adjoint)
  size_t off_Vb, off_Vpb, off_T2mb, off_part_mo, off_R, off_part_p, off_part_h, off_wt;
  // transposed planar copies of Vp (split-BF16x3 W build; see vpt_fits)
  int vpt;
  size_t off_VpT, off_VpU;
  // pipelined adjoint walk: second copies of the per-triple buffers
  int pipe;
  size_t off_W2, off_W8b, off_R2, off_part_p2, off_part_h2;
  size_t total;
  int S_p, S_h;
};

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

static int device_cus() {
  static int cus = [] {
    int dev = 0, n = 256;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
      n = prop.multiProcessorCount;
    return n > 0 ? n : 256;
  }();
  return cus;
}

// Split-K factor for an M x N output with `chunks` K chunks of 16: one full
// round of resident workgroups (two per CU for the FP64 engine and for the
// split-BF16x3 16x16-MFMA tiles, one for its 32x32 tiles), rounded down so
// that no workgroup waits for a second round.  (One round measured faster than two or three: fewer split-K
// partials to write and reduce, same engine time.)
// The split-BF16x3 two-workgroup tiles sum each output tile in FP32 over the
// workgroup's whole K range, so the split count is also raised until no part
// spans more than kB3MaxK terms: the FP32 rounding of those sums then stays
// bounded as v grows (K = v^2 for the particle-side t2 adjoint).  At v = 400 one
// round of workgroups already gives 25 parts of 6400 terms, so this bound only
// acts at larger v.
constexpr int kB3MaxK = 8192;
static int splits_for(int M, int N, int chunks, int prec) {
  const bool b3 = prec == PAMD_PREC_BF16X3;
  const int tiles = std::max(1, b3 ? gemm_tiles_b3(M, N) : gemm_tiles(M, N, prec == PAMD_PREC_FP32X2));
  const int slots = (b3 ? gemm_wgs_per_cu_b3(M, N) : 2) * device_cus();
  int s = slots / tiles;
  if (b3) s = std::max(s, (int)(((long long)chunks * KC + kB3MaxK - 1) / kB3MaxK));
  s = std::max(1, std::min(s, 512));
  return std::min(s, std::max(1, b3 ? chunks / 2 : chunks));
}

// Consecutive k of one occupied pair (i, j) share the W build of the energy walk
// when one triple's W-build GEMM has too few workgroup tiles to fill the GPU:
// about four rounds of the resident workgroups per launch, at most 8 triples,
// their W blocks within 2 GB.  (At nvir = 400 one triple already has ~6000
// tiles: no batching.)
static int energy_batch(int o, int v, int prec) {
  const long long tiles = prec == PAMD_PREC_BF16X3 ? gemm_tiles_b3(v * v, v)
                                                    : gemm_tiles(v * v, v, prec == PAMD_PREC_FP32X2);
  const long long slots = 2LL * device_cus();
  long long b = (4 * slots + tiles - 1) / std::max(1LL, tiles);
  b = std::max(1LL, std::min(8LL, b));
  const long long v3 = (long long)v * v * v;
  while (b > 1 && b * v3 * (long long)sizeof(double) > (2LL << 30)) --b;
  return (int)std::min<long long>(b, o);
}

// Vp, T2m and OOt hold FP64 copies, or their split forms: three bf16 planes
// (split-BF16x3, 6 of the 8 bytes per element) or packed FP32 hi/lo pairs; the
// split precisions add split copies of t2 and of Wbar.
// Transposed planar copies of Vp make every particle-term ovvv operand of the
// split-BF16x3 W build row-contiguous, the faster of the direct engine's two
// staging forms (the big operand of all three passes).  They take two o v^3
// arrays; held when the direct engine runs the W build (nocc and nvir
// multiples of 8, or padded to them) and the copies stay within 48 GB.
static bool vpt_fits(int o, int op, int v, int prec) {
  const double bytes = 2.0 * 8.0 * o * (double)v * v * v;
  return prec == PAMD_PREC_BF16X3 && op % 8 == 0 && v % 8 == 0 && bytes <= 48e9 &&
         gemm_b3p_enabled();
}

// pipe: the adjoint walk runs two triples in flight (run_vjp_pipelined) and
// needs second copies of W, Wbar, the V-bar scratch and the split-K partials
// pad: split-BF16x3 operands with both extents padded to multiples of 8 by zeros.
// Every operand is then 16-byte aligned, so the W build and the ovvv adjoints run
// on the direct engine at every size, and the epilogue is the batched walk's
// (walk64_orbit.hip), which needs whole 8 x 8 x 8 tiles.  Measured, E + VJP at
// o6/v400 (nocc padded): 910 -> 790 ms; at o16/v160 (epilogue alone): 660 -> 636;
// energy at o24/v240 (epilogue alone, 153 -> 65 us per triple): 1601 -> 1479.
// The split-K products keep the unpadded extents: padding would cut their sums
// over (p, q) differently.
static Layout make_layout(int o, int v, int vjp, int prec, bool pipe = false, bool pad = false) {
  Layout L;
  memset(&L, 0, sizeof(L));
  L.pad = pad ? 1 : 0;
  L.op = pad ? (o + 7) / 8 * 8 : o;
  L.vp = pad ? (v + 7) / 8 * 8 : v;
  const size_t d = sizeof(double);
  const size_t vp = L.vp, v2 = vp * vp, v3 = v2 * vp, n = (size_t)o + vp, t2m = o * v2 * L.op;
  const size_t vv = (size_t)v * v;
  size_t off = 0;
  auto take = [&](size_t count) {
    size_t at = off;
    off = align256(off + count * d);
    return at;
  };
  L.off_Vp = take((size_t)o * v3);
  L.off_T2m = take(t2m);
  L.off_OOt = take((size_t)o * o * L.op * vp);
  L.off_OVS = take((size_t)o * o * v2);
  L.off_T2S = take((size_t)o * o * v2);
  const size_t nt = (v + 7) / 8, norb = nt * (nt + 1) * (nt + 2) / 6;
  L.off_orb = take(norb);  // 4 x uint16 per orbit = one double
  L.wbatch = vjp ? 1 : energy_batch(o, L.vp, prec);
  L.off_W = take(v3 * L.wbatch);
  L.off_tri = take((size_t)o * o * o);
  L.off_part_t = take((size_t)kGmax * (pad ? L.wbatch : 1));
  L.off_wt = take((size_t)o);
  if (pad) {
    L.off_t1 = take((size_t)o * vp);
    L.off_fvo = take((size_t)o * vp);
    L.off_mo = take(n);
    L.off_tab = take((size_t)(num_triples(o) + kWalkRun) / 2 + 1);
  }
  if (prec == PAMD_PREC_BF16X3 || prec == PAMD_PREC_FP32X2) {
    L.off_T2g = take((size_t)o * o * v2);
    if (vjp) L.off_W8 = take(v3);
  }
  const int chunks = (int)((vv + KC - 1) / KC);
  L.S_p = splits_for(v, v, chunks, prec);
  L.S_h = splits_for(v, o, chunks, prec);
  if (vjp) {
    L.off_Vb = take(v3);
    L.off_Vpb = take((size_t)o * v3);
    L.off_T2mb = take(t2m);
    L.off_part_mo = take((size_t)kGmax * n);
    L.off_R = take(vr_scratch_doubles(L.vp));
    L.off_part_p = take((size_t)6 * L.S_p * vv);
    L.off_part_h = take((size_t)6 * L.S_h * v * L.op);
  }
  L.vpt = vpt_fits(o, L.op, L.vp, prec) ? 1 : 0;
  if (L.vpt) {
    L.off_VpT = take((size_t)o * v3);
    L.off_VpU = take((size_t)o * v3);
  }
  L.pipe = (vjp && pipe) ? 1 : 0;
  if (L.pipe) {
    L.off_W2 = take(v3);
    if (prec == PAMD_PREC_BF16X3 || prec == PAMD_PREC_FP32X2) L.off_W8b = take(v3);
    L.off_R2 = take(vr_scratch_doubles(L.vp));
    L.off_part_p2 = take((size_t)6 * L.S_p * vv);
    L.off_part_h2 = take((size_t)6 * L.S_h * v * L.op);
  }
  L.total = off;
  return L;
}

// The layout of a plain walk: padded for the split-BF16x3 engine (`plain`, the
// unpadded one, stays where the direct engine is off, `limit` bytes do not hold
// the padded arrays or these are noticeably larger in a workspace that is large
// itself).
static Layout b3_layout(int o, int v, int vjp, int prec, bool pipe, size_t limit, const Layout &plain) {
  const long long vp = (v + 7) / 8 * 8;
  if (prec != PAMD_PREC_BF16X3 || !gemm_b3p_enabled() || vp * vp * vp >= (1LL << 31)) return plain;
  const Layout P = make_layout(o, v, vjp, prec, pipe, true);
  const bool big = P.total > ((size_t)100 << 30) && P.total > plain.total + plain.total / 20;
  return P.total > limit || big ? plain : P;
}

// Planar split-BF16x3 operands: the arrays the walk's descriptors point into
// (Vp, T2m, OOt, t2 copy, Wbar copy), allocated as FP64 (8 bytes per element)
// and holding three bf16 planes of their element count in the first 6 bytes.
// A descriptor built with FP64 element arithmetic is moved onto them: element
// e of an array becomes bf16 element e of its hi plane, with the array's
// element count as the plane stride.
struct PlanarMap {
  const char *base[8];
  long long n[8];
  int count;
};

struct Ctx {
  int o, v, packed, has_fvo, vjp, prec;
  int pad, op, vp;    // extents the arrays are laid out with (Layout)
  double *t1p, *fvop, *mop;  // padded copies (pad)
  int *tab;                  // triples in walk order (pad)
  const double *gT2;  // t2 as a GEMM operand (FP64, or its split copy)
  unsigned short *orb;  // orbit table
  double *gW;         // Wbar as a GEMM operand (= W, or its split copy)
  hipStream_t s;
  const double *mo, *t1, *t2, *ovvv, *ovoo, *ovov, *fvo;
  double *Vp, *T2m, *OOt, *OVS, *T2S, *W, *tri, *part_t;
  double *Vb, *Vpb, *T2mb, *part_mo, *R, *part_p, *part_h;
  int S_p, S_h, G;
  int f32_p, f32_h;   // the split-K parts are FP32 (kPartialF32)
  int wbatch;  // W blocks available to the energy walk's batched W build
  double ebar;
  int shard, nshards;     // this call covers walk triples with index % nshards == shard
  const double *wt_host;  // occupied weights m (host) of a diagonal projector, or null
  double *wt;             // device copy of m
  PlanarMap planes;       // split-BF16x3 operand arrays
  // transposed planar copies of Vp for the W build (split-BF16x3, when the
  // layout holds them): VpT[x][f][p][q] = VpU[x][f][q][p] = Vp[x][p][q][f]
  double *VpT, *VpU;
  // pipelined adjoint walk (pipe = 1): the second set of per-triple buffers
  int pipe;
  double *W2, *gW2, *R2, *part_p2, *part_h2;
  // outputs
  double *t1_bar, *t2_bar, *ovoo_bar, *ovov_bar, *fvo_bar;
};

static bool planarize(const PlanarMap &pm, OpDesc &o) {
  const char *p = (const char *)o.p;
  for (int a = 0; a < pm.count; ++a) {
    if (p < pm.base[a] || p >= pm.base[a] + pm.n[a] * (long long)sizeof(double)) continue;
    const long long e = (p - pm.base[a]) / (long long)sizeof(double);
    o.p = (const double *)(pm.base[a] + 2 * e);
    o.ps = pm.n[a];
    return true;
  }
  return false;
}

// one contraction in the precision of the call that issues it
static hipError_t run_gemm(const Ctx &c, const GemmDesc &d0, int kind,
                           const GemmBatch &bt = no_batch()) {
  if (g_record) {
    if (g_record_launch) g_record_launch->push_back((int)g_record->size());
    g_record->push_back(d0);
    return hipSuccess;
  }
  const double fl = gemm_flops(d0) * bt.nb;
  const hipStream_t s = c.s;
  if (c.prec == PAMD_PREC_BF16X3) {
    GemmDesc d = d0;
    for (int q = 0; q < d.nseg; ++q)
      if (!planarize(c.planes, d.seg[q].A) || !planarize(c.planes, d.seg[q].B))
        return hipErrorInvalidValue;
    return timed(s, kind, fl, 0.0, [&] { return launch_gemm_bf16x3(d, s, bt); });
  }
  if (c.prec == PAMD_PREC_FP32X2)
    return timed(s, kind, fl, 0.0, [&] { return launch_gemm_f32x2(d0, s, bt); });
  return timed(s, kind, fl, 0.0, [&] { return launch_gemm_f64(d0, s, bt); });
}

// Group launches of the adjoint families: env PYSCFAD_AMD_GROUP = 0 never,
// 1 always; unset: when the three bf16 planes of Wbar (6 v^3 bytes, read by
// every product of a family) fit in half of the GPU's 256 MB last-level
// cache.  Measured E+VJP: o16/v160 0.634 -> 0.602 s and o24/v240 5.61 ->
// 5.44 s with groups, o40/v400 134.7 -> 138.6 s (the products of a group then
// stream different ovvv slabs and Wbar orders through the cache at once).
static int group_mode() {
  static const int m = [] {
    const char *e = getenv("PYSCFAD_AMD_GROUP");
    return e ? (e[0] == '0' ? 0 : 1) : -1;
  }();
  return m;
}
constexpr double kGroupWbarBytes = 128.0 * (1 << 20);

// n independent contractions of one kind: in the split-BF16x3 form one group
// launch when their outputs are disjoint (out_disjoint), they fit the direct
// engine's group and grouping is on for their size, else one launch each
static hipError_t run_gemm_group(const Ctx &c, const GemmDesc *ds, int n, int kind,
                                 bool out_disjoint) {
  const int gm = group_mode();
  const bool group = c.prec == PAMD_PREC_BF16X3 && out_disjoint && n <= kMaxGroup &&
                     (gm == 1 || (gm < 0 && 6.0 * c.v * (double)c.v * c.v <= kGroupWbarBytes));
  if (g_record || !group) {
    const int first = g_record ? (int)g_record->size() : 0;
    for (int q = 0; q < n; ++q) {
      const hipError_t e = run_gemm(c, ds[q], kind);
      if (e != hipSuccess) return e;
      if (g_record && g_record_launch && group) g_record_launch->back() = first;
    }
    return hipSuccess;
  }
  GemmDesc d[kMaxGroup];
  double fl = 0.0;
  for (int q = 0; q < n; ++q) {
    d[q] = ds[q];
    for (int p = 0; p < d[q].nseg; ++p)
      if (!planarize(c.planes, d[q].seg[p].A) || !planarize(c.planes, d[q].seg[p].B))
        return hipErrorInvalidValue;
    fl += gemm_flops(d[q]);
  }
  return timed(c.s, kind, fl, 0.0, [&] { return launch_gemm_bf16x3_group(d, n, c.s); });
}

#define PAMD_CHECK(expr)                                                      \
  do {                                                                        \
    hipError_t e_ = (expr);                                                   \
    if (e_ != hipSuccess) {                                                   \
      fprintf(stderr, "pyscfad_amd: %s failed: %s\n", #expr, hipGetErrorString(e_)); \
      return PAMD_ERR_HIP;                                                    \
    }                                                                         \
  } while (0)

// ---------------------------------------------------------------------------
// W build for one triple
// ---------------------------------------------------------------------------
// sums of a product on padded arrays whose unpadded extents are M x N; aligned:
// the direct engine would take it unpadded too
static int b3_sums(const Ctx &c, int M, int N, bool aligned) {
  return c.pad && !aligned ? (int)gemm_b3_sums(M, N) : (int)kSumsAuto;
}

// nb > 1: the W blocks of triples (i, j, k), (i, j, k + 1), ..., (i, j, k + nb - 1)
// in one launch per pass, written to W + b v^3 (every operand slab that names
// k moves by a fixed stride per step of k).
static int build_w(const Ctx &c, int i, int j, int k, int nb = 1) {
  const long long o = c.o, os = c.op, v = c.vp;
  const long long v2 = v * v, v3 = v2 * v, vo = v * os;
  // element strides per step of k of: Vp(k), T2(k, x), T2(x, k), OOt(k, x), OOt(x, k), T2m(k)
  const long long sVp = v3, sT2k_ = o * v2, sT2_k = v2, sOOk_ = o * vo, sOO_k = vo, sT2m = v2 * os;
  auto batch = [&](std::initializer_list<long long> a, std::initializer_list<long long> bo) {
    GemmBatch bt = no_batch();
    int q = 0;
    for (long long x : a) bt.a[q++] = x;
    q = 0;
    for (long long x : bo) bt.bo[q++] = x;
    bt.c = v3;
    bt.nb = nb;
    return bt;
  };
  auto Vp = [&](int x) { return c.Vp + x * v3; };
  auto T2 = [&](int x, int y) { return c.gT2 + (x * o + y) * v2; };
  auto T2m = [&](int x) { return c.T2m + x * v2 * os; };
  auto OOt = [&](int x, int y) { return c.OOt + (x * o + y) * vo; };
  const int V = c.vp, O = c.op;
  const bool whole = c.v % 8 == 0 && c.o % 8 == 0;
  const int sumsC = b3_sums(c, c.v * c.v, c.v, whole), sumsR = b3_sums(c, c.v, c.v * c.v, whole);
  // the ovvv slab of a particle term with its row pair (q, s) read as
  // Vp(x)[q][s][f] ("qs") or Vp(x)[s][q][f] ("sq"), K = f: from Vp itself
  // (K-contiguous), or, when the call holds the transposed copies, from
  // VpT(x)[f][q][s] / VpU(x)[f][q][s] (row-contiguous)
  auto Pqs = [&](int x) {
    return c.VpT ? opR(c.VpT + x * v3, v, 1, V, v2, 1) : opR(Vp(x), v2, v, V, 1, 0);
  };
  auto Psq = [&](int x) {
    return c.VpU ? opR(c.VpU + x * v3, v, 1, V, v2, 1) : opR(Vp(x), v, v2, V, 1, 0);
  };
  // pass C: rows (a,b), cols c
  {
    GemmDesc d = gemm(V * V, V, kStore,
                      {seg(Pqs(i), op1(T2(k, j), v, 1, 0), V, 1.0),      // P1
                       seg(Psq(j), op1(T2(k, i), v, 1, 0), V, 1.0),      // P3
                       seg(opR(T2m(j), os, vo, V, 1, 0), op1(OOt(k, i), os, 1, 0), O, -1.0),   // H5
                       seg(opR(T2m(i), vo, os, V, 1, 0), op1(OOt(k, j), os, 1, 0), O, -1.0)},  // H6
                      out(c.W, v2, v, V, 0, 1, kBig));
    d.sums = sumsC;
    // P1: T2(k,j), P3: T2(k,i), H5: OOt(k,i), H6: OOt(k,j)
    PAMD_CHECK(run_gemm(c, d, kProfWBuild,
                        batch({0, 0, 0, 0}, {sT2k_, sT2k_, sOOk_, sOOk_})));
  }
  // pass B: rows b, cols (a,c)
  {
    GemmDesc d = gemm(V, V * V, kAccumulate,
                      {seg(op1(T2(j, k), v, 1, 0), Pqs(i), V, 1.0),      // P2
                       seg(op1(T2(j, i), v, 1, 0), Psq(k), V, 1.0),      // P5
                       seg(op1(OOt(j, i), os, 1, 0), opR(T2m(k), os, vo, V, 1, 0), O, -1.0),   // H3
                       seg(op1(OOt(j, k), os, 1, 0), opR(T2m(i), vo, os, V, 1, 0), O, -1.0)},  // H4
                      out(c.W, 0, v, kBig, v2, 1, V));
    d.sums = sumsR;
    // P2: T2(j,k) | Vp(i), P5: T2(j,i) | Vp(k), H3: OOt(j,i) | T2m(k), H4: OOt(j,k) | T2m(i)
    PAMD_CHECK(run_gemm(c, d, kProfWBuild,
                        batch({sT2_k, 0, 0, sOO_k}, {0, sVp, sT2m, 0})));
  }
  // pass A: rows a, cols (b,c)
  {
    GemmDesc d = gemm(V, V * V, kAccumulate,
                      {seg(op1(T2(i, k), v, 1, 0), Pqs(j), V, 1.0),      // P4
                       seg(op1(T2(i, j), v, 1, 0), Psq(k), V, 1.0),      // P6
                       seg(op1(OOt(i, j), os, 1, 0), opR(T2m(k), os, vo, V, 1, 0), O, -1.0),   // H1
                       seg(op1(OOt(i, k), os, 1, 0), opR(T2m(j), vo, os, V, 1, 0), O, -1.0)},  // H2
                      out(c.W, 0, v2, kBig, v, 1, V));
    d.sums = sumsR;
    // P4: T2(i,k) | Vp(j), P6: T2(i,j) | Vp(k), H1: OOt(i,j) | T2m(k), H2: OOt(i,k) | T2m(j)
    PAMD_CHECK(run_gemm(c, d, kProfWBuild,
                        batch({sT2_k, 0, 0, sOO_k}, {0, sVp, sT2m, 0})));
  }
  return PAMD_OK;
}

// ---------------------------------------------------------------------------
// adjoint of one triple (c.gW holds Wbar, c.Vb holds Vbar): the V-bar
// reductions into c.R, the adjoint contractions (stream c.s) into Vpb, T2mb
// and the split-K partials c.part_p, c.part_h, and the gather of R and the
// partials into the cotangents
// ---------------------------------------------------------------------------
static int adjoint_vr(const Ctx &c, int i, int j, int k, hipStream_t st) {
  const double v3 = (double)c.v * c.v * c.v;
  VRArgs vr;
  memset(&vr, 0, sizeof(vr));
  vr.parts = kVRS;
  vr.Vb = c.Vb;
  vr.t1 = c.pad ? c.t1p : c.t1;
  vr.fvo = c.pad ? c.fvop : c.fvo;
  vr.ovs = c.OVS;
  vr.t2s = c.T2S;
  vr.o = c.o;
  vr.v = c.vp;
  vr.i = i;
  vr.j = j;
  vr.k = k;
  vr.has_fvo = c.has_fvo;
  vr.R = c.R;
  if (!g_record) {
    const double vb = 2.0 * 8.0 * v3;  // Vbar read twice
    PAMD_CHECK(timed(st, kProfVR, 0.0, vb, [&] { return launch_vr(vr, st); }));
  }
  return PAMD_OK;
}

// pair: 0 all three ovvv adjoints (and hole-term t2 adjoints) of the triple;
// 1 only those into Vpb[k] and T2mb[k] (those into index i and j wait for the
// next triple (i, j, k'), which shares them); 2 those into Vpb[i], Vpb[j],
// T2mb[i], T2mb[j] as four-segment launches that also take the terms of the
// previous triple (i, j, kp) from its own Wbar buffer (prev->gW), plus the
// ones into Vpb[k] and T2mb[k]
static int adjoint_gemms(const Ctx &c, int i, int j, int k, int pair = 0, const Ctx *prev = nullptr,
                         int kp = 0) {
  const long long o = c.o, os = c.op, v = c.vp;
  const long long v2 = v * v, v3 = v2 * v, vo = v * os;
  const int V = c.vp, O = c.op, V0 = c.v, O0 = c.o;
  const int sums_v = b3_sums(c, V0 * V0, V0, V0 % 8 == 0),
            sums_h = b3_sums(c, V0 * V0, O0, V0 % 8 == 0 && O0 % 8 == 0);
  const double *Wb = c.gW;
  auto Vp = [&](int x) { return c.Vp + x * v3; };
  auto Vpb = [&](int x) { return c.Vpb + x * v3; };
  auto T2 = [&](int x, int y) { return c.gT2 + (x * o + y) * v2; };
  auto T2m = [&](int x) { return c.T2m + x * v2 * os; };
  auto T2mb = [&](int x) { return c.T2mb + x * v2 * os; };
  auto OOt = [&](int x, int y) { return c.OOt + (x * o + y) * vo; };

  // the three adjoints into Vpb[i], Vpb[j], Vpb[k] and into T2mb[i], T2mb[j],
  // T2mb[k] write disjoint slabs unless two occupied indices coincide (any two: the
  // projected walk's triples are not sorted, so i == k with another j occurs)
  const bool distinct = i != j && j != k && i != k;
  // ovvv_bar, rows = virtual pairs, cols = f
  if (pair != 0) {
    const double *Wq = prev ? prev->gW : nullptr;
    GemmDesc ds[3];
    int n = 0;
    if (pair == 2) {
      ds[n++] = gemm(V * V, V, kAccumulate,
                     {seg(opR(Wq, v2, v, V, 1, 0), op1(T2(kp, j), 1, v, 1), V, 1.0),
                      seg(opR(Wq, v2, 1, V, v, 1), op1(T2(j, kp), 1, v, 1), V, 1.0),
                      seg(opR(Wb, v2, v, V, 1, 0), op1(T2(k, j), 1, v, 1), V, 1.0),
                      seg(opR(Wb, v2, 1, V, v, 1), op1(T2(j, k), 1, v, 1), V, 1.0)},
                     out(Vpb(i), v2, v, V, 0, 1, kBig));
      ds[n++] = gemm(V * V, V, kAccumulate,
                     {seg(opR(Wq, v, v2, V, 1, 0), op1(T2(kp, i), 1, v, 1), V, 1.0),
                      seg(opR(Wq, v, 1, V, v2, 1), op1(T2(i, kp), 1, v, 1), V, 1.0),
                      seg(opR(Wb, v, v2, V, 1, 0), op1(T2(k, i), 1, v, 1), V, 1.0),
                      seg(opR(Wb, v, 1, V, v2, 1), op1(T2(i, k), 1, v, 1), V, 1.0)},
                     out(Vpb(j), v2, v, V, 0, 1, kBig));
    }
    ds[n++] = gemm(V * V, V, kAccumulate,
                   {seg(opR(Wb, v2, 1, V, v, 1), op1(T2(j, i), 1, v, 1), V, 1.0),
                    seg(opR(Wb, v, 1, V, v2, 1), op1(T2(i, j), 1, v, 1), V, 1.0)},
                   out(Vpb(k), v, v2, V, 0, 1, kBig));
    for (int q = 0; q < n; ++q) {
      ds[q].sums = sums_v;
      PAMD_CHECK(run_gemm(c, ds[q], kProfAdjOvvv));
    }
  } else {
    GemmDesc ds[3] = {
        // Vpb[i][a][b|c][f]: P1 (K=c), P2 (K=b)
        gemm(V * V, V, kAccumulate,
             {seg(opR(Wb, v2, v, V, 1, 0), op1(T2(k, j), 1, v, 1), V, 1.0),
              seg(opR(Wb, v2, 1, V, v, 1), op1(T2(j, k), 1, v, 1), V, 1.0)},
             out(Vpb(i), v2, v, V, 0, 1, kBig)),
        // Vpb[j][b][a|c][f]: P3 (K=c), P4 (K=a)
        gemm(V * V, V, kAccumulate,
             {seg(opR(Wb, v, v2, V, 1, 0), op1(T2(k, i), 1, v, 1), V, 1.0),
              seg(opR(Wb, v, 1, V, v2, 1), op1(T2(i, k), 1, v, 1), V, 1.0)},
             out(Vpb(j), v2, v, V, 0, 1, kBig)),
        // Vpb[k][c][a|b][f]: rows m = y*v + x with x = c: P5 (K=b), P6 (K=a)
        gemm(V * V, V, kAccumulate,
             {seg(opR(Wb, v2, 1, V, v, 1), op1(T2(j, i), 1, v, 1), V, 1.0),
              seg(opR(Wb, v, 1, V, v2, 1), op1(T2(i, j), 1, v, 1), V, 1.0)},
             out(Vpb(k), v, v2, V, 0, 1, kBig)),
    };
    for (GemmDesc &d : ds) d.sums = sums_v;
    PAMD_CHECK(run_gemm_group(c, ds, 3, kProfAdjOvvv, distinct));
  }

  // particle t2_bar pieces: split-K over the virtual pair, partials per problem
  const size_t pp = (size_t)c.S_p * V0 * V0;
  {
    const int mode_p = c.f32_p ? kPartialF32 : kPartial;
    GemmDesc ds[6] = {
        // P1: t2_bar[k,j][c][f] = sum_(a,b) Wb[a,b,c] Vp(i)[a][b][f]
        gemm(V0, V0, mode_p, {seg(opK(Wb, 1, v2, v, V0, 1), opK(Vp(i), 1, v2, v, V0, 1), V0 * V0, 1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_p, c.part_p + 0 * pp),
        // P2: t2_bar[j,k][b][f] = sum_(a,c) Wb[a,b,c] Vp(i)[a][c][f]
        gemm(V0, V0, mode_p, {seg(opK(Wb, v, v2, 1, V0, 0), opK(Vp(i), 1, v2, v, V0, 1), V0 * V0, 1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_p, c.part_p + 1 * pp),
        // P3: t2_bar[k,i][c][f] = sum_(a,b) Wb[a,b,c] Vp(j)[b][a][f]
        gemm(V0, V0, mode_p, {seg(opK(Wb, 1, v2, v, V0, 1), opK(Vp(j), 1, v, v2, V0, 1), V0 * V0, 1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_p, c.part_p + 2 * pp),
        // P4: t2_bar[i,k][a][f] = sum_(b,c) Wb[a,b,c] Vp(j)[b][c][f]
        gemm(V0, V0, mode_p, {seg(opK(Wb, v2, v, 1, V0, 0), opK(Vp(j), 1, v2, v, V0, 1), V0 * V0, 1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_p, c.part_p + 3 * pp),
        // P5: t2_bar[j,i][b][f] = sum_(a,c) Wb[a,b,c] Vp(k)[c][a][f]
        gemm(V0, V0, mode_p, {seg(opK(Wb, v, v2, 1, V0, 0), opK(Vp(k), 1, v, v2, V0, 1), V0 * V0, 1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_p, c.part_p + 4 * pp),
        // P6: t2_bar[i,j][a][f] = sum_(b,c) Wb[a,b,c] Vp(k)[c][b][f]
        gemm(V0, V0, mode_p, {seg(opK(Wb, v2, v, 1, V0, 0), opK(Vp(k), 1, v, v2, V0, 1), V0 * V0, 1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_p, c.part_p + 5 * pp),
    };
    if (c.f32_p)
      for (GemmDesc &d : ds) d.sums = kSumsWhole;
    PAMD_CHECK(run_gemm_group(c, ds, 6, kProfAdjT2P, true));
  }
  // hole ovoo_bar pieces: split-K over the virtual pair
  const int N = c.pad ? c.op : O0;  // (padded: direct loads of T2m's rows)
  const int sums_o = b3_sums(c, V0, O0, V0 % 8 == 0 && O0 % 8 == 0);
  const size_t ph = (size_t)c.S_h * V0 * N;
  {
    const int mode_h = c.f32_h ? kPartialF32 : kPartial;
    GemmDesc ds[6] = {
        // H1: ovoo_bar[i,a,m,j] = -sum_(b,c) Wb[a,b,c] T2m(k)[c][b][m]
        gemm(V0, N, mode_h, {seg(opK(Wb, v2, v, 1, V0, 0), opK(T2m(k), 1, os, vo, V0, 1), V0 * V0, -1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_h, c.part_h + 0 * ph),
        // H2: ovoo_bar[i,a,m,k] = -sum_(b,c) Wb[a,b,c] T2m(j)[b][c][m]
        gemm(V0, N, mode_h, {seg(opK(Wb, v2, v, 1, V0, 0), opK(T2m(j), 1, vo, os, V0, 1), V0 * V0, -1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_h, c.part_h + 1 * ph),
        // H3: ovoo_bar[j,b,m,i] = -sum_(a,c) Wb[a,b,c] T2m(k)[c][a][m]
        gemm(V0, N, mode_h, {seg(opK(Wb, v, v2, 1, V0, 0), opK(T2m(k), 1, os, vo, V0, 1), V0 * V0, -1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_h, c.part_h + 2 * ph),
        // H4: ovoo_bar[j,b,m,k] = -sum_(a,c) Wb[a,b,c] T2m(i)[a][c][m]
        gemm(V0, N, mode_h, {seg(opK(Wb, v, v2, 1, V0, 0), opK(T2m(i), 1, vo, os, V0, 1), V0 * V0, -1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_h, c.part_h + 3 * ph),
        // H5: ovoo_bar[k,c,m,i] = -sum_(a,b) Wb[a,b,c] T2m(j)[b][a][m]
        gemm(V0, N, mode_h, {seg(opK(Wb, 1, v2, v, V0, 1), opK(T2m(j), 1, os, vo, V0, 1), V0 * V0, -1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_h, c.part_h + 4 * ph),
        // H6: ovoo_bar[k,c,m,j] = -sum_(a,b) Wb[a,b,c] T2m(i)[a][b][m]
        gemm(V0, N, mode_h, {seg(opK(Wb, 1, v2, v, V0, 1), opK(T2m(i), 1, vo, os, V0, 1), V0 * V0, -1.0)},
             out(nullptr, 0, 0, 1, 0, 0, 1), c.S_h, c.part_h + 5 * ph),
    };
    for (GemmDesc &d : ds) d.sums = c.f32_h ? (int)kSumsWhole : sums_o;
    PAMD_CHECK(run_gemm_group(c, ds, 6, kProfAdjOvoo, true));
  }
  // hole-term t2 reads: T2mb[x][p][q][m] (= dE/d t2[x,m,p,q])
  if (pair != 0) {
    const double *Wq = prev ? prev->gW : nullptr;
    GemmDesc ds[3];
    int n = 0;
    if (pair == 2) {
      ds[n++] = gemm(V * V, O, kAccumulate,
                     {seg(opR(Wq, v2, 1, V, v, 1), op1(OOt(j, kp), 1, os, 1), V, -1.0),
                      seg(opR(Wq, v2, v, V, 1, 0), op1(OOt(kp, j), 1, os, 1), V, -1.0),
                      seg(opR(Wb, v2, 1, V, v, 1), op1(OOt(j, k), 1, os, 1), V, -1.0),
                      seg(opR(Wb, v2, v, V, 1, 0), op1(OOt(k, j), 1, os, 1), V, -1.0)},
                     out(T2mb(i), vo, os, V, 0, 1, kBig));
      ds[n++] = gemm(V * V, O, kAccumulate,
                     {seg(opR(Wq, v, 1, V, v2, 1), op1(OOt(i, kp), 1, os, 1), V, -1.0),
                      seg(opR(Wq, v, v2, V, 1, 0), op1(OOt(kp, i), 1, os, 1), V, -1.0),
                      seg(opR(Wb, v, 1, V, v2, 1), op1(OOt(i, k), 1, os, 1), V, -1.0),
                      seg(opR(Wb, v, v2, V, 1, 0), op1(OOt(k, i), 1, os, 1), V, -1.0)},
                     out(T2mb(j), vo, os, V, 0, 1, kBig));
    }
    ds[n++] = gemm(V * V, O, kAccumulate,
                   {seg(opR(Wb, v, 1, V, v2, 1), op1(OOt(i, j), 1, os, 1), V, -1.0),
                    seg(opR(Wb, v2, 1, V, v, 1), op1(OOt(j, i), 1, os, 1), V, -1.0)},
                   out(T2mb(k), os, vo, V, 0, 1, kBig));
    for (int q = 0; q < n; ++q) {
      ds[q].sums = sums_h;
      PAMD_CHECK(run_gemm(c, ds[q], kProfAdjT2H));
    }
  } else {
    GemmDesc ds[3] = {
        // T2mb[i]: H4 (p=a,q=c,K=b), H6 (p=a,q=b,K=c)
        gemm(V * V, O, kAccumulate,
             {seg(opR(Wb, v2, 1, V, v, 1), op1(OOt(j, k), 1, os, 1), V, -1.0),
              seg(opR(Wb, v2, v, V, 1, 0), op1(OOt(k, j), 1, os, 1), V, -1.0)},
             out(T2mb(i), vo, os, V, 0, 1, kBig)),
        // T2mb[j]: H2 (p=b,q=c,K=a), H5 (p=b,q=a,K=c)
        gemm(V * V, O, kAccumulate,
             {seg(opR(Wb, v, 1, V, v2, 1), op1(OOt(i, k), 1, os, 1), V, -1.0),
              seg(opR(Wb, v, v2, V, 1, 0), op1(OOt(k, i), 1, os, 1), V, -1.0)},
             out(T2mb(j), vo, os, V, 0, 1, kBig)),
        // T2mb[k]: rows m = q*v + p with p = c: H1 (q=b,K=a), H3 (q=a,K=b)
        gemm(V * V, O, kAccumulate,
             {seg(opR(Wb, v, 1, V, v2, 1), op1(OOt(i, j), 1, os, 1), V, -1.0),
              seg(opR(Wb, v2, 1, V, v, 1), op1(OOt(j, i), 1, os, 1), V, -1.0)},
             out(T2mb(k), os, vo, V, 0, 1, kBig)),
    };
    for (GemmDesc &d : ds) d.sums = sums_h;
    PAMD_CHECK(run_gemm_group(c, ds, 3, kProfAdjT2H, distinct));
  }
  return PAMD_OK;
}

// with_energy: the same launch also sums the orbit epilogue's per-workgroup
// energies of this triple into tri (the walk then skips launch_triple_energy)
static int adjoint_combine(const Ctx &c, int i, int j, int k, hipStream_t st,
                           bool with_energy = false) {
  const double v = c.v, o = c.o, v2 = v * v;
  CombineArgs ca;
  ca.R = c.R;
  ca.part_p = c.part_p;
  ca.part_h = c.part_h;
  ca.S_p = c.S_p;
  ca.S_h = c.S_h;
  ca.f32_p = c.f32_p;
  ca.f32_h = c.f32_h;
  ca.o = c.o;
  ca.v = c.v;
  ca.vp = c.vp;
  ca.op = c.op;
  ca.i = i;
  ca.j = j;
  ca.k = k;
  ca.has_fvo = c.has_fvo;
  ca.t2_bar = c.t2_bar;
  ca.ovov_bar = c.ovov_bar;
  ca.ovoo_bar = c.ovoo_bar;
  ca.t1_bar = c.t1_bar;
  ca.fvo_bar = c.fvo_bar;
  ca.part_t = with_energy ? c.part_t : nullptr;
  ca.G = c.G;
  ca.tri_dst = with_energy ? c.tri + ((size_t)i * c.o + j) * c.o + k : nullptr;
  if (!g_record) {
    const double cb = 8.0 * (6.0 * c.S_p * v2 + 6.0 * c.S_h * v * c.op + 12.0 * v2);
    PAMD_CHECK(timed(st, kProfCombine, 0.0, cb, [&] { return launch_combine(ca, st); }));
  }
  return PAMD_OK;
}

static int adjoint(const Ctx &c, int i, int j, int k, bool with_energy = false) {
  int st = adjoint_vr(c, i, j, k, c.s);
  if (st == PAMD_OK) st = adjoint_gemms(c, i, j, k);
  if (st == PAMD_OK) st = adjoint_combine(c, i, j, k, c.s, with_energy);
  return st;
}

// operand format of a precision
static int split_format(int prec) {
  return prec == PAMD_PREC_BF16X3 ? kSplitBf16x3
                                  : (prec == PAMD_PREC_FP32X2 ? kSplitF32x2 : kSplitNone);
}

// where the orbit epilogue writes Wbar: the GEMM operand copy in the engine's
// format (split forms), or over W (FP64)
static void wbar_out(const Ctx &c, int fmt, OrbitArgs &oa) {
  oa.Wb3 = fmt == kSplitBf16x3 ? (unsigned short *)c.gW : nullptr;
  oa.Wb8 = fmt == kSplitF32x2 ? (unsigned long long *)c.gW : nullptr;
}

// Zero the adjoint accumulators and the cotangent outputs of one call.
static int zero_vjp(const Ctx &c) {
  const int o = c.o, v = c.v;
  const size_t v2 = (size_t)v * v, vp2 = (size_t)c.vp * c.vp;
  PAMD_CHECK(launch_fill(c.Vpb, (size_t)o * vp2 * c.vp, 0.0, c.s));
  PAMD_CHECK(launch_fill(c.T2mb, (size_t)o * c.op * vp2, 0.0, c.s));
  PAMD_CHECK(launch_fill(c.part_mo, (size_t)kGmax * (o + c.vp), 0.0, c.s));
  PAMD_CHECK(launch_fill(c.t1_bar, (size_t)o * v, 0.0, c.s));
  PAMD_CHECK(launch_fill(c.t2_bar, (size_t)o * o * v2, 0.0, c.s));
  PAMD_CHECK(launch_fill(c.ovoo_bar, (size_t)o * v * o * o, 0.0, c.s));
  PAMD_CHECK(launch_fill(c.ovov_bar, (size_t)o * v * o * v, 0.0, c.s));
  PAMD_CHECK(launch_fill(c.fvo_bar, (size_t)v * o, 0.0, c.s));
  return PAMD_OK;
}

// inputs of a call's WalkPrep; the caller adds the outputs
static WalkPrep walk_prep(const Ctx &c, const WalkDims &d) {
  WalkPrep w;
  memset(&w, 0, sizeof(w));
  w.d = d;
  w.mo = c.mo;
  w.t1 = c.t1;
  w.t2 = c.t2;
  w.ovvv = c.ovvv;
  w.ovoo = c.ovoo;
  w.ovov = c.ovov;
  w.fvo = c.has_fvo ? c.fvo : nullptr;
  w.packed = c.packed;
  w.shard = c.shard;
  w.nshards = c.nshards;
  return w;
}

// Layout changes at entry, shared by every walk; returns the orbit count.
static int setup(Ctx &c, long long &norb) {
  const int o = c.o, v = c.v;
  const int fmt = split_format(c.prec);
  const int nt = (v + 7) / 8;
  norb = (long long)nt * (nt + 1) * (nt + 2) / 6;
  PAMD_CHECK(launch_prepare(c.ovvv, c.packed, c.t2, c.ovoo, o, v, c.op, c.vp, c.Vp, c.T2m, c.OOt, fmt, c.s));
  if (c.pad) {
    WalkPrep w = walk_prep(c, walk_dims(o, v));
    w.OVS = c.OVS;
    w.T2S = c.T2S;
    w.t1p = c.t1p;
    w.fvop = c.fvop;
    w.mop = c.mop;
    w.orb = c.orb;
    w.norb = norb;
    w.tri = c.tab;
    w.wb = walk_batches((num_triples(o) - c.shard + c.nshards - 1) / c.nshards, INT_MAX);
    w.zero[0] = c.tri;
    w.nzero[0] = (size_t)o * o * o;
    PAMD_CHECK(launch_walk_prep(w, c.s));
    if (c.wt_host) PAMD_CHECK(launch_walk_upload(c.wt_host, o, c.wt, c.s));
  } else {
    PAMD_CHECK(launch_prep_sym(c.ovov, o, v, 0, c.OVS, c.s));
    PAMD_CHECK(launch_prep_sym(c.t2, o, v, 1, c.T2S, c.s));
    PAMD_CHECK(launch_fill(c.tri, (size_t)o * o * o, 0.0, c.s));
    PAMD_CHECK(launch_orbit_table(norb, c.orb, c.s));
  }
  if (fmt == kSplitBf16x3)
    PAMD_CHECK(launch_split_t2(c.t2, o, v, c.vp, (unsigned short *)c.gT2, c.s));
  if (c.VpT)
    PAMD_CHECK(launch_vp_transposes((const unsigned short *)c.Vp, o, c.vp, (unsigned short *)c.VpT,
                                    (unsigned short *)c.VpU, c.s));
  if (fmt == kSplitF32x2)
    PAMD_CHECK(launch_split_f32x2(c.t2, (size_t)o * o * v * v, (unsigned long long *)c.gT2, c.s));
  // padded: two workgroups per CU, four without the adjoint (LDS)
  c.G = c.pad ? (int)std::min<long long>({norb, (long long)(c.vjp ? 2 : 4) * device_cus(), (long long)kGmax})
              : std::min(orbit_grid(v), kGmax);
  return PAMD_OK;
}

static OrbitArgs orbit_args(const Ctx &c, int i, int j, int k, long long norb) {
  OrbitArgs oa;
  memset(&oa, 0, sizeof(oa));
  oa.W = c.W;
  oa.tab = c.orb;
  oa.Vb = c.Vb;
  oa.t1 = c.t1;
  oa.ovs = c.OVS;
  oa.t2s = c.T2S;
  oa.fvo = c.fvo;
  oa.mo = c.mo;
  oa.o = c.o;
  oa.v = c.v;
  oa.i = i;
  oa.j = j;
  oa.k = k;
  oa.has_fvo = c.has_fvo;
  oa.norb = norb;
  oa.part_t = c.part_t;
  oa.part_mo = c.part_mo;
  return oa;
}

// Epilogue of the t-th triple (i, j, k) of the call's walk on stream st; W: its
// block.  nb > 1 (padded, energy only): also of the nb - 1 triples after it.
static int walk_epilogue(const Ctx &c, long long t, int i, int j, int k, double *W, int nb, long long norb,
                         hipStream_t st) {
  const double v3 = (double)c.v * c.v * c.v;
  const double ob = 8.0 * v3 * (c.vjp ? 3.0 : 1.0) * nb;  // W read (+ Wbar, Vbar written)
  OrbitArgs oa = orbit_args(c, i, j, k, norb);
  oa.W = W;
  if (c.vjp) wbar_out(c, split_format(c.prec), oa);
  oa.vjp = c.vjp;
  oa.ebar = c.ebar;
  if (c.pad) {
    oa.t1 = c.t1p;
    oa.fvo = c.fvop;
    oa.mo = c.mop;
    oa.v = c.vp;
    oa.ws = (long long)c.vp * c.vp;
    oa.tri = c.tab + t;
    oa.nb = nb;
    oa.wt = c.wt_host ? c.wt : nullptr;
    PAMD_CHECK(timed(st, kProfOrbit, 0.0, ob, [&] { return launch_walk_orbit(oa, c.G, st); }));
    return PAMD_OK;
  }
  oa.omega = (i == j || j == k) ? 1.0 : 2.0;
  // a diagonal occupied projector diag(m) weighs the whole triple by
  // (m_i + m_j + m_k) / 3 (the triple energy is symmetric in i, j, k)
  if (c.wt_host) oa.ebar = c.ebar * ((c.wt_host[i] + c.wt_host[j] + c.wt_host[k]) / 3.0);
  PAMD_CHECK(timed(st, kProfOrbit, 0.0, ob, [&] { return launch_orbit(oa, c.G, st); }));
  return PAMD_OK;
}

// Projected walk: for every unordered occupied pair (j, k), all o triples
// (l, j, k) in order of l.  Each W_ljk is built, and the orbit epilogue adds
// ulo[f, l] W and ulo[f, l] Z / D into accA[f], accB[f]; then
// pair_e[j, k] = sum_f <accA[f], accB[f]> = sum_{l,i} mat[l,i] <W_ljk, Z_ijk / D_ijk>.
// With c.vjp, a second pass over l rebuilds W_ljk and runs the projected
// adjoint epilogue (seeds from the finished accA, accB, cotangent
// g = ebar w_jk / 3 with w_jk = 2 off the diagonal) and the plain adjoint
// contractions of that triple; dE/dulo[f, l] gathers g (<W, accB[f]> +
// <accA[f], Z/D>) into ulo_bar.
static int run_projected(Ctx &c, const double *ulo, int nfrag, double *accA, double *accB,
                         double *pair_e, double *dot_part, double *part_u, double *ulo_bar) {
  long long norb = 0;
  int st = setup(c, norb);
  if (st != PAMD_OK) return st;
  const int o = c.o;
  const size_t v3 = (size_t)c.v * c.v * c.v;
  if (c.vjp) {
    st = zero_vjp(c);
    if (st != PAMD_OK) return st;
    PAMD_CHECK(launch_fill(ulo_bar, (size_t)nfrag * o, 0.0, c.s));
  }
  long long tcount = 0;
  const long long nbuild = (long long)o * o * (o + 1) / 2 * (c.vjp ? 2 : 1);
  const auto t_start = std::chrono::steady_clock::now();
  auto progress = [&]() -> int {
    if (g_progress_every > 0 && tcount % g_progress_every == 0) {
      PAMD_CHECK(hipStreamSynchronize(c.s));
      const double el = std::chrono::duration<double>(std::chrono::steady_clock::now() -
                                                       t_start).count();
      fprintf(stderr, "pyscfad_amd: projected (T)%s triples %lld/%lld done, %.1f s\n",
              c.vjp ? "+VJP" : "", tcount, nbuild, el);
      fflush(stderr);
    }
    return PAMD_OK;
  };
  const int fmt = split_format(c.prec);
  for (int j = 0; j < o; ++j)
    for (int k = j; k < o; ++k) {
      PAMD_CHECK(launch_fill(accA, (size_t)nfrag * v3, 0.0, c.s));
      PAMD_CHECK(launch_fill(accB, (size_t)nfrag * v3, 0.0, c.s));
      for (int l = 0; l < o; ++l) {
        g_prof_on = g_prof_every > 0 && (tcount % g_prof_every) == 0;
        ++tcount;
        st = build_w(c, l, j, k);
        if (st != PAMD_OK) return st;
        OrbitArgs oa = orbit_args(c, l, j, k, norb);
        oa.accA = accA;
        oa.accB = accB;
        oa.nfrag = nfrag;
        for (int f = 0; f < nfrag; ++f) oa.u[f] = ulo[(size_t)f * o + l];
        const double ob = 8.0 * (double)v3 * (1.0 + 4.0 * nfrag);  // W read, 2 nfrag RMW
        PAMD_CHECK(timed(c.s, kProfOrbit, 0.0, ob,
                         [&] { return launch_orbit(oa, c.G, c.s, kOrbitProjAcc); }));
        st = progress();
        if (st != PAMD_OK) return st;
      }
      PAMD_CHECK(launch_dot(accA, accB, (size_t)nfrag * v3, dot_part, kGmax, pair_e + j * o + k,
                            c.s));
      if (!c.vjp) continue;
      const double g = c.ebar * (j == k ? 1.0 : 2.0) / 3.0;
      for (int l = 0; l < o; ++l) {
        g_prof_on = g_prof_every > 0 && (tcount % g_prof_every) == 0;
        ++tcount;
        st = build_w(c, l, j, k);
        if (st != PAMD_OK) return st;
        OrbitArgs oa = orbit_args(c, l, j, k, norb);
        wbar_out(c, fmt, oa);
        oa.vjp = 1;
        oa.ebar = g;
        oa.accA = accA;
        oa.accB = accB;
        oa.nfrag = nfrag;
        oa.part_u = part_u;
        for (int f = 0; f < nfrag; ++f) oa.u[f] = ulo[(size_t)f * o + l];
        const double ob = 8.0 * (double)v3 * (3.0 + 2.0 * nfrag);  // W, accA, accB read; Wbar, Vbar
        PAMD_CHECK(timed(c.s, kProfOrbit, 0.0, ob,
                         [&] { return launch_orbit(oa, c.G, c.s, kOrbitProjVjp); }));
        PAMD_CHECK(launch_reduce_ulo(part_u, c.G, nfrag, g, ulo_bar + l, o, c.s));
        st = adjoint(c, l, j, k);
        if (st != PAMD_OK) return st;
        st = progress();
        if (st != PAMD_OK) return st;
      }
    }
  g_prof_on = false;
  if (!g_prof_recs.empty()) PAMD_CHECK(prof_collect());
  return PAMD_OK;
}

// Side stream and events of the pipelined adjoint walk, per host thread and
// device: created once (default priority, non-blocking) and kept for the life
// of the process.
struct PipeRes {
  hipStream_t e;
  hipEvent_t ev[10];  // start, end, W built [2], V-bar reduced [2], adjoint done [2], gathered [2]
  bool ok;
};

static PipeRes *pipe_resources() {
  constexpr int kMaxDev = 64;
  static thread_local PipeRes res[kMaxDev];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) return nullptr;
  PipeRes &r = res[dev];
  if (!r.ok) {
    if (hipStreamCreateWithFlags(&r.e, hipStreamNonBlocking) != hipSuccess) return nullptr;
    for (hipEvent_t &e : r.ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return nullptr;
    r.ok = true;
  }
  return &r;
}

// The adjoint walk with two triples in flight.  The contractions (W builds
// and adjoint GEMMs) run in order on the call's stream G; the memory-bound
// epilogue of each triple (orbit epilogue, triple energy, V-bar reductions,
// gather into the cotangents) runs on the side stream E while G builds the
// next triple's W:
//   G: WB(0) WB(1) ADJ(0) WB(2) ADJ(1) WB(3) ADJ(2) ...
//   E:   ORB(0) VR(0) | COMB(0) ORB(1) VR(1) | COMB(1) ...
// Triple t uses buffer set t % 2 (W, Wbar, V-bar scratch R, split-K
// partials).  Waits: ORB(t) after WB(t); ADJ(t) after VR(t) and after COMB(t-2)
// (which read the partials ADJ(t) overwrites); COMB(t) after ADJ(t).  The
// orders within G and E cover the rest: WB(t+2) follows ADJ(t), which followed
// ORB(t) (the last reader of W[t % 2]); ORB(t+2) follows COMB(t+1) and so
// ADJ(t) (the last reader of Wbar[t % 2]); VR(t+2) follows COMB(t) (the last
// reader of R[t % 2]).  The accumulators shared by all triples (Vpb and T2mb
// on G; the cotangents, triple energies and dE/de partials on E) are each
// written by one stream, in walk order, so the sums are the sequential walk's.
static int run_vjp_pipelined(Ctx &c, long long norb, PipeRes &pr) {
  const int o = c.o;
  std::vector<int> tr;  // triples of this call in walk order, i | j << 10 | k << 20
  {
    long long windex = -1;
    for (int i = 0; i < o; ++i)
      for (int j = i; j < o; ++j)
        for (int k = j; k < o; ++k) {
          if (i == j && j == k) continue;
          ++windex;
          if (c.nshards > 1 && windex % c.nshards != c.shard) continue;
          tr.push_back(i | (j << 10) | (k << 20));
        }
  }
  Ctx cx[2] = {c, c};
  cx[1].W = c.W2;
  cx[1].gW = c.gW2;
  cx[1].R = c.R2;
  cx[1].part_p = c.part_p2;
  cx[1].part_h = c.part_h2;
  for (int a = 0; a < cx[1].planes.count; ++a)
    if (cx[1].planes.base[a] == (const char *)c.gW) cx[1].planes.base[a] = (const char *)c.gW2;
  // Paired ovvv adjoints (env PYSCFAD_AMD_PAIR_OVVV=0 turns them off): consecutive triples
  // (i, j, k), (i, j, k') add into the same Vpb[i] and Vpb[j], so the second
  // one's launches for them also take the first one's terms, from the other
  // Wbar buffer.  That buffer is next written by the orbit epilogue two
  // triples on, which the side stream runs after the gather of the second
  // triple, which waits for its contractions.  Only where Wbar has its own
  // buffer (split forms; FP64 writes Wbar over W, which the W build of the
  // triple after next overwrites before the second triple's contractions).
  // The hole-term t2 adjoints into T2mb[i], T2mb[j] pair the same way.
  // Measured (full walks, split-BF16x3, ovvv adjoints paired): o16/v160 E+VJP
  // 0.541 -> 0.532 s, o24/v240 5.39 -> 5.30 s, o40/v400 127.8 -> 125.2 s.
  // Only ovvv_bar and t2_bar change (the same terms grouped in other FP32
  // sums, ~1e-8 relative).
  static const bool pair_env = [] {
    const char *e = getenv("PYSCFAD_AMD_PAIR_OVVV");
    return !(e && e[0] == '0');
  }();
  const bool pair_on = pair_env && c.gW != c.W && c.gW2 != nullptr;
  if (pair_on && c.prec == PAMD_PREC_BF16X3) {
    const long long v3 = (long long)c.vp * c.vp * c.vp;
    for (int p = 0; p < 2; ++p) {
      PlanarMap &pm = cx[p].planes;
      if (pm.count >= 8) return PAMD_ERR_ARG;
      pm.base[pm.count] = (const char *)cx[1 - p].gW;
      pm.n[pm.count] = v3;
      ++pm.count;
    }
  }
  const hipStream_t G = c.s, E = pr.e;
  hipEvent_t *wb = pr.ev + 2, *vr = pr.ev + 4, *adj = pr.ev + 6, *cmb = pr.ev + 8;
  PAMD_CHECK(hipEventRecord(pr.ev[0], G));
  PAMD_CHECK(hipStreamWaitEvent(E, pr.ev[0], 0));
  const long long n = (long long)tr.size();
  const long long ntrip = (long long)o * (o + 1) * (o + 2) / 6 - o;
  const auto t_start = std::chrono::steady_clock::now();
  auto walk = [&]() -> int {
    if (n == 0) return PAMD_OK;
    auto ijk = [&](long long t, int &i, int &j, int &k) {
      i = tr[t] & 1023;
      j = (tr[t] >> 10) & 1023;
      k = tr[t] >> 20;
    };
    int i, j, k, st;
    bool pend = false;  // the previous triple left its Vpb[i], Vpb[j] adjoints to this one
    int kpend = 0;
    g_prof_on = g_prof_every > 0;
    ijk(0, i, j, k);
    st = build_w(cx[0], i, j, k);
    if (st != PAMD_OK) return st;
    PAMD_CHECK(hipEventRecord(wb[0], G));
    for (long long t = 0; t < n; ++t) {
      const int p = (int)(t & 1);
      const Ctx &C = cx[p];
      g_prof_on = g_prof_every > 0 && (t % g_prof_every) == 0;
      ijk(t, i, j, k);
      // E: epilogue and V-bar reductions of t
      PAMD_CHECK(hipStreamWaitEvent(E, wb[p], 0));
      st = walk_epilogue(C, t, i, j, k, C.W, 1, norb, E);
      if (st != PAMD_OK) return st;
      st = adjoint_vr(C, i, j, k, E);
      if (st != PAMD_OK) return st;
      PAMD_CHECK(hipEventRecord(vr[p], E));
      // G: W build of t + 1
      if (t + 1 < n) {
        int i1, j1, k1;
        ijk(t + 1, i1, j1, k1);
        st = build_w(cx[1 - p], i1, j1, k1);
        if (st != PAMD_OK) return st;
        PAMD_CHECK(hipEventRecord(wb[1 - p], G));
      }
      // G: adjoint contractions of t
      PAMD_CHECK(hipStreamWaitEvent(G, vr[p], 0));
      if (t >= 2) PAMD_CHECK(hipStreamWaitEvent(G, cmb[p], 0));
      if (pend) {
        st = adjoint_gemms(C, i, j, k, 2, &cx[1 - p], kpend);
        pend = false;
      } else if (pair_on && t + 1 < n && (tr[t + 1] & 0xfffff) == (tr[t] & 0xfffff)) {
        st = adjoint_gemms(C, i, j, k, 1);
        pend = true;
        kpend = k;
      } else {
        st = adjoint_gemms(C, i, j, k);
      }
      if (st != PAMD_OK) return st;
      PAMD_CHECK(hipEventRecord(adj[p], G));
      // E: gather of t
      PAMD_CHECK(hipStreamWaitEvent(E, adj[p], 0));
      st = adjoint_combine(C, i, j, k, E, true);  // with the triple's energy
      if (st != PAMD_OK) return st;
      PAMD_CHECK(hipEventRecord(cmb[p], E));
      if (g_progress_every > 0 && (t + 1) % g_progress_every == 0) {
        PAMD_CHECK(hipStreamSynchronize(E));
        PAMD_CHECK(hipStreamSynchronize(G));
        const double el = std::chrono::duration<double>(std::chrono::steady_clock::now() -
                                                         t_start).count();
        fprintf(stderr, "pyscfad_amd: (T)+VJP triples %lld/%lld done, %.1f s\n", t + 1,
                c.nshards > 1 ? n : ntrip, el);
        fflush(stderr);
      }
    }
    return PAMD_OK;
  };
  int st = walk();
  // the call's stream waits for the side stream, also after an error
  hipError_t e = hipEventRecord(pr.ev[1], E);
  if (e == hipSuccess) e = hipStreamWaitEvent(G, pr.ev[1], 0);
  if (e != hipSuccess && st == PAMD_OK) {
    fprintf(stderr, "pyscfad_amd: joining the side stream failed: %s\n", hipGetErrorString(e));
    st = PAMD_ERR_HIP;
  }
  g_prof_on = false;
  if (st == PAMD_OK && !g_prof_recs.empty()) PAMD_CHECK(prof_collect());
  return st;
}

static int run(Ctx &c) {
  const int o = c.o;
  long long norb = 0;
  {
    const int st0 = setup(c, norb);
    if (st0 != PAMD_OK) return st0;
  }
  if (c.vjp) {
    const int st0 = zero_vjp(c);
    if (st0 != PAMD_OK) return st0;
  }
  static const bool pipe_on = [] {
    const char *e = getenv("PYSCFAD_AMD_PIPELINE");
    return !(e && e[0] == '0');
  }();
  if (c.vjp && c.pipe && pipe_on && !g_record) {
    PipeRes *pr = pipe_resources();
    if (pr) return run_vjp_pipelined(c, norb, *pr);
  }
  long long tcount = 0, windex = -1;
  const long long ntrip = (long long)o * (o + 1) * (o + 2) / 6 - o;
  const auto t_start = std::chrono::steady_clock::now();
  if (!c.vjp && c.nshards == 1 && c.wbatch > 1) {
    // energy only, small nvir: the W blocks of up to wbatch consecutive k of one
    // pair (i, j) are built by one launch per pass; each triple's epilogue then
    // reads its own block.  Same triples, same per-triple arithmetic and the
    // same fixed-order sum over tri as the walk below.
    const size_t v3 = (size_t)c.vp * c.vp * c.vp;
    for (int i = 0; i < o; ++i)
      for (int j = i; j < o; ++j)
        for (int kb = (i == j ? j + 1 : j); kb < o; kb += c.wbatch) {
          const int nb = std::min(c.wbatch, o - kb);
          g_prof_on = g_prof_every > 0 && (tcount % g_prof_every) < nb;
          int st = build_w(c, i, j, kb, nb);
          if (st != PAMD_OK) return st;
          if (c.pad) {
            st = walk_epilogue(c, tcount, i, j, kb, c.W, nb, norb, c.s);
            if (st != PAMD_OK) return st;
            PAMD_CHECK(launch_walk_energies(c.tab + tcount, nb, o, c.part_t, c.G, c.tri, c.s));
          }
          for (int b = 0; b < nb; ++b) {
            const int k = kb + b;
            if (!c.pad) {
              st = walk_epilogue(c, tcount, i, j, k, c.W + b * v3, 1, norb, c.s);
              if (st != PAMD_OK) return st;
              PAMD_CHECK(launch_triple_energy(c.part_t, c.G, c.tri + ((size_t)i * o + j) * o + k, c.s));
            }
            ++tcount;
            if (g_progress_every > 0 && tcount % g_progress_every == 0) {
              PAMD_CHECK(hipStreamSynchronize(c.s));
              const double el = std::chrono::duration<double>(std::chrono::steady_clock::now() -
                                                               t_start).count();
              fprintf(stderr, "pyscfad_amd: (T) triples %lld/%lld done, %.1f s\n", tcount, ntrip,
                      el);
              fflush(stderr);
            }
          }
        }
    g_prof_on = false;
    if (!g_prof_recs.empty()) PAMD_CHECK(prof_collect());
    return PAMD_OK;
  }
  for (int i = 0; i < o; ++i)
    for (int j = i; j < o; ++j)
      for (int k = j; k < o; ++k) {
        if (i == j && j == k) continue;
        // round-robin shard of the walk: triple number windex goes to shard windex % nshards
        ++windex;
        if (c.nshards > 1 && windex % c.nshards != c.shard) continue;
        g_prof_on = g_prof_every > 0 && (tcount % g_prof_every) == 0;
        ++tcount;
        int st = build_w(c, i, j, k);
        if (st != PAMD_OK) return st;
        st = walk_epilogue(c, tcount - 1, i, j, k, c.W, 1, norb, c.s);
        if (st != PAMD_OK) return st;
        if (!c.vjp)
          PAMD_CHECK(launch_triple_energy(c.part_t, c.G, c.tri + ((size_t)i * o + j) * o + k, c.s));
        if (c.vjp) {
          st = adjoint(c, i, j, k, true);  // the gather also sums the triple's energy
          if (st != PAMD_OK) return st;
        }
        if (g_progress_every > 0 && tcount % g_progress_every == 0) {
          PAMD_CHECK(hipStreamSynchronize(c.s));
          const double el = std::chrono::duration<double>(std::chrono::steady_clock::now() -
                                                           t_start).count();
          fprintf(stderr, "pyscfad_amd: (T)%s triples %lld/%lld done, %.1f s\n",
                  c.vjp ? "+VJP" : "", tcount, ntrip, el);
          fflush(stderr);
        }
      }
  g_prof_on = false;
  if (!g_prof_recs.empty()) PAMD_CHECK(prof_collect());
  return PAMD_OK;
}

static int check_common(const pamd_ccsdt_config *cfg, const double *mo, const double *t1,
                        const double *t2, const double *ovvv, const double *ovoo,
                        const double *ovov, const double *fvo) {
  if (!cfg || cfg->nocc < 1 || cfg->nvir < 1) return PAMD_ERR_ARG;
  if (!mo || !t1 || !t2 || !ovvv || !ovoo || !ovov) return PAMD_ERR_ARG;
  if (cfg->has_fvo && !fvo) return PAMD_ERR_ARG;
  if (cfg->precision != PAMD_PREC_FP64 && cfg->precision != PAMD_PREC_BF16X3 &&
      cfg->precision != PAMD_PREC_FP32X2)
    return PAMD_ERR_UNSUPPORTED;
  if (cfg->nocc > 1024) return PAMD_ERR_ARG;
  // the engines address an operand within one occupied slab with 32-bit
  // element offsets, and the largest slab is v^3 (W, Wbar, Vp[x])
  if ((long long)cfg->nvir * cfg->nvir * cfg->nvir >= (1LL << 31)) return PAMD_ERR_UNSUPPORTED;
  return PAMD_OK;
}

static void bind_workspace(Ctx &c, const Layout &L, void *ws) {
  char *b = (char *)ws;
  c.Vp = (double *)(b + L.off_Vp);
  c.T2m = (double *)(b + L.off_T2m);
  c.OOt = (double *)(b + L.off_OOt);
  c.OVS = (double *)(b + L.off_OVS);
  c.T2S = (double *)(b + L.off_T2S);
  c.orb = (unsigned short *)(b + L.off_orb);
  c.W = (double *)(b + L.off_W);
  c.wbatch = L.wbatch;
  c.pad = L.pad;
  c.op = L.op;
  c.vp = L.vp;
  if (L.pad) {
    c.t1p = (double *)(b + L.off_t1);
    c.fvop = (double *)(b + L.off_fvo);
    c.mop = (double *)(b + L.off_mo);
    c.tab = (int *)(b + L.off_tab);
  }
  c.tri = (double *)(b + L.off_tri);
  c.part_t = (double *)(b + L.off_part_t);
  c.wt = (double *)(b + L.off_wt);
  const bool packed_ops = c.prec == PAMD_PREC_BF16X3 || c.prec == PAMD_PREC_FP32X2;
  c.gT2 = packed_ops ? (const double *)(b + L.off_T2g) : c.t2;
  c.gW = (packed_ops && c.vjp) ? (double *)(b + L.off_W8) : c.W;
  // (the tiny products are not run by the direct engine, which the copies are for: b3_tiny)
  const bool vpt = L.vpt && L.vp > 16;
  c.VpT = vpt ? (double *)(b + L.off_VpT) : nullptr;
  c.VpU = vpt ? (double *)(b + L.off_VpU) : nullptr;
  {
    const long long o = c.o, op = c.op, v = c.vp, v3 = v * v * v;
    PlanarMap &pm = c.planes;
    pm.count = 0;
    auto add = [&](const void *p, long long n) {
      pm.base[pm.count] = (const char *)p;
      pm.n[pm.count] = n;
      ++pm.count;
    };
    add(c.Vp, o * v3);
    add(c.T2m, o * op * v * v);
    add(c.OOt, o * o * op * v);
    add(c.gT2, o * o * v * v);
    if (c.vjp) add(c.gW, v3);
    if (c.VpT) {
      add(c.VpT, o * v3);
      add(c.VpU, o * v3);
    }
  }
  if (c.vjp) {
    c.Vb = (double *)(b + L.off_Vb);
    c.Vpb = (double *)(b + L.off_Vpb);
    c.T2mb = (double *)(b + L.off_T2mb);
    c.part_mo = (double *)(b + L.off_part_mo);
    c.R = (double *)(b + L.off_R);
    c.part_p = (double *)(b + L.off_part_p);
    c.part_h = (double *)(b + L.off_part_h);
    c.pipe = L.pipe;
    if (L.pipe) {
      c.W2 = (double *)(b + L.off_W2);
      c.gW2 = packed_ops ? (double *)(b + L.off_W8b) : c.W2;
      c.R2 = (double *)(b + L.off_R2);
      c.part_p2 = (double *)(b + L.off_part_p2);
      c.part_h2 = (double *)(b + L.off_part_h2);
    }
  } else {
    c.Vb = c.Vpb = c.T2mb = c.part_mo = c.R = c.part_p = c.part_h = nullptr;
  }
  c.S_p = L.S_p;
  c.S_h = L.S_h;
  // FP32 parts (half the traffic of the reduction) wherever a part is one FP32
  // sum, and two of them leave room for the FP64 result (part_sum_at)
  auto whole = [&](int M, int N) {
    return c.prec == PAMD_PREC_BF16X3 &&
           ((gemm_b3p_enabled() && M % 8 == 0 && N % 8 == 0) || gemm_b3_sums(M, N) == kSumsWhole);
  };
  c.f32_p = L.S_p >= 2 && whole(c.v, c.v);
  c.f32_h = L.S_h >= 2 && whole(c.v, c.o);
}

// ---------------------------------------------------------------------------
// Batched FP64 walk (walk64.h): nb triples per launch.
// ---------------------------------------------------------------------------
constexpr size_t kNoAllocScratchBytes = (size_t)128 << 20;

struct WalkLayout {
  WalkDims d;
  int nb, S, G;
  size_t r_stride, total;
  size_t off_VT, off_TB, off_TBt, off_OVS, off_T2S, off_t1, off_fvo, off_mo, off_orb, off_tri_e, off_tab, off_wt,
      off_W, off_part_t, off_Vb, off_VTb, off_R, off_part, off_vec, off_mo_rows, off_mo2;
};

static WalkLayout walk_layout(int o, int v, int vjp, int nb) {
  WalkLayout L;
  memset(&L, 0, sizeof(L));
  L.d = walk_dims(o, v);
  L.nb = nb;
  const size_t vp = L.d.vp, up = L.d.up, v2 = vp * vp, n = (size_t)o + vp, oo = (size_t)o * o;
  const size_t nt = vp / 8, norb = nt * (nt + 1) * (nt + 2) / 6;
  size_t off = 0;
  auto take = [&](size_t count) {
    const size_t at = off;
    off = align256(off + count * sizeof(double));
    return at;
  };
  // parts of TB's adjoint: enough tiles for 16 rounds of the 1024 SIMDs, each
  // part at least 8 outer steps
  const long long tiles = 6LL * nb * ((vp + 15) / 16) * ((up + 15) / 16);
  L.S = (int)std::max(1LL, std::min({(16 * 1024 + tiles - 1) / tiles, (long long)vp / 8, 8LL}));
  // orbit epilogue: about four rounds of workgroups per launch
  L.G = (int)std::max<size_t>(1, std::min<size_t>({(2048 + (size_t)nb - 1) / nb, norb, (size_t)kGmax}));
  L.off_VT = take((size_t)o * vp * L.d.sp);
  if (vjp) L.off_TB = take(oo * vp * up);
  L.off_TBt = take(oo * vp * up);
  L.off_OVS = take(oo * v2);
  L.off_T2S = take(oo * v2);
  L.off_t1 = take((size_t)o * vp);
  L.off_fvo = take((size_t)o * vp);
  L.off_mo = take(n);
  L.off_orb = take(norb);
  L.off_tri_e = take(oo * o);
  // every shard's table fits: at most one run and one batch's round more
  L.off_tab = take((size_t)(num_triples(o) + kWalkMaxBatch + 2 * kWalkRun) / 2 + 1);
  L.off_wt = take(o);
  L.off_W = take(vp * L.d.ws * nb);
  L.off_part_t = take((size_t)nb * L.G);
  if (vjp) {
    L.off_Vb = take(v2 * vp * nb);
    L.off_VTb = take((size_t)o * vp * L.d.sp);
    L.r_stride = vr_col_blocks((int)vp) > 1 ? vr_scratch_doubles((int)vp) : 10 * v2 + 2 * vp;
    L.off_R = take(L.r_stride * nb);
    L.off_part = take((size_t)nb * 6 * L.S * vp * up);
    L.off_vec = take((size_t)nb * 6 * vp);
    L.off_mo_rows = take((size_t)nb * L.G * n);
    L.off_mo2 = take((size_t)kWalkMoParts * n);
  }
  L.total = off;
  return L;
}

// The batch of a call: as many triples as fit the library's own scratch
// together with the rest when these are all, or 32 (a call without a workspace of
// its own then splits the walk like one with it),
// else as many as 8 GB of blocks hold; fewer when `limit` bytes are there, or
// when an adjoint would hold nearly every triple.
// False when the walk does not apply: slabs beyond 32-bit offsets, not even one
// run in `limit`, or a workspace noticeably larger than the one-triple walk's
// where that is large itself.
static bool walk_pick(int o, int v, int vjp, size_t limit, size_t one_triple_total, WalkLayout &L) {
  if (!walk_dims_ok(walk_dims(o, v))) return false;
  // batch sizes: whole runs, one at least (one occupied orbital has no triples; its
  // empty batch writes the zero cotangents)
  const long long runs = std::max((num_triples(o) + kWalkRun - 1) / kWalkRun, 1LL);
  const int n = (int)std::min<long long>(runs * kWalkRun, kWalkMaxBatch);
  auto largest = [&](size_t bytes) {
    int b = n;
    while (b > 0 && walk_layout(o, v, vjp, b).total > bytes) b -= kWalkRun;
    return b;
  };
  int b = largest(kNoAllocScratchBytes);
  if (b < std::min(n, 32))
    b = std::max(kWalkRun, largest(walk_layout(o, v, vjp, kWalkRun).total + ((size_t)8 << 30)));
  if (vjp) {
    // an adjoint keeps no more than three quarters of what W and Wbar of all
    // triples would take (where that is more than 8 MB): a bound on memory, which a
    // small problem in one batch would pass (o8/v40: 79 instead of 128 MB, and 1.37
    // instead of 1.27 ms)
    const size_t all = (size_t)num_triples(o) * 2 * sizeof(double) * v * v * v;
    const size_t most = std::max<size_t>(all / 4 * 3, (size_t)8 << 20);
    if (walk_layout(o, v, vjp, b).total > most) b = std::max(kWalkRun, largest(most));
  }
  if (walk_layout(o, v, vjp, b).total > limit) b = largest(limit);
  if (b < kWalkRun) return false;
  // batches of equal size, where these take no more than `limit` (fewer triples per
  // batch may take more parts of TB's adjoint)
  L = walk_layout(o, v, vjp, walk_batches(num_triples(o), b).cap);
  if (L.total > limit) L = walk_layout(o, v, vjp, b);
  return L.total <= ((size_t)100 << 30) || L.total <= one_triple_total + one_triple_total / 20;
}

// Inputs, tables and zeroed sums of a call: the triples of wb, or with pairs those
// of the projected walk, in tab; zero[0 .. nzero) = 0.  Returns the orbit count.
static int walk_setup(Ctx &c, const WalkLayout &L, char *b, const WalkBatches *wb, int *tab, double *zero,
                      size_t nzero, long long &norb) {
  auto at = [&](size_t off) { return (double *)(b + off); };
  const WalkDims &d = L.d;
  c.tri = at(L.off_tri_e);
  c.wt = at(L.off_wt);
  const long long nt = d.vp / 8;
  norb = nt * (nt + 1) * (nt + 2) / 6;
  WalkPrep w = walk_prep(c, d);
  w.VT = at(L.off_VT);
  w.TB = c.vjp ? at(L.off_TB) : nullptr;
  w.TBt = at(L.off_TBt);
  w.OVS = at(L.off_OVS);
  w.T2S = at(L.off_T2S);
  w.t1p = at(L.off_t1);
  w.fvop = at(L.off_fvo);
  w.mop = at(L.off_mo);
  w.orb = (unsigned short *)at(L.off_orb);
  w.norb = norb;
  w.tri = tab;
  w.pairs = wb ? 0 : 1;
  if (wb) w.wb = *wb;
  w.zero[0] = zero;
  w.nzero[0] = nzero;
  if (c.vjp) {
    w.zero[1] = at(L.off_mo_rows);
    w.nzero[1] = (size_t)L.nb * L.G * (d.o + d.vp);
  }
  PAMD_CHECK(launch_walk_prep(w, c.s));
  return PAMD_OK;
}

static OrbitArgs walk_orbit_args(const Ctx &c, const WalkLayout &L, char *b, const int *tri, int nb,
                                 long long norb) {
  auto at = [&](size_t off) { return (double *)(b + off); };
  OrbitArgs oa;
  memset(&oa, 0, sizeof(oa));
  oa.W = at(L.off_W);
  oa.tab = (const unsigned short *)at(L.off_orb);
  oa.Vb = c.vjp ? at(L.off_Vb) : nullptr;
  oa.t1 = at(L.off_t1);
  oa.ovs = at(L.off_OVS);
  oa.t2s = at(L.off_T2S);
  oa.fvo = at(L.off_fvo);
  oa.mo = at(L.off_mo);
  oa.o = c.o;
  oa.v = L.d.vp;
  oa.has_fvo = c.has_fvo;
  oa.vjp = c.vjp;
  oa.norb = norb;
  oa.ebar = c.ebar;
  oa.part_t = at(L.off_part_t);
  oa.part_mo = c.vjp ? at(L.off_mo_rows) : nullptr;
  oa.tri = tri;
  oa.nb = nb;
  oa.ws = L.d.ws;
  return oa;
}

// algorithmic flops of one contraction family (W build or an adjoint) of a triple
static double walk_flops(const Ctx &c) { return 12.0 * c.v * (double)c.v * c.v * (c.v + c.o); }

static int walk_build(const Ctx &c, const WalkLayout &L, char *b, const int *tri, int nb) {
  auto at = [&](size_t off) { return (double *)(b + off); };
  PAMD_CHECK(timed(c.s, kProfWBuild, walk_flops(c) * nb, 0.0, [&] {
    return launch_walk_w(L.d, at(L.off_VT), at(L.off_TBt), at(L.off_W), tri, nb, c.s);
  }));
  return PAMD_OK;
}

// adjoint of a batch whose Wbar and Vbar blocks are written; tri_e: also the
// triple energies
static int walk_adjoint(const Ctx &c, const WalkLayout &L, char *b, const int *tri, int nb, bool first,
                        double *tri_e) {
  auto at = [&](size_t off) { return (double *)(b + off); };
  const WalkDims &d = L.d;
  const hipStream_t s = c.s;
  const double v3 = (double)c.v * c.v * c.v, fl = walk_flops(c) * nb;
  if (nb > 0) {
    VRArgs vr;
    memset(&vr, 0, sizeof(vr));
    vr.Vb = at(L.off_Vb);
    vr.t1 = at(L.off_t1);
    vr.fvo = at(L.off_fvo);
    vr.ovs = at(L.off_OVS);
    vr.t2s = at(L.off_T2S);
    vr.o = d.o;
    vr.v = d.vp;
    vr.has_fvo = c.has_fvo;
    vr.R = at(L.off_R);
    vr.parts = 1;
    vr.tri = tri;
    vr.nb = nb;
    vr.r_stride = L.r_stride;
    PAMD_CHECK(timed(s, kProfVR, 0.0, 16.0 * v3 * nb, [&] { return launch_walk_vr(vr, s); }));
  }
  PAMD_CHECK(timed(s, kProfAdjOvvv, fl, 0.0, [&] {
    return launch_walk_vtb(d, at(L.off_W), at(L.off_TB), at(L.off_VTb), tri, nb, first, s);
  }));
  if (nb > 0)
    PAMD_CHECK(timed(s, kProfAdjT2P, fl, 0.0, [&] {
      return launch_walk_tbb(d, at(L.off_W), at(L.off_VT), at(L.off_part), tri, nb, L.S, s);
    }));
  WalkGather g;
  g.d = d;
  g.tri = tri;
  g.nb = nb;
  g.S = L.S;
  g.G = L.G;
  g.has_fvo = c.has_fvo;
  g.first = first;
  g.part = at(L.off_part);
  g.R = at(L.off_R);
  g.r_stride = L.r_stride;
  g.part_t = at(L.off_part_t);
  g.vec = at(L.off_vec);
  g.t1_bar = c.t1_bar;
  g.t2_bar = c.t2_bar;
  g.ovoo_bar = c.ovoo_bar;
  g.ovov_bar = c.ovov_bar;
  g.fvo_bar = c.fvo_bar;
  g.tri_e = tri_e;
  const double cb = 8.0 * 6.0 * L.S * (double)d.vp * d.up * nb;
  PAMD_CHECK(timed(s, kProfCombine, 0.0, cb, [&] { return launch_walk_gather(g, s); }));
  return PAMD_OK;
}

static int walk_finish(const Ctx &c, const WalkLayout &L, char *b, double *ovvv_bar, double *mo_bar) {
  auto at = [&](size_t off) { return (double *)(b + off); };
  PAMD_CHECK(launch_walk_finish(L.d, at(L.off_VTb), c.packed, ovvv_bar, c.t2_bar, at(L.off_mo_rows),
                                L.nb * L.G, at(L.off_mo2), mo_bar, c.s));
  return PAMD_OK;
}

// progress lines (pamd_profile_progress) and launch sampling of a batched walk
struct WalkMeter {
  const char *what;
  long long n, reported;
  std::chrono::steady_clock::time_point start;
  explicit WalkMeter(const char *w, long long total)
      : what(w), n(total), reported(0), start(std::chrono::steady_clock::now()) {}
  void sample(long long t0, int nb) const {
    g_prof_on = g_prof_every > 0 && (t0 + g_prof_every - 1) / g_prof_every * g_prof_every < t0 + nb;
  }
  hipError_t report(long long done, hipStream_t s) {
    if (g_progress_every <= 0 || (done - reported < g_progress_every && done != n)) return hipSuccess;
    reported = done;
    const hipError_t e = hipStreamSynchronize(s);
    if (e != hipSuccess) return e;
    fprintf(stderr, "pyscfad_amd: %s triples %lld/%lld done, %.1f s\n", what, done, n,
            std::chrono::duration<double>(std::chrono::steady_clock::now() - start).count());
    fflush(stderr);
    return hipSuccess;
  }
};

// One call's walk on its stream c.s: c.tri gets the triple energies, and with
// c.vjp every cotangent is complete.
static int run_walk(Ctx &c, const WalkLayout &L, void *ws, double *ovvv_bar, double *mo_bar) {
  char *b = (char *)ws;
  auto at = [&](size_t off) { return (double *)(b + off); };
  const int o = c.o;
  const hipStream_t s = c.s;
  long long norb = 0;
  int *tab = (int *)at(L.off_tab);
  const long long n = (num_triples(o) - c.shard + c.nshards - 1) / c.nshards;
  const WalkBatches wb = walk_batches(n, L.nb);
  int st = walk_setup(c, L, b, &wb, tab, at(L.off_tri_e), (size_t)o * o * o, norb);
  if (st != PAMD_OK) return st;
  if (c.wt_host) PAMD_CHECK(launch_walk_upload(c.wt_host, o, c.wt, s));
  const double v3 = (double)c.v * c.v * c.v;
  WalkMeter meter(c.vjp ? "(T)+VJP" : "(T)", n);
  long long t0 = 0;
  // without triples one empty batch writes the (zero) cotangents
  for (int bt = 0; bt < wb.count; ++bt) {
    const int nb = wb.size(bt);
    const int *tri = tab + (size_t)bt * wb.cap;
    meter.sample(t0, nb);
    if (nb > 0) {
      st = walk_build(c, L, b, tri, nb);
      if (st != PAMD_OK) return st;
      OrbitArgs oa = walk_orbit_args(c, L, b, tri, nb, norb);
      oa.wt = c.wt_host ? c.wt : nullptr;
      const double ob = 8.0 * v3 * (c.vjp ? 3.0 : 1.0) * nb;
      PAMD_CHECK(timed(s, kProfOrbit, 0.0, ob, [&] { return launch_walk_orbit(oa, L.G, s); }));
    }
    if (c.vjp) {
      st = walk_adjoint(c, L, b, tri, nb, bt == 0, c.tri);
      if (st != PAMD_OK) return st;
    } else {
      PAMD_CHECK(launch_walk_energies(tri, nb, o, at(L.off_part_t), L.G, c.tri, s));
    }
    t0 += nb;
    PAMD_CHECK(meter.report(t0, s));
  }
  g_prof_on = false;
  if (!g_prof_recs.empty()) PAMD_CHECK(prof_collect());
  return c.vjp ? walk_finish(c, L, b, ovvv_bar, mo_bar) : PAMD_OK;
}

// (o10/v64, two fragment orbitals, E + VJP: 335 -> 17.6 ms against the one-triple walk.)
// Batched projected walk: np pairs (j, k) at a time, the o triples (l, j, k) of
// each in one batch, whose W blocks stay for the adjoint (the one-triple walk
// builds every W twice).
struct ProjWalkLayout {
  WalkLayout L;
  int np, Ga;  // pairs per batch, workgroups per pair of launch_walk_acc
  size_t off_tab, off_a, off_pair, off_u, off_ulo, total;
};

static ProjWalkLayout proj_walk_layout(int o, int v, int nfrag, int vjp, int np) {
  ProjWalkLayout P;
  P.L = walk_layout(o, v, vjp, np * o);
  P.np = np;
  const size_t nt = P.L.d.vp / 8, norb = nt * (nt + 1) * (nt + 2) / 6, pairs = (size_t)o * (o + 1) / 2;
  // (part_t holds G sums per triple: at least Ga per pair)
  P.Ga = (int)std::min<size_t>({(2048 + (size_t)np - 1) / np, norb, (size_t)P.L.G * o});
  size_t off = P.L.total;
  auto take = [&](size_t count) {
    const size_t at = off;
    off = align256(off + count * sizeof(double));
    return at;
  };
  P.off_tab = take((pairs * o + 1) / 2);
  P.off_a = take(np * nfrag * walk_acc_doubles(P.L.d));
  P.off_pair = take((size_t)o * o);
  P.off_u = take(vjp ? (size_t)np * o * P.L.G * kMaxFrag : 0);
  P.off_ulo = take((size_t)nfrag * o);
  P.total = off;
  return P;
}

// Pairs per batch: all, or as many as a batch of kWalkMaxBatch triples, 8 GB more
// than one pair needs, and `limit` hold.  False as in walk_pick, or when one pair
// has more triples than a batch.
static bool proj_walk_pick(int o, int v, int nfrag, int vjp, size_t limit, size_t one_triple_total,
                           ProjWalkLayout &P) {
  if (!walk_dims_ok(walk_dims(o, v)) || o > kWalkMaxBatch) return false;
  const size_t cap = std::min(limit, proj_walk_layout(o, v, nfrag, vjp, 1).total + ((size_t)8 << 30));
  int np = std::min(o * (o + 1) / 2, kWalkMaxBatch / o);
  while (np > 0 && proj_walk_layout(o, v, nfrag, vjp, np).total > cap) --np;
  if (np < 1) return false;
  const int pairs = o * (o + 1) / 2, batches = (pairs + np - 1) / np;
  P = proj_walk_layout(o, v, nfrag, vjp, (pairs + batches - 1) / batches);
  if (P.total > cap) P = proj_walk_layout(o, v, nfrag, vjp, np);
  return P.total <= ((size_t)100 << 30) || P.total <= one_triple_total + one_triple_total / 20;
}

static int run_projected_walk(Ctx &c, const ProjWalkLayout &P, void *ws, const double *ulo, int nfrag,
                              double *e_out, double *ovvv_bar, double *mo_bar, double *ulo_bar) {
  const WalkLayout &L = P.L;
  char *b = (char *)ws;
  auto at = [&](size_t off) { return (double *)(b + off); };
  const int o = c.o;
  const hipStream_t s = c.s;
  long long norb = 0;
  int *tab = (int *)at(P.off_tab);
  int st = walk_setup(c, L, b, nullptr, tab, at(P.off_pair), (size_t)o * o, norb);
  if (st != PAMD_OK) return st;
  PAMD_CHECK(launch_walk_upload(ulo, (size_t)nfrag * o, at(P.off_ulo), s));
  const double v3 = (double)c.v * c.v * c.v;
  const int pairs = o * (o + 1) / 2;
  WalkMeter meter(c.vjp ? "projected (T)+VJP" : "projected (T)", (long long)pairs * o);
  for (int p0 = 0; p0 < pairs; p0 += P.np) {
    const int np = std::min(P.np, pairs - p0), nb = np * o;
    const int *tri = tab + (size_t)p0 * o;
    meter.sample((long long)p0 * o, nb);
    st = walk_build(c, L, b, tri, nb);
    if (st != PAMD_OK) return st;
    OrbitArgs oa = walk_orbit_args(c, L, b, tri, nb, norb);
    oa.accA = at(P.off_a);
    oa.nfrag = nfrag;
    oa.udev = at(P.off_ulo);
    PAMD_CHECK(timed(s, kProfOrbit, 0.0, 8.0 * v3 * nb, [&] { return launch_walk_acc(oa, P.Ga, np, s); }));
    PAMD_CHECK(launch_walk_pair_energies(at(L.off_part_t), P.Ga, tri, np, o, at(P.off_pair), s));
    if (c.vjp) {
      oa.part_u = at(P.off_u);
      PAMD_CHECK(timed(s, kProfOrbit, 0.0, 8.0 * v3 * (3.0 + 2.0 * nfrag) * nb,
                       [&] { return launch_walk_proj(oa, L.G, s); }));
      PAMD_CHECK(launch_walk_ulo(at(P.off_u), L.G, nfrag, c.ebar, tri, np, o, p0 == 0, ulo_bar, s));
      st = walk_adjoint(c, L, b, tri, nb, p0 == 0, nullptr);
      if (st != PAMD_OK) return st;
    }
    PAMD_CHECK(meter.report((long long)(p0 + np) * o, s));
  }
  g_prof_on = false;
  if (!g_prof_recs.empty()) PAMD_CHECK(prof_collect());
  PAMD_CHECK(launch_projected_total(at(P.off_pair), o, e_out, s));
  return c.vjp ? walk_finish(c, L, b, ovvv_bar, mo_bar) : PAMD_OK;
}

// ---------------------------------------------------------------------------
// Library-owned scratch for pamd_ccsdt_energy_vjp_noalloc: the workspace of
// pamd_ccsdt_energy_vjp in a file-scope device array, so that call allocates
// nothing.  Each GPU holds its own copy for the life of the process; its
// address on a device is looked up once (hipGetSymbolAddress, with that device
// current) and kept per device.  The host-side name `scratch` is never passed
// to a kernel or a copy: only the looked-up address is.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void *g_scratch_ptr[kMaxDevices];

// Address of this device's scratch array (the device current on the calling
// thread), or a PAMD_* error.
static int scratch_on_current_device(void **ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    fprintf(stderr, "pyscfad_amd: hipGetDevice failed: %s\n", hipGetErrorString(e));
    return PAMD_ERR_HIP;
  }
  if (dev < 0 || dev >= kMaxDevices) return PAMD_ERR_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      fprintf(stderr, "pyscfad_amd: hipGetSymbolAddress(scratch) failed on device %d: %s\n", dev,
              hipGetErrorString(e));
      return PAMD_ERR_HIP;
    }
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return PAMD_OK;
}

}  // namespace pamd

using namespace pamd;

extern "C" {

const char *pamd_version(void) { return "pyscfad_amd 0.1.0 (gfx950)"; }

int pamd_ccsdt_workspace_size(const pamd_ccsdt_config *cfg, int with_vjp, size_t *bytes) {
  if (!cfg || !bytes || cfg->nocc < 1 || cfg->nvir < 1) return PAMD_ERR_ARG;
  *bytes = make_layout(cfg->nocc, cfg->nvir, with_vjp ? 1 : 0, cfg->precision, true).total;
  return PAMD_OK;
}

int pamd_ccsdt_preferred_workspace_size(const pamd_ccsdt_config *cfg, int with_vjp, size_t *bytes) {
  if (!cfg || !bytes || cfg->nocc < 1 || cfg->nvir < 1) return PAMD_ERR_ARG;
  const int o = cfg->nocc, v = cfg->nvir, vjp = with_vjp ? 1 : 0;
  const Layout L = make_layout(o, v, vjp, cfg->precision, true);
  *bytes = std::max(L.total, b3_layout(o, v, vjp, cfg->precision, true, (size_t)-1, L).total);
  WalkLayout wl;
  if (cfg->precision == PAMD_PREC_FP64 && walk_pick(o, v, vjp, (size_t)-1, *bytes, wl))
    *bytes = std::max(*bytes, wl.total);
  return PAMD_OK;
}

static int energy_impl(const pamd_ccsdt_config *cfg, const double *mo, const double *t1,
                       const double *t2, const double *ovvv, const double *ovoo,
                       const double *ovov, const double *fvo, void *ws, size_t ws_bytes,
                       hipStream_t s, Ctx &c, int shard = 0, int nshards = 1) {
  int st = check_common(cfg, mo, t1, t2, ovvv, ovoo, ovov, fvo);
  if (st != PAMD_OK) return st;
  Layout L = make_layout(cfg->nocc, cfg->nvir, 0, cfg->precision);
  if (!ws || ws_bytes < L.total) return PAMD_ERR_WORKSPACE;
  memset(&c, 0, sizeof(c));
  c.o = cfg->nocc;
  c.v = cfg->nvir;
  c.packed = cfg->ovvv_packed ? 1 : 0;
  c.has_fvo = cfg->has_fvo ? 1 : 0;
  c.vjp = 0;
  c.prec = cfg->precision;
  c.s = s;
  c.mo = mo;
  c.t1 = t1;
  c.t2 = t2;
  c.ovvv = ovvv;
  c.ovoo = ovoo;
  c.ovov = ovov;
  c.fvo = fvo;
  c.shard = shard;
  c.nshards = nshards;
  WalkLayout wl;
  if (c.prec == PAMD_PREC_FP64 && walk_pick(c.o, c.v, 0, ws_bytes, L.total, wl))
    return run_walk(c, wl, ws, nullptr, nullptr);
  bind_workspace(c, b3_layout(c.o, c.v, 0, c.prec, false, ws_bytes, L), ws);
  return run(c);
}

int pamd_ccsdt_energy(const pamd_ccsdt_config *cfg, const double *mo_energy, const double *t1,
                      const double *t2, const double *ovvv, const double *ovoo, const double *ovov,
                      const double *fvo, void *workspace, size_t workspace_bytes, double *e_out,
                      void *stream) {
  if (!e_out) return PAMD_ERR_ARG;
  Ctx c;
  hipStream_t s = (hipStream_t)stream;
  int st = energy_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, workspace, workspace_bytes,
                       s, c);
  if (st != PAMD_OK) return st;
  PAMD_CHECK(launch_total_energy(c.tri, c.o, e_out, s));
  return PAMD_OK;
}

int pamd_ccsdt_num_triples(int nocc, long long *n) {
  if (nocc < 1 || !n) return PAMD_ERR_ARG;
  *n = (long long)nocc * (nocc + 1) * (nocc + 2) / 6 - nocc;
  return PAMD_OK;
}

int pamd_ccsdt_energy_shard(const pamd_ccsdt_config *cfg, const double *mo_energy,
                            const double *t1, const double *t2, const double *ovvv,
                            const double *ovoo, const double *ovov, const double *fvo, int shard,
                            int nshards, void *workspace, size_t workspace_bytes, double *e_out,
                            void *stream) {
  if (!e_out || nshards < 1 || shard < 0 || shard >= nshards) return PAMD_ERR_ARG;
  Ctx c;
  hipStream_t s = (hipStream_t)stream;
  int st = energy_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, workspace, workspace_bytes,
                       s, c, shard, nshards);
  if (st != PAMD_OK) return st;
  PAMD_CHECK(launch_total_energy(c.tri, c.o, e_out, s));
  return PAMD_OK;
}

int pamd_ccsdt_pair_energy(const pamd_ccsdt_config *cfg, const double *mo_energy, const double *t1,
                           const double *t2, const double *ovvv, const double *ovoo,
                           const double *ovov, const double *fvo, void *workspace,
                           size_t workspace_bytes, double *e_pair, void *stream) {
  if (!e_pair) return PAMD_ERR_ARG;
  Ctx c;
  hipStream_t s = (hipStream_t)stream;
  int st = energy_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, workspace, workspace_bytes,
                       s, c);
  if (st != PAMD_OK) return st;
  PAMD_CHECK(launch_pair_energy(c.tri, c.o, e_pair, s));
  return PAMD_OK;
}

static int vjp_impl(const pamd_ccsdt_config *cfg, const double *mo_energy, const double *t1,
                    const double *t2, const double *ovvv, const double *ovoo, const double *ovov,
                    const double *fvo, const double *wt_host, double et_bar, void *workspace,
                    size_t workspace_bytes, double *e_out, double *mo_energy_bar, double *t1_bar,
                    double *t2_bar, double *ovvv_bar, double *ovoo_bar, double *ovov_bar,
                    double *fvo_bar, double *wt_bar, void *stream, int shard = 0,
                    int nshards = 1, bool pipe = true, bool batched = true) {
  int st = check_common(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo);
  if (st != PAMD_OK) return st;
  if (!e_out || !mo_energy_bar || !t1_bar || !t2_bar || !ovvv_bar || !ovoo_bar || !ovov_bar ||
      !fvo_bar)
    return PAMD_ERR_ARG;
  Layout L = make_layout(cfg->nocc, cfg->nvir, 1, cfg->precision, pipe);
  if (!workspace || workspace_bytes < L.total) return PAMD_ERR_WORKSPACE;
  Ctx c;
  memset(&c, 0, sizeof(c));
  c.o = cfg->nocc;
  c.v = cfg->nvir;
  c.packed = cfg->ovvv_packed ? 1 : 0;
  c.has_fvo = cfg->has_fvo ? 1 : 0;
  c.vjp = 1;
  c.prec = cfg->precision;
  c.s = (hipStream_t)stream;
  c.mo = mo_energy;
  c.t1 = t1;
  c.t2 = t2;
  c.ovvv = ovvv;
  c.ovoo = ovoo;
  c.ovov = ovov;
  c.fvo = fvo;
  c.ebar = et_bar;
  c.wt_host = wt_host;
  c.t1_bar = t1_bar;
  c.t2_bar = t2_bar;
  c.ovoo_bar = ovoo_bar;
  c.ovov_bar = ovov_bar;
  c.fvo_bar = fvo_bar;
  c.shard = shard;
  c.nshards = nshards;
  WalkLayout wl;
  const bool walk =
      batched && c.prec == PAMD_PREC_FP64 && walk_pick(c.o, c.v, 1, workspace_bytes, L.total, wl);
  if (walk) {
    st = run_walk(c, wl, workspace, ovvv_bar, mo_energy_bar);
  } else {
    bind_workspace(c, b3_layout(c.o, c.v, 1, c.prec, pipe, workspace_bytes, L), workspace);
    st = run(c);
  }
  if (st != PAMD_OK) return st;
  const int o = c.o, v = c.v;
  if (wt_host) {
    if (!walk && !c.pad)
      PAMD_CHECK(hipMemcpyAsync(c.wt, wt_host, sizeof(double) * (size_t)o, hipMemcpyHostToDevice,
                                c.s));
    PAMD_CHECK(launch_weighted_energy(c.tri, o, c.wt, et_bar, e_out, wt_bar, c.s));
  } else {
    PAMD_CHECK(launch_total_energy(c.tri, o, e_out, c.s));
  }
  if (walk) return PAMD_OK;
  PAMD_CHECK(launch_reduce_rows(c.part_mo, c.G, o + v, o + c.vp, mo_energy_bar, 0, c.s));
  PAMD_CHECK(launch_fold_ovvv(c.Vpb, o, v, c.vp, c.packed, ovvv_bar, c.s));
  PAMD_CHECK(launch_fold_t2m(c.T2mb, o, v, c.op, c.vp, t2_bar, c.s));
  return PAMD_OK;
}

int pamd_ccsdt_energy_vjp(const pamd_ccsdt_config *cfg, const double *mo_energy, const double *t1,
                          const double *t2, const double *ovvv, const double *ovoo,
                          const double *ovov, const double *fvo, double et_bar, void *workspace,
                          size_t workspace_bytes, double *e_out, double *mo_energy_bar,
                          double *t1_bar, double *t2_bar, double *ovvv_bar, double *ovoo_bar,
                          double *ovov_bar, double *fvo_bar, void *stream) {
  return vjp_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, nullptr, et_bar, workspace,
                  workspace_bytes, e_out, mo_energy_bar, t1_bar, t2_bar, ovvv_bar, ovoo_bar,
                  ovov_bar, fvo_bar, nullptr, stream);
}

int pamd_ccsdt_energy_vjp_shard(const pamd_ccsdt_config *cfg, const double *mo_energy,
                                const double *t1, const double *t2, const double *ovvv,
                                const double *ovoo, const double *ovov, const double *fvo,
                                double et_bar, int shard, int nshards, void *workspace,
                                size_t workspace_bytes, double *e_out, double *mo_energy_bar,
                                double *t1_bar, double *t2_bar, double *ovvv_bar,
                                double *ovoo_bar, double *ovov_bar, double *fvo_bar,
                                void *stream) {
  if (nshards < 1 || shard < 0 || shard >= nshards) return PAMD_ERR_ARG;
  return vjp_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, nullptr, et_bar, workspace,
                  workspace_bytes, e_out, mo_energy_bar, t1_bar, t2_bar, ovvv_bar, ovoo_bar,
                  ovov_bar, fvo_bar, nullptr, stream, shard, nshards);
}

size_t pamd_ccsdt_noalloc_scratch_bytes(void) { return kNoAllocScratchBytes; }

int pamd_ccsdt_noalloc_workspace_size(const pamd_ccsdt_config *cfg, size_t *bytes) {
  if (!cfg || !bytes || cfg->nocc < 1 || cfg->nvir < 1) return PAMD_ERR_ARG;
  *bytes = make_layout(cfg->nocc, cfg->nvir, 1, cfg->precision).total;
  return PAMD_OK;
}

int pamd_ccsdt_energy_vjp_noalloc(const pamd_ccsdt_config *cfg, const double *mo_energy,
                                  const double *t1, const double *t2, const double *ovvv,
                                  const double *ovoo, const double *ovov, const double *fvo,
                                  double et_bar, double *e_out, double *mo_energy_bar,
                                  double *t1_bar, double *t2_bar, double *ovvv_bar,
                                  double *ovoo_bar, double *ovov_bar, double *fvo_bar,
                                  void *stream) {
  int st = check_common(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo);
  if (st != PAMD_OK) return st;
  const Layout L = make_layout(cfg->nocc, cfg->nvir, 1, cfg->precision);
  if (L.total > kNoAllocScratchBytes) {
    fprintf(stderr,
            "pyscfad_amd: pamd_ccsdt_energy_vjp_noalloc: nocc=%d nvir=%d needs %zu bytes of "
            "scratch, more than the library's %zu; use pamd_ccsdt_energy_vjp with a workspace\n",
            cfg->nocc, cfg->nvir, L.total, kNoAllocScratchBytes);
    return PAMD_ERR_WORKSPACE;
  }
  void *ws = nullptr;
  st = scratch_on_current_device(&ws);
  if (st != PAMD_OK) return st;
  g_prof_blocked = true;
  // one triple in flight: no second stream, events or buffer copies
  st = vjp_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, nullptr, et_bar, ws,
                kNoAllocScratchBytes, e_out, mo_energy_bar, t1_bar, t2_bar, ovvv_bar, ovoo_bar,
                ovov_bar, fvo_bar, nullptr, stream, 0, 1, false);
  g_prof_blocked = false;
  return st;
}

int pamd_ccsdt_weighted_energy_vjp(const pamd_ccsdt_config *cfg, const double *mo_energy,
                                   const double *t1, const double *t2, const double *ovvv,
                                   const double *ovoo, const double *ovov, const double *fvo,
                                   const double *occ_weight, double et_bar, void *workspace,
                                   size_t workspace_bytes, double *e_out, double *mo_energy_bar,
                                   double *t1_bar, double *t2_bar, double *ovvv_bar,
                                   double *ovoo_bar, double *ovov_bar, double *fvo_bar,
                                   double *occ_weight_bar, void *stream) {
  if (!occ_weight || !occ_weight_bar) return PAMD_ERR_ARG;
  return vjp_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, occ_weight, et_bar, workspace,
                  workspace_bytes, e_out, mo_energy_bar, t1_bar, t2_bar, ovvv_bar, ovoo_bar,
                  ovov_bar, fvo_bar, occ_weight_bar, stream);
}

// workspace of the projected walk: the plain layout (forward or adjoint), then
// accA, accB (nfrag v^3 each), the pair energies (o^2), the dot partials
// (kGmax) and the per-workgroup dE/dulo sums (kGmax x kMaxFrag)
struct ProjLayout {
  Layout L;
  size_t off_a, off_b, off_p, off_d, off_u, total;
};

static ProjLayout projected_layout(int o, int v, int nfrag, int vjp, int prec) {
  ProjLayout P;
  P.L = make_layout(o, v, vjp, prec);
  const size_t blk = align256(sizeof(double) * (size_t)nfrag * v * v * v);
  P.off_a = P.L.total;
  P.off_b = P.off_a + blk;
  P.off_p = P.off_b + blk;
  P.off_d = P.off_p + align256(sizeof(double) * (size_t)o * o);
  P.off_u = P.off_d + align256(sizeof(double) * kGmax);
  P.total = P.off_u + align256(sizeof(double) * kGmax * kMaxFrag);
  return P;
}

int pamd_ccsdt_projected_workspace_size(const pamd_ccsdt_config *cfg, int nfrag, int with_vjp,
                                        size_t *bytes) {
  if (!cfg || !bytes || cfg->nocc < 1 || cfg->nvir < 1 || nfrag < 1 || nfrag > kMaxFrag)
    return PAMD_ERR_ARG;
  *bytes = projected_layout(cfg->nocc, cfg->nvir, nfrag, with_vjp ? 1 : 0, cfg->precision).total;
  return PAMD_OK;
}

int pamd_ccsdt_projected_preferred_workspace_size(const pamd_ccsdt_config *cfg, int nfrag, int with_vjp,
                                                  size_t *bytes) {
  const int st = pamd_ccsdt_projected_workspace_size(cfg, nfrag, with_vjp, bytes);
  if (st != PAMD_OK) return st;
  ProjWalkLayout pw;
  if (cfg->precision == PAMD_PREC_FP64 &&
      proj_walk_pick(cfg->nocc, cfg->nvir, nfrag, with_vjp ? 1 : 0, (size_t)-1, *bytes, pw))
    *bytes = std::max(*bytes, pw.total);
  return PAMD_OK;
}

static int projected_impl(const pamd_ccsdt_config *cfg, const double *mo_energy, const double *t1,
                          const double *t2, const double *ovvv, const double *ovoo,
                          const double *ovov, const double *fvo, const double *ulo, int nfrag,
                          int vjp, double et_bar, void *workspace, size_t workspace_bytes,
                          double *e_out, double *mo_energy_bar, double *t1_bar, double *t2_bar,
                          double *ovvv_bar, double *ovoo_bar, double *ovov_bar, double *fvo_bar,
                          double *ulo_bar, void *stream, bool batched = true) {
  int st = check_common(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo);
  if (st != PAMD_OK) return st;
  if (!ulo || !e_out || nfrag < 1 || nfrag > kMaxFrag) return PAMD_ERR_ARG;
  if (vjp && (!mo_energy_bar || !t1_bar || !t2_bar || !ovvv_bar || !ovoo_bar || !ovov_bar ||
              !fvo_bar || !ulo_bar))
    return PAMD_ERR_ARG;
  const ProjLayout P = projected_layout(cfg->nocc, cfg->nvir, nfrag, vjp, cfg->precision);
  if (!workspace || workspace_bytes < P.total) return PAMD_ERR_WORKSPACE;
  Ctx c;
  memset(&c, 0, sizeof(c));
  c.o = cfg->nocc;
  c.v = cfg->nvir;
  c.packed = cfg->ovvv_packed ? 1 : 0;
  c.has_fvo = cfg->has_fvo ? 1 : 0;
  c.vjp = vjp;
  c.prec = cfg->precision;
  c.s = (hipStream_t)stream;
  c.mo = mo_energy;
  c.t1 = t1;
  c.t2 = t2;
  c.ovvv = ovvv;
  c.ovoo = ovoo;
  c.ovov = ovov;
  c.fvo = fvo;
  c.ebar = et_bar;
  c.t1_bar = t1_bar;
  c.t2_bar = t2_bar;
  c.ovoo_bar = ovoo_bar;
  c.ovov_bar = ovov_bar;
  c.fvo_bar = fvo_bar;
  ProjWalkLayout pw;
  if (batched && c.prec == PAMD_PREC_FP64 &&
      proj_walk_pick(c.o, c.v, nfrag, vjp, workspace_bytes, P.total, pw)) {
    c.nshards = 1;
    return run_projected_walk(c, pw, workspace, ulo, nfrag, e_out, ovvv_bar, mo_energy_bar, ulo_bar);
  }
  bind_workspace(c, P.L, workspace);
  char *b = (char *)workspace;
  double *pair_e = (double *)(b + P.off_p);
  st = run_projected(c, ulo, nfrag, (double *)(b + P.off_a), (double *)(b + P.off_b), pair_e,
                     (double *)(b + P.off_d), (double *)(b + P.off_u), ulo_bar);
  if (st != PAMD_OK) return st;
  PAMD_CHECK(launch_projected_total(pair_e, c.o, e_out, c.s));
  if (vjp) {
    const int o = c.o, v = c.v;
    PAMD_CHECK(launch_reduce_rows(c.part_mo, c.G, o + v, o + c.vp, mo_energy_bar, 0, c.s));
    PAMD_CHECK(launch_fold_ovvv(c.Vpb, o, v, c.vp, c.packed, ovvv_bar, c.s));
    PAMD_CHECK(launch_fold_t2m(c.T2mb, o, v, c.op, c.vp, t2_bar, c.s));
  }
  return PAMD_OK;
}

int pamd_ccsdt_projected_energy(const pamd_ccsdt_config *cfg, const double *mo_energy,
                                const double *t1, const double *t2, const double *ovvv,
                                const double *ovoo, const double *ovov, const double *fvo,
                                const double *ulo, int nfrag, void *workspace,
                                size_t workspace_bytes, double *e_out, void *stream) {
  return projected_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, ulo, nfrag, 0, 0.0,
                        workspace, workspace_bytes, e_out, nullptr, nullptr, nullptr, nullptr,
                        nullptr, nullptr, nullptr, nullptr, stream);
}

int pamd_ccsdt_projected_energy_vjp(const pamd_ccsdt_config *cfg, const double *mo_energy,
                                    const double *t1, const double *t2, const double *ovvv,
                                    const double *ovoo, const double *ovov, const double *fvo,
                                    const double *ulo, int nfrag, double et_bar, void *workspace,
                                    size_t workspace_bytes, double *e_out, double *mo_energy_bar,
                                    double *t1_bar, double *t2_bar, double *ovvv_bar,
                                    double *ovoo_bar, double *ovov_bar, double *fvo_bar,
                                    double *ulo_bar, void *stream) {
  return projected_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, ulo, nfrag, 1, et_bar,
                        workspace, workspace_bytes, e_out, mo_energy_bar, t1_bar, t2_bar,
                        ovvv_bar, ovoo_bar, ovov_bar, fvo_bar, ulo_bar, stream);
}

int pamd_debug_one_triple_vjp(const pamd_ccsdt_config *cfg, const double *mo_energy, const double *t1,
                              const double *t2, const double *ovvv, const double *ovoo, const double *ovov,
                              const double *fvo, double et_bar, int two_streams, void *workspace,
                              size_t workspace_bytes, double *e_out, double *mo_energy_bar, double *t1_bar,
                              double *t2_bar, double *ovvv_bar, double *ovoo_bar, double *ovov_bar,
                              double *fvo_bar, void *stream) {
  return vjp_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, nullptr, et_bar, workspace, workspace_bytes,
                  e_out, mo_energy_bar, t1_bar, t2_bar, ovvv_bar, ovoo_bar, ovov_bar, fvo_bar, nullptr, stream,
                  0, 1, two_streams != 0, false);
}

int pamd_debug_one_triple_projected_vjp(const pamd_ccsdt_config *cfg, const double *mo_energy, const double *t1,
                                        const double *t2, const double *ovvv, const double *ovoo,
                                        const double *ovov, const double *fvo, const double *ulo, int nfrag,
                                        double et_bar, void *workspace, size_t workspace_bytes, double *e_out,
                                        double *mo_energy_bar, double *t1_bar, double *t2_bar, double *ovvv_bar,
                                        double *ovoo_bar, double *ovov_bar, double *fvo_bar, double *ulo_bar,
                                        void *stream) {
  return projected_impl(cfg, mo_energy, t1, t2, ovvv, ovoo, ovov, fvo, ulo, nfrag, 1, et_bar, workspace,
                        workspace_bytes, e_out, mo_energy_bar, t1_bar, t2_bar, ovvv_bar, ovoo_bar, ovov_bar,
                        fvo_bar, ulo_bar, stream, false);
}

int pamd_debug_walk_batch(int nocc, int nvir, int nfrag, int with_vjp, size_t workspace_bytes, int *triples) {
  if (nocc < 1 || nvir < 1 || nfrag < 0 || nfrag > kMaxFrag || !triples) return PAMD_ERR_ARG;
  const int vjp = with_vjp ? 1 : 0;
  *triples = 0;
  if (nfrag) {
    ProjWalkLayout pw;
    if (proj_walk_pick(nocc, nvir, nfrag, vjp, workspace_bytes,
                       projected_layout(nocc, nvir, nfrag, vjp, PAMD_PREC_FP64).total, pw))
      *triples = pw.np * nocc;
  } else {
    WalkLayout wl;
    if (walk_pick(nocc, nvir, vjp, workspace_bytes, make_layout(nocc, nvir, vjp, PAMD_PREC_FP64, true).total, wl))
      *triples = wl.nb;
  }
  return PAMD_OK;
}

int pamd_debug_walk_bytes(int nocc, int nvir, int nfrag, int with_vjp, size_t workspace_bytes, size_t *bytes) {
  if (nocc < 1 || nvir < 1 || nfrag < 0 || nfrag > kMaxFrag || !bytes) return PAMD_ERR_ARG;
  const int vjp = with_vjp ? 1 : 0;
  *bytes = 0;
  if (nfrag) {
    ProjWalkLayout pw;
    if (proj_walk_pick(nocc, nvir, nfrag, vjp, workspace_bytes,
                       projected_layout(nocc, nvir, nfrag, vjp, PAMD_PREC_FP64).total, pw))
      *bytes = pw.total;
  } else {
    WalkLayout wl;
    if (walk_pick(nocc, nvir, vjp, workspace_bytes, make_layout(nocc, nvir, vjp, PAMD_PREC_FP64, true).total, wl))
      *bytes = wl.total;
  }
  return PAMD_OK;
}

int pamd_debug_gemm_direct_ok(const void *desc) {
  if (!desc) return -PAMD_ERR_ARG;
  GemmDesc d;
  memcpy(&d, desc, sizeof(d));
  return gemm_direct_ok(d) ? 1 : 0;
}

int pamd_debug_gemm_b3p_ok(const void *desc, long long plane_stride) {
  if (!desc) return -PAMD_ERR_ARG;
  GemmDesc d;
  memcpy(&d, desc, sizeof(d));
  for (int q = 0; q < d.nseg; ++q)
    for (OpDesc *op : {&d.seg[q].A, &d.seg[q].B}) {
      // FP64 element address e * 8 -> bf16 element address e * 2
      op->p = (const double *)((uintptr_t)op->p / 4);
      op->ps = plane_stride;
    }
  return gemm_b3p_ok(d) ? 1 : 0;
}

int pamd_debug_gemm_descriptors(int nocc, int nvir, int i, int j, int k, int with_vjp,
                                const unsigned long long *bases, void *out, int max_desc,
                                int *n_desc, int *desc_bytes) {
  if (nocc < 1 || nvir < 1 || !bases || !n_desc || !desc_bytes) return PAMD_ERR_ARG;
  if (i < 0 || j < i || k < j || k >= nocc) return PAMD_ERR_ARG;
  Layout L = make_layout(nocc, nvir, with_vjp ? 1 : 0, PAMD_PREC_FP64);
  Ctx c;
  memset(&c, 0, sizeof(c));
  c.o = c.op = nocc;
  c.v = c.vp = nvir;
  c.vjp = with_vjp ? 1 : 0;
  c.Vp = (double *)bases[0];
  c.T2m = (double *)bases[1];
  c.OOt = (double *)bases[2];
  c.W = (double *)bases[3];
  c.gW = c.W;
  c.t2 = (const double *)bases[4];
  c.gT2 = c.t2;
  c.Vb = (double *)bases[5];
  c.Vpb = (double *)bases[6];
  c.T2mb = (double *)bases[7];
  c.part_p = (double *)bases[8];
  c.part_h = (double *)bases[9];
  c.S_p = L.S_p;
  c.S_h = L.S_h;
  std::vector<GemmDesc> rec;
  g_record = &rec;
  int st = build_w(c, i, j, k);
  if (st == PAMD_OK && with_vjp) st = adjoint(c, i, j, k);
  g_record = nullptr;
  if (st != PAMD_OK) return st;
  *desc_bytes = (int)sizeof(GemmDesc);
  *n_desc = (int)rec.size();
  if (out) {
    const int n = std::min((int)rec.size(), max_desc);
    memcpy(out, rec.data(), sizeof(GemmDesc) * (size_t)n);
  }
  return PAMD_OK;
}

int pamd_debug_adjoint_launches(int nocc, int nvir, int i, int j, int k, const unsigned long long *bases,
                                void *out, int *launch, int max_desc, int *n_desc, int *desc_bytes) {
  if (nocc < 1 || nvir < 1 || !bases || !out || !launch || !n_desc || !desc_bytes) return PAMD_ERR_ARG;
  if (i < 0 || j < 0 || k < 0 || i >= nocc || j >= nocc || k >= nocc) return PAMD_ERR_ARG;
  const Layout L = make_layout(nocc, nvir, 1, PAMD_PREC_BF16X3);
  Ctx c;
  memset(&c, 0, sizeof(c));
  c.prec = PAMD_PREC_BF16X3;
  c.o = c.op = nocc;
  c.v = c.vp = nvir;
  c.vjp = 1;
  c.Vp = (double *)bases[0];
  c.T2m = (double *)bases[1];
  c.OOt = (double *)bases[2];
  c.W = c.gW = (double *)bases[3];
  c.t2 = c.gT2 = (const double *)bases[4];
  c.Vpb = (double *)bases[6];
  c.T2mb = (double *)bases[7];
  c.part_p = (double *)bases[8];
  c.part_h = (double *)bases[9];
  c.S_p = L.S_p;
  c.S_h = L.S_h;
  std::vector<GemmDesc> rec;
  std::vector<int> at;
  g_record = &rec;
  g_record_launch = &at;
  const int st = adjoint_gemms(c, i, j, k);
  g_record = nullptr;
  g_record_launch = nullptr;
  if (st != PAMD_OK) return st;
  *desc_bytes = (int)sizeof(GemmDesc);
  *n_desc = (int)rec.size();
  const int n = std::min((int)rec.size(), max_desc);
  memcpy(out, rec.data(), sizeof(GemmDesc) * (size_t)n);
  memcpy(launch, at.data(), sizeof(int) * (size_t)n);
  return PAMD_OK;
}

int pamd_debug_paired_adjoint_descriptors(int nocc, int nvir, int i, int j, int kp, int k,
                                          const unsigned long long *bases, void *out,
                                          int max_desc, int *n_desc, int *desc_bytes) {
  if (nocc < 1 || nvir < 1 || !bases || !n_desc || !desc_bytes) return PAMD_ERR_ARG;
  if (i < 0 || j < i || kp < j || k <= kp || k >= nocc) return PAMD_ERR_ARG;
  Layout L = make_layout(nocc, nvir, 1, PAMD_PREC_FP64);
  Ctx c1;
  memset(&c1, 0, sizeof(c1));
  c1.o = c1.op = nocc;
  c1.v = c1.vp = nvir;
  c1.vjp = 1;
  c1.Vp = (double *)bases[0];
  c1.T2m = (double *)bases[1];
  c1.OOt = (double *)bases[2];
  c1.W = (double *)bases[3];
  c1.gW = c1.W;
  c1.t2 = (const double *)bases[4];
  c1.gT2 = c1.t2;
  c1.Vb = (double *)bases[5];
  c1.Vpb = (double *)bases[6];
  c1.T2mb = (double *)bases[7];
  c1.part_p = (double *)bases[8];
  c1.part_h = (double *)bases[9];
  c1.S_p = L.S_p;
  c1.S_h = L.S_h;
  Ctx c2 = c1;
  c2.W = (double *)bases[10];
  c2.gW = c2.W;
  std::vector<GemmDesc> rec;
  g_record = &rec;
  int st = adjoint_gemms(c1, i, j, kp, 1);
  if (st == PAMD_OK) st = adjoint_gemms(c2, i, j, k, 2, &c1, kp);
  g_record = nullptr;
  if (st != PAMD_OK) return st;
  *desc_bytes = (int)sizeof(GemmDesc);
  *n_desc = (int)rec.size();
  if (out) {
    const int n = std::min((int)rec.size(), max_desc);
    memcpy(out, rec.data(), sizeof(GemmDesc) * (size_t)n);
  }
  return PAMD_OK;
}

int pamd_profile_enable(int every) {
  if (every < 0) return PAMD_ERR_ARG;
  g_prof_every = every;
  return PAMD_OK;
}

int pamd_profile_progress(int every) {
  if (every < 0) return PAMD_ERR_ARG;
  g_progress_every = every;
  return PAMD_OK;
}

int pamd_profile_reset(void) {
  std::lock_guard<std::mutex> lock(g_prof_mutex);
  memset(g_prof_stat, 0, sizeof(g_prof_stat));
  return PAMD_OK;
}

int pamd_profile_num_kinds(void) { return kProfNum; }

const char *pamd_profile_kind_name(int kind) {
  return (kind >= 0 && kind < kProfNum) ? kProfNames[kind] : "";
}

int pamd_profile_read(int kind, long long *launches, double *ms, double *flops, double *bytes) {
  if (kind < 0 || kind >= kProfNum || !launches || !ms || !flops || !bytes) return PAMD_ERR_ARG;
  std::lock_guard<std::mutex> lock(g_prof_mutex);
  *launches = g_prof_stat[kind].launches;
  *ms = g_prof_stat[kind].ms;
  *flops = g_prof_stat[kind].flops;
  *bytes = g_prof_stat[kind].bytes;
  return PAMD_OK;
}

int pamd_debug_split_factors(int nocc, int nvir, int *S_p, int *S_h) {
  return pamd_debug_split_factors_prec(nocc, nvir, PAMD_PREC_FP64, S_p, S_h);
}

int pamd_debug_split_factors_prec(int nocc, int nvir, int precision, int *S_p, int *S_h) {
  if (nocc < 1 || nvir < 1 || !S_p || !S_h) return PAMD_ERR_ARG;
  if (precision != PAMD_PREC_FP64 && precision != PAMD_PREC_BF16X3 && precision != PAMD_PREC_FP32X2)
    return PAMD_ERR_ARG;
  Layout L = make_layout(nocc, nvir, 1, precision);
  *S_p = L.S_p;
  *S_h = L.S_h;
  return PAMD_OK;
}

}  // extern "C"
