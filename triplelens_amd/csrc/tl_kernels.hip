// HIP kernels of the IRS engine (gfx950).
//
//  trial_*_kernel per light-curve point, all at once: source position, caustic
//                 trial points (src/LightCurves/lcirs.cc:131-165) and the
//                 image polynomial of every solve (tl_coeffs.h).
//  seed_kernel    per light curve, the reference's seed sequence: point images
//                 with the root-reuse chain, then the images of caustic trial
//                 points (src/LightCurves/lcirs.cc:116-165), as pixel seeds.
//  solve_prep_kernel  what a solve of the chain needs that does not depend on
//                 the chain (its first deflation step, its fresh solve).
//  spec_*_kernel  the chain in pieces in parallel, verified, with repair chains
//                 that run beside the fill of the pieces already known.
//  fill_kernel    one persistent, work-stealing launch that grows the image
//                 "amoebae" of a batch of source positions: wavefronts pop
//                 row-check tasks, evaluate 64 pixels per step with the FP64
//                 ray map, record maximal hit runs in a shared run table and
//                 sweep on to the next row.  Counted set and brightness sum are
//                 those of lineFloodFill (lcirs.cc:381-466): every 4-connected
//                 component of hit pixels that holds a hit seed.
//  resolve_kernel folds the per-label partial sums into per-point results.
//
// Compiled with -ffp-contract=off: the hit test rsq < rho^2 is decided on the
// same IEEE values as the reference's irsSIMD.
#include <hip/hip_runtime.h>
#include "tl_engine.h"
#include "tl_roots.h"

namespace tl {

#define AGENT __HIP_MEMORY_SCOPE_AGENT

// Shared state of the fill (run table, labels, queue, counters) is accessed
// only through relaxed agent-scope atomics, which are performed at the
// device's coherence point.  Where one such access must be visible before
// another, mem_order() waits until all of the wave's outstanding memory
// operations have completed; acquire/release orderings are not used because
// on this GPU they write back or invalidate the whole L2 cache.
__device__ __forceinline__ unsigned long long ald(unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, AGENT);
}
__device__ __forceinline__ void ast(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, AGENT);
}
__device__ __forceinline__ bool acas(unsigned long long* p, unsigned long long* expected,
                                     unsigned long long desired) {
  return __hip_atomic_compare_exchange_strong(p, expected, desired, __ATOMIC_RELAXED,
                                              __ATOMIC_RELAXED, AGENT);
}
__device__ __forceinline__ int aldi(int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, AGENT); }
__device__ __forceinline__ void mem_order() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

__device__ __forceinline__ long long wave_sum(long long v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Wave-uniform values in scalar registers (the first active lane's value;
// used where every lane holds the same value or lane 0 holds the result).
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ long long uni64(long long v) {
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long long)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)((unsigned long long)v >> 32));
  return (long long)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double unid(double v) {
  return __longlong_as_double(uni64(__double_as_longlong(v)));
}

// ---------------------------------------------------------------------------
// Plane -> pixel mapping (lcirs.cc:355-378; pixel -> plane is formed where a row is scanned)
// ---------------------------------------------------------------------------
// (long)((x - BL) * N / L + 0.5), with the operand clamped so that the
// conversion is defined for any root.
__device__ __forceinline__ int to_pixel(double v, double bl, double Nd, double L) {
  double t = (v - bl) * Nd / L + 0.5;
  if (!(t > -1.0e9)) t = -1.0e9;
  if (t > 1.0e9) t = 1.0e9;
  return (int)(long long)t;
}

// ---------------------------------------------------------------------------
// Seeds
// ---------------------------------------------------------------------------
__device__ double point_amp_term(const Lens& L, cx z) {
  cx d1 = csub(z, L.z1), d2 = csub(z, L.z2), d3 = csub(z, L.z3);
  cx s = cadd(cadd(cdiv_rc(L.m1, cmul(d1, d1)), cdiv_rc(L.m2, cmul(d2, d2))),
              cdiv_rc(L.m3, cmul(d3, d3)));
  double t = 1.0 / fabs(1.0 - cnorm(s));
  return t == t ? t : 0.0;
}

// ---- wave-cooperative seed search -----------------------------------------
// One wavefront per light curve.  The root-reuse chain is serial; its vectors
// are spread over the lanes (lane k holds coefficient k, or root k) and the
// serial steps read single elements with readlane, so nothing is indexed at
// run time and everything stays in registers.  The independent parts (the
// coefficients, the 10 root polishes, the 10 image tests and the
// caustic-segment tests) run on separate lanes.  Values and their order are
// those of the serial code in tl_math.h, operation for operation.

__device__ __forceinline__ double rl(double v, int k) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, k);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), k);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ cx rlc(const cx& v, int k) { return mk(rl(v.re, k), rl(v.im, k)); }
// The deflation steps J..1 of Laguerre::solveRoots (laguerre.cc:103-167) on
// a wavefront whose lanes all hold the same polynomial p and the same x: the
// root of step J goes to lane 10 - J of rootv.  initv's lane j seeds the
// search of step j.  The accepted x's Horner sums are the next polynomial.
template <int J>
__device__ __forceinline__ void wl_deflate(const cx (&p)[J + 1], cx& rootv, const cx& initv,
                                           const TrigTable* trig, bool& oob) {
  const int ln = __lane_id();
  cx x = rlc(initv, J);
  if constexpr (J == 1) {
    // a root step that fails restarts from (eps, eps), which is what it then
    // leaves as the root (laguerre.cc:120-128)
    if (p[1].re != 0.0 || p[1].im != 0.0) x = cdiv_sel(cneg(p[0]), p[1]);
    else x = mk(kLagEps, kLagEps);
    if (ln == 9) rootv = x;
  } else {
    cx b[J + 1];
    if (!lag_wave<J, true>(p, x, b, trig, oob)) {
      x = mk(kLagEps, kLagEps);
      horner_sums<J>(p, x, b);
    }
    if (ln == 10 - J) rootv = x;
    cx q[J];
#pragma unroll
    for (int j = 0; j < J; j++) q[j] = b[j + 1];
    wl_deflate<J - 1>(q, rootv, initv, trig, oob);
  }
}

// v of the lane n places further round its row of 16 lanes.
template <int N>
__device__ __forceinline__ double row_ror(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x120 + N, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + N, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
template <int N>
__device__ __forceinline__ cx row_times(const cx& v) {
  return cmul(v, mk(row_ror<N>(v.re), row_ror<N>(v.im)));
}

// Laguerre::checkRoots (laguerre.cc:188-198) on roots held one per lane, as
// written (the product in root order).
__device__ __forceinline__ bool wl_check_exact(cx c10, cx a0, const cx& rootv) {
  cx c0 = c10;
  for (int j = 0; j < 10; j++) c0 = cmul(c0, cneg(rlc(rootv, j)));
  if (cabs_(a0) > 1.0e-8) return (1.0 - cabs_(cdiv_sel(c0, a0))) < 1.0e-5;
  return cabs_(csub(c0, a0)) < 1.0e-10;
}

// checkRoots decided from the product taken in any order (a tree over the
// lanes, good to a few units in the last place) where |c0 / a0| is not within
// 1e-9 of its threshold 1 - 1e-5; ten sign changes cancel.
__device__ __forceinline__ bool wl_check(cx c10, cx a0, const cx& rootv) {
  const int ln = __lane_id();
  cx v = ln < 10 ? rootv : mk(1.0, 0.0);
  v = row_times<8>(v);
  v = row_times<4>(v);
  v = row_times<2>(v);
  v = row_times<1>(v);
  const double A = cnorm(cmul(c10, v)), T = cnorm(a0) * ((1.0 - 1.0e-5) * (1.0 - 1.0e-5));
  const bool big = T > 1.0001e-16 && A < 1e300;
  const unsigned long long yes = __ballot(big && A > T * (1.0 + 1e-9));
  if (yes & 1ull) return true;
  const unsigned long long no = __ballot(big && A < T * (1.0 - 1e-9));
  if (no & 1ull) return false;
  return wl_check_exact(c10, a0, rootv);
}

// img_check (imgpoint.cc:72-90) on every lane's root: the residual of the
// lens equation with fused arithmetic, its error bounded by 1e-14 of the sum
// of its terms' magnitudes; where that leaves the comparison with the
// threshold 1e-6 open on some lane below 10, all lanes run img_check itself.
__device__ __forceinline__ bool wl_img_check(const Lens& L, const cx& z, cx zeta) {
  double wr = z.re - zeta.re, wi = z.im - zeta.im;
  double S = fabs(z.re) + fabs(z.im) + fabs(zeta.re) + fabs(zeta.im);
  auto term = [&](double m, const cx& zk) {
    const double dr = z.re - zk.re, di = z.im - zk.im;
    const double r = m * rcp_near(fma(dr, dr, di * di));
    wr = fma(-dr, r, wr);
    wi = fma(-di, r, wi);
    S = fma(fabs(dr) + fabs(di), fabs(r), S);
  };
  term(L.m1, L.z1);
  term(L.m2, L.z2);
  term(L.m3, L.z3);
  const double n = fma(wr, wr, wi * wi), e = 1e-14 * S;
  const bool yes = e < 5e-7 && n < (1e-6 - e) * (1e-6 - e);
  const bool no = n > (1e-6 + e) * (1e-6 + e);
  if (__ballot(!yes && !no && __lane_id() < 10) == 0) return yes;
  return img_check(L, z, zeta, 1.0e-6);
}

// getRootsPrecalculated + getImages (imgpoint.cc:160-274) on a wavefront for
// one solve of the pool: v is lane k's element k of its record (SolvePool),
// freshv the roots of its fresh solve (root r on lane r).  chainv holds
// tempRoots[k] on lane k.  With `slot`, the chained solve's first step starts
// from tempRoots[10] on lane 10 of chainv (a recorded value of the slot the
// reference reads past the end of its vector) instead of 0.  Returns the mask
// of the roots accepted as images (bit k: root k on lane k of chainv).
//
// The reference's sequence (imgpoint.cc:181-206,262-270): a solve from the
// chain's roots (when it has some), replaced by a fresh solve when the roots
// fail checkRoots; then, if the image count is invalid, one more fresh solve.
// A fresh solve depends on the polynomial alone, and so does the chained
// solve's first step (it starts from 0): solve_prep_kernel has done both for
// every solve of the run, and the chain only runs the deflation steps 9..1,
// the polish and the tests.
//
// The record goes through LDS (`rec`, the wave's own 64 doubles): reading it
// back, every lane gets every element by broadcast, 128 bits at a time.
template <bool TRACED>
__device__ __forceinline__ unsigned long long wl_get_images(const Lens& L, double v, cx freshv,
                                                            double* rec, bool slot, cx& chainv,
                                                            int& have, const TrigTable* trig,
                                                            bool binImg, bool& oob) {
  const int ln = __lane_id();
  const int fl = (int)rl(v, kRecFlags);
  if (have) {
    rec[ln] = v;
    const double2* r2 = reinterpret_cast<const double2*>(rec);
    auto get = [&](int k) {
      const double2 e = r2[k / 2];
      return mk(e.x, e.y);
    };
    cx c[11], p[10];
#pragma unroll
    for (int j = 0; j < 10; j++) p[j] = get(kRecDefl + 2 * j);
    cx rootv = get(kRecRoot);
    bool firstOob = (fl & kRecOobFirst) != 0;
    if constexpr (TRACED) {
      if (slot) {
        firstOob = false;
#pragma unroll
        for (int j = 0; j <= 10; j++) c[j] = get(kRecCoef + 2 * j);
        cx x = rlc(chainv, 10), b[11];
        if (!lag_wave<10, true>(c, x, b, trig, firstOob)) {
          x = mk(kLagEps, kLagEps);
          horner_sums<10>(c, x, b);
        }
        rootv = x;
#pragma unroll
        for (int j = 0; j < 10; j++) p[j] = b[j + 1];
      }
    }
    oob |= firstOob;
    wl_deflate<9>(p, rootv, chainv, trig, oob);
    // root r is polished on lane r; the other lanes repeat root 0
#pragma unroll
    for (int j = 0; j <= 10; j++) c[j] = get(kRecCoef + 2 * j);
    bool laneOob = false;
    cx b[11];
    lag_wave<10, false>(c, rootv, b, trig, laneOob);
    oob |= __ballot(laneOob) != 0;
    if (wl_check(c[10], c[0], rootv)) {
      const bool ok = wl_img_check(L, rootv, get(kRecZeta)) && ln < 10;
      const unsigned long long m = __ballot(ok);
      const int n = __builtin_popcountll(m);
      // a valid count: even and at least 4, or for the binary lens odd and at
      // least 3 (imgpoint.cc:236-237)
      if (binImg ? (n % 2 == 1 && n >= 3) : (n % 2 == 0 && n >= 4)) {
        chainv = ln < 10 ? rootv : mk(0.0, 0.0);
        return m;
      }
    }
  }
  chainv = ln < 10 ? freshv : mk(0.0, 0.0);
  have = 1;
  oob |= (fl & kRecOobFresh) != 0;
  return (unsigned long long)(fl & 0x3ff);
}

// The lens as wave-uniform values (a copy that no store of the kernel can
// alias, so that it is not read again at every position).
__device__ __forceinline__ Lens uni_lens(const Lens& g) {
  Lens L;
  L.m1 = unid(g.m1); L.m2 = unid(g.m2); L.m3 = unid(g.m3);
  L.z1 = mk(unid(g.z1.re), unid(g.z1.im));
  L.z2 = mk(unid(g.z2.re), unid(g.z2.im));
  L.z3 = mk(unid(g.z3.re), unid(g.z3.im));
  return L;
}

// Walks a curve's solves in order (the pool holds them so): the record and
// the fresh roots of the coming solve are loaded one solve ahead, and the
// solve counts 64 positions at a time, so that the chain does not wait for
// memory.
struct SolveWalk {
  const int* count;
  const double* rec;  // this lane's element of the coming solve's record
  const cx* fresh;
  int p, pEnd, k, cnt;
  double v;
  cx f;
  __device__ __forceinline__ SolveWalk(const SolvePool& pool, int p0, int end)
      : count(pool.count), p(p0), pEnd(end), k(64), cnt(0) {
    const int ln = __lane_id();
    const size_t sid = (size_t)uni(pool.base[p0]);
    rec = pool.rec + sid * kRecSize + (ln < kRecSize ? ln : 0);
    fresh = pool.fresh + sid * 10 + (ln < 10 ? ln : 0);
    fetch();
  }
  __device__ __forceinline__ void fetch() {
    v = *rec;
    f = *fresh;
    rec += kRecSize;
    fresh += 10;
  }
  // solves of the next position
  __device__ __forceinline__ int position() {
    if (k == 64) {
      const int q = p + __lane_id();
      cnt = q < pEnd ? count[q] : 0;
      k = 0;
    }
    p++;
    return __builtin_amdgcn_readlane(cnt, k++);
  }
  // the next solve's record and fresh roots
  __device__ __forceinline__ void next(double& rv, cx& fv) {
    rv = v;
    fv = f;
    fetch();
  }
};

// Seed pixels of the images in `m` (root order), appended at out[cnt..].
__device__ __forceinline__ void emit_seeds(const CurveDev& C, const cx& chainv,
                                           unsigned long long m, int2* out, int& cnt,
                                           uint32_t& fl) {
  const int ln = __lane_id();
  const int n = __builtin_popcountll(m);
  if ((m >> ln) & 1ull) {
    const int slot = cnt + __builtin_popcountll(m & ((1ull << ln) - 1ull));
    if (slot < kMaxSeeds)
      out[slot] = make_int2(to_pixel(chainv.re, C.blx, C.Nd, C.Ldbl),
                            to_pixel(chainv.im, C.bly, C.Nd, C.Ldbl));
  }
  if (cnt + n > kMaxSeeds) fl |= kFlagSeedOverflow;
  cnt = cnt + n > kMaxSeeds ? kMaxSeeds : cnt + n;
}

// The caustic trial points of one source position in the reference's order
// (lcirs.cc:131-165): for each caustic branch r whose cumulative box meets
// the source square, the segments k = 0..kCccLen-2 are tested 64 at a time;
// the first hit of every run of consecutive hits is a trial point (the
// reference solves only those; `pointTaken` restarts at each branch).  For
// each step that has trial points, onStep(f, trial) receives their mask f
// (bit j: the segment on lane j, in segment order) and every lane's trial
// position.
template <typename OnStep>
__device__ __forceinline__ void scan_trials(const CurveDev& C, cx pos, const cx* caus,
                                            OnStep&& onStep) {
  const int ln = __lane_id();
  for (int r = 0; r < 6; r++) {
    if (!(pos.re + C.rho >= C.boxMin[r].re && pos.re - C.rho <= C.boxMax[r].re &&
          pos.im + C.rho >= C.boxMin[r].im && pos.im - C.rho <= C.boxMax[r].im))
      continue;
    const cx* cr = caus + r * kCccLen;
    bool prevHit = false;
    for (int k0 = 0; k0 < kCccLen - 1; k0 += 64) {
      const int k = k0 + ln;
      cx trial = mk(0.0, 0.0);
      const bool hit = k < kCccLen - 1 &&
                       intersection_check(pos, cr[k], cr[k + 1], C.rho, C.rho2pow, &trial);
      const unsigned long long hm = __ballot(hit);
      const unsigned long long f = hm & ~((hm << 1) | (prevHit ? 1ull : 0ull));
      prevHit = (hm >> 63) & 1ull;
      if (f) onStep(f, trial);
    }
  }
}

// Everything of a light-curve point that does not depend on the root chain,
// all points at once: its source position, the distance to the nearest
// caustic sample, and the list of positions the chain will solve for (the
// centre, then the caustic trial points).  One wavefront per point counts
// the solves, one workgroup turns the counts into places in the pool (point
// order, so that a chain finds its next solve behind the last one), and one
// wavefront per point writes the list.  When the pool is too small nothing is
// written and the host runs the kernels again with a bigger pool.
__global__ void __launch_bounds__(64) trial_count_kernel(TrialArgs a) {
  const int p = blockIdx.x;
  if (p >= a.nPts) return;
  const int ln = __lane_id();
  const CurveDev& C = a.curves[a.ptCurve[p]];
  const unsigned i = (unsigned)(p - C.pointBase);
  const cx pos = traj_pos(mk(C.sx, C.sy), mk(C.ex, C.ey), i, C.lcLength);
  const cx* caus = a.caustics + C.causticBase;
  // distance to the nearest of the curve's caustic samples
  double d2 = 1e300;
  for (int q = ln; q < 6 * kCccLen; q += 64) {
    const double v = cnorm(csub(caus[q], pos));
    d2 = v < d2 ? v : d2;
  }
  for (int o = 32; o >= 1; o >>= 1) {
    const double w2 = __shfl_xor(d2, o, 64);
    d2 = w2 < d2 ? w2 : d2;
  }
  if (ln == 0) {
    a.ptPos[p] = make_double2(pos.re, pos.im);
    a.ptCausD2[p] = d2;
  }
  int n = 1;
  scan_trials(C, pos, caus, [&](unsigned long long f, const cx&) { n += __builtin_popcountll(f); });
  if (ln == 0) a.pool.count[p] = n;
}

// Exclusive prefix sum of the points' solve counts (one workgroup; every
// thread sums a contiguous share), and their total in *cursor.
constexpr int kScanThreads = 1024;
__global__ void __launch_bounds__(kScanThreads) pool_scan_kernel(SolvePool P, int nPts) {
  __shared__ int part[kScanThreads];
  const int t = threadIdx.x;
  const int per = (nPts + kScanThreads - 1) / kScanThreads;
  const int lo = t * per < nPts ? t * per : nPts, hi = lo + per < nPts ? lo + per : nPts;
  int sum = 0;
  for (int p = lo; p < hi; p++) sum += P.count[p];
  part[t] = sum;
  __syncthreads();
  for (int o = 1; o < kScanThreads; o <<= 1) {
    const int v = t >= o ? part[t - o] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int at = part[t] - sum;
  for (int p = lo; p < hi; p++) {
    P.base[p] = at;
    at += P.count[p];
  }
  if (t == kScanThreads - 1) *P.cursor = (unsigned long long)part[t];
}

__global__ void __launch_bounds__(64) trial_list_kernel(TrialArgs a) {
  const int p = blockIdx.x;
  if (p >= a.nPts || *a.pool.cursor > (unsigned long long)a.pool.cap) return;
  const int ln = __lane_id();
  const CurveDev& C = a.curves[a.ptCurve[p]];
  const double2 pp = a.ptPos[p];
  const cx pos = mk(pp.x, pp.y);
  int next = a.pool.base[p];
  if (ln == 0) {
    a.pool.zeta[next] = pos;
    a.pool.owner[next] = p;
  }
  next++;
  if (a.pool.count[p] == 1) return;
  scan_trials(C, pos, a.caustics + C.causticBase, [&](unsigned long long f, const cx& trial) {
    if ((f >> ln) & 1ull) {
      const int sid = next + __builtin_popcountll(f & ((1ull << ln) - 1ull));
      a.pool.zeta[sid] = trial;
      a.pool.owner[sid] = p;
    }
    next += __builtin_popcountll(f);
  });
}

// The image polynomial of every solve in the pool (tl_coeffs.h: the
// reference's rounding), one lane per solve.
__global__ void __launch_bounds__(64) trial_poly_kernel(TrialArgs a, int nSolves) {
  const int sid = blockIdx.x * blockDim.x + threadIdx.x;
  if (sid >= nSolves) return;
  const CurveDev& C = a.curves[a.ptCurve[a.pool.owner[sid]]];
  cx c[11];
  const cx zeta = a.pool.zeta[sid];
  image_poly(C.L, C.fixedPoly, zeta, c);
  cx* rec = reinterpret_cast<cx*>(a.pool.rec + (size_t)sid * kRecSize);
  for (int k = 0; k < 11; k++) rec[k] = c[k];
  rec[kRecZeta / 2] = zeta;
}

// The root solver for one lane per solve, every array in registers (the
// degree is a template argument).
// The deflation steps J..1 of Laguerre::solveRoots (laguerre.cc:103-167) for a
// polynomial of degree DEG: the root found at step J goes to roots[DEG - J].
template <int DEG, int J, bool LOST = false>
__device__ __forceinline__ void lane_deflate(const cx (&p)[J + 1], const cx* init, bool withInit,
                                             cx* roots, const TrigTable* trig, bool& oob) {
  cx x = withInit ? init[J] : mk(kLagEps, kLagEps);
  if constexpr (J == 1) {
    if (p[1].re != 0.0 || p[1].im != 0.0) x = cdiv(cneg(p[0]), p[1]);
    else x = withInit ? mk(kLagEps, kLagEps) : mk(999.0, 999.0);
    roots[DEG - 1] = x;
  } else {
    cx b[J + 1];
    if (!lag_lane<J, LOST>(p, x, b, trig, oob) && withInit) {
      x = mk(kLagEps, kLagEps);
      horner_sums<J>(p, x, b);
    }
    roots[DEG - J] = x;
    cx q[J];
#pragma unroll
    for (int j = 0; j < J; j++) q[j] = b[j + 1];
    lane_deflate<DEG, J - 1, LOST>(q, init, withInit, roots, trig, oob);
  }
}
// solveRoots: the deflation, then each root polished on the full polynomial
// in root order (the roots rotate through roots[0], so one copy of the
// polishing code serves all of them).
template <bool LOST = false>
__device__ __forceinline__ void lane_solve(const cx (&c)[11], const cx* init, bool withInit,
                                           cx* roots, const TrigTable* trig, bool& oob) {
  lane_deflate<10, 10, LOST>(c, init, withInit, roots, trig, oob);
#pragma unroll 1
  for (int j = 0; j < 10; j++) {
    cx x = roots[0], b[11];
    lag_lane<10, LOST>(c, x, b, trig, oob);
#pragma unroll
    for (int k = 0; k < 9; k++) roots[k] = roots[k + 1];
    roots[9] = x;
  }
}

// What a solve of the chain needs that does not depend on the chain, one lane
// per solve: the first deflation step of a chained solve (root and deflated
// polynomial) and the fresh solve (roots and image mask).
__global__ void __launch_bounds__(64) solve_prep_kernel(TrialArgs a, int nSolves) {
  const int sid = blockIdx.x * blockDim.x + threadIdx.x;
  if (sid >= nSolves) return;
  const Lens L = a.curves[a.ptCurve[a.pool.owner[sid]]].L;
  cx* rec = reinterpret_cast<cx*>(a.pool.rec + (size_t)sid * kRecSize);
  cx c[11];
#pragma unroll
  for (int k = 0; k < 11; k++) c[k] = rec[k];
  const cx zeta = rec[kRecZeta / 2];
  cx x = mk(0.0, 0.0), b[11];
  bool oob = false;
  if (!lag_lane<10, true>(c, x, b, a.trig, oob)) {
    x = mk(kLagEps, kLagEps);
    horner_sums<10>(c, x, b);
  }
#pragma unroll
  for (int k = 0; k < 10; k++) rec[kRecDefl / 2 + k] = b[k + 1];
  rec[kRecRoot / 2] = x;
  int fl = oob ? kRecOobFirst : 0;
  cx roots[10];
  oob = false;
  lane_solve<true>(c, nullptr, false, roots, a.trig, oob);
  if (oob) fl |= kRecOobFresh;
#pragma unroll
  for (int k = 0; k < 10; k++) {
    a.pool.fresh[(size_t)sid * 10 + k] = roots[k];
    if (img_check(L, roots[k], zeta, 1.0e-6)) fl |= 1 << k;
  }
  rec[kRecFlags / 2] = mk((double)fl, 0.0);
}

int launch_trials(const TrialArgs& a, hipStream_t s) {
  if (a.nPts <= 0) return 0;
  hipLaunchKernelGGL(trial_count_kernel, dim3(a.nPts), dim3(64), 0, s, a);
  hipLaunchKernelGGL(pool_scan_kernel, dim3(1), dim3(kScanThreads), 0, s, a.pool, a.nPts);
  hipLaunchKernelGGL(trial_list_kernel, dim3(a.nPts), dim3(64), 0, s, a);
  return (int)hipGetLastError();
}

int launch_solve_prep(const TrialArgs& a, int nSolves, hipStream_t s) {
  if (nSolves <= 0) return 0;
  hipLaunchKernelGGL(trial_poly_kernel, dim3((nSolves + 63) / 64), dim3(64), 0, s, a, nSolves);
  hipLaunchKernelGGL(solve_prep_kernel, dim3((nSolves + 63) / 64), dim3(64), 0, s, a, nSolves);
  return (int)hipGetLastError();
}

// image_poly for n positions of one lens, one lane each (test access to the
// device evaluation of the polynomial).
__global__ void __launch_bounds__(64) image_poly_kernel(Lens L, const cx* fixedPoly,
                                                        const cx* zeta, int n, cx* coef) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n) return;
  cx c[11];
  image_poly(L, fixedPoly, zeta[g], c);
  for (int k = 0; k < 11; k++) coef[(size_t)g * 11 + k] = c[k];
}

int launch_image_poly(const Lens& L, const cx* fixedPoly, const cx* zeta, int n, cx* coef,
                      hipStream_t s) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(image_poly_kernel, dim3((n + 63) / 64), dim3(64), 0, s, L, fixedPoly, zeta,
                     n, coef);
  return (int)hipGetLastError();
}

// Workgroup (curve c, piece q): a curve with split = 1 walks the chunk's
// positions as one chain, continuing the curve's root-reuse state.  With
// split = S > 1 the chunk's positions are cut into S contiguous pieces that
// run in parallel; piece 0 continues the chain, the others start from a
// fresh solve.  Each position's solves (centre, then caustic trial points)
// and their polynomials come from the pool, so the chain itself
// only runs the root solves, the image tests and the seed output.
template <bool TRACED>
__global__ void __launch_bounds__(64) seed_kernel(SeedArgs a) {
  __shared__ __align__(16) double rec[64];
  const int c = a.pieces ? uni(a.pieces[blockIdx.x].x) : blockIdx.x / a.maxSplit;
  const int q = a.pieces ? uni(a.pieces[blockIdx.x].y) : blockIdx.x % a.maxSplit;
  if (c >= a.nCurves) return;
  const int ln = __lane_id();
  const CurveDev& C = a.curves[c];
  if (q >= C.split) return;
  const Lens L = uni_lens(C.L);
  const bool binImg = uni(C.binImg) != 0;
  cx chainv = mk(0.0, 0.0);
  int have = 0, calls = 0;
  if (q > 0) {
    // a known start state (the verified speculative chain), else a fresh
    // solve at the piece's first position
    if (a.pieceStart) {
      if (ln < 10) chainv = a.pieceStart[((size_t)a.pieceBase[c] + q) * 10 + ln];
      have = 1;
    }
  } else if (a.chainIn) {
    if (ln <= 10) chainv = a.chainIn[c].tempRoots[ln <= 10 ? ln : 0];
    have = a.chainIn[c].have;
    calls = a.chainIn[c].calls;
  } else {
    if (ln <= 10) chainv = C.chain[ln <= 10 ? ln : 0];
    have = C.chainHave;
    calls = C.chainCalls;
  }
  const bool traced = TRACED && q == 0 && C.slotCount > 0;
  const long long n = (long long)C.lcLength + 1;
  const long long cBegin = n * a.chunk / a.nChunks, cEnd = n * (a.chunk + 1) / a.nChunks;
  const unsigned iBegin = (unsigned)(cBegin + (cEnd - cBegin) * q / C.split);
  const unsigned iEnd = (unsigned)(cBegin + (cEnd - cBegin) * (q + 1) / C.split);
  if (iBegin < iEnd) {
  SolveWalk W(a.pool, C.pointBase + (int)iBegin, C.pointBase + (int)iEnd);
  for (unsigned i = iBegin; i < iEnd; i++) {
    const int p = C.pointBase + (int)i;
    const int nSolve = W.position();
    int cnt = 0;
    uint32_t fl = 0;
    int2* out = a.seeds + (size_t)p * kMaxSeeds;
    double amp = 0.0;
    for (int sIdx = 0; sIdx < nSolve; sIdx++) {
      double rv;
      cx fv;
      W.next(rv, fv);
      const bool slot = traced && have && calls < C.slotCount;
      if (slot && ln == 10) chainv = a.slotTrace[C.slotBase + calls];
      calls++;
      bool oob = false;
      const unsigned long long m =
          wl_get_images<TRACED>(L, rv, fv, rec, slot, chainv, have, a.trig, binImg, oob);
      if (oob) fl |= kFlagKickTable;
      emit_seeds(C, chainv, m, out, cnt, fl);
      if (sIdx == 0) {
        // point-source magnification (getPointAmp, lcbase.cc:17-38) and the
        // magnification-weighted image centroid, summed in root order
        const double term = ((m >> ln) & 1ull) ? point_amp_term(L, chainv) : 0.0;
        const double wx = term * chainv.re, wy = term * chainv.im;
        double sx = 0.0, sy = 0.0;
        unsigned long long mm = m;
        while (mm) {
          const int k = __builtin_ctzll(mm);
          mm &= mm - 1;
          amp += rl(term, k);
          sx += rl(wx, k);
          sy += rl(wy, k);
        }
        // the two largest image magnifications
        double t1 = term;
        for (int o = 32; o >= 1; o >>= 1) {
          const double w2 = __shfl_xor(t1, o, 64);
          t1 = w2 > t1 ? w2 : t1;
        }
        const unsigned long long top = __ballot(term == t1 && ((m >> ln) & 1ull));
        const int topLane = top ? __builtin_ctzll(top) : -1;
        double t2 = (ln == topLane) ? 0.0 : term;
        for (int o = 32; o >= 1; o >>= 1) {
          const double w2 = __shfl_xor(t2, o, 64);
          t2 = w2 > t2 ? w2 : t2;
        }
        if (ln < 10) a.ptRoots[(size_t)p * 10 + ln] = chainv;
        if (ln == 0) {
          a.ptAmp[p] = amp;
          a.ptCen[p] = make_double2(sx / amp, sy / amp);
          const double dist = sqrt(a.ptCausD2[p]);
          // inside a caustic: more images than the 4 (binary: 3) outside
          a.ptCaus[p] = __builtin_popcountll(m) > (binImg ? 3 : 4) ? -dist : dist;
          a.ptPair[p] = amp > 0.0 ? (t1 + t2) / amp : 0.0;
        }
      }
    }
    if (ln == 0) {
      a.nSeeds[p] = cnt;
      a.flags[p] = fl;
      a.cost[p] = (float)(amp * 3.141592653589793 * C.ppr * C.ppr);
    }
  }
  }
  if (q == C.split - 1) {
    if (ln <= 10) a.chainOut[c].tempRoots[ln] = chainv;
    if (ln == 0) {
      a.chainOut[c].have = have;
      a.chainOut[c].calls = calls;
    }
  }
}

// ---- verified speculative chain (SpecArgs) ---------------------------------
// The chain's solves of the walk's next position (centre, then caustic trial
// points), as seed_kernel runs them, without output.  Returns their number.
__device__ __forceinline__ int chain_step(const Lens& L, bool binImg, const TrigTable* trig,
                                          SolveWalk& W, double* rec, cx& chainv, int& have) {
  const int nSolve = W.position();
  for (int sIdx = 0; sIdx < nSolve; sIdx++) {
    double rv;
    cx fv;
    W.next(rv, fv);
    bool oob = false;
    wl_get_images<false>(L, rv, fv, rec, false, chainv, have, trig, binImg, oob);
  }
  return nSolve;
}

// The chain state (roots 0..9 on lanes 0..9) equals the stored one, bit for bit.
__device__ __forceinline__ bool state_equal(const cx& chainv, const cx& st) {
  const bool eq = __double_as_longlong(st.re) == __double_as_longlong(chainv.re) &&
                  __double_as_longlong(st.im) == __double_as_longlong(chainv.im);
  return __ballot(!eq && __lane_id() < 10) == 0;
}

__device__ __forceinline__ void piece_range(const CurveDev& C, int q, int& b, int& e) {
  const long long n = (long long)C.lcLength + 1;
  b = (int)(n * q / C.split);
  e = (int)(n * (q + 1) / C.split);
}

// Round 1: piece q from a fresh solve (piece 0 from the curve's chain state),
// on into the next piece for sp.overlap positions.
__global__ void __launch_bounds__(64) spec_round1_kernel(SeedArgs a, SpecArgs sp) {
  __shared__ __align__(16) double rec[64];
  const int c = blockIdx.x / a.maxSplit, q = blockIdx.x % a.maxSplit;
  if (c >= a.nCurves) return;
  const int ln = __lane_id();
  const CurveDev& C = a.curves[c];
  if (q >= C.split) return;
  const Lens L = uni_lens(C.L);
  const bool binImg = uni(C.binImg) != 0;
  const int pointBase = uni(C.pointBase);
  cx chainv = mk(0.0, 0.0);
  int have = 0;
  if (q == 0) {
    if (ln <= 10) chainv = C.chain[ln <= 10 ? ln : 0];
    have = C.chainHave;
  }
  int b, e;
  piece_range(C, q, b, e);
  int stop = e;
  if (q + 1 < C.split) {
    int b2, e2;
    piece_range(C, q + 1, b2, e2);
    stop = e + sp.overlap < e2 ? e + sp.overlap : e2;
  }
  if (b >= stop) return;
  SolveWalk W(a.pool, C.pointBase + b, C.pointBase + stop);
  for (int i = b; i < stop; i++) {
    const int p = pointBase + i;
    chain_step(L, binImg, a.trig, W, rec, chainv, have);
    cx* dst = (i < e ? sp.own : sp.ext) + (size_t)p * 10;
    if (ln < 10) dst[ln] = chainv;
  }
}

// Whether piece q > 0 agrees with its predecessor's continuation; if not, its
// repair chain stands where that continuation ended.
__global__ void __launch_bounds__(64) spec_agree_kernel(SeedArgs a, SpecArgs sp) {
  const int c = blockIdx.x / a.maxSplit, q = blockIdx.x % a.maxSplit;
  if (c >= a.nCurves) return;
  const int ln = __lane_id();
  const CurveDev& C = a.curves[c];
  if (q == 0 || q >= C.split) return;
  const int gq = sp.pieceBase[c] + q;
  int b, e;
  piece_range(C, q, b, e);
  const int lim = e < b + sp.overlap ? e : b + sp.overlap;
  const int pointBase = uni(C.pointBase);
  // six positions at a time, one root to a lane
  bool agree = false;
  const int r = ln % 10, k = ln / 10;
  for (int i = b; i < lim && !agree; i += 6) {
    bool eq = false;
    if (k < 6 && i + k < lim) {
      const size_t at = ((size_t)pointBase + i + k) * 10 + r;
      const cx v = sp.ext[at], o = sp.own[at];
      eq = __double_as_longlong(v.re) == __double_as_longlong(o.re) &&
           __double_as_longlong(v.im) == __double_as_longlong(o.im);
    }
    const unsigned long long m = __ballot(eq);
    for (int j = 0; j < 6; j++) agree |= ((m >> (10 * j)) & 0x3ffull) == 0x3ffull;
  }
  if (!agree && ln < 10)
    sp.repChain[(size_t)gq * 10 + ln] = sp.ext[((size_t)pointBase + lim - 1) * 10 + ln];
  if (ln == 0) {
    sp.merged[gq] = agree ? 1 : 0;
    sp.repTarget[gq] = kRepairRunning;
    sp.repPos[gq] = make_int2(lim, q);
  }
}

// One segment of the active repair chains, one wavefront each.  A chain is
// serial (its measure is the time per solve, about 20 us), so few wavefronts
// run here for long: they are packed one to a SIMD, four to a workgroup, so
// that they hold few compute units and the fill of the positions already
// known has the others.  With the fill waiting for the last chain instead,
// a 4096-point curve through a central caustic took 55 ms (repair 25, fill
// 23) and the 64-curve batch 241 ms (130, 87).
__global__ void __launch_bounds__(64 * kWalkWaves) spec_walk_kernel(SeedArgs a, SpecArgs sp,
                                                                    int segment) {
  __shared__ __align__(16) double recs[kWalkWaves][64];
  const int ln = __lane_id(), wave = uni((int)threadIdx.x >> 6);
  double* rec = recs[wave];
  const int nActive = uni(sp.info[1 + ((segment - 1) & 1)]);
  for (int w = blockIdx.x * kWalkWaves + wave; w < nActive; w += gridDim.x * kWalkWaves) {
    const int c = uni(sp.active[w].x), q = uni(sp.active[w].y);
    const CurveDev& C = a.curves[c];
    const int gq = uni(sp.pieceBase[c]) + q;
    const int pointBase = uni(C.pointBase), n = uni((int)C.lcLength) + 1, split = uni(C.split);
    const Lens L = uni_lens(C.L);
    const bool binImg = uni(C.binImg) != 0;
    int i = uni(sp.repPos[gq].x), qq = uni(sp.repPos[gq].y);  // qq: the piece the chain is in
    int qe = (int)((long long)n * (qq + 1) / split);
    cx chainv = mk(0.0, 0.0);
    if (ln < 10) chainv = sp.repChain[(size_t)gq * 10 + ln];
    int have = 1, target = kRepairRunning;
    if (i < n) {
      SolveWalk W(a.pool, pointBase + i, pointBase + n);
      int solves = 0;
      for (; i < n && solves < sp.budget; i++) {
        if (i == qe) {
          // entering piece qq + 1: the chain's state before its first position
          const int j = qq - q;
          if (j >= sp.depth) {
            target = kRepairDepth;
            break;
          }
          qq++;
          qe = (int)((long long)n * (qq + 1) / split);
          if (ln < 10) sp.repState[((size_t)gq * sp.depth + j) * 10 + ln] = chainv;
        }
        // the piece's own state, loaded before the solve that it is compared with
        cx own = mk(0.0, 0.0);
        if (ln < 10) own = sp.own[((size_t)pointBase + i) * 10 + ln];
        solves += chain_step(L, binImg, a.trig, W, rec, chainv, have);
        if (state_equal(chainv, own)) {
          target = qq;
          break;
        }
      }
    }
    if (target == kRepairRunning && i >= n) target = kRepairEnd;
    if (ln < 10) sp.repChain[(size_t)gq * 10 + ln] = chainv;
    if (ln == 0) {
      sp.repTarget[gq] = target;
      sp.repPos[gq] = make_int2(i, qq);
    }
  }
}

// The true chain's state before each piece, walking every curve's pieces in
// order from the first whose start is not known (one wavefront per curve, 64
// pieces' records at a time): the true chain at a piece start is either the
// previous piece's own (it agreed with the chain before it, or it is piece 0)
// or a repair chain that has not yet agreed.  Then the repair chains of the
// coming segment: the one the true chain waits for, and those beyond it that
// no other chain in question has run past.
__global__ void __launch_bounds__(64) spec_resolve_kernel(SeedArgs a, SpecArgs sp, int segment) {
  const int c = blockIdx.x;
  if (c >= a.nCurves) return;
  const int ln = __lane_id();
  if (c == 0 && ln == 0) sp.info[1 + ((segment + 1) & 1)] = 0;
  const CurveDev& C = a.curves[c];
  const int split = uni(C.split), g0 = uni(sp.pieceBase[c]);
  const long long n = (long long)uni((int)C.lcLength) + 1;
  const cx* own = sp.own + (size_t)uni(C.pointBase) * 10;
  int q = uni(sp.info[kSpecInfo + c]);
  if (q >= split) return;
  bool viaPiece = uni(sp.front[c].x) != 0;
  int rq = uni(sp.front[c].y);
  int rTarget = viaPiece ? 0 : uni(sp.repTarget[g0 + rq]);
  int rPiece = viaPiece ? 0 : uni(sp.repPos[g0 + rq].y);
  // it may have agreed with the piece it was in at the last resolution
  if (!viaPiece && rTarget == q - 1) viaPiece = true;
  bool failed = false;
  int q0 = q, m = 0, t = 0, rp = 0;  // lane l: the records of piece q0 + l
  auto load = [&]() {
    const int g = g0 + (q0 + ln < split ? q0 + ln : split - 1);
    m = sp.merged[g];
    t = sp.repTarget[g];
    rp = sp.repPos[g].y;
  };
  load();
  for (; q < split; q++) {
    if (q == q0 + 64) {
      q0 = q;
      load();
    }
    const cx* src;
    if (viaPiece) {
      src = own + (n * q / split - 1) * 10;
      if (!__builtin_amdgcn_readlane(m, q - q0)) {
        viaPiece = false;
        rq = q;
        rTarget = __builtin_amdgcn_readlane(t, q - q0);
        rPiece = __builtin_amdgcn_readlane(rp, q - q0);
      }
    } else {
      if (rPiece < q) {
        // the repair chain has not come here: it is running, or gave up
        failed = rTarget != kRepairRunning;
        break;
      }
      src = sp.repState + ((size_t)(g0 + rq) * sp.depth + (q - rq - 1)) * 10;
    }
    if (rTarget == q) viaPiece = true;
    if (ln < 10) sp.start[((size_t)g0 + q) * 10 + ln] = src[ln];
  }
  if (ln == 0) {
    if (failed) sp.info[0] = 1;
    sp.info[kSpecInfo + c] = q;
    sp.front[c] = make_int2(viaPiece ? 1 : 0, rq);
  }
  if (q >= split || failed) return;
  int seen = -1;  // the furthest piece that a chain in question has entered
  for (int p0 = rq; p0 < split; p0 += 64) {
    const int p = p0 + ln;
    const bool there = p < split && (p == rq || p >= q) && !sp.merged[g0 + p];
    int reach = there ? sp.repPos[g0 + p].y : -1;
    const bool running = there && sp.repTarget[g0 + p] == kRepairRunning;
    // the furthest of the lanes below
    int upto = reach;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o, 64);
      if (ln >= o && v > upto) upto = v;
    }
    int before = __shfl_up(upto, 1, 64);
    if (ln == 0 || before < seen) before = seen;
    const bool on = running && (p == rq || before < p);
    const unsigned long long f = __ballot(on);
    int at = 0;
    if (ln == 0 && f) at = atomicAdd(&sp.info[1 + (segment & 1)], __builtin_popcountll(f));
    at = uni(at);
    if (on) sp.active[at + __builtin_popcountll(f & ((1ull << ln) - 1ull))] = make_int2(c, p);
    const int top = __builtin_amdgcn_readlane(upto, 63);
    if (top > seen) seen = top;
  }
}

static bool spec_args_ok(const SeedArgs& a, const SpecArgs& sp) {
  return a.maxSplit >= 1 && (long long)a.nCurves * a.maxSplit <= (1ll << 30) && sp.pieceBase &&
         sp.own && sp.ext && sp.merged && sp.repState && sp.repTarget && sp.repChain &&
         sp.repPos && sp.start && sp.active && sp.front && sp.info && sp.overlap >= 1 &&
         sp.depth >= 1 && sp.budget >= 1 && a.curves && a.trig && a.pool.base && a.pool.count &&
         a.pool.rec && a.pool.fresh;
}

int launch_spec(const SeedArgs& a, const SpecArgs& sp, hipStream_t s) {
  if (a.nCurves <= 0) return 0;
  if (!spec_args_ok(a, sp)) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(spec_round1_kernel, dim3(a.nCurves * a.maxSplit), dim3(64), 0, s, a, sp);
  hipLaunchKernelGGL(spec_agree_kernel, dim3(a.nCurves * a.maxSplit), dim3(64), 0, s, a, sp);
  hipLaunchKernelGGL(spec_resolve_kernel, dim3(a.nCurves), dim3(64), 0, s, a, sp, 0);
  return (int)hipGetLastError();
}

int launch_spec_segment(const SeedArgs& a, const SpecArgs& sp, int segment, int groups,
                        hipStream_t s) {
  if (a.nCurves <= 0) return 0;
  if (!spec_args_ok(a, sp) || segment < 1 || groups < 1) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(spec_walk_kernel, dim3(groups), dim3(64 * kWalkWaves), 0, s, a, sp, segment);
  hipLaunchKernelGGL(spec_resolve_kernel, dim3(a.nCurves), dim3(64), 0, s, a, sp, segment);
  return (int)hipGetLastError();
}

// LightCurveBase::getLC / getPointAmp (lcbase.cc:17-52): positions at
// t = i/(lcLength-1), magnification sum over images (in root order) of
// 1/|1 - |sum m/(z-z_k)^2|^2| (the squares as products; the reference uses
// std::pow(z, 2.0)).  One wavefront per curve, as the seed search.
// The point-source curve's positions as a pool of one solve each.
__global__ void point_list_kernel(TrialArgs a) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= a.nPts) return;
  const CurveDev& C = a.curves[a.ptCurve[p]];
  const int i = p - C.pointBase;
  const cx s = mk(C.sx, C.sy), e = mk(C.ex, C.ey);
  a.pool.zeta[p] = cadd(s, cscale(csub(e, s), i / (C.lcLength - 1.0)));
  a.pool.owner[p] = p;
  a.pool.base[p] = p;
  a.pool.count[p] = 1;
}

__global__ void __launch_bounds__(64) point_lc_kernel(const CurveDev* curves, int nCurves,
                                                      const TrigTable* trig, double* out,
                                                      RootChain* chainOut, SolvePool pool) {
  __shared__ __align__(16) double rec[64];
  const int c = blockIdx.x;
  if (c >= nCurves) return;
  const int ln = __lane_id();
  const CurveDev& C = curves[c];
  const Lens L = uni_lens(C.L);
  const bool binImg = uni(C.binImg) != 0;
  const int pointBase = uni(C.pointBase), len = uni((int)C.lcLength);
  cx chainv = ln <= 10 ? C.chain[ln <= 10 ? ln : 0] : mk(0.0, 0.0);
  int have = C.chainHave;
  SolveWalk W(pool, pointBase, pointBase + len);
  for (int i = 0; i < len; i++) {
    double rv;
    cx fv;
    W.next(rv, fv);
    bool oob = false;
    unsigned long long m = wl_get_images<false>(L, rv, fv, rec, false, chainv, have, trig, binImg, oob);
    const double term = ((m >> ln) & 1ull) ? point_amp_term(L, chainv) : 0.0;
    double amp = 0.0;
    while (m) {
      const int k = __builtin_ctzll(m);
      m &= m - 1;
      amp += rl(term, k);
    }
    if (ln == 0) out[pointBase + i] = amp;
  }
  if (ln <= 10) chainOut[c].tempRoots[ln] = chainv;
  if (ln == 0) {
    chainOut[c].have = have;
    chainOut[c].calls = C.chainCalls + (int)C.lcLength;
  }
}

int launch_point_lc(const TrialArgs& a, int nCurves, double* out, RootChain* chainOut,
                    hipStream_t s) {
  if (nCurves <= 0 || a.nPts <= 0) return 0;
  hipLaunchKernelGGL(point_list_kernel, dim3((a.nPts + 255) / 256), dim3(256), 0, s, a);
  const int rc = launch_solve_prep(a, a.nPts, s);
  if (rc) return rc;
  hipLaunchKernelGGL(point_lc_kernel, dim3(nCurves), dim3(64), 0, s, a.curves, nCurves, a.trig,
                     out, chainOut, a.pool);
  return (int)hipGetLastError();
}

// Offsets, in source radii, of the disk samples of Gould's (2008, ApJ 681,
// 1593) hexadecapole approximation: radius 1/2 on the axes, radius 1 on the
// axes, radius 1 on the diagonals.
constexpr double kSignificant = 1.0e-4;

__constant__ double kRingOff[kRingSamples][2] = {
    {0.5, 0.0}, {0.0, 0.5}, {-0.5, 0.0}, {0.0, -0.5},
    {1.0, 0.0}, {0.0, 1.0}, {-1.0, 0.0}, {0.0, -1.0},
    {0.70710678118654752, 0.70710678118654752}, {-0.70710678118654752, 0.70710678118654752},
    {-0.70710678118654752, -0.70710678118654752}, {0.70710678118654752, -0.70710678118654752}};

// Point magnification (getPointAmp's sum, lcbase.cc:17-38) at the disk
// samples around each position, one wavefront per position.  Every sample
// is solved from the position's own centre roots (the reference's
// root-reuse solve, imgpoint.cc:160-274), so the samples are independent of
// each other and of the order they are visited in.  A sample whose count of
// significant images (each carrying at least kSignificant of the point's
// magnification) differs from the centre's lies across a caustic from it;
// the threshold keeps out the faint images next to a lens whose lens-equation
// residual sits at the acceptance threshold and that come and go between
// nearby points, while an image pair born on a fold is always bright.
// The image polynomial at every disk sample (one lane per sample) for
// ring_lane_kernel: coef[((p * kRingSamples) + s) * 11 + k].
__global__ void __launch_bounds__(64) ring_poly_kernel(const CurveDev* curves, const int* ptCurve,
                                                       const double2* ptPos, int nPts, cx* coef,
                                                       int* cross) {
  const long long g = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (g >= (long long)nPts * kRingSamples) return;
  const int p = (int)(g / kRingSamples), smp = (int)(g % kRingSamples);
  const CurveDev& C = curves[ptCurve[p]];
  if (!C.ring) return;
  const double2 pp = ptPos[p];
  const cx zeta = mk(pp.x + C.rho * kRingOff[smp][0], pp.y + C.rho * kRingOff[smp][1]);
  cx cf[11];
  image_poly(C.L, C.fixedPoly, zeta, cf);
  for (int k = 0; k < 11; k++) coef[(size_t)g * 11 + k] = cf[k];
  if (smp == 0) cross[p] = 0;
}

// lag_check (laguerre.cc:188-198)
template <int DEG>
__device__ __forceinline__ bool lag_check_reg(const cx* coeffs, const cx* roots) {
  cx c0 = coeffs[DEG];
#pragma unroll
  for (int j = 0; j < DEG; j++) c0 = cmul(c0, cneg(roots[j]));
  if (cabs_(coeffs[0]) > 1.0e-8) return (1.0 - cabs_(cdiv(c0, coeffs[0]))) < 1.0e-5;
  return cabs_(csub(c0, coeffs[0])) < 1.0e-10;
}

// Point magnification and significant-image count of the roots marked in
// `mask`, in root order (tlo_ring_amp's significant_images and point_amp):
// sig counts the images carrying at least kSignificant of the sum.
__device__ __forceinline__ double lane_amp(const Lens& L, const cx* roots, unsigned mask,
                                           int& sig) {
  double t[10], amp = 0.0;
#pragma unroll
  for (int k = 0; k < 10; k++) {
    t[k] = 0.0;
    if ((mask >> k) & 1u) {
      t[k] = point_amp_term(L, roots[k]);
      amp += t[k];
    }
  }
  sig = 0;
#pragma unroll
  for (int k = 0; k < 10; k++) sig += ((mask >> k) & 1u) && t[k] >= kSignificant * amp ? 1 : 0;
  return amp;
}

// getRootsPrecalculated + getImages (imgpoint.cc:160-274) on one lane, from
// the root-reuse state chain[0..10] (chain[10] is the slot read past the end:
// 0): the sequence wl_get_images runs on a wavefront, with the Laguerre
// routines above (the same values).  Leaves the roots in chain[0..9] and
// returns the mask of the accepted images among them.
__device__ __forceinline__ unsigned lane_images(const Lens& L, const cx (&cf)[11], cx* chain,
                                                cx zeta, const TrigTable* trig, bool binImg) {
  bool withInit = true, second = false;
  while (true) {
    cx roots[10];
    bool oob = false;
    lane_solve(cf, chain, withInit, roots, trig, oob);
    if (withInit && !lag_check_reg<10>(cf, roots)) {
      withInit = false;
      continue;
    }
#pragma unroll
    for (int k = 0; k < 10; k++) chain[k] = roots[k];
    chain[10] = mk(0.0, 0.0);
    unsigned mask = 0;
    int n = 0;
#pragma unroll
    for (int k = 0; k < 10; k++)
      if (img_check(L, roots[k], zeta, 1.0e-6)) {
        mask |= 1u << k;
        n++;
      }
    // a valid count: even and at least 4, or for the binary lens odd and at
    // least 3 (imgpoint.cc:236-237)
    const bool bad = binImg ? (n % 2 != 1 || n < 3) : (n % 2 != 0 || n < 4);
    if (!bad || second || !withInit) return mask;
    second = true;
    withInit = false;
  }
}

// One lane per disk sample (position g / kRingSamples, sample g %
// kRingSamples): the sample's images by a root-reuse solve from the
// position's own centre roots, its point magnification (root order), and
// whether its count of significant images differs from the centre's
// (cross[p], cleared by ring_poly_kernel, counts those samples).
__global__ void __launch_bounds__(64) ring_lane_kernel(const CurveDev* curves, const int* ptCurve,
                                                       const double2* ptPos, const cx* ptRoots,
                                                       int nPts, const TrigTable* trig,
                                                       double* ring, int* cross, const cx* coef) {
  const long long g = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (g >= (long long)nPts * kRingSamples) return;
  const int p = (int)(g / kRingSamples), smp = (int)(g % kRingSamples);
  const CurveDev& C = curves[ptCurve[p]];
  if (!C.ring) return;
  const Lens L = C.L;
  const double2 pp = ptPos[p];
  cx chain[11];
  unsigned mask0 = 0;
#pragma unroll
  for (int k = 0; k < 10; k++) {
    chain[k] = ptRoots[(size_t)p * 10 + k];
    if (img_check(L, chain[k], mk(pp.x, pp.y), 1.0e-6)) mask0 |= 1u << k;
  }
  chain[10] = mk(0.0, 0.0);
  int sig0 = 0;
  lane_amp(L, chain, mask0, sig0);
  cx cf[11];
#pragma unroll
  for (int k = 0; k < 11; k++) cf[k] = coef[(size_t)g * 11 + k];
  const cx zeta = mk(pp.x + C.rho * kRingOff[smp][0], pp.y + C.rho * kRingOff[smp][1]);
  const unsigned mask = lane_images(L, cf, chain, zeta, trig, C.binImg);
  int sig = 0;
  ring[g] = lane_amp(L, chain, mask, sig);
  if (sig != sig0) atomicAdd(&cross[p], 1);
}

int launch_ring_amp(const CurveDev* curves, const int* ptCurve, const double2* ptPos,
                    const cx* ptRoots, int nPts, const TrigTable* trig, double* ring, int* cross,
                    cx* coef, hipStream_t s) {
  if (nPts <= 0) return 0;
  const long long lanes = (long long)nPts * kRingSamples;
  hipLaunchKernelGGL(ring_poly_kernel, dim3((unsigned)((lanes + 63) / 64)), dim3(64), 0, s, curves,
                     ptCurve, ptPos, nPts, coef, cross);
  hipLaunchKernelGGL(ring_lane_kernel, dim3((unsigned)((lanes + 63) / 64)), dim3(64), 0, s, curves,
                     ptCurve, ptPos, ptRoots, nPts, trig, ring, cross, coef);
  return (int)hipGetLastError();
}

__global__ void clear_flag_bits_kernel(uint32_t* flags, const int* pts, int n, uint32_t bits) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flags[pts[i]] &= ~bits;
}

int launch_clear_flag_bits(uint32_t* flags, const int* pts, int n, uint32_t bits, hipStream_t s) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(clear_flag_bits_kernel, dim3((n + 255) / 256), dim3(256), 0, s, flags, pts, n,
                     bits);
  return (int)hipGetLastError();
}

// Critical curves of many geometries: critical_curves_into with the host's
// step table, every value the host's, and the reference's, to the bit.  The
// 500 steps are a chain (each polishes the last one's roots), but the six
// roots of a step are independent: eight lanes hold a geometry, lane r < 6
// its root r.  A wavefront holds perWave geometries (1 while the launch then
// has at most one wavefront per SIMD, up to 8 beyond).  One lane per geometry
// with the unbracketed iteration took 40 ms for any number of geometries up
// to a few thousand; the chain is bound by its instruction count.
template <int CTRL>
__device__ __forceinline__ cx dpp_times(const cx& v) {
  auto mv = [](double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                            (unsigned)lo));
  };
  return cmul(v, mk(mv(v.re), mv(v.im)));
}

__global__ void __launch_bounds__(64) ccc_kernel(const Lens* lenses, int n, int perWave,
                                                 const CccTable* tab, const TrigTable* trig,
                                                 cx* cc) {
  const int ln = __lane_id(), r = ln & 7;
  const int slot = ln >> 3;
  // lanes without a geometry of their own repeat the wavefront's last one
  const int first = blockIdx.x * perWave;
  int g = first + (slot < perWave ? slot : perWave - 1);
  if (g >= n) g = n - 1;
  const Lens L = lenses[g];
  const bool mine = r < 6 && slot < perWave && first + slot < n;
  const CccPoly st = ccc_poly_static(L);
  cx* out = cc + (size_t)g * 6 * kCccSteps + (size_t)(r < 6 ? r : 0) * kCccSteps;
  cx x = mk(0.0, 0.0);
  bool oob = false;
  for (int j = 0; j < kCccSteps; j++) {
    cx p[7], b[7];
    ccc_poly(L, st, tab->e[j], p);
    bool fresh = j == 0;
    if (!fresh) {
      lag_lane<6>(p, x, b, trig, oob);
      // Laguerre::checkRoots (laguerre.cc:188-198): the product of the roots,
      // taken in any order where it decides (see wl_check), else in root order
      cx v = r < 6 ? x : mk(1.0, 0.0);
      v = dpp_times<0xB1>(v);   // lanes 1, 0, 3, 2
      v = dpp_times<0x4E>(v);   // lanes 2, 3, 0, 1
      v = dpp_times<0x141>(v);  // lanes 7 .. 0
      const double A = cnorm(cmul(p[6], v));
      const double T = cnorm(p[0]) * ((1.0 - 1.0e-5) * (1.0 - 1.0e-5));
      const bool big = T > 1.0001e-16 && A < 1e300;
      const bool yes = big && A > T * (1.0 + 1e-9), no = big && A < T * (1.0 - 1e-9);
      fresh = no;
      if (__ballot(!yes && !no)) {
        cx roots[6];
#pragma unroll
        for (int k = 0; k < 6; k++)
          roots[k] = mk(__shfl(x.re, (ln & ~7) + k, 64), __shfl(x.im, (ln & ~7) + k, 64));
        if (!yes && !no) fresh = !lag_check_reg<6>(p, roots);
      }
    }
    if (__ballot(fresh)) {
      cx roots[6];
      lane_deflate<6, 6>(p, nullptr, false, roots, trig, oob);
      cx y = roots[0];
#pragma unroll
      for (int k = 1; k < 6; k++)
        if (r == k) y = roots[k];
      lag_lane<6>(p, y, b, trig, oob);
      if (fresh) x = y;
    }
    if (mine) out[j] = x;
  }
}

__global__ void caustic_kernel(const Lens* lenses, int n, const cx* cc, cx* ca) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  const size_t per = 6 * kCccSteps;
  if (i < (size_t)n * per) ca[i] = caustic_point(lenses[i / per], cc[i]);
}

int launch_ccc(const Lens* lenses, int n, const CccTable* tab, const TrigTable* trig, cx* cc,
               cx* ca, hipStream_t s) {
  if (n <= 0) return 0;
  int perWave = (n + 1023) / 1024;
  if (perWave > 8) perWave = 8;
  hipLaunchKernelGGL(ccc_kernel, dim3((n + perWave - 1) / perWave), dim3(64), 0, s, lenses, n,
                     perWave, tab, trig, cc);
  const size_t all = (size_t)n * 6 * kCccSteps;
  hipLaunchKernelGGL(caustic_kernel, dim3((unsigned)((all + 255) / 256)), dim3(256), 0, s, lenses,
                     n, cc, ca);
  return (int)hipGetLastError();
}

int launch_seed(const SeedArgs& a, hipStream_t s) {
  if (a.nCurves <= 0) return 0;
  if (a.maxSplit < 1 || (long long)a.nCurves * a.maxSplit > (1ll << 30))
    return (int)hipErrorInvalidValue;
  if (a.pieceStart && !a.pieceBase) return (int)hipErrorInvalidValue;
  const int groups = a.pieces ? a.nPieces : a.nCurves * a.maxSplit;
  if (groups <= 0) return 0;
  if (a.slotTrace)
    hipLaunchKernelGGL(seed_kernel<true>, dim3(groups), dim3(64), 0, s, a);
  else
    hipLaunchKernelGGL(seed_kernel<false>, dim3(groups), dim3(64), 0, s, a);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// Run table: open addressing over 16-byte entries, one slice per group of
// kGroupPoints batch points (group b >> 14).
//   word0 = (row+1) << 39 | xL << 14 | (b & 0x3FFF)   (0 = empty)
//   word1 = label << 32 | xR                        (~0 = not yet written)
// Rows and columns are those of the grid (0 <= row, xL < 2^25 - 1; scans
// never leave the columns [0, N-1]).  A maximal run is identified by (b,
// row, xL): two floods that reach the same run compute the same (xL, xR),
// and the compare-and-swap on word0 lets exactly one of them record it.
// ---------------------------------------------------------------------------
constexpr unsigned long long kEmpty1 = ~0ull;

__device__ __forceinline__ unsigned long long run_key(int b, int row, int xl) {
  return ((unsigned long long)(row + 1) << 39) | ((unsigned long long)(unsigned)xl << 14) |
         (unsigned long long)(b & (kGroupPoints - 1));
}
// Start of a run's probe sequence in its slice: 32-bit multiplicative mixing
// of the key's halves (scalar instructions; the runs of an image differ in
// row and column by small steps, which the two multipliers spread).
__device__ __forceinline__ unsigned hash_run(unsigned long long key) {
  unsigned h = (unsigned)key * 0x9E3779B1u + (unsigned)(key >> 32) * 0x85EBCA77u;
  h ^= h >> 15;
  h *= 0xC2B2AE3Du;
  return h ^ (h >> 13);
}

// A wave-uniform value the compiler knows nothing about.  What a task's rare
// cases need is derived from such copies where they arise: the compiler would
// otherwise compute all of it ahead of the row loop, for every task, and spill
// it.
__device__ __forceinline__ int opq(int x) {
  x = uni(x);
  asm volatile("" : "+s"(x));
  return x;
}
// The launch's arguments, read where they are used (scalar loads from the
// kernel's argument segment) instead of being held in registers: FillArgs is
// the fill kernel's only argument.
typedef const __attribute__((address_space(4))) FillArgs* ArgPtr;
__device__ __forceinline__ ArgPtr opq(ArgPtr a) {
  asm volatile("" : "+s"(a));
  return a;
}

// ---- single-lane memory operations of a wavefront ---------------------------
// A worker's shared-state updates are made by lane 0 alone, with the
// execution mask set around the instruction instead of a branch on the lane
// number: a divergent branch inside the task loop makes the compiler turn
// the loop's uniform branches into masked flow.  Each returning operation
// waits for its result in the same block.
__device__ __forceinline__ unsigned long long cas64_lane0(unsigned long long* p,
                                                          unsigned long long expected,
                                                          unsigned long long desired) {
  typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
  const u64x2 d = {desired, expected};
  unsigned long long old, save;
  asm volatile(
      "s_mov_b64 %1, exec\n\t"
      "s_mov_b64 exec, 1\n\t"
      "global_atomic_cmpswap_x2 %0, %2, %3, off sc0\n\t"
      "s_waitcnt vmcnt(0)\n\t"
      "s_mov_b64 exec, %1"
      : "=&v"(old), "=&s"(save)
      : "v"(p), "v"(d)
      : "memory");
  return (unsigned long long)uni64((long long)old);
}
__device__ __forceinline__ int cas32_lane0(int* p, int expected, int desired) {
  typedef int i32x2 __attribute__((ext_vector_type(2)));
  const i32x2 d = {desired, expected};
  int old;
  unsigned long long save;
  asm volatile(
      "s_mov_b64 %1, exec\n\t"
      "s_mov_b64 exec, 1\n\t"
      "global_atomic_cmpswap %0, %2, %3, off sc0\n\t"
      "s_waitcnt vmcnt(0)\n\t"
      "s_mov_b64 exec, %1"
      : "=&v"(old), "=&s"(save)
      : "v"(p), "v"(d)
      : "memory");
  return uni(old);
}
__device__ __forceinline__ int add32_lane0(int* p, int v) {
  int old;
  unsigned long long save;
  asm volatile(
      "s_mov_b64 %1, exec\n\t"
      "s_mov_b64 exec, 1\n\t"
      "global_atomic_add %0, %2, %3, off sc0\n\t"
      "s_waitcnt vmcnt(0)\n\t"
      "s_mov_b64 exec, %1"
      : "=&v"(old), "=&s"(save)
      : "v"(p), "v"(v)
      : "memory");
  return uni(old);
}
__device__ __forceinline__ void add64_lane0(unsigned long long* p, unsigned long long v) {
  unsigned long long save;
  asm volatile(
      "s_mov_b64 %0, exec\n\t"
      "s_mov_b64 exec, 1\n\t"
      "global_atomic_add_x2 %1, %2, off\n\t"
      "s_mov_b64 exec, %0"
      : "=&s"(save)
      : "v"(p), "v"(v)
      : "memory");
}
__device__ __forceinline__ void or32_lane0(uint32_t* p, uint32_t v) {
  unsigned long long save;
  asm volatile(
      "s_mov_b64 %0, exec\n\t"
      "s_mov_b64 exec, 1\n\t"
      "global_atomic_or %1, %2, off\n\t"
      "s_mov_b64 exec, %0"
      : "=&s"(save)
      : "v"(p), "v"(v)
      : "memory");
}
__device__ __forceinline__ void store64_lane0(unsigned long long* p, unsigned long long v) {
  unsigned long long save;
  asm volatile(
      "s_mov_b64 %0, exec\n\t"
      "s_mov_b64 exec, 1\n\t"
      "global_store_dwordx2 %1, %2, off sc1\n\t"
      "s_mov_b64 exec, %0"
      : "=&s"(save)
      : "v"(p), "v"(v)
      : "memory");
}
__device__ __forceinline__ void store32_lane0(int* p, int v) {
  unsigned long long save;
  asm volatile(
      "s_mov_b64 %0, exec\n\t"
      "s_mov_b64 exec, 1\n\t"
      "global_store_dword %1, %2, off sc1\n\t"
      "s_mov_b64 exec, %0"
      : "=&s"(save)
      : "v"(p), "v"(v)
      : "memory");
}

enum { kInsNew = 1, kInsDup = 0, kInsFull = -1 };

// Records run (b, row, xl, xr) with `label` in the slice of mask + 1 entries
// at tab.  Returns kInsNew, kInsFull, or kInsDup with the label stored by the
// run's first finder in `other`.
__device__ __forceinline__ int insert_run(unsigned long long* tab, unsigned mask, ArgPtr args,
                                          int b, int row, int xl, int xr, int label, int& other) {
  const unsigned long long key = run_key(b, row, xl);
  unsigned idx = hash_run(key) & mask;
  for (int i = 0;;) {
    unsigned long long* e = tab + 2 * (size_t)idx;
    const unsigned long long old = cas64_lane0(e, 0, key);
    if (__builtin_expect(old == 0, 1)) {
      store64_lane0(e + 1, ((unsigned long long)(unsigned)label << 32) |
                               (unsigned long long)(unsigned)xr);
      return kInsNew;
    }
    if (old == key) {
      // the winner writes word1 right after its compare-and-swap
      unsigned long long v = (unsigned long long)uni64((long long)ald(e + 1));
      for (int spin = 0; spin < (1 << 20) && v == kEmpty1; spin++) {
        __builtin_amdgcn_s_sleep(2);
        v = (unsigned long long)uni64((long long)ald(e + 1));
      }
      other = (int)(v >> 32);
      return v == kEmpty1 || other < 0 ? kInsFull : kInsDup;
    }
    idx = (idx + 1) & mask;
    if (++i >= opq(args)->probeLimit) return kInsFull;
  }
}

// ---------------------------------------------------------------------------
// Labels: union-find over flood labels; label b (< nBatch) is the class of
// the reference seeds of batch point b.  Roots link larger index to smaller.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int find_root(int* parent, int x) {
  for (int it = 0; it < (1 << 20); it++) {
    const int p = aldi(&parent[x]);
    if (p == x) return x;
    x = p;
  }
  return x;
}

__device__ __forceinline__ int uni_root(int* parent, int x) {
  for (int it = 0; it < (1 << 20); it++) {
    const int p = uni(aldi(&parent[x]));
    if (p == x) return x;
    x = p;
  }
  return x;
}

__device__ __forceinline__ void unite(int* parent, int a, int b) {
  for (int it = 0; it < (1 << 16) && a != b; it++) {
    const int ra = uni_root(parent, a), rb = uni_root(parent, b);
    if (ra == rb) break;
    const int hi = ra > rb ? ra : rb, lo = ra > rb ? rb : ra;
    if (cas32_lane0(&parent[hi], hi, lo) == hi) break;
  }
}

// ---------------------------------------------------------------------------
// Global task ring (tasks handed between workgroups): bounded
// multi-producer multi-consumer ring with per-slot sequence numbers.  The
// payload is complete before the sequence number that publishes it is
// written (mem_order between them), and a slot is handed back only after its
// payload has been read.
// ---------------------------------------------------------------------------
// A task as four 64-bit words (two ints each, low half first), and back:
// built from the fields, so no task is copied through memory.
__device__ __forceinline__ unsigned long long pack2(int lo, int hi) {
  return (unsigned long long)(unsigned)lo | ((unsigned long long)(unsigned)hi << 32);
}
__device__ __forceinline__ void task_words(const Task& t, unsigned long long (&w)[4]) {
  w[0] = pack2(t.b, t.row);
  w[1] = pack2(t.xa, t.xb);
  w[2] = pack2(t.label, t.kd);
  w[3] = pack2(t.f1, t.f2);
}
__device__ __forceinline__ Task words_task(const unsigned long long (&w)[4]) {
  Task t;
  t.b = (int)(unsigned)w[0]; t.row = (int)(unsigned)(w[0] >> 32);
  t.xa = (int)(unsigned)w[1]; t.xb = (int)(unsigned)(w[1] >> 32);
  t.label = (int)(unsigned)w[2]; t.kd = (int)(unsigned)(w[2] >> 32);
  t.f1 = (int)(unsigned)w[3]; t.f2 = (int)(unsigned)(w[3] >> 32);
  return t;
}

__device__ __forceinline__ bool q_push(ArgPtr args, const Task& t) {
  const ArgPtr a = opq(args);
  unsigned long long* const qtail = a->qtail;
  unsigned long long* const qseq = a->qseq;
  const unsigned long long qcap = a->qcap;
  unsigned long long pos = (unsigned long long)uni64((long long)ald(qtail));
  for (int it = 0; it < (1 << 20); it++) {
    const unsigned long long idx = pos & (qcap - 1);
    const unsigned long long seq = (unsigned long long)uni64((long long)ald(&qseq[idx]));
    const long long dif = (long long)(seq - pos);
    if (dif < 0) return false;  // full
    if (dif == 0) {
      const unsigned long long old = cas64_lane0(qtail, pos, pos + 1);
      if (old == pos) {
        unsigned long long w[4];
        task_words(t, w);
        unsigned long long* dst = reinterpret_cast<unsigned long long*>(&a->qbuf[idx]);
        for (int k = 0; k < 4; k++) store64_lane0(dst + k, w[k]);
        mem_order();
        store64_lane0(&qseq[idx], pos + 1);
        return true;
      }
      pos = old;
    } else {
      pos = (unsigned long long)uni64((long long)ald(qtail));
    }
  }
  return false;
}

__device__ __forceinline__ void flag_point(ArgPtr args, int gp, uint32_t f) {
  or32_lane0(opq(args)->flags + opq(gp), f);
}

__device__ __forceinline__ void afaddi(int* p, int v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, AGENT);
}

// Self-test of the in-range quotient (quot_near) and square root (sqrt_near,
// where lag_step takes it) against the IEEE operations on n operand pairs:
// random sign, exponent and mantissa (one pair in two), the ends of the
// range, and numerators built as the rounded product of the denominator and
// a quotient half an ulp above a random double (roots_check_kernel draws the
// hardest ones).  bad counts the pairs whose results differ in any bit.
__global__ void div_check_kernel(long long n, unsigned long long seed, unsigned long long* bad) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  unsigned long long cnt = 0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (unsigned long long)(i + 1);
    auto next = [&z]() {
      z += 0x9E3779B97F4A7C15ull;
      unsigned long long x = z;
      x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
      x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
      return x ^ (x >> 31);
    };
    auto make = [](unsigned long long r, int elo, int ehi) {
      const unsigned long long mant = r & ((1ull << 52) - 1);
      const int e = elo + (int)((r >> 52) % (unsigned long long)(ehi - elo + 1));
      const unsigned long long sign = (r >> 63) << 63;
      return __longlong_as_double((long long)(sign | ((unsigned long long)(e + 1023) << 52) | mant));
    };
    const unsigned long long r0 = next(), r1 = next(), kind = next() & 7;
    double a, b;
    if (kind < 4) {
      a = make(r0, -500, 9);
      b = make(r1, -500, 499);
    } else if (kind < 6) {
      b = make(r1, -480, 480);
      const double q = make(r0, -15, 15);
      const double h = ldexp(1.0, ilogb(q) - 53);  // half an ulp of q
      a = fma(b, h, b * q);
      if (!(fabs(a) >= 0x1p-500 && fabs(a) < 0x1p10)) a = q;
    } else {
      const double ends[6] = {0x1p-500, 0x1.fffffffffffffp9, 1.0, 0x1.0000000000001p-500,
                              0x1.fffffffffffffp499, 0x1p500};
      a = ends[r0 % 3] * ((r0 >> 8) & 1 ? -1.0 : 1.0);
      b = ends[(r1 % 3) * 2 + ((r1 >> 4) & 1)] * ((r1 >> 8) & 1 ? -1.0 : 1.0);
      if (kind == 7) b = make(r1, -500, 499);
    }
    const double x = quot_near(a, b, rcp_near(b)), y = a / b;
    cnt += __double_as_longlong(x) != __double_as_longlong(y) ? 1 : 0;
    if (edge(b) < kEdge) {
      double r, h;
      sqrt_near(fabs(b), r, h);
      cnt += __double_as_longlong(r) != __double_as_longlong(sqrt(fabs(b))) ? 1 : 0;
    }
  }
  if (cnt) atomicAdd(bad, cnt);
}

int launch_div_check(long long n, unsigned long long seed, unsigned long long* bad,
                     hipStream_t s) {
  if (n <= 0) return 0;
  if (!bad) return (int)hipErrorInvalidValue;
  const long long blocks = (n + 255) / 256;
  hipLaunchKernelGGL(div_check_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256),
                     0, s, n, seed, bad);
  return (int)hipGetLastError();
}

// Self-test of the in-range forms the root solver runs (tl_roots.h) against
// the general ones, to the bit, over the ranges lag_step admits.  Operands that
// it leaves to the general iteration for their mantissas are left out; bad[5]
// counts those among the random ones.
//   bad[0] quot_near: operands 2^-300 .. 2^300, random, and the quotients
//          closest to a rounding boundary: A 2^s = M B -+ j for a denominator
//          B, an odd 54-bit M and j = 1, 3, 5 (one B in four within 2^20
//          units below a power of two, one in eight as far above);
//   bad[1] sqrt_near: 2^-600 .. 2^600, random, and the `nHard` mantissas in
//          hard, whose roots lie closest to a rounding boundary;
//   bad[2] hyp_near against hyp_sel, bad[3] csqrt_near against csqrt_sel:
//          random signs, magnitudes 2^-240 .. 2^240, less than 2^54 apart;
//   bad[4] lag_step's next point, where it gives one, against lag_general's
//          from the same Horner sums, and points it gives although a part of
//          the sums' b[0] that it divides by has edge kEdge (one draw in
//          four); bad[6] counts the points compared.
template <int M>
__device__ __noinline__ void step_check(unsigned long long z, const TrigTable* trig,
                                        unsigned long long& differing,
                                        unsigned long long& compared) {
  auto next = [&z]() {
    z += 0x9E3779B97F4A7C15ull;
    unsigned long long x = z;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
  };
  auto val = [&next]() { return ((double)(long long)next()) * 0x1p-63 * (double)(1 << (next() & 7)); };
  cx b[M + 1];
  for (int j = 0; j <= M; j++) b[j] = mk(val(), val());
  const cx x = mk(val(), val());
  const bool edged = (next() & 3) == 0;
  if (edged) {
    // the larger part is the first divisor
    double& d = fabs(b[0].re) < fabs(b[0].im) ? b[0].im : b[0].re;
    d = __hiloint2double(__double2hiint(d) | 0xFFFF, __double2loint(d));
  }
  cx x1, step, y = x;
  if (!lag_step<M>(b, x, x1, step)) return;
  bool oob = false;
  if (!edged && lag_general<M>(b, y, 1, trig, oob)) return;
  compared++;
  if (edged || __double_as_longlong(y.re) != __double_as_longlong(x1.re) ||
      __double_as_longlong(y.im) != __double_as_longlong(x1.im))
    differing++;
}

__global__ void roots_check_kernel(long long n, unsigned long long seed, const double* hard,
                                   int nHard, const TrigTable* trig, unsigned long long* bad) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  unsigned long long cnt[5] = {0, 0, 0, 0, 0}, skipped = 0, steps = 0;
  auto differ = [](double x, double y) {
    return __double_as_longlong(x) != __double_as_longlong(y) ? 1ull : 0ull;
  };
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (unsigned long long)(i + 1);
    auto next = [&z]() {
      z += 0x9E3779B97F4A7C15ull;
      unsigned long long x = z;
      x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
      x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
      return x ^ (x >> 31);
    };
    // random sign and mantissa, exponent elo .. ehi
    auto make = [&next](int elo, int ehi) {
      const unsigned long long r = next(), e = next();
      const unsigned long long at = (unsigned long long)(1023 + elo) +
                                    e % (unsigned long long)(ehi - elo + 1);
      return __longlong_as_double(
          (long long)((r & 0x800FFFFFFFFFFFFFull) | (at << 52)));
    };
    {
      const double a = make(-300, 299), b = make(-300, 299);
      if (edge(b) < kEdge) cnt[0] += differ(quot_near(a, b, rcp_near(b)), a / b);
      else skipped++;
      const unsigned long long r = next(), kind = next() & 7;
      unsigned long long B = (r & ((1ull << 52) - 1)) | (1ull << 52) | 1ull;
      if (kind < 2) B = (1ull << 53) - ((r & ((1ull << 20) - 1)) | 1ull);
      else if (kind == 2) B = (1ull << 52) + ((r & ((1ull << 20) - 1)) | 1ull);
      unsigned long long inv = B;  // 1 / B modulo 2^64 (Newton)
      for (int k = 0; k < 6; k++) inv *= 2ull - B * inv;
      const int eb = (int)(next() % 500) - 250;
      for (int j = -5; j <= 5; j += 2) {
        const unsigned long long t = (unsigned long long)(long long)j * inv;
        for (int s = 53; s <= 54; s++) {
          const unsigned long long M =
              s == 53 ? (t & ((1ull << 53) - 1)) | (1ull << 53) : t & ((1ull << 54) - 1);
          if (!(M >> 53)) continue;
          // (M B - j) >> s
          unsigned long long lo = M * B, hi = __umul64hi(M, B);
          const unsigned long long d = (unsigned long long)(long long)j;
          hi -= (j < 0 ? ~0ull : 0ull) + (lo < d ? 1ull : 0ull);
          lo -= d;
          const unsigned long long A = (hi << (64 - s)) | (lo >> s);
          if (A >> 53 || !(A >> 52) || (s == 53) != (A >= B)) continue;
          const double x = (double)A, y = ldexp((double)B, eb);
          if (edge(y) < kEdge) cnt[0] += differ(quot_near(x, y, rcp_near(y)), x / y);
        }
      }
    }
    {
      double r, h;
      const double a = fabs(make(-600, 599));
      sqrt_near(a, r, h);
      if (edge(a) < kEdge) cnt[1] += differ(r, sqrt(a));
      else skipped++;
      if (nHard > 0) {
        const double c = ldexp(hard[next() % (unsigned long long)nHard],
                               2 * ((int)(next() % 596) - 298));
        sqrt_near(c, r, h);
        if (edge(c) < kEdge) cnt[1] += differ(r, sqrt(c));
      }
    }
    {
      const double x = make(-240, 239);
      const int e = ilogb(x);
      const int lo = e - 53 < -240 ? -240 : e - 53, hi = e + 53 > 239 ? 239 : e + 53;
      // magnitudes near each other in one pair of two (a radicand's usual case)
      const double y = next() & 1 ? make(lo, hi) : make(e - 1 < -240 ? -240 : e - 1,
                                                        e + 1 > 239 ? 239 : e + 1);
      const double ax = max_abs(x, y), ay = min_abs(x, y);
      if (hyp_in_range(ax, ay)) {
        double n1, n2;
        const double h = hyp_near(ax, ay, n1);
        if (edge(n1) < kEdge) cnt[2] += differ(h, hyp_sel(x, y));
        const cx c0 = csqrt_near(x, y, n1, n2), c1 = csqrt_sel(mk(x, y));
        if (edge(n1) < kEdge && edge(n2) < kEdge) cnt[3] += differ(c0.re, c1.re) | differ(c0.im, c1.im);
        else skipped++;
      }
    }
    step_check<10>(next(), trig, cnt[4], steps);
    step_check<5>(next(), trig, cnt[4], steps);
    step_check<2>(next(), trig, cnt[4], steps);
  }
  for (int k = 0; k < 5; k++)
    if (cnt[k]) atomicAdd(&bad[k], cnt[k]);
  if (skipped) atomicAdd(&bad[5], skipped);
  if (steps) atomicAdd(&bad[6], steps);
}

int launch_roots_check(long long n, unsigned long long seed, const double* hard, int nHard,
                       const TrigTable* trig, unsigned long long* bad, hipStream_t s) {
  if (n <= 0) return 0;
  if (!bad || !trig || nHard < 0 || (nHard > 0 && !hard)) return (int)hipErrorInvalidValue;
  const long long blocks = (n + 255) / 256;
  hipLaunchKernelGGL(roots_check_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256),
                     0, s, n, seed, hard, nHard, trig, bad);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// Row scanning
// ---------------------------------------------------------------------------
// What a fill needs of one batch point, one record of 32 doubles
// (fill_points_kernel): a worker loads it with lane k holding element k and
// reads elements from the lanes, so that a change of position costs one
// dependent load.
enum {
  kPcM1, kPcM2, kPcM3, kPcX1, kPcY1, kPcX2, kPcY2, kPcX3, kPcY3,  // lens
  kPcBlx, kPcBly, kPcStep,  // pixel grid
  kPcPx, kPcPy,             // source position
  kPcRho, kPcRho2, kPcInv,  // radius, its square, 1 / square
  kPcExt,                   // bound of the coordinates' magnitudes (fast rows)
  kPcLo, kPcHi,             // rho^2 -+ the band of rows far from the lenses
  kPcN, kPcGp,              // grid size; global point
  kPcFlags                  // kPt* bits
};
constexpr int kPtBinary = 1;  // irsBinary (m3 = 0)
constexpr int kPtFast = 2;    // lens and grid allow fast rows
constexpr int kPtLimb = 4;    // the profile's square-root term is not zero
constexpr int kPtHeavy = 8;   // predicted rays reach shareRays

// Half-width of the undecided band of the squared distance about rho^2 for
// rays whose terms' magnitudes sum to at most E (see Ray).
__device__ __forceinline__ double ray_band(double E, double rho) {
  const double delta = 0x1p-46 * E;
  return 2.0 * delta * (2.0 * rho + delta);
}
constexpr double kFarRow = 0x1p-10;

__global__ void fill_points_kernel(FillArgs A) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= A.nBatch) return;
  const int gp = A.batchPts[b];
  const CurveDev& C = A.curves[A.ptCurve[gp]];
  double* r = A.points + (size_t)b * kPointRec;
  const Lens& L = C.L;
  const double2 pos = A.ptPos[gp];
  r[kPcM1] = L.m1; r[kPcM2] = L.m2; r[kPcM3] = L.m3;
  r[kPcX1] = L.z1.re; r[kPcY1] = L.z1.im;
  r[kPcX2] = L.z2.re; r[kPcY2] = L.z2.im;
  r[kPcX3] = L.z3.re; r[kPcY3] = L.z3.im;
  r[kPcBlx] = C.blx; r[kPcBly] = C.bly; r[kPcStep] = C.step;
  r[kPcPx] = pos.x; r[kPcPy] = pos.y;
  r[kPcRho] = C.rho; r[kPcRho2] = C.rho2; r[kPcInv] = 1.0 / C.rho2;
  const double ext = fabs(C.blx) + fabs(C.bly) + 2.0 * C.step * (double)C.N + fabs(pos.x) +
                     fabs(pos.y) + fabs(L.z2.re) + fabs(L.z2.im) + fabs(L.z3.re) +
                     fabs(L.z3.im) + fabs(L.z1.re) + fabs(L.z1.im);
  r[kPcExt] = ext;
  r[kPcN] = (double)C.N;
  r[kPcGp] = (double)gp;
  const bool bin = C.binIrs != 0;
  auto mass = [](double m) { return m >= 0x1p-200 && m <= 0x1p10; };
  // E of the rows at least kFarRow from every lens
  const double band =
      ray_band(ext + (fabs(L.m1) + fabs(L.m2) + fabs(L.m3)) * (1.0 / kFarRow), C.rho);
  r[kPcLo] = C.rho2 - band;
  r[kPcHi] = C.rho2 + band;
  const bool fast = band <= 0x1p-10 * C.rho2 && ext <= 0x1p40 && C.rho2 >= 0x1p-200 && C.rho2 <= 0x1p40 && mass(L.m1) &&
                    mass(L.m2) && (bin || mass(L.m3));
  r[kPcFlags] = (double)((bin ? kPtBinary : 0) | (fast ? kPtFast : 0) |
                         (C.ldB != 0.0 ? kPtLimb : 0) |
                         (A.shareRays > 0.0f && A.ptCost[gp] >= A.shareRays ? kPtHeavy : 0));
}

int launch_fill_points(const FillArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(fill_points_kernel, dim3((a.nBatch + 255) / 256), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}

// The rays of one row of one position: the position's constants (wave-uniform)
// and the row's.
//
// Fast rows.  A pixel counts when its ray's squared distance from the source,
// computed by the reference's operations (irs_ray, irs_binary), is below
// rho^2.  Nearly every pixel is far from that boundary, so the distance is
// first formed with fused operations and one reciprocal for the three
// quotients (about 30 instructions instead of 80), and the reference's own
// operations decide only where it lies within [lo, hi].  Both forms use the
// same rounded pixel coordinates and lens distances; from there on each
// rounds at most 20 times, to a relative 2^-53 of the sum of the terms'
// magnitudes, which a row bounds by E = sum m_k / |y - y_k| + ext.  So the
// rays differ by at most delta = 2^-46 E (128 roundings), the squared
// distances near the boundary by 2 rho delta + delta^2, and lo, hi lie twice
// that from rho^2.  Rows at least kFarRow from every lens share one band per
// position; a row closer to one gets its own, and one whose band would exceed
// 2^-10 rho^2, or that passes within 2^-50 of a lens, is evaluated with the
// reference's operations throughout (kRowExact).
//
// A pixel's brightness always comes from the row's own form of the distance
// (never from the one that decided), so its value does not depend on which
// task evaluated it.
constexpr int kRowTriple = 0, kRowBinary = 1, kRowExact = 2;
struct Ray {
  double m1, m2, m3, x1, x2, x3, blx, step, px, inv;
  double f1, f2, f3, e1, e2, e3, ys, lo, hi;
  double pc;  // lane k: element k of the position's record
  int row, mode;
};

// Per-position constants of set_row, in vector registers.
struct RowBase {
  double y1, y2, y3, bly, step, py, lo, hi;
};
__device__ __forceinline__ double to_vgpr(double v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ __forceinline__ RowBase row_base(const Ray& R) {
  RowBase B;
  B.y1 = to_vgpr(rl(R.pc, kPcY1));
  B.y2 = to_vgpr(rl(R.pc, kPcY2));
  B.y3 = to_vgpr(rl(R.pc, kPcY3));
  B.bly = to_vgpr(rl(R.pc, kPcBly));
  B.step = to_vgpr(rl(R.pc, kPcStep));
  B.py = to_vgpr(rl(R.pc, kPcPy));
  B.lo = to_vgpr(rl(R.pc, kPcLo));
  B.hi = to_vgpr(rl(R.pc, kPcHi));
  return B;
}
// Sets the row of a position whose lens and grid allow fast rows (kPtFast) and
// returns whether the row lies far from every lens; else near_row has to
// follow.
__device__ __forceinline__ bool far_row(Ray& R, const RowBase& B, int row) {
  R.row = row;
  const double y = B.bly + B.step * (double)row;
  R.f1 = y - B.y1;
  R.f2 = y - B.y2;
  R.f3 = y - B.y3;
  R.e1 = R.f1 * R.f1;
  R.e2 = R.f2 * R.f2;
  R.e3 = R.f3 * R.f3;
  R.ys = y - B.py;
  R.lo = B.lo;
  R.hi = B.hi;
  return __ballot(min_abs(min_abs(R.f1, R.f2), R.f3) >= kFarRow) != 0;
}
// The row's own band; false when it has to be evaluated exactly.
__device__ __forceinline__ bool near_row(Ray& R, bool bin) {
  const double g1 = fabs(R.f1), g2 = fabs(R.f2), g3 = bin ? 1.0 : fabs(R.f3);
  // the hardware reciprocal's 2^-24 is well inside the factor two
  const double E = rl(R.pc, kPcExt) + R.m1 * __builtin_amdgcn_rcp(g1) +
                   R.m2 * __builtin_amdgcn_rcp(g2) + fabs(R.m3) * __builtin_amdgcn_rcp(g3);
  const double rho2 = rl(R.pc, kPcRho2), band = ray_band(E, rl(R.pc, kPcRho));
  R.lo = rho2 - band;
  R.hi = rho2 + band;
  const bool ok = g1 >= 0x1p-50 && g2 >= 0x1p-50 && g3 >= 0x1p-50 && band <= 0x1p-10 * rho2;
  return __ballot(!ok) == 0;
}
__device__ __forceinline__ void set_row(Ray& R, int flags, int row) {
  const RowBase B = row_base(R);
  const bool bin = (flags & kPtBinary) != 0;
  const bool fast = (far_row(R, B, row) || near_row(R, bin)) && (flags & kPtFast);
  R.mode = fast ? (bin ? kRowBinary : kRowTriple) : kRowExact;
}

// Squared distance in the reference's operations (irsSIMD, lcirs.cc:290-341;
// irsBinary, lcirs.cc:345-353), from y as set_row formed it.
template <bool BIN>
__device__ __forceinline__ double ray_exact(const Ray& R, double x) {
  Lens L;
  L.m1 = R.m1; L.m2 = R.m2; L.m3 = R.m3;
  L.z1 = mk(R.x1, rl(R.pc, kPcY1));
  L.z2 = mk(R.x2, rl(R.pc, kPcY2));
  L.z3 = mk(R.x3, rl(R.pc, kPcY3));
  const double y = rl(R.pc, kPcBly) + rl(R.pc, kPcStep) * (double)R.row, py = rl(R.pc, kPcPy);
  return BIN ? irs_binary(L, x, y, R.px, py) : irs_ray(L, x, y, R.px, py);
}

template <int MODE>
__device__ __forceinline__ double ray_fast(const Ray& R, double x) {
  const double a1 = x - R.x1, a2 = x - R.x2;
  const double q1 = fma(a1, a1, R.e1), q2 = fma(a2, a2, R.e2);
  double nr, ni, Q;
  if (MODE == kRowTriple) {
    const double a3 = x - R.x3;
    const double q3 = fma(a3, a3, R.e3);
    const double q12 = q1 * q2;
    const double w1 = R.m1 * (q2 * q3), w2 = R.m2 * (q1 * q3), w3 = R.m3 * q12;
    Q = q12 * q3;
    nr = fma(w1, a1, fma(w2, a2, w3 * a3));
    ni = fma(w1, R.f1, fma(w2, R.f2, w3 * R.f3));
  } else {
    const double w1 = R.m1 * q2, w2 = R.m2 * q1;
    Q = q1 * q2;
    nr = fma(w1, a1, w2 * a2);
    ni = fma(w1, R.f1, w2 * R.f2);
  }
  const double r = rcp_near(Q);
  const double re = fma(-nr, r, x - R.px), im = fma(-ni, r, R.ys);
  return fma(re, re, im * im);
}

// sqrt(t) for 0 < t <= 1 within a few units in the last place (the hardware
// reciprocal root and one third-order step), as a multiple of 1/kSumScale
// plus kMagic: rounded to the nearest integer multiple by adding 1.5 * 2^52,
// the sum's bits are those of kMagic plus the integer.
constexpr long long kMagicBits = 0x4338000000000000ll;  // the bits of 1.5 * 2^52
__device__ __forceinline__ long long root_bits(double t) {
  const double y = __builtin_amdgcn_rsq(t);
  const double s0 = t * y, h = 0.5 * y;
  const double e = fma(-s0, h, 0.5);
  const double s = fma(s0, fma(1.5 * e, e, e), s0);
  return __double_as_longlong(fma(s, kSumScale, 6755399441055744.0));
}

// The same for any t, 0 where t is not positive.
__device__ __forceinline__ long long root_bits_or_0(double t) {
  const bool pos = t > 0.0;
  return root_bits(pos ? t : 1.0) - (pos ? 0 : (long long)kSumScale);
}

// Evaluates the pixels of columns c .. c + 63 (lane l: column c + l): the hit
// mask, and (LIMB) every hit lane's square root of 1 - r^2/rho^2 as bits.
template <int MODE, bool LIMB>
__device__ __forceinline__ unsigned long long eval_block(const Ray& R, int c, long long& bits) {
  const int ln = __lane_id();
  const double x = R.blx + R.step * (double)(c + ln);
  if (MODE == kRowExact) {
    const double rsq =
        (int)rl(R.pc, kPcFlags) & kPtBinary ? ray_exact<true>(R, x) : ray_exact<false>(R, x);
    if (LIMB) bits = root_bits_or_0(1.0 - rsq * R.inv);
    return __ballot(rsq < rl(R.pc, kPcRho2));
  }
  const double rsq = ray_fast<MODE>(R, x);
  unsigned long long hit = __ballot(rsq < R.lo);
  const unsigned long long miss = __ballot(rsq > R.hi);
  double t = fma(-rsq, R.inv, 1.0);
  if (__builtin_expect(~(hit | miss) != 0, 0)) {
    hit |= ~(hit | miss) & __ballot(ray_exact<MODE == kRowBinary>(R, x) < rl(R.pc, kPcRho2));
    if (LIMB) {
      bits = root_bits_or_0(t);
      return hit;
    }
  }
  if (LIMB) bits = root_bits(t);
  return hit;
}

__device__ __forceinline__ unsigned long long low_bits(int n) {
  return n >= 64 ? ~0ull : (1ull << n) - 1ull;
}

// The maximal hit runs of one row that meet [s, e], left to right.  The row is
// evaluated in steps of 64 pixels over a window that pads [s, e] to whole
// steps on the sides where runs may continue (extL, extR); elsewhere the
// pixel next to [s, e] is a known miss.  A run that reaches the window's right
// edge is followed past it; one that reaches its left edge is left to
// extend_left.
struct RunScan {
  int s, e, ws, we, hi;    // interval, window, last column of the scan
  int c;                   // first column of the current step
  unsigned long long m;    // its hits not yet handed out
  bool extL, extR;
  long long bits;          // (lane) brightness of the step's pixel
  // the run found
  int xl, xr;
  unsigned cnt;
  long long acc;           // (lane) brightness bits of its pixels
  unsigned steps;          // steps evaluated
};

__device__ __forceinline__ void scan_begin(RunScan& Q, int N, int s, int e, bool extL, bool extR) {
  const int len = e - s + 1;
  const int extra = ((len + 63) & ~63) - len;
  const int padL = extL ? (extR ? extra / 2 : extra) : 0;
  const int padR = extR ? extra - padL : 0;
  Q.s = s;
  Q.e = e;
  Q.ws = s - padL < 0 ? 0 : s - padL;
  Q.we = e + padR > N - 1 ? N - 1 : e + padR;
  Q.hi = Q.we;
  Q.c = Q.ws - 64;
  Q.m = 0;
  Q.extL = extL;
  Q.extR = extR;
}

// The next run, or false.  Whole steps inside a run cost their ray tests and
// one accumulation.
template <int MODE, bool LIMB>
__device__ __forceinline__ bool scan_next(const Ray& R, int N, RunScan& Q) {
  const int ln = __lane_id();
  while (true) {
    while (Q.m == 0) {
      Q.c += 64;
      if (Q.c > Q.e || Q.c > Q.hi) return false;  // no later run can meet [s, e]
      const int nb = Q.hi - Q.c + 1;
      Q.m = eval_block<MODE, LIMB>(R, Q.c, Q.bits) & low_bits(nb);
      Q.steps++;
    }
    const int t = __builtin_ctzll(Q.m);
    Q.xl = Q.c + t;
    if (Q.xl > Q.e) return false;
    unsigned long long inv = ~(Q.m >> t);
    int z = inv ? __builtin_ctzll(inv) : 64;
    if (z > 64 - t) z = 64 - t;
    unsigned long long take = low_bits(z) << t;
    if (LIMB) Q.acc = (take >> ln) & 1ull ? Q.bits : 0;
    Q.cnt = (unsigned)z;
    Q.xr = Q.xl + z - 1;
    Q.m &= ~take;
    // follow the run through whole steps
    bool followed = false;
    while (Q.xr == Q.c + 63 || Q.xr == Q.hi) {
      if (Q.xr == Q.hi) {
        if (!(Q.hi == Q.we && Q.extR && Q.we < N - 1)) break;  // its end is known
        Q.hi = N - 1;
        Q.c = Q.we - 63;
        followed = true;
      }
      Q.c += 64;
      const int nb = Q.hi - Q.c + 1;
      Q.m = eval_block<MODE, LIMB>(R, Q.c, Q.bits) & low_bits(nb);
      Q.steps++;
      if (Q.m == ~0ull) {
        if (LIMB) Q.acc += Q.bits;
        Q.cnt += 64;
        Q.xr += 64;
        Q.m = 0;
        continue;
      }
      z = __builtin_ctzll(~Q.m);
      take = low_bits(z);
      if (LIMB) Q.acc += (take >> ln) & 1ull ? Q.bits : 0;
      Q.cnt += (unsigned)z;
      Q.xr += z;
      Q.m &= ~take;
      if (z == 0) break;
    }
    if (followed) Q.m = 0;  // nothing beyond the followed run meets [s, e]
    if (Q.xr >= Q.s) return true;
  }
}

// Follows a run leftwards from column `from` until its first miss or column
// 0; returns the run's first column and adds the pixels taken in.
template <int MODE, bool LIMB>
__device__ __forceinline__ int extend_left(const Ray& R, int from, RunScan& Q) {
  const int ln = __lane_id();
  while (from >= 0) {
    const int c = from - 63;  // the step's columns end at `from`
    long long bits = 0;
    unsigned long long m = eval_block<MODE, LIMB>(R, c, bits);
    if (c < 0) m &= ~low_bits(-c);
    Q.steps++;
    const int z = m == ~0ull ? 64 : __builtin_clzll(~m);  // hits counted from `from` down
    if (LIMB) Q.acc += ln >= 64 - z ? bits : 0;
    Q.cnt += (unsigned)z;
    if (z < 64) return from - z + 1;
    from -= 64;
  }
  return 0;
}

template <int MODE, bool LIMB>
__device__ __forceinline__ bool next_run_in(const Ray& R, int N, RunScan& Q) {
  if (!scan_next<MODE, LIMB>(R, N, Q)) return false;
  if (Q.xl == Q.ws && Q.extL && Q.ws > 0) Q.xl = extend_left<MODE, LIMB>(R, Q.ws - 1, Q);
  return true;
}
__device__ __forceinline__ bool next_run(const Ray& R, int N, bool limb, RunScan& Q) {
  if (R.mode == kRowTriple)
    return limb ? next_run_in<kRowTriple, true>(R, N, Q) : next_run_in<kRowTriple, false>(R, N, Q);
  if (R.mode == kRowBinary)
    return limb ? next_run_in<kRowBinary, true>(R, N, Q) : next_run_in<kRowBinary, false>(R, N, Q);
  return next_run_in<kRowExact, true>(R, N, Q);
}

// ---------------------------------------------------------------------------
// Workgroup task pool (LDS)
// ---------------------------------------------------------------------------
// A fill workgroup has one manager wave and kWorkers worker waves.  The
// workers share a pool of waiting tasks in LDS, guarded by a lock word that
// lane 0 of a wave takes.  `pending` counts the pool's tasks plus the
// workers that hold work (a task in hand or in their own ring); it changes
// only under the lock, so when it reads 0 no worker of the group holds work
// or can make any, and only the manager brings tasks in (seed tasks, or
// tasks that other groups queued in the global ring).  LDS operations of one
// wave are performed in program order; the unlock waits for the wave's LDS
// operations before it releases the word.
constexpr int kWorkers = kFillWaves - 1;
constexpr int kFillStats = 11;   // FillArgs::stats
constexpr int kFeedMax = 16;     // tasks the manager brings in at a time
constexpr int kDonateMax = 8;    // tasks the manager queues for other groups at a time
constexpr int kPoolShare = 16;   // while other groups are idle, workers keep the pool at
                                 // this many tasks

struct GroupPool {
  int lock;
  int pending;     // pool tasks + workers holding work
  int head, count; // the pool ring: count tasks from head on
  int done;        // set by the manager when the fill is over
  int hungry;      // set by the manager while other groups are idle: workers then
                   // move waiting tasks to the pool, and the manager on to the
                   // global ring
  int pad[2];
  Task slot[kPoolCap];
};

#define WGS __HIP_MEMORY_SCOPE_WORKGROUP
__device__ __forceinline__ int lds_ld(int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, WGS); }
__device__ __forceinline__ void lds_st(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, WGS);
}
template <class T>
__device__ __forceinline__ T lds_add(T* p, T v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, WGS);
}
// Waits until the wave's LDS (and scalar) memory operations are done.
__device__ __forceinline__ void lds_wait() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), vmcnt and expcnt not waited for
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
// Lane 0 takes and releases the pool lock.
__device__ __forceinline__ void pool_lock(GroupPool* G) {
  while (true) {
    int expected = 0;
    if (__hip_atomic_compare_exchange_strong(&G->lock, &expected, 1, __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, WGS))
      break;
    __builtin_amdgcn_s_sleep(1);
  }
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
__device__ __forceinline__ void pool_unlock(GroupPool* G) {
  lds_wait();
  lds_st(&G->lock, 0);
}

// A worker's tasks.  A task at rest is eight ints of LDS; a worker moves it
// with lane k < 8 holding int k (the other lanes read and write a scratch
// area, so that no access is under a branch) and reads the fields from the
// lanes.
template <int K>
__device__ __forceinline__ void write_lane(int& v, int x) {
  asm("v_writelane_b32 %0, %1, %2" : "+v"(v) : "s"(uni(x)), "n"(K));
}
__device__ __forceinline__ int task_lanes(const Task& t) {
  int v = 0;
  write_lane<0>(v, t.b);
  write_lane<1>(v, t.row);
  write_lane<2>(v, t.xa);
  write_lane<3>(v, t.xb);
  write_lane<4>(v, t.label);
  write_lane<5>(v, t.kd);
  write_lane<6>(v, t.f1);
  write_lane<7>(v, t.f2);
  return v;
}
__device__ __forceinline__ Task lanes_task(int v) {
  Task t;
  t.b = __builtin_amdgcn_readlane(v, 0);
  t.row = __builtin_amdgcn_readlane(v, 1);
  t.xa = __builtin_amdgcn_readlane(v, 2);
  t.xb = __builtin_amdgcn_readlane(v, 3);
  t.label = __builtin_amdgcn_readlane(v, 4);
  t.kd = __builtin_amdgcn_readlane(v, 5);
  t.f1 = __builtin_amdgcn_readlane(v, 6);
  t.f2 = __builtin_amdgcn_readlane(v, 7);
  return t;
}
// This lane's int of the task at `slot`; lanes 8.. get a place of their own in
// `spare` (64 ints per wave).
__device__ __forceinline__ int* task_int(Task* slot, int* spare) {
  const int ln = __lane_id();
  return ln < 8 ? reinterpret_cast<int*>(slot) + ln : spare + ln;
}

// Takes and releases the pool lock (the whole wave; lane 0's exchange).
__device__ __forceinline__ int lds_cas_lane0(int* p, int expected, int desired) {
  int old;
  unsigned long long save;
  const unsigned at = (unsigned)(unsigned long long)(__attribute__((address_space(3))) int*)p;
  asm volatile(
      "s_mov_b64 %1, exec\n\t"
      "s_mov_b64 exec, 1\n\t"
      "ds_cmpst_rtn_b32 %0, %2, %3, %4\n\t"
      "s_waitcnt lgkmcnt(0)\n\t"
      "s_mov_b64 exec, %1"
      : "=&v"(old), "=&s"(save)
      : "v"(at), "v"(expected), "v"(desired)
      : "memory");
  return uni(old);
}
__device__ __forceinline__ void wave_lock(GroupPool* G) {
  while (lds_cas_lane0(&G->lock, 0, 1) != 0) __builtin_amdgcn_s_sleep(1);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// A worker that holds work adds the (wave-uniform) task t; false when the
// pool is full.
__device__ __forceinline__ bool pool_push(GroupPool* G, const Task& t, int* spare) {
  const int v = task_lanes(t);
  wave_lock(G);
  const int c = uni(lds_ld(&G->count));
  const bool ok = c < kPoolCap;
  if (ok) {
    *task_int(&G->slot[(uni(lds_ld(&G->head)) + c) & (kPoolCap - 1)], spare) = v;
    lds_st(&G->count, c + 1);
    lds_st(&G->pending, uni(lds_ld(&G->pending)) + 1);
  }
  pool_unlock(G);
  return ok;
}

// A worker takes a task of the pool: the newest (newest = true) or the
// oldest.  busy: the worker holds work now (its last task is done and its
// ring is empty): it takes a task (pending - 1) or, with the pool empty,
// gives up its count (pending - 1) and is idle from then on.  !busy: an idle
// worker takes a task and is counted as holding work (pending unchanged),
// or stays idle.  The newest first keeps a group on the sweeps its scouts
// just opened (on the images still growing) before older ones: the
// surrogate's fallback fill of the C2 curve takes ~3% less time with it,
// the heaviest 41 positions ~5% less, C3's fill the same.
__device__ __forceinline__ bool pool_take(GroupPool* G, Task& t, bool busy, bool newest,
                                          int* spare) {
  wave_lock(G);
  const int c = uni(lds_ld(&G->count));
  int v = 0;
  if (c > 0) {
    const int h = uni(lds_ld(&G->head));
    v = *task_int(&G->slot[newest ? (h + c - 1) & (kPoolCap - 1) : h], spare);
    if (!newest) lds_st(&G->head, (h + 1) & (kPoolCap - 1));
    lds_st(&G->count, c - 1);
  }
  if (busy) lds_st(&G->pending, uni(lds_ld(&G->pending)) - 1);
  pool_unlock(G);
  if (c > 0) t = lanes_task(v);
  return c > 0;
}

// Manager: adds the tasks held by lanes [lo, hi) (pending + their number).
// Returns how many fitted; the caller makes room first.
__device__ __forceinline__ int pool_add_lanes(GroupPool* G, const Task& t, int lo, int hi) {
  const int ln = __lane_id();
  int base = 0, fit = 0;
  if (ln == 0) {
    pool_lock(G);
    const int c = lds_ld(&G->count);
    fit = hi - lo < kPoolCap - c ? hi - lo : kPoolCap - c;
    base = lds_ld(&G->head) + c;
  }
  fit = uni(fit);
  base = uni(base);
  if (ln >= lo && ln < lo + fit) G->slot[(base + ln - lo) & (kPoolCap - 1)] = t;
  if (ln == 0) {
    lds_st(&G->count, lds_ld(&G->count) + fit);
    lds_st(&G->pending, lds_ld(&G->pending) + fit);
    pool_unlock(G);
  }
  return fit;
}

// Manager: takes up to n of the pool's oldest tasks into lanes [0, k)
// (pending - k) and returns k.
__device__ __forceinline__ int pool_remove_lanes(GroupPool* G, Task& t, int n) {
  const int ln = __lane_id();
  int k = 0, h = 0;
  if (ln == 0) {
    pool_lock(G);
    const int c = lds_ld(&G->count);
    k = n < c ? n : c;
    h = lds_ld(&G->head);
  }
  k = uni(k);
  h = uni(h);
  if (ln < k) t = G->slot[(h + ln) & (kPoolCap - 1)];
  if (ln == 0) {
    lds_st(&G->head, (h + k) & (kPoolCap - 1));
    lds_st(&G->count, lds_ld(&G->count) - k);
    lds_st(&G->pending, lds_ld(&G->pending) - k);
    pool_unlock(G);
  }
  return k;
}

// Global ring, many tasks per call (manager): lanes [0, n) offer one task
// each; the leading k slots that are free at the tail are claimed with one
// compare-and-swap and written in parallel.  Returns k (the tasks of lanes
// [0, k) are queued).
__device__ __forceinline__ int q_push_lanes(const FillArgs& A, const Task& t, int n) {
  const int ln = __lane_id();
  unsigned long long pos = 0;
  int k = 0;
  for (int it = 0; it < 64; it++) {
    if (ln == 0) pos = ald(A.qtail);
    pos = uni64(pos);
    const bool fr = ln < n && ald(&A.qseq[(pos + ln) & (A.qcap - 1)]) == pos + ln;
    const unsigned long long m = __ballot(fr);
    k = ~m == 0 ? 64 : __builtin_ctzll(~m);
    if (k == 0) return 0;  // full, or another producer moved the tail: try again later
    int ok = 0;
    if (ln == 0) {
      unsigned long long exp = pos;
      ok = acas(A.qtail, &exp, pos + k);
    }
    if (uni(ok)) break;
    k = 0;
  }
  if (ln < k) {
    const unsigned long long idx = (pos + ln) & (A.qcap - 1);
    unsigned long long w[4];
    task_words(t, w);
    unsigned long long* dst = reinterpret_cast<unsigned long long*>(&A.qbuf[idx]);
    ast(&dst[0], w[0]);
    ast(&dst[1], w[1]);
    ast(&dst[2], w[2]);
    ast(&dst[3], w[3]);
    mem_order();
    ast(&A.qseq[idx], pos + ln + 1);
  }
  return k;
}

// Global ring, many tasks per call (manager): takes the leading k <= n
// ready slots at the head into lanes [0, k); returns k.
__device__ __forceinline__ int q_pop_lanes(const FillArgs& A, Task& t, int n) {
  const int ln = __lane_id();
  unsigned long long pos = 0;
  int k = 0;
  for (int it = 0; it < 64; it++) {
    if (ln == 0) pos = ald(A.qhead);
    pos = uni64(pos);
    const bool rd = ln < n && ald(&A.qseq[(pos + ln) & (A.qcap - 1)]) == pos + ln + 1;
    const unsigned long long m = __ballot(rd);
    k = ~m == 0 ? 64 : __builtin_ctzll(~m);
    if (k == 0) return 0;
    int ok = 0;
    if (ln == 0) {
      unsigned long long exp = pos;
      ok = acas(A.qhead, &exp, pos + k);
    }
    if (uni(ok)) break;
    k = 0;
  }
  if (ln < k) {
    const unsigned long long idx = (pos + ln) & (A.qcap - 1);
    unsigned long long w[4];
    const unsigned long long* src = reinterpret_cast<unsigned long long*>(&A.qbuf[idx]);
    w[0] = ald(const_cast<unsigned long long*>(&src[0]));
    w[1] = ald(const_cast<unsigned long long*>(&src[1]));
    w[2] = ald(const_cast<unsigned long long*>(&src[2]));
    w[3] = ald(const_cast<unsigned long long*>(&src[3]));
    mem_order();
    ast(&A.qseq[idx], pos + ln + A.qcap);
    t = words_task(w);
  }
  return k;
}

// Manager: puts the tasks of lanes [lo, hi) back into the pool, or, where it
// is full, into the global ring; waits while both are full (workers keep
// draining the pool), up to the deadline (s_memrealtime ticks).
__device__ __forceinline__ void pool_add_all(const FillArgs& A, GroupPool* G, const Task& t,
                                             int lo, int hi, long long deadline) {
  for (int it = 0; lo < hi; it++) {
    lo += pool_add_lanes(G, t, lo, hi);
    if (lo >= hi) break;
    // lanes [lo, hi) still hold tasks: offer them to the ring from lane 0 on
    Task u = t;
    const int src = __lane_id() + lo;
    u.b = __shfl(t.b, src, 64); u.row = __shfl(t.row, src, 64);
    u.xa = __shfl(t.xa, src, 64); u.xb = __shfl(t.xb, src, 64);
    u.label = __shfl(t.label, src, 64); u.kd = __shfl(t.kd, src, 64);
    u.f1 = __shfl(t.f1, src, 64); u.f2 = __shfl(t.f2, src, 64);
    lo += q_push_lanes(A, u, hi - lo);
    if (lo >= hi) break;
    if ((long long)__builtin_amdgcn_s_memrealtime() > deadline) {
      if (__lane_id() == 0) atomicExch(A.abortFlag, 1);
      break;
    }
    __builtin_amdgcn_s_sleep(16);
  }
}

// Manager: seed tasks [st, st + k) of the batch into lanes [0, k); returns k.
__device__ __forceinline__ int claim_seeds(const FillArgs& A, Task& t, int n) {
  const int ln = __lane_id();
  int st = A.nSeedTasks;
  if (ln == 0 && aldi(A.seedNext) < A.nSeedTasks) st = atomicAdd(A.seedNext, n);
  st = uni(st);
  int k = A.nSeedTasks - st;
  k = k < 0 ? 0 : (k > n ? n : k);
  if (ln < k) {
    const int2 sk = A.seedTasks[st + ln];
    const int gp = A.batchPts[sk.x];
    const int2 px = A.seeds[(size_t)gp * kMaxSeeds + sk.y];
    const long long N = A.curves[A.ptCurve[gp]].N;
    // the reference skips seeds outside rows 1..N-1 (lcirs.cc:386-389)
    const bool rowOk = px.y > 0 && (long long)px.y < N;
    t.b = sk.x; t.row = rowOk ? px.y : -1; t.xa = px.x; t.xb = px.x; t.label = sk.x;
    t.kd = 1; t.f1 = 0; t.f2 = -1;
  }
  return k;
}

// A worker wave's state (uniform across the wave where not marked).
struct Worker {
  ArgPtr A;
  int scoutRows;            // (a hot argument)
  GroupPool* G;             // the workgroup's shared pool
  Task* ring;               // this wave's ring of waiting tasks in LDS:
  int lhead, lcount;        // lcount tasks from lhead on
  Task* out;                // its tasks for the pool: nOut of them
  int nOut;
  Task* back;               // the look-backs recorded by the row's scan: nBack of them
  int nBack;
  int* spare;               // 64 ints of LDS for the lanes without a task int
  Task t;                   // the task in hand
  bool haveCont;            // t is the follow-up kept by this wave
  bool general;             // t is for process_task
  // the position whose constants R holds
  int curB, gp, N, flags;
  unsigned long long* tab;  // its run-table slice
  unsigned tabMask;
  Ray R;
  // totals of new runs, credited to accLabel when the label changes or the
  // wave runs out of work
  int accLabel;
  unsigned accCnt;
  long long accBits;        // (lane) brightness bits, kMagicBits included per pixel
  unsigned nTasks, nIns, nDup, nScout, nScoutRuns, steps;
  unsigned insTicks, nTimed;  // time of the timed inserts, and their number
  bool landed;              // the scout task found a run (new or known)
};

// Task hand-off.  Follow-ups a worker does not continue with go to its own
// ring in LDS (no atomics: one owner); the newest is taken next (depth
// first).  Tasks for the group's pool at once wait in the wave's out buffer
// until the row's scan step is done.  While other workers of the group are
// idle, a worker moves its oldest waiting tasks to the pool; a ring that is
// nearly full spills there too, and a full pool into the global ring.
__device__ __forceinline__ void ring_put(Worker& W, const Task& f) {
  *task_int(&W.ring[(W.lhead + W.lcount) & (kLocalCap - 1)], W.spare) = task_lanes(f);
  W.lcount++;
}

__device__ __forceinline__ Task ring_pop(Worker& W) {
  W.lcount--;
  return lanes_task(*task_int(&W.ring[(W.lhead + W.lcount) & (kLocalCap - 1)], W.spare));
}

// Empties the out buffer into the pool (the ring where the pool is full) and
// moves `give` of the ring's oldest tasks, and as many as make room for the
// next runs' follow-ups, to the pool or the global ring.
constexpr int kOutCap = 8;     // out buffer: a run adds at most 3
constexpr int kRoom = 16;      // ring places kept free (out buffer and a run's follow-ups)
__device__ __forceinline__ void hand_off(Worker& W, int give) {
  while (W.nOut > 0 || give > 0 || W.lcount > kLocalCap - kRoom) {
    const bool out = W.nOut > 0;
    if (!out && W.lcount == 0) break;
    const Task t = lanes_task(
        *task_int(out ? &W.out[W.nOut - 1] : &W.ring[W.lhead], W.spare));
    const bool pooled = pool_push(W.G, t, W.spare);
    if (out) {
      W.nOut--;
      if (!pooled) ring_put(W, t);
      continue;
    }
    if (!pooled && !q_push(W.A, t)) {
      if (W.lcount < kLocalCap - 4) break;  // still room: keep the rest
      flag_point(W.A, W.gp, kFlagQueueFull);  // everything full: the task is lost
    }
    W.lhead = (W.lhead + 1) & (kLocalCap - 1);
    W.lcount--;
    give--;
  }
}

// The totals go to the label as the count and, in two words, the sum of the
// pixels' integers: words (p[0], p[1]) stand for p[1] * 2^32 + p[0], p[0]
// summing the low 32 bits of every value added and p[1] the rest, so that no
// total wraps as long as fewer than 2^32 values are added to it.
__device__ __forceinline__ void flush_acc(Worker& W) {
  if (W.accCnt) {
    const ArgPtr A = opq(W.A);
    add64_lane0(&A->lcount[W.accLabel], W.accCnt);
    if (W.flags & kPtLimb) {
      const unsigned long long v = (unsigned long long)uni64(wave_sum(W.accBits)) -
                                   (unsigned long long)W.accCnt * (unsigned long long)kMagicBits;
      unsigned long long* p = &A->lsum[2 * (size_t)W.accLabel];
      add64_lane0(p, v & 0xFFFFFFFFull);
      if (v >> 32) add64_lane0(p + 1, v >> 32);
    }
  }
  W.accCnt = 0;
  W.accBits = 0;
}

__device__ __forceinline__ Task make_task(int b, int row, int xa, int xb, int label, int kind,
                                          int dir, int f1, int f2) {
  Task f;
  f.b = b; f.row = row; f.xa = xa; f.xb = xb; f.label = label;
  f.kd = kind | (dir < 0 ? 4 : 0);
  f.f1 = f1; f.f2 = f2;
  return f;
}

constexpr int kQueueOnly = 8;  // follow-up flag: never kept by the wave
constexpr int kShare = 16;     // follow-up flag: to the group's pool at once (the wave's
                               // ring when the pool is full)

// A follow-up of a run, dispatched as soon as it is made: the first one that
// may stay with the wave becomes its next step, tasks marked kShare go to the
// group's pool, the others to the wave's ring.
__device__ __forceinline__ void follow(Worker& W, const Task& f, int where) {
  if (where == 0 && !W.haveCont) {
    W.t = f;
    W.haveCont = true;
  } else if (where & kShare) {
    *task_int(&W.out[W.nOut], W.spare) = task_lanes(f);
    W.nOut++;
  } else {
    ring_put(W, f);
  }
}

// A look-back, kept for the end of the row's scan, or queued when two are
// already waiting.
__device__ __forceinline__ void put_back(Worker& W, const Task& f) {
  if (W.nBack < 2) {
    *task_int(&W.back[W.nBack], W.spare) = task_lanes(f);
    W.nBack++;
  } else {
    ring_put(W, f);
  }
}

// Rows a scout jumps from a run of w pixels: scout_jump, shortened in
// proportion where runs are wider than scout_width pixels (0: never), so
// that the rows between two scouts hold about the same number of pixels on
// wide stretches of an image as on narrow ones.  A scout task carries the
// jump it was sent with in the high half of f2 (the low half counts the
// scouts of its chain since the last leap).
constexpr int kMinJump = 16;
__device__ __forceinline__ int scout_jump_for(ArgPtr A, int w) {
  const int jump = A->scoutJump, width = A->scoutWidth;
  if (width <= 0 || w <= width) return jump;
  // below 2^15 and 2^25: the quotient in 64 bits, by the hardware reciprocal
  // would round; the integer division is rare (one run in kMinJump at most)
  const long long j = (long long)jump * width / w;
  const int lo = kMinJump < jump ? kMinJump : jump;
  return j < lo ? lo : (int)j;
}

// What a task scans: a row between columns, in one or two pieces around known
// pixels.
struct Scan {
  int kind, dir, row, label;
  int xa, xb;  // the interval: the known run next to the row (kind 0: the
               // parent, kind 3: the child)
  int k1, k2;  // known pixels within it (none if k1 > k2)
};

// A maximal hit run [xl, xr] of the scan's row was found (cnt pixels, their
// brightness bits per lane in acc): record it, credit its pixels to its label
// and schedule the neighbouring rows.  f1, f2: those of the task in hand (they
// drive sweeps and scouts).  Returns whether a look-back is due: at the row
// the run was reached from, where it reaches past that row's known run and
// its two bounding misses.
__device__ __forceinline__ bool handle_run(Worker& W, const Scan& S, int f1, int f2, int xl, int xr,
                                           unsigned cnt, long long acc, int& labelOut) {
  const int b = W.curB, row = opq(S.row), N = opq(W.N), d = opq(S.dir), kind = opq(S.kind);
  f1 = opq(f1);
  f2 = opq(f2);
  int label = S.label;
  if (__builtin_expect(kind == 2, 0)) {
    W.landed = true;
    // a scout run starts a class of its own
    const ArgPtr A = opq(W.A);
    label = add32_lane0(A->labelNext, 1);
    if (label >= A->labelCap) {
      flag_point(W.A, W.gp, kFlagLabelFull);
      return false;
    }
    store32_lane0(&A->lpoint[label], b);
  }
  labelOut = label;
  int other = 0;
  const int ins = insert_run(W.tab, W.tabMask, W.A, b, row, xl, xr, label, other);
  if (__builtin_expect(ins != kInsNew, 0)) {
    if (ins == kInsFull) {
      flag_point(W.A, W.gp, kFlagHashFull);
    } else {
      W.nDup++;
      if (kind != 2) unite(opq(W.A)->lparent, label, other);
    }
    return false;
  }
  W.nIns++;
  if (xl <= 1 || xr >= N - 2) flag_point(W.A, W.gp, kFlagEdge);
  // at most 2^26 pixels before a flush: their integers stay below 2^62
  if (label != W.accLabel || W.accCnt >= (1u << 25)) {
    flush_acc(W);
    W.accLabel = label;
  }
  W.accCnt += cnt;
  if (W.flags & kPtLimb) W.accBits += acc;
  const int center = (int)(((unsigned)xl + (unsigned)xr) / 2);
  const bool ahead = row + d >= 0 && row + d < N;
  const bool past = row - d >= 0 && row - d < N && (xl < S.xa - 1 || xr > S.xb + 1);
  if (__builtin_expect(kind == 0, 1)) {
    // sweep step: the next row in the direction of travel
    if (ahead) {
      // f2 >= 0: rows since the sweep's anchor, no scout sent yet;
      // f2 < 0: -(rows since the last scout) - 1
      int a1 = f1, a2 = f2 >= 0 ? f2 + 1 : f2 - 1;
      const int rows = a2 >= 0 ? a2 : -a2 - 1;
      if (__builtin_expect(rows >= (a2 >= 0 ? W.scoutRows : kMinJump) && W.scoutRows > 0, 0)) {
        const ArgPtr A = opq(W.A);
        const int J = scout_jump_for(A, xr - xl + 1);
        if (a2 >= 0 || rows >= J) {
          // send a scout ahead along the run's drift, then re-anchor
          const long long rt = (long long)row + (long long)d * J;
          if (rt >= 0 && rt < N) {
            const long long drift = rows > 0 ? (center - a1) / rows : 0;
            const long long pc = center + drift * J;
            const long long adr = drift < 0 ? -drift : drift;
            const long long hw = ((long long)xr - xl) / 2 + adr * J / 4 + 32;
            long long sa = pc - hw, sb = pc + hw;
            if (sa < 0) sa = 0;
            if (sb > N - 1) sb = N - 1;
            if (sa <= sb) {
              // to the wave's ring (the shared queue while some wave is idle),
              // or to the shared queue at once on the images of positions
              // predicted heavy, whose scouts mostly land: sweeps of many
              // small images send many scouts that miss, and queuing each of
              // them at once makes the shared queue's head and tail the
              // bottleneck
              follow(W, make_task(b, (int)rt, (int)sa, (int)sb, -1, 2, d, center, J << 16),
                     kQueueOnly | ((A->scoutShare || (W.flags & kPtHeavy)) ? kShare : 0));
            }
          }
          a1 = center;
          a2 = -1;
        }
      }
      follow(W, make_task(b, row + d, xl, xr, label, 0, d, a1, a2), 0);
    }
    return past;
  }
  if (kind == 1) {
    if (row + 1 < N) follow(W, make_task(b, row + 1, xl, xr, label, 0, 1, center, 0), 0);
    if (row - 1 >= 0) follow(W, make_task(b, row - 1, xl, xr, label, 0, -1, center, 0), 0);
    return false;
  }
  if (kind == 3) {
    // a run found looking back: sweep on away from the run it was reached
    // from, and look back towards that run's row where this one reaches past it
    if (ahead) follow(W, make_task(b, row + d, xl, xr, label, 0, d, center, 0), 0);
    if (past)
      follow(W, make_task(b, row - d, xl, xr, label, 3, -d, S.xa - 1, S.xb + 1), kQueueOnly);
    return false;
  }
  // A scout landed (f1: the column of the run it was sent from, one jump
  // back; f2: that jump's length and the scouts in its chain since the last
  // leap).  The wave sends the next scout straight on at once, with the shift
  // measured over the last jump, and keeps it as its next step, so that the
  // scouts run ahead one task per jump; every leapEvery-th scout also sends a
  // leap scout leapJumps jumps ahead to the shared queue, which starts a
  // chain of its own, so that long images get many chains.  The two sweeps of
  // the new class go to the shared queue for idle waves; they start as if
  // they had just sent a scout.
  W.nScoutRuns++;
  const ArgPtr A = opq(W.A);
  const int count = f2 & 0xFFFF, prevJump = (int)((unsigned)f2 >> 16);
  const int J = scout_jump_for(A, xr - xl + 1);
  // the shift over the last jump, rescaled to this jump
  const long long shift = ((long long)center - f1) * J / (prevJump > 0 ? prevJump : J);
  const long long ash = shift < 0 ? -shift : shift;
  const int leapEvery = A->leapEvery, leapJumps = A->leapJumps;
  const int legs = leapEvery <= 0 || (count + 1) % leapEvery != 0 ? 1 : 2;
  for (int leap = 0; leap < legs && W.scoutRows > 0; leap++) {
    const long long k = leap ? leapJumps : 1;
    const long long rt = (long long)row + (long long)d * J * k;
    if (rt < 0 || rt >= N) continue;
    const long long pc = center + shift * k;
    const long long hw = ((long long)xr - xl) / 2 + ash * k / 4 + 32 * k;
    long long sa = pc - hw, sb = pc + hw;
    if (sa < 0) sa = 0;
    if (sb > N - 1) sb = N - 1;
    if (sa > sb) continue;
    // a leap's chain measures its next shift from the column expected one
    // jump before its landing row
    follow(W,
           make_task(b, (int)rt, (int)sa, (int)sb, -1, 2, d,
                     leap ? (int)(center + shift * (leapJumps - 1)) : center,
                     (J << 16) | (leap ? 0 : (count + 1) & 0xFFFF)),
           leap ? kQueueOnly | kShare : 0);
  }
  for (int e = 1; e >= -1; e -= 2)
    if (row + e >= 0 && row + e < N)
      follow(W, make_task(b, row + e, xl, xr, label, 0, e, center, -1), kShare);
  return false;
}

// ---------------------------------------------------------------------------
// Fill
// ---------------------------------------------------------------------------
// The constants of batch point b, kept while the wave stays on it.
__device__ __forceinline__ void load_position(Worker& W, int b) {
  const ArgPtr A = opq(W.A);
  flush_acc(W);  // under the old position's profile
  W.accLabel = -1;
  W.curB = b;
  const int ln = __lane_id();
  const double pc = A->points[(size_t)b * kPointRec + (ln < kPointRec ? ln : 0)];
  const int g = b >> 14;
  W.tab = A->htab + 2 * (size_t)uni64((long long)A->grpBase[g]);
  W.tabMask = (unsigned)uni64((long long)A->grpMask[g]);
  Ray& R = W.R;
  R.pc = pc;
  R.m1 = rl(pc, kPcM1); R.m2 = rl(pc, kPcM2); R.m3 = rl(pc, kPcM3);
  R.x1 = rl(pc, kPcX1); R.x2 = rl(pc, kPcX2); R.x3 = rl(pc, kPcX3);
  R.blx = rl(pc, kPcBlx); R.step = rl(pc, kPcStep);
  R.px = rl(pc, kPcPx); R.inv = rl(pc, kPcInv);
  W.gp = uni((int)rl(pc, kPcGp));
  W.N = uni((int)rl(pc, kPcN));
  W.flags = uni((int)rl(pc, kPcFlags));
}

// The rows of a sweep (the task in hand, kind 0) on a position whose rows are
// fast: four rows at most, then the caller looks after the hand-off of waiting
// tasks.  This is where a fill spends its time, so it is kept apart from the
// general code: what process_task needs for scouts, seeds and look-backs would
// be live across the row loop and spill.  Further runs go to the wave's ring;
// look-backs end the call (process_task handles them at once: the images'
// other branches start there).  Leaves the sweep's next row in W.t
// (W.haveCont), for process_task (W.general) where it has to be evaluated
// exactly.  TIMED: the inserts are timed (by a call in 16; a branch at every
// insert of the one loop cost each task 1%).
template <int MODE, bool LIMB, bool TIMED>
__device__ __forceinline__ void sweep_rows(Worker& W) {
  const RowBase B = row_base(W.R);
  const int N = W.N, b = W.t.b, d = (W.t.kd & 4) ? -1 : 1;
  int row = W.t.row, xa = W.t.xa, xb = W.t.xb, label = W.t.label, f1 = W.t.f1, f2 = W.t.f2;
  W.haveCont = false;
  if (label != W.accLabel || W.accCnt >= (1u << 25)) {
    flush_acc(W);
    W.accLabel = label;
  }
  while ((unsigned)row < (unsigned)N) {
    if (__builtin_expect(!far_row(W.R, B, row), 0)) {
      if (!near_row(W.R, MODE == kRowBinary)) {
        W.general = true;
        break;
      }
    }
    RunScan Q;
    Q.steps = 0;
    scan_begin(Q, N, xa < 0 ? 0 : xa, xb > N - 1 ? N - 1 : xb, true, true);
    // f2 >= 0: rows since the sweep's anchor, no scout sent yet;
    // f2 < 0: -(rows since the last scout) - 1
    int a1 = f1, a2 = f2 >= 0 ? f2 + 1 : f2 - 1;
    bool have = false;
    int nl = 0, nr = 0;
    while (next_run_in<MODE, LIMB>(W.R, N, Q)) {
      int other = 0;
      const unsigned t0 = TIMED ? (unsigned)__builtin_amdgcn_s_memrealtime() : 0u;
      const int ins = insert_run(W.tab, W.tabMask, W.A, b, row, Q.xl, Q.xr, label, other);
      if (TIMED) {
        W.insTicks += (unsigned)__builtin_amdgcn_s_memrealtime() - t0;
        W.nTimed++;
      }
      if (__builtin_expect(ins != kInsNew, 0)) {
        if (ins == kInsFull) {
          flag_point(W.A, W.gp, kFlagHashFull);
        } else {
          W.nDup++;
          unite(opq(W.A)->lparent, label, other);
        }
        continue;
      }
      W.nIns++;
      W.accCnt += Q.cnt;
      if (LIMB) W.accBits += Q.acc;
      if (__builtin_expect(Q.xl <= 1 || Q.xr >= N - 2, 0)) flag_point(W.A, W.gp, kFlagEdge);
      if (!have) {
        have = true;
        nl = Q.xl;
        nr = Q.xr;
      } else {
        const int r = opq(row) + d;
        if ((unsigned)r < (unsigned)N)
          ring_put(W, make_task(b, r, Q.xl, Q.xr, label, 0, d, a1, a2));
      }
      if (__builtin_expect(Q.xl < xa - 1 || Q.xr > xb + 1, 0)) {
        // the run reaches past its parent and the parent's bounding misses
        const int r = opq(row) - d;
        if ((unsigned)r < (unsigned)N)
          put_back(W, make_task(b, r, Q.xl, Q.xr, label, 3, -d, xa - 1, xb + 1));
      }
      // a flush in time: at most 2^26 pixels, whose integers stay below 2^62
      if (__builtin_expect(W.accCnt >= (1u << 25), 0)) flush_acc(W);
      if (__builtin_expect(W.lcount > kLocalCap - kRoom, 0)) hand_off(W, 0);
    }
    W.steps += Q.steps;
    W.nTasks++;
    if (!have) break;
    const int rows = a2 >= 0 ? a2 : -a2 - 1;
    if (__builtin_expect(rows >= (a2 >= 0 ? W.scoutRows : kMinJump) && W.scoutRows > 0, 0)) {
      const ArgPtr A = opq(W.A);
      const int xl = opq(nl), xr = opq(nr), r0 = opq(row), n = opq(N);
      const int J = scout_jump_for(A, xr - xl + 1);
      if (a2 >= 0 || rows >= J) {
        // send a scout ahead along the run's drift, then re-anchor
        const int center = (int)(((unsigned)xl + (unsigned)xr) / 2);
        const long long rt = (long long)r0 + (long long)d * J;
        if (rt >= 0 && rt < n) {
          const long long drift = rows > 0 ? (center - a1) / rows : 0;
          const long long pc = center + drift * J;
          const long long adr = drift < 0 ? -drift : drift;
          const long long hw = ((long long)xr - xl) / 2 + adr * J / 4 + 32;
          long long sa = pc - hw, sb = pc + hw;
          if (sa < 0) sa = 0;
          if (sb > n - 1) sb = n - 1;
          // to the wave's ring (the pool while some wave is idle), or to the
          // pool at once on the images of positions predicted heavy, whose
          // scouts mostly land: sweeps of many small images send many scouts
          // that miss, and queuing each of them at once makes the queues the
          // bottleneck
          if (sa <= sb)
            follow(W, make_task(b, (int)rt, (int)sa, (int)sb, -1, 2, d, center, J << 16),
                   kQueueOnly | ((A->scoutShare || (W.flags & kPtHeavy)) ? kShare : 0));
        }
        a1 = center;
        a2 = -1;
      }
    }
    row += d;
    xa = nl;
    xb = nr;
    f1 = a1;
    f2 = a2;
    if ((W.nTasks & 3) == 0 || W.nOut + W.nBack > 0) {
      W.haveCont = (unsigned)row < (unsigned)N;
      break;
    }
  }
  W.t.row = row;
  W.t.xa = xa;
  W.t.xb = xb;
  W.t.f1 = f1;
  W.t.f2 = f2;
}

template <int MODE>
__device__ __forceinline__ void sweep_call(Worker& W) {
  const bool limb = (W.flags & kPtLimb) != 0;
  if (__builtin_expect(W.nTasks % 64 < 4, 0))
    limb ? sweep_rows<MODE, true, true>(W) : sweep_rows<MODE, false, true>(W);
  else
    limb ? sweep_rows<MODE, true, false>(W) : sweep_rows<MODE, false, false>(W);
}

// Processes the task in hand and the look-backs recorded meanwhile (up to two;
// the others are queued): the task's row, in one piece or in two around known
// pixels, then each look-back the same way.  The follow-up kept for this wave
// (if any) is left in W.t / W.haveCont.  With backsOnly, the look-backs that
// sweep_rows recorded, leaving W.t / W.haveCont as they are (with nothing in
// hand, the first follow-up is kept).
__device__ __forceinline__ void process_task(Worker& W, bool backsOnly) {
  const Task t = W.t;
  const int kind0 = backsOnly ? 3 : t.kd & 3;
  Scan S;
  S.row = -1;
  int taken = 0;
  W.general = false;
  W.landed = false;
  if (!backsOnly) {
    W.haveCont = false;
    if (t.b != W.curB) load_position(W, t.b);
    S.kind = kind0;
    S.dir = (t.kd & 4) ? -1 : 1;
    S.row = t.row;
    S.label = t.label;
    S.xa = t.xa;
    S.xb = t.xb;
    S.k1 = S.kind == 3 ? t.f1 : 0;
    S.k2 = S.kind == 3 ? t.f2 : -1;
    if ((unsigned)t.row >= (unsigned)W.N) return;
    if (__builtin_expect(S.kind == 1 && (unsigned)t.xa > (unsigned)(W.N - 1), 0)) {
      flag_point(W.A, W.gp, kFlagEdge);  // seed column outside the grid
      return;
    }
  }
  const bool limb = (W.flags & kPtLimb) != 0;
  while (true) {
    if (S.row < 0) {
      if (taken >= W.nBack) break;
      const Task lb = lanes_task(*task_int(&W.back[taken], W.spare));
      taken++;
      S.kind = 3;
      S.dir = (lb.kd & 4) ? -1 : 1;
      S.row = lb.row;
      S.label = lb.label;
      S.xa = lb.xa;
      S.xb = lb.xb;
      S.k1 = lb.f1;
      S.k2 = lb.f2;
    }
    set_row(W.R, W.flags, S.row);
    const int N = W.N;
    const int lo = S.xa < 0 ? 0 : S.xa, hi = S.xb > N - 1 ? N - 1 : S.xb;
    const bool known = S.k1 <= S.k2;
    for (int side = 0; side < (known ? 2 : 1); side++) {
      int s = lo, e = hi;
      bool extL = true, extR = true;
      if (__builtin_expect(known, 0)) {
        if (side == 0) {
          e = hi < S.k1 - 1 ? hi : S.k1 - 1;
          extR = hi < S.k1 - 1;
        } else {
          s = lo > S.k2 + 1 ? lo : S.k2 + 1;
          extL = lo > S.k2 + 1;
        }
      }
      if (s > e) continue;
      RunScan Q;
      Q.steps = 0;
      scan_begin(Q, N, s, e, extL, extR);
      while (next_run(W.R, N, limb, Q)) {
        if (__builtin_expect(W.nOut > kOutCap - 4 || W.lcount > kLocalCap - kRoom, 0))
          hand_off(W, 0);
        int label = 0;
        if (__builtin_expect(handle_run(W, S, t.f1, t.f2, Q.xl, Q.xr, Q.cnt, Q.acc, label), 0)) {
          put_back(W, make_task(W.curB, S.row - S.dir, Q.xl, Q.xr, label, 3, -S.dir, S.xa - 1,
                                S.xb + 1));
        }
      }
      W.steps += Q.steps;
    }
    S.row = -1;
  }
  W.nBack = 0;
  if (__builtin_expect(kind0 == 2, 0)) {
    W.nScout++;
    const int f2 = opq(t.f2);
    const int J = (int)((unsigned)f2 >> 16), count = f2 & 0xFFFF;
    const int J2 = J / 2;
    if (!W.landed && J2 >= kMinJump && opq(W.A)->scoutRetry) {
      // A scout that found nothing (its chain's prediction failed, or the
      // image ends before its row): a retry from the same origin, half the
      // jump ahead, with a window of the same width about the midpoint of the
      // origin column and the failed window's centre.
      const int N = opq(W.N), xa = opq(t.xa), xb = opq(t.xb);
      const int dir = (t.kd & 4) ? -1 : 1;
      const long long rt = (long long)t.row - (long long)dir * (J - J2);
      const long long pc = ((long long)xa + xb) / 2;
      const long long c2 = t.f1 + (pc - t.f1) / 2;
      const long long hw = ((long long)xb - xa) / 2;
      long long sa = c2 - hw, sb = c2 + hw;
      if (sa < 0) sa = 0;
      if (sb > N - 1) sb = N - 1;
      if (rt >= 0 && rt < N && sa <= sb)
        follow(W, make_task(t.b, (int)rt, (int)sa, (int)sb, -1, 2, dir, t.f1, (J2 << 16) | count),
               0);
    }
  }
}

// The manager wave of a fill workgroup.  It keeps the group's pool fed while
// workers are idle (seed tasks first, then tasks that other groups queued in
// the global ring), queues some of a large pool for other groups while any
// group is idle, and runs the end test.  A group joins the global active
// count when it starts, before it takes any task; a group whose `pending`
// count reads 0 with the seed list used up leaves the count and polls the
// global ring, and rejoins the count before it takes tasks from the ring, so
// a task is never queued while the count reads 0.  The fill is over when the
// count is 0 and the ring is empty: no group then holds work, and a group
// that starts later (its compute unit was busy with other kernels) finds
// none and leaves.  So the groups need not all be resident at once.
__device__ __forceinline__ void fill_manager(const FillArgs& A, GroupPool* G, long long t0,
                             unsigned long long& polls) {
  const int ln = __lane_id();
  if (ln == 0) {
    afaddi(A.active, 1);
    mem_order();
  }
  bool counted = true;  // the group is in A.active
  int backoff = 0;
  unsigned long long loops = 0;
  long long nextShareCheck = 0, nextQueueCheck = 0;
  bool othersIdle = false;
  bool seedsLeft = true;  // the batch's seed list is handed out front to back, once
  Task t = make_task(0, 0, 0, 0, 0, 0, 1, 0, 0);
  while (true) {
    loops++;
    const long long now = (long long)__builtin_amdgcn_s_memrealtime();
    if (now - t0 > A.timeLimitTicks) {
      if (ln == 0) atomicExch(A.abortFlag, 1);
      break;
    }
    int pend = 0, cnt = 0;
    if (ln == 0) {
      pend = lds_ld(&G->pending);
      cnt = lds_ld(&G->count);
    }
    pend = uni(pend);
    cnt = uni(cnt);
    const int idle = kWorkers - (pend - cnt);  // workers without work
    if (pend == 0) {
      // the group is idle: seed tasks, else the global ring
      int k = seedsLeft ? claim_seeds(A, t, kFeedMax) : 0;
      seedsLeft = k > 0;
      if (k > 0) {
        pool_add_all(A, G, t, 0, k, t0 + A.timeLimitTicks);
        continue;
      }
      if (counted) {
        if (ln == 0) {
          mem_order();
          afaddi(A.active, -1);
        }
        counted = false;
      }
      polls++;
      if (backoff < A.pollBackoff) backoff++;
      for (int s = 0; s < (1 << backoff); s++) __builtin_amdgcn_s_sleep(16);
      int abortNow = 0, act = 1;
      unsigned long long qh = 0, qt = 0;
      if (ln == 0) {
        if ((polls & 3) == 0) {
          act = aldi(A.active);
          abortNow = aldi(A.abortFlag);
          mem_order();
        }
        qh = ald(A.qhead);
        qt = ald(A.qtail);
      }
      if (uni(abortNow)) break;
      act = uni(act);
      qh = uni64(qh);
      qt = uni64(qt);
      if (qt > qh) {
        // rejoin before taking tasks
        if (ln == 0) {
          afaddi(A.active, 1);
          mem_order();
        }
        counted = true;
        k = q_pop_lanes(A, t, kFeedMax);
        if (k > 0) {
          pool_add_all(A, G, t, 0, k, t0 + A.timeLimitTicks);
          backoff = 0;
        } else {
          if (ln == 0) afaddi(A.active, -1);
          counted = false;
        }
      } else if (act <= 0) {
        break;  // no group holds work and nothing is queued
      }
      continue;
    }
    backoff = 0;
    if (idle > cnt) {
      // workers are waiting: seed tasks, else (at most every ~2 us) the ring
      const int want = idle - cnt + 2 < kFeedMax ? idle - cnt + 2 : kFeedMax;
      int k = seedsLeft ? claim_seeds(A, t, want) : 0;
      seedsLeft = k > 0;
      if (k == 0 && now >= nextQueueCheck) {
        nextQueueCheck = now + 200;
        k = q_pop_lanes(A, t, want);
      }
      if (k > 0) {
        pool_add_all(A, G, t, 0, k, t0 + A.timeLimitTicks);
        continue;
      }
    } else {
      // while some other group is idle (the global count is read at most
      // every ~5 us), the pool's tasks go on to the global ring, and the
      // workers keep the pool topped up
      if (now >= nextShareCheck) {
        nextShareCheck = now + 500;
        int act = 0;
        if (ln == 0) act = aldi(A.active);
        othersIdle = uni(act) < A.nGroups;
        if (ln == 0) lds_st(&G->hungry, othersIdle ? 1 : 0);
      }
      if (othersIdle && cnt >= 2) {
        const int n = cnt / 2 < kDonateMax ? cnt / 2 : kDonateMax;
        const int k = pool_remove_lanes(G, t, n);
        const int q = q_push_lanes(A, t, k);
        if (q < k) pool_add_all(A, G, t, q, k, t0 + A.timeLimitTicks);  // ring full: keep the rest
        if (q > 0) continue;
      }
    }
    __builtin_amdgcn_s_sleep(4);
  }
  if (ln == 0) lds_st(&G->done, 1);
}

// Worker waves take work from their own ring, then from the group's pool;
// a worker that finds neither is idle and waits on the pool until the
// manager ends the fill.
__global__ void __launch_bounds__(kFillThreads) fill_kernel(FillArgs A) {
  __shared__ Task rings[kWorkers][kLocalCap];
  __shared__ GroupPool pool;
  __shared__ Task outs[kWorkers][kOutCap];
  __shared__ Task backs[kWorkers][2];
  __shared__ int spare[kWorkers][64];
  __shared__ unsigned long long sums[kFillStats];
  __shared__ int left;  // workers that have not added theirs
  const int ln = __lane_id();
  const int wave = uni((int)(threadIdx.x / 64));
  const long long t0 = (long long)__builtin_amdgcn_s_memrealtime();
  GroupPool* G = &pool;
  if (threadIdx.x == 0) {
    G->lock = 0;
    G->pending = 0;
    G->head = 0;
    G->count = 0;
    G->done = 0;
    G->hungry = 0;
    left = kWorkers;
  }
  if (threadIdx.x < kFillStats) sums[threadIdx.x] = 0;
  __syncthreads();
  if (wave == 0) {
    unsigned long long polls = 0;
    fill_manager(A, G, t0, polls);
    if (ln == 0) atomicAdd(&A.stats[6], polls);
    return;
  }
  Worker W;
  W.A = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
  W.scoutRows = A.scoutRows;
  W.G = G;
  W.ring = rings[wave - 1];
  W.out = outs[wave - 1];
  W.nOut = 0;
  W.back = backs[wave - 1];
  W.nBack = 0;
  W.spare = spare[wave - 1];
  W.lhead = 0;
  W.lcount = 0;
  W.general = false;
  W.haveCont = false;
  W.curB = -1;
  W.gp = W.N = W.flags = 0;
  W.tab = nullptr;
  W.tabMask = 0;
  W.accLabel = -1;
  W.accCnt = 0;
  W.accBits = 0;
  W.nTasks = W.nIns = W.nDup = W.nScout = W.nScoutRuns = W.steps = 0;
  W.insTicks = W.nTimed = 0;
  const bool newest = A.poolNewest != 0;
  unsigned idlePolls = 0;
  unsigned long long idleTicks = 0;
  bool have = false, busy = false;
  while (true) {
    if (!have && W.lcount > 0) {
      W.t = ring_pop(W);
      have = true;
    }
    if (!have && busy) {
      // own work done: a task of the pool, or idle
      flush_acc(W);
      have = pool_take(G, W.t, true, newest, W.spare);
      busy = have;
    }
    if (!have) {
      const long long ti = (long long)__builtin_amdgcn_s_memrealtime();
      bool over = false;
      while (true) {
        idlePolls++;
        __builtin_amdgcn_s_sleep(24);
        if (uni(lds_ld(&G->done))) {
          over = true;
          break;
        }
        if (uni(lds_ld(&G->count)) > 0 && pool_take(G, W.t, false, newest, W.spare)) break;
        if ((idlePolls & 255) == 0 &&
            (long long)__builtin_amdgcn_s_memrealtime() - t0 >
                opq(W.A)->timeLimitTicks + 100000000ll) {
          // the manager ends the fill at the time limit; this bound only
          // guards against a manager that never does
          over = true;
          break;
        }
      }
      idleTicks += (unsigned long long)((long long)__builtin_amdgcn_s_memrealtime() - ti);
      if (over) break;
      busy = true;
    }
    if ((W.t.kd & 3) == 0) {
      if (W.t.b != W.curB) load_position(W, W.t.b);
      switch (W.flags & (kPtFast | kPtBinary)) {
        case kPtFast:
          sweep_call<kRowTriple>(W);
          break;
        case kPtFast | kPtBinary:
          sweep_call<kRowBinary>(W);
          break;
        default: W.general = true;
      }
    } else {
      W.general = true;
    }
    if (W.general || W.nBack > 0) {
      const bool backs = !W.general;
      W.nTasks += backs ? 0 : 1;
      process_task(W, backs);
    }
    have = W.haveCont;
    // the out buffer's tasks to the pool; every fourth task, waiting ones to
    // idle workers of the group, and while other groups are idle enough to
    // keep the pool topped up for them
    int give = 0;
    if ((W.nTasks & 3) == 0 && W.lcount > 0) {
      const int pend = uni(lds_ld(&G->pending)), cnt = uni(lds_ld(&G->count));
      const int idle = kWorkers - (pend - cnt);
      if (idle > cnt || (uni(lds_ld(&G->hungry)) && cnt < kPoolShare)) give = W.lcount > 2 ? 2 : 1;
    }
    if (W.nOut + give > 0) hand_off(W, give);
    if ((W.nTasks & 255) == 0) {
      const long long now = (long long)__builtin_amdgcn_s_memrealtime();
      const ArgPtr a = opq(W.A);
      if (now - t0 > a->timeLimitTicks) {
        store32_lane0(a->abortFlag, 1);
        break;
      }
      if (uni(aldi(a->abortFlag))) break;
    }
  }
  flush_acc(W);
  const unsigned long long busyTicks =
      (unsigned long long)((long long)__builtin_amdgcn_s_memrealtime() - t0) - idleTicks;
  // The workgroup's counters go to the launch's from its last worker: 3840
  // waves that add to one address take turns (a 17-point curve 1.62 -> 1.37 ms
  // with ten counters added by 256).
  if (ln == 0) {
    const unsigned long long v[kFillStats] = {W.nTasks, 64ull * W.steps, W.nIns, W.nDup, busyTicks,
                                              W.insTicks, idlePolls, 1, W.nScout,
                                              W.nScoutRuns, W.nTimed};
    for (int k = 0; k < kFillStats; k++) lds_add(&sums[k], v[k]);
    if (lds_add(&left, -1) == 1)
      for (int k = 0; k < kFillStats; k++) atomicAdd(&A.stats[k], lds_add(&sums[k], 0ull));
  }
}

// Workgroups of fill_kernel that can be resident on the device at once (a
// larger launch is correct, its surplus groups run after the others).
int fill_resident_workgroups() {
  int perCu = 0, dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, fill_kernel, kFillThreads, 0) !=
      hipSuccess)
    return 0;
  return perCu * cus;
}

int launch_fill(const FillArgs& a, int nWorkgroups, hipStream_t s) {
  hipLaunchKernelGGL(fill_kernel, dim3(nWorkgroups), dim3(kFillThreads), 0, s, a);
  return (int)hipGetLastError();
}

__global__ void clear_u64_kernel(unsigned long long* p, unsigned long long n, unsigned long long v) {
  for (unsigned long long i = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; i < n;
       i += (unsigned long long)gridDim.x * blockDim.x)
    p[i] = v;
}

int launch_clear_u64(unsigned long long* p, unsigned long long n, unsigned long long v,
                     hipStream_t s) {
  if (n == 0) return 0;
  unsigned long long blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(clear_u64_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
  return (int)hipGetLastError();
}

// Resets the run table (word0 = 0, word1 = ~0), labels, queue slots and
// counters before a fill launch.  A plain kernel (no memset nodes), so that
// the sequence can be captured in a graph.
__global__ void fill_reset_kernel(FillArgs A) {
  const unsigned long long tid = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x;
  const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
  for (unsigned long long i = tid; i < A.htabEntries; i += stride) {
    A.htab[2 * i] = 0;
    A.htab[2 * i + 1] = kEmpty1;
  }
  for (unsigned long long i = tid; i < (unsigned long long)A.labelCap; i += stride) {
    A.lparent[i] = (int)i;
    A.lpoint[i] = i < (unsigned long long)A.nBatch ? (int)i : -1;
    A.lcount[i] = 0;
    A.lsum[2 * i] = 0;
    A.lsum[2 * i + 1] = 0;
  }
  for (unsigned long long i = tid; i < A.qcap; i += stride) A.qseq[i] = i;
  if (tid == 0) {
    *A.qhead = 0;
    *A.qtail = 0;
    *A.active = 0;
    *A.seedNext = 0;
    *A.labelNext = A.nBatch;
    *A.abortFlag = 0;
    for (int k = 0; k < kFillStats; k++) A.stats[k] = 0;
  }
}

int launch_fill_reset(const FillArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(fill_reset_kernel, dim3(2048), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}

// Adds every label whose class holds the reference-seed label of its point
// to that point's totals.
__global__ void resolve_kernel(FillArgs A, int nLabels, unsigned long long* ptCount,
                               unsigned long long* ptSum) {
  const int L = blockIdx.x * blockDim.x + threadIdx.x;
  if (L >= nLabels) return;
  const int b = A.lpoint[L];
  if (b < 0 || b >= A.nBatch) return;
  if (A.lcount[L] == 0) return;
  const int r = find_root(A.lparent, L);
  const int rb = find_root(A.lparent, b);
  if (r != rb) return;
  atomicAdd(&ptCount[b], A.lcount[L]);
  // the label's split total into the point's, word by word (the point's
  // total is hi * 2^32 + lo like the labels'; its low word may carry past
  // 2^64 only after 2^32 labels)
  const unsigned long long lo = A.lsum[2 * (size_t)L], hi = A.lsum[2 * (size_t)L + 1];
  atomicAdd(&ptSum[2 * (size_t)b], lo);
  if (hi) atomicAdd(&ptSum[2 * (size_t)b + 1], hi);
}

int launch_resolve(const FillArgs& a, int nLabels, unsigned long long* ptCount,
                   unsigned long long* ptSum,
                   hipStream_t s) {
  if (nLabels <= 0) return 0;
  hipLaunchKernelGGL(resolve_kernel, dim3((nLabels + 255) / 256), dim3(256), 0, s, a, nLabels,
                     ptCount, ptSum);
  return (int)hipGetLastError();
}

}  // namespace tl
