// Temporally blocked 2D Yee step for gfx950 (TMz, TEz and the studies' lossy
// TMz): TB time steps per launch on register-resident tiles.
//
// A block of W waves holds an extended tile of W*K planes (x) by 64 rows (y,
// one per lane): wave w owns K planes, every lane its row of those planes.
// The tile's own cells are the inner (W*K - 2 TB) x (64 - 2 TB); the TB-cell
// ghost frame on every side is loaded and stepped like the rest and discarded:
// each step (E then H) moves the region that depends on values outside the
// tile one cell inwards from each side, so after TB steps the inner cells are
// exact.  The launch reads field/psi set ((n0 / TB) & 1) and writes the inner
// cells' state to the other set, so no tile races another.
//
// Per step the only exchanges are the y neighbours (DPP lane shifts) and,
// between waves, one plane before the E and one before the H half-step through
// LDS.  Every half-step updates the planes that do not need the exchanged
// plane between the LDS write and the barrier, so the waves' skew is absorbed
// there.
//
// What bounds it: instruction issue.  A field value passes through HBM once
// per TB steps, so the kernel is lean in the inner loop instead:
//   - the class of a wave (not of a tile) picks one of four step bodies:
//     planes outside the x slabs, the source and the capture planes with all
//     rows outside the y slabs (bulk curls alone, 11 vector instructions per
//     cell and step); the same planes with y-slab rows (the y psi terms run on
//     every lane and are selected, as the update ranges are); planes in the x
//     slabs or at the x limits; planes with the source or a capture;
//   - the per-plane 1/kappa stay in scalar registers over the launch.
//
// The arithmetic is written with explicit fused multiply-adds, the ones the
// two-kernel forms (k_*_e2 / k_*_h2, k_tmzl_e / k_tmzl_h) compile to, so every
// shape and every class gives the same bits, infinite and NaN ones included.
//
// Field monitors.  The running DFTs of the study drivers (one per field, over
// any box) ride along: their sums of the wave's cells sit in registers over
// the launch, each step folded as k_monitor folds it (product and sum in
// double, rounded to T), so a whole-plane phasor costs one read and one write
// of its sums per 8 steps instead of a kernel per step.  us per step, two
// kernels and the monitor kernel / blocked: TEz study 4170 x 430 with two
// planes 36.8 / 10.0 (11.2 with a branch per cell round the sums' loads), lossy
// TMz 2787 x 430 with three 33.2 / 10.9, bound by the conversions and FP64
// operations of the fold.
#pragma once
#include "fdtd_kernels.h"

namespace oidt {

// A uniform / per-lane value the compiler may not connect with its origin: what
// is derived from it is formed again after a long stretch of code instead of
// being kept in registers across it.
__device__ __forceinline__ int opaque_uniform(int v) {
  asm volatile("" : "+s"(v));
  return v;
}
template <typename U>
__device__ __forceinline__ U opaque_value(U v) {
  asm volatile("" : "+v"(v));
  return v;
}

// p = b * p + t in place (the compiler otherwise accumulates into t and copies
// it back to p in every step).
__device__ __forceinline__ void psi_step(float& p, float b, float t) {
  asm("v_fma_f32 %0, %1, %0, %2" : "+v"(p) : "v"(b), "v"(t));
}
__device__ __forceinline__ void psi_step(double& p, double b, double t) {
  asm("v_fma_f64 %0, %1, %0, %2" : "+v"(p) : "v"(b), "v"(t));
}

// The fields by their role in the step:
//   A  exchanged before E (TMz Hy, TEz Hz): E reads it at i+1
//   B  exchanged after E  (TMz Ez, TEz Ey): H reads it at i-1
//   C  read at j+-1 only  (TMz Hx, TEz Ex)
// px / py are the E psi of the x / y slabs (TMz ez_x, ez_y; TEz ey_x, ex_y),
// qx / qy the H psi (TMz hy_x, hx_y; TEz hz_x, hz_y).
template <int SCH>
struct Blocked2d;
template <>
struct Blocked2d<SCHEME_TMZ> {
  static constexpr int A = F_HY, B = F_EZ, C = F_HX;
  static constexpr int PX = F_EZ, PY = F_EZ, QX = F_HY, QY = F_HX;   // psi components
  static constexpr int SRC = F_EZ;
};
// The lossy TMz form differences the other way round: E reads A at i-1, H
// reads B at i+1.
template <>
struct Blocked2d<SCHEME_TMZ_LOSSY> : Blocked2d<SCHEME_TMZ> {};
template <>
struct Blocked2d<SCHEME_TEZ> {
  static constexpr int A = F_HZ, B = F_EY, C = F_EX;
  static constexpr int PX = F_EY, PY = F_EX, QX = F_HZ, QY = F_HZ;
  static constexpr int SRC = F_HZ;
};

// CPML cells of the lossy TMz form (k_tmzl_e, k_tmzl_h): row and coefficient
// are the distance from the grid edge.
__device__ __forceinline__ int slab_e_lossy(int x, int e, int N, int& d, int& ci) {
  if (x < N) { d = ci = x; return 0; }
  if (e - x < N) { d = ci = e - x; return 1; }
  return -1;
}
__device__ __forceinline__ int slab_h_lossy(int x, int e, int N, int& d, int& ci) {
  if (x >= 1 && x < N) { d = ci = x; return 0; }
  if (e - 1 - x >= 1 && e - 1 - x < N) { d = ci = e - 1 - x; return 1; }
  return -1;
}

// Roles with a monitor, as bits of a kernel's MON.
enum : int { MON_A = 1, MON_B = 2, MON_C = 4 };

// MON: the roles a run's monitors may take (0: the kernel ignores monitors);
// smon[slot]: first monitor of the run in `mons` and their number, at most one
// per field.
template <typename T, int SCH, int TB, int W, int K, int MON>
__device__ __forceinline__ void blocked_step_2d(const Slot<T>* __restrict__ slots, const int4* __restrict__ tiles,
                                                int ntiles, int tstep, const Monitor<T>* __restrict__ mons,
                                                const int2* __restrict__ smon) {
  using R = Blocked2d<SCH>;
  constexpr bool tm = SCH != SCHEME_TEZ, lossy = SCH == SCHEME_TMZ_LOSSY;
  constexpr int P = W * K;                           // planes of the extended tile
  constexpr int TX = P - 2 * TB, TY = 64 - 2 * TB;   // inner cells of a tile
  static_assert(TX > 0 && TY > 0 && kChunk % TB == 0, "blocking depth");
  constexpr unsigned es = sizeof(T);
  __shared__ T xA[W][64];   // A of each wave's first plane, before E
  __shared__ T xB[W][64];   // B of each wave's last plane, after E
  const int lane = threadIdx.x;
  const int w = wave_id();
  // The chunk's first step is a multiple of kChunk and kChunk / TB is even:
  // the set a launch reads follows from its place in the chunk.
  const bool odd = ((tstep / TB) & 1) != 0;
  for (int tt = xcd_block(); tt < ntiles; tt += gridDim.x) {
    const int4 tl = tiles[tt];
    const Slot<T>& s = slots[tl.x];
    // Everything the loads below need, requested together: a launch over a
    // small grid is a chain of dependent loads, so the branch must not
    // split it.
    const int n0 = s.base + tstep, nt = s.nt, active = s.active;
    const int nx = s.nx, ny = s.ny, N = s.N, ib = s.ib, ie = s.ie, jb = s.jb, je = s.je;
    const T* const gA = odd ? s.f2[R::A] : s.f[R::A];
    const T* const gB = odd ? s.f2[R::B] : s.f[R::B];
    const T* const gC = odd ? s.f2[R::C] : s.f[R::C];
    const uint8_t* const gm = s.mat;
    const T* const ike0 = s.ike[0];
    const T* const ike1 = s.ike[1];
    const T* const ikh0 = s.ikh[0];
    const T* const ikh1 = s.ikh[1];
    asm volatile("" ::"s"(n0), "s"(nt), "s"(active), "s"(nx), "s"(ny), "s"(N), "s"(ib), "s"(ie), "s"(jb), "s"(je),
                 "s"(gA), "s"(gB), "s"(gC), "s"(gm), "s"(ike0), "s"(ike1), "s"(ikh0), "s"(ikh1));
    if (!active || n0 >= nt) continue;      // uniform over the block
    const int nsteps = min(TB, nt - n0);
    const int i0 = tl.y, j0 = tl.z;               // first inner cell
    const int ib0 = i0 - TB + w * K, ib00 = ib0;  // this wave's first plane
    const int j = j0 - TB + lane;
    const bool jok = j >= 0 && j < ny;
    const int jc = min(max(j, 0), ny - 1);
    // ---- fields and material of the wave's cells, from set A.  Cells outside
    // the grid read the nearest one inside: no step updates them, and the
    // rows and planes that are updated lie at least one cell inside the grid,
    // so nothing updated reads them.
    T a[K], bf[K], c[K];
    unsigned m[K];
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const unsigned idx = (unsigned)min(max(ib0 + q, 0), nx - 1) * ny + jc;
      a[q] = ldg<T>(gA, idx * es);
      bf[q] = ldg<T>(gB, idx * es);
      c[q] = ldg<T>(gC, idx * es);
      m[q] = ldg<uint8_t>(gm, idx);
    }
    // ---- row (y-only) constants of this lane
    // update rows: TMz Ez, Hy [jb, je), Hx (jb, je); TEz Ex [jb, je), Ey and Hz
    // (jb, je); lossy TMz E [1, je), H [0, je)
    const bool yin = jok && j >= jb && j < je, yin1 = jok && (lossy || j > jb) && j < je;
    int dye = 0, cye = 0, dyh = 0, cyh = 0;
    auto se = [&](int x, int b_, int e_, int& d, int& ci) {
      return lossy ? slab_e_lossy(x, e_, N, d, ci) : slab_e(x, b_, e_, N, d, ci);
    };
    auto sh = [&](int x, int b_, int e_, int& d, int& ci) {
      return lossy ? slab_h_lossy(x, e_, N, d, ci) : slab_h(x, b_, e_, N, d, ci);
    };
    const int sye = yin ? se(j, jb, je, dye, cye) : -1;
    const int syh = yin1 ? sh(j, jb, je, dyh, cyh) : -1;
    const T ikye = yin ? ldg<T>(ike1, j * es) : T(0), ikyh = yin1 ? ldg<T>(ikh1, j * es) : T(0);
    const T bey = sye >= 0 ? s.be[cye] : T(0), cey = sye >= 0 ? s.ceo[cye] : T(0);
    const T bhy = syh >= 0 ? s.bh[cyh] : T(0), chy = syh >= 0 ? s.cho[cyh] : T(0);
    const bool has_src = s.src_field == R::SRC;
    const bool jsrc = jok && has_src && j >= s.sy0 && j < s.sy1;
    // ---- class of this wave (see above)
    const int sx0 = s.sx0, sx1 = s.sx1, port0 = s.port[0], port1 = s.port[1];
    auto meets = [&](int lo, int hi) { return ib0 < hi && ib0 + K > lo; };
    const bool ports = !lossy && s.nf > 0;   // nothing folds the captures of a run without frequencies
    const bool special = (has_src && meets(sx0, sx1)) || (ports && (meets(port0, port0 + 2) || meets(port1, port1 + 2)));
    const bool xplain = ib0 >= ib + N && ib0 + K <= ie - N && !special;
    const bool yplain = j0 - TB >= jb + N && j0 - TB + 64 <= je - N;
    // Where plane ib0 + l is updated and its x-slab cells, lane l = 0..K-1 (a
    // vector register serves all the wave's planes; the values of one plane
    // are read from its lane).  Roles: bit 0 x in [ib, ie), 1 x in (ib, ie)
    // (lossy: [0, ie)), 2 source, 3 E slab, 4 H slab, 5..8 capture at port0, port1, port0 + 1,
    // port1 + 1.  re / rh: row of the E / H psi slab, kHi added on its high
    // side.
    constexpr int kHi = 1 << 24;
    struct XCell { int f, re, rh, cxe, cxh; };
    auto xcells = [&](int l) {
      XCell x{};
      const int i = ib00 + l;
      const bool iok = i >= 0 && i < nx;
      const bool xin = iok && i >= ib && i < ie, xin1 = iok && (lossy || i > ib) && i < ie;
      const bool inner = ports && iok && i >= i0 && i < i0 + TX;
      int dxe = 0, dxh = 0;
      const int sxe = xin ? se(i, ib, ie, dxe, x.cxe) : -1;
      const int sxh = xin1 ? sh(i, ib, ie, dxh, x.cxh) : -1;
      x.re = dxe + (sxe == 1 ? kHi : 0);
      x.rh = dxh + (sxh == 1 ? kHi : 0);
      x.f = (xin ? 1 : 0) | (xin1 ? 2 : 0) | (iok && i >= sx0 && i < sx1 ? 4 : 0) | (sxe >= 0 ? 8 : 0) |
            (sxh >= 0 ? 16 : 0) | (inner && i == port0 ? 32 : 0) | (inner && i == port1 ? 64 : 0) |
            (inner && i == port0 + 1 ? 128 : 0) | (inner && i == port1 + 1 ? 256 : 0);
      return x;
    };
    auto at = [](int v, int q) { return __builtin_amdgcn_readlane(v, q); };
    // rows of the x psi: E (TMz Ez, TEz Ey) and H (TMz Hy, TEz Hz); first
    // planes of the y psi: E (TMz Ez, TEz Ex) and H (TMz Hx, TEz Hz)
    const bool yxe = tm ? yin : yin1, yxh = tm && !lossy ? yin : yin1;
    const int pye = tm ? ib : ib + 1, pyh = lossy ? 0 : pye;
    // ---- coefficients
    T cb0[K], cb1[K], kx[K], kh[K];
    // lane q loads plane q's 1/kappa; each then sits in a scalar register
    T lkx = T(0), lkh = T(0);
    if (lane < K) {
      const int i = ib0 + lane;
      const bool xin = i >= ib && i < ie, xin1 = (lossy ? i >= 0 : i > ib) && i < ie;
      lkx = xin ? ldg<T>(ike0, i * es) : T(0);
      lkh = xin1 ? ldg<T>(ikh0, i * es) : T(0);
    }
    // cb0: TMz cb (lossy CURL_H), TEz cb of Ex; cb1: TEz cb of Ey, lossy MOD_E
    constexpr int c0 = tm ? 2 : 0, c1 = lossy ? 0 : 1;
    const T v00 = s.cbv[c0][0], v01 = s.cbv[c0][1], v02 = s.cbv[c0][2], v03 = s.cbv[c0][3];
    const T v10 = s.cbv[c1][0], v11 = s.cbv[c1][1], v12 = s.cbv[c1][2], v13 = s.cbv[c1][3];
#pragma unroll
    for (int q = 0; q < K; ++q) {
      kx[q] = lane_get(lkx, q);
      kh[q] = lane_get(lkh, q);
      cb0[q] = cb_of(v00, v01, v02, v03, m[q], c0);
      cb1[q] = tm && !lossy ? T(0) : cb_of(v10, v11, v12, v13, m[q], c1);
    }
    const T db = s.db, dxT = s.dxT, dtmu = s.dtmu;
    // CLS 0: anything; 1: bulk only; 2: no x slab or limit, source or capture;
    // 3: no source or capture.
    auto tile = [&](auto cls) {
      constexpr int CLS = decltype(cls)::value;
      constexpr bool kX = CLS == 0 || CLS == 3;    // x slabs and limits
      constexpr bool kSp = CLS == 0;               // source and capture
      // ---- source waveform (lane t: step n0 + t) and capture ring
      const bool jcap = kSp && lane >= TB && lane < TB + TY && j >= s.wy0 && j <= s.wy1;
      const T jvl = kSp && has_src && lane < nsteps ? s.jsrc[n0 + lane] : T(0);
      OIDT_GLOBAL T* const ring = s.ring;
      const int pcells = s.pcells, nplanes = s.nplanes;
      const int cw = j - s.wy0;
      // ---- psi of the slabs this wave can meet
      T px[K], py[K], qx[K], qy[K];
#pragma unroll
      for (int q = 0; q < K; ++q) px[q] = py[q] = qx[q] = qy[q] = T(0);
      OIDT_GLOBAL T* const* psiA = odd ? s.psi2 : s.psi;
      if (CLS != 1 && !yplain) {
        // low-side array plus the side's byte distance: 32-bit lane offsets
        const T* gpy = psiA[psi_id(R::PY, 1, 0)];
        const T* gqy = psiA[psi_id(R::QY, 1, 0)];
        const unsigned oe = (unsigned)dye * es + (sye == 1 ? s.psi_hi[1] : 0u);
        const unsigned oh = (unsigned)dyh * es + (syh == 1 ? s.psi_hi[1] : 0u);
#pragma unroll
        for (int q = 0; q < K; ++q) {
          const int i = ib0 + q;
          if (i >= pye && i < ie && sye >= 0) py[q] = ldg<T>(gpy, (unsigned)(i * N) * es + oe);
          if (i >= pyh && i < ie && syh >= 0) qy[q] = ldg<T>(gqy, (unsigned)(i * N) * es + oh);
        }
      }
      // x-slab coefficients, lane q plane q
      T lbe = T(0), lce = T(0), lbh = T(0), lch = T(0);
      int lf = 0;
      if (kX) {
        const XCell x = xcells(lane);
        lf = x.f;
        lbe = (lf & 8) ? s.be[x.cxe] : T(0);
        lce = (lf & 8) ? s.ceo[x.cxe] : T(0);
        lbh = (lf & 16) ? s.bh[x.cxh] : T(0);
        lch = (lf & 16) ? s.cho[x.cxh] : T(0);
#pragma unroll
        for (int q = 0; q < K; ++q) {
          const int f = at(x.f, q), re = at(x.re, q), rh = at(x.rh, q);
          if ((f & 8) && yxe) px[q] = ldg<T>(psiA[psi_id(R::PX, 0, re >= kHi)], (unsigned)((re & (kHi - 1)) * ny + jc) * es);
          if ((f & 16) && yxh) qx[q] = ldg<T>(psiA[psi_id(R::QX, 0, rh >= kHi)], (unsigned)((rh & (kHi - 1)) * ny + jc) * es);
        }
      }
      // A cell outside a component's update range keeps its value by a select in
      // every step where an updated neighbour along x or y reads it (TMz A / C,
      // TEz A / A, lossy TMz B / B) and on the source planes (TMz B, TEz A: the
      // source drives cells outside the ranges too).  The other cells outside a
      // range hold zero and are read by nothing that is updated: the steps let
      // them go, captures and the final store take the zero, and monitors fold
      // nothing there.  (A zero factor instead of the selects also keeps a
      // finite cell, but turns it NaN beside an infinite neighbour.  A 600 x 240
      // FP64 solve, the case with the largest difference: 8.44 ms with zero
      // factors, 8.54 so.)
      constexpr bool sxA = !lossy, syA = !tm;
      constexpr bool sxB = lossy, syB = lossy;
      constexpr bool sxC = false, syC = tm && !lossy;
      // update planes (bits of the x flags) and rows
      constexpr unsigned upA = 2u, upB = 1u, upC = tm && !lossy ? 1u : 2u;
      const bool yA = yxh, yB = yxe, yC = tm ? yin1 : yin;
      auto updates = [&](bool sx, unsigned xin, bool sy, bool yr) {
        return (!kX || !sx || xin != 0u) && (CLS == 1 || !sy || yr);
      };
      // With few planes the flags, masks and slab coefficients stay in scalar
      // registers over the steps; with many they are formed again in every
      // step (they would spill).
      auto flags = [&](int q) -> unsigned {
        if constexpr (!kX) return 3u;
        else return (unsigned)at(K <= 2 ? lf : opaque_value(lf), q);
      };
      auto coef = [&](const T& v, int q) { return lane_get(K <= 2 ? v : opaque_value(v), q); };
      auto cap = [&](int t, int plane, T v) {
        ring[((size_t)(tstep + t) * nplanes + plane) * pcells + cw] = v;
      };
      // E half-step of plane q; up: A of plane q + 1 (lossy: q - 1)
      auto e_half = [&](int q, T up, int t, T jv) {
        const unsigned f = flags(q);
        const T dx = lossy ? a[q] - up : up - a[q];
        if constexpr (lossy) {
          const T dy = lane_prev(c[q]) - c[q];
          const T ch = cb0[q];
          T e = fmadd(cb1[q], bf[q], ch * fmadd(dy, ikye, dx * kx[q]));
          if (kSp && (f & 4u)) e = jsrc ? e - jv : e;   // (the box lies inside the update range)
          if (CLS != 1) {
            const T chdx = ch * dxT;
            if (kX && (f & 8u)) {
              px[q] = fmadd(coef(lce, q), dx, coef(lbe, q) * px[q]);
              e = fmadd(chdx, px[q], e);
            }
            py[q] = fmadd(cey, dy, bey * py[q]);
            e = sye >= 0 ? fmadd(chdx, py[q], e) : e;
          }
          bf[q] = updates(sxB, f & upB, syB, yB) ? e : bf[q];
        } else if constexpr (tm) {
          const T dy = lane_next(c[q]) - c[q];
          const T cb = cb0[q];
          T e = fmadd(cb, fmadd(dx, kx[q], -(dy * ikye)), bf[q]);
          const T kept = kSp && jsrc ? bf[q] - jv : bf[q];
          if (kSp && (f & 4u)) e = jsrc ? e - jv : e;
          if (kX && (f & 8u)) {
            px[q] = fmadd(coef(lbe, q), px[q], coef(lce, q) * dx);
            e = fmadd(cb, px[q], e);
          }
          if (CLS != 1) {
            psi_step(py[q], bey, cey * dy);
            e = sye >= 0 ? fmadd(-cb, py[q], e) : e;
          }
          if (kSp && (f & 4u)) e = (f & upB) && yB ? e : kept;
          bf[q] = e;
        } else {
          const T dy = lane_next(a[q]) - a[q];
          T ex = fmadd(cb0[q] * dy, ikye, c[q]);
          T ey = fmadd(cb1[q] * -dx, kx[q], bf[q]);
          if (CLS != 1) {
            psi_step(py[q], bey, cey * dy);
            ex = sye >= 0 ? fmadd(cb0[q], py[q], ex) : ex;
          }
          if (kX && (f & 8u)) {
            px[q] = fmadd(coef(lbe, q), px[q], coef(lce, q) * dx);
            ey = fmadd(-cb1[q], px[q], ey);
          }
          c[q] = ex;
          bf[q] = ey;
        }
        if (kSp && (f & 96u) && jcap) {
          const T v = sxB || (tm && (f & 4u)) || ((f & upB) && yB) ? bf[q] : T(0);
          if (f & 32u) cap(t, 0, v);
          if (f & 64u) cap(t, 3, v);
        }
      };
      // H half-step of plane q; dn: B of plane q - 1 (lossy: q + 1)
      auto h_half = [&](int q, T dn, int t, T jv) {
        const unsigned f = flags(q);
        const T dx = lossy ? dn - bf[q] : bf[q] - dn;
        T h;
        if constexpr (lossy) {
          const T dy = bf[q] - lane_next(bf[q]);
          T hx = fmadd(db * dy, ikyh, c[q]);
          h = fmadd(db * dx, kh[q], a[q]);
          if (CLS != 1) {
            if (kX && (f & 16u)) {
              qx[q] = fmadd(coef(lch, q), dx, coef(lbh, q) * qx[q]);
              h = fmadd(dtmu, qx[q], h);
            }
            qy[q] = fmadd(chy, dy, bhy * qy[q]);
            hx = syh >= 0 ? fmadd(dtmu, qy[q], hx) : hx;
          }
          c[q] = updates(sxC, f & upC, syC, yC) ? hx : c[q];
          h = updates(sxA, f & upA, syA, yA) ? h : a[q];
        } else if constexpr (tm) {
          const T dy = bf[q] - lane_prev(bf[q]);
          T hx = fmadd(db * -dy, ikyh, c[q]);
          if (CLS != 1) {
            psi_step(qy[q], bhy, chy * dy);
            hx = syh >= 0 ? fmadd(-db, qy[q], hx) : hx;
          }
          c[q] = updates(sxC, f & upC, syC, yC) ? hx : c[q];
          h = a[q];
          if (!kX || (f & upA)) {
            h = fmadd(db * dx, kh[q], h);
            if (kX && (f & 16u)) {
              qx[q] = fmadd(coef(lbh, q), qx[q], coef(lch, q) * dx);
              h = fmadd(db, qx[q], h);
            }
          }
        } else {
          const T dy = c[q] - lane_prev(c[q]);
          T kept = a[q];
          h = fmadd(db, fmadd(dy, ikyh, -(dx * kh[q])), a[q]);
          if (kSp && (f & 4u)) {
            h = jsrc ? h - jv : h;
            kept = jsrc ? kept - jv : kept;
          }
          if (kX && (f & 16u)) {
            qx[q] = fmadd(coef(lbh, q), qx[q], coef(lch, q) * dx);
            h = fmadd(-db, qx[q], h);
          }
          if (CLS != 1) {
            psi_step(qy[q], bhy, chy * dy);
            h = syh >= 0 ? fmadd(db, qy[q], h) : h;
          }
          h = updates(sxA, f & upA, syA, yA) ? h : kept;
        }
        a[q] = h;
        if (kSp && (f & 480u) && jcap) {
          const T v = syA || yA ? h : T(0);   // its planes are selected
          if (f & 32u) cap(t, 1, v);
          if (f & 128u) cap(t, 2, v);
          if (f & 64u) cap(t, 4, v);
          if (f & 256u) cap(t, 5, v);
        }
      };
      // ---- monitors: running sums of this wave's cells, weights (lane t:
      // record of step n0 + t), steps with a record
      constexpr int NM = MON == 0 ? 1 : 3;
      T mre[NM][K], mim[NM][K];
      double lcr[NM], lci[NM], msc[NM];
      unsigned mvalid[NM];
      const Monitor<T>* mon[NM];
      bool mafter[NM];
      // the own rows and planes [lo, hi) of monitor m of role r: of its box, and
      // inside the update range unless the steps keep the role's other cells
      struct MonBox { int lo, hi; bool row; };
      auto box = [&](int r, const Monitor<T>& m) {
        MonBox x;
        const int xb = r == 0 ? (sxA ? 0 : lossy ? 0 : ib + 1) : r == 1 ? (sxB ? 0 : ib) : (lossy ? 0 : ib + 1);
        const int xe = (r == 0 ? sxA : r == 1 ? sxB : sxC) ? nx : ie;
        x.lo = max(max(i0, m.x0), xb);
        x.hi = min(min(i0 + TX, m.x0 + m.ex), xe);
        x.row = lane >= TB && lane < TB + TY && j >= m.y0 && j < m.y0 + m.ey &&
                (r == 0 ? syA || yA : r == 1 ? syB || yB : syC || yC);
        return x;
      };
      if constexpr (MON != 0) {
        const int2 sm = smon[tl.x];
#pragma unroll
        for (int r = 0; r < NM; ++r) {
          mvalid[r] = 0;
          mon[r] = nullptr;
          if (!(MON & (1 << r))) continue;
          const int field = r == 0 ? R::A : r == 1 ? R::B : R::C;
          for (int k = 0; k < sm.y; ++k)
            if (mons[sm.x + k].field == field) mon[r] = mons + sm.x + k;
          lcr[r] = lci[r] = 0.0;
          if (mon[r]) {
            const Monitor<T>& m = *mon[r];
            const int rec = n0 + lane + m.shift;
            const bool has = lane < nsteps && rec >= 0 && rec < m.nrec;
            // a wave whose planes all lie in the ghost frame folds nothing
            mvalid[r] = ib0 + K > i0 && ib0 < i0 + TX ? (unsigned)__ballot(has) : 0u;
            lcr[r] = has ? m.cs[2 * rec] : 0.0;
            lci[r] = has ? m.cs[2 * rec + 1] : 0.0;
            msc[r] = m.scale;
            mafter[r] = m.after_h != 0;
            const MonBox x = box(r, m);
#pragma unroll
            for (int q = 0; q < K; ++q) {
              const int i = ib0 + q, cell = (i - m.x0) * m.ey + (j - m.y0);
              const bool in = i >= x.lo && i < x.hi && x.row;
              mre[r][q] = in ? m.re[cell] : T(0);
              mim[r][q] = in ? m.im[cell] : T(0);
            }
          }
        }
      }
      auto fold = [&](int t, bool after) {
        if constexpr (MON != 0) {
#pragma unroll
          for (int r = 0; r < NM; ++r) {
            if (!(MON & (1 << r)) || !((mvalid[r] >> t) & 1u) || mafter[r] != after) continue;
            const double cr = lane_get(lcr[r], t), ci = lane_get(lci[r], t), sc = msc[r];
#pragma unroll
            for (int q = 0; q < K; ++q) {
              const double v = sc * (double)(r == 0 ? a[q] : r == 1 ? bf[q] : c[q]);
              mre[r][q] = (T)fmadd(v, cr, (double)mre[r][q]);
              mim[r][q] = (T)fmadd(v, ci, (double)mim[r][q]);
            }
          }
        }
      };
      // first and last plane in the order of the E half-step: E takes its
      // neighbour from the wave that holds the plane after `last`, H from the
      // one before `first`
      constexpr int first = lossy ? K - 1 : 0, last = lossy ? 0 : K - 1;
      const bool wnext = lossy ? w > 0 : w + 1 < W, wprev = lossy ? w + 1 < W : w > 0;
      const int wn = lossy ? w - 1 : w + 1, wp = lossy ? w + 1 : w - 1;
      xA[w][lane] = a[first];
      for (int t = 0; t < nsteps; ++t) {
        const T jv = kSp ? lane_get(jvl, t) : T(0);
#pragma unroll
        for (int u = 0; u + 1 < K; ++u) {
          const int q = lossy ? K - 1 - u : u;
          e_half(q, a[lossy ? q - 1 : q + 1], t, jv);
        }
        lds_barrier();
        e_half(last, wnext ? xA[wn][lane] : a[last], t, jv);
        xB[w][lane] = bf[last];
        fold(t, false);
#pragma unroll
        for (int u = 1; u < K; ++u) {
          const int q = lossy ? K - 1 - u : u;
          h_half(q, bf[lossy ? q + 1 : q - 1], t, jv);
        }
        lds_barrier();
        h_half(first, wprev ? xB[wp][lane] : bf[first], t, jv);
        xA[w][lane] = a[first];
        fold(t, true);
      }
      if constexpr (MON != 0) {
#pragma unroll
        for (int r = 0; r < NM; ++r) {
          if (!(MON & (1 << r)) || !mvalid[r]) continue;
          const Monitor<T>& m = *mon[r];
          const MonBox x = box(r, m);
          if (!x.row) continue;
#pragma unroll
          for (int q = 0; q < K; ++q) {
            const int i = ib0 + q, cell = (i - m.x0) * m.ey + (j - m.y0);
            if (i >= x.lo && i < x.hi) {
              m.re[cell] = mre[r][q];
              m.im[cell] = mim[r][q];
            }
          }
        }
      }
      // ---- the inner cells to set B (fields unconditionally: cells no step
      // updates hold the same value in both sets)
      const int ib1 = opaque_uniform(ib00);
      const int js = j0 - TB + opaque_value(lane);
      const bool own = js >= j0 && js < j0 + TY && js < ny;   // j0 >= 0
      const bool yins = js >= jb && js < je, yins1 = (lossy || js > jb) && js < je;
      const bool yxes = tm ? yins : yins1, yxhs = tm && !lossy ? yins : yins1;
      // the planes' slab rows, read while every lane is active (the lanes that
      // hold them lie in the ghost frame and store nothing)
      int xf[K], xre[K], xrh[K];
      if (kX) {
        const XCell x = xcells(opaque_value(lane));
#pragma unroll
        for (int q = 0; q < K; ++q) {
          xf[q] = at(x.f, q);
          xre[q] = at(x.re, q);
          xrh[q] = at(x.rh, q);
        }
      }
      OIDT_GLOBAL T* const* fB = odd ? s.f : s.f2;
      OIDT_GLOBAL T* const* psiB = odd ? s.psi : s.psi2;
      T* oA = fB[R::A];
      T* oB = fB[R::B];
      T* oC = fB[R::C];
      if (own) {
#pragma unroll
        for (int q = 0; q < K; ++q) {
          const int i = ib1 + q;
          if (i < i0 || i >= i0 + TX || i >= nx) continue;
          // selected in every step, or updated
          auto clean = [&](bool sx, unsigned up, bool sy, bool yr) {
            return (!kX || sx || ((unsigned)xf[q] & up) != 0u) && (CLS == 1 || sy || yr);
          };
          const unsigned idx = (unsigned)i * ny + js;
          stg_nt<T>(oA, idx * es, clean(sxA, upA, syA, yxhs) ? a[q] : T(0));
          stg_nt<T>(oB, idx * es, clean(sxB, upB, syB, yxes) || (kSp && tm && (xf[q] & 4)) ? bf[q] : T(0));
          stg_nt<T>(oC, idx * es, clean(sxC, upC, syC, tm ? yins1 : yins) ? c[q] : T(0));
        }
        if (CLS != 1 && !yplain) {
          int dyes = 0, dyhs = 0, unused = 0;
          const int syes = yins ? se(js, jb, je, dyes, unused) : -1;
          const int syhs = yins1 ? sh(js, jb, je, dyhs, unused) : -1;
          T* opy = psiB[psi_id(R::PY, 1, 0)];
          T* oqy = psiB[psi_id(R::QY, 1, 0)];
          const unsigned oe = (unsigned)dyes * es + (syes == 1 ? s.psi_hi[1] : 0u);
          const unsigned oh = (unsigned)dyhs * es + (syhs == 1 ? s.psi_hi[1] : 0u);
#pragma unroll
          for (int q = 0; q < K; ++q) {
            const int i = ib1 + q;
            if (i < i0 || i >= i0 + TX || i >= ie) continue;
            if (syes >= 0 && i >= pye) stg<T>(opy, (unsigned)(i * N) * es + oe, py[q]);
            if (syhs >= 0 && i >= pyh) stg<T>(oqy, (unsigned)(i * N) * es + oh, qy[q]);
          }
        }
        if (kX) {
#pragma unroll
          for (int q = 0; q < K; ++q) {
            const int i = ib1 + q;
            if (i < i0 || i >= i0 + TX) continue;
            if ((xf[q] & 8) && yxes)
              stg<T>(psiB[psi_id(R::PX, 0, xre[q] >= kHi)], (unsigned)((xre[q] & (kHi - 1)) * ny + js) * es, px[q]);
            if ((xf[q] & 16) && yxhs)
              stg<T>(psiB[psi_id(R::QX, 0, xrh[q] >= kHi)], (unsigned)((xrh[q] & (kHi - 1)) * ny + js) * es, qx[q]);
          }
        }
      }
    };
    if (special)
      tile(std::integral_constant<int, 0>{});
    else if (!xplain)
      tile(std::integral_constant<int, 3>{});
    else if (yplain)
      tile(std::integral_constant<int, 1>{});
    else
      tile(std::integral_constant<int, 2>{});

    lds_barrier();   // the next tile reuses the exchange planes
  }
}

// MW: waves per SIMD to keep registers for (see launch_blocked2d).
template <typename T, int TB, int W, int K, int MW>
__global__ __launch_bounds__(64 * W, MW) void k_tmz_tb(const Slot<T>* __restrict__ slots,
                                                       const int4* __restrict__ tiles, int ntiles, int tstep) {
  blocked_step_2d<T, SCHEME_TMZ, TB, W, K, 0>(slots, tiles, ntiles, tstep, nullptr, nullptr);
}

template <typename T, int TB, int W, int K, int MW, int MON>
__global__ __launch_bounds__(64 * W, MW) void k_tez_tb(const Slot<T>* __restrict__ slots,
                                                       const int4* __restrict__ tiles, int ntiles, int tstep,
                                                       const Monitor<T>* __restrict__ mons,
                                                       const int2* __restrict__ smon) {
  blocked_step_2d<T, SCHEME_TEZ, TB, W, K, MON>(slots, tiles, ntiles, tstep, mons, smon);
}

template <typename T, int TB, int W, int K, int MW, int MON>
__global__ __launch_bounds__(64 * W, MW) void k_tmzl_tb(const Slot<T>* __restrict__ slots,
                                                        const int4* __restrict__ tiles, int ntiles, int tstep,
                                                        const Monitor<T>* __restrict__ mons,
                                                        const int2* __restrict__ smon) {
  blocked_step_2d<T, SCHEME_TMZ_LOSSY, TB, W, K, MON>(slots, tiles, ntiles, tstep, mons, smon);
}

}  // namespace oidt
