// Force interaction of the SPH step on gfx950 (FP32 pair arithmetic).
//
// Physics follow the reference GPU kernels KerInteractionForcesFluid /
// KerInteractionForcesFluidBox / KerInteractionForcesBound (JSphGpu_ker.cu:
// 450-990): for every fluid particle the neighbour cell rows are visited
// z-outer, y-inner, fluid cells first and then boundary cells, the particles of
// a row in ascending sorted index, all contributions in one accumulator set;
// distances from the cell-relative FP32 PosCell.
//
// Three fluid kernels produce the same sums in the same order (fluid_form says
// which runs):
//  - k_forces_fluid_rows: one lane per particle looping over its rows (the
//    reference's structure). A wave executes the pair body whenever any lane
//    has a neighbour, so most lanes idle (about a quarter of them do work on a
//    jittered lattice).
//  - k_forces_fluid_tile: a wave walks the rows shared by its lanes
//    once, stages each row in LDS with coalesced loads, lets every lane run a
//    cheap conservative distance test against the staged candidates and queue
//    its hits in LDS, then evaluates the exact pair body for the queued pairs
//    in wave-uniform batches (every lane busy), so the expensive body runs
//    only for real pairs. Queue order is the scan order, so the summation
//    order is unchanged.
//  - k_forces_fluid_team: four lanes per particle, four consecutive pairs at a
//    time, whose terms are then added in order (small and middle sizes).
// One condition on "the same": the rows kernel takes the pairs within 2h among the
// cells next to each particle's own, the other two those among the cells of a group
// of particles. They differ by pairs two cells apart (2h or more, but for
// rounding) whose FP32 distance rounds to 2h or less: the kernel gradient is nil
// there, but their dot/r^2 enters the maximum viscdt.
#include <cfloat>
#include <cstring>
#include <map>
#include <mutex>
#include <type_traits>
#include "ensemble.h"
#include "sph_math.h"

using namespace dsph;

namespace {

constexpr unsigned kBsForces = 128;
constexpr unsigned kBs = 256;

// Per-interaction preparation: pressure (EOS once per particle; each pair sees
// the same value the reference computes per pair) and the reciprocal density
// (v_rcp_f32, as a fast-math quotient by rho computes it).
__device__ inline float2 prep_one(float rho, const Cte& c) {
  return make_float2(eos_press(rho, c), fast_rcp(rho));
}

__global__ void __launch_bounds__(kBs) k_prep(unsigned n, const float4* __restrict__ velrho,
    float2* __restrict__ press, Cte c) {
  const unsigned p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  press[p] = prep_one(velrho[p].w, c);
}

// XCD-aware block order. The dispatcher sends block i to XCD i % 8; each
// XCD has its own L2. Renumbering so that XCD x runs one contiguous range of
// logical blocks keeps neighbouring particles (which read the same neighbour
// data) on the same L2.
constexpr unsigned kNumXcd = 8;
__device__ inline unsigned xcd_block(unsigned i, unsigned nblocks) {
  const unsigned per = nblocks / kNumXcd, rem = nblocks % kNumXcd;
  const unsigned x = i % kNumXcd, k = i / kNumXcd;
  return x * per + min(x, rem) + k;
}

struct Acc {
  float ax, ay, az, ar, visc, delta;
  float s[6];   // two_strain {xx,xy,xz,yy,yz,zz}
  float g[9];   // full velocity gradient (learned closure features)
  float4 sh;    // shifting: sum m/rho gradW (x = FLT_MAX: cancelled), w = -sum m/rho r.gradW
  float npc[3], nps[3];  // no-penetration: boundary neighbours counted and corrections, per axis
};

__device__ inline void acc_init(Acc& a) {
  a.ax = a.ay = a.az = a.ar = a.visc = a.delta = 0;
  a.sh = make_float4(0, 0, 0, 0);
#pragma unroll
  for (int k = 0; k < 3; k++) a.npc[k] = a.nps[k] = 0;
#pragma unroll
  for (int k = 0; k < 6; k++) a.s[k] = 0;
#pragma unroll
  for (int k = 0; k < 9; k++) a.g[k] = 0;
}

struct P1 {
  float4 ps, vr;
  float press, rrho;
  float tau[6];
  bool ftp1;   // floating particle (FT kernels only)
};

// Whether the series of pow_invgamma serves every pair: |ddtgz dz| < 1e-2.
__device__ inline bool ddt_series(const Cte& c) {
  return fabsf(c.ddtgz) * (2.f * c.h) * 1.01f < 1e-2f;
}

// Exact pair body for fluid p1 and neighbour p2 (KerInteractionForcesFluidBox,
// JSphGpu_ker.cu:539-777, in-scope options). boundp2 selects the boundary
// variant (mass, viscosity, no SPS tau of p2, delta-SPH rules).
// pair_eval takes the neighbour's PosCell, velrho and {pressure, 1/rho} already loaded
// and applies the exact neighbour test rr2 <= (2h)^2, rr2 >= ALMOSTZERO.
// MDBC2: boundary neighbours in mDBC2 mode (boundmode, tangential velocity):
// no mass when their ghost node is dry, viscous terms against the tangential
// velocity (JSphGpu_ker.cu:585-588, 725-730; velocities kept for continuity,
// MDBC2_KEEPVEL).
// SHIFT: standard shifting (JSphGpu_ker.cu:677-684): accumulates m2/rho2 gradW
// and -m2/rho2 r.gradW; a boundary neighbour cancels it (x = FLT_MAX) for
// shiftmode 1 (no boundaries) and, for shiftmode 2, when it is fixed.
// FT: floating bodies. A floating neighbour (code type floating, in the
// fluid range) has its body's particle mass ftomassp[type value], stops the
// Molteni-Colagrossi term when it is not heavier than 1.2 fluid particles,
// takes no part in the Fourtakas term and gives no SPS tau; a floating p1
// has no density diffusion and no strain (JSphGpu_ker.cu:570-583, 668,
// 755-766, 838-843).
// NOPEN: mDBC2 no-penetration sums against boundary neighbours, with the
// velocity relative to their motion velocity (motionvel, float3 per
// particle; NULL = fixed boundaries) (MDBC2_NoPen, JSphGpu_ker.cu:686-707
// with ComputeNoPenVel, :428-440).
template <int TVISCO, int TDDT, bool VELGRAD, bool MDBC2 = false, bool SHIFT = false,
          bool FT = false, bool NOPEN = false>
__device__ __forceinline__ void pair_eval(bool boundp2, unsigned p2, const float4& ps2,
    const float4& vr2, float2 pr2, const P1& q, const float* __restrict__ tau, float viscob,
    float viscof, const Cte& c, Acc& a, const uint8_t* __restrict__ bmode = nullptr,
    const float* __restrict__ tangenvel = nullptr, int shiftmode = 0,
    const typecode* __restrict__ code = nullptr, const float* __restrict__ ftomassp = nullptr,
    const float* __restrict__ boundnor = nullptr, const float* __restrict__ motionvel = nullptr) {
  const float3 dr = pscel_dr(q.ps, ps2, c.pcs);
  const float rr2 = dr.x * dr.x + dr.y * dr.y + dr.z * dr.z;
  if (!(rr2 <= c.ks2 && rr2 >= kAlmostZero)) return;
  float massp2 = boundp2 ? c.massb : c.massf;
  if (MDBC2 && boundp2 && bmode[p2] == DSPH_BMODE_MDBC2OFF) massp2 = 0.f;
  bool ftp2 = false;
  if (FT && !boundp2) {
    const unsigned cd = code[p2];
    ftp2 = code_type(cd) == kCodeTypeFloating;
    if (ftp2) {
      const float ftm = ftomassp[cd & kCodeMaskValue];
      if (TDDT == DSPH_DDT_DDT && ftm <= massp2 * 1.2f) a.delta = FLT_MAX;
      massp2 = ftm;
    }
  }
  const float visco = boundp2 ? viscob : viscof;
  const float fac = wendland_fac(rr2, c);
  const float frx = fac * dr.x, fry = fac * dr.y, frz = fac * dr.z;
  const float4& vr1 = q.vr;
  {
    const float prs = (q.press + pr2.x) * (q.rrho * pr2.y);
    const float p_vpm = -prs * massp2;
    a.ax += p_vpm * frx; a.ay += p_vpm * fry; a.az += p_vpm * frz;
  }
  float dvx = vr1.x - vr2.x, dvy = vr1.y - vr2.y, dvz = vr1.z - vr2.z;
  const float rrho2 = pr2.y;
  a.ar += massp2 * (dvx * frx + dvy * fry + dvz * frz) * (vr1.w * rrho2);
  const float cbar = c.cs0;
  const float dot3 = dr.x * frx + dr.y * fry + dr.z * frz;
  const float rr2eta = fast_rcp(rr2 + c.eta2);
  if (TDDT == DSPH_DDT_DDT && a.delta != FLT_MAX) {
    const float rhop1over2 = vr1.w * rrho2;
    const float visc_densi = c.ddtkh * cbar * (rhop1over2 - 1.f) * rr2eta;
    const float delta = visc_densi * dot3 * massp2;
    // A boundary neighbour cancels the term with DBC only (JSphGpu_ker.cu:665).
    a.delta = ((boundp2 && c.tboundary == DSPH_BC_DBC) ? FLT_MAX : a.delta + delta);
  }
  if ((TDDT == DSPH_DDT_DDT2 && a.delta != FLT_MAX && !(FT && ftp2)) ||
      (TDDT == DSPH_DDT_DDT2FULL && !boundp2 && !(FT && (ftp2 || a.delta == FLT_MAX)))) {
    const float rh = 1.f + c.ddtgz * dr.z;
    const float u = rh - 1.f;
    const float ser = u * (c.pc1 + u * (c.pc2 + u * (c.pc3 + u * c.pc4)));
    float pw = 1.f + ser;
    if (!ddt_series(c) && !(fabsf(u) < 1e-2f)) pw = powf(rh, c.invgamma);
    const float drho = c.rhopzero * pw - c.rhopzero;
    const float visc_densi = c.ddtkh * cbar * ((vr2.w - vr1.w) - drho) * rr2eta;
    const float delta = visc_densi * dot3 * massp2 * rrho2;
    a.delta = (boundp2 ? FLT_MAX : a.delta - delta);
  }
  if (SHIFT && a.sh.x != FLT_MAX) {
    const float massrho = massp2 * rrho2;
    const bool noshift = boundp2 && (shiftmode == 1 ||
                                     (shiftmode == 2 && code_type(code[p2]) == kCodeTypeFixed));
    a.sh.x = noshift ? FLT_MAX : a.sh.x + massrho * frx;
    a.sh.y += massrho * fry;
    a.sh.z += massrho * frz;
    a.sh.w -= massrho * dot3;
  }
  if (NOPEN && boundp2) {
    // A boundary neighbour of the first layer (|normal| < 1.75 dp) within
    // 1.25 dp, with the particle less than 0.75 |normal| away along the
    // normal: per axis, a particle moving towards the wall (v relative to
    // the wall's motion velocity) gets -(3 - 4 max(|dr/n|, 1/4)) v n^2.
    if (sqrtf(rr2) < 1.25f * c.dp) {
      const float* bn = boundnor + 3 * size_t(p2);
      const float norm = sqrtf(bn[0] * bn[0] + bn[1] * bn[1] + bn[2] * bn[2]);
      const float nrm[3] = {fast_div(bn[0], norm), fast_div(bn[1], norm), fast_div(bn[2], norm)};
      const float d[3] = {dr.x, dr.y, dr.z};
      const float* mv = motionvel ? motionvel + 3 * size_t(p2) : nullptr;
      const float v[3] = {mv ? q.vr.x - mv[0] : q.vr.x, mv ? q.vr.y - mv[1] : q.vr.y,
                          mv ? q.vr.z - mv[2] : q.vr.z};
      if (nrm[0] * dr.x + nrm[1] * dr.y + nrm[2] * dr.z < 0.75f * norm && norm < 1.75f * c.dp) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
          if (d[k] * nrm[k] < 0.75f && fabsf(nrm[k]) > 0.001f * c.dp && v[k] * nrm[k] < 0.f) {
            const float ratio = fmaxf(fabsf(fast_div(d[k], nrm[k])), 0.25f);
            const float factor = -4.f * ratio + 3.f;
            a.npc[k] += 1.f;
            a.nps[k] -= factor * v[k] * nrm[k] * nrm[k];
          }
        }
      }
    }
  }
  if (MDBC2 && boundp2) {
    const float* tv = tangenvel + 3 * size_t(p2);
    dvx = vr1.x - tv[0]; dvy = vr1.y - tv[1]; dvz = vr1.z - tv[2];
  }
  const float dot = dr.x * dvx + dr.y * dvy + dr.z * dvz;
  const float dot_rr2 = dot * rr2eta;
  a.visc = fmaxf(dot_rr2, a.visc);
  if (TVISCO == DSPH_VISCO_ARTIFICIAL) {
    // No branch: a term of zero leaves the sums as they are.
    const float amubar = c.h * dot_rr2;
    const float robar = (vr1.w + vr2.w) * 0.5f;
    float pi_visc = fast_div(-visco * cbar * amubar, robar) * massp2;
    pi_visc = dot < 0 ? pi_visc : 0.f;
    a.ax -= pi_visc * frx; a.ay -= pi_visc * fry; a.az -= pi_visc * frz;
  } else {
    const float robar2 = (vr1.w + vr2.w);
    const float temp = fast_div(4.f * visco, (rr2 + c.eta2) * robar2);
    const float vtemp = massp2 * temp * dot3;
    a.ax += vtemp * dvx; a.ay += vtemp * dvy; a.az += vtemp * dvz;
  }
  if (TVISCO == DSPH_VISCO_LAMINARSPS) {
    float sxx = q.tau[0], sxy = q.tau[1], sxz = q.tau[2], syy = q.tau[3], syz = q.tau[4],
          szz = q.tau[5];
    if (!boundp2 && !(FT && ftp2)) {
      const float* t2 = tau + 6 * size_t(p2);
      sxx += t2[0]; sxy += t2[1]; sxz += t2[2]; syy += t2[3]; syz += t2[4]; szz += t2[5];
    }
    a.ax += massp2 * (sxx * frx + sxy * fry + sxz * frz);
    a.ay += massp2 * (sxy * frx + syy * fry + syz * frz);
    a.az += massp2 * (sxz * frx + syz * fry + szz * frz);
    if (!(FT && q.ftp1)) {
      const float volp2 = -massp2 * rrho2;
      float dv = dvx * volp2; a.s[0] += dv * frx; a.s[1] += dv * fry; a.s[2] += dv * frz;
      dv = dvy * volp2;       a.s[1] += dv * frx; a.s[3] += dv * fry; a.s[4] += dv * frz;
      dv = dvz * volp2;       a.s[2] += dv * frx; a.s[4] += dv * fry; a.s[5] += dv * frz;
    }
  }
  if (VELGRAD) {
    // Full gradient G_ij = sum_b -m_b/rho_b (v_a-v_b)_i dW/dx_j.
    const float volp2 = -massp2 * rrho2;
    const float ux = dvx * volp2, uy = dvy * volp2, uz = dvz * volp2;
    a.g[0] += ux * frx; a.g[1] += ux * fry; a.g[2] += ux * frz;
    a.g[3] += uy * frx; a.g[4] += uy * fry; a.g[5] += uy * frz;
    a.g[6] += uz * frx; a.g[7] += uz * fry; a.g[8] += uz * frz;
  }
}

// Reference-structured pair: loads PosCell first and the rest only for a
// real neighbour.
template <int TVISCO, int TDDT, bool VELGRAD, bool MDBC2 = false, bool SHIFT = false,
          bool FT = false, bool NOPEN = false>
__device__ __forceinline__ void pair_body(bool boundp2, unsigned p2, const P1& q,
    const float4* __restrict__ poscell, const float4* __restrict__ velrho,
    const float2* __restrict__ press, const float* __restrict__ tau, float viscob, float viscof,
    const Cte& c, Acc& a, const uint8_t* __restrict__ bmode = nullptr,
    const float* __restrict__ tangenvel = nullptr, int shiftmode = 0,
    const typecode* __restrict__ code = nullptr, const float* __restrict__ ftomassp = nullptr,
    const float* __restrict__ boundnor = nullptr, const float* __restrict__ motionvel = nullptr) {
  const float4 ps2 = poscell[p2];
  const float3 dr = pscel_dr(q.ps, ps2, c.pcs);
  const float rr2 = dr.x * dr.x + dr.y * dr.y + dr.z * dr.z;
  if (!(rr2 <= c.ks2 && rr2 >= kAlmostZero)) return;
  pair_eval<TVISCO, TDDT, VELGRAD, MDBC2, SHIFT, FT, NOPEN>(
      boundp2, p2, ps2, velrho[p2], press[p2], q, tau, viscob, viscof, c, a, bmode, tangenvel,
      shiftmode, code, ftomassp, boundnor, motionvel);
}

template <int TVISCO>
__device__ inline void load_p1(unsigned p1, const float4* __restrict__ poscell,
                               const float4* __restrict__ velrho, const float2* __restrict__ press,
                               const float* __restrict__ tau, P1& q) {
  q.ps = poscell[p1];
  q.vr = velrho[p1];
  const float2 pr1 = press[p1];
  q.press = pr1.x;
  q.rrho = pr1.y;
  q.ftp1 = false;
#pragma unroll
  for (int k = 0; k < 6; k++)
    q.tau[k] = (TVISCO == DSPH_VISCO_LAMINARSPS) ? tau[6 * size_t(p1) + k] : 0.f;
}

template <int TVISCO, int TDDT, bool VELGRAD>
__device__ inline void store_results(unsigned p1, const Acc& a, float* __restrict__ viscdt,
                                     float* __restrict__ ar, float* __restrict__ ace,
                                     float* __restrict__ strain, float* __restrict__ velgrad) {
  if (a.ar != 0 || a.ax != 0 || a.ay != 0 || a.az != 0 || a.visc != 0) {
    float arp1 = a.ar;
    if (TDDT != DSPH_DDT_NONE && a.delta != FLT_MAX) arp1 += a.delta;
    ar[p1] += arp1;
    float* ap = ace + 3 * size_t(p1);
    ap[0] += a.ax; ap[1] += a.ay; ap[2] += a.az;
    if (a.visc > viscdt[p1]) viscdt[p1] = a.visc;
    if (TVISCO == DSPH_VISCO_LAMINARSPS) {
      float* sp = strain + 6 * size_t(p1);
#pragma unroll
      for (int k = 0; k < 6; k++) sp[k] += a.s[k];
    }
  }
  if (VELGRAD) {
    float* gp = velgrad + 9 * size_t(p1);
#pragma unroll
    for (int k = 0; k < 9; k++) gp[k] = a.g[k];
  }
}

__device__ inline NgLimits p1_limits(unsigned p1, const unsigned* __restrict__ dcell,
                                     const DivData& dvd) {
  const unsigned cel = dcell[p1];
  const int cx = int(dcel_cellx(dvd.domcellcode, cel)) - dvd.czx;
  const int cy = int(dcel_celly(dvd.domcellcode, cel)) - dvd.czy;
  const int cz = int(dcel_cellz(dvd.domcellcode, cel)) - dvd.czz;
  return ng_limits(cx, cy, cz, dvd);
}

// ------------------------------------------------------------ reference-order rows kernel
template <int TVISCO, int TDDT, bool VELGRAD, bool MDBC2 = false, bool SHIFT = false,
          bool FT = false, bool NOPEN = false>
__device__ __forceinline__ void fluid_rows_body(unsigned p1, float viscob, float viscof,
    const DivData& dvd, const Cte& c, const unsigned* __restrict__ dcell,
    const float4* __restrict__ poscell, const float4* __restrict__ velrho,
    const float2* __restrict__ press, const float* __restrict__ tau, float* __restrict__ viscdt,
    float* __restrict__ ar, float* __restrict__ ace, float* __restrict__ strain,
    float* __restrict__ velgrad, const uint8_t* __restrict__ bmode = nullptr,
    const float* __restrict__ tangenvel = nullptr, int shiftmode = 0,
    const typecode* __restrict__ code = nullptr, float4* __restrict__ shiftposfs = nullptr,
    const float* __restrict__ ftomassp = nullptr, const float* __restrict__ boundnor = nullptr,
    float4* __restrict__ nopenshift = nullptr, const float* __restrict__ motionvel = nullptr) {
  Acc a;
  acc_init(a);
  if (SHIFT) a.sh = shiftposfs[p1];
  P1 q;
  load_p1<TVISCO>(p1, poscell, velrho, press, tau, q);
  if (FT) {
    q.ftp1 = code_type(code[p1]) == kCodeTypeFloating;
    if (q.ftp1 && TDDT != DSPH_DDT_NONE) a.delta = FLT_MAX;
  }
  const NgLimits l = p1_limits(p1, dcell, dvd);
  for (int kind = 0; kind < 2; kind++) {
    const int base = kind == 0 ? int(dvd.cellfluid) : 0;
    for (int z = l.z0; z < l.z1; z++)
      for (int y = l.y0; y < l.y1; y++) {
        unsigned pini, pfin;
        row_range(dvd.begincell, base + z * dvd.ncw + y * dvd.ncx, l.x0, l.x1, pini, pfin);
        for (unsigned p2 = pini; p2 < pfin; p2++)
          pair_body<TVISCO, TDDT, VELGRAD, MDBC2, SHIFT, FT, NOPEN>(
              kind == 1, p2, q, poscell, velrho, press, tau, viscob, viscof, c, a, bmode,
              tangenvel, shiftmode, code, ftomassp, boundnor, motionvel);
      }
  }
  store_results<TVISCO, TDDT, VELGRAD>(p1, a, viscdt, ar, ace, strain, velgrad);
  if (SHIFT) shiftposfs[p1] = a.sh;
  if (NOPEN) {
    // Mean correction per axis over the boundary neighbours that asked for
    // one; w = 10 marks a particle to correct (JSphGpu_ker.cu:958-976).
    float4 ns = make_float4(0, 0, 0, 0);
    if (a.npc[0] > 0.f) { ns.x = fast_div(a.nps[0], a.npc[0]); ns.w = 10.f; }
    if (a.npc[1] > 0.f) { ns.y = fast_div(a.nps[1], a.npc[1]); ns.w = 10.f; }
    if (a.npc[2] > 0.f) { ns.z = fast_div(a.nps[2], a.npc[2]); ns.w = 10.f; }
    nopenshift[p1] = ns;
  }
}

template <int TVISCO, int TDDT, bool VELGRAD, bool MDBC2, bool SHIFT = false, bool FT = false,
          bool NOPEN = false>
__global__ void __launch_bounds__(kBsForces) k_forces_fluid_rows(
    unsigned n, unsigned pinit, float viscob, float viscof, DivData dvd, Cte c,
    const unsigned* __restrict__ dcell, const float4* __restrict__ poscell,
    const float4* __restrict__ velrho, const float2* __restrict__ press,
    const float* __restrict__ tau, float* __restrict__ viscdt, float* __restrict__ ar,
    float* __restrict__ ace, float* __restrict__ strain, float* __restrict__ velgrad,
    const uint8_t* __restrict__ bmode, const float* __restrict__ tangenvel, int shiftmode = 0,
    const typecode* __restrict__ code = nullptr, float4* __restrict__ shiftposfs = nullptr,
    const float* __restrict__ ftomassp = nullptr, const float* __restrict__ boundnor = nullptr,
    float4* __restrict__ nopenshift = nullptr, const float* __restrict__ motionvel = nullptr) {
  const unsigned p = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (p >= n) return;
  fluid_rows_body<TVISCO, TDDT, VELGRAD, MDBC2, SHIFT, FT, NOPEN>(
      p + pinit, viscob, viscof, dvd, c, dcell, poscell, velrho, press, tau, viscdt, ar, ace,
      strain, velgrad, bmode, tangenvel, shiftmode, code, shiftposfs, ftomassp, boundnor,
      nopenshift, motionvel);
}

// Boundary particle against one fluid neighbour that passed the neighbour
// test (KerInteractionForcesBound, JSphGpu_ker.cu:450-493): density rate and
// the viscous dt term.
__device__ __forceinline__ void bound_pair(const float4& vr1, const float3& dr, float rr2,
                                           const float4& vr2, float massp2, const Cte& c,
                                           float& arp1, float& visc) {
  const float fac = wendland_fac(rr2, c);
  const float frx = fac * dr.x, fry = fac * dr.y, frz = fac * dr.z;
  const float dvx = vr1.x - vr2.x, dvy = vr1.y - vr2.y, dvz = vr1.z - vr2.z;
  arp1 += massp2 * (dvx * frx + dvy * fry + dvz * frz) * fast_div(vr1.w, vr2.w);
  const float dot = dr.x * dvx + dr.y * dvy + dr.z * dvz;
  const float dot_rr2 = fast_div(dot, rr2 + c.eta2);
  visc = fmaxf(dot_rr2, visc);
}

// ------------------------------------------------------------ cell-row tile kernel
constexpr unsigned kTile = 64;   // candidates staged in LDS per tile (one bit each)
constexpr unsigned kMinBatch = 16;
constexpr unsigned kScanBlock = 8;  // staged candidates tested per loop trip
#ifndef DSPH_RING_TILES
#define DSPH_RING_TILES 8
#endif
// Tiles of hit masks kept per wave (8 bytes per lane and tile).
constexpr unsigned kRingTiles = DSPH_RING_TILES;
#ifndef DSPH_TILE_WAVES
#define DSPH_TILE_WAVES 1
#endif
// Waves per workgroup of the single-case tile kernel: the waves of one
// workgroup run on one CU and take consecutive groups of 64 particles, so
// they share the L1 copy of their common neighbour rows.
constexpr unsigned kTileWaves = DSPH_TILE_WAVES;

// Orders the LDS accesses of one wave whose lanes exchange data through LDS.
// The LDS executes the instructions of a wave in issue order, so fences at
// wavefront scope (which keep the compiler from moving accesses across them)
// are all that is needed; there is no workgroup barrier, as the waves of a
// workgroup run loops of different lengths.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int CTRL>
__device__ __forceinline__ unsigned dpp_u(unsigned v) {
  return unsigned(__builtin_amdgcn_update_dpp(0, int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __uint_as_float(dpp_u<CTRL>(__float_as_uint(v)));
}
constexpr int kDppRor1 = 0x121, kDppRor2 = 0x122, kDppRor4 = 0x124, kDppRor8 = 0x128;  // in 16 lanes
__device__ __forceinline__ unsigned lane_u(unsigned v, int lane) {
  return unsigned(__builtin_amdgcn_readlane(int(v), lane));
}
__device__ __forceinline__ float lane_f(float v, int lane) {
  return __uint_as_float(lane_u(__float_as_uint(v), lane));
}
__device__ __forceinline__ unsigned wave_min_u32(unsigned v) {
  v = min(v, dpp_u<kDppRor8>(v));
  v = min(v, dpp_u<kDppRor4>(v));
  v = min(v, dpp_u<kDppRor2>(v));
  v = min(v, dpp_u<kDppRor1>(v));
  return min(min(lane_u(v, 0), lane_u(v, 16)), min(lane_u(v, 32), lane_u(v, 48)));
}
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) { return ~wave_min_u32(~v); }
__device__ __forceinline__ float wave_min_f32(float v) {
  v = fminf(v, dpp_f<kDppRor8>(v));
  v = fminf(v, dpp_f<kDppRor4>(v));
  v = fminf(v, dpp_f<kDppRor2>(v));
  v = fminf(v, dpp_f<kDppRor1>(v));
  return fminf(fminf(lane_f(v, 0), lane_f(v, 16)), fminf(lane_f(v, 32), lane_f(v, 48)));
}
// Shifts the result of d <= thr into bit 0 of bits (bits = 2*bits + (thr >= d)):
// a compare into VCC and an add with carry, two instructions per candidate.
__device__ __forceinline__ void shift_in_le(unsigned& bits, float d, float thr) {
  asm("v_cmp_ge_f32_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc"
      : "+v"(bits)
      : "v"(thr), "v"(d)
      : "vcc");
}

// Conservative distance test of one lane against the first nblk blocks of 8
// staged candidates (wave-uniform nblk <= 8): bit k of the result is set when
// candidate k passes d = |q2|^2 - 2 q1.q2 <= thr. Bits of candidates beyond
// the staged ones are undefined (the caller masks them with its window).
__device__ __forceinline__ unsigned long long scan_tile(const float4* tile, unsigned nblk,
                                                        float m2x, float m2y, float m2z,
                                                        float thr) {
  unsigned w[2];
#pragma unroll
  for (unsigned h = 0; h < 2; h++) {
    const unsigned nb = min(nblk - min(nblk, 4u * h), 4u);
    unsigned b = 0;
#pragma unroll 1
    for (unsigned i = 0; i < nb; i++) {
#pragma unroll
      for (unsigned k = 0; k < kScanBlock; k++) {
        const float4 f = tile[32 * h + kScanBlock * i + k];
        float d = fmaf(m2x, f.x, f.w);
        d = fmaf(m2y, f.y, d);
        d = fmaf(m2z, f.z, d);
        shift_in_le(b, d, thr);
      }
    }
    // Candidate 32h + j is at bit 8nb-1-j: left-align it to bit 31-j, reverse.
    w[h] = nb ? __builtin_bitreverse32(b << (32u - kScanBlock * nb)) : 0u;
  }
  return ((unsigned long long)w[1] << 32) | w[0];
}

// One wave = 64 consecutive fluid particles (sorted order). Lanes in the same
// cell row (cy, cz) form a group (normally the whole wave); the group walks
// the union of its lanes' neighbour rows once, fluid cells then boundary
// cells, z-outer / y-inner (JSphGpu_ker.cu:867-896), 64 particles at a time with
// coalesced loads. Those within 2h of the box around the group's particles
// (about half) are appended, in order, to a tile in LDS (position relative to
// the box centre and its square; the particle's index beside it). Every lane
// tests the 64 entries of a full tile (LDS broadcast) with a conservative distance
// bound and keeps its hits as a 64-bit mask; the masks and indices of the last
// kRing tiles stay in LDS. The exact pair body then runs for the queued pairs in
// wave-uniform batches (every lane busy), each lane popping its hits in tile
// and bit order, i.e. in the reference's summation order: the results equal
// k_forces_fluid_rows bit for bit. Loads of the next pair are issued before
// the arithmetic of the current one.
// Bound by the VALU and the gathers, both near their limits at 6.1M particles: one
// VALU instruction per 3.2 cycles and SIMD (1030 a particle; an FMA of vector
// registers alone measured 2.9), and the texture data path of a CU busy 87 % of the
// cycles (two 16-byte gathers a pair, 55 % of them from L1). The box test halves the
// tiles to scan and lets a ring of 8 tiles even out the lanes better than 12 tiles of
// whole rows did: 6.1M particles 8.04 -> 7.12 ms (rings of 6 / 10 / 12: 7.38 / 7.30 / 7.32),
// 1.6M 2.15 -> 1.88 ms, a step of 3.0M particles in 2-D 1.99 -> 1.85 ms.
// LDS of one wave of the tile kernel.
template <unsigned kRing>
struct TileLds {
  float4 tile[2 * kTile];   // the tiles being filled: position in the group's frame, its square
  unsigned long long masks[kRing][64];
  unsigned index[kRing * kTile];   // particle of each staged neighbour | kind << 31
};

template <int TVISCO, int TDDT, bool VELGRAD, unsigned kRing, bool MDBC2 = false,
          bool SHIFT = false, bool EOS7 = false>
__device__ __forceinline__ void fluid_tile_body(unsigned p, bool valid, unsigned pinit,
    float viscob, float viscof, const DivData& dvd, const Cte& c,
    const unsigned* __restrict__ dcell, const float4* __restrict__ poscell, const float4* __restrict__ velrho,
    const float2* __restrict__ press, const float* __restrict__ tau, float* __restrict__ viscdt,
    float* __restrict__ ar, float* __restrict__ ace, float* __restrict__ strain,
    float* __restrict__ velgrad, TileLds<kRing>& lds, const uint8_t* __restrict__ bmode = nullptr,
    const float* __restrict__ tangenvel = nullptr, int shiftmode = 0,
    const typecode* __restrict__ code = nullptr, float4* __restrict__ shiftposfs = nullptr) {
  auto& masks = lds.masks;
  const unsigned lane = threadIdx.x & 63u;
  const unsigned p1 = (valid ? p : 0) + pinit;
  Acc a;
  acc_init(a);
  P1 q;
  load_p1<TVISCO>(p1, poscell, velrho, press, tau, q);
  if (SHIFT) a.sh = shiftposfs[p1];
  int cx, cy, cz;
  {
    const unsigned cel = dcell[p1];
    cx = int(dcel_cellx(dvd.domcellcode, cel)) - dvd.czx;
    cy = int(dcel_celly(dvd.domcellcode, cel)) - dvd.czy;
    cz = int(dcel_cellz(dvd.domcellcode, cel)) - dvd.czz;
  }
  const int s = dvd.scelldiv;
  const int pfx = pscel_fx(q.ps.w), pfy = pscel_fy(q.ps.w), pfz = pscel_fz(q.ps.w);

  // Queue state. wt: tiles scanned (uniform). Per lane: rt = tile being
  // consumed, cm = its remaining hits, tb = its first place in index,
  // len = queued hits. Invariant: len > 0 => cm != 0; len == 0 => rt == wt.
  unsigned wt = 0, rt = 0, tb = 0, len = 0;
  unsigned long long cm = 0;
  auto pop = [&](unsigned& j) {
    const unsigned bit = unsigned(__builtin_ctzll(cm));  // cm != 0 while len > 0
    j = lds.index[tb + bit];  // kind in bit 31
    cm &= cm - 1ull;
    len--;
    if (!cm) {
      if (len) {
        do {
          rt++;
          cm = masks[rt % kRing][lane];
        } while (!cm);
        tb = rt % kRing * kTile;
      } else {
        rt = wt;
      }
    }
  };
  // Pops the next queued pair and issues its loads (32-bit offsets from the
  // array bases).
  // EOS7 (gamma = 7): the neighbour's {press, 1/rho} are evaluated from its
  // density with the functions k_prep applies (so the same bits; the power is
  // four FP64 products) instead of being gathered: two gathers per pair
  // instead of three. Otherwise they are loaded.
  auto issue = [&](unsigned& j, float4& ps2, float4& vr2, float2& pr2) {
    pop(j);
    const unsigned jj = j & 0x7fffffffu;
    ps2 = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(poscell) + (jj << 4));
    vr2 = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(velrho) + (jj << 4));
    if (!EOS7)
      pr2 = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(press) + (jj << 3));
  };
  auto eval = [&](unsigned j, const float4& ps2, const float4& vr2, const float2& pr2) {
    const float2 pr =
        EOS7 ? make_float2(c.cteb * (pow7_f64(vr2.w * c.ovrhopzero) - 1.0f), fast_rcp(vr2.w))
             : pr2;
    pair_eval<TVISCO, TDDT, VELGRAD, MDBC2, SHIFT>((j >> 31) != 0, j & 0x7fffffffu, ps2, vr2,
                                                   pr, q, tau, viscob, viscof, c, a, bmode,
                                                   tangenvel, shiftmode, code);
  };
  // k wave-uniform iterations; each lane pops up to k of its queued pairs.
  // Two register sets alternate so the loads of the next pair are in flight
  // during the arithmetic of the current one. With kFull every lane has at
  // least k queued pairs, so no lane test is needed.
  auto process = [&](unsigned k, auto full) {
    constexpr bool kFull = decltype(full)::value;
    unsigned ja = 0, jb = 0;
    float4 psa = make_float4(0, 0, 0, 0), vra = psa, psb = psa, vrb = psa;
    float2 pra = make_float2(0, 0), prb = pra;
    bool ha = k != 0 && (kFull || len != 0);
    if (ha) issue(ja, psa, vra, pra);
    for (unsigned i = 0; i < k; i += 2) {
      const bool hb = i + 1 < k && (kFull || len != 0);
      if (hb) issue(jb, psb, vrb, prb);
      if (ha) eval(ja, psa, vra, pra);
      ha = i + 2 < k && (kFull || len != 0);
      if (ha) issue(ja, psa, vra, pra);
      if (hb) eval(jb, psb, vrb, prb);
    }
  };
  using Full = std::true_type;
  using Some = std::false_type;

  bool pending = valid;
  for (;;) {
    const unsigned long long pend = __ballot(pending);
    if (!pend) break;
    const int leader = __ffsll((long long)pend) - 1;
    const int gy = __builtin_amdgcn_readlane(cy, leader), gz = __builtin_amdgcn_readlane(cz, leader);
    const int rfx = __builtin_amdgcn_readlane(pfx, leader),
              rfy = __builtin_amdgcn_readlane(pfy, leader),
              rfz = __builtin_amdgcn_readlane(pfz, leader);
    const bool member = pending && cy == gy && cz == gz;
    pending = pending && !member;
    const int gxmin = __builtin_amdgcn_readlane(cx, leader);
    const int gxmax = int(~wave_min_u32(member ? ~unsigned(cx) : 0xffffffffu));
    const int X0 = gxmin - min(gxmin, s), X1 = gxmax + min(dvd.ncx - gxmax - 1, s) + 1;
    const int Y0 = gy - min(gy, s), Y1 = gy + min(dvd.ncy - gy - 1, s) + 1;
    const int Z0 = gz - min(gz, s), Z1 = gz + min(dvd.ncz - gz - 1, s) + 1;
    // Positions relative to the leader's PosCell, the box of the group's
    // particles, and the lane's threshold of the expanded distance test
    // |q1|^2 + |q2|^2 - 2 q1.q2 <= thr (q relative to the box centre).
    // Rounding: of the coordinates below 2^-22 Q with Q = max|q1| + 2h, of the
    // expanded form below 8 * 2^-24 * (2Q)^2: covered by 4e-5 (2h)^2 + 2e-6 Q^2.
    const float q1x = c.pcs * float(pfx - rfx) + q.ps.x, q1y = c.pcs * float(pfy - rfy) + q.ps.y,
                q1z = c.pcs * float(pfz - rfz) + q.ps.z;
    // A position that is not finite, or whose square may not be, stays out of the
    // box: all neighbours of the group pass (0 + |q2|^2 <= inf; not a position that
    // is not finite) and go to its exact test. (A pass of steps at 6.1M particles,
    // without any of this / so: 373.1 / 373.9 ms; all bits or-ed into the hits of each
    // tile instead, in another run: 364.9 / 367.8.)
    const bool near = member && q1x * q1x + q1y * q1y + q1z * q1z < 1e30f, far = member && !near;
    const float bx0 = wave_min_f32(near ? q1x : FLT_MAX),
                bx1 = -wave_min_f32(near ? -q1x : FLT_MAX);
    const float by0 = wave_min_f32(near ? q1y : FLT_MAX),
                by1 = -wave_min_f32(near ? -q1y : FLT_MAX);
    const float bz0 = wave_min_f32(near ? q1z : FLT_MAX),
                bz1 = -wave_min_f32(near ? -q1z : FLT_MAX);
    const float ox = 0.5f * (bx0 + bx1), oy = 0.5f * (by0 + by1), oz = 0.5f * (bz0 + bz1);
    const float ex = 0.5f * (bx1 - bx0), ey = 0.5f * (by1 - by0), ez = 0.5f * (bz1 - bz0);
    const float qx = q1x - ox, qy = q1y - oy, qz = q1z - oz;
    const float s1 = qx * qx + qy * qy + qz * qz;
    const float qm = sqrtf(ex * ex + ey * ey + ez * ez) + 1.01f * sqrtf(c.ks2);
    const float reach2 = c.ks2 * 1.00004f + 2.0e-6f * qm * qm;
    const float box2 = __ballot(far) ? __builtin_inff() : reach2;
    const float thr = far ? __builtin_inff() : reach2 - s1;
    const float m2x = far ? 0.f : -2.f * qx, m2y = far ? 0.f : -2.f * qy,
                m2z = far ? 0.f : -2.f * qz;
    const int ny = Y1 - Y0, nrows = ny * (Z1 - Z0);
    // Rows of the group, fluid cells then boundary cells, one a lane (18 in
    // all, or 50 of half cells); 64 neighbours of a row at a time. Those near
    // the group's box are appended to the tile being filled (index wt; fill
    // entries, the ones past 64 belong to the next).
    int r0 = 0;
    unsigned rini = 0, rfin = 0, t = 0, gfin = 0, kbit = 0, fill = 0;
    unsigned long long rows = 0;
    for (bool more = true; more;) {
      if (t >= gfin) {
        while (!rows && r0 < 2 * nrows) {
          const int r = r0 + int(lane);
          rini = rfin = 0;
          if (r < 2 * nrows) {
            const int rk = r >= nrows ? r - nrows : r;
            const int z = Z0 + rk / ny, y = Y0 + rk % ny;
            row_range(dvd.begincell,
                      (r >= nrows ? 0 : int(dvd.cellfluid)) + z * dvd.ncw + y * dvd.ncx, X0, X1,
                      rini, rfin);
          }
          rows = __ballot(rfin > rini);
          r0 += 64;
        }
        more = rows != 0;
        if (more) {
          const int rr = __builtin_ctzll(rows);
          rows &= rows - 1;
          t = lane_u(rini, rr);
          gfin = lane_u(rfin, rr);
          kbit = r0 - 64 + rr >= nrows ? 0x80000000u : 0u;
        }
      }
      if (more) {
        // The places of tiles wt and wt + 1 must have been consumed by every lane.
        while (wt + 1 >= kRing && wave_min_u32(rt) + kRing <= wt + 1) process(kMinBatch, Some());
        const bool in = t + lane < gfin;
        const unsigned p2 = in ? t + lane : t;
        t += 64;
        const float4 f = *reinterpret_cast<const float4*>(
            reinterpret_cast<const char*>(poscell) + (p2 << 4));
        const float x = c.pcs * float(pscel_fx(f.w) - rfx) + f.x - ox,
                    y = c.pcs * float(pscel_fy(f.w) - rfy) + f.y - oy,
                    z = c.pcs * float(pscel_fz(f.w) - rfz) + f.z - oz;
        const float hx = fmaxf(fabsf(x) - ex, 0.f), hy = fmaxf(fabsf(y) - ey, 0.f),
                    hz = fmaxf(fabsf(z) - ez, 0.f);
        const bool keep = in && hx * hx + hy * hy + hz * hz <= box2;
        const unsigned long long kept = __ballot(keep);
        wave_sync();
        if (keep) {
          const unsigned i = fill + __builtin_amdgcn_mbcnt_hi(
                                        unsigned(kept >> 32),
                                        __builtin_amdgcn_mbcnt_lo(unsigned(kept), 0));
          lds.tile[(wt * kTile + i) % (2 * kTile)] = make_float4(x, y, z, x * x + y * y + z * z);
          const unsigned e = wt % kRing * kTile + i;
          lds.index[e >= kRing * kTile ? e - kRing * kTile : e] = p2 | kbit;
        }
        fill += unsigned(__popcll(kept));
        wave_sync();
      }
      if (fill >= kTile || (!more && fill)) {
        // Hits of this lane among the entries of the tile (blocks of 8 up to the
        // last one; the rest drops).
        const unsigned nt = min(fill, kTile);
        unsigned long long hm = 0;
        if (member)
          hm = scan_tile(lds.tile + (wt & 1) * kTile, (nt + kScanBlock - 1) / kScanBlock, m2x, m2y,
                         m2z, thr) &
               (~0ull >> (kTile - nt));
        masks[wt % kRing][lane] = hm;
        if (len == 0) {
          // Caught up: consume the new tile directly.
          cm = hm;
          tb = wt % kRing * kTile;
          rt = hm ? wt : wt + 1;
        }
        len += unsigned(__popcll(hm));
        wt++;
        fill -= nt;
        if (!more && fill) more = true;   // a last, partial tile
        const unsigned mn = wave_min_u32(member ? len : 0xffffffffu);
        if (mn >= kMinBatch) {
          // All 64 lanes have mn pairs queued (the usual case: one group,
          // all lanes valid): batches without per-lane tests.
          if (wave_min_u32(len) >= mn) process(mn, Full());
          else process(mn, Some());
        }
      }
    }
  }
  process(wave_max_u32(len), Some());
  if (valid) {
    store_results<TVISCO, TDDT, VELGRAD>(p1, a, viscdt, ar, ace, strain, velgrad);
    if (SHIFT) shiftposfs[p1] = a.sh;
  }
}

// Waves per SIMD the register allocation of the tile kernel must allow. The
// kernel's speed is set by the latency of its neighbour gathers, so by the
// waves that cover it: 5 (96 registers, a few bytes spilled outside the pair
// loop) for the artificial and laminar accumulator sets, measured 10% faster
// than the 4 waves of the unconstrained allocation; 4 (128 registers) for
// the larger sets, which would otherwise get 3.
template <int TVISCO, bool VELGRAD, bool MDBC2, bool SHIFT>
constexpr int tile_min_waves() {
  return (TVISCO != DSPH_VISCO_LAMINARSPS && !VELGRAD && !MDBC2 && !SHIFT) ? 5 : 4;
}

template <int TVISCO, int TDDT, bool VELGRAD, unsigned kRing, bool MDBC2 = false,
          bool SHIFT = false, bool EOS7 = false>
__global__ void __launch_bounds__(64 * kTileWaves)
__attribute__((amdgpu_waves_per_eu(tile_min_waves<TVISCO, VELGRAD, MDBC2, SHIFT>(), 8)))
k_forces_fluid_tile(
    unsigned n, unsigned pinit, float viscob, float viscof, DivData dvd, Cte c,
    const unsigned* __restrict__ dcell, const float4* __restrict__ poscell, const float4* __restrict__ velrho,
    const float2* __restrict__ press, const float* __restrict__ tau, float* __restrict__ viscdt,
    float* __restrict__ ar, float* __restrict__ ace, float* __restrict__ strain,
    float* __restrict__ velgrad, const uint8_t* __restrict__ bmode = nullptr,
    const float* __restrict__ tangenvel = nullptr, int shiftmode = 0,
    const typecode* __restrict__ code = nullptr, float4* __restrict__ shiftposfs = nullptr) {
  __shared__ TileLds<kRing> lds[kTileWaves];
  const unsigned w = threadIdx.x >> 6;
  const unsigned p =
      (xcd_block(blockIdx.x, gridDim.x) * kTileWaves + w) * 64 + (threadIdx.x & 63u);
  fluid_tile_body<TVISCO, TDDT, VELGRAD, kRing, MDBC2, SHIFT, EOS7>(
      p, p < n, pinit, viscob, viscof, dvd, c, dcell, poscell, velrho, press, tau,
      viscdt, ar, ace, strain, velgrad, lds[w], bmode, tangenvel, shiftmode, code, shiftposfs);
}

// Boundary particle p1 against fluid neighbours (KerInteractionForcesBound,
// JSphGpu_ker.cu:450-533).
// FT: a floating neighbour has its body's particle mass (JSphGpu_ker.cu:470-483).
template <bool FT = false>
__device__ __forceinline__ void bound_body(unsigned p1, const DivData& dvd, const Cte& c,
    const unsigned* __restrict__ dcell, const float4* __restrict__ poscell,
    const float4* __restrict__ velrho, float* __restrict__ viscdt, float* __restrict__ ar,
    const typecode* __restrict__ code = nullptr, const float* __restrict__ ftomassp = nullptr) {
  float visc = 0, arp1 = 0;
  const float4 ps1 = poscell[p1];
  const float4 vr1 = velrho[p1];
  const NgLimits l = p1_limits(p1, dcell, dvd);
  for (int z = l.z0; z < l.z1; z++)
    for (int y = l.y0; y < l.y1; y++) {
      unsigned pini, pfin;
      row_range(dvd.begincell, int(dvd.cellfluid) + z * dvd.ncw + y * dvd.ncx, l.x0, l.x1,
                pini, pfin);
      for (unsigned p2 = pini; p2 < pfin; p2++) {
        const float4 ps2 = poscell[p2];
        const float3 dr = pscel_dr(ps1, ps2, c.pcs);
        const float rr2 = dr.x * dr.x + dr.y * dr.y + dr.z * dr.z;
        if (rr2 <= c.ks2 && rr2 >= kAlmostZero) {
          const float4 vr2 = velrho[p2];
          float massp2 = c.massf;
          if (FT) {
            const unsigned cd = code[p2];
            if (code_type(cd) == kCodeTypeFloating) massp2 = ftomassp[cd & kCodeMaskValue];
          }
          bound_pair(vr1, dr, rr2, vr2, massp2, c, arp1, visc);
        }
      }
    }
  if (arp1 != 0 || visc != 0) {
    ar[p1] += arp1;
    if (visc > viscdt[p1]) viscdt[p1] = visc;
  }
}

template <bool FT = false>
__global__ void __launch_bounds__(kBsForces) k_forces_bound(unsigned n, DivData dvd, Cte c,
    const unsigned* __restrict__ dcell, const float4* __restrict__ poscell,
    const float4* __restrict__ velrho, float* __restrict__ viscdt, float* __restrict__ ar,
    const typecode* __restrict__ code = nullptr, const float* __restrict__ ftomassp = nullptr) {
  const unsigned p1 = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (p1 >= n) return;
  bound_body<FT>(p1, dvd, c, dcell, poscell, velrho, viscdt, ar, code, ftomassp);
}

// Arrays of one interaction (the options' arrays are null when unused).
struct TeamArrays {
  const unsigned* __restrict__ dcell;
  const float4* __restrict__ poscell;
  const float4* __restrict__ velrho;
  const float2* __restrict__ press;
  const float* __restrict__ tau;
  float* __restrict__ viscdt;
  float* __restrict__ ar;
  float* __restrict__ ace;
  float* __restrict__ strain;
  const uint8_t* __restrict__ bmode;
  const float* __restrict__ tangenvel;
  const typecode* __restrict__ code;
  const float* __restrict__ ftomassp;
};

// ------------------------------------------------------------ team kernel
// The tile kernel's sums with four lanes per particle: a wave works on 16
// consecutive particles (a "team" of four lanes each). Rows shared by the wave's
// particles are walked once, 64 neighbours at a time with coalesced loads; a
// neighbour farther than 2h from the box around the particles is dropped, the
// others go to a ring in LDS with all that the pair body reads. Every 64 of
// them the lanes of a team test a quarter each with the conservative bound and
// append their hits, in order, to the team's queue. The pair body then runs
// for four consecutive hits of every team at a time, one per lane, and writes
// the factors of its terms to LDS; each lane then adds one component (ax, ay,
// az, ar; the density diffusion on all lanes) of the four pairs one after the other.
// So every sum runs over the neighbours in the rows' order with the rows
// kernel's roundings: identical bits.
//
// Why: with one lane per particle (tile kernel) a wave is a serial chain
// of some 300 gathers and pair bodies, and below about 1e5 particles few
// waves share the chip; four lanes per particle make four times the waves
// with a quarter of the chain, and data in LDS replaces the gathers. Bound by the
// latency of that chain: 80k fluid particles issue one VALU instruction per 6.6
// cycles and SIMD, 10k (638 waves for 1024 SIMDs) one per 27; texture data path 32
// and 10 % of the cycles, LDS bank conflicts 7 and 2 %. us, tile -> team (dam breaks,
// artificial viscosity): 26k particles, 10k of them fluid, 321 -> 111; 141k (80k)
// 381 -> 253; 253k (157k) 428 -> 414; 357k (234k) 531 -> 578. Boundary interaction,
// one lane per particle -> team: 26k 229 -> 46, 141k 243 -> 49, 6.1M 406 -> 196.
// Computed share of busy lanes in the pair body for particles in lattice order:
// ring of 128 77 %, 192 86 %, 256 94 % (but a wave less per SIMD).
constexpr unsigned kTeam = 4;             // lanes per particle
constexpr unsigned kTeamP = 64 / kTeam;   // particles per wave
constexpr unsigned kRingN = 192;          // neighbours kept in LDS (8-bit queue entries)
constexpr unsigned kQueue = 128;          // hits a team may have queued
constexpr int kSpan = 4;                  // cells of a row that one group spans
constexpr int kCellBias = 128;            // cell offsets are kept as bytes
constexpr int kNear = 8;                  // PosCell cells a group spans beside its first particle

constexpr int kDppSwap1 = 0xB1;  // quad_perm [1,0,3,2]
constexpr int kDppSwap2 = 0x4E;  // quad_perm [2,3,0,1]
template <int J>
__device__ __forceinline__ float team_lane(float v) { return dpp_f<J * 0x55>(v); }  // lane J of the team

__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }
// Minimum / maximum over the wave of a value that is equal within each team.
__device__ __forceinline__ float teams_min(float v) {
  v = fminf(v, dpp_f<kDppRor4>(v));
  v = fminf(v, dpp_f<kDppRor8>(v));
  return fminf(fminf(lane_f(v, 0), lane_f(v, 16)), fminf(lane_f(v, 32), lane_f(v, 48)));
}
__device__ __forceinline__ int teams_max_i(int v) {
  v = max(v, int(dpp_u<kDppRor4>(unsigned(v))));
  v = max(v, int(dpp_u<kDppRor8>(unsigned(v))));
  return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// Constants of the pair body, moved to vector registers (pin): a VALU
// instruction with a scalar register operand issues in 5 cycles on gfx950,
// with vector registers and literals only in 2.9 (measured, v_fma_f32).
struct PairK {
  float pcs, ks2, invh, bwenh, eta2, mass;
  float dk, ddtgz, rho0, pc1, pc2, pc3, pc4;  // dk = ddtkh cs0
  float visk, h;                              // artificial: -visco cs0; else 4 visco
  bool series;  // |ddtgz dz| < 1e-2 for every pair: the series of pow_invgamma serves all
};
template <int TVISCO, int TDDT>
__device__ __forceinline__ PairK pair_k(const Cte& c, bool boundp2, float visco) {
  PairK k;
  k.pcs = c.pcs; k.ks2 = c.ks2; k.invh = c.invh; k.bwenh = c.bwenh; k.eta2 = c.eta2;
  k.mass = boundp2 ? c.massb : c.massf;
  k.dk = c.ddtkh * c.cs0; k.ddtgz = c.ddtgz; k.rho0 = c.rhopzero;
  k.pc1 = c.pc1; k.pc2 = c.pc2; k.pc3 = c.pc3; k.pc4 = c.pc4;
  k.visk = TVISCO == DSPH_VISCO_ARTIFICIAL ? -visco * c.cs0 : 4.f * visco;
  k.h = c.h;
  k.series = ddt_series(c);
  pin(k.pcs); pin(k.ks2); pin(k.invh); pin(k.bwenh); pin(k.eta2); pin(k.mass);
  pin(k.visk);
  if (TVISCO == DSPH_VISCO_ARTIFICIAL) pin(k.h);
  if (TDDT != DSPH_DDT_NONE) pin(k.dk);
  if (TDDT == DSPH_DDT_DDT2 || TDDT == DSPH_DDT_DDT2FULL) {
    pin(k.ddtgz); pin(k.rho0); pin(k.pc1); pin(k.pc2); pin(k.pc3); pin(k.pc4);
  }
  return k;
}

// What a neighbour carries beside position, velocity, density, pressure and
// 1/rho (only the options that use it).
struct P2x {
  float mass;        // FT, MDBC2: of this neighbour
  unsigned flags;    // kNb*
  float t[6];        // SPS: tau of a fluid neighbour; MDBC2: tangential velocity of a wall's
};
constexpr unsigned kNbFloating = 1, kNbLight = 2;

template <int TVISCO, bool MDBC2, bool FT, bool KB>
__device__ __forceinline__ void load_p2x(unsigned p2, const Cte& c, const TeamArrays& A, P2x& o) {
  o.mass = 0.f;
  o.flags = 0;
  if (FT && !KB) {
    o.mass = c.massf;
    const unsigned cd = A.code[p2];
    if (code_type(cd) == kCodeTypeFloating) {
      const float ftm = A.ftomassp[cd & kCodeMaskValue];
      o.flags = kNbFloating | (ftm <= c.massf * 1.2f ? kNbLight : 0u);
      o.mass = ftm;
    }
  }
  if (MDBC2 && KB) {
    o.mass = A.bmode[p2] == DSPH_BMODE_MDBC2OFF ? 0.f : c.massb;
#pragma unroll
    for (int i = 0; i < 3; i++) o.t[i] = A.tangenvel[3 * size_t(p2) + i];
  }
  if (TVISCO == DSPH_VISCO_LAMINARSPS && !KB) {
#pragma unroll
    for (int i = 0; i < 6; i++) o.t[i] = A.tau[6 * size_t(p2) + i];
  }
}

// Factors of the terms of one pair, as pair_eval adds them one after the other:
//   a += p fr;  artificial: a += c fr, laminar: a += c dv;  SPS: a += m e,
//   strain += u fr;  ar += mar rr;  delta -= dl.
struct Terms {
  float p, c, mar, dl, frx, fry, frz, rr;
  float dvx, dvy, dvz, ex, ey, ez, m, ux, uy, uz;
};

// The terms of fluid particle q and a neighbour (pair_eval, expression by
// expression); all zero but fr unless ok. KB: boundary neighbour.
template <int TVISCO, int TDDT, bool MDBC2, bool FT, bool KB>
__device__ __forceinline__ void pair_terms(bool ok, const float3& dr, float rr2, const float4& vr2,
    float2 pr2, const P2x& x, const P1& q, const PairK& k, const Cte& c, Terms& t, float& visc,
    bool& cancel) {
  const float4& vr1 = q.vr;
  const float mass = (FT && !KB) || (MDBC2 && KB) ? x.mass : k.mass;
  const bool ftp2 = FT && !KB && (x.flags & kNbFloating);
  const float rad = fast_sqrt(rr2);
  const float qq = rad * k.invh;
  const float wqq1 = 1.f - 0.5f * qq;
  const float fac = k.bwenh * wqq1 * wqq1 * wqq1;
  t.frx = fac * dr.x; t.fry = fac * dr.y; t.frz = fac * dr.z;
  const float frx = t.frx, fry = t.fry, frz = t.frz;
  const float rrho2 = pr2.y;
  const float prs = (q.press + pr2.x) * (q.rrho * rrho2);
  const float p = -prs * mass;
  float dvx = vr1.x - vr2.x, dvy = vr1.y - vr2.y, dvz = vr1.z - vr2.z;
  const float mar = mass * (dvx * frx + dvy * fry + dvz * frz);
  const float rr = vr1.w * rrho2;
  const float dot3 = dr.x * frx + dr.y * fry + dr.z * frz;
  const float rr2eta = fast_rcp(rr2 + k.eta2);
  float dl = 0.f;
  if (TDDT == DSPH_DDT_DDT) {
    const float rhop1over2 = vr1.w * rrho2;
    const float visc_densi = k.dk * (rhop1over2 - 1.f) * rr2eta;
    const float delta = visc_densi * dot3 * mass;
    dl = -delta;
    // A boundary neighbour cancels the term with DBC only (JSphGpu_ker.cu:665).
    if (ok && KB && c.tboundary == DSPH_BC_DBC) cancel = true;
    if (ok && FT && !KB && (x.flags & kNbLight)) cancel = true;
  }
  if (TDDT == DSPH_DDT_DDT2 && KB && ok) cancel = true;
  if (!KB && (TDDT == DSPH_DDT_DDT2 || TDDT == DSPH_DDT_DDT2FULL)) {
    const float rh = 1.f + k.ddtgz * dr.z;
    const float u = rh - 1.f;
    const float s = u * (k.pc1 + u * (k.pc2 + u * (k.pc3 + u * k.pc4)));
    float pw = 1.f + s;
    if (!k.series && !(fabsf(u) < 1e-2f)) pw = powf(rh, c.invgamma);
    const float drho = k.rho0 * pw - k.rho0;
    const float visc_densi = k.dk * ((vr2.w - vr1.w) - drho) * rr2eta;
    const float delta = visc_densi * dot3 * mass * rrho2;
    dl = ftp2 ? 0.f : delta;
  }
  if (MDBC2 && KB) {
    dvx = vr1.x - x.t[0]; dvy = vr1.y - x.t[1]; dvz = vr1.z - x.t[2];
  }
  const float dot = dr.x * dvx + dr.y * dvy + dr.z * dvz;
  const float dot_rr2 = dot * rr2eta;
  float cc;
  if (TVISCO == DSPH_VISCO_ARTIFICIAL) {
    const float amubar = k.h * dot_rr2;
    const float robar = (vr1.w + vr2.w) * 0.5f;
    const float pi_visc = fast_div(k.visk * amubar, robar) * mass;
    cc = dot < 0 ? -pi_visc : 0.f;
  } else {
    const float robar2 = (vr1.w + vr2.w);
    const float temp = fast_div(k.visk, (rr2 + k.eta2) * robar2);
    cc = mass * temp * dot3;
  }
  const unsigned keep = ok ? 0xffffffffu : 0u;
  auto only = [&](float v) { return __uint_as_float(__float_as_uint(v) & keep); };
  visc = fmaxf(ok ? dot_rr2 : visc, visc);
  t.p = only(p); t.c = only(cc); t.mar = only(mar); t.dl = only(dl); t.rr = only(rr);
  if (TVISCO != DSPH_VISCO_ARTIFICIAL) { t.dvx = only(dvx); t.dvy = only(dvy); t.dvz = only(dvz); }
  if (TVISCO == DSPH_VISCO_LAMINARSPS) {
    float sxx = q.tau[0], sxy = q.tau[1], sxz = q.tau[2], syy = q.tau[3], syz = q.tau[4],
          szz = q.tau[5];
    if (!KB && !ftp2) {
      sxx += x.t[0]; sxy += x.t[1]; sxz += x.t[2]; syy += x.t[3]; syz += x.t[4]; szz += x.t[5];
    }
    t.m = only(mass);
    t.ex = only(sxx * frx + sxy * fry + sxz * frz);
    t.ey = only(sxy * frx + syy * fry + syz * frz);
    t.ez = only(sxz * frx + syz * fry + szz * frz);
    const float volp2 = -mass * rrho2;
    const bool strain = !(FT && q.ftp1);
    t.ux = strain ? only(dvx * volp2) : 0.f;
    t.uy = strain ? only(dvy * volp2) : 0.f;
    t.uz = strain ? only(dvz * volp2) : 0.f;
  }
}

// LDS of one wave. kP: pressures; kX: floats of option data per neighbour; kM:
// its mass; kT: float4 of terms per lane.
template <bool kP, unsigned kX, bool kM, unsigned kT>
struct TeamLds {
  float4 pos[kRingN];   // PosCell position, bytes {cell offsets x, y, z, flags}
  float4 vr[kRingN];    // velocity and density
  float pr[kP ? kRingN : 1];    // pressure
  float m[kM ? kRingN : 1];
  float x[kX ? kX * kRingN : 1];
  float4 scan[2 * 4 * 17];      // position in the group's frame, its square (17: bank spread)
  float4 term[kTeamP * (kT * kTeam + 1)];   // a team's records, padded: bank spread
  alignas(4) uint8_t queue[kTeamP][kQueue + 4];   // (+ 4: bank spread)
};
template <int TVISCO, bool MDBC2>
constexpr unsigned team_kx() {
  return TVISCO == DSPH_VISCO_LAMINARSPS ? 6 : (MDBC2 ? 3 : 0);
}
template <int TVISCO, bool BP1>
constexpr unsigned team_kt() {
  return BP1 ? 1 : (TVISCO == DSPH_VISCO_ARTIFICIAL ? 2 : (TVISCO == DSPH_VISCO_LAMINAR ? 3 : 5));
}

// Particles [pw, min(pw+16, n)) of those from pinit on. BP1: boundary
// particles (bound_pair over fluid cells). kInMap: all positions are inside the
// map (an ensemble excludes others when it divides).
template <int TVISCO, int TDDT, bool MDBC2, bool FT, bool BP1, bool kInMap = false>
__device__ __forceinline__ void team_body(unsigned pw, unsigned n, unsigned pinit, float viscob,
    float viscof, const DivData& dvd, const Cte& c, const TeamArrays& A,
    TeamLds<!BP1, team_kx<TVISCO, MDBC2>(), MDBC2 || FT, team_kt<TVISCO, BP1>()>& lds) {
  constexpr unsigned kX = team_kx<TVISCO, MDBC2>();
  constexpr bool kM = MDBC2 || FT;
  constexpr bool kSps = TVISCO == DSPH_VISCO_LAMINARSPS;
  const unsigned lane = threadIdx.x & 63u;
  const unsigned k = lane & (kTeam - 1), team = lane / kTeam;
  const unsigned p = pw + team;
  const bool valid = p < n;
  const unsigned p1 = (valid ? p : 0) + pinit;
  P1 q;
  q.ps = A.poscell[p1];
  // A particle whose position is not finite or far from its PosCell cell
  // (dsph_update_poscell gives these for positions outside the map) joins no group:
  // one lane walks its rows.
  const float lim = float(kNear) * c.pcs;
  const bool fit =
      kInMap || (fabsf(q.ps.x) <= lim && fabsf(q.ps.y) <= lim && fabsf(q.ps.z) <= lim);
  if (__builtin_expect(!fit, 0)) {
    q.ps.x = q.ps.y = q.ps.z = 0.f;
    if (valid && k == 0) {
      if constexpr (BP1)
        bound_body<FT>(p1, dvd, c, A.dcell, A.poscell, A.velrho, A.viscdt, A.ar, A.code,
                       A.ftomassp);
      else
        fluid_rows_body<TVISCO, TDDT, false, MDBC2, false, FT>(
            p1, viscob, viscof, dvd, c, A.dcell, A.poscell, A.velrho, A.press, A.tau, A.viscdt,
            A.ar, A.ace, A.strain, nullptr, A.bmode, A.tangenvel, 0, A.code, nullptr, A.ftomassp);
    }
  }
  q.vr = A.velrho[p1];
  q.press = q.rrho = 0.f;
  if (!BP1) {
    const float2 pr1 = A.press[p1];
    q.press = pr1.x;
    q.rrho = pr1.y;
  }
  q.ftp1 = FT && !BP1 && code_type(A.code[p1]) == kCodeTypeFloating;
#pragma unroll
  for (int i = 0; i < 6; i++) q.tau[i] = kSps ? A.tau[6 * size_t(p1) + i] : 0.f;
  // This lane's sums: component k of {ax, ay, az, ar}, the diffusion, the
  // largest dot_rr2 of its pairs, strain diagonal k and off-diagonal k
  // (xy, xz, yz).
  float s = 0.f, delta = 0.f, visc = 0.f, sd = 0.f, so = 0.f;
  bool cancel = q.ftp1;
  int cx, cy, cz;
  {
    const unsigned cel = A.dcell[p1];
    cx = int(dcel_cellx(dvd.domcellcode, cel)) - dvd.czx;
    cy = int(dcel_celly(dvd.domcellcode, cel)) - dvd.czy;
    cz = int(dcel_cellz(dvd.domcellcode, cel)) - dvd.czz;
  }
  const int pfx = pscel_fx(q.ps.w), pfy = pscel_fy(q.ps.w), pfz = pscel_fz(q.ps.w);
  const int sc = dvd.scelldiv;
  float f1x = 0, f1y = 0, f1z = 0;  // own cell offsets from the group's, biased

  // Neighbours are numbered as they are appended: [tail, scanned) tested and in
  // the ring, [scanned, head) in the ring only (uniform). Queue of the team:
  // qh taken, qn appended, qe[b] appended up to the end of the b-th block of
  // 64 from tail on.
  unsigned head = 0, scanned = 0, tail = 0;
  unsigned qh = 0, qn = 0, qe[3] = {0, 0, 0};
  uint8_t* const queue = lds.queue[team];
  const unsigned kf = k < 3 ? 0xffffffffu : 0u;
  const float* const term = reinterpret_cast<const float*>(lds.term);
  constexpr unsigned kRec = 4 * team_kt<TVISCO, BP1>();   // floats per record
  const unsigned tbase = team * (kTeam * kRec + 4);

  // Records of the last round, added during the next one: their way through LDS
  // and the chain of additions are covered by the pair body.
  struct Rec { float2 ac[4]; float f[4], d[4], e[4], m[4], uk[4], ua[4], ub[4], fa[4], fb[4]; };
  float dlp = 0.f;   // this lane's diffusion term of the last round
  auto read = [&](Rec& v) {
#pragma unroll
    for (unsigned j = 0; j < kTeam; j++) {
      const float* const r = term + tbase + j * kRec;
      v.ac[j] = *reinterpret_cast<const float2*>(r + (BP1 || k < 3 ? 0 : 2));
      if (BP1) continue;
      v.f[j] = r[4 + k];
      if (TVISCO != DSPH_VISCO_ARTIFICIAL) v.d[j] = r[8 + k];
      if (kSps) {
        const unsigned ia = k < 2 ? 0 : 1, ib = k == 0 ? 1 : 2;
        v.e[j] = r[12 + k]; v.m[j] = r[19]; v.uk[j] = r[16 + k];
        v.ua[j] = r[16 + ia]; v.ub[j] = r[16 + ib]; v.fa[j] = r[4 + ia]; v.fb[j] = r[4 + ib];
      }
    }
  };
  auto add = [&](const Rec& v) {
    const float dl[4] = {team_lane<0>(dlp), team_lane<1>(dlp), team_lane<2>(dlp),
                         team_lane<3>(dlp)};
#pragma unroll
    for (unsigned j = 0; j < kTeam; j++) {
      s += v.ac[j].x * (BP1 ? v.ac[j].y : v.f[j]);
      if (BP1) continue;
      if (TVISCO == DSPH_VISCO_ARTIFICIAL)
        s += v.ac[j].y * __uint_as_float(__float_as_uint(v.f[j]) & kf);
      else
        s += v.ac[j].y * v.d[j];
      if (kSps) {
        s += v.m[j] * v.e[j];
        // Strain: diagonal u_k fr_k, off-diagonals xy, xz, yz.
        sd += __uint_as_float(__float_as_uint(v.uk[j]) & kf) * v.f[j];
        so += v.ua[j] * v.fb[j];
        so += v.ub[j] * v.fa[j];
      }
      if (TDDT != DSPH_DDT_NONE) delta = delta - dl[j];
    }
  };

  struct Nb { float4 ps, vr; float pr; P2x x; bool has; };
  // Evaluates the next four hits of every team, one a lane, its times.
  auto process = [&](auto kb, const PairK& pk, int its) {
    constexpr bool KB = decltype(kb)::value;
    auto fetch = [&](Nb& b) {
      const unsigned i = qh + k;
      b.has = int(qn - i) > 0;
      const unsigned e = queue[i & (kQueue - 1)];
      qh = min(qh + kTeam, qn);
      b.ps = lds.pos[e];
      b.vr = lds.vr[e];
      if (!BP1) b.pr = lds.pr[e];
      if (kM) b.x.mass = lds.m[e];
      constexpr unsigned kNx = kSps && !KB ? 6u : (MDBC2 && KB ? 3u : 0u);
#pragma unroll
      for (unsigned j = 0; j < kNx; j++) b.x.t[j] = lds.x[kX * e + j];
    };
    auto eval = [&](Nb& b) {
      const unsigned w = __float_as_uint(b.ps.w);
      b.x.flags = w >> 24;
      float3 dr;
      dr.x = q.ps.x - b.ps.x + pk.pcs * (f1x - float(w & 0xffu));
      dr.y = q.ps.y - b.ps.y + pk.pcs * (f1y - float((w >> 8) & 0xffu));
      dr.z = q.ps.z - b.ps.z + pk.pcs * (f1z - float((w >> 16) & 0xffu));
      const float rr2 = dr.x * dr.x + dr.y * dr.y + dr.z * dr.z;
      const bool ok = b.has && rr2 <= pk.ks2 && rr2 >= kAlmostZero;
      float* const rec = reinterpret_cast<float*>(lds.term) + tbase + k * kRec;
      Rec r;
      read(r);
      wave_sync();
      if constexpr (BP1) {
        const float mass = FT ? b.x.mass : pk.mass;
        const float rad = fast_sqrt(rr2);
        const float qq = rad * pk.invh;
        const float wqq1 = 1.f - 0.5f * qq;
        const float fac = pk.bwenh * wqq1 * wqq1 * wqq1;
        const float frx = fac * dr.x, fry = fac * dr.y, frz = fac * dr.z;
        const float dvx = q.vr.x - b.vr.x, dvy = q.vr.y - b.vr.y, dvz = q.vr.z - b.vr.z;
        const float mar = mass * (dvx * frx + dvy * fry + dvz * frz);
        const float rr = fast_div(q.vr.w, b.vr.w);
        const float dot = dr.x * dvx + dr.y * dvy + dr.z * dvz;
        const float dot_rr2 = fast_div(dot, rr2 + pk.eta2);
        visc = fmaxf(ok ? dot_rr2 : visc, visc);
        add(r);
        *reinterpret_cast<float2*>(rec) = make_float2(ok ? mar : 0.f, ok ? rr : 0.f);
      } else {
        Terms t;
        pair_terms<TVISCO, TDDT, MDBC2, FT, KB>(ok, dr, rr2, b.vr,
                                                make_float2(b.pr, fast_rcp(b.vr.w)), b.x, q, pk, c,
                                                t, visc, cancel);
        add(r);
        dlp = t.dl;
        float4* const rec4 = reinterpret_cast<float4*>(rec);
        // Lane 3 takes the density rate: no second factor for it.
        rec4[0] = make_float4(t.p, t.c, t.mar, 0.f);
        rec4[1] = make_float4(t.frx, t.fry, t.frz, t.rr);
        if (TVISCO != DSPH_VISCO_ARTIFICIAL) rec4[2] = make_float4(t.dvx, t.dvy, t.dvz, 0.f);
        if (kSps) {
          rec4[3] = make_float4(t.ex, t.ey, t.ez, 0.f);
          rec4[4] = make_float4(t.ux, t.uy, t.uz, t.m);
        }
      }
      wave_sync();
    };
    if (its <= 0) return;
    Nb u, v;
    fetch(u);
    for (;;) {
      if (--its > 0) fetch(v);
      eval(u);
      if (its <= 0) break;
      if (--its > 0) fetch(u);
      eval(v);
      if (its <= 0) break;
    }
  };
  // Tests nb <= 64 neighbours from scanned on and queues the hits.
  auto scan = [&](unsigned nb, bool member, float m2x, float m2y, float m2z, float thr) {
    wave_sync();
    const float4* const f0 = lds.scan + (scanned & 64u ? 68u : 0u) + 17 * k;
    unsigned bits = 0;
#pragma unroll
    for (unsigned j = 0; j < 16; j++) {
      const float4 f = f0[j];
      float d = fmaf(m2x, f.x, f.w);
      d = fmaf(m2y, f.y, d);
      d = fmaf(m2z, f.z, d);
      shift_in_le(bits, d, thr);
    }
    // Neighbour 16 k + j is at bit 15 - j.
    bits = __builtin_bitreverse32(bits) >> 16;
    const int nk = min(max(int(nb) - int(16 * k), 0), 16);
    bits = member ? bits & ((1u << nk) - 1u) : 0u;
    const unsigned a = unsigned(__popc(bits));
    const unsigned b1 = dpp_u<kDppSwap1>(a), pair = a + b1, pair2 = dpp_u<kDppSwap2>(pair);
    unsigned w = qn + (k & 1 ? b1 : 0u) + (k & 2 ? pair2 : 0u);
    qn += pair + pair2;
    const unsigned e0 = scanned % kRingN + 16 * k;
    while (__ballot(bits != 0)) {
      if (bits) {
        queue[w & (kQueue - 1)] = uint8_t(e0 + unsigned(__builtin_ctz(bits)));
        bits &= bits - 1u;
        w++;
      }
    }
    const unsigned blk = (scanned - tail) / 64;
#pragma unroll
    for (unsigned j = 0; j < 3; j++) qe[j] = blk == j ? qn : qe[j];
    scanned += nb;
    wave_sync();
  };

  // A lane without a hit reads some entry of the queue and the neighbour it names,
  // whose contents do not count but for a finite position (the kernel gradient
  // is not masked): entries name places of the ring and positions are finite
  // from the start (neighbours with a position that is not fail the box test).
  static_assert(sizeof(lds.queue) % 4 == 0, "the queues are cleared word by word");
  for (unsigned i = lane; i < sizeof(lds.queue) / 4; i += 64)
    reinterpret_cast<unsigned*>(lds.queue)[i] = 0u;
  for (unsigned i = lane; i < kRingN; i += 64) lds.pos[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (unsigned i = 0; i < kRec; i++) reinterpret_cast<float*>(lds.term)[tbase + k * kRec + i] = 0.f;
  wave_sync();

  bool pending = valid && fit;
  for (;;) {
    const unsigned long long pend = __ballot(pending);
    if (!pend) break;
    const int leader = __builtin_ctzll(pend);
    const int gx = __builtin_amdgcn_readlane(cx, leader), gy = __builtin_amdgcn_readlane(cy, leader),
              gz = __builtin_amdgcn_readlane(cz, leader);
    const int rfx = __builtin_amdgcn_readlane(pfx, leader), rfy = __builtin_amdgcn_readlane(pfy, leader),
              rfz = __builtin_amdgcn_readlane(pfz, leader);
    const bool member = pending && cy == gy && cz == gz && unsigned(cx - gx) < unsigned(kSpan) &&
                        max(max(abs(pfx - rfx), abs(pfy - rfy)), abs(pfz - rfz)) <= kNear;
    pending = pending && !member;
    const int gxmax = gx + int(-teams_min(member ? -float(cx - gx) : 0.f));
    const int X0 = gx - min(gx, sc), X1 = gxmax + min(dvd.ncx - gxmax - 1, sc) + 1;
    const int Y0 = gy - min(gy, sc), Y1 = gy + min(dvd.ncy - gy - 1, sc) + 1;
    const int Z0 = gz - min(gz, sc), Z1 = gz + min(dvd.ncz - gz - 1, sc) + 1;
    // Positions relative to the leader's PosCell, the box of the group's
    // particles, and the lane's threshold of the expanded distance test
    // |q1|^2 + |q2|^2 - 2 q1.q2 <= thr (q relative to the box centre).
    // Rounding: coordinates are below 2^4 cells, so a distance is off by less
    // than 2^-18 cells, covered by the 4e-5 of the box test and of thr; the
    // expanded form by 8 * 2^-24 * (2Q)^2 with Q = max|q1| + 2h.
    if (member) {
      f1x = float(pfx - rfx + kCellBias);
      f1y = float(pfy - rfy + kCellBias);
      f1z = float(pfz - rfz + kCellBias);
    }
    const float q1x = c.pcs * float(pfx - rfx) + q.ps.x, q1y = c.pcs * float(pfy - rfy) + q.ps.y,
                q1z = c.pcs * float(pfz - rfz) + q.ps.z;
    const float bx0 = teams_min(member ? q1x : FLT_MAX), bx1 = -teams_min(member ? -q1x : FLT_MAX);
    const float by0 = teams_min(member ? q1y : FLT_MAX), by1 = -teams_min(member ? -q1y : FLT_MAX);
    const float bz0 = teams_min(member ? q1z : FLT_MAX), bz1 = -teams_min(member ? -q1z : FLT_MAX);
    float ox = 0.5f * (bx0 + bx1), oy = 0.5f * (by0 + by1), oz = 0.5f * (bz0 + bz1);
    float ex = 0.5f * (bx1 - bx0), ey = 0.5f * (by1 - by0), ez = 0.5f * (bz1 - bz0);
    float box2 = c.ks2 * 1.00004f, pcs = c.pcs;
    pin(ox); pin(oy); pin(oz); pin(ex); pin(ey); pin(ez); pin(box2); pin(pcs);
    const float qx = q1x - ox, qy = q1y - oy, qz = q1z - oz;
    const float s1 = qx * qx + qy * qy + qz * qz;
    const float qm = sqrtf(ex * ex + ey * ey + ez * ez) + 1.01f * sqrtf(c.ks2);
    const float thr = c.ks2 * 1.00004f - s1 + 2.0e-6f * qm * qm;
    const float m2x = -2.f * qx, m2y = -2.f * qy, m2z = -2.f * qz;
    const int ny = Y1 - Y0, nrows = ny * (Z1 - Z0);

    auto kind = [&](auto kb) {
      constexpr bool KB = decltype(kb)::value;
      const PairK pk = pair_k<TVISCO, TDDT>(c, KB, KB ? viscob : viscof);
      // Rows r0.. of the group, one a lane (9 in all, or 25 of half cells).
      int r0 = 0;
      unsigned rini = 0, rfin = 0;
      unsigned long long rows = 0;
      auto load_rows = [&]() {
        const int r = r0 + int(lane);
        rini = rfin = 0;
        if (r < nrows) {
          const int z = Z0 + r / ny, y = Y0 + r % ny;
          const int2* bc =
              dvd.begincell + ((KB ? 0 : int(dvd.cellfluid)) + z * dvd.ncw + y * dvd.ncx);
          for (int cl = X0; cl < X1; cl += 4) {   // row_range, four loads at a time
            int2 be[4];
#pragma unroll
            for (int j = 0; j < 4; j++) be[j] = bc[min(cl + j, X1 - 1)];
#pragma unroll
            for (int j = 0; j < 4; j++)
              if (be[j].y) {
                if (!rfin) rini = unsigned(be[j].x);
                rfin = unsigned(be[j].y);
              }
          }
        }
        rows = __ballot(rfin > rini);
        r0 += 64;
      };
      // The next 64 to come: their positions are loaded while the current
      // ones are worked on.
      unsigned t = 0, gfin = 0, ni = 0;
      float4 nps = make_float4(0, 0, 0, 0);
      bool nin = false;
      auto advance = [&]() {
        if (t >= gfin) {
          while (!rows) {
            if (r0 >= nrows) return false;
            load_rows();
          }
          const int rr = __builtin_ctzll(rows);
          rows &= rows - 1;
          t = unsigned(__builtin_amdgcn_readlane(int(rini), rr));
          gfin = unsigned(__builtin_amdgcn_readlane(int(rfin), rr));
        }
        nin = t + lane < gfin;
        ni = nin ? t + lane : t;
        t += 64;
        nps = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(A.poscell) +
                                               (ni << 4));
        return true;
      };
      bool more = advance();
      if (!more) return;
      bool held = false;   // 64 neighbours in registers
      float4 ps = nps, vr = nps;
      float pr = 0;
      unsigned ci = 0, add = 0;
      int dx = 0, dy = 0, dz = 0;
      float x = 0, y = 0, z = 0, s2 = 0;
      bool keep = false;
      unsigned long long kept = 0;
      for (;;) {
        if (!held && more) {
          const bool in = nin;
          ps = nps;
          ci = ni;
          vr = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(A.velrho) +
                                                (ci << 4));
          if (!BP1)
            pr = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(A.press) +
                                                 (ci << 3));
          more = advance();
          // Box test.
          dx = pscel_fx(ps.w) - rfx; dy = pscel_fy(ps.w) - rfy; dz = pscel_fz(ps.w) - rfz;
          x = pcs * float(dx) + ps.x - ox;
          y = pcs * float(dy) + ps.y - oy;
          z = pcs * float(dz) + ps.z - oz;
          const float hx = fmaxf(fabsf(x) - ex, 0.f), hy = fmaxf(fabsf(y) - ey, 0.f),
                      hz = fmaxf(fabsf(z) - ez, 0.f);
          s2 = x * x + y * y + z * z;
          keep = in && hx * hx + hy * hy + hz * hz <= box2 && s2 < 1e30f;
          kept = __ballot(keep);
          add = unsigned(__popcll(kept));
          held = true;
        }
        // Append them if the ring has room, or make room by using up its
        // oldest block; test a block of 64 if the queues have room (64 hits at
        // most), or make room there; at the end use up all.
        int its = 0;
        bool fin = false;
        if (held && head - scanned < 64) {
          if (head + add - tail <= kRingN) {
            if (keep) {
              const unsigned rank = __builtin_amdgcn_mbcnt_hi(
                  unsigned(kept >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(kept), 0));
              const unsigned si = (head + rank) & 127u;
              lds.scan[si + (si >> 4)] = make_float4(x, y, z, s2);
              const unsigned i = head % kRingN + rank, e = min(i, i - kRingN);
              P2x o;
              load_p2x<TVISCO, MDBC2, FT, KB>(ci, c, A, o);
              const unsigned w = (unsigned(dx + kCellBias) & 0xffu) |
                                 ((unsigned(dy + kCellBias) & 0xffu) << 8) |
                                 ((unsigned(dz + kCellBias) & 0xffu) << 16) | (o.flags << 24);
              lds.pos[e] = make_float4(ps.x, ps.y, ps.z, __uint_as_float(w));
              lds.vr[e] = vr;
              if (!BP1) lds.pr[e] = pr;
              if (kM) lds.m[e] = o.mass;
              constexpr unsigned kNx = kSps && !KB ? 6u : (MDBC2 && KB ? 3u : 0u);
#pragma unroll
              for (unsigned j = 0; j < kNx; j++) lds.x[kX * e + j] = o.t[j];
            }
            head += add;
            held = false;
          } else {
            its = (teams_max_i(int(qe[0] - qh)) + 3) >> 2;
            tail += 64;
            qe[0] = qe[1]; qe[1] = qe[2];
          }
        }
        const unsigned left = head - scanned;
        const bool end = !held && !more;
        if (left >= 64 || (end && left)) {
          const int over = teams_max_i(int(qn - qh)) - int(kQueue - 64);
          if (over > 0) {
            its = (over + 3) >> 2;
          } else {
            scan(min(left, 64u), member, m2x, m2y, m2z, thr);
            // Rounds that every team of the group can fill.
            its = -teams_max_i(member ? -int(qn - qh) : -0x7fffffff) >> 2;
          }
        } else if (end) {
          its = (teams_max_i(int(qn - qh)) + 3) >> 2;
          fin = true;
        }
        process(kb, pk, its);
        if (fin) break;
      }
      head = scanned = tail = 0;
    };
    kind(std::false_type());
    if constexpr (!BP1) kind(std::true_type());
  }
  {
    Rec r;
    read(r);
    add(r);
  }
  // Lane 0 of the team gathers the sums.
  visc = fmaxf(visc, dpp_f<kDppSwap1>(visc));
  visc = fmaxf(visc, dpp_f<kDppSwap2>(visc));
  if constexpr (BP1) {
    if (valid && k == 0 && (s != 0 || visc != 0)) {
      A.ar[p1] += s;
      if (visc > A.viscdt[p1]) A.viscdt[p1] = visc;
    }
  } else {
    unsigned can = cancel ? 1u : 0u;
    can |= dpp_u<kDppSwap1>(can);
    can |= dpp_u<kDppSwap2>(can);
    Acc a;
    acc_init(a);
    a.ax = team_lane<0>(s); a.ay = team_lane<1>(s); a.az = team_lane<2>(s); a.ar = team_lane<3>(s);
    a.visc = visc;
    a.delta = can ? FLT_MAX : delta;
    if (kSps) {
      a.s[0] = team_lane<0>(sd); a.s[3] = team_lane<1>(sd); a.s[5] = team_lane<2>(sd);
      a.s[1] = team_lane<0>(so); a.s[2] = team_lane<1>(so); a.s[4] = team_lane<2>(so);
    }
    if (valid && k == 0)
      store_results<TVISCO, TDDT, false>(p1, a, A.viscdt, A.ar, A.ace, A.strain, nullptr);
  }
}

// Three waves per SIMD are what the LDS of ring, queues and records allows (12
// waves per CU; a ring of 256 with 8 of them: 12.0 ms where this takes 10.6).
template <int TVISCO, int TDDT, bool MDBC2, bool FT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 8)))
k_forces_fluid_team(unsigned n, unsigned pinit, float viscob, float viscof, DivData dvd, Cte c,
                    TeamArrays A) {
  __shared__ TeamLds<true, team_kx<TVISCO, MDBC2>(), MDBC2 || FT, team_kt<TVISCO, false>()> lds;
  team_body<TVISCO, TDDT, MDBC2, FT, false>(xcd_block(blockIdx.x, gridDim.x) * kTeamP, n, pinit,
                                            viscob, viscof, dvd, c, A, lds);
}

template <bool FT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_forces_bound_team(unsigned n, DivData dvd, Cte c, TeamArrays A) {
  __shared__ TeamLds<false, 0, FT, 1> lds;
  team_body<DSPH_VISCO_ARTIFICIAL, DSPH_DDT_NONE, false, FT, true>(
      xcd_block(blockIdx.x, gridDim.x) * kTeamP, n, 0, 0.f, 0.f, dvd, c, A, lds);
}

TeamArrays team_arrays(const dsph_inter_parms* t, const float2* press) {
  TeamArrays A;
  A.dcell = t->d_dcell;
  A.poscell = (const float4*)t->d_poscell;
  A.velrho = (const float4*)t->d_velrho;
  A.press = press;
  A.tau = t->d_spstaurho2;
  A.viscdt = t->d_viscdt;
  A.ar = t->d_ar;
  A.ace = t->d_ace;
  A.strain = t->d_sps2strain;
  A.bmode = t->d_boundmode;
  A.tangenvel = t->d_tangenvel;
  A.code = t->d_code;
  A.ftomassp = t->d_ftomassp;
  return A;
}

enum class FluidForm { kTeam, kTile, kRows };

// Form of the fluid interaction (all give the same bits).
// Teams win while the chip is not full of the tile kernel's waves of 64
// particles, the tile kernel (5 waves per SIMD against 3, fewer LDS accesses
// per pair) above. Measured, us, team / tile:
//   artificial  3-D   80k fluid particles 253 / 379, 157k 424 / 443, 234k 591 / 528
//   laminar     3-D   80k 280 / 378, 157k 467 / 437, 234k 656 / 519
//   Laminar+SPS 3-D   80k 451 / 490, 157k 781 / 565
//   artificial  2-D (step)  120k 453 / 465, 480k 769 / 662
//   mDBC2 (laminar, step)   122k 1466 / 1567
// Floating bodies have no tile kernel; against rows: 92k 1020 / 2286 (step),
// 380k 2640 / 3343. Shifting has no team kernel: which boundary neighbour
// cancels it first decides what is summed.
FluidForm fluid_form(const dsph_ctx* ctx, const dsph_inter_parms* t) {
  if (ctx->forces_kernel != 0 || t->d_nopenshift) return FluidForm::kRows;
  if (t->d_ftomassp) return FluidForm::kTeam;
  if (t->d_boundmode && (t->d_shiftposfs || t->d_velgrad)) return FluidForm::kRows;
  if (t->d_shiftposfs || t->d_velgrad) return FluidForm::kTile;
  const unsigned most = t->tvisco == DSPH_VISCO_ARTIFICIAL ? 180000u
                        : t->tvisco == DSPH_VISCO_LAMINAR  ? 140000u
                                                           : 100000u;
  const unsigned npf = t->np - t->npb;
  return npf <= (ctx->cte.simulate2d ? most / 4 * 3 : most) ? FluidForm::kTeam : FluidForm::kTile;
}

template <int TVISCO, int TDDT, bool VELGRAD>
void launch_fluid(dsph_ctx* ctx, const dsph_inter_parms* t, const DivData& dvd, const Cte& c,
                  const float2* press) {
  KTimer kt(ctx, "k_forces_fluid");
  const unsigned npf = t->np - t->npb;
  const FluidForm form = fluid_form(ctx, t);
  if (form == FluidForm::kTeam) {
    if constexpr (!VELGRAD) {
      const unsigned g = grid_for(npf, kTeamP);
      const TeamArrays A = team_arrays(t, press);
      if (t->d_ftomassp)
        k_forces_fluid_team<TVISCO, TDDT, false, true><<<g, 64, 0, ctx->stream>>>(
            npf, t->npb, t->viscob, t->viscof, dvd, c, A);
      else if (t->d_boundmode)
        k_forces_fluid_team<TVISCO, TDDT, true, false><<<g, 64, 0, ctx->stream>>>(
            npf, t->npb, t->viscob, t->viscof, dvd, c, A);
      else
        k_forces_fluid_team<TVISCO, TDDT, false, false><<<g, 64, 0, ctx->stream>>>(
            npf, t->npb, t->viscob, t->viscof, dvd, c, A);
    }
  } else if (t->d_nopenshift) {
    // mDBC2 with no penetration: the one-lane-per-particle kernel with the
    // no-penetration sums (shifting and floating bodies are refused with it
    // by dsph_interaction_forces).
    k_forces_fluid_rows<TVISCO, TDDT, VELGRAD, true, false, false, true>
        <<<grid_for(npf, kBsForces), kBsForces, 0, ctx->stream>>>(
            npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell, (const float4*)t->d_poscell,
            (const float4*)t->d_velrho, press, t->d_spstaurho2, t->d_viscdt, t->d_ar, t->d_ace,
            t->d_sps2strain, t->d_velgrad, t->d_boundmode, t->d_tangenvel, 0, nullptr, nullptr,
            nullptr, t->d_boundnor, (float4*)t->d_nopenshift, t->d_motionvel);
  } else if (t->d_ftomassp) {
    // Floating bodies, rows kernel requested (shifting, mDBC2 and the velocity gradient are refused with them
    // by dsph_interaction_forces).
    if constexpr (!VELGRAD)
      k_forces_fluid_rows<TVISCO, TDDT, false, false, false, true>
          <<<grid_for(npf, kBsForces), kBsForces, 0, ctx->stream>>>(
              npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell, (const float4*)t->d_poscell,
              (const float4*)t->d_velrho, press, t->d_spstaurho2, t->d_viscdt, t->d_ar, t->d_ace,
              t->d_sps2strain, nullptr, nullptr, nullptr, 0, t->d_code, nullptr, t->d_ftomassp);
  } else if (t->d_shiftposfs && t->d_boundmode) {
    // Shifting with mDBC2 boundaries: the one-lane-per-particle kernel with
    // both rules (a boundary switched off has mass 0 in the shifting sums
    // too, JSphGpu_ker.cu:586-588, 733-740).
    k_forces_fluid_rows<TVISCO, TDDT, false, true, true><<<grid_for(npf, kBsForces), kBsForces,
                                                          0, ctx->stream>>>(
        npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell, (const float4*)t->d_poscell,
        (const float4*)t->d_velrho, press, t->d_spstaurho2, t->d_viscdt, t->d_ar, t->d_ace,
        t->d_sps2strain, nullptr, t->d_boundmode, t->d_tangenvel, t->shiftmode, t->d_code,
        (float4*)t->d_shiftposfs);
  } else if (t->d_shiftposfs && form == FluidForm::kTile) {
    // Shifting in the tile kernel (no penetration and the velocity gradient
    // are refused with shifting by dsph_interaction_forces).
    k_forces_fluid_tile<TVISCO, TDDT, false, kRingTiles, false, true>
        <<<grid_for(npf, 64 * kTileWaves), 64 * kTileWaves, 0, ctx->stream>>>(
        npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell,
        (const float4*)t->d_poscell, (const float4*)t->d_velrho, press, t->d_spstaurho2,
        t->d_viscdt, t->d_ar, t->d_ace, t->d_sps2strain, nullptr, nullptr, nullptr, t->shiftmode,
        t->d_code, (float4*)t->d_shiftposfs);
  } else if (t->d_shiftposfs) {
    k_forces_fluid_rows<TVISCO, TDDT, false, false, true><<<grid_for(npf, kBsForces), kBsForces,
                                                           0, ctx->stream>>>(
        npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell, (const float4*)t->d_poscell,
        (const float4*)t->d_velrho, press, t->d_spstaurho2, t->d_viscdt, t->d_ar, t->d_ace,
        t->d_sps2strain, nullptr, nullptr, nullptr, t->shiftmode, t->d_code,
        (float4*)t->d_shiftposfs);
  } else if (t->d_boundmode && form == FluidForm::kTile) {
    // mDBC2 boundaries in the tile kernel.
    k_forces_fluid_tile<TVISCO, TDDT, false, kRingTiles, true>
        <<<grid_for(npf, 64 * kTileWaves), 64 * kTileWaves, 0, ctx->stream>>>(
        npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell,
        (const float4*)t->d_poscell, (const float4*)t->d_velrho, press, t->d_spstaurho2,
        t->d_viscdt, t->d_ar, t->d_ace, t->d_sps2strain, nullptr, t->d_boundmode, t->d_tangenvel);
  } else if (t->d_boundmode) {
    // mDBC2 with the velocity gradient (learned closure) or the rows kernel
    // requested: the one-lane-per-particle kernel.
    k_forces_fluid_rows<TVISCO, TDDT, VELGRAD, true><<<grid_for(npf, kBsForces), kBsForces, 0,
                                                       ctx->stream>>>(
        npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell, (const float4*)t->d_poscell,
        (const float4*)t->d_velrho, press, t->d_spstaurho2, t->d_viscdt, t->d_ar, t->d_ace,
        t->d_sps2strain, t->d_velgrad, t->d_boundmode, t->d_tangenvel);
  } else if (form == FluidForm::kTile) {
    // gamma = 7 without the gradient output: the neighbour pressure is
    // evaluated in the kernel instead of being gathered (Laminar+SPS too: 127
    // registers, no spill, 9 % faster on the wave flume).
    constexpr bool kEos7Built = !VELGRAD;
    if (kEos7Built && c.gamma == 7.f)
      k_forces_fluid_tile<TVISCO, TDDT, false, kRingTiles, false, false, kEos7Built>
          <<<grid_for(npf, 64 * kTileWaves), 64 * kTileWaves, 0, ctx->stream>>>(
              npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell,
              (const float4*)t->d_poscell, (const float4*)t->d_velrho, press,
              t->d_spstaurho2, t->d_viscdt, t->d_ar, t->d_ace, t->d_sps2strain, nullptr);
    else
      k_forces_fluid_tile<TVISCO, TDDT, VELGRAD, kRingTiles>
          <<<grid_for(npf, 64 * kTileWaves), 64 * kTileWaves, 0, ctx->stream>>>(
              npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell,
              (const float4*)t->d_poscell, (const float4*)t->d_velrho, press,
              t->d_spstaurho2, t->d_viscdt, t->d_ar, t->d_ace, t->d_sps2strain, t->d_velgrad);
  } else {
    k_forces_fluid_rows<TVISCO, TDDT, VELGRAD, false><<<grid_for(npf, kBsForces), kBsForces, 0,
                                                        ctx->stream>>>(
        npf, t->npb, t->viscob, t->viscof, dvd, c, t->d_dcell, (const float4*)t->d_poscell,
        (const float4*)t->d_velrho, press, t->d_spstaurho2, t->d_viscdt, t->d_ar, t->d_ace,
        t->d_sps2strain, t->d_velgrad, nullptr, nullptr);
  }
}

template <int TVISCO, bool VELGRAD>
int dispatch_ddt(dsph_ctx* ctx, const dsph_inter_parms* t, const DivData& dvd, const Cte& c,
                 const float2* press) {
  switch (t->tdensity) {
    case DSPH_DDT_NONE: launch_fluid<TVISCO, DSPH_DDT_NONE, VELGRAD>(ctx, t, dvd, c, press); break;
    case DSPH_DDT_DDT: launch_fluid<TVISCO, DSPH_DDT_DDT, VELGRAD>(ctx, t, dvd, c, press); break;
    case DSPH_DDT_DDT2: launch_fluid<TVISCO, DSPH_DDT_DDT2, VELGRAD>(ctx, t, dvd, c, press); break;
    case DSPH_DDT_DDT2FULL:
      launch_fluid<TVISCO, DSPH_DDT_DDT2FULL, VELGRAD>(ctx, t, dvd, c, press);
      break;
    default: return set_error(ctx, DSPH_E_ARG, "dsph_interaction_forces: invalid tdensity");
  }
  return DSPH_OK;
}

// ---------------------------------------------------------------- ensembles
// The same bodies over the cases of an ensemble; the block map gives the case
// and the first case-local index of each workgroup.
__global__ void k_fill_u32(unsigned* __restrict__ a, unsigned n, unsigned v) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

__global__ void __launch_bounds__(kBs) k_ens_prep(const EnsCase* __restrict__ cases,
    const EnsState* __restrict__ st, const EnsBlock* __restrict__ pmap,
    const float4* __restrict__ velrho, float2* __restrict__ press) {
  const EnsBlock e = pmap[blockIdx.x];
  if (!st[e.x].active) return;
  const unsigned l = e.y + threadIdx.x;
  if (l >= st[e.x].np) return;
  const EnsCase& ec = cases[e.x];
  press[ec.p0 + l] = prep_one(velrho[ec.p0 + l].w, ec.c);
}

template <int TVISCO, int TDDT, unsigned kRing, bool EOS7>
__global__ void __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(tile_min_waves<TVISCO, false, false, false>(), 8)))
k_ens_fluid_tile(const EnsCase* __restrict__ cases,
    const EnsState* __restrict__ st, const EnsBlock* __restrict__ wmap,
    const unsigned* __restrict__ dcell, const float4* __restrict__ poscell, const float4* __restrict__ velrho,
    const float2* __restrict__ press, float* __restrict__ viscdt, float* __restrict__ ar,
    float* __restrict__ ace) {
  __shared__ TileLds<kRing> lds;
  const EnsBlock e = wmap[xcd_block(blockIdx.x, gridDim.x)];
  if (!st[e.x].active) return;
  const EnsCase& ec = cases[e.x];
  const unsigned npf = st[e.x].np - ec.npb;
  if (e.y >= npf) return;
  const unsigned p = e.y + threadIdx.x;
  fluid_tile_body<TVISCO, TDDT, false, kRing, false, false, EOS7>(
      p, p < npf, ec.p0 + ec.npb, ec.viscob, ec.viscof,
                                              ec.dvd, ec.c, dcell, poscell,
                                              velrho, press, nullptr, viscdt, ar, ace, nullptr,
                                              nullptr, lds);
}

// Persistent form of k_ens_fluid_tile: a grid sized to the resident waves
// pulls work items (waves of 64 fluid particles, entries of wmap) in chunks of
// `chunk` consecutive items from counters, until the list is exhausted. The
// list is split into kNumXcd contiguous segments, one per XCD (block i runs
// on XCD i % 8), so neighbouring particles stay on one L2; a wave drains its
// own XCD's segment first, then helps the others. Every wave leaves once each
// segment's counter has passed its end (counters only grow), so the grid
// drains. ctr[0..kNumXcd) must be zero at launch. Items are independent:
// the schedule changes no result.
template <int TVISCO, int TDDT, unsigned kRing, bool EOS7>
__global__ void __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(tile_min_waves<TVISCO, false, false, false>(), 8)))
k_ens_fluid_tile_persist(const EnsCase* __restrict__ cases,
    const EnsState* __restrict__ st, const EnsBlock* __restrict__ wmap, unsigned nitems,
    unsigned chunk, unsigned* __restrict__ ctr,
    const unsigned* __restrict__ dcell, const float4* __restrict__ poscell, const float4* __restrict__ velrho,
    const float2* __restrict__ press, float* __restrict__ viscdt, float* __restrict__ ar,
    float* __restrict__ ace) {
  __shared__ TileLds<kRing> lds;
  const unsigned per = nitems / kNumXcd, rem = nitems % kNumXcd;
  const unsigned x0 = blockIdx.x % kNumXcd;
  for (unsigned s = 0; s < kNumXcd; s++) {
    const unsigned x = (x0 + s) % kNumXcd;
    const unsigned seg0 = x * per + min(x, rem), segn = per + (x < rem ? 1u : 0u);
    for (;;) {
      unsigned i0 = 0;
      if (threadIdx.x == 0) i0 = atomicAdd(ctr + x, chunk);
      i0 = __builtin_amdgcn_readfirstlane(i0);
      if (i0 >= segn) break;
      const unsigned i1 = min(i0 + chunk, segn);
      for (unsigned i = i0; i < i1; i++) {
        const EnsBlock e = wmap[seg0 + i];
        if (!st[e.x].active) continue;
        const EnsCase& ec = cases[e.x];
        const unsigned npf = st[e.x].np - ec.npb;
        if (e.y >= npf) continue;
        const unsigned p = e.y + threadIdx.x;
        fluid_tile_body<TVISCO, TDDT, false, kRing, false, false, EOS7>(
            p, p < npf, ec.p0 + ec.npb, ec.viscob, ec.viscof, ec.dvd, ec.c, dcell,
            poscell, velrho, press, nullptr, viscdt, ar, ace, nullptr, nullptr, lds);
      }
    }
  }
}

template <int TVISCO, int TDDT>
__global__ void __launch_bounds__(64) k_ens_fluid_rows(const EnsCase* __restrict__ cases,
    const EnsState* __restrict__ st, const EnsBlock* __restrict__ wmap,
    const unsigned* __restrict__ dcell, const float4* __restrict__ poscell,
    const float4* __restrict__ velrho, const float2* __restrict__ press,
    float* __restrict__ viscdt, float* __restrict__ ar, float* __restrict__ ace) {
  const EnsBlock e = wmap[xcd_block(blockIdx.x, gridDim.x)];
  if (!st[e.x].active) return;
  const EnsCase& ec = cases[e.x];
  const unsigned l = e.y + threadIdx.x;
  if (l >= st[e.x].np - ec.npb) return;
  fluid_rows_body<TVISCO, TDDT, false>(ec.p0 + ec.npb + l, ec.viscob, ec.viscof, ec.dvd, ec.c,
                                       dcell, poscell, velrho, press, nullptr, viscdt, ar, ace,
                                       nullptr, nullptr);
}

// Any block size up to kEnsBsBoundMax; bmap has one entry per block of
// blockDim.x boundary particles.
__global__ void __launch_bounds__(kEnsBsBoundMax) k_ens_bound(const EnsCase* __restrict__ cases,
    const EnsState* __restrict__ st, const EnsBlock* __restrict__ bmap,
    const unsigned* __restrict__ dcell, const float4* __restrict__ poscell,
    const float4* __restrict__ velrho, float* __restrict__ viscdt, float* __restrict__ ar) {
  const EnsBlock e = bmap[xcd_block(blockIdx.x, gridDim.x)];
  if (!st[e.x].active) return;
  const unsigned l = e.y + threadIdx.x;
  if (l >= st[e.x].npbok) return;
  const EnsCase& ec = cases[e.x];
  bound_body<false>(ec.p0 + l, ec.dvd, ec.c, dcell, poscell, velrho, viscdt, ar);
}

// The boundary interaction of an ensemble with teams (k_forces_bound_team per
// case): bmap has one entry per 64 boundary particles, four waves each.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_ens_bound_team(const EnsCase* __restrict__ cases, const EnsState* __restrict__ st,
    const EnsBlock* __restrict__ bmap, TeamArrays A) {
  __shared__ TeamLds<false, 0, false, 1> lds;
  const unsigned b = xcd_block(blockIdx.x, gridDim.x);
  const EnsBlock e = bmap[b / kTeam];
  if (!st[e.x].active) return;
  const unsigned npbok = st[e.x].npbok, l0 = e.y + (b % kTeam) * kTeamP;
  if (l0 >= npbok) return;
  const EnsCase& ec = cases[e.x];
  // The rows walk costs 12 bytes of spills here (185 -> 216 us for 20 cases).
  team_body<DSPH_VISCO_ARTIFICIAL, DSPH_DDT_NONE, false, false, true, true>(
      l0, npbok, ec.p0, 0.f, 0.f, ec.dvd, ec.c, A, lds);
}

template <int TVISCO, int TDDT, bool EOS7>
void launch_ens_fluid(dsph_ctx* ctx, int variant, const EnsCase* cases, const EnsState* st,
                      const EnsBlock* wmap, unsigned nb, const EnsPersist* pers,
                      const unsigned* dcell,
                      const float4* poscell, const float4* velrho,
                      const float2* press, float* viscdt, float* ar, float* ace) {
  if (pers) {
    const unsigned g = pers->grid;
    switch (variant) {
      case kEnsTileRing8:
        k_ens_fluid_tile_persist<TVISCO, TDDT, 8, EOS7><<<g, 64, 0, ctx->stream>>>(
            cases, st, wmap, nb, pers->chunk, pers->ctr, dcell, poscell, velrho, press,
            viscdt, ar, ace);
        break;
      case kEnsTileRing12:
        k_ens_fluid_tile_persist<TVISCO, TDDT, 12, EOS7><<<g, 64, 0, ctx->stream>>>(
            cases, st, wmap, nb, pers->chunk, pers->ctr, dcell, poscell, velrho, press,
            viscdt, ar, ace);
        break;
      default:
        k_ens_fluid_tile_persist<TVISCO, TDDT, 16, EOS7><<<g, 64, 0, ctx->stream>>>(
            cases, st, wmap, nb, pers->chunk, pers->ctr, dcell, poscell, velrho, press,
            viscdt, ar, ace);
        break;
    }
    return;
  }
  switch (variant) {
    case kEnsTileRing8:
      k_ens_fluid_tile<TVISCO, TDDT, 8, EOS7><<<nb, 64, 0, ctx->stream>>>(
          cases, st, wmap, dcell, poscell, velrho, press, viscdt, ar, ace);
      break;
    case kEnsTileRing12:
      k_ens_fluid_tile<TVISCO, TDDT, 12, EOS7><<<nb, 64, 0, ctx->stream>>>(
          cases, st, wmap, dcell, poscell, velrho, press, viscdt, ar, ace);
      break;
    case kEnsTileRing16:
      k_ens_fluid_tile<TVISCO, TDDT, 16, EOS7><<<nb, 64, 0, ctx->stream>>>(
          cases, st, wmap, dcell, poscell, velrho, press, viscdt, ar, ace);
      break;
    default:
      k_ens_fluid_rows<TVISCO, TDDT><<<nb, 64, 0, ctx->stream>>>(
          cases, st, wmap, dcell, poscell, velrho, press, viscdt, ar, ace);
      break;
  }
}

}  // namespace

namespace dsph {

int ens_prep(dsph_ctx* ctx, const EnsCase* cases, const EnsState* st, const EnsBlock* pmap,
             unsigned npblocks, const float4* velrho, float2* press) {
  if (!npblocks) return DSPH_OK;
  KTimer kt(ctx, "k_prep");
  k_ens_prep<<<npblocks, kBs, 0, ctx->stream>>>(cases, st, pmap, velrho, press);
  DSPH_LAUNCHED(ctx, "k_ens_prep");
  return DSPH_OK;
}

int ens_forces_fluid(dsph_ctx* ctx, int variant, int tvisco, int tddt, bool eos7,
                     const EnsCase* cases, const EnsState* st, const EnsBlock* wmap,
                     unsigned nblocks, const EnsPersist* pers, const unsigned* dcell,
                     const float4* poscell,
                     const float4* velrho, const float2* press,
                     float* viscdt, float* ar, float* ace) {
  if (!nblocks) return DSPH_OK;
  DSPH_REQUIRE(ctx, variant >= 0 && variant < kEnsNumVariants, "ensemble: invalid kernel variant");
  if (pers) {
    DSPH_REQUIRE(ctx, variant != kEnsRows64, "ensemble: the persistent form runs the tile kernel");
    DSPH_REQUIRE(ctx, pers->ctr && pers->grid && pers->chunk,
                 "ensemble: persistent launch without counters, grid or chunk");
    // The counters start at zero (fill kernel: safe inside a captured graph).
    k_fill_u32<<<1, kNumXcd, 0, ctx->stream>>>(pers->ctr, kNumXcd, 0u);
    DSPH_LAUNCHED(ctx, "k_fill_u32");
  }
  KTimer kt(ctx, "k_forces_fluid");
#define DSPH_ENS_FLUID(V, D)                                                              \
  (eos7 ? launch_ens_fluid<V, D, true>(ctx, variant, cases, st, wmap, nblocks, pers, dcell,   \
                                       poscell, velrho, press, viscdt, ar, ace)         \
        : launch_ens_fluid<V, D, false>(ctx, variant, cases, st, wmap, nblocks, pers, dcell,  \
                                        poscell, velrho, press, viscdt, ar, ace))
  if (tvisco == DSPH_VISCO_ARTIFICIAL && tddt == DSPH_DDT_DDT2FULL)
    DSPH_ENS_FLUID(DSPH_VISCO_ARTIFICIAL, DSPH_DDT_DDT2FULL);
  else if (tvisco == DSPH_VISCO_ARTIFICIAL && tddt == DSPH_DDT_NONE)
    DSPH_ENS_FLUID(DSPH_VISCO_ARTIFICIAL, DSPH_DDT_NONE);
  else if (tvisco == DSPH_VISCO_LAMINAR && tddt == DSPH_DDT_DDT2FULL)
    DSPH_ENS_FLUID(DSPH_VISCO_LAMINAR, DSPH_DDT_DDT2FULL);
  else if (tvisco == DSPH_VISCO_LAMINAR && tddt == DSPH_DDT_NONE)
    DSPH_ENS_FLUID(DSPH_VISCO_LAMINAR, DSPH_DDT_NONE);
  else
    return set_error(ctx, DSPH_E_ARG,
                     "ensembles are built for artificial or laminar viscosity with "
                     "DDT2Full or no density diffusion");
#undef DSPH_ENS_FLUID
  DSPH_LAUNCHED(ctx, "k_ens_fluid");
  return DSPH_OK;
}

int ens_forces_bound(dsph_ctx* ctx, const EnsCase* cases, const EnsState* st,
                     const EnsBlock* bmap, unsigned nblocks, unsigned bs, const unsigned* dcell,
                     const float4* poscell, const float4* velrho, float* viscdt, float* ar) {
  if (!nblocks) return DSPH_OK;
  DSPH_REQUIRE(ctx, bs >= 64 && bs <= kEnsBsBoundMax && bs % 64 == 0,
               "ensemble: boundary block size must be a multiple of 64 up to 256");
  KTimer kt(ctx, "k_forces_bound");
  k_ens_bound<<<nblocks, bs, 0, ctx->stream>>>(cases, st, bmap, dcell, poscell, velrho,
                                              viscdt, ar);
  DSPH_LAUNCHED(ctx, "k_ens_bound");
  return DSPH_OK;
}

int ens_forces_bound_team(dsph_ctx* ctx, const EnsCase* cases, const EnsState* st,
                          const EnsBlock* bmap64, unsigned nblocks, const unsigned* dcell,
                          const float4* poscell, const float4* velrho, float* viscdt, float* ar) {
  if (!nblocks) return DSPH_OK;
  KTimer kt(ctx, "k_forces_bound");
  TeamArrays A = {};
  A.dcell = dcell;
  A.poscell = poscell;
  A.velrho = velrho;
  A.viscdt = viscdt;
  A.ar = ar;
  k_ens_bound_team<<<nblocks * kTeam, 64, 0, ctx->stream>>>(cases, st, bmap64, A);
  DSPH_LAUNCHED(ctx, "k_ens_bound_team");
  return DSPH_OK;
}

}  // namespace dsph

extern "C" {

int dsph_ctx_set_option(dsph_ctx* ctx, int key, int value) {
  if (!ctx) return DSPH_E_ARG;
  switch (key) {
    case DSPH_OPT_FORCES_KERNEL:
      DSPH_REQUIRE(ctx, value == 0 || value == 1, "forces kernel must be 0 (staged) or 1 (rows)");
      ctx->forces_kernel = value;
      return DSPH_OK;
    case DSPH_OPT_BOUND_KERNEL:
      DSPH_REQUIRE(ctx, value >= 0 && value <= 2,
                   "boundary kernel must be 0 (auto), 1 (staged) or 2 (rows)");
      ctx->bound_kernel = value;
      return DSPH_OK;
    default: return set_error(ctx, DSPH_E_ARG, "unknown option");
  }
}

}  // extern "C"

namespace {

// Argument checks shared by the interaction entry points.
int check_inter_parms(dsph_ctx* ctx, const dsph_inter_parms* t) {
  if (!ctx->cte_set) return set_error(ctx, DSPH_E_STATE, "constants not set");
  DSPH_REQUIRE(ctx, t->tkernel == DSPH_KERNEL_WENDLAND, "only the Wendland kernel is built");
  DSPH_REQUIRE(ctx, t->np >= t->npb && t->npb >= t->npbok, "invalid particle counts");
  DSPH_REQUIRE(ctx, t->np < DSPH_NP_LIMIT,
               "dsph_interaction_forces: np >= DSPH_NP_LIMIT (2^28: 32-bit byte offsets)");
  DSPH_REQUIRE(ctx, t->d_dcell && t->d_poscell && t->d_velrho && t->d_viscdt && t->d_ar &&
                        t->d_ace && t->divdata.d_beginendcell,
               "dsph_interaction_forces: null array");
  DSPH_REQUIRE(ctx, !t->d_boundmode || t->d_tangenvel, "mDBC2 needs boundmode and tangenvel");
  DSPH_REQUIRE(ctx, !t->d_shiftposfs || (t->shiftmode >= 1 && t->shiftmode <= 3 && t->d_code),
               "shifting needs shiftmode 1..3 and the particle codes");
  DSPH_REQUIRE(ctx, !t->d_shiftposfs || (!t->d_nopenshift && !t->d_velgrad),
               "shifting with mDBC2 no penetration or the velocity gradient is not built");
  DSPH_REQUIRE(ctx, !t->d_ftomassp || t->d_code, "floating bodies need the particle codes");
  DSPH_REQUIRE(ctx, !t->d_ftomassp || (!t->d_shiftposfs && !t->d_boundmode && !t->d_velgrad),
               "floating bodies with shifting, mDBC2 or the velocity gradient are not built");
  DSPH_REQUIRE(ctx, !t->d_nopenshift || (t->d_boundmode && t->d_boundnor),
               "no penetration needs mDBC2 (boundmode, tangenvel) and the boundary normals");
  const bool sps = t->tvisco == DSPH_VISCO_LAMINARSPS;
  DSPH_REQUIRE(ctx, !sps || (t->d_spstaurho2 && t->d_sps2strain),
               "Laminar+SPS needs spstaurho2 and sps2strain");
  return DSPH_OK;
}

// The interaction with the per-particle preparation in press (np
// entries): k_prep, the fluid kernel, the boundary kernel.
int interaction_forces(dsph_ctx* ctx, const dsph_inter_parms* t, float2* press) {
  const Cte c = make_cte(ctx->cte);
  const DivData dvd = make_divdata(t->divdata);
  const unsigned npf = t->np - t->npb;
  int rc = DSPH_OK;
  if (npf) {
    {
      KTimer kt(ctx, "k_prep");
      k_prep<<<grid_for(t->np, kBs), kBs, 0, ctx->stream>>>(
          t->np, (const float4*)t->d_velrho, press, c);
    }
    const bool vg = t->d_velgrad != nullptr;
    switch (t->tvisco) {
      case DSPH_VISCO_ARTIFICIAL:
        rc = vg ? dispatch_ddt<DSPH_VISCO_ARTIFICIAL, true>(ctx, t, dvd, c, press)
                : dispatch_ddt<DSPH_VISCO_ARTIFICIAL, false>(ctx, t, dvd, c, press);
        break;
      case DSPH_VISCO_LAMINAR:
        rc = vg ? dispatch_ddt<DSPH_VISCO_LAMINAR, true>(ctx, t, dvd, c, press)
                : dispatch_ddt<DSPH_VISCO_LAMINAR, false>(ctx, t, dvd, c, press);
        break;
      case DSPH_VISCO_LAMINARSPS:
        rc = vg ? dispatch_ddt<DSPH_VISCO_LAMINARSPS, true>(ctx, t, dvd, c, press)
                : dispatch_ddt<DSPH_VISCO_LAMINARSPS, false>(ctx, t, dvd, c, press);
        break;
      default: return set_error(ctx, DSPH_E_ARG, "dsph_interaction_forces: invalid tvisco");
    }
    if (rc) return rc;
    DSPH_LAUNCHED(ctx, "k_forces_fluid");
  }
  if (t->npbok) {
    KTimer kt(ctx, "k_forces_bound");
    if (ctx->forces_kernel == 0 && ctx->bound_kernel != 2) {
      // Teams beat one lane per particle at every size (us, dam breaks of 26k / 141k /
      // 6.1M particles 46 / 49 / 196 against 229 / 243 / 406, wave flume of 1.1M
      // 128 against 326).
      const unsigned g = grid_for(t->npbok, kTeamP);
      const TeamArrays A = team_arrays(t, press);
      if (t->d_ftomassp)
        k_forces_bound_team<true><<<g, 64, 0, ctx->stream>>>(t->npbok, dvd, c, A);
      else
        k_forces_bound_team<false><<<g, 64, 0, ctx->stream>>>(t->npbok, dvd, c, A);
    } else if (t->d_ftomassp)
      k_forces_bound<true><<<grid_for(t->npbok, kBsForces), kBsForces, 0, ctx->stream>>>(
          t->npbok, dvd, c, t->d_dcell, (const float4*)t->d_poscell,
          (const float4*)t->d_velrho, t->d_viscdt, t->d_ar, t->d_code, t->d_ftomassp);
    else
      k_forces_bound<false><<<grid_for(t->npbok, kBsForces), kBsForces, 0, ctx->stream>>>(
          t->npbok, dvd, c, t->d_dcell, (const float4*)t->d_poscell,
          (const float4*)t->d_velrho, t->d_viscdt, t->d_ar);
    DSPH_LAUNCHED(ctx, "k_forces_bound");
  }
  return DSPH_OK;
}

// Scratch of dsph_interaction_forces_noalloc: {press, 1/rho} (float2) for
// DSPH_NOALLOC_NP_MAX particles.
// Every GPU holds its own copy for the life of the process; host code uses
// the device address that hipGetSymbolAddress gives on each device, never
// the array's name.
constexpr size_t kNoallocBytes = size_t(DSPH_NOALLOC_NP_MAX) * sizeof(float2);
static __device__ __align__(256) unsigned char scratch[kNoallocBytes];

}  // namespace

namespace dsph {

// Device address of the no-alloc scratch on the current device (the
// context's device), looked up once per device.
int noalloc_scratch_init(dsph_ctx* ctx) {
  static std::mutex mu;
  static std::map<int, void*> addr;
  std::lock_guard<std::mutex> lock(mu);
  auto it = addr.find(ctx->device);
  if (it == addr.end()) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return set_error(ctx, DSPH_E_LAUNCH,
                       std::string("hipGetSymbolAddress(no-alloc scratch): ") +
                           hipGetErrorString(e));
    it = addr.emplace(ctx->device, ptr).first;
  }
  ctx->noalloc_scratch = it->second;
  return DSPH_OK;
}

}  // namespace dsph

extern "C" {

int dsph_interaction_forces(dsph_ctx* ctx, const dsph_inter_parms* t) {
  if (!ctx || !t) return DSPH_E_ARG;
  int rc = check_inter_parms(ctx, t);
  if (rc) return rc;
  if (t->np - t->npb) {
    rc = ensure_prep_scratch(ctx, t->np);
    if (rc) return rc;
  }
  return interaction_forces(ctx, t, reinterpret_cast<float2*>(ctx->prep_press));
}

int dsph_interaction_forces_noalloc(dsph_ctx* ctx, const dsph_inter_parms* t) {
  if (!ctx || !t) return DSPH_E_ARG;
  DSPH_REQUIRE(ctx, t->np <= DSPH_NOALLOC_NP_MAX,
               "dsph_interaction_forces_noalloc: np " + std::to_string(t->np) +
                   " > DSPH_NOALLOC_NP_MAX (" + std::to_string(DSPH_NOALLOC_NP_MAX) +
                   "); use dsph_interaction_forces");
  int rc = check_inter_parms(ctx, t);
  if (rc) return rc;
  if (!ctx->noalloc_scratch)
    return set_error(ctx, DSPH_E_STATE, "no-alloc scratch address not set up for this device");
  unsigned char* base = static_cast<unsigned char*>(ctx->noalloc_scratch);
  return interaction_forces(ctx, t, reinterpret_cast<float2*>(base));
}

}  // extern "C"
