// fdm_quad.h -- the batched F-16 step with each aircraft's substep spread over four cooperating
// wavefronts, so that at 16,384 engagements every SIMD holds two of them.
//
// One lane per aircraft; every 64 aircraft get four wavefronts ("roles") of one workgroup (two
// such groups, or one in a small batch):
//   kin   the integrator: pose and motion, frames, gravity, forces, moments, accelerations, and
//         the late (Mach) terms of the side, roll and yaw axes;
//   aero  mass properties, the rest of the aero build-up, and the history shift of a step of one
//         or two substeps;
//   fcs   the flight control system, the previous-frame auxiliary values, sin/cos of the Earth
//         angle and, after the last substep, most of the 17-value output;
//   air   atmosphere, engine, fuel.
// They trade values through LDS at three workgroup barriers per substep.  Attitude and position
// of a substep need only the rates and velocities of the one before, so the kin role forms the
// next pose while the others still work on the forces, and the atmosphere and the FCS channels
// of substep t run beside the late aero terms of substep t - 1:
//   before X2  kin: pose of t (frames, altitude, gravity);  fcs: sin/cos for t + 1
//   X2 -> X3   kin: lateral late terms, geometry, gyroscopic terms of t - 1;  aero: longitudinal
//              terms of t - 1;  fcs: channels of t that read the previous frame;  air: atmosphere
//   X3 -> X1   kin: accelerations of t - 1, motion of t;  aero: mass;  fcs: pitch loop;
//              air: spools
//   X1 -> X2   kin: quaternion rate, stores, (next pose);  aero: geometry, alpha-beta terms;
//              fcs: Mach, calibrated airspeed, load factors, ground speed;  air: engine
// (the loop below is rotated so that each piece appears once; iteration S only finishes the
// forces of the last substep).  Per substep at one wavefront per SIMD the four windows take
// 1.5, 1.05 and 0.55 us where the order propagate, atmosphere, aero, engine of the one-lane
// kernel took 1.6, 1.25 and 1.3: a lone wavefront issues one instruction every 4-5 clocks,
// VALU or not (fp64 included, no extra latency when dependent), so a window costs the longest
// role's instruction count and the split is chosen to make those equal.  Measured per step
// (tail-chase, HIP-graph replay), four roles in that order and in this one: 2,048 engagements
// 26.5 -> 24.0 us, 64 with the 17-value output 28.0 -> 24.3, 16,384 with it 35.9 -> 32.4 and
// without 32.4 -> 31.0 (there two wavefronts share each SIMD and issue during 75 % of its time),
// 65,536 115 -> 110; the single-precision build 16,384 26.0 -> 22.1, 64 23.8 -> 19.1.  The env step
// at 16,384 engagements 59.9 -> 52.9 us (of which the supersonic passes left to the last substep
// 3.4).
//
// Every value is formed by the component functions of fdm_device.h with the operands the
// one-lane kernel gives them, so all three kernels agree bit for bit.  An aero axis is summed
// in the generated order (the lateral early sums go from aero to kin), and a value that its
// writer forms again in the window its reader still reads it in is kept in two blocks by
// substep parity (sin/cos, surfaces, mass, local axes, gravity).
//
// The two groups of a workgroup map their roles to waves in opposite orders, so each SIMD
// (wave w and w + 4 of the workgroup) holds two roles that are busy in different phases: the
// SIMD pairs are (kin, fcs) and (air, aero).  Within a pair, kin and aero, which are on the
// substep's critical path, run at raised wave priority (s_setprio), so their instructions issue
// first whenever both waves have one ready: 31.4 -> 29.7 us per step at 16k engagements, with
// the pairs (kin, air) and (fcs, aero) 30.1.  Only with two groups per workgroup: with one, a
// SIMD holds one wave.
#pragma once
#include "fdm_image.h"
#include "fdm_split.h"

namespace f16 {
// A state value's store in the last substeps: a relaxed store at system scope, the same bytes as
// a plain store, written through the L2 as it is issued rather than left dirty there for the
// write-back that ends the kernel.  Each role stores a value in the phase of the last substep
// that makes it final (kin: position, velocity, rates, attitude, Earth angle and quaternion rate
// after X1, the accelerations at the end; fcs: PIDs, surface positions and auxiliary values
// before X2, alpha at the end; air: engine and fuel before X2), so most of the 27 MB of a 16k launch
// drains while the last substep still computes.  Per step (HIP-graph replay, tail-chase
// engagements, measured when it was introduced): 32.2 -> 31.7 us at 16k, 124 -> 117 us at 65,536,
// 25.9 -> 25.7 us at 4,096; the one-launch env step unchanged.  Plain stores at the same places gain
// about a third of that,
// streaming (non-temporal) ones two thirds.
// The pointer is named a global one.  Those that went through an empty asm are generic to the
// compiler, and a flat store counts as an LDS access too: every barrier and LDS read after the
// stores of the last substep waited for their write-through (fp64, six substeps of 64 / 16,384 /
// 65,536 engagements: 24.3 -> 23.9, 32.3 -> 31.6, 114.9 -> 112.0 us; fp32 at 64: 19.6 -> 19.1).
typedef __attribute__((address_space(1))) double GlobalDouble;
__device__ __forceinline__ void put(double* p, double v) {
  __hip_atomic_store((GlobalDouble*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr int kQuadGroups = 2;                   // 64-aircraft groups per workgroup
constexpr int kQuadBlock = 256 * kQuadGroups;    // threads per workgroup
constexpr int kQuadAircraft = 64 * kQuadGroups;  // aircraft per workgroup

enum QuadRole : int { kRoleKin = 0, kRoleAero = 1, kRoleFcs = 2, kRoleAir = 3 };

// role of wave w (0..3) of group g
__device__ __forceinline__ int quad_role(int g, int w) {
  // waves w and w + 4 share a SIMD: the SIMD pairs are (kin, fcs) and (air, aero)
  constexpr int kOrder[2][4] = {{kRoleKin, kRoleAir, kRoleAero, kRoleFcs},
                                {kRoleFcs, kRoleAero, kRoleAir, kRoleKin}};
  return kOrder[g][w];
}

// LDS exchange fields, [group][field][lane].
enum QuadField : int {
  // written before X2
  kQAlt, kQCtcp,                                         // kin (pose)
  kQCs,                                                  // fcs: cos, sin in the block of the
                                                         // substep's parity
  kQAlpha = kQCs + 4, kQBeta, kQE1, kQE3, kQE5,          // aero
  kQThrust, kQFuel,                                      // air
  // written before X3
  kQLef, kQFlap,                                         // fcs
  kQSurf,                                                // fcs: aileron, rudder, parity blocks
  kQAx0 = kQSurf + 4, kQAx1, kQAx2, kQAx3, kQAx4, kQAx5,              // aero (0, 2, 4), kin (1, 3, 5)
  // written before X1
  kQU, kQV, kQW, kQP, kQQ, kQR,                          // kin
  kQElev,                                                // fcs
  kQRho, kQSound, kQPres,                                // air
  kQMass, kQJ, kQJinv = kQJ + 6, kQRp = kQJinv + 6, kQCg = kQRp + 3,   // aero, parity block 0
  kQMassB = kQCg + 3,                                    // aero, parity block 1 (19 fields)
  // after the last substep: whether what each role stored is finite
  kQFinKin = kQMassB + (kQMassB - kQMass), kQFinFcs, kQFinAero,
  // the kin role's own slots: values it reads once per substep, kept out of registers across the
  // phases that do not use them
  kQPba, kQPpd = kQPba + 3, kQPpq = kQPpd + 3,           // previous accelerations and rates
  kQQuat = kQPpq + 3,                                    // this substep's quaternion
  kQLoc = kQQuat + 4,                                    // body axes' north and east components,
                                                         // parity blocks (read by fcs)
  kQGrav = kQLoc + 12,                                   // gravity, parity blocks
  kQPosOut = kQGrav + 6,                                 // the last substep's position, for the output
  kQuadFields = kQPosOut + 3
};
__device__ __forceinline__ int quad_mass_block(int t) { return (t & 1) ? kQMassB - kQMass : 0; }

// Wave priority N for the rest of this phase, when priorities are in use (two groups per
// workgroup: two waves per SIMD to arbitrate between).
template <int N, bool P>
__device__ __forceinline__ void quad_prio() {
  if constexpr (P) __builtin_amdgcn_s_setprio(N);
}

typedef double QuadX[kQuadFields][64];

// ---- kin: the integrator, and the late terms of the side, roll and yaw axes.  `fin`: report
// the finite flag of every state value it stores through x[kQFinKin] after one more barrier.
template <int FCS_RATE, bool PRIO, class Image>
__device__ __forceinline__ void quad_kin(const Image& image, double* __restrict__ s, long ld, int S, bool store,
                                         double* __restrict__ out_base, long obs_ld,
                                         const double* __restrict__ T, QuadX& x, int lane,
                                         bool fin) {
#define F(k) s[(long)(k) * ld]
  Aircraft a;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    a.p[j] = F(F16S_POS + j); a.v[j] = F(F16S_VEL + j); a.wi[j] = F(F16S_PQRI + j);
    a.ai[j] = F(F16S_UVWIDOT + j); a.wdi[j] = F(F16S_PQRIDOT + j);
    a.vh1[j] = F(F16S_DIVEL + j); a.vh2[j] = F(F16S_DIVEL + 3 + j); a.ah1[j] = F(F16S_DUVW + j);
    x[kQPba + j][lane] = F(F16S_PBA + j); x[kQPpd + j][lane] = F(F16S_PPQRIDOT + j);
    x[kQPpq + j][lane] = F(F16S_PPQRI + j);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) { a.q[j] = F(F16S_Q + j); a.qd[j] = F(F16S_QDOT + j); }
  a.epa = F(F16S_EPA);
  image.store();
  {   // the first substep's Earth angle (the later ones come from the fcs role)
    double ce, se;
    sincos(a.epa + kRot * kDt, &se, &ce);
    x[kQCs][lane] = ce;
    x[kQCs + 1][lane] = se;
  }
  const bool out = out_base != nullptr && store;   // its part of the 17-value output
  for (int t = 0;; ++t) {
    const int slot = S - 1 - t;
    // ---- pose of substep t: attitude, position, frames, gravity
    quad_prio<3, PRIO>();
#pragma unroll
    for (int j = 0; j < 4; ++j) x[kQQuat + j][lane] = a.q[j];     // substep t - 1's
    if (t < S) {
      propagate_pose(a);
      const double ce = x[kQCs + 2 * (t & 1)][lane], se = x[kQCs + 2 * (t & 1) + 1][lane];
      Kin k;
      double L[3][3], euler[3];
      kin_pose(a.p, a.q, ce, se, false, k, L, euler);
      const double alt = k.radius - kSemiMajor;
      x[kQAlt][lane] = alt; x[kQCtcp][lane] = k.ctcp;
      double gi[3];
      gravity(k, gi);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        x[kQLoc + 6 * (t & 1) + j][lane] = L[j][0]; x[kQLoc + 6 * (t & 1) + 3 + j][lane] = L[j][1];
        x[kQGrav + 3 * (t & 1) + j][lane] = gi[j];
      }
    }
    __syncthreads();
    // ---- X2 -> X3: late terms of the lateral axes and the force-free part of the accelerations
    // of substep t - 1
    quad_prio<2, PRIO>();
    double B[3][3];
    AccelPre pre;
    Mass mb;
    AuxGeo g;
    if (t > 0) {
      const int mo = quad_mass_block(t - 1);
      const double uvw[3] = {x[kQU][lane], x[kQV][lane], x[kQW][lane]};
      g = aux_geometry(uvw);
      {
        const double alpha = x[kQAlpha][lane], beta = x[kQBeta][lane];
        const int so = kQSurf + 2 * ((t - 1) & 1);
        const double ail = x[so][lane], rud = x[so + 1][lane];
        const double qbar = 0.5 * x[kQRho][lane] * g.vt2;
        const double mach = fm_div(g.vt, x[kQSound][lane]);
        F16_AERO_BRACKETS_MACH;
        F16_AERO_LOOKUPS_MACH;
        x[kQAx1][lane] = F16_AERO_SIDE_SCALE * (x[kQE1][lane] + F16_AERO_SIDE_LATE);
        x[kQAx3][lane] = F16_AERO_ROLL_SCALE * (x[kQE3][lane] + F16_AERO_ROLL_LATE);
        x[kQAx5][lane] = F16_AERO_YAW_SCALE * (x[kQE5][lane] + F16_AERO_YAW_LATE);
      }
      __builtin_amdgcn_sched_barrier(0);   // not interleaved with the above: registers
      {
        const double wpqr[3] = {x[kQP][lane], x[kQQ][lane], x[kQR][lane]};
        double q[4], J[6];
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = x[kQQuat + j][lane];
        body_dcm(q, B);
#pragma unroll
        for (int j = 0; j < 6; ++j) { J[j] = x[mo + kQJ + j][lane]; mb.Jinv[j] = x[mo + kQJinv + j][lane]; }
        accel_pre(B, wpqr, J, x[mo + kQMass][lane], pre);
      }
    }
    __syncthreads();
    // ---- X3 -> X1: forces, moments and accelerations of substep t - 1, motion of substep t
    quad_prio<3, PRIO>();
    if (t > 0) {
      const int mo = quad_mass_block(t - 1), go = kQGrav + 3 * ((t - 1) & 1);
      const double ax[6] = {x[kQAx0][lane], x[kQAx1][lane], x[kQAx2][lane], x[kQAx3][lane],
                            x[kQAx4][lane], x[kQAx5][lane]};
      const double thrust = x[kQThrust][lane];
      const double gi[3] = {x[go][lane], x[go + 1][lane], x[go + 2][lane]};
#pragma unroll
      for (int j = 0; j < 3; ++j) { mb.rp[j] = x[mo + kQRp + j][lane]; mb.cg[j] = x[mo + kQCg + j][lane]; }
      double Fb[3], Mb[3];
      forces_moments(ax, g, mb, thrust, Fb, Mb);
      Accel ac;
      accel_post(B, pre, mb.Jinv, Fb, Mb, gi, ac);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        a.ai[i] = ac.ai[i]; a.wdi[i] = ac.wdi[i];
        x[kQPba + i][lane] = ac.pba[i]; x[kQPpd + i][lane] = ac.wdi[i]; x[kQPpq + i][lane] = ac.ppq[i];
      }
    }
    if (t >= S) break;
    propagate_motion(a);   // leaves the values the histories take: v in vh1, a in ah1
    {
    double uvw[3], wpqr[3], Bt[3][3];
    body_dcm(a.q, Bt);
    body_motion(Bt, a.p, a.v, a.wi, uvw, wpqr);
    x[kQU][lane] = uvw[0]; x[kQV][lane] = uvw[1]; x[kQW][lane] = uvw[2];
    x[kQP][lane] = wpqr[0]; x[kQQ][lane] = wpqr[1]; x[kQR][lane] = wpqr[2];
    }
    __syncthreads();
    // ---- X1 -> X2: quaternion rate, the state's stores, and the next pose
    quad_prio<3, PRIO>();
    if (store && slot <= 2) {       // values pushed onto the histories at the start of this substep
      double* h = s;                // the history addresses are formed here (see the stores
      asm volatile("" : "+v"(h));   // after the loop)
#define H(k) h[(long)(k) * ld]
#pragma unroll
      for (int j = 0; j < 4; ++j) put(&H(F16S_DQ + 4 * slot + j), a.qd[j]);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        put(&H(F16S_DPQRI + 3 * slot + j), a.wdi[j]);
        put(&H(F16S_DIVEL + 3 * slot + j), a.vh1[j]);
        put(&H(F16S_DUVW + 3 * slot + j), a.ah1[j]);
      }
#undef H
    }
    quat_rate(a);
    if (slot == 0 && out) {
      // the output's addresses are formed here from a pointer the compiler cannot see through,
      // not hoisted above the loop
      GlobalDouble* o = (GlobalDouble*)out_base;
      asm volatile("" : "+v"(o));
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        o[(long)j * obs_ld] = a.p[j];
        o[(long)(3 + j) * obs_ld] = a.v[j];
        x[kQPosOut + j][lane] = a.p[j];   // for the fcs role's part of the output
      }
    }
    if (store && slot == 0) {
      double* h = s;
      asm volatile("" : "+v"(h));
#define H(k) h[(long)(k) * ld]
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        put(&H(F16S_POS + j), a.p[j]); put(&H(F16S_VEL + j), a.v[j]); put(&H(F16S_PQRI + j), a.wi[j]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) { put(&H(F16S_Q + j), a.q[j]); put(&H(F16S_QDOT + j), a.qd[j]); }
      put(&H(F16S_EPA), a.epa);
#undef H
    }
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    a.pba[j] = x[kQPba + j][lane]; a.ppd[j] = x[kQPpd + j][lane]; a.ppq[j] = x[kQPpq + j][lane];
  }
  quad_prio<0, PRIO>();
  // the state's addresses are formed here, from a pointer the compiler cannot see through:
  // hoisted above the substep loop they would stay live across it, 2 registers each
  asm volatile("" : "+v"(s));
  if (store && S > 0) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      put(&F(F16S_UVWIDOT + j), a.ai[j]); put(&F(F16S_PQRIDOT + j), a.wdi[j]);
      put(&F(F16S_PBA + j), a.pba[j]); put(&F(F16S_PPQRIDOT + j), a.ppd[j]);
      put(&F(F16S_PPQRI + j), a.ppq[j]);
    }
  }
#undef F
  if (fin) {
    unsigned m = fin_acc(0u, a.epa);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      m = fin_acc(fin_acc(fin_acc(fin_acc(m, a.p[j]), a.v[j]), a.wi[j]), a.ai[j]);
      m = fin_acc(fin_acc(fin_acc(fin_acc(m, a.wdi[j]), a.pba[j]), a.ppd[j]), a.ppq[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) m = fin_acc(fin_acc(m, a.q[j]), a.qd[j]);
    x[kQFinKin][lane] = m < kFinInf ? 1.0 : 0.0;
    __syncthreads();
  }
}

// ---- aero: mass properties, and the six axes of the aero build-up but the lateral axes' late
// terms.  Holds no state, and in a step of one or two substeps shifts the history entries that
// outlive it: all loaded at once while the other roles load their states, where the kin role
// shifted them one entry after the other before its first pose (one substep of 64 / 16,384 /
// 65,536 engagements: 12.05 / 15.9 / 59.2 -> 9.5 / 13.2 / 46.4 us; two: 14.0 / 18.5 / 64.7 ->
// 12.2 / 16.6 / 58.0).
template <int FCS_RATE, bool PRIO, class Image>
__device__ __forceinline__ void quad_aero(const Image& image, double* __restrict__ s, long ld,
                                          int S, bool store, const double* __restrict__ T,
                                          QuadX& x, int lane, bool fin) {
  double vt = 0.0, vt2 = 0.0, alpha = 0.0, q = 0.0, lef = 0.0, flap = 0.0;
  unsigned hist_m = 0u;   // as split_flight: only the entries shifted when S < 3 need a test
  if (store && S > 0 && S < 3) {
#define F(k) s[(long)(k) * ld]
    double e[2][13];      // entries 0 and (S = 1) 1, which become S and 2
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (k > 0 && S == 2) break;
#pragma unroll
      for (int j = 0; j < 4; ++j) e[k][j] = F(F16S_DQ + 4 * k + j);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        e[k][4 + j] = F(F16S_DPQRI + 3 * k + j);
        e[k][7 + j] = F(F16S_DIVEL + 3 * k + j);
        e[k][10 + j] = F(F16S_DUVW + 3 * k + j);
      }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (k > 0 && S == 2) break;
      const int to = k + S;
#pragma unroll
      for (int j = 0; j < 13; ++j) hist_m = fin_acc(hist_m, e[k][j]);
#pragma unroll
      for (int j = 0; j < 4; ++j) F(F16S_DQ + 4 * to + j) = e[k][j];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        F(F16S_DPQRI + 3 * to + j) = e[k][4 + j];
        F(F16S_DIVEL + 3 * to + j) = e[k][7 + j];
        F(F16S_DUVW + 3 * to + j) = e[k][10 + j];
      }
    }
#undef F
  }
  image.store();
  for (int t = 0;; ++t) {
    __syncthreads();
    // ---- X2 -> X3: the Mach and elevator terms of substep t - 1
    quad_prio<2, PRIO>();
    if (t > 0) {
      const double rho = x[kQRho][lane], sound = x[kQSound][lane], elev = x[kQElev][lane];
      const double qbar = 0.5 * rho * vt2;
      const double mach = fm_div(vt, sound);
      constexpr double kclge = kCLge;
      constexpr double gear = kGearPos<FCS_RATE>;
      constexpr double beta = 0.0;                  // (no longitudinal term reads it)
      double bi2vel, ci2vel;
      aero_rates(vt, bi2vel, ci2vel);
      F16_AERO_BRACKETS_AB;
      F16_AERO_LOOKUPS_AB;
      F16_AERO_BRACKETS_MACH;
      F16_AERO_BRACKETS_ELEV;
      F16_AERO_LOOKUPS_MACH;
      F16_AERO_LOOKUPS_ELEV;
      const double e0 = F16_AERO_DRAG_EARLY, e2 = F16_AERO_LIFT_EARLY, e4 = F16_AERO_PITCH_EARLY;
      x[kQAx0][lane] = F16_AERO_DRAG_SCALE * (e0 + F16_AERO_DRAG_LATE);
      x[kQAx2][lane] = F16_AERO_LIFT_SCALE * (e2 + F16_AERO_LIFT_LATE);
      x[kQAx4][lane] = F16_AERO_PITCH_SCALE * (e4 + F16_AERO_PITCH_LATE);
    }
    __syncthreads();
    if (t >= S) break;
    // ---- X3 -> X1: mass, CG, inertia
    quad_prio<3, PRIO>();
    {
      const int mo = quad_mass_block(t);
      const Mass mb = mass_props(x[kQFuel][lane]);
      x[mo + kQMass][lane] = mb.mass;
#pragma unroll
      for (int j = 0; j < 6; ++j) { x[mo + kQJ + j][lane] = mb.J[j]; x[mo + kQJinv + j][lane] = mb.Jinv[j]; }
#pragma unroll
      for (int j = 0; j < 3; ++j) { x[mo + kQRp + j][lane] = mb.rp[j]; x[mo + kQCg + j][lane] = mb.cg[j]; }
    }
    __syncthreads();
    // ---- X1 -> X2: geometry and the alpha-beta terms
    quad_prio<3, PRIO>();
    {
      const double uvw[3] = {x[kQU][lane], x[kQV][lane], x[kQW][lane]};
      const AuxGeo g = aux_geometry(uvw);
      alpha = g.alpha; vt = g.vt; vt2 = g.vt2;
      const double beta = g.beta;
      x[kQAlpha][lane] = alpha; x[kQBeta][lane] = beta;
      const double ail = x[kQSurf + 2 * (t & 1)][lane], rud = x[kQSurf + 2 * (t & 1) + 1][lane];
      lef = x[kQLef][lane]; flap = x[kQFlap][lane];
      double bi2vel, ci2vel;
      aero_rates(vt, bi2vel, ci2vel);
      const double p = x[kQP][lane], r = x[kQR][lane];
      q = x[kQQ][lane];
      F16_AERO_BRACKETS_AB;
      F16_AERO_LOOKUPS_AB;
      x[kQE1][lane] = F16_AERO_SIDE_EARLY;
      x[kQE3][lane] = F16_AERO_ROLL_EARLY;
      x[kQE5][lane] = F16_AERO_YAW_EARLY;
    }
  }
  quad_prio<0, PRIO>();
  if (fin) {
    x[kQFinAero][lane] = hist_m < kFinInf ? 1.0 : 0.0;
    __syncthreads();
  }
}

// ---- fcs: the FCS channels, the previous-frame auxiliary values, and sin/cos of the Earth angle.
template <int FCS_RATE, bool PRIO, class Image>
__device__ __forceinline__ void quad_fcs(const Image& image, double* __restrict__ s, long ld,
                                         const double* __restrict__ act4, int S, bool store,
                                         const double* __restrict__ T, QuadX& x, int lane,
                                         bool fin, double* __restrict__ keep,
                                         double* __restrict__ out_base = nullptr,
                                         long obs_ld = 0) {
#define F(k) s[(long)(k) * ld]
  Aircraft a;
#pragma unroll
  for (int j = 0; j < 3; ++j) { a.pid_ip[j] = F(F16S_PID + 3 * j); a.pid_io[j] = F(F16S_PID + 3 * j + 2); }
#pragma unroll
  for (int j = 0; j < 9; ++j) a.pa[j] = F(F16S_PAUX + j);
  a.k_tef = F(F16S_KIN); a.k_ail = F(F16S_KIN + 1); a.k_ele = F(F16S_KIN + 2); a.k_lef = F(F16S_KIN + 5);
  a.epa = F(F16S_EPA);   // tracked with the kin role's increments; never stored here
  a.epa += kRot * kDt;
  const double c_ail = act4[0], c_ele = act4[1], c_rud = act4[2];
  image.store();
  if (keep && store) { keep[0] = c_ail; keep[1] = c_ele; keep[2] = c_rud; keep[3] = act4[3]; }
  double k_rud = 0.0;
  unsigned ip2_m = 0u;
  for (int t = 0;; ++t) {
    // ---- before X2: sin/cos of the next substep's Earth angle
    quad_prio<0, PRIO>();
    if (t + 1 < S) {
      a.epa += kRot * kDt;
      double sn, cn;
      sincos(a.epa, &sn, &cn);
      x[kQCs + 2 * ((t + 1) & 1)][lane] = cn;
      x[kQCs + 2 * ((t + 1) & 1) + 1][lane] = sn;
    }
    __syncthreads();
    // ---- X2 -> X3: the rest of substep t - 1's auxiliary values, then substep t's channels that
    // read only those
    quad_prio<1, PRIO>();
    if (t > 0) a.pa[0] = x[kQAlpha][lane];
    FcsOut fc;
    double esch = 0.0;
    if (t < S) {
      if (store && t + 1 == S) {   // PID input_prev2 = input_prev before the final update
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          F(F16S_PID + 3 * j + 1) = a.pid_ip[j];
          ip2_m = fin_acc(ip2_m, a.pid_ip[j]);
        }
      }
      esch = fcs_prev_frame<FCS_RATE>(a, c_ail, c_ele, c_rud, T, fc);
      k_rud = fc.k_rud;
      x[kQSurf + 2 * (t & 1)][lane] = fc.ail; x[kQSurf + 2 * (t & 1) + 1][lane] = fc.rud;
      x[kQLef][lane] = fc.lef; x[kQFlap][lane] = fc.flap;
    }
    __syncthreads();
    if (t >= S) break;
    // ---- X3 -> X1: the pitch loop
    quad_prio<0, PRIO>();
    fcs_pitch<FCS_RATE>(a, esch, x[kQCtcp][lane], fc);
    x[kQElev][lane] = fc.elev;
    __syncthreads();
    // ---- X1 -> X2: Mach number, calibrated airspeed, body rates
    quad_prio<0, PRIO>();
    if (store && t + 1 == S) {
      double* h = s;
      asm volatile("" : "+v"(h));
#define H(k) h[(long)(k) * ld]
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        put(&H(F16S_PID + 3 * j), a.pid_ip[j]); put(&H(F16S_PID + 3 * j + 2), a.pid_io[j]);
      }
      put(&H(F16S_KIN), a.k_tef); put(&H(F16S_KIN + 1), a.k_ail); put(&H(F16S_KIN + 2), a.k_ele);
      put(&H(F16S_KIN + 3), k_rud); put(&H(F16S_KIN + 4), kGearPos<FCS_RATE>);
      put(&H(F16S_KIN + 5), a.k_lef);
#undef H
    }
    {
      const double u = x[kQU][lane], v = x[kQV][lane], w = x[kQW][lane];
      const double vt = fm_sqrt((u * u + w * w) + v * v);   // aux_geometry's
      const double mach = fm_div(vt, x[kQSound][lane]);
      a.pa[1] = mach;
      // between substeps the channels only test the airspeed against 250 kt and less, so the ten
      // supersonic passes (every wavefront with one supersonic aircraft makes them) are left to
      // the last substep, whose value is stored
      a.pa[2] = vc_knots(mach, x[kQPres][lane], t + 1 == S);
      a.pa[6] = x[kQP][lane]; a.pa[7] = x[kQQ][lane]; a.pa[8] = x[kQR][lane];
      const int mo = quad_mass_block(t);
      const double cg[3] = {x[mo + kQCg][lane], x[mo + kQCg + 1][lane], x[mo + kQCg + 2][lane]};
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        a.pba[j] = x[kQPba + j][lane]; a.ppd[j] = x[kQPpd + j][lane]; a.ppq[j] = x[kQPpq + j][lane];
      }
      load_factors(a, cg, a.pa[4], a.pa[5]);
      const int lo = kQLoc + 6 * (t & 1);
      const double vn = x[lo][lane] * u + x[lo + 1][lane] * v + x[lo + 2][lane] * w;
      const double ve = x[lo + 3][lane] * u + x[lo + 4][lane] * v + x[lo + 5][lane] * w;
      a.pa[3] = fm_sqrt(vn * vn + ve * ve);
    }
    if (store && t + 1 == S) {   // all but alpha, which the aero role forms in this window
      double* h = s;
      asm volatile("" : "+v"(h));
#pragma unroll
      for (int j = 1; j < 9; ++j) put(&h[(long)(F16S_PAUX + j) * ld], a.pa[j]);
    }
  }
  quad_prio<0, PRIO>();
  asm volatile("" : "+v"(s));   // as in quad_kin: the store addresses are formed here
  if (store && S > 0) put(&F(F16S_PAUX), a.pa[0]);
#undef F
  if (out_base != nullptr && store && S > 0) {
    // the output but position and velocity, formed here while the kin and aero roles finish the
    // last substep: the Euler angles' inverse trigonometry stays out of the loop
    double p[3], q[4], euler[3], L[3][3];
#pragma unroll
    for (int j = 0; j < 3; ++j) p[j] = x[kQPosOut + j][lane];
#pragma unroll
    for (int j = 0; j < 4; ++j) q[j] = x[kQQuat + j][lane];
    const int cs = kQCs + 2 * ((S - 1) & 1);
    Kin k;
    kin_pose(p, q, x[cs][lane], x[cs + 1][lane], true, k, L, euler);
    const double u = x[kQU][lane], v = x[kQV][lane], w = x[kQW][lane];
    GlobalDouble* o = (GlobalDouble*)out_base;
    asm volatile("" : "+v"(o));
#pragma unroll
    for (int j = 0; j < 3; ++j) o[(long)(6 + j) * obs_ld] = euler[j];
    o[9L * obs_ld] = u; o[10L * obs_ld] = v; o[11L * obs_ld] = w;
    o[12L * obs_ld] = x[kQAlpha][lane]; o[13L * obs_ld] = x[kQBeta][lane];
    o[14L * obs_ld] = a.pa[1];
    o[15L * obs_ld] = fm_sqrt((u * u + w * w) + v * v);
    o[16L * obs_ld] = k.radius - kSemiMajor;
  }
  if (fin) {
    unsigned m = fin_acc(fin_acc(fin_acc(ip2_m, a.k_tef), a.k_ail), a.k_ele);
    m = fin_acc(fin_acc(m, k_rud), a.k_lef);
#pragma unroll
    for (int j = 0; j < 3; ++j) m = fin_acc(fin_acc(m, a.pid_ip[j]), a.pid_io[j]);
#pragma unroll
    for (int j = 0; j < 9; ++j) m = fin_acc(m, a.pa[j]);
    x[kQFinFcs][lane] = m < kFinInf ? 1.0 : 0.0;
    __syncthreads();
  }
}

// ---- air: atmosphere, engine and fuel.  With `fin` non-null, fin[0] <- 1 if all 101 state
// values are finite (its own, and the other roles' flags after the last barrier).
template <int FCS_RATE, bool PRIO, class Image>
__device__ __forceinline__ void quad_air(const Image& image, double* __restrict__ s, long ld,
                                         const double* __restrict__ act4, int S, bool store,
                                         const double* __restrict__ T, QuadX& x, int lane,
                                         unsigned char* __restrict__ fin) {
#define F(k) s[(long)(k) * ld]
  Aircraft a;
  a.fuel = F(F16S_FUEL);
  a.n1 = F(F16S_ENG); a.n2 = F(F16S_ENG + 1); a.n2n = F(F16S_ENG + 2); a.ff = F(F16S_ENG + 3);
  const double c_thr = act4[3];
  image.store();
  for (int t = 0;; ++t) {
    x[kQFuel][lane] = a.fuel;
    __syncthreads();
    // ---- X2 -> X3: the atmosphere of substep t
    quad_prio<1, PRIO>();
    Atmos at;
    if (t < S) at = isa(x[kQAlt][lane], T);
    __syncthreads();
    if (t >= S) break;
    // ---- X3 -> X1: the spools
    quad_prio<0, PRIO>();
    x[kQRho][lane] = at.rho; x[kQSound][lane] = at.a; x[kQPres][lane] = at.P;
    const double aug = engine_spool(a, c_thr, at);
    __syncthreads();
    // ---- X1 -> X2: Mach number, thrust, fuel flow
    quad_prio<0, PRIO>();
    {
      const double u = x[kQU][lane], v = x[kQV][lane], w = x[kQW][lane];
      const double vt = fm_sqrt((u * u + w * w) + v * v);   // aux_geometry's
      const double mach = fm_div(vt, at.a);
      double burn;
      x[kQThrust][lane] = engine_thrust(a, aug, at, mach, T, burn);
      a.fuel -= burn;
    }
    if (store && t + 1 == S) {
      double* h = s;
      asm volatile("" : "+v"(h));
#define H(k) h[(long)(k) * ld]
      put(&H(F16S_ENG), a.n1); put(&H(F16S_ENG + 1), a.n2); put(&H(F16S_ENG + 2), a.n2n);
      put(&H(F16S_ENG + 3), a.ff); put(&H(F16S_FUEL), a.fuel);
#undef H
    }
  }
  quad_prio<0, PRIO>();
#undef F
  if (fin) {
    unsigned m = fin_acc(fin_acc(fin_acc(fin_acc(0u, a.fuel), a.n1), a.n2), a.n2n);
    m = fin_acc(m, a.ff);
    __syncthreads();
    if (store)
      fin[0] = (m < kFinInf && x[kQFinKin][lane] != 0.0 && x[kQFinFcs][lane] != 0.0 &&
                x[kQFinAero][lane] != 0.0) ? 1 : 0;
  }
}

// ------------------------------------------------------------------ the kernel
// The four-role form: each 64 aircraft on four wavefronts, G groups per
// workgroup of 256 G threads.  G = 2: 16,384 engagements put two wavefronts on every SIMD (at
// most 256 registers each) where the two-wave kernel has one, the two groups' roles paired on
// each SIMD by quad_role.  G = 1: a batch too small to give every CU a two-group workgroup
// spreads over twice as many CUs, one wavefront per SIMD (the two group orders alternate
// between workgroups).  The same results bit for bit.  OBS: the 17-value output is written
// (its own instantiation: 207 registers with it, 191 without).
template <int FCS_RATE, bool OBS, int G>
__global__ __launch_bounds__(256 * G) void fdm_step_quad_kernel(
    double* __restrict__ st, long ld, const double* __restrict__ act, int nac, int S,
    double* __restrict__ obs, long obs_ld, unsigned char* __restrict__ fin,
    double* __restrict__ act_keep) {
  static_assert(G == 1 || G == kQuadGroups, "one or two 64-aircraft groups per workgroup");
  __shared__ double T[F16M_IMAGE_LEN];
  __shared__ QuadX X[G];
  ImageCopy<256 * G> image;   // stored by the roles once their state loads are issued
  image.load(T);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wave >> 2;
  const int role = quad_role(G == 1 ? (int)(blockIdx.x & 1) : grp, wave & 3);
  const int i = blockIdx.x * (64 * G) + grp * 64 + lane;
  const bool store = i < nac;
  const int ia = store ? i : nac - 1;   // lanes past the batch shadow the last aircraft
  constexpr bool kPrio = G == kQuadGroups;   // two waves per SIMD to arbitrate between
  if (role == kRoleKin)
    quad_kin<FCS_RATE, kPrio>(image, st + ia, ld, S, store, OBS ? obs + ia : nullptr, obs_ld, T, X[grp],
                              lane, fin != nullptr);
  else if (role == kRoleAero)
    quad_aero<FCS_RATE, kPrio>(image, st + ia, ld, S, store, T, X[grp], lane, fin != nullptr);
  else if (role == kRoleFcs)
    quad_fcs<FCS_RATE, kPrio>(image, st + ia, ld, act + 4L * ia, S, store, T, X[grp], lane,
                              fin != nullptr, act_keep ? act_keep + 4L * ia : nullptr,
                              OBS ? obs + ia : nullptr, obs_ld);
  else
    quad_air<FCS_RATE, kPrio>(image, st + ia, ld, act + 4L * ia, S, store, T, X[grp], lane,
                              fin ? fin + ia : nullptr);
}

}  // namespace f16
