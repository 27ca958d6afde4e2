// The MD step (the path g6_step runs), one kernel per step for systems of up
// to a few thousand molecules (k_md_step) and two beyond:
//
//   k_md_pre   64 molecules per block, one Gear role per wave, state held
//              in registers: rigid_correct with the forces of the previous
//              k_md_main, kinetic and kinetic-tensor partials, rigid_predict,
//              rigid_setmatrix, the per-molecule record read by k_md_main
//              (predicted COM in FP64, site offsets in the pair precision),
//              Address_Assign binning into fixed-capacity cell lists of this
//              step's parity, and the Verlet-skin test that decides whether
//              rows are rebuilt.
//   close      one block: Nose_Correct / Nose_Predict from the kinetic
//              energies, and the cell lists of the other parity cleared
//              (block 0 of k_md_main); after the last step of a call, and
//              every step of the barostat, also the block partials reduced in
//              a fixed order into the thermo record (energies, temperature,
//              pressure, conserved H; k_md_close).  Pair partials alternate
//              between two parities.
//   k_md_main  one wavefront per molecule i:
//              (1) if a rebuild is due, i's own neighbour row: every j != i
//                  (small systems), or every j != i of the cells whose box
//                  lies within rc + skin of i (a 5^3 stencil of cells of edge
//                  >= (rc+skin)/2), that passes the reference's FP64
//                  minimum-image test dd < (rc+skin)^2, sorted by j;
//              (2) the pair forces of i with every listed j whose FP64 COM
//                  distance passes dd < rc^2 - the reference's
//                  Interaction_Compress2 test, so the interacting set is the
//                  reference's - via pair_sites (g6_pair.h);
//              (3) wave reduction of i's force and lab torque (the work of
//                  rigid_collectforce), stored for the corrector;
//              (4) block partials of energy and virial.
//   k_md_step  k_md_main's work and, for the block's four molecules, the
//              corrector and the next step's k_md_pre.
// A step is k_md_step, or k_md_pre(correct previous, predict) + k_md_main;
// block 0 of the pair kernel first does the close work of the previous step
// (k_md_close runs on its own only around the first and last step of a run).
// A run of steps ends with the correctors and k_md_close, so every g6_step
// call leaves the state of the reference's loop end (after Nose_Correct,
// Mixture.F90:2282).  Cell lists, rebuild flags and partials alternate so that
// no kernel needs a grid-wide barrier; both forms give the same bits.
// Each unordered pair is evaluated in both rows, so no molecule's force
// needs an atomic, rows are sorted and every reduction runs in a fixed
// order: results are deterministic.  Energies and the virial are halved.
#include <type_traits>

#include "g6_md_common.h"

// Everything written in this file is FP64 bookkeeping in the reference's
// operation order: no FMA contraction (the pragma is set by g6_md_common.h).
// The FP32 pair arithmetic lives in g6_pair.h, outside the pragma, and may
// contract.

namespace g6 {

__device__ inline float fma_r(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ inline double fma_r(double a, double b, double c) { return __builtin_fma(a, b, c); }

// force (C0 = 0) or lab torque (C0 = 3) of molecule i from the tile
// kernel's partials, summed in a fixed order (as k_part_reduce)
template <int C0>
__device__ inline void part_sum(const MdBuf &b, int i, double (&f)[3]) {
  const float *p = b.part + (size_t)i * b.nds * 6 + C0;
  for (int q = 0; q < b.nds; q++)
#pragma unroll
    for (int a = 0; a < 3; a++) f[a] += (double)p[q * 6 + a];
}

// value of lane l of the quad
template <int L>
__device__ inline double quad_d(double v) {
  return dpp_d<L * 0x55>(v);
}
// sum over the quad in a fixed order, in every lane
__device__ inline double quad_sum_d(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  return v;
}

// kinetic energy of four molecules from their sums of |dx(1)|^2 and w^2
__device__ inline double kin_energy(const ModelTable &mt, double dt, double et, double ex,
                                    double ey, double ez) {
  return et * mt.mass * 0.5 * (1.0 / (dt * dt)) +
         (ex * mt.Ixx + ey * mt.Iyy + ez * mt.Izz) * 0.5;
}

// ---- kernel A --------------------------------------------------------------
// A block updates 64 molecules (one per lane) with one role per wave:
//   wave 0  translation: com, dx[5][3]; record COM, binning, skin test
//   wave 1  angular velocity w[5][3]
//   wave 2  quaternion components a, b of every derivative; wave 3 c, d
// Every component is computed with the operation order of rigid_correct
// (RigidModule.F90:1255-1487, with the Nose drag) and rigid_predict
// (RigidModule.F90:480-559); values cross waves only through LDS, so the
// split changes no bit of the result.  The roles are wave-uniform, so no
// wave executes another role's code.
// blk is the block's index within its system (blockIdx.x for one system).
template <int BOX>
__device__ __forceinline__ void md_pre_body(const ModelTable &mt, const Geom &g, const MdBuf &b,
                                            double dt, int nose_active, int do_correct,
                                            int do_predict, int do_sites, int list, int half,
                                            int blk) {
  constexpr bool NPT = BOX == kBoxBaro;
  __shared__ double s_w0[3][64], s_W[12][64];
  __shared__ double s_q0[4][64], s_p[4][64], s_r[4][64], s_s[4][64], s_qn[4][64];
  __shared__ double s_ew[3][16];
  const int n = g.n;
  const int role = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int i = blk * 64 + lane;
  const bool ok = i < n;
  const bool q2 = role == 2;  // wave 2: components a, b; wave 3: c, d
  // the group of four molecules of lanes 4 l .. 4 l + 3
  const int grp = blk * 16 + (lane >> 2);
  const bool grp_ok = (lane & 3) == 0 && grp * 4 < n;
  // the block's kinetic partials
  const int nb64 = (n + 63) / 64;
  double *ek = b.stepek + blk;
  double et = 0.0;
  double S[20];  // wave 0: com, dx; wave 1: w; waves 2-3: q (all four)
#pragma unroll
  for (int k = 0; k < 20; k++) S[k] = 0.0;
  const double zeta0 = nose_active ? b.nose[3] : 0.0;
  // translational drag: Nose, plus the Andersen dilation
  // (RigidModule.F90:1275-1305): v1 / (2*3*v0) on every axis in the
  // orthorhombic mode, v1 / (2*v0) on z alone in the orz mode
  const bool orz = NPT && b.box[16] == 2.0;
  const double acoeff = !NPT ? 0.0
                        : orz ? b.anders[3] / (2.0 * b.anders[2])
                              : b.anders[3] / (2.0 * 3.0 * b.anders[2]);
  const double nc = zeta0 * dt, exr = nc;
  const double ext[3] = {nc * 0.5 + (orz ? 0.0 : acoeff), nc * 0.5 + (orz ? 0.0 : acoeff),
                         nc * 0.5 + acoeff};
  const BoxNow bx = box_now<BOX>(g, b);
  // every global load is issued here, ahead of the first barrier
  double F[3] = {0, 0, 0}, t[9], tl[3] = {0, 0, 0}, cref[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < 9; a++) t[a] = 0.0;
  if (ok) {
    if (role == 0) {
#pragma unroll
      for (int a = 0; a < 3; a++) S[a] = b.com[a * n + i];
#pragma unroll
      for (int k = 0; k < 15; k++) S[3 + k] = b.dx[k * n + i];
      if (do_correct) {
        if (b.part) part_sum<0>(b, i, F);
        else
#pragma unroll
          for (int a = 0; a < 3; a++) F[a] = b.frc[a * n + i];
      }
      if (do_sites && b.half_skin2 > 0.0)
#pragma unroll
        for (int a = 0; a < 3; a++) cref[a] = b.com_ref[a * n + i];
    } else if (role == 1) {
#pragma unroll
      for (int k = 0; k < 15; k++) S[k] = b.w[k * n + i];
      if (do_correct) {
#pragma unroll
        for (int a = 0; a < 9; a++) t[a] = b.tmat[a * n + i];
        if (b.part) part_sum<3>(b, i, tl);
        else
#pragma unroll
          for (int a = 0; a < 3; a++) tl[a] = b.frc[(3 + a) * n + i];
      }
    } else {
#pragma unroll
      for (int k = 0; k < 20; k++) S[k] = b.quat[k * n + i];
    }
  }
  // ---- corrector ----
  if (do_correct) {
    if (role == 1) {
#pragma unroll
      for (int a = 0; a < 3; a++) s_w0[a][lane] = S[a];  // the old w, for nw
    }
    __syncthreads();
    if (role == 0) {
      if (ok) {
        const double tf = dt * dt * 0.5 * mt.inv_mass;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          double nf = F[a] * tf;
          nf = nf - S[3 + a] * ext[a];
          const double d = nf - S[6 + a];
          S[a] = S[a] + kG5_0 * d;
          S[3 + a] = S[3 + a] + kG5_1 * d;
          S[6 + a] = nf;
          S[9 + a] = S[9 + a] + kG5_3 * d;
          S[12 + a] = S[12 + a] + kG5_4 * d;
          S[15 + a] = S[15 + a] + kG5_5 * d;
        }
      }
      // Rigid_Ek and Rigid_PressureTensor sums (RigidModule.F90:576-619),
      // upper triangle
      const double v[3] = {ok ? S[3] : 0.0, ok ? S[4] : 0.0, ok ? S[5] : 0.0};
      const double vv = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
      et = quad_sum_d(vv);
      const double u[8] = {vv,          v[0] * v[0], v[0] * v[1], v[0] * v[2],
                           v[1] * v[1], v[1] * v[2], v[2] * v[2], 0.0};
      double e0, e1;
      wsum_eight(u, lane, e0, e1);
      if (lane >> 2 == 1) {  // columns 0 and 4..6, then 7..9
        const int c = lane & 3;
        ek[(size_t)(c == 0 ? 0 : 3 + c) * nb64] = e0;
        if (c < 3) ek[(size_t)(7 + c) * nb64] = e1;
      }
    } else if (role == 1) {
      if (ok) {
        // rigid_collectforce's body-frame torque (RigidModule.F90:301-306)
        const double tq0 = t[0] * tl[0] + t[3] * tl[1] + t[6] * tl[2];
        const double tq1 = t[1] * tl[0] + t[4] * tl[1] + t[7] * tl[2];
        const double tq2 = t[2] * tl[0] + t[5] * tl[1] + t[8] * tl[2];
        const double wx = S[0], wy = S[1], wz = S[2];
        double nf[3];
        nf[0] = (tq0 + (mt.Iyy - mt.Izz) * wy * wz) * dt * mt.inv_ixx;
        nf[1] = (tq1 + (mt.Izz - mt.Ixx) * wz * wx) * dt * mt.inv_iyy;
        nf[2] = (tq2 + (mt.Ixx - mt.Iyy) * wx * wy) * dt * mt.inv_izz;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          nf[a] = nf[a] - S[a] * exr;
          const double d = nf[a] - S[3 + a];
          S[a] = S[a] + kG4_0 * d;
          S[3 + a] = nf[a];
          S[6 + a] = S[6 + a] + kG4_2 * d;
          S[9 + a] = S[9 + a] + kG4_3 * d;
          S[12 + a] = S[12 + a] + kG4_4 * d;
        }
      }
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const double w0 = ok ? S[c] : 0.0, e = quad_sum_d(w0 * w0), es = wsum63_quads(e);
        if (lane == 63) ek[(size_t)(1 + c) * nb64] = es;
        if ((lane & 3) == 0) s_ew[c][lane >> 2] = e;
      }
#pragma unroll
      for (int k = 0; k < 12; k++) s_W[k][lane] = S[k];
    } else {
      const double wx = s_w0[0][lane], wy = s_w0[1][lane], wz = s_w0[2][lane];
      const double qa = S[0], qb = S[1], qc = S[2], qd = S[3];
      if (q2) {
        const double nwa = (-wx * qb + wy * qc - wz * qd) * dt * 0.5;
        const double nwb = (wx * qa - wy * qd - wz * qc) * dt * 0.5;
        S[0] = S[0] + kG4_0 * (nwa - S[4]);
        S[1] = S[1] + kG4_0 * (nwb - S[5]);
      } else {
        const double nwc = (-wx * qd - wy * qa + wz * qb) * dt * 0.5;
        const double nwd = (wx * qc + wy * qb + wz * qa) * dt * 0.5;
        S[2] = S[2] + kG4_0 * (nwc - S[6]);
        S[3] = S[3] + kG4_0 * (nwd - S[7]);
      }
      if (q2) {
        s_q0[0][lane] = S[0];
        s_q0[1][lane] = S[1];
      } else {
        s_q0[2][lane] = S[2];
        s_q0[3][lane] = S[3];
      }
    }
    __syncthreads();
    if (role == 0 && grp_ok)
      b.stepkin[grp] = kin_energy(mt, dt, et, s_ew[0][lane >> 2], s_ew[1][lane >> 2],
                                  s_ew[2][lane >> 2]);
    // quaternion derivatives from the corrected w: own components, then
    // the partner's through LDS
    double w1x = 0, w1y = 0, w1z = 0, w2x = 0, w2y = 0, w2z = 0, w3x = 0, w3y = 0, w3z = 0,
           w4x = 0, w4y = 0, w4z = 0, qa = 0, qb = 0, qc = 0, qd = 0;
    if (role >= 2) {
      w1x = s_W[0][lane]; w1y = s_W[1][lane]; w1z = s_W[2][lane];
      w2x = s_W[3][lane]; w2y = s_W[4][lane]; w2z = s_W[5][lane];
      w3x = s_W[6][lane]; w3y = s_W[7][lane]; w3z = s_W[8][lane];
      w4x = s_W[9][lane]; w4y = s_W[10][lane]; w4z = s_W[11][lane];
      S[0] = s_q0[0][lane]; S[1] = s_q0[1][lane]; S[2] = s_q0[2][lane]; S[3] = s_q0[3][lane];
      qa = S[0]; qb = S[1]; qc = S[2]; qd = S[3];
      if (q2) {
        s_p[0][lane] = (-w1x * qb + w1y * qc - w1z * qd) * dt * 0.5;
        s_p[1][lane] = (w1x * qa - w1y * qd - w1z * qc) * dt * 0.5;
      } else {
        s_p[2][lane] = (-w1x * qd - w1y * qa + w1z * qb) * dt * 0.5;
        s_p[3][lane] = (w1x * qc + w1y * qb + w1z * qa) * dt * 0.5;
      }
    }
    __syncthreads();
    double pa = 0, pb = 0, pc = 0, pd = 0;
    if (role >= 2) {
      pa = s_p[0][lane]; pb = s_p[1][lane]; pc = s_p[2][lane]; pd = s_p[3][lane];
      if (q2) {
        s_r[0][lane] = (-w2x * qb + w2y * qc - w2z * qd - w1x * pb + w1y * pc - w1z * pd) * dt * 0.25;
        s_r[1][lane] = (w2x * qa - w2y * qd - w2z * qc + w1x * pa - w1y * pd - w1z * pc) * dt * 0.25;
      } else {
        s_r[2][lane] = (-w2x * qd - w2y * qa + w2z * qb - w1x * pd - w1y * pa + w1z * pb) * dt * 0.25;
        s_r[3][lane] = (w2x * qc + w2y * qb + w2z * qa + w1x * pc + w1y * pb + w1z * pa) * dt * 0.25;
      }
    }
    __syncthreads();
    double ra = 0, rb = 0, rc_ = 0, rd = 0;
    if (role >= 2) {
      ra = s_r[0][lane]; rb = s_r[1][lane]; rc_ = s_r[2][lane]; rd = s_r[3][lane];
      if (q2) {
        s_s[0][lane] = (-w3x * qb + w3y * qc - w3z * qd - w1x * rb + w1y * rc_ - w1z * rd - w2x * pb +
                        w2y * pc - w2z * pd) * dt * (1.0 / 6.0);
        s_s[1][lane] = (w3x * qa - w3y * qd - w3z * qc + w1x * ra - w1y * rd - w1z * rc_ + w2x * pa -
                        w2y * pd - w2z * pc) * dt * (1.0 / 6.0);
      } else {
        s_s[2][lane] = (-w3x * qd - w3y * qa + w3z * qb - w1x * rd - w1y * ra + w1z * rb - w2x * pd -
                        w2y * pa + w2z * pb) * dt * (1.0 / 6.0);
        s_s[3][lane] = (w3x * qc + w3y * qb + w3z * qa + w1x * rc_ + w1y * rb + w1z * ra + w2x * pc +
                        w2y * pb + w2z * pa) * dt * (1.0 / 6.0);
      }
    }
    __syncthreads();
    if (role >= 2) {
      const double sa = s_s[0][lane], sb = s_s[1][lane], sc = s_s[2][lane], sd = s_s[3][lane];
      S[4] = pa; S[5] = pb; S[6] = pc; S[7] = pd;
      S[8] = ra; S[9] = rb; S[10] = rc_; S[11] = rd;
      S[12] = sa; S[13] = sb; S[14] = sc; S[15] = sd;
      if (q2) {
        S[16] = (-w4x * qb + w4y * qc - w4z * qd - w3x * pb + w3y * pc - w3z * pd - w2x * rb +
                 w2y * rc_ - w2z * rd - w1x * sb + w1y * sc - w1z * sd) * dt * (1.0 / 8.0);
        S[17] = (w4x * qa - w4y * qd - w4z * qc + w3x * pa - w3y * pd - w3z * pc + w2x * ra -
                 w2y * rd - w2z * rc_ + w1x * sa - w1y * sd - w1z * sc) * dt * (1.0 / 8.0);
      } else {
        S[18] = (-w4x * qd - w4y * qa + w4z * qb - w3x * pd - w3y * pa + w3z * pb - w2x * rd -
                 w2y * ra + w2z * rb - w1x * sd - w1y * sa + w1z * sb) * dt * (1.0 / 8.0);
        S[19] = (w4x * qc + w4y * qb + w4z * qa + w3x * pc + w3y * pb + w3z * pa + w2x * rc_ +
                 w2y * rb + w2z * ra + w1x * sc + w1y * sb + w1z * sa) * dt * (1.0 / 8.0);
      }
    }
  }
  // ---- predictor ----
  if (do_predict) {
    if (role == 0) {
#pragma unroll
      for (int a = 0; a < 3; a++) {
        S[a] = S[a] + S[3 + a] + S[6 + a] + S[9 + a] + S[12 + a] + S[15 + a];
        S[3 + a] = S[3 + a] + 2.0 * S[6 + a] + 3.0 * S[9 + a] + 4.0 * S[12 + a] + 5.0 * S[15 + a];
        S[6 + a] = S[6 + a] + 3.0 * S[9 + a] + 6.0 * S[12 + a] + 10.0 * S[15 + a];
        S[9 + a] = S[9 + a] + 4.0 * S[12 + a] + 10.0 * S[15 + a];
        S[12 + a] = S[12 + a] + 5.0 * S[15 + a];
      }
    } else if (role == 1) {
#pragma unroll
      for (int a = 0; a < 3; a++) {
        S[a] = S[a] + S[3 + a] + S[6 + a] + S[9 + a] + S[12 + a];
        S[3 + a] = S[3 + a] + 2.0 * S[6 + a] + 3.0 * S[9 + a] + 4.0 * S[12 + a];
        S[6 + a] = S[6 + a] + 3.0 * S[9 + a] + 6.0 * S[12 + a];
        S[9 + a] = S[9 + a] + 4.0 * S[12 + a];
      }
    } else {
      if (q2) {
        predict_qc<0>(S);
        predict_qc<1>(S);
        s_qn[0][lane] = S[0];
        s_qn[1][lane] = S[1];
      } else {
        predict_qc<2>(S);
        predict_qc<3>(S);
        s_qn[2][lane] = S[2];
        s_qn[3][lane] = S[3];
      }
    }
    __syncthreads();
    if (role >= 2) {
      // all four predicted components, normalised in the order of rigid_predict
      S[0] = s_qn[0][lane]; S[1] = s_qn[1][lane]; S[2] = s_qn[2][lane]; S[3] = s_qn[3][lane];
      const double re = 1.0 / sqrt(S[0] * S[0] + S[1] * S[1] + S[2] * S[2] + S[3] * S[3]);
#pragma unroll
      for (int a = 0; a < 4; a++) S[a] = S[a] * re;
    }
  }
  if (ok && (do_predict || do_correct)) {
    if (role == 0) {
#pragma unroll
      for (int a = 0; a < 3; a++) b.com[a * n + i] = S[a];
#pragma unroll
      for (int k = 0; k < 15; k++) b.dx[k * n + i] = S[3 + k];
    } else if (role == 1) {
#pragma unroll
      for (int k = 0; k < 15; k++) b.w[k * n + i] = S[k];
    } else if (q2) {
      store_qc<0>(b, n, i, S);
    } else {
      store_qc<2>(b, n, i, S);
    }
  }
  if (do_sites && ok) {
    if (role == 0) {
      double *rec = b.rec + ((size_t)half * n + i) * b.rs;
#pragma unroll
      for (int a = 0; a < 3; a++) {
        rec[a] = S[a];
        if (b.scan) b.comp[(3 * half + a) * n + i] = S[a];
      }
      if (!b.scan) {
        int jc[3], nd[3];
        grid_nd<BOX>(g, nd);
  #pragma unroll
        for (int a = 0; a < 3; a++) {
          double d = S[a];
          const double o = round(d * bx.invL[a]) * bx.L[a];
          d = d - o;
          int j = (int)round(d * bx.cellinv[a]);
          if (j < 0) j += nd[a];
          j = ((j % nd[a]) + nd[a]) % nd[a];
          jc[a] = j;
        }
        const int c = (jc[2] * nd[1] + jc[1]) * nd[0] + jc[0];
        b.cell[i] = c;
        // slot 0 of a cell row is its count; residents follow
        int *cr = b.cellres + ((size_t)list * g.ncell + c) * b.cell_cap;
        const int slot = atomicAdd(cr, 1) + 1;
        if (slot < b.cell_cap)
          cr[slot] = i;
        else
          raise_flag(b.flags, 3);  // cell capacity exceeded
      }
      if (b.half_skin2 > 0.0) {
        // a pair of the rows moves by at most twice the largest displacement
        // plus |L - L_ref| (image shifts of one box per axis)
        double h2 = b.half_skin2;
        if (NPT) {
          const double e0 = bx.L[0] - b.box[9], e1 = bx.L[1] - b.box[10], e2 = bx.L[2] - b.box[11];
          const double h = sqrt(b.half_skin2) - 0.5 * sqrt(e0 * e0 + e1 * e1 + e2 * e2);
          h2 = h > 0.0 ? h * h : -1.0;
        }
        const double e0 = S[0] - cref[0], e1 = S[1] - cref[1], e2 = S[2] - cref[2];
        if (e0 * e0 + e1 * e1 + e2 * e2 > h2) b.flags[2 + list] = 1;
      } else if (i == 0) {
        b.flags[2 + list] = 1;  // no skin: the reference rebuilds every step
      }
      if (NPT && i == 0 &&
          (bx.L[0] < b.box[12] * b.box[15] || bx.L[1] < b.box[13] * b.box[15] ||
           bx.L[2] < b.box[14] * b.box[15]))
        raise_flag(b.flags, 5);  // cells below (rc+skin)/2
    } else if (role >= 2) {
      // rigid_setmatrix and the site offsets; the two waves split the stores
      const double qa = S[0], qb = S[1], qc = S[2], qd = S[3];
      t[0] = (qa * qa + qb * qb - (qc * qc + qd * qd));
      t[1] = -2.0 * (qa * qd + qb * qc);
      t[2] = 2.0 * (qb * qd - qa * qc);
      t[3] = 2.0 * (qa * qd - qb * qc);
      t[4] = qa * qa + qc * qc - (qb * qb + qd * qd);
      t[5] = -2.0 * (qa * qb + qc * qd);
      t[6] = 2.0 * (qa * qc + qb * qd);
      t[7] = 2.0 * (qa * qb - qc * qd);
      t[8] = qa * qa + qd * qd - (qb * qb + qc * qc);
      if (q2) {
#pragma unroll
        for (int a = 0; a < 5; a++) b.tmat[a * n + i] = t[a];
      } else {
#pragma unroll
        for (int a = 5; a < 9; a++) b.tmat[a * n + i] = t[a];
      }
      double *rec = b.rec + ((size_t)half * n + i) * b.rs;
      float *recf = reinterpret_cast<float *>(rec + 4);
      const int nq = mt.nsite - 1, mid = (nq + 1) / 2;
      const int s0 = q2 ? 0 : mid, s1 = q2 ? mid : nq;
      for (int s = s0; s < s1; s++) {
        const double r0 = t[0] * mt.bx[s] + t[1] * mt.by[s] + t[2] * mt.bz[s];
        const double r1 = t[3] * mt.bx[s] + t[4] * mt.by[s] + t[5] * mt.bz[s];
        const double r2 = t[6] * mt.bx[s] + t[7] * mt.by[s] + t[8] * mt.bz[s];
        if (b.rs == kRecF) {
          recf[s * 3 + 0] = (float)r0;
          recf[s * 3 + 1] = (float)r1;
          recf[s * 3 + 2] = (float)r2;
        } else {
          rec[4 + s * 3 + 0] = r0;
          rec[4 + s * 3 + 1] = r1;
          rec[4 + s * 3 + 2] = r2;
        }
      }
    }
  }
}

template <int BOX>
__global__ __launch_bounds__(256) void k_md_pre(ModelTable mt, Geom g, MdBuf b, double dt,
                                                int nose_active, int do_correct, int do_predict,
                                                int do_sites, int list, int half) {
  md_pre_body<BOX>(mt, g, b, dt, nose_active, do_correct, do_predict, do_sites, list, half,
                   blockIdx.x);
}

// Ladder form: one launch over the blocks of every system of a ladder;
// map[blockIdx.x] names the system and its block (system < 0: an idle block
// that pads the XCD interleave).
__global__ __launch_bounds__(256) void k_md_pre_lad(ModelTable mt, const MdRep *__restrict__ reps,
                                                    const int2 *__restrict__ map, int do_correct,
                                                    int do_predict, int list, int half) {
  const int2 m = map[blockIdx.x];
  if (m.x < 0) return;
  const Geom g = reps[m.x].g;
  const MdBuf b = reps[m.x].b;
  md_pre_body<kBoxCube>(mt, g, b, reps[m.x].dt, reps[m.x].nose_active, do_correct, do_predict,
                        do_predict, list, half, m.y);
}

template <bool NPT>
__global__ __launch_bounds__(1024) void k_md_close(ModelTable mt, MdBuf b, int n, int ncell,
                                                   double box_vol, CloseArgs ca) {
  __shared__ double s_red[4][kRed];
  close_body<NPT, true>(mt, b, n, ncell, box_vol, ca, s_red);
}

// ---- kernel B --------------------------------------------------------------

// Cell stencil of the MD grid: per axis na offsets from lo; on an axis of
// nd >= 5 cells the 5 offsets -2..2 are distinct cells and are pruned by
// their distance from the molecule, on a shorter axis every cell is taken
// once (no pruning).
struct Stencil {
  int na[3], lo[3], nst;
  bool prune[3], any;
};
__device__ inline Stencil stencil_of(const int (&nd)[3]) {
  Stencil st;
  st.nst = 1;
  st.any = false;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    st.prune[a] = nd[a] >= 5;
    st.na[a] = st.prune[a] ? 5 : nd[a];
    st.lo[a] = st.prune[a] ? -2 : -((nd[a] - 1) / 2);
    st.nst *= st.na[a];
    st.any = st.any || st.prune[a];
  }
  return st;
}

// Distance in cell units from a point at u (cell units from the centre of
// its cell, |u| <= 1/2) to the cell at offset o, which spans [o-1/2, o+1/2];
// shrunk by 1e-9 so that rounding in the binning never drops a cell.
__device__ inline double cell_gap(int o, double u) {
  const double a = (double)o - 0.5 - u, c = u - (double)o - 0.5;
  return fmax(0.0, fmax(a, c) - 1e-9);
}

__device__ inline double frac_in_cell(const BoxNow &bx, double x, int a) {
  const double d = x - round(x * bx.invL[a]) * bx.L[a];
  const double t = d * bx.cellinv[a];
  return t - round(t);
}

// The FP64 minimum-image test of Interaction_Compress2 at rc + skin for one
// candidate: whether j is in i's row, and its image shift code.
__device__ inline bool row_test(const BoxNow &bx, const MdBuf &b, double rr, double d0, double d1,
                                double d2, int &code) {
  const double k0 = round(d0 * bx.invL[0]), k1 = round(d1 * bx.invL[1]),
               k2 = round(d2 * bx.invL[2]);
  d0 = d0 - k0 * bx.L[0];
  d1 = d1 - k1 * bx.L[1];
  d2 = d2 - k2 * bx.L[2];
  const double dd = d0 * d0 + d1 * d1 + d2 * d2;
  const bool pass = dd < rr;
  code = ((int)k0 & 1023) | (((int)k1 & 1023) << 10) | (((int)k2 & 1023) << 20);
  if (pass && (fabs(k0) > 511.0 || fabs(k1) > 511.0 || fabs(k2) > 511.0)) raise_flag(b.flags, 2);
  return pass;
}

// Row of molecule i from a scan of every molecule in index order: the row
// comes out sorted, with no cell lists.  Four candidates per lane are loaded
// together (the COM components are read from the arrays the predictor wrote,
// which are contiguous in j), so the cost is n / 64 tests per lane and no
// latency of cell counts, search and sort.  Taken up to kScanMax molecules.
template <int BOX>
__device__ inline int scan_row(const Geom &g, const MdBuf &b, const double *com, int i, int lane,
                               double xi, double yi, double zi, int *nj, int *nc) {
  const BoxNow bx = box_now<BOX>(g, b);
  const int n = g.n, cap = b.maxnb;
  const unsigned long long lt = (1ull << lane) - 1ull;
  int base = 0;
  for (int j0 = 0; j0 < n; j0 += 256) {
    double x[4], y[4], z[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = min(j0 + 64 * u + lane, n - 1);
      x[u] = com[j];
      y[u] = com[n + j];
      z[u] = com[2 * n + j];
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = j0 + 64 * u + lane;
      int code = 0;
      const bool pass =
          j < n && j != i && row_test(bx, b, g.rr, xi - x[u], yi - y[u], zi - z[u], code);
      const unsigned long long mask = __ballot(pass);
      const int pos = base + __popcll(mask & lt);
      if (pass) {
        if (pos < cap) {
          nj[pos] = j;
          nc[pos] = code;
        } else {
          raise_flag(b.flags, 4);  // neighbour-row capacity exceeded
        }
      }
      base += __popcll(mask);
    }
  }
  return min(base, cap);
}

// Row of molecule i from the cell lists, sorted by j so that the force sums
// do not depend on the order in which the binning atomics filled the cells.
// The sort places every entry at the number of smaller j in the row: a bit
// per molecule index in LDS (a window of 32 * kRowWords indices at a time),
// the words' running counts, and the bits below j in its word.  (Counting the
// smaller entries of the row per entry is 3 passes of 176 LDS reads at 4096
// molecules, skin 1.8 A, twice the instructions of a step without a build; it
// stays where the windows are many.)
constexpr int kWindowEntries = 18;
template <int BOX>
__device__ inline int cell_row(const Geom &g, const MdBuf &b, const double *rec, int list, int i,
                               int lane, double xi, double yi, double zi, int *s_j, int *nj,
                               int *nc) {
  const BoxNow bx = box_now<BOX>(g, b);
  const int n = g.n;
  int *s_c = s_j + b.maxnb;
  unsigned *s_bit = reinterpret_cast<unsigned *>(s_c + b.maxnb);
  int *s_cnt = reinterpret_cast<int *>(s_bit + kRowWords);
  int *s_beg = s_cnt + kRowWords, *s_pre = s_beg + 128;
  int nd[3];
  grid_nd<BOX>(g, nd);
  const int nx = nd[0], ny = nd[1], nz = nd[2];
  const int c = b.cell[i];
  const int cx = c % nx, cy = (c / nx) % ny, cz = c / (nx * ny);
  const Stencil st = stencil_of(nd);
  const double ux = frac_in_cell(bx, xi, 0), uy = frac_in_cell(bx, yi, 1),
               uz = frac_in_cell(bx, zi, 2);
  const int *res = b.cellres + (size_t)list * g.ncell * b.cell_cap;
  int carry = 0;
  for (int e0 = 0; e0 < st.nst; e0 += 64) {
    const int e = e0 + lane;
    int len = 0;
    if (e < st.nst) {
      const int ox = st.lo[0] + e % st.na[0], oy = st.lo[1] + (e / st.na[0]) % st.na[1],
                oz = st.lo[2] + e / (st.na[0] * st.na[1]);
      bool keep = true;
      if (BOX == kBoxCube && st.any) {  // in cell units of the cube
        const double gx = cell_gap(ox, ux), gy = cell_gap(oy, uy), gz = cell_gap(oz, uz);
        keep = gx * gx + gy * gy + gz * gz <= g.rr * (bx.cellinv[0] * bx.cellinv[0]);
      } else if (st.any) {  // the gap to the cell in A on the pruned axes
        const double gx = st.prune[0] ? cell_gap(ox, ux) / bx.cellinv[0] : 0.0;
        const double gy = st.prune[1] ? cell_gap(oy, uy) / bx.cellinv[1] : 0.0;
        const double gz = st.prune[2] ? cell_gap(oz, uz) / bx.cellinv[2] : 0.0;
        keep = gx * gx + gy * gy + gz * gz <= g.rr;
      }
      const int c2 = ((((cz + oz) % nz + nz) % nz) * ny + ((cy + oy) % ny + ny) % ny) * nx +
                     ((cx + ox) % nx + nx) % nx;
      s_beg[e] = c2 * b.cell_cap + 1;
      if (keep) len = min(res[(size_t)c2 * b.cell_cap], b.cell_cap - 1);
    }
    int inc = len;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(inc, d, 64);
      if (lane >= d) inc += v;
    }
    if (e < st.nst) s_pre[e + 1] = carry + inc;
    carry += __shfl(inc, 63, 64);
  }
  if (lane == 0) s_pre[0] = 0;
  wsync();
  const int total = s_pre[st.nst];
  int base = 0;
  const int cap = b.maxnb;
  for (int t0 = 0; t0 < total; t0 += 64) {
    const int t = t0 + lane;
    bool pass = false;
    int j = 0, code = 0;
    if (t < total) {
      int lo = 0, hi = st.nst;  // s_pre[lo] <= t < s_pre[hi]
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (s_pre[mid] <= t) lo = mid;
        else hi = mid;
      }
      j = res[s_beg[lo] + (t - s_pre[lo])];
      if (j != i) {
        const double *recj = rec + (size_t)j * b.rs;
        pass = row_test(bx, b, g.rr, xi - recj[0], yi - recj[1], zi - recj[2], code);
      }
    }
    const unsigned long long mask = __ballot(pass);
    const int pos = base + __popcll(mask & ((1ull << lane) - 1ull));
    if (pass) {
      if (pos < cap) {
        s_j[pos] = j;
        s_c[pos] = code;
      } else {
        raise_flag(b.flags, 4);  // neighbour-row capacity exceeded
      }
    }
    base += __popcll(mask);
  }
  wsync();
  const int m = min(base, cap);
  // The windows cost by the molecules of the system, counting the smaller
  // entries by the square of the row's: the line lies at kWindowEntries row
  // entries a window.  Step with rows rebuilt, windows / counting, rows of 102
  // entries: 4096 molecules 31.4 / 34.8 us, 16,384 94 / 97, 32,768 169 / 160,
  // 65,536 389 / 308; of 38 entries: 8192 43.2 / 42.3, 32,768 129 / 112; of 242:
  // 32,768 268 / 323, 65,536 599 / 616.
  if ((n + 32 * kRowWords - 1) / (32 * kRowWords) * kWindowEntries > m) {
    for (int t = lane; t < m; t += 64) {
      const int key = s_j[t];
      int rank = 0;
      for (int u = 0; u < m; u++) rank += s_j[u] < key;
      nj[rank] = key;
      nc[rank] = s_c[t];
    }
    return m;
  }
  // windows of the index range: the bits of the entries, the running counts
  // of the words (two words per lane of the wave), the entries' places
  int below = 0;
  for (int w0 = 0; w0 < n; w0 += 32 * kRowWords) {
#pragma unroll
    for (int u = 0; u < kRowWords / 64; u++) s_bit[64 * u + lane] = 0u;
    wsync();
    for (int t = lane; t < m; t += 64) {
      const unsigned q = (unsigned)(s_j[t] - w0);
      if (q < 32u * kRowWords) atomicOr(&s_bit[q >> 5], 1u << (q & 31));
    }
    wsync();
    int cnt[kRowWords / 64], sum = 0;
#pragma unroll
    for (int u = 0; u < kRowWords / 64; u++) {
      cnt[u] = __popc(s_bit[lane * (kRowWords / 64) + u]);
      sum += cnt[u];
    }
    int inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(inc, d, 64);
      if (lane >= d) inc += v;
    }
    int run = below + inc - sum;
#pragma unroll
    for (int u = 0; u < kRowWords / 64; u++) {
      s_cnt[lane * (kRowWords / 64) + u] = run;
      run += cnt[u];
    }
    below += __shfl(inc, 63, 64);
    wsync();
    for (int t = lane; t < m; t += 64) {
      const int key = s_j[t];
      const unsigned q = (unsigned)(key - w0);
      if (q < 32u * kRowWords) {
        const int rank = s_cnt[q >> 5] + __popc(s_bit[q >> 5] & ((1u << (q & 31)) - 1u));
        nj[rank] = key;
        nc[rank] = s_c[t];
      }
    }
    wsync();
  }
  return m;
}

// neighbour-row build of molecule i into nbr[i*maxnb ...], in the order of
// j; returns the row length (also stored).
template <int BOX>
__device__ inline int build_row(const Geom &g, const MdBuf &b, int list, int half, int i, int lane,
                                int *s_sort) {
  constexpr bool NPT = BOX == kBoxBaro;
  const int n = g.n;
  const double *rec = b.rec + (size_t)half * n * b.rs;
  const double *reci = rec + (size_t)i * b.rs;
  const double xi = reci[0], yi = reci[1], zi = reci[2];
  int *nj = b.nbr_j + (size_t)i * b.maxnb;
  int *nc = b.nbr_code + (size_t)i * b.maxnb;
  const int m = b.scan ? scan_row<BOX>(g, b, b.comp + (size_t)3 * half * n, i, lane, xi, yi, zi, nj,
                                       nc)
                       : cell_row<BOX>(g, b, rec, list, i, lane, xi, yi, zi, s_sort, nj, nc);
  wsync();  // the force loop reads entries other lanes wrote
  if (lane == 0) {
    b.nbr_cnt[i] = m;
    b.com_ref[i] = xi;
    b.com_ref[n + i] = yi;
    b.com_ref[2 * n + i] = zi;
    if (NPT && i == 0) {  // the box the rows were built in
      const BoxNow bx = box_now<BOX>(g, b);
      b.box[9] = bx.L[0];
      b.box[10] = bx.L[1];
      b.box[11] = bx.L[2];
    }
  }
  return m;
}

// A wave's interacting entries in its LDS region: the index of j and the COM
// separation in the pair precision, one 16-byte entry (FP32) or an index and
// three component arrays (FP64).
template <typename R>
struct PairList;
template <>
struct PairList<float> {
  float4 *e;
  __device__ PairList(unsigned char *reg, int) : e(reinterpret_cast<float4 *>(reg)) {}
  __device__ void put(int p, int j, double d0, double d1, double d2) {
    e[p] = make_float4((float)d0, (float)d1, (float)d2, __int_as_float(j));
  }
  __device__ void get(int p, int &j, float (&d)[3]) const {
    const float4 v = e[p];
    d[0] = v.x;
    d[1] = v.y;
    d[2] = v.z;
    j = __float_as_int(v.w);
  }
};
template <>
struct PairList<double> {
  int *j_;
  double *d_;
  int stride;
  __device__ PairList(unsigned char *reg, int cap)
      : j_(reinterpret_cast<int *>(reg)),
        d_(reinterpret_cast<double *>(reg + (4 * cap + 15) / 16 * 16)),
        stride((8 * cap + 15) / 16 * 2) {}
  __device__ void put(int p, int j, double d0, double d1, double d2) {
    j_[p] = j;
    d_[p] = d0;
    d_[stride + p] = d1;
    d_[2 * stride + p] = d2;
  }
  __device__ void get(int p, int &j, double (&d)[3]) const {
    j = j_[p];
    d[0] = d_[p];
    d[1] = d_[stride + p];
    d[2] = d_[2 * stride + p];
  }
};

// image shift of axis A in a row entry's code (10-bit signed fields)
template <int A>
__device__ inline int shift_of(int code) {
  return (int)((unsigned)code << (22 - 10 * A)) >> 22;
}

// The pair forces on molecule i by its wave: its row is rebuilt if a rebuild
// is due, the row's pairs within rc are compacted into the wave's LDS region
// `reg`, then evaluated.  The results are each lane's sums over its own pairs
// (two or three in a liquid) in the pair precision.
template <typename R>
struct PairOut {
  R F[3], T[3], e, v[9];
  int npair, nlist;  // wave-uniform counts
};
template <int M, typename R, int BOX, class Mid>
__device__ __forceinline__ void pair_phase(const Geom &g, const MdBuf &b, const PairK<R> &pk,
                                           int rebuild, int list, int half, int i, int lane,
                                           unsigned char *reg, PairOut<R> &o, Mid &&mid) {
  using T = Traits<M>;
  const int cap = b.maxnb;
  const BoxNow bl = box_now<BOX>(g, b);
  const double *rec = b.rec + (size_t)half * g.n * b.rs;
  const int *nj = b.nbr_j + (size_t)i * cap;
  const int *nc = b.nbr_code + (size_t)i * cap;
  // the first round of row entries is fetched with the row length (or
  // right after a rebuild)
  int jj[4], cc[4];
  int m;
  if (rebuild) {
    m = build_row<BOX>(g, b, list, half, i, lane, reinterpret_cast<int *>(reg));
    o.nlist = m;
  } else {
    m = b.nbr_cnt[i];
  }
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int k = 64 * u + lane;
    jj[u] = k < cap ? nj[k] : i;
    cc[u] = k < cap ? nc[k] : 0;
  }
  // entries at or past the row length hold stale or never-written values:
  // they are replaced before any of them forms an address
#pragma unroll
  for (int u = 0; u < 4; u++) {
    if (64 * u + lane >= m) {
      jj[u] = i;
      cc[u] = 0;
    }
  }
  const double *reci = rec + (size_t)i * b.rs;
  const double xi = reci[0], yi = reci[1], zi = reci[2];
  // pass 1: the reference's FP64 interaction test on every row entry; the
  // entries that pass are compacted in row order into LDS
  PairList<R> pl(reg, cap);
  wsync();  // the sort buffers of build_row share this region
  int np = 0;
  // four entries per lane per round: the index loads, then the record
  // loads, are in flight together; whole waves past the row are skipped
  for (int k0 = 0; k0 < m; k0 += 256) {
    if (k0 > 0) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int k = k0 + 64 * u + lane;
        jj[u] = k < m ? nj[k] : i;
        cc[u] = k < m ? nc[k] : 0;
      }
    }
    double xj[4], yj[4], zj[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (k0 + 64 * u >= m) break;
      const double *recj = rec + (size_t)jj[u] * b.rs;
      xj[u] = recj[0];
      yj[u] = recj[1];
      zj[u] = recj[2];
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (k0 + 64 * u >= m) break;
      const int code = cc[u];
      const double d0 = (xi - xj[u]) - (double)shift_of<0>(code) * bl.L[0];
      const double d1 = (yi - yj[u]) - (double)shift_of<1>(code) * bl.L[1];
      const double d2 = (zi - zj[u]) - (double)shift_of<2>(code) * bl.L[2];
      const bool pass = k0 + 64 * u + lane < m && d0 * d0 + d1 * d1 + d2 * d2 < g.rc2;
      const unsigned long long mask = __ballot(pass);
      if (pass) pl.put(np + __popcll(mask & ((1ull << lane) - 1ull)), jj[u], d0, d1, d2);
      np += __popcll(mask);
    }
  }
  o.npair = np;
  mid();
  wsync();
  // pass 2: the interacting pairs, densely, two per lane per round
  R ri[T::NS][3];
  RecSites<M, R>::load(reci, ri);
  R(&Fr)[3] = o.F;
  R(&Tr)[3] = o.T;
  R(&vr)[9] = o.v;
  auto eval = [&](R d0, R d1, R d2, const R (&rj)[T::NS][3]) {
    R Fp[3], Tp[3];
    const R e = pair_on_i<M, R>(pk, d0 * d0 + d1 * d1 + d2 * d2, d0, d1, d2, ri, rj, Fp, Tp);
    Fr[0] += Fp[0]; Fr[1] += Fp[1]; Fr[2] += Fp[2];
    Tr[0] += Tp[0]; Tr[1] += Tp[1]; Tr[2] += Tp[2];
    o.e += e;
    // pair virial d (x) F, fused multiply-adds
    const R dd3[3] = {d0, d1, d2};
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int c = 0; c < 3; c++) vr[3 * a + c] = fma_r(dd3[a], Fp[c], vr[3 * a + c]);
  };
  for (int k0 = 0; k0 < np; k0 += 128) {
    const int ka = k0 + lane, kb = k0 + 64 + lane;
    R da[3] = {R(0), R(0), R(0)}, db[3] = {R(0), R(0), R(0)};
    int ja = i, jb = i;
    if (ka < np) pl.get(ka, ja, da);
    if (kb < np) pl.get(kb, jb, db);
    R ra[T::NS][3], rb[T::NS][3];
    RecSites<M, R>::load(rec + (size_t)ja * b.rs, ra);
    RecSites<M, R>::load(rec + (size_t)jb * b.rs, rb);
    if (ka < np) eval(da[0], da[1], da[2], ra);
    if (kb < np) eval(db[0], db[1], db[2], rb);
  }
}

template <typename R>
__device__ inline void pair_zero(PairOut<R> &o) {
#pragma unroll
  for (int a = 0; a < 3; a++) o.F[a] = o.T[a] = R(0);
  o.e = R(0);
#pragma unroll
  for (int q = 0; q < 9; q++) o.v[q] = R(0);
  o.npair = o.nlist = 0;
}

// The wave's force and lab torque of its molecule: lane l < 6 component l.
template <typename R>
__device__ inline double force_torque(const PairOut<R> &o, int lane) {
  const double v[6] = {(double)o.F[0], (double)o.F[1], (double)o.F[2],
                       (double)o.T[0], (double)o.T[1], (double)o.T[2]};
  return wsum_six(v, lane);
}

// each lane's energy and virial into its wave's LDS region [10][64], which
// the compacted entries no longer need
template <typename R>
__device__ inline void park_sums(const PairOut<R> &o, unsigned char *reg, int lane,
                                 double (&s_cnt)[2]) {
  double *acc = reinterpret_cast<double *>(reg);
  acc[lane] = (double)o.e;
#pragma unroll
  for (int q = 0; q < 9; q++) acc[(1 + q) * 64 + lane] = (double)o.v[q];
  if (lane == 0) {
    s_cnt[0] = (double)o.npair;
    s_cnt[1] = (double)o.nlist;
  }
}
// block partial of quantity q (energy, virial) from the parked lanes, in a
// fixed order: thread (q, seg) sums lanes seg, seg+16, ... of the 256 (for
// each u the 16 threads of a DPP row read 16 consecutive doubles: no bank
// conflict), compensated (TwoSum over the 16 terms and the row), halved
// (every pair is met from both sides)
__device__ inline void block_sum(const unsigned char *s_dyn, int reg_bytes, int q, int seg,
                                 double *out) {
  double r = 0.0, rc = 0.0;
#pragma unroll
  for (int u = 0; u < 16; u++) {
    const int L = seg + 16 * u;
    two_sum_acc(r, rc,
                reinterpret_cast<const double *>(s_dyn + (size_t)(L >> 6) * reg_bytes)[q * 64 + (L & 63)]);
  }
  rowsum16_dd(r, rc);
  if (seg == 0) out[q] = 0.5 * (r + rc);
}

// blk is the block's index within its system and nblk the system's block
// count (blockIdx.x and gridDim.x for one system).
template <int M, typename R, int BOX>
__device__ __forceinline__ void md_main_body(const Geom &g, const MdBuf &b, const PairK<R> &pk,
                                             double *out, int parity, int reg_bytes, int blk,
                                             int nblk) {
  extern __shared__ __align__(16) unsigned char s_dyn[];  // [4][reg_bytes]
  __shared__ double s_cnt[4][2];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n = g.n;
  const int i = blk * 4 + wid;
  unsigned char *reg = s_dyn + (size_t)wid * reg_bytes;
  PairOut<R> o;
  pair_zero(o);
  if (i < n) {
    pair_phase<M, R, BOX>(g, b, pk, b.flags[2 + parity], parity, 0, i, lane, reg, o, [] {});
    const double ft = force_torque(o, lane);
    if (out) {
      // molecule force (lab) and body torque, as rigid_collectforce
      const double t0 = __shfl(ft, 3, 64), t1 = __shfl(ft, 4, 64), t2 = __shfl(ft, 5, 64);
      if (lane < 3) {
        const double *t = b.tmat + i;
        out[lane * n + i] = ft;
        out[(3 + lane) * n + i] = t[lane * n] * t0 + t[(3 + lane) * n] * t1 + t[(6 + lane) * n] * t2;
      }
    } else if (lane < 6) {
      b.frc[lane * n + i] = ft;
    }
    wsync();  // every lane has read the compacted entries
  }
  park_sums(o, reg, lane, s_cnt[wid]);
  __syncthreads();
  double *part = b.blockpart + ((size_t)parity * nblk + blk) * kBP;
  if (threadIdx.x < 160) {
    block_sum(s_dyn, reg_bytes, threadIdx.x >> 4, threadIdx.x & 15, part);
  } else if (threadIdx.x < 162) {
    const int q = threadIdx.x - 160;
    part[10 + q] = 0.5 * (s_cnt[0][q] + s_cnt[1][q] + s_cnt[2][q] + s_cnt[3][q]);
  }
}

// Waves per SIMD the row kernel is compiled for (register budget)
template <int M, typename R>
constexpr int main_waves_per_eu() {
  // FP32 TIP4P and SPC/E rows fit in 96 VGPRs: five waves per SIMD, so that a
  // 4096-molecule grid plus the step-close block (1025 blocks) is resident
  // at once on 256 CUs (four waves per SIMD leave the last block waiting for
  // a slot, which set the kernel's end)
  if (sizeof(R) == 4 && (M == G6_TIP4P || M == G6_SPCE || M == G6_OPLSMEOH)) return 5;
  return (M != G6_ST2 && M != G6_NVDE && sizeof(R) == 4) ? 4 : 1;
}

// ---- the step kernel ---------------------------------------------------------
// One kernel per step of a fixed-box system on the rows: the pair forces of
// step q at the predicted positions, the corrector of the block's four
// molecules with the Nose drag, and their predictor, records, binning and
// skin test for step q + 1.  A step of two kernels (predictor and forces) at
// 4096 molecules spent 6 us in the per-molecule kernel, which is latency
// alone, and a launch boundary between them.
//
// The corrector needs zeta of this step, that is, the whole system's kinetic
// energy of the step before.  That step's kernel left the kinetic energy of
// every block of four molecules, and every block sums them again, in the same
// order, in the shadow of its pair phase: 1024 values at 4096 molecules.  No
// block waits for another.
//
// Buffers alternate so that no block writes what another may still read:
// records, scanned COMs, the thermostat state and the partials by parity,
// cell lists and rebuild flags in threes (read, filled, cleared).
//
// Roles after the pair phase, 16 lanes each (a quad per molecule, a lane per
// component): wave 0 translation, binning and skin test; wave 1 angular
// velocity; wave 2 quaternions, rotation and site offsets; wave 3 kinetic
// sums; waves 1 to 3 the block's energy and virial sums.  Every component
// keeps md_pre_body's operation order, which is the reference's, so the
// states are the same bits as the two-kernel step's.

struct StepArgs {
  int parity;       // of this step's records, partials and thermostat state
  int list;         // cell list and rebuild flag of this step
  int first, last;  // no step before (the thermostat state is this step's) / after
  int nose_active;
  double dt;
};

// blk: the index of the block's four molecules, one per wave; nblk: the
// system's blocks.
template <int M, typename R, int BOX>
__device__ __forceinline__ void md_step_body(const ModelTable &mt, const Geom &g, const MdBuf &b,
                                             const PairK<R> &pk, const StepArgs &st, int reg_bytes,
                                             int blk, int nblk) {
  extern __shared__ __align__(16) unsigned char s_dyn[];  // [4][reg_bytes]
  __shared__ double s_cnt[4][2], s_kin[4], s_z[9];
  __shared__ double s_st[kStateRows * 4];   // the Gear state of the block's molecules
  __shared__ double s_ft[4][6];             // force and lab torque
  __shared__ double s_v[4][3], s_W[4][12];  // corrected dx(1) and w levels 0..3
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n = g.n;
  const int par = st.parity;
  const int rebuild = b.flags[2 + st.list];
  // What the corrector reads - the state block's columns of the molecules, the
  // kinetic energies and the thermostat state of the step before - is fetched
  // ahead of the pairs and parked in LDS once the row has been tested: each
  // block starts on cold caches, and a load after the pairs would add a
  // memory latency to the step (4096 molecules: 0.8 us of 19).
  const bool kin_sum = st.nose_active && !st.first;
  const double *kin_in = b.stepkin + (size_t)(1 - par) * nblk;
  double pst, pkin[4], pz = 0.0;
  {
    const int row = threadIdx.x >> 2, i = blk * 4 + (threadIdx.x & 3);
    pst = row < kStateRows && i < n ? b.com[(size_t)row * n + i] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int k = threadIdx.x + 256 * u;
    pkin[u] = kin_sum && k < nblk ? kin_in[k] : 0.0;
  }
  if (threadIdx.x < 9) pz = b.nose[9 * (st.first ? par : 1 - par) + threadIdx.x];
  auto park = [&]() {
    if (threadIdx.x < kStateRows * 4) s_st[threadIdx.x] = pst;
    if (threadIdx.x < 9) s_z[threadIdx.x] = pz;
    if (kin_sum) {
      double s = 0.0;
#pragma unroll
      for (int u = 0; u < 4; u++) s += pkin[u];
#pragma unroll 4
      for (int k = threadIdx.x + 1024; k < nblk; k += 256) s += kin_in[k];
      s = wsum63(s);
      if (lane == 63) s_kin[wid] = s;
    }
  };
  unsigned char *reg = s_dyn + (size_t)wid * reg_bytes;
  PairOut<R> o;
  pair_zero(o);
  if (blk * 4 + wid < n)
    pair_phase<M, R, BOX>(g, b, pk, rebuild, st.list, par, blk * 4 + wid, lane, reg, o, park);
  else
    park();
  const double ft = force_torque(o, lane);
  if (lane < 6) s_ft[wid][lane] = ft;
  wsync();  // every lane has read the compacted entries
  park_sums(o, reg, lane, s_cnt[wid]);
  __syncthreads();
  double *part = b.blockpart + ((size_t)par * nblk + blk) * kBP;

  // lane m * 4 + a holds component a of molecule m
  const int m = (lane >> 2) & 3, a = lane & 3;
  const int i = blk * 4 + m;
  const bool ok = lane < 16 && i < n;
  const int ax = a < 3 ? a : 0;
  double S[6], X[4], cref = 0.0;
#pragma unroll
  for (int k = 0; k < 6; k++) S[k] = 0.0;
#pragma unroll
  for (int k = 0; k < 4; k++) X[k] = 0.0;
  auto state = [&](int row) { return s_st[row * 4 + m]; };
  if (wid == 0) {
#pragma unroll
    for (int k = 0; k < 6; k++) S[k] = state(3 * k + ax);  // com, dx levels
    cref = state(kRowRef + ax);
  } else if (wid == 1) {
#pragma unroll
    for (int k = 0; k < 5; k++) S[k] = state(kRowW + 3 * k + ax);
#pragma unroll
    for (int c = 0; c < 4; c++) X[c] = state(kRowQ + c);
  } else if (wid == 2) {
#pragma unroll
    for (int k = 0; k < 5; k++) S[k] = state(kRowQ + 4 * k + a);
#pragma unroll
    for (int c = 0; c < 3; c++) X[c] = state(kRowW + c);
  }
  const int rs = b.rs;
  double *rec = b.rec + (size_t)(1 - par) * n * rs;  // the next step's records
  double *com = b.com;
  const double dt = st.dt;
  if (wid < 2) {
    // zeta of this step: the state of the step before, corrected with its
    // temperature and predicted (the step close stores the same values)
    double zeta0 = 0.0;
    if (st.nose_active) {
      double z[9];
#pragma unroll
      for (int q = 0; q < 9; q++) z[q] = s_z[q];
      if (!st.first) {
        const double ek = s_kin[0] + s_kin[1] + s_kin[2] + s_kin[3];
        nose_correct(z, temperature_of(ek, n));
        nose_predict(z);
      }
      zeta0 = z[3];
    }
    const double nc = zeta0 * dt;
    if (wid == 0) {
      if (!ok || a == 3) {
        // idle lanes and the quads' fourth lanes carry zeros
      } else {
        const double tf = dt * dt * 0.5 * mt.inv_mass;
        double nf = s_ft[m][a] * tf;
        nf = nf - S[1] * (nc * 0.5);
        const double d = nf - S[2];
        if (rebuild) cref = S[0];  // the rows of this step were built here
        S[0] = S[0] + kG5_0 * d;
        S[1] = S[1] + kG5_1 * d;
        S[2] = nf;
        S[3] = S[3] + kG5_3 * d;
        S[4] = S[4] + kG5_4 * d;
        S[5] = S[5] + kG5_5 * d;
      }
      if (lane < 16 && a < 3) s_v[m][a] = S[1];
    } else {
      // rigid_collectforce's body-frame torque with the rotation matrix of
      // the predicted orientation
      const double qa = X[0], qb = X[1], qc = X[2], qd = X[3];
      double t[3];  // column a
      if (a == 0) {
        t[0] = (qa * qa + qb * qb - (qc * qc + qd * qd));
        t[1] = 2.0 * (qa * qd - qb * qc);
        t[2] = 2.0 * (qa * qc + qb * qd);
      } else if (a == 1) {
        t[0] = -2.0 * (qa * qd + qb * qc);
        t[1] = qa * qa + qc * qc - (qb * qb + qd * qd);
        t[2] = 2.0 * (qa * qb - qc * qd);
      } else {
        t[0] = 2.0 * (qb * qd - qa * qc);
        t[1] = -2.0 * (qa * qb + qc * qd);
        t[2] = qa * qa + qd * qd - (qb * qb + qc * qc);
      }
      const double tq = t[0] * s_ft[m][3] + t[1] * s_ft[m][4] + t[2] * s_ft[m][5];
      const double di = a == 0 ? mt.Iyy - mt.Izz : a == 1 ? mt.Izz - mt.Ixx : mt.Ixx - mt.Iyy;
      const double ii = a == 0 ? mt.inv_ixx : a == 1 ? mt.inv_iyy : mt.inv_izz;
      const double w1 = dpp_d<0xC9>(S[0]);  // lanes a + 1 and a + 2 of the three
      const double w2 = dpp_d<0xD2>(S[0]);
      if (ok && a < 3) {
        double nf = (tq + di * w1 * w2) * dt * ii;
        nf = nf - S[0] * nc;
        const double d = nf - S[1];
        S[0] = S[0] + kG4_0 * d;
        S[1] = nf;
        S[2] = S[2] + kG4_2 * d;
        S[3] = S[3] + kG4_3 * d;
        S[4] = S[4] + kG4_4 * d;
      }
      if (lane < 16 && a < 3)
#pragma unroll
        for (int k = 0; k < 4; k++) s_W[m][3 * k + a] = S[k];
    }
  } else {
    block_sum(s_dyn, reg_bytes, 4 * (wid - 2) + (lane >> 4), lane & 15, part);
  }
  // quaternion corrector of level 0 (with the uncorrected w).  Component a
  // of a product with (wx, wy, wz) is -+wx q(a^1) -+ wy q(a^2) -+ wz q(a^3)
  const double sx = (a & 1) ? 1.0 : -1.0, sy = (a == 0 || a == 3) ? 1.0 : -1.0,
               sz = a >= 2 ? 1.0 : -1.0;
  auto turn3 = [](double wx, double wy, double wz, double q1, double q2, double q3) {
    return wx * q1 + wy * q2 + wz * q3;
  };
  if (wid == 2) {
    const double nw = turn3(sx * X[0], sy * X[1], sz * X[2], dpp_d<0xB1>(S[0]), dpp_d<0x4E>(S[0]),
                            dpp_d<0x1B>(S[0])) * dt * 0.5;
    S[0] = S[0] + kG4_0 * (nw - S[1]);
  }
  __syncthreads();

  if (wid == 0) {
    if (!st.last && ok && a < 3) {
      S[0] = S[0] + S[1] + S[2] + S[3] + S[4] + S[5];
      S[1] = S[1] + 2.0 * S[2] + 3.0 * S[3] + 4.0 * S[4] + 5.0 * S[5];
      S[2] = S[2] + 3.0 * S[3] + 6.0 * S[4] + 10.0 * S[5];
      S[3] = S[3] + 4.0 * S[4] + 10.0 * S[5];
      S[4] = S[4] + 5.0 * S[5];
    }
    if (ok && a < 3)
#pragma unroll
      for (int k = 0; k < 6; k++) com[(size_t)(3 * k + a) * n + i] = S[k];
    if (!st.last) {
      const bool scan = b.scan != 0;
      const int nl = st.list == 2 ? 0 : st.list + 1;  // the next step's list
      if (ok && a < 3) {
        rec[(size_t)i * rs + a] = S[0];
        if (scan) b.comp[(3 * (1 - par) + a) * n + i] = S[0];
      }
      if (!scan) {
        const int e = BOX == kBoxCube ? 0 : ax;
        const double L = g.L[e], invL = g.invL[e], ci = g.cellinv[e];
        const int nda = g.nd[e];
        double d = S[0];
        const double os = round(d * invL) * L;
        d = d - os;
        int j = (int)round(d * ci);
        if (j < 0) j += nda;
        j = ((j % nda) + nda) % nda;
        const int j0 = __builtin_amdgcn_mov_dpp(j, 0x00, 0xF, 0xF, false);
        const int j1 = __builtin_amdgcn_mov_dpp(j, 0x55, 0xF, 0xF, false);
        const int j2 = __builtin_amdgcn_mov_dpp(j, 0xAA, 0xF, 0xF, false);
        if (ok && a == 0) {
          const int c = (j2 * g.nd[BOX == kBoxCube ? 0 : 1] + j1) * g.nd[0] + j0;
          b.cell[i] = c;
          const int cap = b.cell_cap;
          int *cr = b.cellres + ((size_t)nl * g.ncell + c) * cap;
          const int slot = atomicAdd(cr, 1) + 1;
          if (slot < cap)
            cr[slot] = i;
          else
            raise_flag(b.flags, 3);  // cell capacity exceeded
        }
      }
      const double h2 = b.half_skin2;
      if (h2 > 0.0) {
        const double e = S[0] - cref, ee = e * e;
        const double e0 = quad_d<0>(ee), e1 = quad_d<1>(ee), e2 = quad_d<2>(ee);
        if (ok && a == 0 && e0 + e1 + e2 > h2) b.flags[2 + nl] = 1;
      } else if (ok && a == 0 && i == 0) {
        b.flags[2 + nl] = 1;  // no skin: the reference rebuilds every step
      }
    }
  } else if (wid == 1) {
    if (!st.last && ok && a < 3) {
      S[0] = S[0] + S[1] + S[2] + S[3] + S[4];
      S[1] = S[1] + 2.0 * S[2] + 3.0 * S[3] + 4.0 * S[4];
      S[2] = S[2] + 3.0 * S[3] + 6.0 * S[4];
      S[3] = S[3] + 4.0 * S[4];
    }
    if (ok && a < 3)
#pragma unroll
      for (int k = 0; k < 5; k++) com[(size_t)(kRowW + 3 * k + a) * n + i] = S[k];
    // the last two energy and virial sums (rows of 16 lanes) and the counts
    if (lane < 32) block_sum(s_dyn, reg_bytes, 8 + (lane >> 4), lane & 15, part);
    else if (lane < 34) {
      const int q = lane - 32;
      part[10 + q] = 0.5 * (s_cnt[0][q] + s_cnt[1][q] + s_cnt[2][q] + s_cnt[3][q]);
    }
  } else if (wid == 2) {
    // quaternion derivatives from the corrected w: level k + 1 of component
    // a from the lower levels' partner components
    double w1[3], w2[3], w3[3], w4[3];
    {
      const double sg[3] = {sx, sy, sz};
#pragma unroll
      for (int c = 0; c < 3; c++) {
        w1[c] = sg[c] * s_W[m][c];
        w2[c] = sg[c] * s_W[m][3 + c];
        w3[c] = sg[c] * s_W[m][6 + c];
        w4[c] = sg[c] * s_W[m][9 + c];
      }
    }
    const double q1 = dpp_d<0xB1>(S[0]), q2 = dpp_d<0x4E>(S[0]), q3 = dpp_d<0x1B>(S[0]);
    const double p = (w1[0] * q1 + w1[1] * q2 + w1[2] * q3) * dt * 0.5;
    const double p1 = dpp_d<0xB1>(p), p2 = dpp_d<0x4E>(p), p3 = dpp_d<0x1B>(p);
    const double r = (w2[0] * q1 + w2[1] * q2 + w2[2] * q3 + w1[0] * p1 + w1[1] * p2 + w1[2] * p3) *
                     dt * 0.25;
    const double r1 = dpp_d<0xB1>(r), r2 = dpp_d<0x4E>(r), r3 = dpp_d<0x1B>(r);
    const double s = (w3[0] * q1 + w3[1] * q2 + w3[2] * q3 + w1[0] * r1 + w1[1] * r2 + w1[2] * r3 +
                      w2[0] * p1 + w2[1] * p2 + w2[2] * p3) * dt * (1.0 / 6.0);
    const double s1 = dpp_d<0xB1>(s), s2 = dpp_d<0x4E>(s), s3 = dpp_d<0x1B>(s);
    const double u = (w4[0] * q1 + w4[1] * q2 + w4[2] * q3 + w3[0] * p1 + w3[1] * p2 + w3[2] * p3 +
                      w2[0] * r1 + w2[1] * r2 + w2[2] * r3 + w1[0] * s1 + w1[1] * s2 + w1[2] * s3) *
                     dt * (1.0 / 8.0);
    S[1] = p;
    S[2] = r;
    S[3] = s;
    S[4] = u;
    if (!st.last) {
      S[0] = S[0] + S[1] + S[2] + S[3] + S[4];
      S[1] = S[1] + 2.0 * S[2] + 3.0 * S[3] + 4.0 * S[4];
      double qa = quad_d<0>(S[0]), qb = quad_d<1>(S[0]), qc = quad_d<2>(S[0]),
             qd = quad_d<3>(S[0]);
      const double re = 1.0 / sqrt(qa * qa + qb * qb + qc * qc + qd * qd);
      qa = qa * re;
      qb = qb * re;
      qc = qc * re;
      qd = qd * re;
      S[0] = S[0] * re;
      double t[9];
      t[0] = (qa * qa + qb * qb - (qc * qc + qd * qd));
      t[1] = -2.0 * (qa * qd + qb * qc);
      t[2] = 2.0 * (qb * qd - qa * qc);
      t[3] = 2.0 * (qa * qd - qb * qc);
      t[4] = qa * qa + qc * qc - (qb * qb + qd * qd);
      t[5] = -2.0 * (qa * qb + qc * qd);
      t[6] = 2.0 * (qa * qc + qb * qd);
      t[7] = 2.0 * (qa * qb - qc * qd);
      t[8] = qa * qa + qd * qd - (qb * qb + qc * qc);
      // lane a places sites a and a + 4
      const int nq = mt.nsite - 1;
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const int q = 4 * k + a;
        if (!ok || q >= nq) continue;
        const double bx = mt.bx[q], by = mt.by[q], bz = mt.bz[q];
        const double r0 = t[0] * bx + t[1] * by + t[2] * bz;
        const double r1 = t[3] * bx + t[4] * by + t[5] * bz;
        const double r2 = t[6] * bx + t[7] * by + t[8] * bz;
        double *ri = rec + (size_t)i * rs + 4;
        if (sizeof(R) == 4) {
          float *rf = reinterpret_cast<float *>(ri) + 3 * q;
          rf[0] = (float)r0;
          rf[1] = (float)r1;
          rf[2] = (float)r2;
        } else {
          ri[3 * q] = r0;
          ri[3 * q + 1] = r1;
          ri[3 * q + 2] = r2;
        }
      }
    }
    if (ok)
#pragma unroll
      for (int k = 0; k < 5; k++) com[(size_t)(kRowQ + 4 * k + a) * n + i] = S[k];
  } else {
    // kinetic partials of the block: lane (q, molecule) one term of quantity
    // q (Rigid_Ek and Rigid_PressureTensor sums, as md_pre_body's), summed
    // over the quad; then the block's kinetic energy
    const int q = lane >> 2;
    double e = 0.0;
    if (q == 0) e = s_v[a][0] * s_v[a][0] + s_v[a][1] * s_v[a][1] + s_v[a][2] * s_v[a][2];
    else if (q < 4) e = s_W[a][q - 1] * s_W[a][q - 1];
    else if (q < kEkLen) {
      const int l = q < 7 ? 0 : q < 9 ? 1 : 2;  // xx xy xz yy yz zz
      const int h = q < 7 ? q - 4 : q < 9 ? q - 6 : 2;
      e = s_v[a][l] * s_v[a][h];
    }
    e = quad_sum_d(e);
    const size_t grp = (size_t)par * nblk + blk;
    if (a == 0 && q < kEkLen) b.stepek[grp * kEkLen + q] = e;
    const double et = __shfl(e, 0, 64), ex = __shfl(e, 4, 64), ey = __shfl(e, 8, 64),
                 ez = __shfl(e, 12, 64);
    if (lane == 0) b.stepkin[grp] = kin_energy(mt, dt, et, ex, ey, ez);
  }
}

// The force phase of a step whose corrector is a kernel of its own; block 0
// closes the previous step while the other blocks run the rows (ca.mode != 0).
template <int M, typename R, int BOX>
__global__ __launch_bounds__(256, (main_waves_per_eu<M, R>())) void k_md_main(ModelTable mt, Geom g,
                                                                            MdBuf b, PairK<R> pk,
                                                                            double *out, int parity,
                                                                            CloseArgs ca,
                                                                            int reg_bytes) {
  const int close = ca.mode != 0;
  if (close && blockIdx.x == 0) {
    __shared__ double s_close[4][kRed];
    close_body<false, false>(mt, b, g.n, g.ncell, box_volume(g.L), ca, s_close);
    return;
  }
  md_main_body<M, R, BOX>(g, b, pk, out, parity, reg_bytes, blockIdx.x - close, gridDim.x - close);
}

// Workgroups are dealt to the eight XCDs round-robin by index.  The index-th
// of nblk workgroups takes this block of four molecules: those of one XCD a
// contiguous run, so the cache lines of the state arrays (16 molecules of one
// component) and the records that near molecules share stay in one XCD's L2.
__device__ inline int xcd_run(int index, int nblk) {
  const int q = nblk >> 3, r = nblk & 7, x = index & 7, p = index >> 3;
  return x < r ? x * (q + 1) + p : r * (q + 1) + (x - r) * q + p;
}

template <int M, typename R, int BOX>
__global__ __launch_bounds__(256, (main_waves_per_eu<M, R>())) void k_md_step(
    ModelTable mt, Geom g, MdBuf b, PairK<R> pk, StepArgs st, CloseArgs ca, int reg_bytes) {
  // block 0 closes the previous step while the other blocks step
  const int close = ca.mode != 0;
  if (close && blockIdx.x == 0) {
    __shared__ double s_close[4][kRed];
    close_body<false, false>(mt, b, g.n, g.ncell, box_volume(g.L), ca, s_close);
    return;
  }
  const int nblk = gridDim.x - close;
  md_step_body<M, R, BOX>(mt, g, b, pk, st, reg_bytes, xcd_run(blockIdx.x - close, nblk), nblk);
}

// Ladder forms (map as k_md_pre_lad; the block of index -1 of each system
// closes that system's previous step).
// Arguments of the close in or around step q of a call of k steps: the pair
// and kinetic partials of the step before, the thermostat state from its half
// into this step's, and the list after next cleared.
__device__ __host__ inline CloseArgs step_close_args(const MdBuf &b, int nose_active, int nblk,
                                                     double dt, int mode, int parity, int list) {
  CloseArgs ca;
  ca.mode = mode;
  ca.nose_active = nose_active;
  ca.ngrp = ca.nblk_main = nblk;
  ca.dt = dt;
  ca.bpart = b.blockpart + (size_t)(1 - parity) * nblk * kBP;
  ca.ek = b.stepek + (size_t)(1 - parity) * nblk * kEkLen;
  ca.fine = 1;
  ca.kin = b.stepkin + (size_t)(1 - parity) * nblk;
  ca.nose_in = b.nose + 9 * (1 - parity);
  ca.nose_out = b.nose + 9 * parity;
  ca.clear = 1 << ((list + 2) % 3);
  return ca;
}
// the closes before the first step (mode 2: the thermostat state of the call's
// start, predicted into the first step's half; lists 1 and 2 cleared) and
// after the last (mode 1: the last step has parity 0; every list cleared)
__device__ __host__ inline CloseArgs step_end_args(const MdBuf &b, int nose_active, int nblk,
                                                   double dt, int mode, int k) {
  CloseArgs ca = step_close_args(b, nose_active, nblk, dt, mode, 1, 0);
  ca.nose_in = b.nose;
  ca.nose_out = b.nose + (mode == 2 ? 9 * ((k - 1) & 1) : 0);
  ca.clear = mode == 2 ? 6 : 7;
  return ca;
}

// the close of a step whose corrector was k_md_pre: the pair partials of
// src_parity, the kinetic partials and the thermostat state in the first halves
__device__ __host__ inline CloseArgs pre_close_args(const MdBuf &b, int n, int nose_active,
                                                    int nblk, double dt, int mode, int clear,
                                                    int src_parity) {
  CloseArgs ca;
  ca.mode = mode;
  ca.nose_active = nose_active;
  ca.ngrp = (n + 3) / 4;
  ca.nblk_main = nblk;
  ca.dt = dt;
  ca.bpart = b.blockpart + (size_t)src_parity * nblk * kBP;
  ca.ek = b.stepek;
  ca.fine = 0;
  ca.kin = b.stepkin;
  ca.nose_in = ca.nose_out = b.nose;
  ca.clear = clear;
  return ca;
}

template <int M, typename R>
__global__ __launch_bounds__(256, (main_waves_per_eu<M, R>())) void k_md_main_lad(
    ModelTable mt, const MdRep *__restrict__ reps, const int2 *__restrict__ map, PairK<R> pk,
    int parity, int close_mode, int reg_bytes) {
  const int2 m = map[blockIdx.x];
  if (m.x < 0) return;
  const Geom g = reps[m.x].g;
  const MdBuf b = reps[m.x].b;
  const int nm = reps[m.x].nblk_main;
  if (m.y < 0) {
    if (close_mode) {
      __shared__ double s_close[4][kRed];
      const CloseArgs ca = pre_close_args(b, g.n, reps[m.x].nose_active, nm, reps[m.x].dt,
                                          close_mode, 1 << (1 - parity), 1 - parity);
      close_body<false, false>(mt, b, g.n, g.ncell, box_volume(g.L), ca, s_close);
    }
    return;
  }
  md_main_body<M, R, kBoxCube>(g, b, pk, nullptr, parity, reg_bytes, m.y, nm);
}

template <int M, typename R>
__global__ __launch_bounds__(256, (main_waves_per_eu<M, R>())) void k_md_step_lad(
    ModelTable mt, const MdRep *__restrict__ reps, const int2 *__restrict__ map, PairK<R> pk,
    StepArgs st, int reg_bytes) {
  const int2 m = map[blockIdx.x];
  if (m.x < 0) return;
  const Geom g = reps[m.x].g;
  const MdBuf b = reps[m.x].b;
  const int nm = reps[m.x].nblk_main;
  StepArgs s1 = st;
  s1.nose_active = reps[m.x].nose_active;
  s1.dt = reps[m.x].dt;
  if (m.y < 0) {
    if (!st.first) {
      __shared__ double s_close[4][kRed];
      const CloseArgs ca = step_close_args(b, s1.nose_active, nm, s1.dt, 1 | 2, st.parity, st.list);
      close_body<false, false>(mt, b, g.n, g.ncell, box_volume(g.L), ca, s_close);
    }
    return;
  }
  md_step_body<M, R, kBoxCube>(mt, g, b, pk, s1, reg_bytes, m.y, nm);
}

// block r closes system r before (mode 2) or after (mode 1) the k steps of a
// call; one: they run as step kernels
__global__ __launch_bounds__(1024) void k_md_close_lad(ModelTable mt,
                                                       const MdRep *__restrict__ reps, int mode,
                                                       int k, int one) {
  __shared__ double s_red[4][kRed];
  const MdRep &r = reps[blockIdx.x];
  const MdBuf b = r.b;
  const CloseArgs ca =
      one ? step_end_args(b, r.nose_active, r.nblk_main, r.dt, mode, k)
          : pre_close_args(b, r.g.n, r.nose_active, r.nblk_main, r.dt, mode, mode == 2 ? 2 : 7,
                           (k - 1) & 1);
  close_body<false, true>(mt, b, r.g.n, r.g.ncell, box_volume(r.g.L), ca, s_red);
}

__global__ void k_flag_set(int *flags, int k, int v) {
  if (threadIdx.x == 0) flags[k] = v;
}

void md_launch_flag(System &s, int k, int v) { k_flag_set<<<1, 64, 0, s.stream>>>(s.md.flags, k, v); }

void md_launch_pre(System &s, bool correct, bool predict, bool sites, int list, int half) {
  const int nb = pre_blocks(s.n), na = s.nose_active ? 1 : 0;
  const int co = correct ? 1 : 0, pr = predict ? 1 : 0, si = sites ? 1 : 0;
  auto launch = [&](auto kern) {
    kern<<<nb, 256, 0, s.stream>>>(s.mt, s.geo_md, s.md, s.dt, na, co, pr, si, list, half);
  };
  if (s.andersen) launch(k_md_pre<kBoxBaro>);
  else if (is_cubic(s)) launch(k_md_pre<kBoxCube>);
  else launch(k_md_pre<kBoxOrtho>);
}

static CloseArgs close_args(System &s, int mode, int clear, int src_parity) {
  return pre_close_args(s.md, s.n, s.nose_active ? 1 : 0, s.nblk_md, s.dt, mode, clear, src_parity);
}

static void launch_close(System &s, const CloseArgs &ca) {
  auto launch = [&](auto kern) {
    kern<<<1, 1024, 0, s.stream>>>(s.mt, s.md, s.n, s.geo_md.ncell, box_volume(s.Lb), ca);
  };
  if (s.andersen) launch(k_md_close<true>);
  else launch(k_md_close<false>);
}

void md_launch_close(System &s, int mode, int clear, int src_parity) {
  launch_close(s, close_args(s, mode, clear, src_parity));
}

template <typename R>
static const PairK<R> &pair_k(const System &s);
template <>
const PairK<float> &pair_k<float>(const System &s) { return s.pkf; }
template <>
const PairK<double> &pair_k<double>(const System &s) { return s.pkd; }

// calls f with the pair-kernel layout and the pair precision of a system
// (or ladder) as std::integral_constant and a value of the type
template <class F>
static void with_model(int kmodel, int prec, F &&f) {
  auto pr = [&](auto m) {
    if (prec == G6_FP32) f(m, 0.0f);
    else f(m, 0.0);
  };
  if (kmodel == G6_TIP4P) pr(std::integral_constant<int, G6_TIP4P>());
  else if (kmodel == G6_TIP5P) pr(std::integral_constant<int, G6_TIP5P>());
  else if (kmodel == G6_SPCE) pr(std::integral_constant<int, G6_SPCE>());
  else if (kmodel == G6_NVDE) pr(std::integral_constant<int, G6_NVDE>());
  else if (kmodel == G6_OPLSMEOH) pr(std::integral_constant<int, G6_OPLSMEOH>());
  else pr(std::integral_constant<int, G6_ST2>());
}

void md_launch_main(System &s, double *out, int parity, int close_mode) {
  const CloseArgs ca =
      close_args(s, close_mode, close_mode ? 1 << (1 - parity) : 0, 1 - parity);
  if (s.tiles) {
    md_launch_tile(s, parity, ca);
    if (out) md_launch_part_reduce(s, out);
    return;
  }
  with_model(s.kmodel, s.prec, [&](auto mm, auto rr) {
    constexpr int M = decltype(mm)::value;
    using R = decltype(rr);
    const int rb = main_region_bytes(s.md.maxnb, (int)sizeof(R));
    auto launch = [&](auto kern) {
      kern<<<s.nblk_md + (ca.mode ? 1 : 0), 256, 4 * (size_t)rb, s.stream>>>(
          s.mt, s.geo_md, s.md, pair_k<R>(s), out, parity, ca, rb);
    };
    if (s.andersen) launch(k_md_main<M, R, kBoxBaro>);
    else if (is_cubic(s)) launch(k_md_main<M, R, kBoxCube>);
    else launch(k_md_main<M, R, kBoxOrtho>);
  });
}

// step q of k has parity (k - 1 - q) mod 2: the last one leaves its records,
// partials and thermostat state in the first halves
static StepArgs step_args(int q, int k) {
  StepArgs st{};
  st.parity = (k - 1 - q) & 1;
  st.list = q % 3;
  st.first = q == 0;
  st.last = q == k - 1;
  return st;
}

void md_launch_step(System &s, int q, int k) {
  StepArgs st = step_args(q, k);
  st.nose_active = s.nose_active ? 1 : 0;
  st.dt = s.dt;
  const CloseArgs ca = step_close_args(s.md, st.nose_active, s.nblk_md, s.dt, q > 0 ? 1 | 2 : 0,
                                       st.parity, st.list);
  with_model(s.kmodel, s.prec, [&](auto mm, auto rr) {
    constexpr int M = decltype(mm)::value;
    using R = decltype(rr);
    const int rb = main_region_bytes(s.md.maxnb, (int)sizeof(R));
    auto launch = [&](auto kern) {
      kern<<<s.nblk_md + (ca.mode ? 1 : 0), 256, 4 * (size_t)rb, s.stream>>>(
          s.mt, s.geo_md, s.md, pair_k<R>(s), st, ca, rb);
    };
    if (is_cubic(s)) launch(k_md_step<M, R, kBoxCube>);
    else launch(k_md_step<M, R, kBoxOrtho>);
  });
}

void md_launch_step_close(System &s, int mode, int k) {
  launch_close(s, step_end_args(s.md, s.nose_active ? 1 : 0, s.nblk_md, s.dt, mode, k));
}

void md_launch_pre_lad(Ladder &l, bool correct, bool predict, int list, int half) {
  k_md_pre_lad<<<l.grid_pre, 256, 0, l.stream>>>(l.mt, l.reps, l.map_pre, correct ? 1 : 0,
                                                 predict ? 1 : 0, list, half);
}

void md_launch_close_lad(Ladder &l, int mode, int k) {
  k_md_close_lad<<<(int)l.sys.size(), 1024, 0, l.stream>>>(l.mt, l.reps, mode, k,
                                                          l.one_kernel ? 1 : 0);
}

template <typename R>
static const PairK<R> &pair_k(const Ladder &l);
template <>
const PairK<float> &pair_k<float>(const Ladder &l) { return l.pkf; }
template <>
const PairK<double> &pair_k<double>(const Ladder &l) { return l.pkd; }

void md_launch_step_lad(Ladder &l, int q, int k) {
  const StepArgs st = step_args(q, k);
  with_model(l.model, l.prec, [&](auto mm, auto rr) {
    constexpr int M = decltype(mm)::value;
    using R = decltype(rr);
    k_md_step_lad<M, R><<<l.grid_main, 256, 4 * (size_t)l.reg_bytes, l.stream>>>(
        l.mt, l.reps, l.map_main, pair_k<R>(l), st, l.reg_bytes);
  });
}

void md_launch_main_lad(Ladder &l, int parity, int close_mode) {
  with_model(l.model, l.prec, [&](auto mm, auto rr) {
    constexpr int M = decltype(mm)::value;
    using R = decltype(rr);
    k_md_main_lad<M, R><<<l.grid_main, 256, 4 * (size_t)l.reg_bytes, l.stream>>>(
        l.mt, l.reps, l.map_main, pair_k<R>(l), parity, close_mode, l.reg_bytes);
  });
}

}  // namespace g6
