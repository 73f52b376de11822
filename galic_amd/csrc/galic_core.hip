// galic_core.hip -- the plain FP64 path on gfx950: orbit integration with
// binning, the incremental merit with accept/reject, commit and global fit.
//
// Built with -ffp-contract=off: every a*b+c rounds twice, as in the reference's
// x86-64 build, so results agree with the reference to rounding.
//
// Kernels and the reference code they replace:
//   k_orbit64        produce_orbit_response_field_mod   orbit_response.c:155-491
//   k_inst_init      calc_disp_components + add_to_energy_grid in
//                    calc_all_response_fields           main.c:226-229
//   k_eval_apply64   eval_fit_mod x2 + accept + deltas  main.c:460-505, 1021-1217
//   k_commit         commit_updates                     main.c:808-841
//   k_fit_stacks     calc_global_fit: Allreduce+smooth  main.c:256-292
//   k_fit_sums       calc_global_fit: merit sums        main.c:294-359
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "galic_ctx.h"
#include "galic_kernels.h"
#include "galic_merit.h"

namespace galic {

// ------------------------------------------------------------------ orbits --

// Four lanes integrate one orbit.  A launch has far fewer orbits than the GPU has lanes (a rep's
// trials, a batch of single orbits), so its time is the longest orbit's chain of steps, and a
// step's latency is mostly the length of its instruction stream: about 1100 FP64 instructions
// with one lane per orbit, 600 with four.  The lanes of a quad hold the same state bit for bit
// and share the step's independent pieces, one each: the three square roots, the four log
// indices (R and z on the force and the density grid, with their divisions), the divisions of
// the force and of the velocity components, the four table taps and the four cells of a binning
// event.  Every value is formed by the operations, in the order, of the lookups in
// galic_device.h, so the results do not depend on the split.  Measured against one lane per
// orbit: a single orbit's step 2.5 -> 1.5 us; 6000 orbits on 64^2 grids 32 -> 16 ms; the initial
// pass of 2e4 particles 35 -> 22 ms, of 2e5 (bound by the atomics on the Loc grids) 217 -> 138 ms.

// Lane k's value in all four lanes of the quad.
template <int K>
__device__ __forceinline__ double quad_get(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), K * 0x55, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), K * 0x55, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ int quad_first(int v) { return __builtin_amdgcn_mov_dpp(v, 0, 0xF, 0xF, true); }

// Register-resident accumulator of the lane's cell of the 2x2 block (lane bit 0: R + 1, bit 1:
// z + 1) for consecutive binning events that hit the same block: flushed to memory only when
// the block changes.
struct Run64 {
  int quad;  // iz*Nbin + iR of the lower-left cell, -1 when empty
  double w[kFields];
};

// Adds a run to the orbit's private slot (trial evaluation; cell-major: a cell's 5 fields are
// contiguous) or to the Loc grid of the particle's type (initial response pass).  Atomics without
// return in both: the slot belongs to one orbit, but a load, add and store would make the wave
// wait for memory at every flush.
__device__ __forceinline__ void run_flush(const Run64 &r, int q, int nb, int ngrid, double fac, double *slot,
                                          double *loc) {
  if(r.quad < 0) return;
  const int c = r.quad + (q & 1) + (q >> 1) * nb;
  if(slot) {
    double *s = slot + (size_t)c * kFields;
#pragma unroll
    for(int f = 0; f < kFields; f++) atomicAdd(&s[f], fac * r.w[f]);
  } else {
#pragma unroll
    for(int f = 0; f < kFields; f++) atomicAdd(&loc[(size_t)f * ngrid + c], fac * r.w[f]);
  }
}

// Starts an empty run in the block of cell (iR, iz).
__device__ __forceinline__ void run_start(Run64 &r, int nb, int iR, int iz, int4 &bb) {
  r.quad = iz * nb + iR;
#pragma unroll
  for(int f = 0; f < kFields; f++) r.w[f] = 0;
  bb.x = min(bb.x, iR);
  bb.y = max(bb.y, iR + 1);
  bb.z = min(bb.z, iz);
  bb.w = max(bb.w, iz + 1);
}

// One binning event in the run's block: trapezoid half weights (orbit_response.c:277-319).
__device__ __forceinline__ void bin_event64(Run64 &r, int q, double fR, double fz, double dt, double vr2, double vt2,
                                            double vq2, double vp2) {
  const double m = 0.5 * dt * ((q & 1) ? fR : 1 - fR) * ((q & 2) ? fz : 1 - fz);
  r.w[F_M] += m;
  r.w[F_R] += m * vr2;
  r.w[F_T] += m * vt2;
  r.w[F_Q] += m * vq2;
  r.w[F_P] += m * vp2;
}

// Persistent quads: qpw quads of each wave take orbits from the launch's counter, the next one
// when their orbit ends, so orbits of different length keep the wave busy.  A freshly taken orbit
// spends one pass of the loop on the lookups at its start point.  Every quad leaves once the
// counter passes the orbit count.
__global__ void __launch_bounds__(64) k_orbit64(DevModel M, OrbitArgs A, int qpw) {
  const int lane = threadIdx.x, q = lane & 3;
  if((lane >> 2) >= qpw) return;
  const int nb = M.DG_Nbin, ngrid = nb * nb, fb = M.FG_Nbin;
  const bool odd = q & 1, upper = q & 2;
  // the lane's constants: log index (lanes 0, 1 the force grid, 2, 3 the density grid), force term
  // (lane 2 the halo, 3 the bulge) and timestep limit (odd lanes the orbital one)
  const double l_rmin = upper ? M.DG_Rmin : M.FG_Rmin, l_lf = upper ? M.DG_logFac : M.FG_logFac;
  const double l_off = upper ? 0.5 : 0.0, l_fac = odd ? M.fo : M.fc;
  const double l_GM = odd ? M.G * M.Bulge_Mass : M.G * M.Halo_Mass;
  const double l_a = odd ? M.Bulge_A : M.Halo_A, l_eps = 1.0e-6 * l_a;

  int o = 0, type = 0, tovs = 0;
  double x = 0, y = 0, z = 0, vx = 0, vy = 0, vz = 0, timespan = 0, fac = 0;
  double ax = 0, ay = 0, az = 0, cellsize = 0, fR = 0, fz = 0, E0 = 0;
  double vr2 = 0, vt2 = 0, vq2 = 0, vp2 = 0, tall = 0, radsign_previous = 0, dt = 0;
  double *slot = nullptr, *loc = nullptr;
  int iR = 0, iz = 0, norbit = 0, flag = 0, status = 0;
  long long steps = 0;
  Run64 run;
  run.quad = -1;
  int4 bb = make_int4(nb, -1, nb, -1);
  bool take = true, fresh = false, streams = false;
  while(true) {
    if(take) {
      int t = 0;
      if(q == 0) t = (int)atomicAdd(A.counter, 1u);
      o = quad_first(t);
      if(o >= A.n) break;
      if(A.order) o = A.order[o];
      type = A.otype[o];
      tovs = M.tovs[type];
      streams = (A.vstream_nz >> type) & 1u;
      x = A.ox[o]; y = A.oy[o]; z = A.oz[o];
      vx = A.ovx[o]; vy = A.ovy[o]; vz = A.ovz[o];
      timespan = A.otint[o];
      fac = A.omass[o] / timespan;  // mass/t with t == timespan at the end (see tall)
      slot = A.slots ? A.slots + (size_t)(o - A.slot_base) * A.slot_stride : nullptr;
      loc = A.loc ? A.loc + (size_t)type * kFields * ngrid : nullptr;
      E0 = 0.5 * (vx * vx + vy * vy + vz * vz) + potential64(M, x, y, z);
      run.quad = -1;
      bb = make_int4(nb, -1, nb, -1);
      tall = radsign_previous = 0;
      norbit = flag = status = 0;
      steps = 0;
      take = false;
      fresh = true;
    }
    if(!fresh) {
      // get_timestep (orbit_response.c:16-26), with the cell of the previous position
      const double v2 = vx * vx + vy * vy + vz * vz, a2 = ax * ax + ay * ay + az * az;
      const double tl = l_fac * ((odd ? M.V200 : cellsize) / sqrt(odd ? a2 : v2));
      const double t1 = quad_get<1>(tl), t2 = quad_get<0>(tl);
      dt = (t1 < t2) ? t1 : t2;
      if(timespan < dt + tall) {
        dt = timespan - tall;
        flag = 1;
      }
      if(!(dt >= 0 && dt <= timespan)) {  // NaN state: stop instead of running to the step cap
        status = GALIC_ERR_ARG;
      } else {
        bin_event64(run, q, fR, fz, dt, vr2, vt2, vq2, vp2);  // (in the block of the step before)
        vx += 0.5 * dt * ax;
        vy += 0.5 * dt * ay;
        vz += 0.5 * dt * az;
        x += dt * vx;
        y += dt * vy;
        z += dt * vz;
      }
    }
    if(status == 0) {
      const double R2 = x * x + y * y, r2 = x * x + y * y + z * z;
      // orbit_response.c:222-273: Q and T of the velocity decomposition
      double Q0, Q1, Q2, q2;
      if(tovs == 2) {
        Q0 = -y;
        Q1 = x;
        Q2 = 0;
        q2 = Q0 * Q0 + Q1 * Q1;
      } else {
        Q0 = y * (-1.0) - z * 0.0;
        Q1 = z * 0.0 - x * (-1.0);
        Q2 = x * 0.0 - y * 0.0;
        q2 = Q0 * Q0 + Q1 * Q1 + Q2 * Q2;
      }
      const double root = sqrt(upper ? q2 : odd ? r2 : R2);
      const double R = quad_get<0>(root), r = quad_get<1>(root), qn = quad_get<2>(root);
      const double bin = log((odd ? fabs(z) : R) / l_rmin + 1.0) / l_lf - l_off;
      const double jd = quad_get<0>(bin), id = quad_get<1>(bin);
      double br = quad_get<2>(bin), bz = quad_get<3>(bin);
      // densitygrid_get_cell (grid.c:494-534)
      if(br < 0) br = 0;
      if(bz < 0) bz = 0;
      iR = (int)br;
      fR = br - iR;
      iz = (int)bz;
      fz = bz - iz;
      if(iR >= nb - 1) {
        iR = nb - 2;
        fR = 1;
      }
      if(iz >= nb - 1) {
        iz = nb - 2;
        fz = 1;
      }
      // the lane's taps: its node of the force tables and of the streaming table, and the cell size
      const int jbin = (int)jd, ibin = (int)id;
      const double jfac = jd - jbin, ifac = id - ibin;
      const bool on = M.use_table && ibin < fb - 1 && jbin < fb - 1;
      double tR = 0, tz = 0;
      if(on) {
        const int k = (ibin + (q >> 1)) * fb + jbin + (q & 1);
        tR = M.FG_DPotDR[k];
        tz = M.FG_DPotDz[k];
      }
      // get_vstream (disp_fields.c:118-132) through forcegrid_get_cell (grid.c:15-55)
      double sR = jd < 0 ? 0 : jd, sz = id < 0 ? 0 : id;
      int jR = (int)sR, jz = (int)sz;
      double gR = sR - jR, gz = sz - jz;
      if(jR >= fb - 1) {
        jR = fb - 2;
        gR = 1;
      }
      if(jz >= fb - 1) {
        jz = fb - 2;
        gz = 1;
      }
      // (a table of zeros, as the isotropic components have, gives vstr = 0 without its load)
      const double tv = streams ? M.FG_Vstream[type][(jz + (q >> 1)) * fb + jR + (q & 1)] : 0;
      cellsize = M.DG_CellSize[iz * nb + iR];
      // forcegrid_get_acceleration (grid.c:122-197): lanes 0, 1 the direction cosines, 2, 3 the
      // closed forms of halo and bulge
      const double quot = (upper ? l_GM : odd ? y : x) / (upper ? (r + l_eps) * (r + l_a) * (r + l_a) : R);
      const double hal = quad_get<2>(quot), bul = quad_get<3>(quot);
      ax = ay = az = 0;
      if(on) {
        const double wi = upper ? ifac : 1 - ifac, wj = odd ? jfac : 1 - jfac;
        const double pR = tR * wi * wj, pz = tz * wi * wj;
        const double accR = quad_get<0>(pR) + quad_get<1>(pR) + quad_get<2>(pR) + quad_get<3>(pR);
        double accz = quad_get<0>(pz) + quad_get<1>(pz) + quad_get<2>(pz) + quad_get<3>(pz);
        if(z < 0) accz = -accz;
        const double c = quad_get<0>(quot), s = quad_get<1>(quot);
        ax = accR * (R > 0 ? c : 1.0);
        ay = accR * (R > 0 ? s : 0.0);
        az = accz;
      } else if(M.use_table) {
        ax = -hal * x * M.halo_offgrid_fac;
        ay = -hal * y * M.halo_offgrid_fac;
        az = -hal * z * M.halo_offgrid_fac;
      }
      if(M.add_halo) {
        ax += -hal * x;
        ay += -hal * y;
        az += -hal * z;
      }
      if(M.add_bulge) {
        ax += -bul * x;
        ay += -bul * y;
        az += -bul * z;
      }
      if(!fresh) {
        vx += 0.5 * dt * ax;
        vy += 0.5 * dt * ay;
        vz += 0.5 * dt * az;
      }
      // the decomposition at the end of a step is also the one at the start of the next
      double vstr = 0;
      if(streams) {
        const double pv = tv * (odd ? gR : 1 - gR) * (upper ? gz : 1 - gz);
        vstr = quad_get<0>(pv) + quad_get<2>(pv) + quad_get<1>(pv) + quad_get<3>(pv);
      }
      double num, den;
      if(tovs == 2) {
        const double v_dot_x = vx * x + vy * y, v_dot_Q = vx * Q0 + vy * Q1;
        num = odd ? v_dot_Q : v_dot_x * v_dot_x;
        den = odd ? qn : R2;
      } else {
        const double v_dot_x = vx * x + vy * y + vz * z, v_dot_Q = vx * Q0 + vy * Q1 + vz * Q2;
        const double T0 = y * Q2 - z * Q1, T1 = z * Q0 - x * Q2, T2 = x * Q1 - y * Q0;
        const double v_dot_T = vx * T0 + vy * T1 + vz * T2;
        num = upper ? v_dot_T * v_dot_T : odd ? v_dot_Q : v_dot_x * v_dot_x;
        den = upper ? T0 * T0 + T1 * T1 + T2 * T2 : odd ? qn : r2;
      }
      const double comp = num / den;
      vr2 = quad_get<0>(comp);
      vt2 = tovs == 2 ? vz * vz : quad_get<2>(comp);
      const double vq = quad_get<1>(comp);
      vq2 = vq * vq;
      vp2 = (vq - vstr) * (vq - vstr);
      if(fresh) {
        fresh = false;
        if(timespan > 0) {
          run_start(run, nb, iR, iz, bb);
          continue;
        }
        status = GALIC_ERR_ARG;  // the reference would loop until its step cap
      } else {
        if(iz * nb + iR != run.quad) {
          run_flush(run, q, nb, ngrid, fac, slot, loc);
          run_start(run, nb, iR, iz, bb);
        }
        bin_event64(run, q, fR, fz, dt, vr2, vt2, vq2, vp2);
        tall += dt;
        const double radsign = vx * x + vy * y + vz * z;
        if(radsign > 0 && radsign_previous < 0) norbit++;
        radsign_previous = radsign;
        steps++;
        if(steps > M.max_steps) status = GALIC_ERR_STEPCAP;
      }
    }
    if(flag || status) {
      if(steps > 0)
        run_flush(run, q, nb, ngrid, fac, slot, loc);
      else
        bb = make_int4(nb, -1, nb, -1);  // nothing was binned
      const double e1 = 0.5 * (vx * vx + vy * vy + vz * vz) + potential64(M, x, y, z);
      if(q == 0) {
        A.tall[o] = tall;
        A.norbit[o] = norbit;
        A.steps[o] = steps;
        A.e0[o] = E0;
        A.e1[o] = e1;
        A.bbox[o] = bb;
        A.status[o] = status;
        orbit_stats_add(A.stats, steps, status, o);
      }
      take = true;
    }
  }
}

// Expected steps of each orbit, its time span over the timestep at its start (orbit_response.c:16-26):
// the key by which a launch takes its longest orbits first.
__global__ void k_expect_steps(DevModel M, int n, const double *ox, const double *oy, const double *oz,
                               const double *ovx, const double *ovy, const double *ovz, const double *otint,
                               unsigned int *key, int *ord) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  if(o >= n) return;
  const double x = ox[o], y = oy[o], z = oz[o], vx = ovx[o], vy = ovy[o], vz = ovz[o];
  double ax, ay, az, fR, fz;
  int iR, iz;
  accel64(M, x, y, z, fg_index64(M, x, y, z), ax, ay, az);
  cell64(x, y, z, M.DG_Rmin, M.DG_logFac, M.DG_Nbin, iR, iz, fR, fz);
  const double t1 = M.fo * M.V200 / sqrt(ax * ax + ay * ay + az * az);
  const double t2 = M.fc * M.DG_CellSize[iz * M.DG_Nbin + iR] / sqrt(vx * vx + vy * vy + vz * vz);
  const double s = otint[o] / (t1 < t2 ? t1 : t2);
  key[o] = s > 0 && s < 4e9 ? (unsigned int)s : 0u;
  ord[o] = o;
}

// --------------------------------------------------- instantaneous moments --

// calc_disp_components_for_particle + add_to_energy_grid for every particle
// (main.c:226-229); atomics replace the serial accumulation.
__global__ void k_inst_init(DevModel M, Particles P, double *locI, double *locM, int ngrid) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if(n >= P.n) return;
  const int t = P.type[n];
  double x = P.x[n], y = P.y[n], z = P.z[n];
  double vr2, vt2, vp2, vq2;
  disp_components64(M, t, x, y, z, P.vx[n], P.vy[n], P.vz[n], vr2, vt2, vp2, vq2);
  P.vr2[n] = vr2;
  P.vt2[n] = vt2;
  P.vp2[n] = vp2;
  P.vq2[n] = vq2;
  int iR, iz;
  double fR, fz;
  cell64(x, y, z, M.EG_Rmin, M.EG_logFac, M.EG_Nbin, iR, iz, fR, fz);
  const int nb = M.EG_Nbin;
  const double mass = P.mass[n];
  double w[4] = {(1 - fR) * (1 - fz), (fR) * (1 - fz), (1 - fR) * (fz), (fR) * (fz)};
  int c[4] = {iz * nb + iR, iz * nb + iR + 1, (iz + 1) * nb + iR, (iz + 1) * nb + iR + 1};
  double val[4] = {vr2 * mass, vt2 * mass, vp2 * mass, vq2 * mass};
  double *li = locI + (size_t)t * 4 * ngrid;
  for(int k = 0; k < 4; k++) {
    atomicAdd(&locM[(size_t)t * ngrid + c[k]], w[k] * mass);
    for(int f = 0; f < 4; f++) atomicAdd(&li[(size_t)f * ngrid + c[k]], w[k] * val[f]);
  }
}

// ------------------------------------------------------------------- merit --

// Block-wide sum of up to 8 doubles per thread with a fixed reduction order.
template <int NV>
__device__ void block_sum(double (&v)[NV], double *lds) {
  const int tid = threadIdx.x, nt = blockDim.x;
  for(int k = 0; k < NV; k++) lds[k * nt + tid] = v[k];
  __syncthreads();
  for(int s = nt / 2; s > 0; s >>= 1) {
    if(tid < s)
      for(int k = 0; k < NV; k++) lds[k * nt + tid] += lds[k * nt + tid + s];
    __syncthreads();
  }
  for(int k = 0; k < NV; k++) v[k] = lds[k * nt];
  __syncthreads();
}

// Change of the instantaneous terms (main.c:1125-1176) when the particle's
// squared components change by mass*diff at its energy-grid cell.
__device__ double inst_delta(const DevModel &M, const double *S, const double *W, const int *cutB_of, int t,
                             double x, double y, double z, double mass, const double (&dnew)[4],
                             const double (&dold)[4], double lowdisp, int &c0, double (&cw)[4], int (&cc)[4]) {
  const int L = M.EG_L, nb = M.EG_Nbin, Nstack = GALIC_NSTACK(L);
  int iR, iz;
  double fR, fz;
  cell64(x, y, z, M.EG_Rmin, M.EG_logFac, nb, iR, iz, fR, fz);
  cw[0] = (1 - fR) * (1 - fz);
  cw[1] = (fR) * (1 - fz);
  cw[2] = (1 - fR) * (fz);
  cw[3] = (fR) * (fz);
  cc[0] = iz * nb + iR;
  cc[1] = iz * nb + iR + 1;
  cc[2] = (iz + 1) * nb + iR;
  cc[3] = (iz + 1) * nb + iR + 1;
  c0 = cc[0];
  const double *MR = S + ST_EMR * Nstack, *MT = S + ST_EMT * Nstack;
  const int stI[4] = {ST_IR, ST_IT, ST_IP, ST_IQ};
  const int stE[4] = {ST_ER, ST_ET, ST_EP, ST_EQ};
  int node[4];
  for(int k = 0; k < 4; k++) node[k] = cutB_of[cc[k]];
  double total = 0;
  const int tovs = M.tovs[t];
  for(int f = 0; f < 4; f++) {
    if(f == I_Q && (tovs == 0 || t == 2)) continue;  // main.c:1195
    double val = (dnew[f] - dold[f]) * mass;           // add_to_energy_grid scales by mass first
    const double *I = S + stI[f] * Nstack, *E = S + stE[f] * Nstack;
    for(int k = 0; k < 4; k++) {
      int nd = node[k];
      bool first = true;
      for(int j = 0; j < k; j++)
        if(node[j] == nd) first = false;
      if(!first) continue;
      double delta = 0;
      for(int j = k; j < 4; j++)
        if(node[j] == nd) delta += cw[j] * val;
      double mr = MR[nd], mt = MT[nd];
      if(mr > 0 && mt > 0) {
        double tgt = E[nd] / mt;
        double den = tgt > lowdisp ? tgt : lowdisp;
        double before = fabs(I[nd] / mr - tgt) / den;
        double after = fabs((I[nd] + delta) / mr - tgt) / den;
        total += after - before;
      }
    }
  }
  return total;
}

// One workgroup per trial.  The trial's old and new orbit responses sit in two
// private slots; the change of every orbit-averaged merit term is evaluated on
// the fixed cut of the density target (the cut nodes never change, because the
// targets are fixed): fine-level nodes inside the orbits' bounding box directly,
// coarse nodes from a pyramid of the difference built in LDS.  This equals
// F_try - F_base of main.c:464-465 up to rounding.
__global__ void __launch_bounds__(256) k_eval_apply64(DevModel M, EvalArgs A) {
  extern __shared__ double lds[];
  const int i = A.block_base + blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
  const int L = M.DG_L, nb = M.DG_Nbin, ngrid = nb * nb, Nstack = GALIC_NSTACK(L);
  const int ncoarse = (Nstack - ngrid);
  // coarse levels 0..L-1 in LDS, or in this workgroup's HBM scratch where they do not fit (levels 8, 9)
  double *cs = A.cs_global ? A.cs_global + (size_t)blockIdx.x * A.cs_stride : lds;
  double *red = A.cs_global ? lds : lds + ncoarse;  // reduction scratch, 8*nt
  __shared__ int s_accept;

  const int p = A.tidx[i];
  const int t = A.P.type[p];
  const double *S = A.stacks + (size_t)t * ST_COUNT * Nstack;
  const double *W = A.weights + (size_t)t * W_COUNT * Nstack;
  const int oo = 2 * i - A.slot_base, on = 2 * i + 1 - A.slot_base;
  const double *so = A.slots + (size_t)oo * A.slot_stride;
  const double *sn = A.slots + (size_t)on * A.slot_stride;
  const int4 bo = A.bbox[2 * i], bn = A.bbox[2 * i + 1];
  int r0 = min(bo.x, bn.x), r1 = max(bo.y, bn.y), z0 = min(bo.z, bn.z), z1 = max(bo.w, bn.w);
  if(r1 < r0 || z1 < z0) {  // no binning event (cannot happen after a successful orbit launch)
    r0 = z0 = 0;
    r1 = z1 = -1;
  }
  const int pr0 = r0 >> 1, pr1 = r1 >> 1, pz0 = z0 >> 1, pz1 = z1 >> 1;
  const int npr = (r1 < r0) ? 0 : pr1 - pr0 + 1, npz = (z1 < z0) ? 0 : pz1 - pz0 + 1;
  const int offL = GALIC_STACKOFFSET(L, 0, 0), offL1 = GALIC_STACKOFFSET(L - 1, 0, 0);

  double phi[kFields];
  const int stR[kFields] = {ST_RM, ST_RSR, ST_RST, ST_RSQ, ST_RSP};
  const int stT[kFields] = {ST_MT, ST_ER, ST_ET, ST_EQ, ST_EP};
  (void)npr; (void)npz; (void)pr0; (void)pz0; (void)offL; (void)offL1; (void)pr1; (void)pz1;
  for(int f = 0; f < kFields; f++) {
    CutTerm C;
    C.R = S + stR[f] * Nstack;
    C.T = S + stT[f] * Nstack;
    C.den = W + W_A * Nstack;
    C.ratio = (f == F_M) ? nullptr : W + (W_SR + f - 1) * Nstack;
    const double *fo = so + f, *fn = sn + f;  // cell-major slots: field f of cell c at c*5 + f
    phi[f] = cut_sum_field(C, [&](int cell) { return fn[(size_t)cell * kFields] - fo[(size_t)cell * kFields]; }, r0,
                           r1, z0, z1, L, cs);
  }
  double sums[kFields];
  for(int f = 0; f < kFields; f++) sums[f] = phi[f];
  block_sum<kFields>(sums, red);

  const double x = A.P.x[p], y = A.P.y[p], z = A.P.z[p], mass = A.P.mass[p];
  const double tvx = A.tvx[i], tvy = A.tvy[i], tvz = A.tvz[i];
  double dnew[4], dold[4] = {A.P.vr2[p], A.P.vt2[p], A.P.vp2[p], A.P.vq2[p]};
  if(tid == 0) {
    disp_components64(M, t, x, y, z, tvx, tvy, tvz, dnew[0], dnew[1], dnew[2], dnew[3]);
    const double *fit = A.fit + (size_t)t * 16;
    int c0, cc[4];
    double cw[4];
    double vinst = inst_delta(M, S, W, A.cutB_of + (size_t)t * ngrid, t, x, y, z, mass, dnew, dold, A.lowdisp,
                              c0, cw, cc);
    const double MT = A.MType[t];
    double dF = sums[F_M] / MT +
                (A.fac[t][0] * sums[F_R] + A.fac[t][1] * sums[F_T] + A.fac[t][3] * sums[F_P] +
                 A.fac[t][2] * sums[F_Q]) / MT / 4 +
                fit[5] / fit[6] * vinst;
    int acc = (dF < 0);
    A.accept[i] = acc;
    A.dF[i] = dF;
    s_accept = acc;
    const int ono = A.norbit[2 * i], onn = A.norbit[2 * i + 1];
    A.P.orbits[p] = acc ? onn : ono;
    if(acc) {
      A.P.vx[p] = tvx;
      A.P.vy[p] = tvy;
      A.P.vz[p] = tvz;
      double *lid = A.locI_d + (size_t)t * 4 * ngrid;
      for(int f = 0; f < 4; f++) {
        double val = (dnew[f] - dold[f]) * mass;
        for(int k = 0; k < 4; k++) atomicAdd(&lid[(size_t)f * ngrid + cc[k]], cw[k] * val);
      }
      A.P.vr2[p] = dnew[0];
      A.P.vt2[p] = dnew[1];
      A.P.vp2[p] = dnew[2];
      A.P.vq2[p] = dnew[3];
    }
  }
  __syncthreads();
  const int acc = s_accept;
  // deltas of accepted orbits (main.c:477-486), then clear both slots
  const int nr = (r1 < r0) ? 0 : r1 - r0 + 1, nzz = (z1 < z0) ? 0 : z1 - z0 + 1;
  double *lad = A.locA_d + (size_t)t * kFields * ngrid;
  double *wo = (double *)so, *wn = (double *)sn;
  for(int k = tid; k < nr * nzz; k += nt) {
    int cell = (z0 + k / nr) * nb + (r0 + k % nr);
    for(int f = 0; f < kFields; f++) {
      size_t o = (size_t)cell * kFields + f;
      if(acc) {
        double d = wn[o] - wo[o];
        if(d != 0) atomicAdd(&lad[(size_t)f * ngrid + cell], d);
      }
      wo[o] = 0;
      wn[o] = 0;
    }
  }
}

// ----------------------------------------------------------- commit / fit --

// commit_updates (main.c:808-841): Loc += delta, delta = 0
__global__ void k_commit(double *loc, double *delta, size_t n) {
  size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(k >= n) return;
  loc[k] += delta[k];
  delta[k] = 0;
}

// The cuts of calc_stack_difference (grid.c:1090: the recursion stops where l >= maxlevel or ref
// < thresh) and what the merit needs on them.  Positions never move and the targets are fixed, so
// the cuts are the same at every call.  A node is on a cut when it stops the recursion and none of
// its ancestors does: every node, tile and cell looks down its own path from the root, so the
// passes over the stacks (30 ms a type on the host at 512^2 cells) are a few microseconds here.
__device__ __forceinline__ int cut_level(const double *ref, double thresh, int L, int l, int i, int j) {
  for(int a = 0; a < l; a++)
    if(ref[GALIC_STACKOFFSET(a, i >> (l - a), j >> (l - a))] < thresh) return a;
  return (l >= L || ref[GALIC_STACKOFFSET(l, i, j)] < thresh) ? l : l + 1;  // (l + 1: the recursion goes on)
}

// Per node: min(dist, R200/20) and Tm/E_x on the cut of DGs_MassTarget (grid.c:1078-1084,
// 1128-1133), 1 on the cut of EGs_MassResponse.
__global__ void k_cut_weights(CutArgs A) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y, L = A.L, Ns = GALIC_NSTACK(L);
  if(o >= Ns) return;
  int l = 0;
  while(l < L && o >= GALIC_STACKOFFSET(l + 1, 0, 0)) l++;
  const int k = o - GALIC_STACKOFFSET(l, 0, 0), i = k >> l, j = k & ((1 << l) - 1);
  const double *S = A.stacks + (size_t)t * ST_COUNT * Ns;
  double *W = A.weights + (size_t)t * W_COUNT * Ns;
  double w[W_COUNT] = {0, 0, 0, 0, 0, 0};
  if(A.present[t]) {
    const double *Tm = S + ST_MT * Ns;
    if(cut_level(Tm, A.thr_d[t], L, l, i, j) == l) {
      const double d = S[ST_DIST * Ns + o];
      w[W_A] = (d < A.rlim) ? d : A.rlim;
      const int st[4] = {ST_ER, ST_ET, ST_EQ, ST_EP};
      for(int f = 0; f < 4; f++) {
        const double e = S[st[f] * Ns + o];
        w[W_SR + f] = (e > 0) ? Tm[o] / e : 0.0;
      }
    }
    if(cut_level(S + ST_EMR * Ns, A.thr_s[t], L, l, i, j) == l) w[W_B] = 1.0;
  }
  for(int f = 0; f < W_COUNT; f++) W[(size_t)f * Ns + o] = w[f];
}

// Per fine cell: its node on the cut of EGs_MassResponse.
__global__ void k_cut_cells(CutArgs A) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y, L = A.L, ng = 1 << (2 * L);
  if(c >= ng) return;
  const int i = c >> L, j = c & ((1 << L) - 1);
  int node = 0;
  if(A.present[t]) {
    const int l = cut_level(A.stacks + ((size_t)t * ST_COUNT + ST_EMR) * GALIC_NSTACK(L), A.thr_s[t], L, L, i, j);
    node = GALIC_STACKOFFSET(l, i >> (L - l), j >> (L - l));
  }
  A.cutB_of[(size_t)t * ng + c] = node;
}

// Per 16 x 16-cell tile (Morton index), the levels of its nodes on the cut of DGs_MassTarget: bit u
// for level L-u inside the tile (u = 0..4), bit 5 when the tile lies inside a cut node above its
// level.  One wave per tile.
__global__ void __launch_bounds__(64) k_cut_tiles(CutArgs A) {
  const int L = A.L, lt = L - 4, ntile = 1 << (2 * lt), m = blockIdx.x, t = blockIdx.y, lane = threadIdx.x;
  int tz = 0, tr = 0;
  for(int b = 0; b < lt; b++) {
    tr |= ((m >> (2 * b)) & 1) << b;
    tz |= ((m >> (2 * b + 1)) & 1) << b;
  }
  unsigned int bits = 0;
  if(A.present[t]) {
    const double *Tm = A.stacks + ((size_t)t * ST_COUNT + ST_MT) * GALIC_NSTACK(L);
    for(int u = 0; u <= 4; u++) {
      const int n = 16 >> u;
      bool on = false;
      for(int q = lane; q < n * n; q += 64)
        on = on || cut_level(Tm, A.thr_d[t], L, L - u, tz * n + q / n, tr * n + q % n) == L - u;
      if(__ballot(on)) bits |= 1u << u;
    }
    if(cut_level(Tm, A.thr_d[t], L, lt, tz, tr) < lt) bits |= 32u;
  }
  if(lane == 0) A.tcut[(size_t)t * ntile + m] = (unsigned char)bits;
}

// One workgroup per (type, stack): copy the fine level from a Loc grid and
// build the coarse levels as in smooth_stack (grid.c:1247-1265).
__global__ void k_fit_stacks(FitArgs A) {
  const int job = blockIdx.x;  // type*10 + k
  const int t = job / 10 + 1, k = job % 10;
  if(!A.present[t]) return;
  const int L = A.L, nb = 1 << L, ngrid = nb * nb, Nstack = GALIC_NSTACK(L);
  double *S = A.stacks + (size_t)t * ST_COUNT * Nstack;
  const int dst[10] = {ST_RM, ST_RSR, ST_RST, ST_RSQ, ST_RSP, ST_EMR, ST_IR, ST_IT, ST_IP, ST_IQ};
  double *st = S + (size_t)dst[k] * Nstack;
  const double *src;
  if(k < 5)
    src = A.locA + ((size_t)t * kFields + k) * ngrid;
  else if(k == 5)
    src = A.locM + (size_t)t * ngrid;
  else
    src = A.locI + ((size_t)t * 4 + (k - 6)) * ngrid;
  const int off = GALIC_STACKOFFSET(L, 0, 0);
  for(int c = threadIdx.x; c < ngrid; c += blockDim.x) st[off + c] = src[c];
  __syncthreads();
  for(int l = L - 1; l >= 0; l--) {
    int n = 1 << l;
    for(int q = threadIdx.x; q < n * n; q += blockDim.x) {
      int i = q / n, j = q % n;
      st[GALIC_STACKOFFSET(l, i, j)] = st[GALIC_STACKOFFSET(l + 1, 2 * i, 2 * j)] +
                                       st[GALIC_STACKOFFSET(l + 1, 2 * i + 1, 2 * j)] +
                                       st[GALIC_STACKOFFSET(l + 1, 2 * i, 2 * j + 1)] +
                                       st[GALIC_STACKOFFSET(l + 1, 2 * i + 1, 2 * j + 1)];
    }
    __syncthreads();
  }
}

// calc_global_fit's stacks for grids of 32 x 32 cells and more, in tiles: workgroup (tile,
// stack) copies the tile's 32 x 32 fine cells into the stack and forms the tile's nodes of
// levels L-1 .. L-5 in LDS, each parent the sum of its four children in smooth_stack's order
// (grid.c:1247-1265); k_fit_top then forms the levels above the tiles.  The same sums in the
// same order as k_fit_stacks, spread over many workgroups.
constexpr int FIT_TILE = 32;
__global__ void __launch_bounds__(256) k_fit_tiles(FitArgs A) {
  __shared__ double lv[2][FIT_TILE * FIT_TILE];
  const int job = blockIdx.y;  // type*10 + k
  const int t = job / 10 + 1, k = job % 10;
  if(!A.present[t]) return;
  const int L = A.L, nb = 1 << L, ngrid = nb * nb, Nstack = GALIC_NSTACK(L), ts = nb / FIT_TILE;
  const int tz = blockIdx.x / ts, tr = blockIdx.x % ts;
  double *S = A.stacks + (size_t)t * ST_COUNT * Nstack;
  const int dst[10] = {ST_RM, ST_RSR, ST_RST, ST_RSQ, ST_RSP, ST_EMR, ST_IR, ST_IT, ST_IP, ST_IQ};
  double *st = S + (size_t)dst[k] * Nstack;
  const double *src;
  if(k < 5)
    src = A.locA + ((size_t)t * kFields + k) * ngrid;
  else if(k == 5)
    src = A.locM + (size_t)t * ngrid;
  else
    src = A.locI + ((size_t)t * 4 + (k - 6)) * ngrid;
  const int off = GALIC_STACKOFFSET(L, 0, 0);
  for(int q = threadIdx.x; q < FIT_TILE * FIT_TILE; q += blockDim.x) {
    const int c = (tz * FIT_TILE + q / FIT_TILE) * nb + tr * FIT_TILE + q % FIT_TILE;
    const double v = src[c];
    st[off + c] = v;
    lv[0][q] = v;
  }
  __syncthreads();
  int cur = 0;
  for(int u = 1; u <= 5; u++) {
    const int n = FIT_TILE >> u, l = L - u;
    const double *ch = lv[cur];
    for(int q = threadIdx.x; q < n * n; q += blockDim.x) {
      const int i = q / n, j = q % n, m = 2 * n;
      const double v = ch[(2 * i) * m + 2 * j] + ch[(2 * i + 1) * m + 2 * j] + ch[(2 * i) * m + 2 * j + 1] +
                       ch[(2 * i + 1) * m + 2 * j + 1];
      lv[1 - cur][q] = v;
      st[GALIC_STACKOFFSET(l, tz * n + i, tr * n + j)] = v;
    }
    cur = 1 - cur;
    __syncthreads();
  }
}

// The levels above the tiles of k_fit_tiles (L-6 .. 0), one workgroup per stack.
__global__ void k_fit_top(FitArgs A) {
  const int job = blockIdx.x;
  const int t = job / 10 + 1, k = job % 10;
  if(!A.present[t]) return;
  const int L = A.L, Nstack = GALIC_NSTACK(L);
  const int dst[10] = {ST_RM, ST_RSR, ST_RST, ST_RSQ, ST_RSP, ST_EMR, ST_IR, ST_IT, ST_IP, ST_IQ};
  double *st = A.stacks + (size_t)t * ST_COUNT * Nstack + (size_t)dst[k] * Nstack;
  for(int l = L - 6; l >= 0; l--) {
    const int n = 1 << l;
    for(int q = threadIdx.x; q < n * n; q += blockDim.x) {
      const int i = q / n, j = q % n;
      st[GALIC_STACKOFFSET(l, i, j)] = st[GALIC_STACKOFFSET(l + 1, 2 * i, 2 * j)] +
                                       st[GALIC_STACKOFFSET(l + 1, 2 * i + 1, 2 * j)] +
                                       st[GALIC_STACKOFFSET(l + 1, 2 * i, 2 * j + 1)] +
                                       st[GALIC_STACKOFFSET(l + 1, 2 * i + 1, 2 * j + 1)];
    }
    __syncthreads();
  }
}

// The cut sums of calc_global_fit spread over nblk workgroups per type: partial sums of
// the five merit terms per workgroup, summed in workgroup order by k_fit_final.
__global__ void __launch_bounds__(256) k_fit_partial(FitArgs A, double *part, int nblk) {
  __shared__ double red[5 * 256];
  const int t = blockIdx.y + 1, b = blockIdx.x;
  if(!A.present[t]) return;
  const int L = A.L, Nstack = GALIC_NSTACK(L);
  const double *S = A.stacks + (size_t)t * ST_COUNT * Nstack;
  const double *W = A.weights + (size_t)t * W_COUNT * Nstack;
  const double *den = W + W_A * Nstack, *cutB = W + W_B * Nstack;
  const double *Rm = S + ST_RM * Nstack, *Tm = S + ST_MT * Nstack;
  const double *MR = S + ST_EMR * Nstack, *MT = S + ST_EMT * Nstack;
  const int stI[4] = {ST_IR, ST_IT, ST_IP, ST_IQ};
  const int stE[4] = {ST_ER, ST_ET, ST_EP, ST_EQ};
  double v[5] = {0, 0, 0, 0, 0};
  for(int node = b * blockDim.x + threadIdx.x; node < Nstack; node += nblk * blockDim.x) {
    if(den[node] != 0) v[0] += fabs(Rm[node] - Tm[node]) / den[node];
    if(cutB[node] != 0 && MR[node] > 0 && MT[node] > 0)
      for(int f = 0; f < 4; f++) {
        const double *I = S + stI[f] * Nstack, *E = S + stE[f] * Nstack;
        double tgt = E[node] / MT[node];
        double dd = tgt > A.lowdisp ? tgt : A.lowdisp;
        v[1 + f] += fabs(I[node] / MR[node] - tgt) / dd;
      }
  }
  block_sum<5>(v, red);
  if(threadIdx.x == 0)
    for(int f = 0; f < 5; f++) part[((size_t)blockIdx.y * nblk + b) * 5 + f] = v[f];
}

// The bookkeeping of main.c:294-359 from the partial sums (one thread per type).
__global__ void k_fit_final(FitArgs A, const double *part, int nblk) {
  const int t = blockIdx.x + 1;
  if(!A.present[t] || threadIdx.x != 0) return;
  double v[5] = {0, 0, 0, 0, 0};
  for(int b = 0; b < nblk; b++)
    for(int f = 0; f < 5; f++) v[f] += part[((size_t)blockIdx.x * nblk + b) * 5 + f];
  const int Nstack = GALIC_NSTACK(A.L);
  const double *Tm = A.stacks + (size_t)t * ST_COUNT * Nstack + ST_MT * Nstack;
  double *fit = A.fit + (size_t)t * 16;
  double s = v[0] * (1.0 / Tm[0]);
  double sr = v[1], st = v[2], sp = v[3], sq = v[4];
  int tovs = A.tovs[t];
  double cnt;
  if(tovs == 0 || tovs == 1) {
    cnt = 3.0;
    sq = 0;
  } else
    cnt = 4.0;
  if(fit[8] == 0) {
    fit[5] = s / ((sr + st + sp + sq) / cnt);
    fit[8] = 1;
  }
  double rf = fit[5];
  sr *= rf;
  st *= rf;
  sp *= rf;
  sq *= rf;
  fit[0] = s;
  fit[1] = sr;
  fit[2] = st;
  fit[3] = sp;
  fit[4] = sq;
  fit[6] = cnt;
  fit[7] = s + (sr + st + sp + sq) / cnt;
}

// One workgroup per type: the cut sums of calc_global_fit and the Srelfac
// bookkeeping (main.c:294-359).  fit[t][.] = S, Sdisp_r, Sdisp_t, Sdisp_p,
// Sdisp_q, Srelfac, Srelfac_count, Sall, firstrun flag.
__global__ void k_fit_sums(FitArgs A) {
  extern __shared__ double red[];
  const int t = blockIdx.x + 1;
  if(!A.present[t]) return;
  const int L = A.L, Nstack = GALIC_NSTACK(L);
  const double *S = A.stacks + (size_t)t * ST_COUNT * Nstack;
  const double *W = A.weights + (size_t)t * W_COUNT * Nstack;
  const double *den = W + W_A * Nstack, *cutB = W + W_B * Nstack;
  const double *Rm = S + ST_RM * Nstack, *Tm = S + ST_MT * Nstack;
  const double *MR = S + ST_EMR * Nstack, *MT = S + ST_EMT * Nstack;
  const int stI[4] = {ST_IR, ST_IT, ST_IP, ST_IQ};
  const int stE[4] = {ST_ER, ST_ET, ST_EP, ST_EQ};
  double v[5] = {0, 0, 0, 0, 0};
  for(int node = threadIdx.x; node < Nstack; node += blockDim.x) {
    if(den[node] != 0) v[0] += fabs(Rm[node] - Tm[node]) / den[node];
    if(cutB[node] != 0 && MR[node] > 0 && MT[node] > 0)
      for(int f = 0; f < 4; f++) {
        const double *I = S + stI[f] * Nstack, *E = S + stE[f] * Nstack;
        double tgt = E[node] / MT[node];
        double dd = tgt > A.lowdisp ? tgt : A.lowdisp;
        v[1 + f] += fabs(I[node] / MR[node] - tgt) / dd;
      }
  }
  block_sum<5>(v, red);
  if(threadIdx.x == 0) {
    double *fit = A.fit + (size_t)t * 16;
    double s = v[0] * (1.0 / Tm[0]);
    double sr = v[1], st = v[2], sp = v[3], sq = v[4];
    int tovs = A.tovs[t];
    double cnt;
    if(tovs == 0 || tovs == 1) {
      cnt = 3.0;
      sq = 0;
    } else
      cnt = 4.0;
    if(fit[8] == 0) {
      fit[5] = s / ((sr + st + sp + sq) / cnt);
      fit[8] = 1;
    }
    double rf = fit[5];
    sr *= rf;
    st *= rf;
    sp *= rf;
    sq *= rf;
    fit[0] = s;
    fit[1] = sr;
    fit[2] = st;
    fit[3] = sp;
    fit[4] = sq;
    fit[6] = cnt;
    fit[7] = s + (sr + st + sp + sq) / cnt;
  }
}

// ------------------------------------------------------- trial preparation --

// Orbit o = 2i is the trial's current velocity, o = 2i+1 its trial velocity.
__global__ void k_prepare_trials(int ntrial, const int *tidx, const double *tvx, const double *tvy,
                                 const double *tvz, Particles P, OrbitIn O) {
  int o = blockIdx.x * blockDim.x + threadIdx.x;
  if(o >= 2 * ntrial) return;
  int i = o >> 1, p = tidx[i];
  O.pidx[o] = p;
  O.ox[o] = P.x[p];
  O.oy[o] = P.y[p];
  O.oz[o] = P.z[p];
  O.omass[o] = P.mass[p];
  O.otint[o] = P.tint[p];
  O.otype[o] = P.type[p];
  if(o & 1) {
    O.ovx[o] = tvx[i];
    O.ovy[o] = tvy[i];
    O.ovz[o] = tvz[i];
  } else {
    O.ovx[o] = P.vx[p];
    O.ovy[o] = P.vy[p];
    O.ovz[o] = P.vz[p];
  }
}

// Orbit o = particle (base + o) with its current velocity (initial response pass).
__global__ void k_prepare_all(int n, int base, Particles P, OrbitIn O) {
  int o = blockIdx.x * blockDim.x + threadIdx.x;
  if(o >= n) return;
  int p = base + o;
  O.pidx[o] = p;
  O.ox[o] = P.x[p];
  O.oy[o] = P.y[p];
  O.oz[o] = P.z[p];
  O.ovx[o] = P.vx[p];
  O.ovy[o] = P.vy[p];
  O.ovz[o] = P.vz[p];
  O.omass[o] = P.mass[p];
  O.otint[o] = P.tint[p];
  O.otype[o] = P.type[p];
}

__global__ void k_store_orbits(int n, int base, const int *norbit, int *orbits) {
  int o = blockIdx.x * blockDim.x + threadIdx.x;
  if(o < n) orbits[base + o] = norbit[o];
}

// The response fields of orbits as the caller takes them, five FP64 grids per orbit, from their
// cell-major slots, which are zero again after it.  A workgroup turns 256 cells in LDS; the copy
// to the host bounds the whole.  (A call for 64 orbits on 64^2 grids: 15.7 ms with the slots copied and
// turned on the host, 13.4 ms so, 12.7 of them the orbits.)
template <typename T>
__global__ void __launch_bounds__(kFieldCells) k_fields_out(int ngrid, int nblk, T *slots, double *out) {
  __shared__ T cell[kFieldCells * kFields];
  const int o = blockIdx.x / nblk, c0 = blockIdx.x % nblk * kFieldCells, nc = min(kFieldCells, ngrid - c0);
  T *src = slots + ((size_t)o * ngrid + c0) * kFields;
  for(int i = threadIdx.x; i < nc * kFields; i += kFieldCells) {
    cell[i] = src[i];
    src[i] = 0;
  }
  __syncthreads();
  if((int)threadIdx.x < nc)
    for(int f = 0; f < kFields; f++)
      out[((size_t)o * kFields + f) * ngrid + c0 + threadIdx.x] = (double)cell[threadIdx.x * kFields + f];
}
template __global__ void k_fields_out<double>(int ngrid, int nblk, double *slots, double *out);
template __global__ void k_fields_out<float>(int ngrid, int nblk, float *slots, double *out);

}  // namespace galic
