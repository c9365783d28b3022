// FP64 explicit solve with the reference's operation order.  This file is
// compiled with -ffp-contract=off so every product and sum rounds as in the
// reference C++ (BatchedFiberRVEAnalysisExplicitTeamOuterLoop.h:180-437,
// BatchedFiberRVEAnalysisExplicitBase.h:155-287).
#include "root64.hpp"
#include "solve64_ieee.hpp"

namespace mf {
namespace kern {

// l = sqrt(x) and rl = 1 / l from the hardware's reciprocal square root
__device__ inline void sqrt64(double x, double &l, double &rl) {
  root64(x, __builtin_amdgcn_rsq(x), l, rl);
}
typedef __attribute__((address_space(4))) Law64 law_const;
// Three doubles per item in LDS as one 16-byte (x, y) array and one 8-byte z
// array: gathering random items takes 20 CU cycles a wave (in-order ones 8),
// against 32 (12) for records of 24 bytes or three arrays, and 34 (16) for
// records of 32 bytes; stores cost the same 21-35 in every layout.
typedef double v2d __attribute__((ext_vector_type(2), aligned(16)));
typedef __attribute__((address_space(3))) v2d lds_v2d;
typedef __attribute__((address_space(3))) double lds_double;
struct Lds3 {
  uint32_t xy, z;  // byte addresses of the arrays
  __device__ __forceinline__ void get(uint32_t i, double (&v)[3]) const {
    const v2d p = *reinterpret_cast<const lds_v2d *>((uintptr_t)(xy + 16u * i));
    v[0] = p.x;
    v[1] = p.y;
    v[2] = *reinterpret_cast<const lds_double *>((uintptr_t)(z + 8u * i));
  }
  __device__ __forceinline__ void put(uint32_t i, const double (&v)[3]) const {
    *reinterpret_cast<lds_v2d *>((uintptr_t)(xy + 16u * i)) = v2d{v[0], v[1]};
    *reinterpret_cast<lds_double *>((uintptr_t)(z + 8u * i)) = v[2];
  }
};
// Force of a nonlinear fiber (react64 with the stretch lr, g = (lr^2 - 1)/2
// and 1/l0 at hand): both extensions are one formula with selected constants.
__device__ inline double nonlinear64(const law_const &q, double lr, double g, double l0,
                                     double rl0) {
#pragma clang fp contract(off)
  const bool hi = lr > q.lt, lo = lr < q.lc;
  if (hi || lo)
    return div64(q.alpha, l0, rl0) * (hi ? q.Kt : q.Kc) * (lr - (hi ? q.lt : q.lc)) * l0 +
           (hi ? q.bt : q.bc);
  return q.alpha * lr * (exp(q.B * g) - 1);
}
// Hides a register's value from the compiler: what is derived from it is
// computed where it is used, not before a loop.
template <class T>
__device__ __forceinline__ void keep_packed(T &v) {
  asm volatile("" : "+v"(v));
}
// ---- pieces shared by the FP64 kernels for fast64 RVEs ---------------------
// Initial positions of every node (as solve64) and the boundary records.
template <int B>
__device__ __forceinline__ void init_positions64(const SolveArgs &a, const RveDev &R,
                                                 const double (&F)[9], bool ramp,
                                                 const Lds3 &pos, double *bst) {
#pragma clang fp contract(off)
  for (int r = threadIdx.x; r < R.N; r += B) {
    const int64_t g = R.node_off + r;
    double xp[3], inc[3], x[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) xp[d] = a.x_in[3 * g + d];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      inc[k] = (F[3 * k + 0] - (k == 0 ? 1.0 : 0.0)) * xp[0] +
               (F[3 * k + 1] - (k == 1 ? 1.0 : 0.0)) * xp[1] +
               (F[3 * k + 2] - (k == 2 ? 1.0 : 0.0)) * xp[2];
      const double up = a.u_in[3 * g + k];
      x[k] = a.X[3 * g + k] + (ramp ? up : inc[k] + up);
      if (r >= R.Nf) {
        bst[6 * (r - R.Nf) + k] = x[k];
        bst[6 * (r - R.Nf) + 3 + k] = ramp ? inc[k] : 0.0;
      }
    }
    pos.put(r, x);
  }
}
// Positions of the boundary nodes after step k (waves from the last one down,
// which hold the fewest free nodes).  k / S by S's reciprocal is exact:
// quotients of 31-bit numbers keep 2^-32 ulp from a rounding boundary.
template <int B>
__device__ __forceinline__ void move_boundary64(int k, double S, double rS, int amplitude,
                                                int Nf, int Nb, const Lds3 &pos,
                                                const double *bst) {
#pragma clang fp contract(off)
  const int b0 = B - 1 - (int)threadIdx.x;
  if (b0 < Nb) {
    const double alpha = amplitude64(div64(k, S, rS), amplitude);
    for (int b = b0; b < Nb; b += B) {
      const double *q = bst + 6 * b;
      double x[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) x[d] = q[d] + alpha * q[3 + d];
      pos.put(Nf + b, x);
    }
  }
}
// Force of a fiber of length l with reaction rid: one pass per law among the
// wave's fibers, its constants in scalar registers (fibers are listed by law,
// so nearly every wave has one).
__device__ __forceinline__ double law64(const law_const *laws, int rid, double l, double l0,
                                        double r0) {
#pragma clang fp contract(off)
  const double lr = div64(l, l0, r0);
  const double g = 1.0 / 2.0 * (lr * lr - 1);
  double frc = 0.0;
  for (bool todo = true; todo;) {
    const int u = __builtin_amdgcn_readfirstlane(rid);
    int k = u;  // hidden: known to equal rid below, it would load per lane
    asm volatile("" : "+s"(k));
    if (u == rid) {
      const law_const &q = laws[k];
      if (q.type == MF_REACTION_LINEAR)
        frc = lr * q.E * q.A * g;
      else
        frc = nonlinear64(q, lr, g, l0, r0);
      todo = false;
    }
  }
  return frc;
}
// Free nodes drift in place with their updated velocities.
template <int B, int NPT>
__device__ __forceinline__ void drift64(int Nf, double h, const double (&vr)[NPT][3],
                                        const Lds3 &pos) {
#pragma clang fp contract(off)
#pragma unroll
  for (int s = 0; s < NPT; ++s) {
    const int r = s * B + (int)threadIdx.x;
    if (r < Nf) {
      double x[3];
      pos.get(r, x);
#pragma unroll
      for (int d = 0; d < 3; ++d) x[d] = x[d] + 2 * h * vr[s][d];
      pos.put(r, x);
    }
  }
}
__device__ __forceinline__ double load_double(__amdgpu_buffer_rsrc_t rs, int vo, int so) {
  typedef uint32_t u2 __attribute__((ext_vector_type(2)));
  const u2 q = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(rs, vo, so, 0));
  return __hiloint2double((int)q.y, (int)q.x);
}
// FinalizeData + computeCauchyStress (as solve64) from the final positions.
template <int B>
__device__ __forceinline__ void finalize64(const SolveArgs &a, const RveDev &R, int rv, int sid,
                                           int step, int status, bool ramp, const Lds3 &pos,
                                           const double *bst, double *red) {
#pragma clang fp contract(off)
  const int tid = threadIdx.x, Nf = R.Nf, Nb = R.Nb;
  const int64_t nb = R.node_off;
  const int32_t *gw = a.ell_w + R.ell_off;
  const double *gl0 = a.ell_l0 + R.ell_off;
  __syncthreads();  // the last refresh reduction has been read by every wave
  double st[6] = {0, 0, 0, 0, 0, 0};
  const int flags = a.solve_flags[sid];
  const double alpha_end = ramp ? ramp_alpha(step, a.n_steps, a.amplitude) : 0.0;
  for (int b = tid; b < Nb; b += B) {
    const int r = Nf + b;
    double xb[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) xb[d] = bst[6 * b + d] + alpha_end * bst[6 * b + 3 + d];
    const int base = a.slice_base[R.slice_off + r / kWave] + (r & (kWave - 1));
    const int dg = a.deg[nb + r];
    double f1 = 0.0, f2 = 0.0, f3 = 0.0;
    for (int j = 0; j < dg; ++j) {
      const int idx = base + j * kWave;
      const int32_t wv = gw[idx];
      const double l0 = gl0[idx];
      double p[3];
      pos.get(wv & 0xFFFFFF, p);
      const double dx = p[0] - xb[0];
      const double dy = p[1] - xb[1];
      const double dz = p[2] - xb[2];
      const double l = sqrt(dx * dx + dy * dy + dz * dz);
      const double t = react64(a.laws[R.react_off + ((uint32_t)wv >> 24)], l0, l) / l;
      f1 = f1 - dx * t;
      f2 = f2 - dy * t;
      f3 = f3 - dz * t;
    }
    st[0] += xb[0] * f1;
    st[1] += xb[1] * f2;
    st[2] += xb[2] * f3;
    st[3] += 0.5 * (xb[1] * f3 + xb[2] * f2);
    st[4] += 0.5 * (xb[0] * f3 + xb[2] * f1);
    st[5] += 0.5 * (xb[0] * f2 + xb[1] * f1);
    if (flags & kWriteX)
      for (int d = 0; d < 3; ++d) a.x_out[3 * (nb + r) + d] = xb[d];
    if (flags & kWriteU)
      for (int d = 0; d < 3; ++d) a.u_out[3 * (nb + r) + d] = xb[d] - a.X[3 * (nb + r) + d];
  }
  for (int r = tid; r < Nf; r += B) {
    const int64_t g = nb + r;
    double x[3];
    pos.get(r, x);
    if (flags & kWriteX)
      for (int d = 0; d < 3; ++d) a.x_out[3 * g + d] = x[d];
    if (flags & kWriteU)
      for (int d = 0; d < 3; ++d) a.u_out[3 * g + d] = x[d] - a.X[3 * g + d];
  }
  block_sum<B, 6>(st, red);
  if (tid == 0) {
    const double sv = R.scale / a.V[rv];
    bool bad = false;
    for (int i = 0; i < 6; ++i) {
      double v = st[i] * sv;
      a.sigma[6 * (int64_t)sid + i] = v;
      bad = bad || !isfinite(v);
    }
    if (bad && status == MF_STATUS_OK) status = MF_STATUS_NAN;
    a.status[sid] = status;
    a.steps[sid] = step;
  }
}

// ============================================================================
// FP64 kernel, each fiber evaluated once per step
// ============================================================================
// Bitwise the result of solve64: at end b the difference vector is exactly
// the negation of end a's (x_a - x_b = -(x_b - x_a) in IEEE arithmetic), so
// the length, the force, t = f/l and d t of a fiber are the same numbers at
// both ends, up to the sign.  A fiber phase computes d t once per fiber with
// a free end into a 24-byte LDS record; a node phase sums each free node's
// records in its ELL order, subtracting at end a and adding at end b, which
// are solve64's roundings (an FMA by +-1 rounds as the addition does).
//
// What bounds it: FP64 instruction issue and LDS in turn, between two barriers
// (0.66 of the SIMD cycles and 0.63 of the LDS cycles on 1024 RVEs of 500
// nodes, 0.27 of the latter bank conflicts of the gathers).  So nothing that does
// not change is computed or loaded in the step loop: a lane keeps its FPL fibers
// (both ends' ranks, l0, 1/l0) and its nodes' first record references
// (16 bits each) in registers, reaction constants are formed once
// per batch, quotients by l0, m and l multiply by a reciprocal and correct
// the result (div64), the two half kicks of a step share their quotient
// except after a refresh, and the shortest fiber is a by-product of the
// fiber phase.  Positions need one buffer: the node phase reads records only.
//
// 1024 linear RVEs of 500 nodes, 1000 steps: 10.3 ms with solve64, 5.3 ms
// with this split and an entry at a time in the node phase, 4.4 ms with four
// entries in flight and the (x, y), z arrays.  One RVE of 250 nodes on a CU
// of its own: 2.9 us a step, now 1.1 us.
//
// fast64 RVEs only (lengths and masses far inside the FP64 range).
template <int B, int NPT, int FPL, bool LIN>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(4)))
void solve64f(SolveArgs a) {
#pragma clang fp contract(off)
  constexpr int NW = B / kWave;
  // record references of a node held in registers: nodes are sorted by
  // degree, so only the first slot has nodes of more than eight fibers, and
  // in networks of mean degree 5 hardly any of more than kRefs0
  constexpr int kRefs = 8, kRefs0 = NPT == 1 ? 16 : 12;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int sid = a.order ? a.order[blockIdx.x] : (int)blockIdx.x;
  const int rv = a.solve_rve[sid];
  const RveDev R = a.rves[rv];
  const double eta_r = a.eta_rve ? a.eta_rve[rv] : a.eta;
  const int N = R.N, Nf = R.Nf, Nb = R.Nb, M = R.M, Mf = R.m_free;
  const int64_t nb = R.node_off;

  // LDS carve (mirrors lds_bytes)
  const uint32_t at =
      (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char *)smem);
  const int Ne = (N + 1) & ~1, Me = (M + 2) & ~1;  // keep 16-byte alignment
  const Lds3 pos{at, at + 16u * Ne};                                   // [N]
  const Lds3 rec{at + 24u * Ne, at + 24u * Ne + 16u * Me};             // [M + 1], record M zero
  size_t off = 24 * ((size_t)Ne + Me);
  double *red = reinterpret_cast<double *>(smem + off);
  off += sizeof(double) * NW * kRedStride;
  double *bst = reinterpret_cast<double *>(smem + off);  // [Nb][6] x_b0, g

  const int32_t *gw = a.ell_w + R.ell_off;
  const double *gl0 = a.ell_l0 + R.ell_off;
  const int32_t *gfr = a.ell_fref + R.ell_off;
  const int32_t *fst = a.fstream + 4 * R.fib_off;
  // constant for the whole launch: read with scalar loads
  const law_const *laws = reinterpret_cast<const law_const *>(
      reinterpret_cast<uintptr_t>(a.laws + R.react_off));
  if (tid == 0) rec.put(M, {0.0, 0.0, 0.0});

  double F[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) F[i] = a.solve_F[9 * (int64_t)sid + i];
  const bool ramp = a.mode == MF_MODE_RAMP;

  init_positions64<B>(a, R, F, ramp, pos, bst);
  // the lane's fibers: both ends' ranks (16 bits each), reference length and its reciprocal, reaction ids (3 bits a slot)
  uint32_t fab[FPL];
  double fl0[FPL], fr0[FPL];
  int frid = 0;
#pragma unroll
  for (int k = 0; k < FPL; ++k) {
    const int e = k * B + tid;
    fab[k] = 0;
    fl0[k] = fr0[k] = 1.0;
    if (e < Mf) {
      const int sa = fst[4 * e + 2];
      fab[k] = (uint32_t)fst[4 * e] | (uint32_t)fst[4 * e + 1] << 16;
      fl0[k] = gl0[sa];
      fr0[k] = 1.0 / fl0[k];
      frid |= (int)((uint32_t)gw[sa] >> 24) << (3 * k);
    }
  }
  __syncthreads();

  // with two nodes per thread their positions stay in LDS only: 12 registers
  // that would spill
  constexpr bool kXReg = NPT == 1;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  double xr[kXReg ? NPT : 1][3], vr[NPT][3], mr[NPT], rm[NPT];
  int Dr[NPT];
  uint32_t refs[NPT][kRefs0 / 2];  // 16 bits: record | (node is end a) << 15
#pragma unroll
  for (int s = 0; s < NPT; ++s) {
    const int r = s * B + tid;
    const int k = s * NW + wave, sl = R.slice_off + k;  // slice of the wave's nodes
    mr[s] = r < Nf ? a.mass[nb + r] : 1.0;
    rm[s] = 1.0 / mr[s];
    if (kXReg && r < Nf) pos.get(r, xr[s]);
    vr[s][0] = vr[s][1] = vr[s][2] = 0.0;
    // waves past Nf never gather
    Dr[s] = k * kWave < Nf ? a.slice_D[sl] : 0;
    const int base = (k * kWave < Nf ? a.slice_base[sl] : 0) + lane;
#pragma unroll
    for (int j = 0; j < (s == 0 ? kRefs0 : kRefs); ++j) {
      const uint32_t q = j < Dr[s] ? (uint32_t)gfr[base + j * kWave] : (uint32_t)M;
      const uint32_t w = (q & 0x7FFFu) | q >> 31 << 15;
      refs[s][j / 2] = j & 1 ? refs[s][j / 2] | w << 16 : w;
    }
  }

  const double linE = laws[0].E, linA = laws[0].A;  // LIN

  const double c_sound = R.c_sound;
  // d t of the lane's fibers at the current positions into the records;
  // returns the smallest of their squared lengths (the square root of the
  // smallest is the smallest of the square roots: rounding is monotonic)
  auto fiber_phase = [&]() __attribute__((always_inline)) {
    double l2min = __builtin_inf();
#pragma unroll
    for (int k = 0; k < FPL; ++k) {
      const int e = k * B + tid;
      if (e < Mf) {
        double pa[3], pb[3];
        pos.get(fab[k] & 0xFFFFu, pa);
        pos.get(fab[k] >> 16, pb);
        const double dx = pb[0] - pa[0];
        const double dy = pb[1] - pa[1];
        const double dz = pb[2] - pa[2];
        const double l2 = dx * dx + dy * dy + dz * dz;
        double l, rl;
        sqrt64(l2, l, rl);
        l2min = __builtin_fmin(l2min, l2);
        double frc;
        if (LIN) {
          const double lr = div64(l, fl0[k], fr0[k]);
          frc = lr * linE * linA * (1.0 / 2.0 * (lr * lr - 1));
        } else {
          frc = law64(laws, (frid >> (3 * k)) & 7, l, fl0[k], fr0[k]);
        }
        const double t = div64(frc, l, rl);
        rec.put(e, {dx * t, dy * t, dz * t});
      }
    }
    return l2min;
  };
  // lengths of the fibers between two boundary nodes (refresh steps only)
  auto outer_min = [&](double l2min) {
    for (int e = Mf + tid; e < M; e += B) {
      double pa[3], pb[3];
      pos.get(fst[4 * e], pa);
      pos.get(fst[4 * e + 1], pb);
      const double dx = pb[0] - pa[0], dy = pb[1] - pa[1], dz = pb[2] - pa[2];
      l2min = __builtin_fmin(l2min, dx * dx + dy * dy + dz * dz);
    }
    return l2min;
  };
  // internal force of a slot's node from the records, in ELL order.  Four
  // entries' loads are in flight at once (past the list, the zero record's):
  // one at a time, each waited for its own, which took half of a step on
  // RVEs that leave a CU's other wave slots empty.
  auto node_force = [&](int s, double (&f)[3]) __attribute__((always_inline)) {
    f[0] = f[1] = f[2] = 0.0;
    const int D = Dr[s], nr = s == 0 ? kRefs0 : kRefs;
#pragma unroll
    for (int j0 = 0; j0 < nr; j0 += 4) {
      if (j0 > 0 && j0 >= D) break;
      double q[4][3];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t w = refs[s][(j0 + j) / 2];
        rec.get((j & 1 ? w >> 16 : w) & 0x7FFFu, q[j]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t w = refs[s][(j0 + j) / 2];
        // -1 at end a, +1 at end b
        const double sg =
            __hiloint2double((int)(((j & 1 ? w : w << 16) & 0x80000000u) | 0x3FF00000u), 0);
#pragma unroll
        for (int d = 0; d < 3; ++d) f[d] = __builtin_fma(sg, q[j][d], f[d]);
      }
    }
    if (__builtin_expect(D > nr, 0)) {
      const int base = a.slice_base[R.slice_off + s * NW + wave] + lane;
      for (int j = nr; j < D; ++j) {
        const uint32_t q = (uint32_t)gfr[base + j * kWave];
        double p[3];
        rec.get(q & 0x7FFFu, p);
        const double sg = __hiloint2double((int)((q & 0x80000000u) | 0x3FF00000u), 0);
#pragma unroll
        for (int d = 0; d < 3; ++d) f[d] = __builtin_fma(sg, p[d], f[d]);
      }
    }
  };
  const double S = a.n_steps, rS = 1.0 / S;

  // ---- RunInitialization (TeamOuterLoop.h:215-289) and the main loop
  // (TeamOuterLoop.h:340-371).  One pass: forces at the current positions,
  // the closing half kick of the step that led there, the opening half kick
  // and drift of the next.  The first pass (step -1) has no closing kick.
  int step = -1, due = 0;
  double residual = 10.0, h = 0.0;
  int status = MF_STATUS_OK;
  const int freq = a.freq;
  for (;;) {
    // the packed words stay packed: unpacked once before the loop, they would
    // take twice the registers and spill
    keep_packed(frid);
#pragma unroll
    for (int k = 0; k < FPL; ++k) keep_packed(fab[k]);
#pragma unroll
    for (int s = 0; s < NPT; ++s)
#pragma unroll
      for (int j = 0; j < (s == 0 ? kRefs0 : kRefs) / 2; ++j) keep_packed(refs[s][j]);
    double l2min = fiber_phase();
    __syncthreads();  // records published
    // steps 0, freq, 2 freq, ...: counted, a remainder would cost each step
    // a division
    const bool refresh = step < 0 || step == due;
    const double h1 = h;
    if (__builtin_expect(refresh, 0)) {
      if (step >= 0) due += freq;
      // the residual takes a pass over the records of its own, so that the
      // other steps need not keep the forces until the sums are known
      double rsum = 0.0;
#pragma unroll
      for (int s = 0; s < NPT; ++s) {
        if (s * B + tid < Nf) {
          double f[3];
          node_force(s, f);
          double rn = 0.0;
#pragma unroll
          for (int d = 0; d < 3; ++d) rn += f[d] * f[d];
          rsum += rn;
        }
      }
      l2min = outer_min(l2min);
      block_min_sum<B>(l2min, rsum, red);
      const double lmin = sqrt(l2min);
      h = a.crit * ((lmin < 1.0e300 ? lmin : 1.0e300) / c_sound) * 0.5;
      if (step >= 0) residual = sqrt(rsum);
    }
    if (step >= 0) {
      bool stop = false;
      ++step;
      if (ramp) {
        stop = step >= a.n_steps;
      } else if (!(residual > a.tol)) {
        stop = true;
      } else if (step >= a.max_steps) {
        status = MF_STATUS_STEP_CAP;
        stop = true;
      }
      if (stop) break;
    } else {
      step = 0;
    }
    // half kicks and drift of free nodes (TeamOuterLoop.h:144-175)
#pragma unroll
    for (int s = 0; s < NPT; ++s) {
      const int r = s * B + tid;
      if (r < Nf) {
        double f[3];
        node_force(s, f);
        double x[3];
        if (kXReg) {
#pragma unroll
          for (int d = 0; d < 3; ++d) x[d] = xr[s][d];
        } else {
          pos.get(r, x);
        }
        const double mass = mr[s] * eta_r;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const double ft = -f[d] - mass * vr[s][d];
          const double a2 = div64(h * ft, mr[s], rm[s]);
          double a1 = a2;
          if (__builtin_expect(refresh, 0)) {
            asm volatile("");  // not computed in the other steps
            a1 = div64(h1 * ft, mr[s], rm[s]);
          }
          const double vl = vr[s][d] + a1 + a2;
          vr[s][d] = vl;
          x[d] = x[d] + 2 * h * vl;
          if (kXReg) xr[s][d] = x[d];
        }
        pos.put(r, x);
      }
    }
    if (ramp) move_boundary64<B>(step + 1, S, rS, a.amplitude, Nf, Nb, pos, bst);
    __syncthreads();  // positions published, record reads done
  }
  if (residual != residual) status = MF_STATUS_NAN;

  finalize64<B>(a, R, rv, sid, step, status, ramp, pos, bst, red);
}

// ============================================================================
// FP64 node-centric kernel for RVEs whose force records do not fit LDS
// ============================================================================
// solve64's results bit for bit with solve64f's arithmetic (fast64 RVEs):
// every free node gathers its fibers in ELL order, each fiber evaluated at
// both ends.  Only the positions (one buffer) and the boundary state live in
// LDS, so RVEs of up to ~5000 nodes fit; the lists stream from L2 through
// buffer resources, one entry ahead.  Velocities are updated while the old
// positions are still being gathered; after a barrier the nodes drift in place.
template <int B, int NPT>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(B / 256)))
void solve64n(SolveArgs a) {
#pragma clang fp contract(off)
  constexpr int NW = B / kWave;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int sid = a.order ? a.order[blockIdx.x] : (int)blockIdx.x;
  const int rv = a.solve_rve[sid];
  const RveDev R = a.rves[rv];
  const double eta_r = a.eta_rve ? a.eta_rve[rv] : a.eta;
  const int N = R.N, Nf = R.Nf, Nb = R.Nb, M = R.M;
  const int64_t nb = R.node_off;

  // LDS carve (mirrors lds_bytes)
  const uint32_t at =
      (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char *)smem);
  const int Ne = (N + 1) & ~1;
  const Lds3 pos{at, at + 16u * Ne};  // [N]
  size_t off = 24 * (size_t)Ne;
  double *red = reinterpret_cast<double *>(smem + off);
  off += sizeof(double) * NW * kRedStride;
  double *bst = reinterpret_cast<double *>(smem + off);  // [Nb][6] x_b0, g

  const int32_t *gw = a.ell_w + R.ell_off;
  const double *gl0 = a.ell_l0 + R.ell_off;
  const law_const *laws = reinterpret_cast<const law_const *>(
      reinterpret_cast<uintptr_t>(a.laws + R.react_off));
  // the RVE's free-node entries as raw buffers (loads past the end return 0)
  const int entries = R.ell_free_entries;
  const __amdgpu_buffer_rsrc_t rsw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int32_t *>(gw), 0, entries * 4, kBufRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsl = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<double *>(gl0), 0, entries * 8, kBufRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<double *>(a.ell_r0 + R.ell_off), 0, entries * 8, kBufRsrcWord3);

  double F[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) F[i] = a.solve_F[9 * (int64_t)sid + i];
  const bool ramp = a.mode == MF_MODE_RAMP;
  init_positions64<B>(a, R, F, ramp, pos, bst);
  __syncthreads();

  // masses and degrees (8 bits a slot) are reloaded or packed: four nodes per
  // thread leave few registers for the force
  double vr[NPT][3], rm[NPT];
  int Dr[NPT], base[NPT];
  uint32_t degs = 0;
#pragma unroll
  for (int s = 0; s < NPT; ++s) {
    const int r = s * B + tid;
    const int k = s * NW + wave, sl = R.slice_off + k;  // slice of the wave's nodes
    rm[s] = r < Nf ? 1.0 / a.mass[nb + r] : 1.0;
    vr[s][0] = vr[s][1] = vr[s][2] = 0.0;
    Dr[s] = k * kWave < Nf ? a.slice_D[sl] : 0;
    base[s] = k * kWave < Nf ? a.slice_base[sl] : 0;
    degs |= (uint32_t)(r < Nf ? a.deg[nb + r] : 0) << (8 * s);
  }

  const double c_sound = R.c_sound;
  struct Entry {
    int32_t w;
    double l0, r0;
  };
  // internal force of a slot's node, in ELL order
  auto node_force = [&](int s, const double (&x)[3], double (&f)[3])
                        __attribute__((always_inline)) {
    f[0] = f[1] = f[2] = 0.0;
    const int D = Dr[s];
    auto entry = [&](int j) __attribute__((always_inline)) {
      Entry q;
      const int so = base[s] + j * kWave;
      q.w = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(rsw, lane * 4, so * 4, 0);
      q.l0 = load_double(rsl, lane * 8, so * 8);
      q.r0 = load_double(rsr, lane * 8, so * 8);
      return q;
    };
    const int dg = (int)(degs >> (8 * s) & 255u);
    Entry nx = entry(0);
    for (int j = 0; j < D; ++j) {
      const Entry q = nx;
      nx = entry(j + 1 < D ? j + 1 : j);
      if (j < dg) {
        double p[3];
        pos.get((uint32_t)q.w & 0xFFFFFFu, p);
        const double dx = p[0] - x[0], dy = p[1] - x[1], dz = p[2] - x[2];
        double l, rl;
        sqrt64(dx * dx + dy * dy + dz * dz, l, rl);
        const double t = div64(law64(laws, (int)((uint32_t)q.w >> 24), l, q.l0, q.r0), l, rl);
        f[0] = f[0] - dx * t;
        f[1] = f[1] - dy * t;
        f[2] = f[2] - dz * t;
      }
    }
  };

  // ---- RunInitialization (TeamOuterLoop.h:215-289) and the main loop
  // (TeamOuterLoop.h:340-371), organised as in solve64f
  int step = -1, due = 0;
  double residual = 10.0, h = 0.0;
  int status = MF_STATUS_OK;
  const int freq = a.freq;
  const double S = a.n_steps, rS = 1.0 / S;
  for (;;) {
    keep_packed(degs);
    const bool refresh = step < 0 || step == due;
    const double h1 = h;
    if (__builtin_expect(refresh, 0)) {
      if (step >= 0) due += freq;
      double l2min = __builtin_inf(), none = 0.0;
      const int32_t *fb = a.fib + 2 * R.fib_off;
      for (int e = tid; e < M; e += B) {
        double pa[3], pb[3];
        pos.get(fb[2 * e], pa);
        pos.get(fb[2 * e + 1], pb);
        const double dx = pb[0] - pa[0], dy = pb[1] - pa[1], dz = pb[2] - pa[2];
        l2min = __builtin_fmin(l2min, dx * dx + dy * dy + dz * dz);
      }
      block_min_sum<B>(l2min, none, red);
      const double lmin = sqrt(l2min);
      h = a.crit * ((lmin < 1.0e300 ? lmin : 1.0e300) / c_sound) * 0.5;
    }
    double rsum = 0.0;
#pragma unroll
    for (int s = 0; s < NPT; ++s) {
      const int r = s * B + tid;
      if (r < Nf) {
        double x[3], f[3];
        pos.get(r, x);
        node_force(s, x, f);
        double rn = 0.0;
        const double m = a.mass[nb + r], mass = m * eta_r;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          rn += f[d] * f[d];
          const double ft = -f[d] - mass * vr[s][d];
          const double a2 = div64(h * ft, m, rm[s]);
          double a1 = a2;
          if (__builtin_expect(refresh, 0)) {
            asm volatile("");  // not computed in the other steps
            a1 = div64(h1 * ft, m, rm[s]);
          }
          vr[s][d] = vr[s][d] + a1 + a2;
        }
        rsum += rn;
      }
    }
    if (__builtin_expect(refresh && step >= 0, 0)) {
      // slots 2-3 of the scratch: waves may still read slots 0-1 above
      double none = 0.0;
      block_min_sum<B>(none, rsum, red + 2);
      residual = sqrt(rsum);
    }
    if (step >= 0) {
      bool stop = false;
      ++step;
      if (ramp) {
        stop = step >= a.n_steps;
      } else if (!(residual > a.tol)) {
        stop = true;
      } else if (step >= a.max_steps) {
        status = MF_STATUS_STEP_CAP;
        stop = true;
      }
      if (stop) break;
    } else {
      step = 0;
    }
    __syncthreads();  // every gather of the old positions is done
    drift64<B, NPT>(Nf, h, vr, pos);
    if (ramp) move_boundary64<B>(step + 1, S, rS, a.amplitude, Nf, Nb, pos, bst);
    __syncthreads();  // positions published
  }
  if (residual != residual) status = MF_STATUS_NAN;
  finalize64<B>(a, R, rv, sid, step, status, ramp, pos, bst, red);
}

// ============================================================================
// FP64 fiber-once kernel for large RVEs
// ============================================================================
// solve64f's results for RVEs whose force records do not fit LDS, or whose
// fibers the registers of a forced thread count.  Records
// hold t = f/l alone (8 bytes), and a node's gather recomputes d from the
// positions, so these must stay until every gather is done: one buffer, and
// the nodes drift in place after a barrier.  In RVEs with fibers of both laws
// the nonlinear fibers come first in the stream and in every node's list, so
// the records are formed in two rounds, nonlinear then linear, in the same
// storage: a 4000-node RVE keeps 96 KB of positions and ~40 KB of records.
// Fiber and list data stream from L2.  257 toe-law RVEs of 200-4000 nodes, 600
// steps, whose largest RVEs end the batch: 11.8 ms, against 13.1 ms with the
// node-centric kernel above, which evaluates every fiber twice, in waves of
// mixed laws, and 20.4 ms with solve64.
template <int B, int NPT>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(4)))
void solve64t(SolveArgs a) {
#pragma clang fp contract(off)
  constexpr int NW = B / kWave;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int sid = a.order ? a.order[blockIdx.x] : (int)blockIdx.x;
  const int rv = a.solve_rve[sid];
  const RveDev R = a.rves[rv];
  const double eta_r = a.eta_rve ? a.eta_rve[rv] : a.eta;
  const int N = R.N, Nf = R.Nf, Nb = R.Nb, M = R.M, Mf = R.m_free;
  const int64_t nb = R.node_off;

  // LDS carve (mirrors lds_bytes)
  const uint32_t at =
      (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char *)smem);
  const int Ne = (N + 1) & ~1, Te = (R.t_records + 1) & ~1;
  const Lds3 pos{at, at + 16u * Ne};  // [N]
  const uint32_t trec = at + 24u * Ne;  // [t_records]
  size_t off = 24 * (size_t)Ne + 8 * (size_t)Te;
  double *red = reinterpret_cast<double *>(smem + off);
  off += sizeof(double) * NW * kRedStride;
  double *bst = reinterpret_cast<double *>(smem + off);  // [Nb][6] x_b0, g

  const uint32_t *fab = a.fs_ab + R.fib_off;
  const double2 *flr = a.fs_lr + R.fib_off;
  const law_const *laws = reinterpret_cast<const law_const *>(
      reinterpret_cast<uintptr_t>(a.laws + R.react_off));
  // the RVE's free-node entries as raw buffers (loads past the end return 0)
  const int list_bytes = R.ell_free_entries * 4;
  const __amdgpu_buffer_rsrc_t rsw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int32_t *>(a.ell_w + R.ell_off), 0, list_bytes, kBufRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsf = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int32_t *>(a.ell_fref + R.ell_off), 0, list_bytes, kBufRsrcWord3);
  // fibers [0, n1) and list entries of the first round; none: one round
  const bool mixed = R.n_nl > 0 && R.n_nl < Mf;
  const int n1 = mixed ? R.n_nl : 0;

  double F[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) F[i] = a.solve_F[9 * (int64_t)sid + i];
  const bool ramp = a.mode == MF_MODE_RAMP;
  init_positions64<B>(a, R, F, ramp, pos, bst);
  __syncthreads();

  // masses are reloaded; degrees and first-round counts take 8 bits a slot
  double vr[NPT][3], rm[NPT];
  int Dr[NPT], D1[NPT], J2[NPT], base[NPT];  // J2: where a lane's second round may begin
  uint32_t degs = 0, cnts = 0;
#pragma unroll
  for (int s = 0; s < NPT; ++s) {
    const int r = s * B + tid;
    const int k = s * NW + wave, sl = R.slice_off + k;  // slice of the wave's nodes
    rm[s] = r < Nf ? 1.0 / a.mass[nb + r] : 1.0;
    vr[s][0] = vr[s][1] = vr[s][2] = 0.0;
    Dr[s] = k * kWave < Nf ? a.slice_D[sl] : 0;
    base[s] = k * kWave < Nf ? a.slice_base[sl] : 0;
    const int dg = r < Nf ? a.deg[nb + r] : 0;
    int cnt = 0;
    if (mixed)
      while (cnt < dg && (a.ell_fref[R.ell_off + base[s] + cnt * kWave + lane] & 0x7FFFFFFF) < n1)
        ++cnt;
    degs |= (uint32_t)dg << (8 * s);
    cnts |= (uint32_t)cnt << (8 * s);
    int first = r < Nf ? cnt : 255;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      cnt = max(cnt, __shfl_xor(cnt, o, kWave));
      first = min(first, __shfl_xor(first, o, kWave));
    }
    D1[s] = __builtin_amdgcn_readfirstlane(cnt);
    J2[s] = min(__builtin_amdgcn_readfirstlane(first), Dr[s]);
  }

  const double c_sound = R.c_sound;
  // t of fibers [e0, e1) into the records; returns the smallest squared length
  auto fiber_round = [&](int e0, int e1, double l2min) __attribute__((always_inline)) {
    int e = e0 + tid;
    uint32_t ab = e < e1 ? fab[e] : 0;
    double2 lr = e < e1 ? flr[e] : make_double2(1.0, 1.0);
    for (; e < e1; e += B) {
      const uint32_t ab0 = ab;
      const double2 lr0 = lr;
      const int en = e + B < e1 ? e + B : e;  // the next fiber loads meanwhile
      ab = fab[en];
      lr = flr[en];
      double pa[3], pb[3];
      pos.get(stream_a(ab0), pa);
      pos.get(stream_b(ab0), pb);
      const double dx = pb[0] - pa[0], dy = pb[1] - pa[1], dz = pb[2] - pa[2];
      const double l2 = dx * dx + dy * dy + dz * dz;
      double l, rl;
      sqrt64(l2, l, rl);
      l2min = __builtin_fmin(l2min, l2);
      const double frc = law64(laws, stream_law(ab0), l, lr0.x, lr0.y);
      *reinterpret_cast<lds_double *>((uintptr_t)(trec + 8u * (uint32_t)(e - e0))) =
          div64(frc, l, rl);
    }
    return l2min;
  };
  // adds entries [j0, j1) of a slot's list to its force: those of the round
  // whose first fiber is e0, the lane's own being [c0, c1)
  auto gather = [&](int s, int j0, int j1, int c0, int c1, int e0, const double (&x)[3],
                    double (&f)[3]) __attribute__((always_inline)) {
    auto word = [&](__amdgpu_buffer_rsrc_t rs, int j) __attribute__((always_inline)) {
      return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, lane * 4,
                                                             (base[s] + j * kWave) * 4, 0);
    };
    uint32_t wn = word(rsw, j0), tn = word(rsf, j0);
    for (int j = j0; j < j1; ++j) {
      const uint32_t w = wn & 0xFFFFFFu, q = tn & 0x7FFFFFFFu;
      const int jn = j + 1 < j1 ? j + 1 : j;
      wn = word(rsw, jn);
      tn = word(rsf, jn);
      if (j >= c0 && j < c1) {
        double p[3];
        pos.get(w, p);
        const double t = *reinterpret_cast<const lds_double *>((uintptr_t)(trec + 8u * (q - e0)));
        f[0] = f[0] - (p[0] - x[0]) * t;
        f[1] = f[1] - (p[1] - x[1]) * t;
        f[2] = f[2] - (p[2] - x[2]) * t;
      }
    }
  };

  // ---- RunInitialization (TeamOuterLoop.h:215-289) and the main loop
  // (TeamOuterLoop.h:340-371), organised as in solve64f
  int step = -1, due = 0;
  double residual = 10.0, h = 0.0;
  int status = MF_STATUS_OK;
  const int freq = a.freq;
  const double S = a.n_steps, rS = 1.0 / S;
  for (;;) {
    keep_packed(degs);
    keep_packed(cnts);
    const bool refresh = step < 0 || step == due;
    const double h1 = h;
    double l2min = __builtin_inf();
    double f[NPT][3];
#pragma unroll
    for (int s = 0; s < NPT; ++s) f[s][0] = f[s][1] = f[s][2] = 0.0;
    if (mixed) {
      l2min = fiber_round(0, n1, l2min);
      __syncthreads();  // first round's records published
#pragma unroll
      for (int s = 0; s < NPT; ++s) {
        const int r = s * B + tid;
        if (r < Nf) {
          double x[3];
          pos.get(r, x);
          gather(s, 0, D1[s], 0, (int)(cnts >> (8 * s) & 255u), 0, x, f[s]);
        }
      }
      __syncthreads();  // and read
    }
    l2min = fiber_round(n1, Mf, l2min);
    if (__builtin_expect(refresh, 0)) {
      if (step >= 0) due += freq;
      double none = 0.0;
      for (int e = Mf + tid; e < M; e += B) {  // between two boundary nodes
        double pa[3], pb[3];
        pos.get(stream_a(fab[e]), pa);
        pos.get(stream_b(fab[e]), pb);
        const double dx = pb[0] - pa[0], dy = pb[1] - pa[1], dz = pb[2] - pa[2];
        l2min = __builtin_fmin(l2min, dx * dx + dy * dy + dz * dz);
      }
      block_min_sum<B>(l2min, none, red);
      const double lmin = sqrt(l2min);
      h = a.crit * ((lmin < 1.0e300 ? lmin : 1.0e300) / c_sound) * 0.5;
    }
    __syncthreads();  // records published
    double rsum = 0.0;
#pragma unroll
    for (int s = 0; s < NPT; ++s) {
      const int r = s * B + tid;
      if (r < Nf) {
        double x[3];
        pos.get(r, x);
        gather(s, J2[s], Dr[s], (int)(cnts >> (8 * s) & 255u), (int)(degs >> (8 * s) & 255u), n1,
               x, f[s]);
        double rn = 0.0;
        const double m = a.mass[nb + r], mass = m * eta_r;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          rn += f[s][d] * f[s][d];
          const double ft = -f[s][d] - mass * vr[s][d];
          const double a2 = div64(h * ft, m, rm[s]);
          double a1 = a2;
          if (__builtin_expect(refresh, 0)) {
            asm volatile("");  // not computed in the other steps
            a1 = div64(h1 * ft, m, rm[s]);
          }
          vr[s][d] = vr[s][d] + a1 + a2;
        }
        rsum += rn;
      }
    }
    if (__builtin_expect(refresh && step >= 0, 0)) {
      // slots 2-3 of the scratch: waves may still read slots 0-1 above
      double none = 0.0;
      block_min_sum<B>(none, rsum, red + 2);
      residual = sqrt(rsum);
    }
    if (step >= 0) {
      bool stop = false;
      ++step;
      if (ramp) {
        stop = step >= a.n_steps;
      } else if (!(residual > a.tol)) {
        stop = true;
      } else if (step >= a.max_steps) {
        status = MF_STATUS_STEP_CAP;
        stop = true;
      }
      if (stop) break;
    } else {
      step = 0;
    }
    __syncthreads();  // every gather of the old positions is done
    drift64<B, NPT>(Nf, h, vr, pos);
    if (ramp) move_boundary64<B>(step + 1, S, rS, a.amplitude, Nf, Nb, pos, bst);
    __syncthreads();  // positions published
  }
  if (residual != residual) status = MF_STATUS_NAN;
  finalize64<B>(a, R, rv, sid, step, status, ramp, pos, bst, red);
}

// ============================================================================
// FP64 kernel with the state in global memory (any RVE size)
// ============================================================================
// The RVEs no LDS/register kernel holds (more free nodes than lanes, or
// positions beyond LDS).  Per node the arithmetic and its order are
// solve64's; positions (double-buffered), velocities and forces live in a
// per-solve global scratch, a.gstate + blockIdx.x * a.gstride doubles laid
// out [2][3][Np] positions, [3][Np] velocities, [3][Np] forces, and each
// thread loops over its free nodes r = tid, tid + B, ...  The workgroup
// barrier orders its waves' global accesses (one CU).  LDS keeps the
// reduction scratch, the boundary state and the reaction table.
template <int B>
__global__ __launch_bounds__(B) void solve64g(SolveArgs a) {
#pragma clang fp contract(off)
  constexpr int NW = B / kWave;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x;
  const int sid = a.order ? a.order[blockIdx.x] : (int)blockIdx.x;
  const int rv = a.solve_rve[sid];
  const RveDev R = a.rves[rv];
  const double eta_r = a.eta_rve ? a.eta_rve[rv] : a.eta;
  const int N = R.N, Nf = R.Nf, Nb = R.Nb, M = R.M;
  const int Np = (N + 1) & ~1, Nbp = (Nb + 1) & ~1;
  const int64_t nb = R.node_off;

  // LDS carve (mirrors lds_bytes)
  size_t off = 0;
  double *red = reinterpret_cast<double *>(smem);
  off += sizeof(double) * NW * kRedStride;
  double *bst = reinterpret_cast<double *>(smem + off);
  off += sizeof(double) * 6 * Nbp;
  Law64 *rxs = reinterpret_cast<Law64 *>(smem + off);
  // global state of this solve
  double *pos = a.gstate + (size_t)blockIdx.x * (size_t)a.gstride;  // [2][3][Np]
  double *gv = pos + 6 * (size_t)Np;                                // [3][Np]
  double *gf = gv + 3 * (size_t)Np;                                 // [3][Np]

  const int32_t *gw = a.ell_w + R.ell_off;
  const double *gl0 = a.ell_l0 + R.ell_off;
  if (tid < R.n_react) rxs[tid] = a.laws[R.react_off + tid];
  const bool lin_only =
      R.n_react == 1 && a.reacts[R.react_off].type == MF_REACTION_LINEAR;
  const Lin64 lin{a.reacts[R.react_off].E, a.reacts[R.react_off].A};

  double F[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) F[i] = a.solve_F[9 * (int64_t)sid + i];
  const bool ramp = a.mode == MF_MODE_RAMP;

  // ---- initial state (as solve64) -------------------------------------------
  for (int r = tid; r < N; r += B) {
    const int64_t g = nb + r;
    double xp[3], up[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      xp[d] = a.x_in[3 * g + d];
      up[d] = a.u_in[3 * g + d];
    }
    double inc[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      inc[k] = (F[3 * k + 0] - (k == 0 ? 1.0 : 0.0)) * xp[0] +
               (F[3 * k + 1] - (k == 1 ? 1.0 : 0.0)) * xp[1] +
               (F[3 * k + 2] - (k == 2 ? 1.0 : 0.0)) * xp[2];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double u = ramp ? up[k] : inc[k] + up[k];
      const double x = a.X[3 * g + k] + u;
      pos[k * Np + r] = x;
      pos[3 * Np + k * Np + r] = x;
      if (r < Nf) gv[k * Np + r] = 0.0;
    }
    if (r >= Nf) {
      const int b = r - Nf;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        bst[k * Nbp + b] = pos[k * Np + r];
        bst[(3 + k) * Nbp + b] = ramp ? inc[k] : 0.0;
      }
    }
  }
  __syncthreads();

  const double c_sound = R.c_sound;
  int cur = 0;
  // internal force at node r (free or boundary) from the positions in buffer
  // `buf`: the node's fibers in increasing fiber index
  auto node_force = [&](int r, int buf, double (&f)[3]) {
    const double *P = pos + buf * 3 * Np;
    const double x0 = P[r], x1 = P[Np + r], x2 = P[2 * Np + r];
    const int base = a.slice_base[R.slice_off + r / kWave] + (r & (kWave - 1));
    const int dg = a.deg[nb + r];
    double fx = 0.0, fy = 0.0, fz = 0.0;
    for (int j = 0; j < dg; ++j) {
      const int idx = base + j * kWave;
      const int32_t wv = gw[idx];
      const double l0 = gl0[idx];
      const int w = wv & 0xFFFFFF;
      const double dx = P[w] - x0;
      const double dy = P[Np + w] - x1;
      const double dz = P[2 * Np + w] - x2;
      const double l = sqrt(dx * dx + dy * dy + dz * dz);
      double frc;
      if (lin_only) {
        double lr = l / l0;
        double gs = 1.0 / 2.0 * (lr * lr - 1);
        frc = lr * lin.E * lin.A * gs;
      } else {
        frc = react64(rxs[(uint32_t)wv >> 24], l0, l);
      }
      const double t = frc / l;
      fx = fx - dx * t;
      fy = fy - dy * t;
      fz = fz - dz * t;
    }
    f[0] = fx;
    f[1] = fy;
    f[2] = fz;
  };
  auto min_length = [&](int buf) {
    const double *P = pos + buf * 3 * Np;
    double lmin = 1.0e300;
    const int32_t *fb = a.fib + 2 * R.fib_off;
    for (int e = tid; e < M; e += B) {
      const int n1 = fb[2 * e], n2 = fb[2 * e + 1];
      double x1 = P[n2] - P[n1];
      double x2 = P[Np + n2] - P[Np + n1];
      double x3 = P[2 * Np + n2] - P[2 * Np + n1];
      double l = sqrt(x1 * x1 + x2 * x2 + x3 * x3);
      lmin = l < lmin ? l : lmin;
    }
    return lmin;
  };

  // ---- RunInitialization (TeamOuterLoop.h:215-289) ---------------------------
  double resid_local = 0.0;
  for (int r = tid; r < Nf; r += B) {
    double fint[3];
    node_force(r, cur, fint);
    const double mr = a.mass[nb + r];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double mass = mr * eta_r;
      double fdamp = mass * gv[d * Np + r];
      gf[d * Np + r] = -fint[d] - fdamp;
    }
  }
  double lmin = min_length(cur);
  block_min_sum<B>(lmin, resid_local, red);
  double dt_crit = lmin / c_sound;

  // ---- main loop (TeamOuterLoop.h:340-371) -----------------------------------
  int step = 0;
  double residual = 10.0;
  int status = MF_STATUS_OK;
  const int freq = a.freq;
  for (;;) {
    const double h = a.crit * dt_crit * 0.5;
    const int nxt = cur ^ 1;
    const double *Pc = pos + cur * 3 * Np;
    double *Pn = pos + nxt * 3 * Np;
    // updates(): half kick + drift of free nodes (TeamOuterLoop.h:157-175)
    for (int r = tid; r < Nf; r += B) {
      const double mr = a.mass[nb + r];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double vl = gv[d * Np + r] + h * gf[d * Np + r] / mr;
        gv[d * Np + r] = vl;
        Pn[d * Np + r] = Pc[d * Np + r] + 2 * h * vl;
      }
    }
    if (ramp && tid < Nb) {
      const double alpha = ramp_alpha(step + 1, a.n_steps, a.amplitude);
      for (int b = tid; b < Nb; b += B) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
          Pn[d * Np + Nf + b] = bst[d * Nbp + b] + alpha * bst[(3 + d) * Nbp + b];
      }
    }
    __syncthreads();
    cur = nxt;
    const bool refresh = (step % freq) == 0;
    double rsum = 0.0;
    for (int r = tid; r < Nf; r += B) {
      double fint[3];
      node_force(r, cur, fint);
      const double mr = a.mass[nb + r];
      double rn = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double mass = mr * eta_r;
        double fdamp = mass * gv[d * Np + r];
        double lres = -fint[d];
        gf[d * Np + r] = lres - fdamp;
        rn += lres * lres;
      }
      rsum += rn;
    }
    if (refresh) {
      double lm = min_length(cur);
      block_min_sum<B>(lm, rsum, red);
      dt_crit = lm / c_sound;
      residual = sqrt(rsum);
    }
    // updateAccelVels(): second half kick (TeamOuterLoop.h:144-156)
    for (int r = tid; r < Nf; r += B) {
      const double mr = a.mass[nb + r];
#pragma unroll
      for (int d = 0; d < 3; ++d) gv[d * Np + r] += h * gf[d * Np + r] / mr;
    }
    ++step;
    if (ramp) {
      if (step >= a.n_steps) break;
    } else {
      if (!(residual > a.tol)) break;
      if (step >= a.max_steps) {
        status = MF_STATUS_STEP_CAP;
        break;
      }
    }
  }
  if (residual != residual) status = MF_STATUS_NAN;

  // ---- FinalizeData + computeCauchyStress (as solve64) ----------------------
  const double *P = pos + cur * 3 * Np;
  __syncthreads();
  double st[6] = {0, 0, 0, 0, 0, 0};
  const int flags = a.solve_flags[sid];
  const double alpha_end = ramp ? ramp_alpha(step, a.n_steps, a.amplitude) : 0.0;
  for (int b = tid; b < Nb; b += B) {
    const int r = Nf + b;
    double xb[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) xb[d] = bst[d * Nbp + b] + alpha_end * bst[(3 + d) * Nbp + b];
    const int base = a.slice_base[R.slice_off + r / kWave] + (r & (kWave - 1));
    const int dg = a.deg[nb + r];
    double f1 = 0.0, f2 = 0.0, f3 = 0.0;
    for (int j = 0; j < dg; ++j) {
      const int idx = base + j * kWave;
      const int32_t wv = gw[idx];
      const double l0 = gl0[idx];
      const int w = wv & 0xFFFFFF;
      const double dx = P[w] - xb[0];
      const double dy = P[Np + w] - xb[1];
      const double dz = P[2 * Np + w] - xb[2];
      const double l = sqrt(dx * dx + dy * dy + dz * dz);
      double frc;
      if (lin_only) {
        double lr = l / l0;
        double gs = 1.0 / 2.0 * (lr * lr - 1);
        frc = lr * lin.E * lin.A * gs;
      } else {
        frc = react64(rxs[(uint32_t)wv >> 24], l0, l);
      }
      const double t = frc / l;
      f1 = f1 - dx * t;
      f2 = f2 - dy * t;
      f3 = f3 - dz * t;
    }
    st[0] += xb[0] * f1;
    st[1] += xb[1] * f2;
    st[2] += xb[2] * f3;
    st[3] += 0.5 * (xb[1] * f3 + xb[2] * f2);
    st[4] += 0.5 * (xb[0] * f3 + xb[2] * f1);
    st[5] += 0.5 * (xb[0] * f2 + xb[1] * f1);
    if (flags & kWriteX)
      for (int d = 0; d < 3; ++d) a.x_out[3 * (nb + r) + d] = xb[d];
    if (flags & kWriteU)
      for (int d = 0; d < 3; ++d) a.u_out[3 * (nb + r) + d] = xb[d] - a.X[3 * (nb + r) + d];
  }
  // free nodes: u = x - X (TeamOuterLoop.h:427-432)
  for (int r = tid; r < Nf; r += B) {
    const int64_t g = nb + r;
    if (flags & kWriteX)
      for (int d = 0; d < 3; ++d) a.x_out[3 * g + d] = P[d * Np + r];
    if (flags & kWriteU)
      for (int d = 0; d < 3; ++d) a.u_out[3 * g + d] = P[d * Np + r] - a.X[3 * g + d];
  }
  block_sum<B, 6>(st, red);
  if (tid == 0) {
    const double sv = R.scale / a.V[rv];
    bool bad = false;
    for (int i = 0; i < 6; ++i) {
      double v = st[i] * sv;
      a.sigma[6 * (int64_t)sid + i] = v;
      bad = bad || !isfinite(v);
    }
    if (bad && status == MF_STATUS_OK) status = MF_STATUS_NAN;
    a.status[sid] = status;
    a.steps[sid] = step;
  }
}

}  // namespace kern

// shapes with their incidence lists in LDS (solve64l.hip)
hipError_t launch_solve64l(const Variant &v, const SolveArgs &a, int n_blocks, size_t lds,
                           hipStream_t s);

hipError_t launch_solve64(const Variant &v, const SolveArgs &a, int n_blocks,
                  size_t lds, hipStream_t s) {
  if (v.flags & kEllInLds) return launch_solve64l(v, a, n_blocks, lds, s);
#define MF_VARIANT_LAUNCH(P, B, N, F)                                        \
  if constexpr (P == MF_PREC_FP64 && !((F) & kEllInLds))                     \
    if (v.block == B && v.npt == N && (v.flags & ~kEnergy) == F) {          \
    auto k = (v.flags & kEnergy) ? kern::solve64<B, N, F, true>              \
                                 : kern::solve64<B, N, F, false>;            \
    if (lds > 64 * 1024)                                                     \
      (void)hipFuncSetAttribute((const void *)k,                             \
                                hipFuncAttributeMaxDynamicSharedMemorySize, \
                                (int)kMaxLds);                               \
    hipLaunchKernelGGL(k, dim3(n_blocks), dim3(B), lds, s, a);               \
    return hipGetLastError();                                                \
  }
  MF_VARIANT_LIST(MF_VARIANT_LAUNCH)
#undef MF_VARIANT_LAUNCH
#define MF_FONCE_LAUNCH(B, N, FPL, LIN)                                       \
  if (v.block == B && v.npt == N && v.flags == (kFiberOnce | ((LIN) ? kLinearOnly : 0))) { \
    auto k = kern::solve64f<B, N, FPL, LIN>;                                 \
    if (lds > 64 * 1024)                                                     \
      (void)hipFuncSetAttribute((const void *)k,                             \
                                hipFuncAttributeMaxDynamicSharedMemorySize, \
                                (int)kMaxLds);                               \
    hipLaunchKernelGGL(k, dim3(n_blocks), dim3(B), lds, s, a);               \
    return hipGetLastError();                                                \
  }
#define MF_FONCE_LAUNCH2(B, N, FPL) \
  MF_FONCE_LAUNCH(B, N, FPL, true)  \
  MF_FONCE_LAUNCH(B, N, FPL, false)
  MF_FONCE_LIST(MF_FONCE_LAUNCH2)
#undef MF_FONCE_LAUNCH2
#undef MF_FONCE_LAUNCH
#define MF_NODE64_LAUNCH(B, N)                                                \
  if (v.block == B && v.npt == N && v.flags == kFast64) {                    \
    auto k = kern::solve64n<B, N>;                                           \
    if (lds > 64 * 1024)                                                     \
      (void)hipFuncSetAttribute((const void *)k,                             \
                                hipFuncAttributeMaxDynamicSharedMemorySize, \
                                (int)kMaxLds);                               \
    hipLaunchKernelGGL(k, dim3(n_blocks), dim3(B), lds, s, a);               \
    return hipGetLastError();                                                \
  }
  MF_NODE64_LIST(MF_NODE64_LAUNCH)
#undef MF_NODE64_LAUNCH
#define MF_FONCE_L_LAUNCH(B, N)                                               \
  if (v.block == B && v.npt == N && v.flags == (kFiberOnce | kFast64)) {     \
    auto k = kern::solve64t<B, N>;                                           \
    if (lds > 64 * 1024)                                                     \
      (void)hipFuncSetAttribute((const void *)k,                             \
                                hipFuncAttributeMaxDynamicSharedMemorySize, \
                                (int)kMaxLds);                               \
    hipLaunchKernelGGL(k, dim3(n_blocks), dim3(B), lds, s, a);               \
    return hipGetLastError();                                                \
  }
  MF_TREC64_LIST(MF_FONCE_L_LAUNCH)
#undef MF_FONCE_L_LAUNCH
  if (v.block == 1024 && v.flags == kGlobalState) {
    auto k = kern::solve64g<1024>;
    if (lds > 64 * 1024)
      (void)hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)kMaxLds);
    hipLaunchKernelGGL(k, dim3(n_blocks), dim3(1024), lds, s, a);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}

}  // namespace mf
