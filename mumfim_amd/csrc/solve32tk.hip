// The tangent-linear kernels that gain where values stay where they are used
// instead of being moved out of the step loop: three directions per workgroup
// (64 toe-law RVEs of 1850 nodes, 200 steps: 3.04 -> 2.55 ms) and, of one
// direction, three nodes per lane (300 RVEs of 2600 nodes, half toe law 14.4 ->
// 13.4 ms, linear 12.6 -> 12.2 ms) and the two narrow shapes (8 RVEs of 200
// nodes, half toe law 0.82 -> 0.79 ms).  The others lose by it and are compiled
// without (solve32t.hip).
#include <type_traits>

#include "solve32t.hpp"

namespace mf {
namespace kern {

// ============================================================================
// Three directions per workgroup
// ============================================================================
// The base solve does not depend on the direction, so one workgroup carries
// kTlDirs of an RVE's six derivatives along it: neighbour records, reference
// vectors, stretch and reaction law of an incidence are evaluated once for
// three directions (~40 instructions), and each direction adds ~15 of its
// own, against ~55 for one direction alone.  The derivative rows of a node
// take two 16-byte LDS words and the spare word of its displacement, so a
// gather reads four words for three directions instead of three for one.
// Three is what a node's registers (10 + 6 per direction, up to three nodes
// per thread at 768 threads) and LDS (75 bytes per node, RVEs of up to ~2170
// nodes) hold; larger RVEs run the one-direction kernel.  Every rounding is
// that kernel's: the contractions its compilation chose are spelt out.
// 256 RVEs of 1000-2000 nodes, 800 steps: 27.4 ms with one direction per
// workgroup, 15.4 ms with three; the same bits.  768 threads (three waves per
// SIMD) rather than 1024: at 128 registers a lane this shape spills in the
// step loop and took 34.4 ms.
template <int B, int NPT>
__global__ __launch_bounds__(B)
__attribute__((amdgpu_waves_per_eu(B == 768 ? 3 : 4)))
void solve32tk(SolveArgs a) {
  constexpr int K = kTlDirs, NW = B / kWave;
  static_assert(K == 3, "the record layout holds three directions");
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  // solves sid, sid + 1, sid + 2: one RVE, consecutive directions
  const int sid = a.order ? a.order[blockIdx.x] : (int)blockIdx.x * K;
  if (!a.solve_G || !a.dsigma) {  // launched outside a tangent-linear set
    if (tid < K) {
      for (int i = 0; i < 6; ++i) a.sigma[6 * (int64_t)(sid + tid) + i] = __builtin_nan("");
      a.status[sid + tid] = MF_STATUS_NAN;
    }
    return;
  }
  const int rv = a.solve_rve[sid];
  const RveDev R = a.rves[rv];
  const int N = R.N, Nf = R.Nf, Nb = R.Nb, M = R.M;
  const int Np = (N + 1) & ~1, Nbp = (Nb + 1) & ~1;
  const int64_t nb = R.node_off;

  // LDS carve (mirrors lds_bytes).  Derivatives of directions 0, 1, 2:
  // dA = (0x 0y 0z 1x), dB = (1y 1z 2x 2y), pos.w = 2z
  size_t off = 0;
  float4 *pos = reinterpret_cast<float4 *>(smem);  // [Np] displacement hi, 2z
  off += sizeof(float4) * Np;
  float4 *dA = reinterpret_cast<float4 *>(smem + off);
  off += sizeof(float4) * Np;
  float4 *dB = reinterpret_cast<float4 *>(smem + off);
  off += sizeof(float4) * Np;
  int4 *Xs = reinterpret_cast<int4 *>(smem + off);  // [Np] reference X, fixed point
  off += sizeof(int4) * Np;
  double *red = reinterpret_cast<double *>(smem + off);
  off += sizeof(double) * NW * kRedStride;
  double *bst = reinterpret_cast<double *>(smem + off);  // [Nbp][6] u_b0, g
  off += sizeof(double) * 6 * Nbp;
  float *dbst = reinterpret_cast<float *>(smem + off);  // [Nbp][12] dg = G x_b
  off += sizeof(float) * 12 * Nbp;
  float4 *rtab = reinterpret_cast<float4 *>(smem + off);  // packed reaction table

  const int32_t *gw = a.ell_w + R.ell_off;
  const float *gil = a.ell_il + R.ell_off;
  // said to be uniform: otherwise every list load becomes a loop over lanes
  const int list_bytes =
      __builtin_amdgcn_readfirstlane(R.ell_free_entries) * (int)sizeof(int32_t);
  const __amdgpu_buffer_rsrc_t rsw =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t *>(gw), 0, list_bytes, kBufRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsil =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(gil), 0, list_bytes, kBufRsrcWord3);
  if (tid < R.n_react) pack_react_table(a.reacts[R.react_off + tid], rtab + kReactTabStride * tid);
  int nl_rid = -1;
  float ea_half_lin = 0.0f;
  const bool mix2 = mix2_table(a.reacts + R.react_off, R.n_react, nl_rid, ea_half_lin);
  const ReactDev nlq = a.reacts[R.react_off + (nl_rid < 0 ? 0 : nl_rid)];
  const bool lin_only =
      R.n_react == 1 && a.reacts[R.react_off].type == MF_REACTION_LINEAR;
  const float lin_EA_half = a.reacts[R.react_off].EA_half;
  const float eta = (float)(a.eta_rve ? a.eta_rve[rv] : a.eta);
  const double inv_S = 1.0 / a.n_steps;

  float uh[NPT][3], ul[NPT][3], vr[NPT][3], imr[NPT];
  float du[NPT][K][3], dv[NPT][K][3];
  // slice width and base (wave-uniform); Dn: with one linear and one
  // nonlinear reaction, entries [0, Dn) hold the wave's nonlinear fibers
  // (nodes list them first) and later entries are linear on every lane
  int Dr[NPT], sbase[NPT], Dn[NPT];
  {
    double F[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) F[i] = a.solve_F[9 * (int64_t)sid + i];
    for (int r = tid; r < N; r += B) {
      const int64_t g = nb + r;
      double xp[3], u[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        xp[d] = a.x_in[3 * g + d];
        u[d] = a.u_in[3 * g + d];
      }
      pos[r] = make_float4((float)u[0], (float)u[1], (float)u[2], 0.0f);
      dA[r] = dB[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      Xs[r] = make_int4((int)rint(a.X[3 * g] * R.xq_scale),
                        (int)rint(a.X[3 * g + 1] * R.xq_scale),
                        (int)rint(a.X[3 * g + 2] * R.xq_scale), 0);
      if (r >= Nf) {
        const int b = r - Nf;
        double inc[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
          inc[k] = (F[3 * k + 0] - (k == 0 ? 1.0 : 0.0)) * xp[0] +
                   (F[3 * k + 1] - (k == 1 ? 1.0 : 0.0)) * xp[1] +
                   (F[3 * k + 2] - (k == 2 ? 1.0 : 0.0)) * xp[2];
        bnd_set(bst + 6 * b, u, inc);
        for (int q = 0; q < K; ++q) {
          const double *G = a.solve_G + 9 * (int64_t)(sid + q);
          for (int k = 0; k < 3; ++k)
            dbst[12 * b + 3 * q + k] =
                (float)(G[3 * k + 0] * xp[0] + G[3 * k + 1] * xp[1] + G[3 * k + 2] * xp[2]);
        }
      }
    }
  }
#pragma unroll
  for (int s = 0; s < NPT; ++s) {
    const int r = s * B + tid;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double u = r < Nf ? a.u_in[3 * (nb + r) + d] : 0.0;
      uh[s][d] = (float)u;
      ul[s][d] = (float)(u - (double)uh[s][d]);
      vr[s][d] = 0.0f;
#pragma unroll
      for (int q = 0; q < K; ++q) du[s][q][d] = dv[s][q][d] = 0.0f;
    }
    imr[s] = r < Nf ? (float)(1.0 / a.mass[nb + r]) : 0.0f;
    const int k = s * NW + wave, sl = R.slice_off + k;  // slice of the wave's nodes
    Dr[s] = __builtin_amdgcn_readfirstlane(k * kWave < Nf ? a.slice_D[sl] : 0);
    sbase[s] = __builtin_amdgcn_readfirstlane(k * kWave < Nf ? a.slice_base[sl] : 0);
    int cnt = 0;
    if (mix2 && r < Nf) {
      const int dg = a.deg[nb + r];
      while (cnt < dg && (int)((uint32_t)gw[sbase[s] + lane + cnt * kWave] >> 24) == nl_rid) ++cnt;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cnt = max(cnt, __shfl_xor(cnt, o, kWave));
    Dn[s] = __builtin_amdgcn_readfirstlane(cnt);
  }
  __syncthreads();

  const float inv_c = (float)(1.0 / R.c_sound);
  const float xq_inv = R.xq_inv;
  auto rows = [&](int w, float w2z, float (&d)[K][3]) __attribute__((always_inline)) {
    const float4 A = ld16(dA + w), Bq = ld16(dB + w);
    d[0][0] = A.x;
    d[0][1] = A.y;
    d[0][2] = A.z;
    d[1][0] = A.w;
    d[1][1] = Bq.x;
    d[1][2] = Bq.y;
    d[2][0] = Bq.z;
    d[2][1] = Bq.w;
    d[2][2] = w2z;
  };
  auto put = [&](int r, float x, float y, float z, const float (&d)[K][3])
                 __attribute__((always_inline)) {
    pos[r] = make_float4(x, y, z, d[2][2]);
    dA[r] = make_float4(d[0][0], d[0][1], d[0][2], d[1][0]);
    dB[r] = make_float4(d[1][1], d[1][2], d[2][0], d[2][1]);
  };
  // internal force of a slot's node and its derivatives (ELL padding names
  // the node itself with 1/l0 = 0: zero force, zero derivatives)
  auto node_force = [&](int s, float (&f)[3], float (&df)[K][3]) __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      f[d] = 0.0f;
#pragma unroll
      for (int q = 0; q < K; ++q) df[q][d] = 0.0f;
    }
    const int D = Dr[s];
    if (D <= 0) return;
    const int4 Xv = ld16(Xs + s * B + tid);
    const int vo = (sbase[s] + lane) * (int)sizeof(int32_t), Dm = D - 1;
    auto entry = [&](int jj, int32_t &wv, float &il) __attribute__((always_inline)) {
      const int so = jj * (kWave * (int)sizeof(int32_t));
      wv = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(rsw, vo, so, 0);
      il = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsil, vo, so, 0));
    };
    int32_t wv_n, wv_nn;
    float il_n, il_nn;
    entry(0, wv_n, il_n);
    entry(min(1, Dm), wv_nn, il_nn);
    // entries [j0, j1) under one law, chosen outside the loop
    auto run = [&](int j0, int j1, auto LAWC) __attribute__((always_inline)) {
      constexpr int LAW = decltype(LAWC)::value;
#pragma clang loop unroll(disable)
      for (int j = j0; j < j1; ++j) {
        const int32_t wv = wv_n;
        const float il = il_n;
        wv_n = wv_nn;
        il_n = il_nn;
        entry(min(j + 2, Dm), wv_nn, il_nn);
        const int w = wv & 0xFFFFFF;
        const float4 q4 = ld16(pos + w);
        const int4 xq = ld16(Xs + w);
        float dw[K][3];
        rows(w, q4.w, dw);
        const float cx = (float)(xq.x - Xv.x), cy = (float)(xq.y - Xv.y),
                    cz = (float)(xq.z - Xv.z);
        const float gx = (q4.x - uh[s][0]) - ul[s][0];
        const float gy = (q4.y - uh[s][1]) - ul[s][1];
        const float gz = (q4.z - uh[s][2]) - ul[s][2];
        const float dx = fmaf(xq_inv, cx, gx), dy = fmaf(xq_inv, cy, gy),
                    dz = fmaf(xq_inv, cz, gz);
        // l^2 - l0^2 = (d0 + d) . delta
        const float sl = fmaf(gz, fmaf(xq_inv, cz, dz),
                              fmaf(gx, fmaf(xq_inv, cx, dx), gy * fmaf(xq_inv, cy, dy)));
        const float il2 = il * il, e2 = sl * il2;
        float t, dt;
        if (LAW == kLawLin) {
          dt = lin_EA_half * il;
          t = dt * e2;
        } else if (LAW == kLawMixLin) {
          dt = ea_half_lin * il;
          t = dt * e2;
        } else if (LAW == kLawMixNl) {
          t = react32_mix2_dt(nlq, ea_half_lin, (int)((uint32_t)wv >> 24) == nl_rid, e2, il, dt);
        } else {
          t = react32_tab_dt(rtab, (uint32_t)wv >> 24, e2, il, dt);
        }
        f[0] = fmaf(-dx, t, f[0]);
        f[1] = fmaf(-dy, t, f[1]);
        f[2] = fmaf(-dz, t, f[2]);
#pragma unroll
        for (int q = 0; q < K; ++q) {
          // d(l^2 - l0^2) = 2 d . dd
          const float ddx = dw[q][0] - du[s][q][0], ddy = dw[q][1] - du[s][q][1],
                      ddz = dw[q][2] - du[s][q][2];
          const float dot = fmaf(ddz, dz, fmaf(ddx, dx, ddy * dy));
          const float dtt = il2 * (dot + dot) * dt;
          df[q][0] = df[q][0] - fmaf(ddx, t, dx * dtt);
          df[q][1] = df[q][1] - fmaf(ddy, t, dy * dtt);
          df[q][2] = df[q][2] - fmaf(ddz, t, dz * dtt);
        }
      }
    };
    if (lin_only) {
      run(0, D, std::integral_constant<int, kLawLin>{});
    } else if (mix2) {
      const int dn = min(Dn[s], D);
      run(0, dn, std::integral_constant<int, kLawMixNl>{});
      run(dn, D, std::integral_constant<int, kLawMixLin>{});
    } else {
      run(0, D, std::integral_constant<int, kLawTab>{});
    }
  };
  // shortest fiber's l^2 (lowest index on ties) and its derivatives
  auto min_length2 = [&](float (&dl2)[K]) {
    float lmin = 3.0e38f, none = 0.0f;
    int imin = 0x7FFFFFFF;
    const int32_t *fb = a.fib + 2 * R.fib_off;
    auto vec = [&](int e, float &x1, float &x2, float &x3) {
      const int n1 = fb[2 * e], n2 = fb[2 * e + 1];
      const float4 p1 = pos[n1], p2 = pos[n2];
      const int4 X1 = Xs[n1], X2 = Xs[n2];
      x1 = fmaf(xq_inv, (float)(X2.x - X1.x), p2.x - p1.x);
      x2 = fmaf(xq_inv, (float)(X2.y - X1.y), p2.y - p1.y);
      x3 = fmaf(xq_inv, (float)(X2.z - X1.z), p2.z - p1.z);
    };
    for (int e = tid; e < M; e += B) {
      float x1, x2, x3;
      vec(e, x1, x2, x3);
      const float l2 = fmaf(x3, x3, fmaf(x1, x1, x2 * x2));
      if (l2 < lmin) {  // fibers visited in increasing index per thread
        lmin = l2;
        imin = e;
      }
    }
    block_argmin<B>(lmin, imin, none, red);
#pragma unroll
    for (int q = 0; q < K; ++q) dl2[q] = 0.0f;
    if (imin < M) {
      float x1, x2, x3, d1[K][3], d2[K][3];
      vec(imin, x1, x2, x3);
      const int n1 = fb[2 * imin], n2 = fb[2 * imin + 1];
      rows(n1, pos[n1].w, d1);
      rows(n2, pos[n2].w, d2);
#pragma unroll
      for (int q = 0; q < K; ++q) {
        const float d = fmaf(x3, d2[q][2] - d1[q][2],
                             fmaf(x2, d2[q][1] - d1[q][1], x1 * (d2[q][0] - d1[q][0])));
        dl2[q] = d + d;
      }
    }
    return lmin;
  };

  const float crit_half = (float)(a.crit * 0.5);
  // h = crit/2 sqrt(l2) / c and dh = crit/2 dl2 / (2 sqrt(l2) c)
  auto step_size = [&](float l2, const float (&dl2)[K], float (&dh)[K]) {
    const float l = sqrtf(l2);
#pragma unroll
    for (int q = 0; q < K; ++q) dh[q] = crit_half * (0.5f * dl2[q] / l) * inv_c;
    return crit_half * (l * inv_c);
  };
  // Both half kicks between two drifts use one acceleration: v += (h_k +
  // h_{k+1}) a.  The first pass (step -1) kicks with h_0 alone.
  float h_prev = 0.0f, dh_prev[K] = {0.0f, 0.0f, 0.0f};
  int step = -1, due = 0;
  double residual = 10.0;
  const int freq = a.freq;
  for (;;) {
    const bool refresh = step < 0 || step == due;
    float h = h_prev, dh[K];
#pragma unroll
    for (int q = 0; q < K; ++q) dh[q] = dh_prev[q];
    if (__builtin_expect(refresh, 0)) {
      if (step >= 0) due += freq;
      float dl2[K];
      const float l2 = min_length2(dl2);
      h = step_size(l2, dl2, dh);
    }
    const float hk = h_prev + h;
    float dhk[K];
#pragma unroll
    for (int q = 0; q < K; ++q) dhk[q] = dh_prev[q] + dh[q];
    double rsum = 0.0;
#pragma unroll
    for (int s = 0; s < NPT; ++s) {
      if (s * B + tid < Nf) {
        float f[3], df[K][3];
        node_force(s, f, df);
        if (refresh) rsum += (double)dot3f(f[0], f[1], f[2], f[0], f[1], f[2]);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const float acc = fmaf(imr[s], -f[d], -(vr[s][d] * eta));
          vr[s][d] = fmaf(hk, acc, vr[s][d]);
#pragma unroll
          for (int q = 0; q < K; ++q) {
            const float dacc = fmaf(imr[s], -df[q][d], -(dv[s][q][d] * eta));
            dv[s][q][d] = dv[s][q][d] + fmaf(dhk[q], acc, hk * dacc);
          }
        }
      }
    }
    if (__builtin_expect(refresh && step >= 0, 0)) {
      double none = 0.0;
      block_min_sum<B>(none, rsum, red + 4);
      residual = sqrt(rsum);
    }
    h_prev = h;
#pragma unroll
    for (int q = 0; q < K; ++q) dh_prev[q] = dh[q];
    if (++step >= a.n_steps) break;
    __syncthreads();  // every read of the last step's positions done
    const float h2 = h_prev + h_prev;
#pragma unroll
    for (int s = 0; s < NPT; ++s) {
      const int r = s * B + tid;
      if (r < Nf) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const float y = fmaf(h2, vr[s][d], ul[s][d]);
          const float sh = uh[s][d] + y;
          ul[s][d] = y - (sh - uh[s][d]);
          uh[s][d] = sh;
#pragma unroll
          for (int q = 0; q < K; ++q)
            du[s][q][d] = du[s][q][d] +
                          fmaf(dh_prev[q] + dh_prev[q], vr[s][d], h2 * dv[s][q][d]);
        }
        put(r, uh[s][0], uh[s][1], uh[s][2], du[s]);
      }
    }
    if (tid < Nb) {
      const double alpha = ramp_alpha_step(step + 1, inv_S, a.amplitude);
      const float af = (float)alpha;
      for (int b = tid; b < Nb; b += B) {
        float ub[3], d[K][3];
        bnd_step(bst + 6 * b, alpha, ub);
#pragma unroll
        for (int i = 0; i < 3 * K; ++i) d[i / 3][i % 3] = dbst[12 * b + i] * af;
        put(Nf + b, ub[0], ub[1], ub[2], d);
      }
    }
    __syncthreads();
  }
  int status = residual != residual ? MF_STATUS_NAN : MF_STATUS_OK;

  const double alpha_end = ramp_alpha(step, a.n_steps, a.amplitude);
  const int flags = a.solve_flags[sid];  // the first solve's; the others commit nothing
  __syncthreads();  // every read of the step's positions done
  for (int b = tid; b < Nb; b += B) {
    double ub[3];
    float d[K][3];
    bnd_disp(bst + 6 * b, alpha_end, ub);
    const float af = (float)alpha_end;
    for (int i = 0; i < 3 * K; ++i) d[i / 3][i % 3] = dbst[12 * b + i] * af;
    put(Nf + b, (float)ub[0], (float)ub[1], (float)ub[2], d);
  }
  __syncthreads();
  // boundary force of the node and its derivative along direction q (none:
  // q < 0), one direction at a time: d sigma = s/V sum_b sym(dx_b (x) f_b +
  // x_b (x) df_b) from the hi parts and the derivatives, sigma from the full
  // displacements (lb, Pl: low parts, or null)
  auto row = [&](int r, float w2z, int q, float (&d)[3]) __attribute__((always_inline)) {
    const float4 A = ld16(dA + r), Bq = ld16(dB + r);
    d[0] = q == 0 ? A.x : q == 1 ? A.w : Bq.z;
    d[1] = q == 0 ? A.y : q == 1 ? Bq.x : Bq.w;
    d[2] = q == 0 ? A.z : q == 1 ? Bq.y : w2z;
  };
  auto bgather = [&](int r, const float4 hb, const float4 lb, const float4 *Pl, int q,
                     float (&f)[3], float (&df)[3]) __attribute__((always_inline)) {
    const int4 Xb = Xs[r];
    float db[3];
    row(r, hb.w, q, db);
    const int base = a.slice_base[R.slice_off + r / kWave] + (r & (kWave - 1));
    const int dg = a.deg[nb + r];
    for (int d = 0; d < 3; ++d) f[d] = df[d] = 0.0f;
    for (int j = 0; j < dg; ++j) {
      const int idx = base + j * kWave;
      const int32_t wv = gw[idx];
      const float il = gil[idx];
      const int w = wv & 0xFFFFFF;
      const float4 qh = pos[w];
      const float4 ql = Pl ? Pl[w] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      const int4 xq = Xs[w];
      const float cx = (float)(xq.x - Xb.x), cy = (float)(xq.y - Xb.y), cz = (float)(xq.z - Xb.z);
      const float gx = (qh.x - hb.x) + (ql.x - lb.x);
      const float gy = (qh.y - hb.y) + (ql.y - lb.y);
      const float gz = (qh.z - hb.z) + (ql.z - lb.z);
      const float dx = fmaf(xq_inv, cx, gx), dy = fmaf(xq_inv, cy, gy), dz = fmaf(xq_inv, cz, gz);
      const float sl = fmaf(gz, fmaf(xq_inv, cz, dz),
                            fmaf(gx, fmaf(xq_inv, cx, dx), gy * fmaf(xq_inv, cy, dy)));
      const float il2 = il * il, e2 = sl * il2;
      const unsigned rid = (uint32_t)wv >> 24;
      float t, dt;
      if (lin_only) {
        dt = lin_EA_half * il;
        t = dt * e2;
      } else {
        t = mix2 ? react32_mix2_dt(nlq, ea_half_lin, (int)rid == nl_rid, e2, il, dt)
                 : react32_tab_dt(rtab, rid, e2, il, dt);
      }
      f[0] = fmaf(-dx, t, f[0]);
      f[1] = fmaf(-dy, t, f[1]);
      f[2] = fmaf(-dz, t, f[2]);
      if (!Pl) {
        float dw[3];
        row(w, qh.w, q, dw);
        const float ddx = dw[0] - db[0], ddy = dw[1] - db[1], ddz = dw[2] - db[2];
        const float dot = fmaf(ddz, dz, fmaf(ddx, dx, ddy * dy));
        const float dtt = (dt + dt) * dot * il2;
        df[0] = df[0] - fmaf(ddx, t, dx * dtt);
        df[1] = df[1] - fmaf(ddy, t, dy * dtt);
        df[2] = df[2] - fmaf(ddz, t, dz * dtt);
      }
    }
  };
  const double sv = R.scale / a.V[rv];
  int badq = 0;  // directions with a derivative that is not finite
#pragma clang loop unroll(disable)
  for (int q = 0; q < K; ++q) {
    double ds[6] = {0, 0, 0, 0, 0, 0};
    for (int b = tid; b < Nb; b += B) {
      const int r = Nf + b;
      double ub[3], xb[3];
      bnd_disp(bst + 6 * b, alpha_end, ub);
      for (int d = 0; d < 3; ++d) xb[d] = a.X[3 * (nb + r) + d] + ub[d];
      float f[3], df[3], db[3];
      const float4 hb = pos[r];
      row(r, hb.w, q, db);
      bgather(r, hb, make_float4(0.0f, 0.0f, 0.0f, 0.0f), nullptr, q, f, df);
      const double fb[3] = {f[0], f[1], f[2]};
      const double dxb[3] = {db[0], db[1], db[2]}, dfb[3] = {df[0], df[1], df[2]};
      ds[0] += dxb[0] * fb[0] + xb[0] * dfb[0];
      ds[1] += dxb[1] * fb[1] + xb[1] * dfb[1];
      ds[2] += dxb[2] * fb[2] + xb[2] * dfb[2];
      ds[3] += 0.5 * (dxb[1] * fb[2] + xb[1] * dfb[2] + dxb[2] * fb[1] + xb[2] * dfb[1]);
      ds[4] += 0.5 * (dxb[0] * fb[2] + xb[0] * dfb[2] + dxb[2] * fb[0] + xb[2] * dfb[0]);
      ds[5] += 0.5 * (dxb[0] * fb[1] + xb[0] * dfb[1] + dxb[1] * fb[0] + xb[1] * dfb[0]);
    }
    block_sum_lane0<B, 6>(ds, red);
    if (tid == 0)
      for (int i = 0; i < 6; ++i) {
        const double w = ds[i] * sv;
        a.dsigma[6 * (int64_t)(sid + q) + i] = w;
        badq |= !isfinite(w) ? 1 << q : 0;
      }
    __syncthreads();  // thread 0 has read red
  }
  __syncthreads();  // the derivative rows are free: dA takes the low parts
  float4 *Pl = dA;
#pragma unroll
  for (int s = 0; s < NPT; ++s) {
    const int r = s * B + tid;
    if (r < Nf) Pl[r] = make_float4(ul[s][0], ul[s][1], ul[s][2], 0.0f);
  }
  for (int b = tid; b < Nb; b += B) {
    double ub[3];
    bnd_disp(bst + 6 * b, alpha_end, ub);
    const float4 hb = pos[Nf + b];
    Pl[Nf + b] = make_float4((float)(ub[0] - (double)hb.x), (float)(ub[1] - (double)hb.y),
                             (float)(ub[2] - (double)hb.z), 0.0f);
  }
  __syncthreads();
  double st[6] = {0, 0, 0, 0, 0, 0};
  for (int b = tid; b < Nb; b += B) {
    const int r = Nf + b;
    double ub[3], xb[3];
    bnd_disp(bst + 6 * b, alpha_end, ub);
    for (int d = 0; d < 3; ++d) xb[d] = a.X[3 * (nb + r) + d] + ub[d];
    float f[3], df[3];
    bgather(r, pos[r], Pl[r], Pl, 0, f, df);
    const double g1 = f[0], g2 = f[1], g3 = f[2];
    st[0] += xb[0] * g1;
    st[1] += xb[1] * g2;
    st[2] += xb[2] * g3;
    st[3] += 0.5 * (xb[1] * g3 + xb[2] * g2);
    st[4] += 0.5 * (xb[0] * g3 + xb[2] * g1);
    st[5] += 0.5 * (xb[0] * g2 + xb[1] * g1);
    if (flags & kWriteX)
      for (int d = 0; d < 3; ++d) a.x_out[3 * (nb + r) + d] = xb[d];
    if (flags & kWriteU)
      for (int d = 0; d < 3; ++d) a.u_out[3 * (nb + r) + d] = ub[d];
  }
#pragma unroll
  for (int s = 0; s < NPT; ++s) {
    const int r = s * B + tid;
    if (r < Nf) {
      const int64_t g = nb + r;
      for (int d = 0; d < 3; ++d) {
        const double u = (double)uh[s][d] + (double)ul[s][d];
        if (flags & kWriteX) a.x_out[3 * g + d] = a.X[3 * g + d] + u;
        if (flags & kWriteU) a.u_out[3 * g + d] = u;
      }
    }
  }
  block_sum_lane0<B, 6>(st, red);
  if (tid == 0) {
    bool bad = false;
    for (int i = 0; i < 6; ++i) {
      st[i] = st[i] * sv;
      bad = bad || !isfinite(st[i]);
    }
    for (int q = 0; q < K; ++q) {
      for (int i = 0; i < 6; ++i) a.sigma[6 * (int64_t)(sid + q) + i] = st[i];
      a.status[sid + q] =
          (bad || (badq >> q & 1)) && status == MF_STATUS_OK ? MF_STATUS_NAN : status;
      a.steps[sid + q] = step;
    }
  }
}

}  // namespace kern

hipError_t launch_solve32tk(const Variant &v, const SolveArgs &a, int n_blocks, size_t lds,
                            hipStream_t s) {
#define MF_TLK_LAUNCH(K, B, N, DIRS)                                         \
  if (v.block == B && v.npt == N && variant_fpl(v.flags) == DIRS) {          \
    auto k = kern::K<B, N>;                                                  \
    if (lds > 64 * 1024)                                                     \
      (void)hipFuncSetAttribute((const void *)k,                             \
                                hipFuncAttributeMaxDynamicSharedMemorySize, \
                                (int)kMaxLds);                               \
    hipLaunchKernelGGL(k, dim3(n_blocks), dim3(B), lds, s, a);               \
    return hipGetLastError();                                                \
  }
#define MF_TLK_LAUNCH3(B, N) MF_TLK_LAUNCH(solve32tk, B, N, kTlDirs)
#define MF_TLK_LAUNCH1(B, N) MF_TLK_LAUNCH(solve32t, B, N, 0)
  MF_TLK_LIST(MF_TLK_LAUNCH3)
  MF_TL_K_LIST(MF_TLK_LAUNCH1)
#undef MF_TLK_LAUNCH1
#undef MF_TLK_LAUNCH3
#undef MF_TLK_LAUNCH
  return hipErrorInvalidValue;
}

}  // namespace mf
