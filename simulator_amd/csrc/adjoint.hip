// adjoint.hip -- reverse-mode gradient of a cloth rollout on gfx950.
//
// The forward is the plain fused step (k_verlet) with the parameters under
// study: stiffness of the three spring types, the velocity damping and the
// rest-length scale; the initial state is x_cur = x0, x_prev = x0 - v0 dt.
// The backward differentiates that step with the contacts of the forward
// held fixed: a vertex projected in a step is moved by the fixed plane
// projection (I - n n^T) u + (n . a) n, and the contact normal entering the
// next step's force projection F - (c . F) c is a constant.
//
// Per step (state x = (P, Q) -> (P', Q'), adjoints lP', lQ' -> lP, lQ):
//   u = 2P - Q + w (I - c c^T) F(P, Q),  w = dt^2 / m
//   free vertex:      P' = u, Q' = P          -> lu = lP',  lP += lQ'
//   projected vertex: P' = Q' = Pi(u)         -> lu = (I - n n^T)(lP' + lQ')
//   pinned vertex:    P' = Q' = P             -> lP += lP' + lQ'
//   lP += 2 lu, lQ -= lu, lF = w (I - c c^T) lu,
//   F = g m + damp v + sum_j f(d, dv), v = (P - Q)/dt, d = P_i - P_j + eps,
//   f = alpha d/L, alpha = -k (L - rest) + kd (dv . d)/L.
// A step back has two parts: the force part (lu, lF and the vertex-local terms;
// no neighbour needed) and the spring part (the spring terms, gathered per
// vertex: for a spring i->j the side of f_ij weighted by lF_i and, by the
// symmetry of the spring set (checked at creation), the side of f_ji weighted
// by lF_j).  One launch takes the spring part of step t and the force part of
// step t - 1, which needs only what this vertex has just finished
// (k_adj_step); k_adj_force opens a run of steps.
//
// A trajectory of up to keep_limit() bytes keeps every state of the forward, and
// the backward steps through them.  A longer one keeps checkpoints every
// `ckpt` steps; each segment is recomputed forward with its per-step states
// kept, then stepped back.  The states are the same either way.  Parameter
// gradients: FP32 sums per step and block of 256 vertices, accumulated per
// block in FP64 (k_adj_acc), reduced in FP64 on the GPU at the end.
#include <cstdlib>
#include <cstring>
#include <memory>

#include "cc_device.h"
#include "cc_sim.h"

namespace cc {

constexpr int ADJ_THREADS = 256;
constexpr int NPARAM = 5;   // k0, k1, k2, damp, rest_scale
// All states of a rollout are kept up to this size (36 bytes per vertex and
// step): 128 x 128 vertices over 200 steps take 118 MB, and recomputing them
// took 1.1 of the 3.6 ms of their backward.  1 GiB is a 1/288 of the card; a
// program that holds many handles, or little memory, sets CC_ADJ_KEEP_MB.
constexpr size_t ADJ_KEEP_MB = 1024;
static size_t keep_limit() {
  const char* e = std::getenv("CC_ADJ_KEEP_MB");
  return (e ? (size_t)std::clamp(std::atoll(e), 0ll, 1ll << 30) : ADJ_KEEP_MB) << 20;
}

struct AdjArgs {
  float dt, inv_dt, w, damp, kd, k0, k1, k2, rest_scale, eps;
};

// Vector-Jacobian product of one spring force with the weight lam:
// gd = (df/dd)^T lam, gdv = (df/ddv)^T lam, dl = (d/L) . lam.
__device__ inline void spring_vjp(f3 d, f3 dv, float ks, float rest, float kd, f3 lam, f3& gd, f3& gdv,
                                  float& dl, float& L) {
  L = sqrtf(fmaf(d.z, d.z, fmaf(d.y, d.y, d.x * d.x)));
  const float il = 1.0f / L;
  const f3 u = mk(d.x * il, d.y * il, d.z * il);
  const float ud = fmaf(u.z, dv.z, fmaf(u.y, dv.y, u.x * dv.x));
  const float alpha = fmaf(-ks, L - rest, kd * ud);
  const float l = fmaf(u.z, lam.z, fmaf(u.y, lam.y, u.x * lam.x));
  const float kl = kd * il;
  // d alpha / d d = -ks u + kd (dv - (u . dv) u) / L;  d u / d d = (I - u u^T) / L
  const f3 da = mk(fmaf(-ks, u.x, kl * fmaf(-ud, u.x, dv.x)), fmaf(-ks, u.y, kl * fmaf(-ud, u.y, dv.y)),
                   fmaf(-ks, u.z, kl * fmaf(-ud, u.z, dv.z)));
  const float al = alpha * il;
  gd = mk(fmaf(da.x, l, al * fmaf(-u.x, l, lam.x)), fmaf(da.y, l, al * fmaf(-u.y, l, lam.y)),
          fmaf(da.z, l, al * fmaf(-u.z, l, lam.z)));
  gdv = mk(u.x * (kd * l), u.y * (kd * l), u.z * (kd * l));
  dl = l;
}

// Sum over a wave of 64 vertices (one per lane), valid in lane 0.
template <int K>
__device__ inline void wave_sum(float (&v)[K]) {
#pragma unroll
  for (int k = 0; k < K; ++k)
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_down(v[k], off, 64);
}

// The force part of a step for one vertex: its adjoint lP, lQ after the step,
// the contact normals before (c) and after (nn) it, its state s before it.
struct AdjForce {
  f3 lF, gp, gq;     // lF, and the vertex-local terms of lP, lQ before the step
  float damp;        // lF . vel
};
__device__ inline AdjForce adj_force(f3 lP, f3 lQ, bool pinned, f3 c, f3 nn, f3 sp, f3 sq, const AdjArgs& a) {
  AdjForce r{mk(0.0f, 0.0f, 0.0f), mk(0.0f, 0.0f, 0.0f), mk(0.0f, 0.0f, 0.0f), 0.0f};
  if (pinned) {
    r.gp = lP + lQ;
    return r;
  }
  f3 lu;
  if (nn.x != 0.0f || nn.y != 0.0f || nn.z != 0.0f) {
    const f3 s2 = lP + lQ;
    const float ns = fmaf(nn.z, s2.z, fmaf(nn.y, s2.y, nn.x * s2.x));
    lu = mk(fmaf(-nn.x, ns, s2.x), fmaf(-nn.y, ns, s2.y), fmaf(-nn.z, ns, s2.z));
  } else {
    lu = lP;
    r.gp = lQ;
  }
  r.gp = mk(fmaf(2.0f, lu.x, r.gp.x), fmaf(2.0f, lu.y, r.gp.y), fmaf(2.0f, lu.z, r.gp.z));
  r.gq = mk(-lu.x, -lu.y, -lu.z);
  const float cl = fmaf(c.z, lu.z, fmaf(c.y, lu.y, c.x * lu.x));
  r.lF = mk(a.w * fmaf(-c.x, cl, lu.x), a.w * fmaf(-c.y, cl, lu.y), a.w * fmaf(-c.z, cl, lu.z));
  const f3 vel = mk((sp.x - sq.x) * a.inv_dt, (sp.y - sq.y) * a.inv_dt, (sp.z - sq.z) * a.inv_dt);
  r.damp = fmaf(r.lF.z, vel.z, fmaf(r.lF.y, vel.y, r.lF.x * vel.x));   // F += damp * vel
  const float dd = a.damp * a.inv_dt;
  r.gp = mk(fmaf(dd, r.lF.x, r.gp.x), fmaf(dd, r.lF.y, r.gp.y), fmaf(dd, r.lF.z, r.gp.z));
  r.gq = mk(fmaf(-dd, r.lF.x, r.gq.x), fmaf(-dd, r.lF.y, r.gq.y), fmaf(-dd, r.lF.z, r.gq.z));
  return r;
}

__global__ __launch_bounds__(ADJ_THREADS) void k_adj_force(
    uint32_t n, const uint32_t* __restrict__ row, const float* __restrict__ state,
    const float* __restrict__ c_in, const float* __restrict__ c_out, const float* __restrict__ lp,
    const float* __restrict__ lq, AdjArgs a, float* __restrict__ lf, float* __restrict__ locp,
    float* __restrict__ locq, float* __restrict__ part) {
  const uint32_t i = blockIdx.x * ADJ_THREADS + threadIdx.x;
  float g[1] = {0.0f};
  if (i < n) {
    const size_t o = 3 * (size_t)i;
    const AdjForce r = adj_force(ld3(lp + o), ld3(lq + o), (row[i] & PIN_BIT) != 0, ld3(c_in + o), ld3(c_out + o),
                                 ld3(state + 2 * o), ld3(state + 2 * o + 3), a);
    st3(lf + o, r.lF);
    st3(locp + o, r.gp);
    st3(locq + o, r.gq);
    g[0] = r.damp;
  }
  wave_sum(g);
  if ((threadIdx.x & 63u) == 0 && i < n) part[NPARAM * (size_t)(i >> 6) + 3] = g[0];
}

// One spring's adjoint terms (the forward's f_ij in F_i and f_ji in F_j):
// gp += a1, gq -= v1 / dt, gp -= a2, gq += v2 / dt, in that order, and its
// parts gk0 .. gk2 (its type's, the others 0) and gr of the gradients of the
// stiffnesses and of rest_scale.  All zero for an empty slot.
struct AdjTerm {
  f3 a1, v1, a2, v2;
  float gk0, gk1, gk2, gr;
};
__device__ inline AdjTerm adj_spring(f3 pi, f3 vi, f3 lFi, f3 pj, f3 vj, f3 lFj, uint2 r, bool real,
                                     const AdjArgs& a, float ks0, float ks1, float ks2) {
  AdjTerm o;
  const uint32_t ty = r.x >> 30;
  const float rest0 = __uint_as_float(r.y), rest = rest0 * a.rest_scale;
  const float ks = ty == 0 ? ks0 : (ty == 1 ? ks1 : ks2);
  f3 gd;
  float dl, L;
  // f_ij, in F_i
  spring_vjp(mk((pi.x - pj.x) + a.eps, (pi.y - pj.y) + a.eps, (pi.z - pj.z) + a.eps), vi - vj, ks, rest, a.kd, lFi,
             gd, o.v1, dl, L);
  o.a1 = mk(fmaf(o.v1.x, a.inv_dt, gd.x), fmaf(o.v1.y, a.inv_dt, gd.y), fmaf(o.v1.z, a.inv_dt, gd.z));
  const float gk = -(L - rest) * dl;
  o.gr = ks * rest0 * dl;
  // f_ji, in F_j (the same type and rest length)
  spring_vjp(mk((pj.x - pi.x) + a.eps, (pj.y - pi.y) + a.eps, (pj.z - pi.z) + a.eps), vj - vi, ks, rest, a.kd, lFj,
             gd, o.v2, dl, L);
  o.a2 = mk(fmaf(o.v2.x, a.inv_dt, gd.x), fmaf(o.v2.y, a.inv_dt, gd.y), fmaf(o.v2.z, a.inv_dt, gd.z));
  // by a mask and not by a select, as in spring_scale
  uint32_t keep = real ? ~0u : 0u;
  asm("" : "+v"(keep));
  auto masked = [keep](float v) { return __uint_as_float(__float_as_uint(v) & keep); };
  auto masked3 = [&](f3 v) { return mk(masked(v.x), masked(v.y), masked(v.z)); };
  o.a1 = masked3(o.a1);
  o.v1 = masked3(o.v1);
  o.a2 = masked3(o.a2);
  o.v2 = masked3(o.v2);
  o.gr = masked(o.gr);
  o.gk0 = masked(ty == 0 ? gk : 0.0f);
  o.gk1 = masked(ty == 1 ? gk : 0.0f);
  o.gk2 = masked(ty == 2 ? gk : 0.0f);
  return o;
}
// Its sum into gp, gq and the parameter gradients g = {k0, k1, k2, -, rest_scale}.
__device__ inline void adj_add(const AdjTerm& o, float inv_dt, f3& gp, f3& gq, float (&g)[NPARAM]) {
  gp = gp + o.a1;
  gq = mk(fmaf(-o.v1.x, inv_dt, gq.x), fmaf(-o.v1.y, inv_dt, gq.y), fmaf(-o.v1.z, inv_dt, gq.z));
  g[0] += o.gk0;
  g[1] += o.gk1;
  g[2] += o.gk2;
  g[4] += o.gr;
  gp = gp - o.a2;
  gq = mk(fmaf(o.v2.x, inv_dt, gq.x), fmaf(o.v2.y, inv_dt, gq.y), fmaf(o.v2.z, inv_dt, gq.z));
}
// adj_add of lane K's terms in every lane of the quad, the operands read across
// lanes by the additions themselves (see quad_add of cc_step.h for the wait).
template <int K, int NB>
__device__ inline void quad_adj_add(const AdjTerm (&t)[NB], float inv_dt, f3& gp, f3& gq, float (&g)[NPARAM]) {
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    const AdjTerm& o = t[k];
#define CC_LANE " quad_perm:[%c[K],%c[K],%c[K],%c[K]] row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %[ax], %0" CC_LANE "v_add_f32_dpp %1, %[ay], %1" CC_LANE "v_add_f32_dpp %2, %[az], %2" CC_LANE
        "v_fmac_f32_dpp %3, -%[vx], %[dt]" CC_LANE "v_fmac_f32_dpp %4, -%[vy], %[dt]" CC_LANE
        "v_fmac_f32_dpp %5, -%[vz], %[dt]" CC_LANE
        : "+v"(gp.x), "+v"(gp.y), "+v"(gp.z), "+v"(gq.x), "+v"(gq.y), "+v"(gq.z)
        : [ax] "v"(o.a1.x), [ay] "v"(o.a1.y), [az] "v"(o.a1.z), [vx] "v"(o.v1.x), [vy] "v"(o.v1.y),
          [vz] "v"(o.v1.z), [dt] "v"(inv_dt), [K] "n"(K));
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %[g0], %0" CC_LANE "v_add_f32_dpp %1, %[g1], %1" CC_LANE "v_add_f32_dpp %2, %[g2], %2" CC_LANE
        "v_add_f32_dpp %3, %[gr], %3" CC_LANE
        : "+v"(g[0]), "+v"(g[1]), "+v"(g[2]), "+v"(g[4])
        : [g0] "v"(o.gk0), [g1] "v"(o.gk1), [g2] "v"(o.gk2), [gr] "v"(o.gr), [K] "n"(K));
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, -%[ax], %0" CC_LANE "v_add_f32_dpp %1, -%[ay], %1" CC_LANE
        "v_add_f32_dpp %2, -%[az], %2" CC_LANE
        "v_fmac_f32_dpp %3, %[vx], %[dt]" CC_LANE "v_fmac_f32_dpp %4, %[vy], %[dt]" CC_LANE
        "v_fmac_f32_dpp %5, %[vz], %[dt]" CC_LANE
        : "+v"(gp.x), "+v"(gp.y), "+v"(gp.z), "+v"(gq.x), "+v"(gq.y), "+v"(gq.z)
        : [ax] "v"(o.a2.x), [ay] "v"(o.a2.y), [az] "v"(o.a2.z), [vx] "v"(o.v2.x), [vy] "v"(o.v2.y),
          [vz] "v"(o.v2.z), [dt] "v"(inv_dt), [K] "n"(K));
#undef CC_LANE
  }
}

// What a launch of k_adj_step reads and writes: step t's records and springs,
// and for the force part of step t - 1 its state and contact normals (state1
// null: the first step of a run, whose adjoint goes to lp, lq).
struct AdjStep {
  const float *state, *lf, *locp, *locq;          // of step t
  const float *state1, *c_in1, *c_out1;           // of step t - 1
  float *lf1, *locp1, *locq1;                     // out: the force part of step t - 1
  float *lp, *lq;                                 // out: dL/dx_cur, dL/dx_prev before step t
  float *part, *part1;                            // out: parameter sums of 64 vertices each, of steps t, t - 1
};

// The spring part of step t and the force part of step t - 1.  LANES lanes per
// vertex (4: a quad, each lane a quarter of the springs, their terms added in
// row order in every lane); the parameter sums go out per 64 vertices, so they
// add the same numbers in the same order either way.  EW > 0: `rec` holds EW
// records per vertex (the forward's fixed-width rows); EW == 0: the merged CSR
// at `row`.  Bound by the chain
// from the records to the gathers and by the terms' instructions (two square
// roots and divisions each), one wave per SIMD at 128 x 128.  So the records load
// with the vertex's own data, the gathers are waited for once, empty slots are
// masked and the sums read across lanes by the additions themselves: 200 steps
// back take 1.16 ms (5.6 us a step) against 1.28 without (6.2), and 3.6 with two
// launches a step (9.2 + 2.9), one lane per vertex and the states recomputed (5.3).
template <int EW, int LANES>
__global__ __launch_bounds__(ADJ_THREADS) void k_adj_step(uint32_t n, const uint32_t* __restrict__ row,
                                                          const uint2* __restrict__ rec, AdjStep S, AdjArgs a) {
  constexpr bool QUAD = LANES == 4;
  constexpr int NB = EW && QUAD ? EW / 4 : (QUAD ? 3 : (EW ? 6 : 4));   // springs of a lane at a time
  constexpr bool PRE = EW > 0 && QUAD;   // all records load with the vertex's own data
  constexpr uint32_t VERTS = ADJ_THREADS / LANES;
  __shared__ float sg[QUAD ? VERTS : 1][NPARAM];
  const uint32_t v = threadIdx.x / LANES, i = blockIdx.x * VERTS + v;
  const int e = (int)(threadIdx.x % LANES);
  float g[NPARAM] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  if (i < n) {
    const size_t o = 3 * (size_t)i;
    uint2 er[NB];
    if constexpr (PRE) {
#pragma unroll
      for (int k = 0; k < NB; ++k) er[k] = rec[(size_t)i * EW + (uint32_t)(e * NB + k)];
    }
    const uint32_t r0raw = row[i], r1raw = EW ? 0u : row[i + 1];
    const f3 pi = ld3(S.state + 2 * o), qi = ld3(S.state + 2 * o + 3);
    const f3 lFi = ld3(S.lf + o);
    f3 gp = ld3(S.locp + o), gq = ld3(S.locq + o);
    // the force part's own loads, early
    f3 c1 = mk(0.0f, 0.0f, 0.0f), n1 = c1, p1 = c1, q1 = c1;
    if (S.state1) {
      c1 = ld3(S.c_in1 + o);
      n1 = ld3(S.c_out1 + o);
      p1 = ld3(S.state1 + 2 * o);
      q1 = ld3(S.state1 + 2 * o + 3);
    }
    const f3 vi = mk((pi.x - qi.x) * a.inv_dt, (pi.y - qi.y) * a.inv_dt, (pi.z - qi.z) * a.inv_dt);
    // in registers, as in step_vertex (selects between fields of `a` become loads)
    const float ks0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(a.k0)));
    const float ks1 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(a.k1)));
    const float ks2 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(a.k2)));
    // places in this vertex's own records (EW), or in all of them
    const uint2* __restrict__ recs = EW ? rec + (size_t)i * EW : rec;
    const uint32_t r0 = EW ? 0u : r0raw & ROW_MASK, r1 = EW ? (uint32_t)EW : r1raw & ROW_MASK;
    for (uint32_t k0 = r0; PRE || k0 < r1; k0 += NB * LANES) {
      bool real[NB];
      float sj[NB][6], lj[NB][3];
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const uint32_t at = k0 + (uint32_t)(e * NB + k);
        if (!PRE) er[k] = recs[EW ? at : min(at, r1 - 1)];
        real[k] = EW ? (er[k].x & PAD_TYPE) != PAD_TYPE : at < r1;
        if (!EW && !real[k]) er[k] = make_uint2(i | PAD_TYPE, 0u);
      }
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const uint32_t j = er[k].x & END_MASK;
        const float2* s2 = reinterpret_cast<const float2*>(S.state + 6 * (size_t)j);
        const float2 u = s2[0], w = s2[1], x = s2[2];
        sj[k][0] = u.x; sj[k][1] = u.y; sj[k][2] = w.x; sj[k][3] = w.y; sj[k][4] = x.x; sj[k][5] = x.y;
        for (int c = 0; c < 3; ++c) lj[k][c] = S.lf[3 * (size_t)j + c];
      }
      // waited for once: the compiler issues some of them at their first use
      // otherwise, one memory round trip after another
#pragma unroll
      for (int k = 0; k < NB; ++k)
        asm volatile("" ::"v"(sj[k][0]), "v"(sj[k][1]), "v"(sj[k][2]), "v"(sj[k][3]), "v"(sj[k][4]), "v"(sj[k][5]),
                     "v"(lj[k][0]), "v"(lj[k][1]), "v"(lj[k][2]));
      AdjTerm t[NB];
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const f3 pj = mk(sj[k][0], sj[k][1], sj[k][2]);
        const f3 vj = mk((sj[k][0] - sj[k][3]) * a.inv_dt, (sj[k][1] - sj[k][4]) * a.inv_dt,
                         (sj[k][2] - sj[k][5]) * a.inv_dt);
        t[k] = adj_spring(pi, vi, lFi, pj, vj, mk(lj[k][0], lj[k][1], lj[k][2]), er[k], real[k], a,
                          ks0, ks1, ks2);
        if constexpr (!QUAD) adj_add(t[k], a.inv_dt, gp, gq, g);
      }
      if constexpr (QUAD) {
        quad_adj_add<0>(t, a.inv_dt, gp, gq, g);
        quad_adj_add<1>(t, a.inv_dt, gp, gq, g);
        quad_adj_add<2>(t, a.inv_dt, gp, gq, g);
        quad_adj_add<3>(t, a.inv_dt, gp, gq, g);
      }
      if (PRE) break;
    }
    if (S.state1) {
      const AdjForce r = adj_force(gp, gq, (r0raw & PIN_BIT) != 0, c1, n1, p1, q1, a);
      g[3] = r.damp;
      if (!QUAD || e == 0) st3(S.lf1 + o, r.lF);
      if (!QUAD || e == 1) st3(S.locp1 + o, r.gp);
      if (!QUAD || e == 2) st3(S.locq1 + o, r.gq);
    } else {
      if (!QUAD || e == 0) st3(S.lp + o, gp);
      if (!QUAD || e == 1) st3(S.lq + o, gq);
    }
    if (QUAD && e == 3)
      for (int k = 0; k < NPARAM; ++k) sg[v][k] = g[k];
  }
  uint32_t v0 = i;                       // this lane's vertex in the sums
  if constexpr (QUAD) {                  // one vertex per lane again, in the first wave
    static_assert(VERTS == 64, "one wave of vertices per block");
    __syncthreads();
    if (threadIdx.x >= VERTS) return;
    v0 = blockIdx.x * VERTS + threadIdx.x;
    for (int k = 0; k < NPARAM; ++k) g[k] = v0 < n ? sg[threadIdx.x][k] : 0.0f;
  }
  wave_sum(g);
  if ((threadIdx.x & 63u) == 0 && v0 < n) {
    const size_t w = NPARAM * (size_t)(v0 >> 6);
    for (int k = 0; k < NPARAM; ++k)
      if (k != 3) S.part[w + k] = g[k];
    if (S.state1) S.part1[w + 3] = g[3];
  }
}

// acc[b] += the sums of L steps, last step first, over blocks of ADJ_THREADS
// vertices (four waves each, added in order in FP32): one workgroup per block.
// Bound by the latency of the loads: all threads fetch ACC_STEPS steps' sums
// together, then one thread per parameter adds them in order (200 steps of 16,384
// vertices: 6 us against 31 with one thread per sum fetching its own).
constexpr uint32_t ACC_STEPS = 256;
__global__ __launch_bounds__(256) void k_adj_acc(const float* __restrict__ part, uint32_t L, uint32_t nw,
                                                 double* __restrict__ acc) {
  __shared__ float f[ACC_STEPS * NPARAM];
  const uint32_t w0 = 4 * blockIdx.x;
  double s = threadIdx.x < NPARAM ? acc[blockIdx.x * NPARAM + threadIdx.x] : 0.0;
  for (uint32_t t = L; t > 0;) {
    const uint32_t k = min(t, ACC_STEPS);
#pragma unroll
    for (uint32_t r = 0; r < NPARAM; ++r) {
      const uint32_t q = r * 256 + threadIdx.x, u = q / NPARAM, p = q % NPARAM;
      if (u >= k) continue;
      const float* x = part + NPARAM * ((size_t)(t - 1 - u) * nw + w0) + p;
      float v = 0.0f;
      v += x[0];
      v += w0 + 1 < nw ? x[NPARAM] : 0.0f;
      v += w0 + 2 < nw ? x[2 * NPARAM] : 0.0f;
      v += w0 + 3 < nw ? x[3 * NPARAM] : 0.0f;
      f[q] = v;
    }
    __syncthreads();
    if (threadIdx.x < NPARAM) {
#pragma unroll 8
      for (uint32_t u = 0; u < k; ++u) s += (double)f[u * NPARAM + threadIdx.x];
    }
    __syncthreads();
    t -= k;
  }
  if (threadIdx.x < NPARAM) acc[blockIdx.x * NPARAM + threadIdx.x] = s;
}

// out[p] = sum over blocks of acc[p], in FP64 (one workgroup)
__global__ __launch_bounds__(256) void k_reduce_f64(const double* __restrict__ acc, uint32_t nblk,
                                                    double* __restrict__ out) {
  __shared__ double part[256];
  for (int p = 0; p < NPARAM; ++p) {
    double s = 0.0;
    for (uint32_t b = threadIdx.x; b < nblk; b += 256) s += acc[NPARAM * (size_t)b + p];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) out[p] = part[0];
    __syncthreads();
  }
}

struct Adj {
  Sim* S = nullptr;
  uint32_t n = 0, nsteps = 0, ckpt = 0, nck = 0, nblk = 0;
  cc_params prm{};
  StepArgs sa{};
  AdjArgs aa{};
  bool have_forward = false;
  bool keep = false;                     // seg_state / seg_contact hold every state of the forward
  DBuf<float> st[2], contact;
  DBuf<float> ck_state, ck_contact;      // [nck][6n], [nck][3n]
  DBuf<float> seg_state, seg_contact;    // [ckpt+1][6n], [ckpt+1][3n]
  DBuf<float> lp, lq, lf[2], locp[2], locq[2];
  DBuf<float> part;                      // [ckpt][ceil(n / 64)][NPARAM]
  DBuf<double> acc, out;
  ~Adj() {
    if (S && S->stream) (void)hipStreamSynchronize(S->stream);   // before the buffers are freed
  }
};

static void check_symmetric(const Sim& S) {
  std::vector<uint2> rec(S.rec.n);
  copy_on(rec.data(), S.rec.p, rec.size() * sizeof(uint2), hipMemcpyDeviceToHost, S.stream);
  const std::vector<uint32_t>& row = S.h_row;
  for (uint32_t i = 0; i < S.n; ++i)
    for (uint32_t k = row[i] & ROW_MASK; k < (row[i + 1] & ROW_MASK); ++k) {
      const uint32_t j = rec[k].x & END_MASK, t = rec[k].x >> 30;
      bool found = false;
      for (uint32_t e = row[j] & ROW_MASK; e < (row[j + 1] & ROW_MASK) && !found; ++e)
        found = (rec[e].x & END_MASK) == i && (rec[e].x >> 30) == t && rec[e].y == rec[k].y;
      CC_REQUIRE(found, "cc_adj_create: the spring set is not symmetric (every spring i->j needs j->i "
                        "of the same type and rest length)");
    }
}

// The buffers of a rollout of nsteps steps: all its states, or checkpoints.
static void alloc_adj(Adj& A, Sim& S, uint32_t nsteps, uint32_t ckpt_every, bool keep) {
  A.S = &S;
  A.n = S.n;
  A.nsteps = nsteps;
  A.keep = keep;
  A.ckpt = keep ? nsteps : std::min(ckpt_every, nsteps);
  A.nck = (uint32_t)(((size_t)nsteps + A.ckpt - 1) / A.ckpt);
  A.nblk = grid_for(S.n, ADJ_THREADS);
  const size_t n3 = 3 * (size_t)S.n, n6 = 6 * (size_t)S.n;
  A.seg_state.alloc(((size_t)A.ckpt + 1) * n6);
  A.seg_contact.alloc(((size_t)A.ckpt + 1) * n3);
  if (!keep) {
    for (int b = 0; b < 2; ++b) A.st[b].alloc(n6);
    A.contact.alloc(n3);
    A.ck_state.alloc(A.nck * n6);
    A.ck_contact.alloc(A.nck * n3);
  }
  A.lp.alloc(n3);
  A.lq.alloc(n3);
  for (int b = 0; b < 2; ++b) {
    A.lf[b].alloc(n3);
    A.locp[b].alloc(n3);
    A.locq[b].alloc(n3);
  }
  A.part.alloc((size_t)A.ckpt * grid_for(S.n, 64) * NPARAM);
  A.acc.alloc(NPARAM * (size_t)A.nblk);
  A.out.alloc(NPARAM);
}

}  // namespace cc

using namespace cc;

struct cc_adj {
  Adj a;
};

extern "C" {

int cc_adj_create(cc_sim* sim, uint32_t nsteps, uint32_t ckpt_every, cc_adj** out) {
  return guard([&] {
    CC_REQUIRE(sim && out && nsteps >= 1 && ckpt_every >= 1, "cc_adj_create: bad argument");
    Sim& S = sim->s;
    CC_REQUIRE(!S.body.moving(), "cc_adj_create: a moving body is not supported (static or no body)");
    *out = nullptr;
    CC_HIP(hipDeviceSynchronize());
    check_symmetric(S);
    // Every state where that takes little memory; checkpoints otherwise, also
    // when any part of that memory is not to be had.
    const size_t keep_bytes = ((size_t)nsteps + 1) * 9 * S.n * sizeof(float);
    std::unique_ptr<cc_adj> h(new cc_adj);
    try {
      alloc_adj(h->a, S, nsteps, ckpt_every, keep_bytes <= keep_limit());
    } catch (const Error& e) {
      if (e.code != CC_ERR_ALLOC || !h->a.keep) throw;
      h.reset();           // the first attempt's memory goes before the second
      h.reset(new cc_adj);
      alloc_adj(h->a, S, nsteps, ckpt_every, false);
    }
    *out = h.release();
  });
}

int cc_adj_destroy(cc_adj* adj) {
  return guard([&] {
    if (!adj) return;
    (void)hipStreamSynchronize(adj->a.S->stream);
    delete adj;
  });
}

int cc_adj_forward(cc_adj* adj, const float* x0, const float* v0, const double theta[5], float* x_final) {
  return guard([&] {
    CC_REQUIRE(adj && x0 && theta, "cc_adj_forward: bad argument");
    Adj& A = adj->a;
    Sim& S = *A.S;
    hipStream_t s = S.stream;
    CC_HIP(hipDeviceSynchronize());
    A.prm = S.prm;
    for (int t = 0; t < 3; ++t) A.prm.k[t] = (float)theta[t];
    A.prm.damp = (float)theta[3];
    A.prm.rest_scale = (float)theta[4];
    A.sa = step_args(A.prm, S.ntypes);
    A.aa.dt = A.prm.dt;
    A.aa.inv_dt = A.sa.inv_dt;
    A.aa.w = A.sa.dt2 * A.sa.inv_mass;
    A.aa.damp = A.prm.damp;
    A.aa.kd = A.prm.kd;
    A.aa.k0 = A.prm.k[0];
    A.aa.k1 = A.prm.k[1];
    A.aa.k2 = A.prm.k[2];
    A.aa.rest_scale = A.prm.rest_scale;
    A.aa.eps = A.prm.eps;
    const size_t n3 = 3 * (size_t)A.n, n6 = 6 * (size_t)A.n;
    std::vector<float> packed(n6);
    for (uint32_t i = 0; i < A.n; ++i)
      for (int c = 0; c < 3; ++c) {
        const float x = x0[3 * (size_t)i + c], v = v0 ? v0[3 * (size_t)i + c] : 0.0f;
        packed[6 * (size_t)i + c] = x;
        packed[6 * (size_t)i + 3 + c] = x - v * A.prm.dt;
      }
    float* const x_in = A.keep ? A.seg_state.p : A.st[0].p;
    float* const c_in = A.keep ? A.seg_contact.p : A.contact.p;
    CC_HIP(hipMemcpyAsync(x_in, packed.data(), n6 * sizeof(float), hipMemcpyHostToDevice, s));
    CC_HIP(hipMemsetAsync(c_in, 0, n3 * sizeof(float), s));
    const float* x_out = nullptr;
    if (A.keep) {
      for (uint32_t t = 0; t < A.nsteps; ++t)
        S.launch_step(A.seg_state.p + t * n6, A.seg_state.p + (t + 1) * n6, A.seg_contact.p + t * n3,
                      A.seg_contact.p + (t + 1) * n3, A.sa, 0, s);
      x_out = A.seg_state.p + A.nsteps * n6;
    } else {
      int cur = 0;
      for (uint32_t t = 0; t < A.nsteps; ++t) {
        if (t % A.ckpt == 0) {
          const uint32_t c = t / A.ckpt;
          CC_HIP(hipMemcpyAsync(A.ck_state.p + c * n6, A.st[cur].p, n6 * sizeof(float), hipMemcpyDeviceToDevice, s));
          CC_HIP(hipMemcpyAsync(A.ck_contact.p + c * n3, A.contact.p, n3 * sizeof(float), hipMemcpyDeviceToDevice, s));
        }
        S.launch_step(A.st[cur].p, A.st[cur ^ 1].p, A.contact.p, A.contact.p, A.sa, 0, s);
        cur ^= 1;
      }
      x_out = A.st[cur].p;
    }
    if (x_final) {
      CC_HIP(hipMemcpyAsync(packed.data(), x_out, n6 * sizeof(float), hipMemcpyDeviceToHost, s));
      CC_HIP(hipStreamSynchronize(s));
      for (uint32_t i = 0; i < A.n; ++i)
        for (int c = 0; c < 3; ++c) x_final[3 * (size_t)i + c] = packed[6 * (size_t)i + c];
    }
    CC_HIP(hipStreamSynchronize(s));
    A.have_forward = true;
  });
}

int cc_adj_backward(cc_adj* adj, const float* dl_dx_final, double dl_dtheta[5], float* dl_dv0, float* dl_dx0) {
  return guard([&] {
    CC_REQUIRE(adj && dl_dx_final, "cc_adj_backward: bad argument");
    Adj& A = adj->a;
    CC_REQUIRE(A.have_forward, "cc_adj_backward: call cc_adj_forward first");
    Sim& S = *A.S;
    hipStream_t s = S.stream;
    const size_t n3 = 3 * (size_t)A.n, n6 = 6 * (size_t)A.n;
    CC_HIP(hipMemcpyAsync(A.lp.p, dl_dx_final, n3 * sizeof(float), hipMemcpyHostToDevice, s));
    A.lq.zero(s);
    A.acc.zero(s);
    // four lanes per vertex up to the size where the forward's step takes them
    // (us per step back, one lane / four: 13.5 / 13.1 at 65,536 vertices, 20.2 /
    // 19.0 at 90,000, 21.8 / 21.2 at 108,900, 23.9 / 24.2 at 131,044)
    const bool quads = A.n <= QUAD_MAX_N, ell = S.ell_w == ELL_W;
    const uint2* recs = ell ? S.ell.p : S.rec.p;
    auto kern = ell ? (quads ? k_adj_step<ELL_W, 4> : k_adj_step<ELL_W, 1>)
                    : (quads ? k_adj_step<0, 4> : k_adj_step<0, 1>);
    const unsigned grid = grid_for(A.n, quads ? ADJ_THREADS / 4 : ADJ_THREADS);
    const uint32_t nw = grid_for(A.n, 64);
    auto part = [&](uint32_t j) { return A.part.p + (size_t)j * nw * NPARAM; };
    for (uint32_t c = A.nck; c-- > 0;) {
      const uint32_t t0 = c * A.ckpt, t1 = std::min(t0 + A.ckpt, A.nsteps), L = t1 - t0;
      if (!A.keep) {
        // the segment forward again, keeping every state
        CC_HIP(hipMemcpyAsync(A.seg_state.p, A.ck_state.p + c * n6, n6 * sizeof(float), hipMemcpyDeviceToDevice, s));
        CC_HIP(hipMemcpyAsync(A.seg_contact.p, A.ck_contact.p + c * n3, n3 * sizeof(float), hipMemcpyDeviceToDevice,
                              s));
        for (uint32_t j = 0; j < L; ++j)   // contact normals of step j in, of step j + 1 out
          S.launch_step(A.seg_state.p + j * n6, A.seg_state.p + (j + 1) * n6, A.seg_contact.p + j * n3,
                        A.seg_contact.p + (j + 1) * n3, A.sa, 0, s);
      }
      auto st = [&](uint32_t j) { return A.seg_state.p + j * n6; };
      auto ct = [&](uint32_t j) { return A.seg_contact.p + j * n3; };
      int cur = 0;
      k_adj_force<<<A.nblk, ADJ_THREADS, 0, s>>>(A.n, S.row.p, st(L - 1), ct(L - 1), ct(L), A.lp.p, A.lq.p, A.aa,
                                                 A.lf[0].p, A.locp[0].p, A.locq[0].p, part(L - 1));
      CC_LAUNCHED();
      for (uint32_t j = L; j-- > 0;) {
        AdjStep D{};
        D.state = st(j);
        D.lf = A.lf[cur].p;
        D.locp = A.locp[cur].p;
        D.locq = A.locq[cur].p;
        D.part = part(j);
        if (j > 0) {
          D.part1 = part(j - 1);
          D.state1 = st(j - 1);
          D.c_in1 = ct(j - 1);
          D.c_out1 = ct(j);
          D.lf1 = A.lf[cur ^ 1].p;
          D.locp1 = A.locp[cur ^ 1].p;
          D.locq1 = A.locq[cur ^ 1].p;
        } else {
          D.lp = A.lp.p;
          D.lq = A.lq.p;
        }
        kern<<<grid, ADJ_THREADS, 0, s>>>(A.n, S.row.p, recs, D, A.aa);
        CC_LAUNCHED();
        cur ^= 1;
      }
      k_adj_acc<<<A.nblk, 256, 0, s>>>(A.part.p, L, nw, A.acc.p);
      CC_LAUNCHED();
    }
    k_reduce_f64<<<1, 256, 0, s>>>(A.acc.p, A.nblk, A.out.p);
    CC_LAUNCHED();
    std::vector<float> lp(n3), lq(n3);
    double g[NPARAM];
    CC_HIP(hipMemcpyAsync(lp.data(), A.lp.p, n3 * sizeof(float), hipMemcpyDeviceToHost, s));
    CC_HIP(hipMemcpyAsync(lq.data(), A.lq.p, n3 * sizeof(float), hipMemcpyDeviceToHost, s));
    CC_HIP(hipMemcpyAsync(g, A.out.p, sizeof(g), hipMemcpyDeviceToHost, s));
    CC_HIP(hipStreamSynchronize(s));
    if (dl_dtheta) std::memcpy(dl_dtheta, g, sizeof(g));
    for (size_t k = 0; k < n3; ++k) {   // x_cur = x0, x_prev = x0 - v0 dt
      if (dl_dx0) dl_dx0[k] = lp[k] + lq[k];
      if (dl_dv0) dl_dv0[k] = -A.prm.dt * lq[k];
    }
  });
}

}  // extern "C"
