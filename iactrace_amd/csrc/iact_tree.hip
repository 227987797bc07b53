// The spot tree: image and gradients of primary-only, hard-binned renders with
// far or parallel sources, summed per (run of samples, source) instead of per
// ray wherever all rays of the run provably meet the same pixel.
//
// A far source (source_qs 0) or a parallel one gives every sample of a facet
// the same u, and a sample's ray carries value / |u| (u.m) nrwh (m, nrwh from
// its record).  If the rays of a run of samples all meet pixel P and no
// obstruction can reach any of them, the run adds value / |u| (u.S) to P with
// S = sum nrwh m, whatever the number of samples; the gradients of such a run
// follow from G[P] and S in the same way.  The kernels walk a tree of runs per
// facet -- 1024 samples, 64, 16, single rays; the records are Morton-sorted,
// so a run is compact on the facet -- and split a (run, source) pair only
// where the run's spot may cross a pixel boundary or a shadow edge.  Single
// rays are traced with the arithmetic of the other kernels, and a pair is
// resolved only with a margin above its rounding, so every ray lands on the
// pixel that the per-ray kernels give it.
//
// The spot of a run.  With U = (u.An, u.Au, u.Av), a = U.y / U.x,
// b = U.z / U.x and (da, db) the offset from a reference direction (a0, b0),
// the hit of sample j in grid coordinates is exactly
//   g_j = P_j + (Q_j.d) s_j,   s_j = 1 / (1 + h_j.d),   d = (da, db)
// (the plane hit is a homography of the direction).  Writing s for the run's
// s (its mean h) and d' = s d,
//   g_j = P_j + Q_j.d' - (dh_j.d')(Q.d') + rem,
//   |rem| <= s |dh_j.d| (s_j |dQ_j.d| + s s_j |dh_j.d| |Q.d|).
// P, Q and h vary almost linearly over a compact run, so each is stored as
// its mean, its slopes over the run's two facet coordinates x (scaled by the
// run's half extents X) and the largest residuals: the spot lies within
//   ext = |J1 + K1.d' - (Q.d') H1.d'| + |J2 + ...| + W + V |d|_1
// of the run's centre in each form that bounds a pixel (two for squares, three
// for hexagons).  W holds the rounding margin.  Any slopes give a valid bound;
// they are the least-squares ones, or zero where that is tighter (rough
// mirrors).
#include <math.h>
#include <string.h>

#include "iact_abi_internal.h"

namespace iact {

constexpr int kWaves = 8;  // of a block
constexpr float kTreeEps = 2e-6f;  // margin: some four times the fp32 rounding of a hit

// Node words: 0-1 P, 2-5 Q (u: a, b; v: a, b), 6-7 h, 8-11 J (u: 1, 2; v: 1,
// 2), 12-19 K (u1: a, b; u2; v1; v2), 20-23 H (1: a, b; 2), 24-26 W, 27 V,
// 28-30 S, 31: the node is worth testing.

// ------------------------------------------------------------------ frame
// Block 0: the reference direction -- the mean (a, b) over the sources, the
// sign of U.x that most have, and the largest |d|_1, at most eight times its
// mean (sources beyond it are traced per ray).  frame: a0, b0, tau, sign, and
// the walk's work counter, cleared.
// At most 8192 sources are looked at (the frame steers the bounds' tightness,
// not their validity).  Other blocks: the hexagonal table in 16 bits with two
// border entries on every side; -1 is an empty cell, -2 one whose six
// neighbours are empty too.
__global__ __launch_bounds__(1024) void k_tree_frame(const double* src, int ns, int source_type,
                                                     DevSensor S, float* frame, int16_t* table) {
  const int t = threadIdx.x;
  if (blockIdx.x > 0) {
    const int w = S.tr + 4, i = (blockIdx.x - 1) * 1024 + t;
    if (i >= (S.tq + 4) * w) return;
    const int q = i / w - 2, r = i % w - 2;
    auto at = [&](int a, int b) {
      return a >= 0 && a < S.tq && b >= 0 && b < S.tr ? max(S.table[a * S.tr + b], -1) : -1;
    };
    int v = at(q, r);
    if (v < 0 && at(q + 1, r) < 0 && at(q - 1, r) < 0 && at(q, r + 1) < 0 && at(q, r - 1) < 0 &&
        at(q + 1, r - 1) < 0 && at(q - 1, r + 1) < 0)
      v = -2;
    table[i] = (int16_t)v;
    return;
  }
  __shared__ float red[6][16];
  const long long stride = max(1, (ns + 8191) / 8192);
  const float sg = source_type == IACT_SOURCE_POINT ? -1.f : 1.f;
  auto dir = [&](long long s, float& a, float& b, float& sn) {
    const double x = src[3 * s], y = src[3 * s + 1], z = src[3 * s + 2];
    const double il = 1.0 / sqrt(x * x + y * y + z * z);
    const f3 u = sg * mk3((float)(x * il), (float)(y * il), (float)(z * il));
    const f3 U = sensor_dirs(S, u);
    a = U.y / U.x;
    b = U.z / U.x;
    sn = U.x > 1e-2f ? 1.f : (U.x < -1e-2f ? -1.f : 0.f);
  };
  float v[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // (n, a, b) for U.x < 0, then > 0
  for (long long s = t * stride; s < ns; s += 1024 * stride) {
    float a, b, sn;
    dir(s, a, b, sn);
    const int o = sn > 0.f ? 3 : 0;
    if (sn != 0.f) {
      v[0] += o ? 0.f : 1.f;
      v[1] += o ? 0.f : a;
      v[2] += o ? 0.f : b;
      v[3] += o ? 1.f : 0.f;
      v[4] += o ? a : 0.f;
      v[5] += o ? b : 0.f;
    }
  }
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const float w = wave_sum(v[i]);
    if ((t & 63) == 0) red[i][t >> 6] = w;
  }
  __syncthreads();
  float tot[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    tot[i] = 0.f;
    for (int w = 0; w < 16; ++w) tot[i] += red[i][w];
  }
  const bool pos = tot[3] > tot[0];
  const float n = pos ? tot[3] : tot[0], sign = pos ? 1.f : -1.f;
  const float a0 = (pos ? tot[4] : tot[1]) / fmaxf(n, 1.f);
  const float b0 = (pos ? tot[5] : tot[2]) / fmaxf(n, 1.f);
  float mx = 0.f, sum = 0.f;
  for (long long s = t * stride; s < ns; s += 1024 * stride) {
    float a, b, sn;
    dir(s, a, b, sn);
    if (sn == sign) {
      const float tau = fabsf(a - a0) + fabsf(b - b0);
      mx = fmaxf(mx, tau);
      sum += tau;
    }
  }
  __syncthreads();
  const float ws = wave_sum(sum);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  if ((t & 63) == 0) {
    red[0][t >> 6] = ws;
    red[1][t >> 6] = mx;
  }
  __syncthreads();
  if (t == 0) {
    float m = 0.f, s = 0.f;
    for (int w = 0; w < 16; ++w) {
      s += red[0][w];
      m = fmaxf(m, red[1][w]);
    }
    frame[0] = a0;
    frame[1] = b0;
    // (a sparse look at many sources may miss the outermost ones)
    frame[2] = n > 0.f ? fminf(m * (stride > 1 ? 1.05f : 1.001f), 8.f * s / n) +
                             4e-6f * (1.f + fabsf(a0) + fabsf(b0))
                       : -1.f;
    frame[3] = sign;
    ((uint32_t*)frame)[4] = 0u;  // the walk's work counter
  }
}

// ------------------------------------------------------------------ nodes
template <int G, class Op>
IACT_DEV float group_all(float v, Op op) {  // over 16 or 64 lanes, to each of them
  v = op(v, dpp_f<0xB1>(v));
  v = op(v, dpp_f<0x4E>(v));
  v = op(v, dpp_f<0x141>(v));
  v = op(v, dpp_f<0x140>(v));
  if (G == 64) {
    v = op(v, __shfl_xor(v, 16, 64));
    v = op(v, __shfl_xor(v, 32, 64));
  }
  return v;
}
template <int G>
IACT_DEV float group_sum(float v) {
  return group_all<G>(v, [](float a, float b) { return a + b; });
}
template <int G>
IACT_DEV float group_max(float v) {
  return group_all<G>(v, [](float a, float b) { return fmaxf(a, b); });
}

// One sample's exact spot coefficients (file comment), its coordinates x, y in
// the facet frame, and the magnitudes that bound the rounding of its hit.
struct SpotSample {
  float v[8];  // P (u, v), Q (ua, ub, va, vb), h (a, b)
  float x, y, mu, mv;
  f3 p, s;     // point, nrwh m
  bool ok;     // a hit in front of the sample, all terms finite
};
IACT_DEV SpotSample spot_sample(const TreeParams& K, const float4* rec, const m3& R, float a0,
                                float b0, float tau, float sign) {
  const Sample s = unpack_record(RecRaw{rec[0], rec[1], rec[2], rec[3]});
  SpotSample o;
  const f3 B0 = mk3(K.b0[0], K.b0[1], K.b0[2]), B1 = mk3(K.b1[0], K.b1[1], K.b1[2]);
  const f3 B2 = mk3(K.b2[0], K.b2[1], K.b2[2]);
  const f3 u0 = fma3(a0, B1, fma3(b0, B2, B0));
  const float w1 = dot(s.m, B1), w2 = dot(s.m, B2), C0 = dot(s.m, u0);
  const float D0 = fmaf(s.N.x, C0, 1.f), iD = 1.f / D0;
  const float rE = fmaf(s.N.y, C0, a0) * iD, rF = fmaf(s.N.z, C0, b0) * iD;
  const float ha = s.N.x * w1 * iD, hb = s.N.x * w2 * iD;
  o.v[0] = fmaf(s.G.kt, rE, s.G.ku);
  o.v[1] = fmaf(s.G.kt, rF, s.G.kv);
  o.v[2] = s.G.kt * (fmaf(s.N.y, w1, 1.f) * iD - rE * ha);
  o.v[3] = s.G.kt * (s.N.y * w2 * iD - rE * hb);
  o.v[4] = s.G.kt * (s.N.z * w1 * iD - rF * ha);
  o.v[5] = s.G.kt * (fmaf(s.N.z, w2, 1.f) * iD - rF * hb);
  o.v[6] = ha;
  o.v[7] = hb;
  const f3 l = mulT(R, s.q);
  o.x = l.x;
  o.y = l.y;
  o.p = s.p;
  o.s = s.nrwh * s.m;
  const float nu = sqrtf(dot(u0, u0)), cm = 2.f * nu, k = fabsf(s.G.kt * iD);
  const float dD = nu + fabsf(s.N.x) * cm;
  o.mu = fabsf(s.G.ku) + k * (fmaf(K.n_au, nu, fabsf(s.N.y) * cm) + fabsf(rE) * dD) +
         (fabsf(o.v[2]) + fabsf(o.v[3])) * tau;
  o.mv = fabsf(s.G.kv) + k * (fmaf(K.n_av, nu, fabsf(s.N.z) * cm) + fabsf(rF) * dD) +
         (fabsf(o.v[4]) + fabsf(o.v[5])) * tau;
  // t = kt / (U.x D) > 0 with U.x of the frame's sign; |D| well above 0
  o.ok = s.G.kt * D0 * sign > 0.f && fabsf(D0) > 1e-3f && o.mu < 1e7f && o.mv < 1e7f &&
         fabsf(o.s.x) + fabsf(o.s.y) + fabsf(o.s.z) < 1e30f && tau >= 0.f;
  return o;
}

// Counts, means and central moments of a group's samples.
struct SpotMoments {
  float n, mx, my, sxx, sxy, syy;
  float mv[8], cx[8], cy[8];
};
template <int G>
IACT_DEV SpotMoments spot_moments(const SpotSample& s, bool act) {
  const int base = lane_id() & ~(G - 1);
  SpotMoments m;
  const float w = act ? 1.f : 0.f;
  m.n = fmaxf(group_sum<G>(w), 1.f);
  const float in = 1.f / m.n;
  const float x0 = __shfl(s.x, base, 64), y0 = __shfl(s.y, base, 64);
  const float dx = act ? s.x - x0 : 0.f, dy = act ? s.y - y0 : 0.f;
  const float ex = group_sum<G>(dx) * in, ey = group_sum<G>(dy) * in;
  m.mx = x0 + ex;
  m.my = y0 + ey;
  m.sxx = group_sum<G>(dx * dx) - m.n * ex * ex;
  m.sxy = group_sum<G>(dx * dy) - m.n * ex * ey;
  m.syy = group_sum<G>(dy * dy) - m.n * ey * ey;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float v0 = __shfl(s.v[k], base, 64);
    const float dv = act ? s.v[k] - v0 : 0.f;
    const float ev = group_sum<G>(dv) * in;
    m.mv[k] = v0 + ev;
    m.cx[k] = group_sum<G>(dv * dx) - m.n * ev * ex;
    m.cy[k] = group_sum<G>(dv * dy) - m.n * ev * ey;
  }
  return m;
}
// Least-squares slopes; zero for a degenerate group.
IACT_DEV void spot_slopes(const SpotMoments& m, float* sx, float* sy) {
  const float det = m.sxx * m.syy - m.sxy * m.sxy;
  const float id = det > 1e-4f * m.sxx * m.syy ? 1.f / det : 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    sx[k] = (m.syy * m.cx[k] - m.sxy * m.cy[k]) * id;
    sy[k] = (m.sxx * m.cy[k] - m.sxy * m.cx[k]) * id;
  }
}
// The forms that bound a pixel, as combinations of (u, v).
template <int KIND>
IACT_DEV void spot_forms(float u, float v, float* f) {
  if (KIND == IACT_SENSOR_HEX) {
    f[0] = fmaf(2.f, u, v);
    f[1] = fmaf(2.f, v, u);
    f[2] = u - v;
  } else {
    f[0] = u;
    f[1] = v;
    f[2] = 0.f;
  }
}
// Largest deviations of a group's samples from its linear model.
struct SpotExtent {
  // X, Y; per form the residual of P, the deviation of P, the residual and the
  // deviation of Q, the largest |Q|; the residual, deviation and largest |h|;
  // the magnitudes; the distance from the ball's centre
  float e[23];
};
template <int KIND>
IACT_DEV void spot_extent(const SpotSample& s, bool act, float mx, float my, const float* mv,
                          const float* sx, const float* sy, f3 c, SpotExtent& E) {
  if (!act) return;
  const float x = s.x - mx, y = s.y - my;
  float d[8], r[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    d[k] = s.v[k] - mv[k];
    r[k] = d[k] - fmaf(sx[k], x, sy[k] * y);
  }
  auto up = [&](int i, float v) { E.e[i] = fmaxf(E.e[i], fabsf(v)); };
  up(0, x);
  up(1, y);
  float f[3], g[3];
  spot_forms<KIND>(r[0], r[1], f);
  spot_forms<KIND>(d[0], d[1], g);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    up(2 + i, f[i]);
    up(5 + i, g[i]);
  }
  spot_forms<KIND>(r[2], r[4], f);
  spot_forms<KIND>(r[3], r[5], g);
#pragma unroll
  for (int i = 0; i < 3; ++i) up(8 + i, fmaxf(fabsf(f[i]), fabsf(g[i])));
  spot_forms<KIND>(d[2], d[4], f);
  spot_forms<KIND>(d[3], d[5], g);
#pragma unroll
  for (int i = 0; i < 3; ++i) up(11 + i, fmaxf(fabsf(f[i]), fabsf(g[i])));
  spot_forms<KIND>(s.v[2], s.v[4], f);
  spot_forms<KIND>(s.v[3], s.v[5], g);
#pragma unroll
  for (int i = 0; i < 3; ++i) up(14 + i, fmaxf(fabsf(f[i]), fabsf(g[i])));
  up(17, fmaxf(fabsf(r[6]), fabsf(r[7])));
  up(18, fmaxf(fabsf(d[6]), fabsf(d[7])));
  up(19, fmaxf(fabsf(s.v[6]), fabsf(s.v[7])));
  up(20, s.mu);
  up(21, s.mv);
  const f3 w = s.p - c;
  up(22, sqrtf(dot(w, w)));
}
// Node words from a group's model and extents.  useful: the largest W, in
// half pixels, for which a test is worth its instructions (a 16-sample node's
// test costs two of its sixteen rays, a patch's a tenth of what it may save;
// tops are always tested: they drop the pairs that miss the camera).
template <int KIND>
IACT_DEV void store_node(const TreeParams& K, float* o, float* ball, float tau, bool ok,
                         float useful, const float* mv, const float* sx, const float* sy, f3 S,
                         f3 c, const SpotExtent& E) {
  const float* e = E.e;
  const int nf = KIND == IACT_SENSOR_HEX ? 3 : 2;
  const float hm = e[19] * tau;
  ok = ok && hm <= 0.25f && K.hu > 0.f && K.hv > 0.f;
  const float sm = 1.f / (1.f - fminf(hm, 0.5f));
  float W[3], Wb[3], V = 0.f, Vb = 0.f, cl = 0.f, cb = 0.f;
  float mag[3];
  spot_forms<KIND>(e[20], e[21], mag);
  mag[2] = e[20] + e[21];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    W[i] = Wb[i] = 0.f;
    if (i >= nf) continue;
    const float mu = fmaf(kTreeEps, mag[i], 3e-5f);
    float js[3], ks[3];
    spot_forms<KIND>(sx[0], sx[1], js);
    spot_forms<KIND>(sy[0], sy[1], ks);
    const float rem = sm * sm * tau * e[18] * fmaf(sm * e[18] * tau, e[14 + i], e[11 + i]);
    W[i] = e[2 + i] + mu;
    Wb[i] = e[5 + i] + mu;
    V = fmaxf(V, 1.01f * (sm * e[8 + i] + sm * sm * e[14 + i] * tau * e[17] + rem));
    Vb = fmaxf(Vb, 1.01f * (sm * e[11 + i] + sm * sm * e[14 + i] * tau * e[18] + rem));
    cl += W[i] + fabsf(js[i]) * e[0] + fabsf(ks[i]) * e[1];
    cb += Wb[i];
  }
  // the slopes tighten the bound unless the samples scatter (rough mirrors)
  const bool lin = cl + nf * 0.5f * tau * V <= cb + nf * 0.5f * tau * Vb;
  const float X = lin ? e[0] : 0.f, Y = lin ? e[1] : 0.f;
  float w[IACT_NODE_WORDS];
#pragma unroll
  for (int k = 0; k < 8; ++k) w[k] = mv[k];
  w[8] = sx[0] * X;
  w[9] = sy[0] * Y;
  w[10] = sx[1] * X;
  w[11] = sy[1] * Y;
  w[12] = sx[2] * X;
  w[13] = sx[3] * X;
  w[14] = sy[2] * Y;
  w[15] = sy[3] * Y;
  w[16] = sx[4] * X;
  w[17] = sx[5] * X;
  w[18] = sy[4] * Y;
  w[19] = sy[5] * Y;
  w[20] = sx[6] * X;
  w[21] = sx[7] * X;
  w[22] = sy[6] * Y;
  w[23] = sy[7] * Y;
  float wm = 0.f;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    w[24 + i] = lin ? W[i] : Wb[i];
    wm = fmaxf(wm, w[24 + i]);
  }
  w[27] = lin ? V : Vb;
  w[28] = S.x;
  w[29] = S.y;
  w[30] = S.z;
  w[31] = ok && wm < useful * fminf(K.hu, K.hv) ? 1.f : 0.f;
  float4* o4 = (float4*)o;
#pragma unroll
  for (int i = 0; i < IACT_NODE_WORDS / 4; ++i)
    o4[i] = make_float4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
  *(float4*)ball = make_float4(c.x, c.y, c.z, fmaf(e[22], 1.000001f, 1e-6f));
}

// A group of G lanes (one sample each) to one node, written by its first lane.
template <int KIND, int G>
IACT_DEV void group_node(const TreeParams& K, const SpotSample& s, bool act, float tau,
                         float useful, float* nodes, float* balls, long long id, bool store,
                         SpotMoments& m, f3& S, f3& c) {
  const int base = lane_id() & ~(G - 1);
  m = spot_moments<G>(s, act);
  float sx[8], sy[8];
  spot_slopes(m, sx, sy);
  S = mk3(group_sum<G>(act ? s.s.x : 0.f), group_sum<G>(act ? s.s.y : 0.f),
          group_sum<G>(act ? s.s.z : 0.f));
  const f3 p0 = mk3(__shfl(s.p.x, base, 64), __shfl(s.p.y, base, 64), __shfl(s.p.z, base, 64));
  const f3 dp = act ? s.p - p0 : mk3(0.f, 0.f, 0.f);
  c = p0 + (1.f / m.n) * mk3(group_sum<G>(dp.x), group_sum<G>(dp.y), group_sum<G>(dp.z));
  SpotExtent E;
#pragma unroll
  for (int i = 0; i < 23; ++i) E.e[i] = 0.f;
  spot_extent<KIND>(s, act, m.mx, m.my, m.mv, sx, sy, c, E);
#pragma unroll
  for (int i = 0; i < 23; ++i) E.e[i] = group_max<G>(E.e[i]);
  const uint64_t bad = __ballot(act && !s.ok);
  const uint64_t mine = G == 64 ? ~0ull : 0xffffull << base;
  if (lane_id() == base && store)
    store_node<KIND>(K, nodes + IACT_NODE_WORDS * id, balls + 4 * id, tau, (bad & mine) == 0ull,
                     useful, m.mv, sx, sy, S, c, E);
}

// One block of four waves per (facet, top): a wave per patch of 64 records
// makes the patch's node and its four leaves' (wave reductions), then the
// block makes the top's from the patches' moments and a second pass over the
// samples.  87 us for 875 x 1024 samples: the reductions' VALU.
template <int KIND>
__global__ __launch_bounds__(256) void k_tree_nodes(TraceArgs A, TreeParams K, float* nodes, float* balls) {
  __shared__ float mom[16][36];
  __shared__ float model[32];
  __shared__ int emax[23];
  __shared__ int bad;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
  const int f = blockIdx.x / K.n_top, top = blockIdx.x - f * K.n_top;
  const cptr<float> fr = as_const(K.frame);
  const float a0 = fr[0], b0 = fr[1], tau = fr[2], sign = fr[3];
  const m3 R = facet_rotation(A.rotations, f);
  const int m0 = top * kTopSamples;
  const int npt = (min(kTopSamples, A.M - m0) + 63) / 64;
  const long long base = (long long)f * K.per_facet;
  const float4* recs = (const float4*)A.recs + 4 * ((size_t)f * A.M);
  if (threadIdx.x < 23) emax[threadIdx.x] = 0;
  if (threadIdx.x == 0) bad = 0;
  __syncthreads();
  bool any_bad = false;
  for (int p = wave; p < npt; p += 4) {
    const int m = m0 + 64 * p + lane;
    const bool act = m < A.M;
    const SpotSample s =
        spot_sample(K, recs + 4 * (size_t)(act ? m : A.M - 1), R, a0, b0, tau, sign);
    any_bad |= __any(act && !s.ok);
    SpotMoments mm;
    f3 S, c;
    const int leaf = top * (kTopSamples / 16) + 4 * p + (lane >> 4);
    group_node<KIND, 16>(K, s, act, tau, 0.65f, nodes, balls, base + K.n_top + K.n_patch + leaf,
                         leaf < K.n_leaf, mm, S, c);
    const int patch = top * (kTopSamples / 64) + p;
    group_node<KIND, 64>(K, s, act, tau, 0.8f, nodes, balls, base + K.n_top + patch, true, mm, S,
                         c);
    if (lane == 0) {
      float* o = mom[p];
      o[0] = mm.n;
      o[1] = mm.mx;
      o[2] = mm.my;
      o[3] = mm.sxx;
      o[4] = mm.sxy;
      o[5] = mm.syy;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        o[6 + k] = mm.mv[k];
        o[14 + k] = mm.cx[k];
        o[22 + k] = mm.cy[k];
      }
      o[30] = S.x;
      o[31] = S.y;
      o[32] = S.z;
      o[33] = c.x;
      o[34] = c.y;
      o[35] = c.z;
    }
  }
  if (any_bad && lane == 0) atomicOr(&bad, 1);
  __syncthreads();
  // the top's moments from its patches' (lane = patch of the first wave)
  float sx[8], sy[8], mv[8];
  if (wave == 0) {
    const float* o = mom[lane & 15];
    const bool act = (lane & 15) < npt;
    SpotMoments m;
    const float n = act ? o[0] : 0.f;
    m.n = group_sum<16>(n);
    const float in = 1.f / m.n;
    const float dx0 = act ? o[1] - mom[0][1] : 0.f, dy0 = act ? o[2] - mom[0][2] : 0.f;
    const float ex = group_sum<16>(n * dx0) * in, ey = group_sum<16>(n * dy0) * in;
    m.mx = mom[0][1] + ex;
    m.my = mom[0][2] + ey;
    const float dx = dx0 - ex, dy = dy0 - ey;
    m.sxx = group_sum<16>(act ? fmaf(n * dx, dx, o[3]) : 0.f);
    m.sxy = group_sum<16>(act ? fmaf(n * dx, dy, o[4]) : 0.f);
    m.syy = group_sum<16>(act ? fmaf(n * dy, dy, o[5]) : 0.f);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float d0 = act ? o[6 + k] - mom[0][6 + k] : 0.f;
      const float ev = group_sum<16>(n * d0) * in;
      m.mv[k] = mom[0][6 + k] + ev;
      m.cx[k] = group_sum<16>(act ? fmaf(n * dx, d0 - ev, o[14 + k]) : 0.f);
      m.cy[k] = group_sum<16>(act ? fmaf(n * dy, d0 - ev, o[22 + k]) : 0.f);
    }
    spot_slopes(m, sx, sy);
    f3 c = mk3(0.f, 0.f, 0.f);
    if (act) c = n * in * mk3(o[33] - mom[0][33], o[34] - mom[0][34], o[35] - mom[0][35]);
    c = mk3(mom[0][33], mom[0][34], mom[0][35]) +
        mk3(group_sum<16>(c.x), group_sum<16>(c.y), group_sum<16>(c.z));
    if (lane == 0) {
      model[0] = m.mx;
      model[1] = m.my;
      model[2] = c.x;
      model[3] = c.y;
      model[4] = c.z;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        model[5 + k] = m.mv[k];
        model[13 + k] = sx[k];
        model[21 + k] = sy[k];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    mv[k] = model[5 + k];
    sx[k] = model[13 + k];
    sy[k] = model[21 + k];
  }
  const f3 c = mk3(model[2], model[3], model[4]);
  SpotExtent E;
#pragma unroll
  for (int i = 0; i < 23; ++i) E.e[i] = 0.f;
  for (int p = wave; p < npt; p += 4) {
    const int m = m0 + 64 * p + lane;
    const bool act = m < A.M;
    const SpotSample s =
        spot_sample(K, recs + 4 * (size_t)(act ? m : A.M - 1), R, a0, b0, tau, sign);
    spot_extent<KIND>(s, act, model[0], model[1], mv, sx, sy, c, E);
  }
#pragma unroll
  for (int i = 0; i < 23; ++i) {
    const float v = group_max<64>(E.e[i]);
    if (lane == 0) atomicMax(emax + i, __float_as_int(v));  // (v >= 0: ordered as integers)
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double S0 = 0.0, S1 = 0.0, S2 = 0.0;
    for (int p = 0; p < npt; ++p) {
      S0 += (double)mom[p][30];
      S1 += (double)mom[p][31];
      S2 += (double)mom[p][32];
    }
#pragma unroll
    for (int i = 0; i < 23; ++i) E.e[i] = __int_as_float(emax[i]);
    const long long id = base + top;
    store_node<KIND>(K, nodes + IACT_NODE_WORDS * id, balls + 4 * id, tau, bad == 0, 1e9f, mv,
                     sx, sy, mk3((float)S0, (float)S1, (float)S2), c, E);
  }
}

// ------------------------------------------------------------------ walk
// LDS of a block (byte offsets): the item's sources, the lists and sums at
// fixed offsets, then the image (fp64, see lds_add) or the image gradient (fp32)
// behind one spare entry, the staged table, the candidate list with each wave's
// selection from it, and the per-source gradient sums (fp64: value, then sum G nrwh m).
template <int MODE>
struct TreeLds {
  using Img = std::conditional_t<MODE == 0, double, float>;
  static constexpr uint32_t src = 0;  // u, value / |u|, da, db (, 1 / |e|): see scaled_inv
  static constexpr uint32_t l0 = src + (MODE == 2 ? 7u : 6u) * kTreeSources * 4u;
  static constexpr uint32_t wl = l0 + kTreeSources * 2u;
  static constexpr uint32_t pc = wl + kWaves * 2u * kTreeSources * 2u;
  static constexpr uint32_t red = pc + kWaves * 64u * 2u;
  static constexpr uint32_t img = red + 256u;
};
template <int MODE>
__host__ __device__ inline uint32_t tree_tab_at(int n_pixels) {
  return (TreeLds<MODE>::img +
          (uint32_t)(n_pixels + 1) * (uint32_t)sizeof(typename TreeLds<MODE>::Img) + 15u) &
         ~15u;
}
__host__ __device__ inline uint32_t tree_lc_at(uint32_t tab_at, int table_words) {
  return (tab_at + (uint32_t)table_words * 2u + 15u) & ~15u;
}
__host__ __device__ inline uint32_t tree_gm_at(uint32_t lc_at, int n_ob) {
  return (lc_at + (uint32_t)n_ob * 2u + 15u) & ~15u;
}
__host__ __device__ inline uint32_t tree_acc_at(uint32_t gm_at, int n_ob) {
  return gm_at + (uint32_t)((n_ob + 63) / 64) * 8u * (uint32_t)kWaves;
}
template <int MODE>
static size_t tree_lds_bytes(int n_pixels, int table_words, int n_ob, int n_acc) {
  const uint32_t lc = tree_lc_at(tree_tab_at<MODE>(n_pixels), table_words);
  return (size_t)tree_acc_at(tree_gm_at(lc, n_ob), n_ob) +
         (size_t)n_acc * kTreeSources * sizeof(double);
}
static int table_words(const DevSensor& S) {
  return S.kind == IACT_SENSOR_HEX ? (S.tq + 4) * (S.tr + 4) : 0;
}

// Hard pixel of a hit, as square_pixel_hit and hex_pixel_hit, on the 16-bit
// table (two border entries; negative entries are empty).
template <int KIND, bool EDGE>
IACT_DEV int tree_pixel(const DevSensor& S, const int16_t* tab, float u, float v, bool ok) {
  if (KIND == IACT_SENSOR_SQUARE) return square_pixel_hit<EDGE>(S, u, v, ok);
  const float a = floorf(fmaf(2.f, u, v)), b = floorf(fmaf(-2.f, v, -u)), c = floorf(v - u);
  const int row =
      floor_i32(__builtin_amdgcn_fmed3f(fmaf(a - c, 1.f / 3.f, 2.5f), 0.f, S.tq_f + 3.f));
  const int col =
      floor_i32(__builtin_amdgcn_fmed3f(fmaf(c - b, 1.f / 3.f, 2.5f), 0.f, S.tr_f + 3.f));
  const int pid = tab[__umul24((unsigned)row, (unsigned)(S.tr + 4)) + (unsigned)col];
  bool good = ok & (pid >= 0);
  if (EDGE && S.edge)
    good = good & !(hex_norm_axial(u - (float)(row - 2), v - (float)(col - 2)) > S.edge_thr);
  return good ? pid : -1;
}

constexpr int kUnresolved = -2;

// Where the spot of node nd lies for direction offset (da, db): a pixel that
// holds all of it, -1 if all of it misses the camera, kUnresolved otherwise
// (also for NaN offsets).
template <int KIND>
IACT_DEV int node_test(const DevSensor& S, const TreeParams& K, const int16_t* tab,
                       cptr<float> nd, float da, float db) {
  const float s = frcp(1.f + fmaf(nd[6], da, nd[7] * db));
  const float xa = s * da, xb = s * db;
  const float qu = fmaf(nd[2], xa, nd[3] * xb), qv = fmaf(nd[4], xa, nd[5] * xb);
  const float u = nd[0] + qu, v = nd[1] + qv;
  const float h1 = fmaf(nd[20], xa, nd[21] * xb), h2 = fmaf(nd[22], xa, nd[23] * xb);
  const float gu1 = fmaf(-qu, h1, fmaf(nd[12], xa, fmaf(nd[13], xb, nd[8])));
  const float gu2 = fmaf(-qu, h2, fmaf(nd[14], xa, fmaf(nd[15], xb, nd[9])));
  const float gv1 = fmaf(-qv, h1, fmaf(nd[16], xa, fmaf(nd[17], xb, nd[10])));
  const float gv2 = fmaf(-qv, h2, fmaf(nd[18], xa, fmaf(nd[19], xb, nd[11])));
  const float vt = nd[27] * (fabsf(da) + fabsf(db));
  if (KIND == IACT_SENSOR_SQUARE) {
    const float eu = fabsf(gu1) + fabsf(gu2) + (nd[24] + vt);
    const float ev = fabsf(gv1) + fabsf(gv2) + (nd[25] + vt);
    const float cu = floorf(u), cv = floorf(v);
    const bool off = (u + eu < 0.f) | (u - eu > S.wf) | (v + ev < 0.f) | (v - ev > S.hf);
    const float fu = fabsf(u - cu - 0.5f) + eu, fv = fabsf(v - cv - 0.5f) + ev;
    const bool one = (fu < K.hu) & (fv < K.hv) & (cu >= 0.f) & (cu < S.wf) &
                     (cv >= 0.f) & (cv < S.hf);
    const int pix = (int)(__umul24((unsigned)floor_i32(cv), (unsigned)S.width) +
                          (unsigned)floor_i32(cu));
    return off ? -1 : (one ? pix : kUnresolved);
  }
  const float e1 = fabsf(fmaf(2.f, gu1, gv1)) + fabsf(fmaf(2.f, gu2, gv2)) + (nd[24] + vt);
  const float e2 = fabsf(fmaf(2.f, gv1, gu1)) + fabsf(fmaf(2.f, gv2, gu2)) + (nd[25] + vt);
  const float e3 = fabsf(gu1 - gv1) + fabsf(gu2 - gv2) + (nd[26] + vt);
  const float a = floorf(fmaf(2.f, u, v)), b = floorf(fmaf(-2.f, v, -u)), c = floorf(v - u);
  const float cu = floorf(fmaf(a - c, 1.f / 3.f, 0.5f)), cv = floorf(fmaf(c - b, 1.f / 3.f, 0.5f));
  const float du = u - cu, dv = v - cv;
  const float fm = fmaxf(fmaxf(fabsf(fmaf(2.f, du, dv)) + e1, fabsf(fmaf(2.f, dv, du)) + e2),
                         fabsf(du - dv) + e3);
  const int row = floor_i32(__builtin_amdgcn_fmed3f(cu + 2.f, 0.f, S.tq_f + 3.f));
  const int col = floor_i32(__builtin_amdgcn_fmed3f(cv + 2.f, 0.f, S.tr_f + 3.f));
  const int code = tab[__umul24((unsigned)row, (unsigned)(S.tr + 4)) + (unsigned)col];
  // within 2 of the centre in every form lie only the cell and its neighbours
  return fm < K.hu ? max(code, -1) : (code == -2 && fm < 1.99f ? -1 : kUnresolved);
}

IACT_DEV int lanes_below(uint64_t mask) {  // set bits below the lane's own
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Wave-private list in LDS: one list grows from the front, one from the back.
struct WaveList {
  uint16_t* l;
  int n, m;  // entries at the front, at the back
};
IACT_DEV void push(WaveList& w, bool front, bool back, int v) {
  const uint64_t bf = __ballot(front), bb = __ballot(back);
  if (front) w.l[w.n + lanes_below(bf)] = (uint16_t)v;
  if (back) w.l[kTreeSources - 1 - (w.m + lanes_below(bb))] = (uint16_t)v;
  w.n += __popcll(bf);
  w.m += __popcll(bb);
}
IACT_DEV void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Shadow bits of a leaf's nq <= 16 samples for obstruction j along the lane's
// direction d: bit i is set when the ray of sample i (its point in lane i of
// myp) meets it.  The decisions are the per-ray tests' own (their expressions).
// Lanes without `need` may get any bits.  A cylinder that every ray of the
// leaf's ball (c, rho) can only meet on its side, well inside its ends and in
// front -- the line's closest approach to the axis, give or take the chord,
// lies within [0, h] and t > 0 by margins far above rounding -- is decided by
// its discriminant alone: a quarter of the whole test's instructions.
IACT_DEV uint32_t shade_bits(const iact_obstructions& ob, int j, f3 myp, int nq, f3 d, f3 c,
                             float rho, bool need) {
  uint32_t bits = 0u;
  const int c0 = ob.n_cylinders, c1 = c0 + ob.n_boxes;
  if (j < c0) {
    const cptr<float> q = as_const(ob.cylinders) + 8 * j;
    const CylDir D = cyl_dir(d, q);
    const f3 p1 = mk3(q[0], q[1], q[2]), ax = mk3(q[3], q[4], q[5]);
    const float h = q[6], r = q[7];
    float oca, cc;
    f3 ocp;
    cyl_axial(c - p1, ax, r, oca, ocp, cc);
    const float ia = frsq(D.a), dd = fmaf(D.rda, D.rda, D.a);
    const float tc = -dot(ocp, D.rdp) * (ia * ia), yc = fmaf(tc, D.rda, oca);
    const float dt = 1.01f * (r + rho) * ia, dy = fmaf(dt, fabsf(D.rda), 1.01f * rho);
    const float mg = fmaf(1e-4f, h, 5e-3f);
    const bool side = D.a > 1e-3f * dd && (tc - dt) * fsqrt(dd) > 5e-3f && yc - dy > mg &&
                      yc + dy < h - mg;
    if (__all(side || !need)) {
      cyl_axial(myp - p1, ax, r, oca, ocp, cc);  // of the lane's sample
      for (int i = 0; i < nq; ++i) {
        float b;
        bits |= cyl_disc(lane_value(ocp, i), lane_value(cc, i), D, b) >= 0.f ? 1u << i : 0u;
      }
    } else {
      for (int i = 0; i < nq; ++i)
        bits |= hit_cylinder_dir(lane_value(myp, i), D, q) < 1e10f ? 1u << i : 0u;
    }
  } else if (j < c1) {
    const cptr<float> q = as_const(ob.boxes) + 6 * (j - c0);
    const BoxDir D = box_dir(d);
    for (int i = 0; i < nq; ++i)
      bits |= hit_box_dir(lane_value(myp, i), D, q) < 1e10f ? 1u << i : 0u;
  } else {
    const int c2 = c1 + ob.n_spheres, c3 = c2 + ob.n_oriented_boxes;
    for (int i = 0; i < nq; ++i) {
      const f3 o = lane_value(myp, i);
      const float t = j < c2   ? hit_sphere(o, d, as_const(ob.spheres) + 4 * (j - c1))
                      : j < c3 ? hit_oriented_box(o, d, as_const(ob.oriented_boxes) + 15 * (j - c2))
                               : hit_triangle(o, d, as_const(ob.triangles) + 9 * (j - c3));
      bits |= t < 1e10f ? 1u << i : 0u;
    }
  }
  return bits;
}

// A far point source's u is kept as e times the power of two 2^x that brings |u|
// to (1, 2], with 1 / |e| = 2^x / |u|.  No decision and no term of a ray changes but
// by that power, and value / |u| keeps fp32's range: at |e| = 1e10 m, value / |e| of
// a flux of 1e-29 is subnormal, and so is its product with a small image gradient
// (rotation gradients of fluxes and image gradients of 2^-55 were off by 0.6 of the
// largest, ray by ray 2e-6).
IACT_DEV float scaled_inv(float ie) { return __builtin_amdgcn_frexp_mantf(ie); }  // 1 / |u|
IACT_DEV float per_metre(float v, float ie) {                                     // v 2^x
  return __builtin_ldexpf(v, __builtin_amdgcn_frexp_expf(ie));
}

// A work item is a block of kTreeSources sources against one top of a facet.
// The block's threads test the top for one source each and list the sources it
// does not resolve; each wave then takes patches of the top, tests the listed
// sources (64 at a time) on the patch, lists what is left, tests that on the
// patch's leaves and traces what is left there ray by ray -- always 64 pairs
// per instruction, whatever the fraction that splits.  MODE 0: image; 1:
// rotation gradients; 2: also positions, values, sources.
// VALU issue bounds it (82-87 % of the busy cycles), about half in the rays of
// unresolved leaves.  One ray per (sample, source) took 3693 us for 382 facets
// x 4096 samples x 4096 sources without obstructions and a square camera, this
// 960; 12732 against 4200 us for 875 x 1024 x 16384 behind a box and four masts,
// a hexagonal camera and smooth mirrors.  Eight waves share one image; a CU holds
// three blocks of a kernel of up to 80 VGPRs, two of the others (obstructed
// images 97-105, clear gradients 79-102).  Four-wave blocks: 5007 against 4611 us.
// Six waves per SIMD for the obstructed gradients: 6.23 against 6.43 ms for an
// iteration of five pointings; the image kernels need no bound (4528 against
// 4537 us with one).
template <int SRC, int KIND, int OBST, int MODE>
__global__ __launch_bounds__(64 * kWaves)
__attribute__((amdgpu_waves_per_eu(OBST && MODE ? 6 : 1))) void k_tree(AdjArgs B, TreeParams K) {
  const TraceArgs& A = B.T;
  constexpr int NS = kTreeSources, NT = 64 * kWaves;
  extern __shared__ __align__(16) char sm[];
  const int P = A.S.n_pixels;
  const int tw = KIND == IACT_SENSOR_HEX ? (A.S.tq + 4) * (A.S.tr + 4) : 0;
  const int n_ob = OBST ? n_obstructions(A.ob) : 0;
  using L = TreeLds<MODE>;
  auto* img = (typename L::Img*)(sm + L::img) + 1;  // (MODE > 0: the gradient; [-1] = 0)
  const uint32_t tab_at = tree_tab_at<MODE>(P), lc_at = tree_lc_at(tab_at, tw);
  int16_t* tab = (int16_t*)(sm + tab_at);
  float* sx = (float*)(sm + L::src);
  float *sy = sx + NS, *sz = sx + 2 * NS, *svi = sx + 3 * NS, *sda = sx + 4 * NS;
  float *sdb = sx + 5 * NS, *sinv = sx + 6 * NS;
  const uint32_t gm_at = tree_gm_at(lc_at, n_ob);
  double* acc = (double*)(sm + tree_acc_at(gm_at, n_ob));  // (MODE 2)
  uint16_t* l0 = (uint16_t*)(sm + L::l0);
  uint16_t* lc = (uint16_t*)(sm + lc_at);
  float* red = (float*)(sm + L::red);          // 32 floats
  int* cnt = (int*)(sm + L::red + 128);        // 4 ints
  uint32_t& work_next = *(uint32_t*)(sm + L::red + 144);
  double* tot = (double*)(sm + L::red + 160);  // 6 doubles
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint16_t* wl1 = (uint16_t*)(sm + L::wl) + (2 * wave) * NS;
  uint16_t* wl2 = wl1 + NS;
  uint16_t* pc = (uint16_t*)(sm + L::pc) + 64 * wave;
  uint64_t* gm = (uint64_t*)(sm + gm_at) + wave * ((n_ob + 63) / 64);
  if (tid == 0) img[-1] = 0;
  for (int i = tid; i < P; i += NT) img[i] = MODE ? B.grad_image[i] : 0.f;
  for (int i = tid; i < tw; i += NT) tab[i] = K.table[i];
  const cptr<float> fr = as_const(K.frame);
  const float a0 = fr[0], b0 = fr[1], tau = fr[2], sign = fr[3];
  const long long total = (long long)A.nf * A.M;
  // the lean per-ray trace serves the launch (see k_trace_sm)
  const bool lean = as_const((const uint32_t*)(A.recs + IACT_REC_WORDS * total))[0] == 0u &&
                    !A.S.edge && (KIND != IACT_SENSOR_SQUARE || A.S.v_scale == 1.f);
  const bool want_src = MODE == 2 && B.g_src, want_val = MODE == 2 && B.g_val;
  const bool want_pos = MODE == 2 && B.g_pos;

  // Items are handed out by a counter: their costs differ by far (a block of
  // sources off the camera ends at its top).  The next item is asked for while
  // one is walked.
  uint32_t* const work = (uint32_t*)K.frame + 4;
  for (uint32_t item = blockIdx.x; item < K.items;) {
    const uint32_t ftp = fdiv(item, K.d_sb);
    const int sb = (int)(item - ftp * K.n_sb);
    const uint32_t ft = fdiv(ftp, K.d_part);
    const int part = (int)(ftp - ft * K.n_part);
    const int f = (int)fdiv(ft, K.d_top), top = (int)ft - f * K.n_top;
    const int npt = (min(kTopSamples, A.M - top * kTopSamples) + 63) / 64;
    const long long nbase = (long long)f * K.per_facet;
    const cptr<float> tnode = as_const(K.nodes) + IACT_NODE_WORDS * (nbase + top);
    const cptr<float> tball = as_const(K.balls) + 4 * (nbase + top);
    uint32_t next = 0u;  // (thread 0's; used when the item is done)
    if (tid == 0) next = gridDim.x + atomicAdd(work, 1u);
    if (tid < 4) cnt[tid] = 0;
    if (MODE && tid < 6) tot[tid] = 0.0;
    if (MODE == 2) {
      for (int i = tid; i < K.n_acc * NS; i += NT) acc[i] = 0.0;
    }
    f3 T = mk3(0.f, 0.f, 0.f), Gp = mk3(0.f, 0.f, 0.f);  // lane's torque and dL/dpos
    constexpr float inf = __builtin_inff();
    // ---- the item's sources
    const cptr<float> fp = as_const(A.positions) + 3 * f;
    const f3 pos = mk3(fp[0], fp[1], fp[2]);
    f3 dsum = mk3(0.f, 0.f, 0.f);  // of the unit directions towards them
#pragma unroll
    for (int r = 0; r < NS; r += NT) {
      const int si = r + tid, sidx = sb * NS + si;
      const bool valid = sidx < A.ns;
      const int sl = valid ? sidx : A.ns - 1;
      const double* sp = A.sources + 3 * (size_t)sl;
      const f3 e = source_offset<SRC>(sp[0], sp[1], sp[2], pos);
      const float value = valid ? A.values[sl] : 0.f;
      const float ie = frsq(dot(e, e));
      const bool far = valid && (SRC != IACT_SOURCE_POINT || source_qs(A, e) == 0.f);
      const bool scaled = SRC == IACT_SOURCE_POINT && far;
      const float pw = scaled ? per_metre(1.f, ie) : 1.f;
      const float vi =
          value * (SRC == IACT_SOURCE_POINT ? (scaled ? scaled_inv(ie) : ie) : 1.f);
      const f3 U = sensor_dirs(A.S, e);
      const float iu = frcp(U.x);
      float da = fmaf(U.y, iu, -a0);
      float db = fmaf(U.z, iu, -b0);
      // a value that is not finite spreads as it does ray by ray: to every pixel
      // that one of its rays meets, shaded or not, and to every facet's gradients
      const bool finite = MODE || fabsf(vi) < inf;
      if (MODE && far) T = T + mk3(0.f * vi, 0.f * vi, 0.f * vi);
      if (MODE == 2 && scaled) Gp = Gp + mk3(0.f * vi, 0.f * vi, 0.f * vi);
      if (!(far && finite && U.x * ie * sign > 1e-3f && fabsf(da) + fabsf(db) <= tau)) {
        da = __builtin_nanf("");                // no node's test resolves it
        db = !far ? da : (finite ? 0.f : inf);  // (NaN: not far, inf: not shaded)
      }
      sx[si] = pw * e.x;
      sy[si] = pw * e.y;
      sz[si] = pw * e.z;
      svi[si] = vi;
      sda[si] = da;
      sdb[si] = db;
      if (MODE == 2) sinv[si] = SRC == IACT_SOURCE_POINT ? ie : 1.f;
      if (OBST && valid) dsum = dsum - ie * e;
    }
    // ---- obstruction candidates of the item: those the cone of its sources'
    // directions (with the parallax of near ones: a ray's direction is e + q,
    // |q| at most the distance of the top's farthest sample from the facet
    // position) can reach from the top's ball
    const f3 tc = mk3(tball[0], tball[1], tball[2]);
    const float trho = tball[3];
    f3 ax = mk3(0.f, 0.f, 1.f);
    float tn = -1.f;
    if (OBST && !A.cull_all) {
      const float wx = wave_sum(dsum.x), wy = wave_sum(dsum.y), wz = wave_sum(dsum.z);
      if (lane == 0) {
        red[3 * wave] = wx;
        red[3 * wave + 1] = wy;
        red[3 * wave + 2] = wz;
      }
      __syncthreads();
      f3 sum = mk3(0.f, 0.f, 0.f);
#pragma unroll
      for (int i = 0; i < kWaves; ++i)
        sum = sum + mk3(red[3 * i], red[3 * i + 1], red[3 * i + 2]);
      const float la = dot(sum, sum);
      if (la > 0.f) ax = frsq(la) * sum;
      // the largest tan(angle + parallax), from the chord (acos of a cosine
      // next to 1 would be off by 3e-4 rad); beyond 80 degrees: no culling
      float tg = 0.f;
      const f3 tq = tc - pos;
      const float qmax = trho + 1.0001f * fsqrt(dot(tq, tq));
#pragma unroll
      for (int r = 0; r < NS; r += NT) {
        const int si = r + tid;
        const f3 e = mk3(sx[si], sy[si], sz[si]);
        const float ie = frsq(dot(e, e));
        const f3 ch = -ie * e - ax;
        const float c2 = dot(ch, ch), cs = fmaf(-0.5f, c2, 1.f);
        float g = cs > 0.17f ? fsqrt(c2 * fmaf(-0.25f, c2, 1.f)) * frcp(cs) : 1e30f;
        if (SRC == IACT_SOURCE_POINT && !(sdb[si] == sdb[si])) {  // (far: below 2^-30)
          const float sp = qmax * ie, cp2 = fmaf(-sp, sp, 1.f);
          const float tp = cp2 > 0.03f ? sp * frsq(cp2) : 1e30f;
          g = g * tp < 0.9f ? (g + tp) * frcp(fmaf(-g, tp, 1.f)) : 1e30f;
        }
        if (!(g < 5.6f)) g = 1e30f;  // (NaN too)
        if (sb * NS + si < A.ns) tg = fmaxf(tg, g);
      }
      tg = group_max<64>(tg);
      if (lane == 0) red[24 + wave] = tg;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kWaves; ++i) tg = fmaxf(tg, red[24 + i]);
      // + 2e-4 rad
      tn = tg < 5.6f ? fmaf(1.0001f, tg, 2e-4f) * frcp(fmaf(-2e-4f, tg, 1.f)) : -1.f;
    } else {
      __syncthreads();
    }
    if (OBST) {
      for (int j0 = 0; j0 < n_ob; j0 += NT) {
        const int j = j0 + tid;
        const bool keep = j < n_ob && (tn < 0.f || obstruction_reaches(A.ob, j, tc, trho, ax, tn));
        const uint64_t bk = __ballot(keep);
        int at = 0;
        if (lane == 0 && bk) at = atomicAdd(cnt + 2, __popcll(bk));
        at = __builtin_amdgcn_readfirstlane(at);
        if (keep) lc[at + lanes_below(bk)] = (uint16_t)j;
      }
      __syncthreads();
    }
    const int nlc = OBST ? __builtin_amdgcn_readfirstlane(cnt[2]) : 0;
    // can a candidate (one per lane of id, chosen by mask) reach a ray of the
    // ball (c, rho) towards the lane's source?
    auto reached = [&](uint64_t mask, int id, f3 c, float rho, f3 d, bool act) {
      bool sus = false;
      while (mask != 0ull) {
        const int k = __builtin_ctzll(mask);
        mask &= mask - 1ull;
        sus |= line_reaches(A.ob, __builtin_amdgcn_readlane(id, k), c, rho, d);
        if (__all(sus || !act)) break;
      }
      return sus;
    };
    f3 Aw = mk3(0.f, 0.f, 0.f), Dw = mk3(0.f, 0.f, 0.f);
    float w1 = 0.f;
    // a pair resolved to pixel pix adds its node's rays at once
    auto add_pair = [&](cptr<float> nd, int pix, f3 u, float vi, int si) {
      if (pix < 0) return;
      const f3 S = mk3(nd[28], nd[29], nd[30]);
      const float us = dot(u, S);
      if (MODE == 0) {
        lds_add(img + pix, vi * us);
      } else {
        const float g = img[pix], w = g * vi;
        Aw = fma3(w, u, Aw);
        if (MODE == 2) {
          const float ie = sinv[si], i1 = SRC == IACT_SOURCE_POINT ? scaled_inv(ie) : 1.f;
          if (want_pos && SRC == IACT_SOURCE_POINT) {
            const float wm = per_metre(w, ie);
            w1 += wm;
            Dw = fma3(wm * us * (i1 * i1), u, Dw);
          }
          if (want_val) lds_add(acc + si, g * (us * i1));
          if (want_src) {
            lds_add(acc + NS + si, g * S.x);
            lds_add(acc + 2 * NS + si, g * S.y);
            lds_add(acc + 3 * NS + si, g * S.z);
          }
        }
      }
    };
    // the resolved pairs of one node share S: torque = S x sum w u
    auto end_node = [&](cptr<float> nd) {
      if (MODE && nd[31] != 0.f) {  // (an untested node's S may not be finite)
        const f3 S = mk3(nd[28], nd[29], nd[30]);
        T = T + cross(S, Aw);
        Aw = mk3(0.f, 0.f, 0.f);
        if (MODE == 2) {
          Gp = Gp + (fma3(w1, S, mk3(-Dw.x, -Dw.y, -Dw.z)));
          Dw = mk3(0.f, 0.f, 0.f);
          w1 = 0.f;
        }
      }
    };
    auto flush = [&]() {
      if (MODE) {
        const float t0 = wave_sum(T.x), t1 = wave_sum(T.y), t2 = wave_sum(T.z);
        float g0 = 0.f, g1 = 0.f, g2 = 0.f;
        if (want_pos) {
          g0 = wave_sum(Gp.x);
          g1 = wave_sum(Gp.y);
          g2 = wave_sum(Gp.z);
        }
        if (lane == 0) {
          const auto ad = [&](int i, float v) {
            __hip_atomic_fetch_add(tot + i, (double)v, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
          };
          ad(0, t0);
          ad(1, t1);
          ad(2, t2);
          if (want_pos) {
            ad(3, g0);
            ad(4, g1);
            ad(5, g2);
          }
        }
        T = mk3(0.f, 0.f, 0.f);
        Gp = mk3(0.f, 0.f, 0.f);
      }
    };
    // ---- the top
#pragma unroll
    for (int r = 0; r < NS; r += NT) {
      const int si = r + tid;
      const bool valid = sb * NS + si < A.ns;
      const f3 e = mk3(sx[si], sy[si], sz[si]);
      const bool far = valid && (SRC != IACT_SOURCE_POINT || sdb[si] == sdb[si]);
      bool sus = false;
      if (OBST && nlc > 0) {
        if (nlc <= 64 && !A.cull_all) {
          const int id = lane < nlc ? lc[lane] : 0;
          sus = reached(nlc == 64 ? ~0ull : (1ull << nlc) - 1ull, id, tc, trho,
                        -(frsq(dot(e, e)) * e), far);
        } else {
          sus = true;
        }
      }
      int code = kUnresolved;
      if (tnode[31] != 0.f) code = node_test<KIND>(A.S, K, tab, tnode, sda[si], sdb[si]);
      // (a suspect that misses the camera needs no shadow test)
      if (!far || (sus && code != -1)) code = kUnresolved;
      if (code >= 0 && part == 0) add_pair(tnode, code, e, svi[si], si);
      const bool split = far && code == kUnresolved, near = valid && !far;
      const uint64_t bf = __ballot(split), bn = __ballot(near);
      int at = 0;
      if (lane == 0) {
        if (bf) at = atomicAdd(cnt, __popcll(bf));
        if (bn) at |= atomicAdd(cnt + 1, __popcll(bn)) << 16;
      }
      at = __builtin_amdgcn_readfirstlane(at);
      if (split) l0[(at & 0xffff) + lanes_below(bf)] = (uint16_t)si;
      if (near) l0[NS - 1 - (at >> 16) - lanes_below(bn)] = (uint16_t)si;
    }
    end_node(tnode);
    flush();
    __syncthreads();
    const int n0 = __builtin_amdgcn_readfirstlane(cnt[0]);
    const int nn = __builtin_amdgcn_readfirstlane(cnt[1]);
    // ---- patches (and, where there are few patches for the waves, segments of
    // the list), taken by the waves one by one.  A part of one patch has as many
    // segments as waves where four of them would be longer than a batch of 64
    // sources (rough mirrors and near sources leave most of the list: 875 x 512
    // samples x 300 sources behind masts, 24 arcsec: 648 us with four, 492 so)
    const int p0 = (npt * part) / (int)K.n_part, p1 = (npt * (part + 1)) / (int)K.n_part;
    const int np1 = p1 - p0;
    const int left = n0 + nn;
    const int lseg = np1 >= kWaves ? 0 : 2 * np1 >= kWaves ? 1 : np1 > 1 || left <= 256 ? 2 : 3;
    const int nseg = 1 << lseg, nun = left == 0 ? 0 : (p1 - p0) << lseg;
    auto take = [&]() {
      int u = 0;
      if (lane == 0) u = atomicAdd(cnt + 3, 1);
      return __builtin_amdgcn_readfirstlane(u);
    };
    for (int un = take(); un < nun; un = take()) {
      const int p = p0 + (un >> lseg), seg = un & (nseg - 1);
      const int patch = top * (kTopSamples / 64) + p;
      const int mp = patch * 64, np = min(64, A.M - mp), nleaf = (np + 15) / 16;
      const int jp = f * A.M + mp;  // first record
      const cptr<float> pnode = as_const(K.nodes) + IACT_NODE_WORDS * (nbase + K.n_top + patch);
      const cptr<float> pball = as_const(K.balls) + 4 * (nbase + K.n_top + patch);
      const long long lid0 = nbase + K.n_top + K.n_patch + 4 * patch;
      const f3 bc = mk3(pball[0], pball[1], pball[2]);
      const float brho = pball[3];
      // the patch's candidates: groups of 64 of the item's list (rarely more
      // than one), one per lane, selected by a mask (kept in LDS)
      const int ngrp = OBST ? (nlc + 63) >> 6 : 0;
      bool cand = false;
      for (int g = 0; g < ngrp; ++g) {
        const int i = 64 * g + lane;
        const uint64_t mk =
            __ballot(i < nlc && (tn < 0.f || obstruction_reaches(A.ob, lc[min(i, nlc - 1)], bc,
                                                                 brho, ax, tn)));
        if (lane == 0) gm[g] = mk;
        cand |= mk != 0ull;
      }
      if (OBST) wave_lds_fence();
      int pid = 0;
      uint64_t pmask = 0ull;
      auto load_group = [&](int g) {
        pid = lc[min(64 * g + lane, nlc - 1)];
        const uint64_t mk = gm[g];
        pmask = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)mk) |
                (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(mk >> 32)) << 32;
      };

      // the gradients of a lane's rays of one source, N = sum G nrwh m
      auto add_rays = [&](f3 N, f3 u, float vi, int si) {
        T = T + vi * cross(N, u);
        if (MODE == 2) {
          const float ie = sinv[si], i1 = SRC == IACT_SOURCE_POINT ? scaled_inv(ie) : 1.f;
          const float un = dot(u, N) * i1;
          if (want_pos && SRC == IACT_SOURCE_POINT)
            Gp = Gp + per_metre(vi, ie) * fma3(-un * i1, u, N);
          if (want_val) lds_add(acc + si, un);
          if (want_src) {
            lds_add(acc + NS + si, N.x);
            lds_add(acc + 2 * NS + si, N.y);
            lds_add(acc + 3 * NS + si, N.z);
          }
        }
      };
      // Rays of listed pairs, with the per-ray kernels' arithmetic: ns samples
      // from record j0.  Full waves: lane = source, the records one after
      // another in scalar registers, pixel runs as in k_trace_sm.  A rest of at
      // most 48 pairs: the wave is 4 SPL sources times 16 / SPL parts of sixteen
      // samples, SPL records per lane in vector registers, so a short list
      // fills the lanes.  BITS: shadow bits per pair (short lists, second form).
      // SPL: four took 1050 us against 1163 with one (and fewer adds per ray)
      // without obstructions; beside the shadow code four spills the waves'
      // occupancy (7004 us with obstructions, 4359 with two, 4528 with one).
      auto trace_far = [&](auto gen, auto bits_t, const uint16_t* list, const uint16_t* bits,
                           int n, int j0, int ns) {
        constexpr bool GEN = decltype(gen)::value;
        constexpr bool BITS = decltype(bits_t)::value;
        int done = 0;
        if (!BITS) {
          for (; n - done > 48; done += 64) {
            const bool act = done + lane < n;
            const int si = list[act ? done + lane : done];
            const f3 u = mk3(sx[si], sy[si], sz[si]);
            const float vi = act ? svi[si] : 0.f;
            const f3 Ud = sensor_dirs(A.S, u);
            const float rs = SRC == IACT_SOURCE_POINT ? frsq(dot(u, u)) : 1.f;
            int run_pix = -1;
            float run_l = 0.f;
            f3 N = mk3(0.f, 0.f, 0.f);
            const float4* rp = (const float4*)A.recs + 4 * (size_t)j0;
            RecRaw cur = fetch_record(rp);
            for (int j = 0; j < ns; ++j) {
              rp += 4;
              const RecRaw nxt = fetch_record(rp);
              const Sample s = unpack_record(cur);
              const float cu = dot(u, s.m);
              float gu, gv;
              const bool ok = grid_hit<GEN>(s.G, s.N, Ud, cu, gu, gv, rs);
              const int pix = tree_pixel<KIND, GEN>(A.S, tab, gu, gv, ok);
              if (MODE == 0) {
                if (pix != run_pix) {
                  lds_add(img + run_pix, vi * run_l);
                  run_pix = pix;
                  run_l = 0.f;
                }
                run_l = fmaf(cu, s.nrwh, run_l);
              } else {
                N = fma3(img[pix] * s.nrwh, s.m, N);
              }
              cur = nxt;
            }
            if (MODE == 0)
              lds_add(img + run_pix, vi * run_l);
            else if (act)
              add_rays(N, u, vi, si);
          }
          if (done >= n) return;
        }
        constexpr int SPL = !OBST ? 4 : MODE == 0 ? 2 : 1, SRCS = 4 * SPL;
        const int part = lane / SRCS, slot = lane % SRCS;
#pragma unroll 1
        for (int q = 0; q < ns; q += 16) {
          // (samples past the end of the run are its last one again, dropped)
          Sample smp[SPL];
          const int sm0 = q + SPL * part;
#pragma unroll
          for (int k = 0; k < SPL; ++k) {
            const float4* rp = (const float4*)A.recs + 4 * (size_t)(j0 + min(sm0 + k, ns - 1));
            smp[k] = unpack_record(RecRaw{rp[0], rp[1], rp[2], rp[3]});
          }
#pragma unroll 1
          for (int i = done; i < n; i += SRCS) {
            const int at = min(i + slot, n - 1);
            const int si = list[at];
            const uint32_t drop = (BITS ? (uint32_t)bits[at] >> (SPL * part) : 0u) |
                                  (i + slot < n ? ~0u << min(max(ns - sm0, 0), SPL) : ~0u);
            const f3 u = mk3(sx[si], sy[si], sz[si]);
            const float vi = svi[si];
            const f3 Ud = sensor_dirs(A.S, u);
            const float rs = SRC == IACT_SOURCE_POINT ? frsq(dot(u, u)) : 1.f;
            int run_pix = -1;
            float run_l = 0.f;
            f3 N = mk3(0.f, 0.f, 0.f);
#pragma unroll
            for (int k = 0; k < SPL; ++k) {
              const Sample& s = smp[k];
              const float cu = dot(u, s.m);
              float gu, gv;
              const bool ok = grid_hit<GEN>(s.G, s.N, Ud, cu, gu, gv, rs);
              const int pix = tree_pixel<KIND, GEN>(A.S, tab, gu, gv,
                                                    ok & (((drop >> k) & 1u) == 0u));
              if (MODE == 0) {
                if (pix != run_pix) {
                  if (k > 0) lds_add(img + run_pix, vi * run_l);
                  run_pix = pix;
                  run_l = 0.f;
                }
                run_l = fmaf(cu, s.nrwh, run_l);
              } else {
                N = fma3(img[pix] * s.nrwh, s.m, N);
              }
            }
            if (MODE == 0)
              lds_add(img + run_pix, vi * run_l);
            else
              add_rays(N, u, vi, si);
          }
        }
      };

      // ---- far sources
      const int s0 = n0 * seg / nseg, ns0 = n0 * (seg + 1) / nseg - s0;
      if (ns0 > 0) {
        bool leaves = false;
        for (int q = 0; q < nleaf; ++q)
          leaves |= as_const(K.nodes)[IACT_NODE_WORDS * (lid0 + q) + 31] != 0.f;
        const bool ptest = npt > 1 && pnode[31] != 0.f;
        const uint16_t* l1 = l0 + s0;
        int n1 = ns0, m1 = 0;
        if (ptest || cand) {
          WaveList w = {wl1, 0, 0};
          for (int i = 0; i < ns0; i += 64) {
            const bool act = i + lane < ns0;
            const int si = l0[s0 + (act ? i + lane : 0)];
            const f3 u = mk3(sx[si], sy[si], sz[si]);
            bool sus = false;
            if (OBST && cand) {
              const f3 dn = -(frsq(dot(u, u)) * u);
              for (int g = 0; g < ngrp; ++g) {
                load_group(g);
                sus |= pmask != 0ull && (A.cull_all || reached(pmask, pid, bc, brho, dn, act));
              }
              if (MODE == 0) sus = sus && sdb[si] != inf;
            }
            int code = kUnresolved;
            if (ptest) code = node_test<KIND>(A.S, K, tab, pnode, sda[si], sdb[si]);
            if (!act || (sus && code != -1)) code = kUnresolved;
            if (code >= 0) add_pair(pnode, code, u, svi[si], si);
            const bool left = act && code == kUnresolved;
            push(w, left && !sus, left && sus, si);
          }
          wave_lds_fence();
          end_node(pnode);
          l1 = wl1;
          n1 = w.n;
          m1 = w.m;
        }
        // ---- unshadowed pairs of the patch: leaf by leaf (a patch whose leaves
        // are not worth a test is traced as one run)
        for (int q = 0; n1 > 0 && q < (leaves ? nleaf : 1); ++q) {
          const cptr<float> lnode = as_const(K.nodes) + IACT_NODE_WORDS * (lid0 + q);
          const uint16_t* l2 = l1;
          int n2 = n1;
          if (leaves && nleaf > 1 && lnode[31] != 0.f) {
            WaveList w = {wl2, 0, 0};
            for (int i = 0; i < n1; i += 64) {
              const bool act = i + lane < n1;
              const int si = l1[act ? i + lane : 0];
              int code = node_test<KIND>(A.S, K, tab, lnode, sda[si], sdb[si]);
              if (!act) code = kUnresolved;
              if (code >= 0) add_pair(lnode, code, mk3(sx[si], sy[si], sz[si]), svi[si], si);
              push(w, act && code == kUnresolved, false, si);
            }
            wave_lds_fence();
            end_node(lnode);
            l2 = wl2;
            n2 = w.n;
          }
          if (n2 == 0) continue;
          const int nq = leaves ? min(16, np - 16 * q) : np;
          if (lean)
            trace_far(std::false_type{}, std::false_type{}, l2, nullptr, n2, jp + 16 * q, nq);
          else
            trace_far(std::true_type{}, std::false_type{}, l2, nullptr, n2, jp + 16 * q, nq);
        }
        // ---- shadow suspects of the patch, 64 at a time: per leaf the shadow
        // bits of each pair's sixteen rays, candidate by candidate and only
        // those that reach the patch (then the leaf) along the pair's direction.
        // A pair whose pixel is known needs no rays: its lit samples' sum.
        for (int i = 0; OBST && i < m1; i += 64) {
          const bool act = i + lane < m1;
          const int si = wl1[NS - 1 - (act ? i + lane : 0)];
          const f3 u = mk3(sx[si], sy[si], sz[si]);
          const float vi = svi[si], da1 = sda[si], db1 = sdb[si];
          const f3 dn = -(frsq(dot(u, u)) * u);
          const f3 ds = SRC == IACT_SOURCE_POINT ? dn : -u;  // as the per-ray tests have it
          uint64_t pm = 0ull, um = 0ull;  // the lane's, the wave's candidates
          auto patch_group = [&](int g) {
            load_group(g);
            pm = um = 0ull;
            for (uint64_t b = pmask; b != 0ull;) {
              const int k = __builtin_ctzll(b);
              b &= b - 1ull;
              const bool r =
                  act && (A.cull_all ||
                          line_reaches(A.ob, __builtin_amdgcn_readlane(pid, k), bc, brho, dn));
              pm |= r ? 1ull << k : 0ull;
              um |= __any(r) ? 1ull << k : 0ull;
            }
          };
          for (int q = 0; q < nleaf; ++q) {
            const cptr<float> lnode = as_const(K.nodes) + IACT_NODE_WORDS * (lid0 + q);
            const cptr<float> lb = as_const(K.balls) + 4 * (lid0 + q);
            const f3 lcn = mk3(lb[0], lb[1], lb[2]);
            const float lrho = lb[3];
            const int nq = min(16, np - 16 * q), j0 = jp + 16 * q;
            int code = kUnresolved;
            if (lnode[31] != 0.f) code = node_test<KIND>(A.S, K, tab, lnode, da1, db1);
            const bool need = act && code != -1;
            // lane i < 16 holds sample i's point
            const float* pr = A.recs + IACT_REC_WORDS * (size_t)(j0 + min(lane & 15, nq - 1)) + 13;
            const f3 myp = mk3(pr[0], pr[1], pr[2]);
            const uint32_t all = (1u << nq) - 1u;
            uint32_t bits = 0u;
            for (int g = 0; g < ngrp; ++g) {
              if (ngrp > 1 || q == 0) patch_group(g);
              uint64_t lm = um;
              if (!A.cull_all)
                lm &= __ballot(((um >> lane) & 1ull) &&
                               (tn < 0.f || obstruction_reaches(A.ob, pid, lcn, lrho, ax, tn)));
              while (lm != 0ull) {
                const int k = __builtin_ctzll(lm);
                lm &= lm - 1ull;
                const int j = __builtin_amdgcn_readlane(pid, k);
                bool r = need && ((pm >> k) & 1ull) && bits != all;
                if (!__any(r)) continue;
                r = r && (A.cull_all || line_reaches(A.ob, j, lcn, lrho, dn));
                if (!__any(r)) continue;
                const uint32_t tb = shade_bits(A.ob, j, myp, nq, ds, lcn, lrho, r);
                bits |= r ? tb : 0u;
              }
            }
            const bool res = code >= 0 && act;
            if (res && bits == 0u) add_pair(lnode, code, u, vi, si);
            end_node(lnode);
            const bool part = res && bits != 0u && bits != all;
            if (__any(part)) {
              f3 N = mk3(0.f, 0.f, 0.f);
              for (int s = 0; s < nq; ++s) {
                const Sample smp = unpack_record(fetch_record((const float4*)A.recs + 4 * (size_t)(j0 + s)));
                N = fma3(((bits >> s) & 1u) ? 0.f : smp.nrwh, smp.m, N);
              }
              if (part) {
                if (MODE == 0)
                  lds_add(img + code, vi * dot(u, N));
                else
                  add_rays(img[code] * N, u, vi, si);
              }
            }
            const bool left = act && code == kUnresolved && bits != all;
            if (__any(left)) {
              WaveList w = {wl2, 0, 0}, wb = {pc, 0, 0};
              push(w, left, false, si);
              push(wb, left, false, (int)bits);
              wave_lds_fence();
              if (lean)
                trace_far(std::false_type{}, std::true_type{}, wl2, pc, w.n, j0, nq);
              else
                trace_far(std::true_type{}, std::true_type{}, wl2, pc, w.n, j0, nq);
              wave_lds_fence();
            }
          }
        }
      }

      // ---- near sources (u = q + e differs from sample to sample): per ray
      const int t0 = nn * seg / nseg, nt = nn * (seg + 1) / nseg - t0;
      if (SRC == IACT_SOURCE_POINT && nt > 0) {
        for (int i = 0; i < nt; i += 64) {
          const bool act = i + lane < nt;
          const int si = l0[NS - 1 - (t0 + (act ? i + lane : 0))];
          const f3 e1 = mk3(sx[si], sy[si], sz[si]);
          // (value / |e| is kept: the value again from memory)
          const float val = act ? A.values[min(sb * NS + si, A.ns - 1)] : 0.f;
          int run_pix = -1;
          float run_v = 0.f, gval = 0.f;
          f3 gs3 = mk3(0.f, 0.f, 0.f);
          const float4* rp = (const float4*)A.recs + 4 * (size_t)jp;
          RecRaw cur = fetch_record(rp);
          for (int j = 0; j < np; ++j) {
            rp += 4;
            const RecRaw nxt = fetch_record(rp);
            const Sample s = unpack_record(cur);
            const f3 u = s.q + e1;
            const float i1 = frsq(dot(u, u));
            const float cu = dot(u, s.m);
            const f3 d = i1 * u;
            float sh = 1.f;
            if (OBST && cand) {
              for (int g = 0; g < ngrp; ++g) {
                if (ngrp > 1 || j == 0) load_group(g);
                sh *= shadow_factor_list(A.ob, pid, pmask, s.p, -d, act);
              }
            }
            float gu, gv;
            const bool ok = grid_hit<true>(s.G, s.N, sensor_dirs(A.S, u), cu, gu, gv, i1);
            const int pix = tree_pixel<KIND, true>(A.S, tab, gu, gv, ok && act);
            const float c2 = cu * i1;
            if (MODE == 0) {
              if (pix != run_pix) {
                lds_add(img + run_pix, val * run_v);
                run_pix = pix;
                run_v = 0.f;
              }
              run_v = fmaf(c2 * sh, s.nrwh, run_v);
            } else {
              // dL/dn = dc d, dL/dp = dc / |u| (n - (d.n) d), dc = G value sh nrw;
              // n = -m / 2, nrw = -2 nrwh, d.n = -c2 / 2
              const float g = img[pix] * sh;
              const float b = g * s.nrwh, bv = b * val;
              const f3 gp = (bv * i1) * fma3(-c2, d, s.m);
              T = T + cross(s.q, gp) + cross(bv * s.m, d);
              Gp = Gp + gp;
              if (MODE == 2) {
                gval = fmaf(b, c2, gval);
                gs3 = gs3 - gp;
              }
            }
            cur = nxt;
          }
          if (MODE == 0) lds_add(img + run_pix, val * run_v);
          if (MODE == 2 && act) {
            if (want_val) lds_add(acc + si, gval);
            if (want_src) {
              lds_add(acc + NS + si, gs3.x);
              lds_add(acc + 2 * NS + si, gs3.y);
              lds_add(acc + 3 * NS + si, gs3.z);
            }
          }
        }
      }
      flush();
    }
    if (tid == 0) work_next = next;
    __syncthreads();
    if (MODE) {
      if (tid < 3 && tot[tid] != 0.0) unsafeAtomicAdd(B.torque + 3 * f + tid, tot[tid]);
      if (want_pos && tid < 3 && tot[3 + tid] != 0.0)
        unsafeAtomicAdd(B.g_pos + 3 * f + tid, tot[3 + tid]);
    }
    for (int r = 0; (want_val || want_src) && r < NS; r += NT) {
      const int si = r + tid, sidx = sb * NS + si;
      if (sidx >= A.ns) break;
      const long long so = B.src_perm ? (long long)B.src_perm[sidx] : (long long)sidx;
      if (want_val && acc[si] != 0.0) unsafeAtomicAdd(B.g_val + so, acc[si]);
      if (want_src) {
        const f3 N = mk3((float)acc[NS + si], (float)acc[2 * NS + si], (float)acc[3 * NS + si]);
        const f3 d = scaled_inv(sinv[si]) * mk3(sx[si], sy[si], sz[si]);
        // far: dL/dsrc = -value / |u| (N - (d.N) d); near sources have theirs
        // summed already; parallel: value N (1 / |u| is 1)
        const f3 g = SRC == IACT_SOURCE_POINT
                         ? (sdb[si] == sdb[si]
                                ? per_metre(-svi[si], sinv[si]) * fma3(-dot(d, N), d, N)
                                : N)
                         : svi[si] * N;
        unsafeAtomicAdd(B.g_src + 3 * so, (double)g.x);
        unsafeAtomicAdd(B.g_src + 3 * so + 1, (double)g.y);
        unsafeAtomicAdd(B.g_src + 3 * so + 2, (double)g.z);
      }
    }
    item = __builtin_amdgcn_readfirstlane(work_next);
    if (MODE) __syncthreads();  // (the sums above are read before they are cleared)
  }
  if (MODE == 0) {
    __syncthreads();
    float* part = A.partials + (size_t)blockIdx.x * P;
    for (int i = tid; i < P; i += NT) part[i] = (float)img[i];
  }
}

// The image from the blocks' partial images, summed in fp64: one block per 64
// pixels, a wave per sixteenth of the partials.  Leaves the walk's work counter
// cleared for a gradient walk of the same tree.
__global__ __launch_bounds__(1024) void k_sum_partials(const float* part, int n, int P, float* out,
                                                       uint32_t* work) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *work = 0u;
  __shared__ double red[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + lane;
  double s = 0.0;
  if (i < P) {
    int b = w;
    for (; b + 112 < n; b += 128) {  // eight loads in flight
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = part[(size_t)(b + 16 * k) * P + i];
#pragma unroll
      for (int k = 0; k < 8; ++k) s += (double)v[k];
    }
    for (; b < n; b += 16) s += (double)part[(size_t)b * P + i];
  }
  red[w][lane] = s;
  __syncthreads();
  if (w == 0 && i < P) {
    for (int k = 1; k < 16; ++k) s += red[k][lane];
    out[i] = (float)s;
  }
}

// ------------------------------------------------------------------ host
static size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

TreeLayout tree_layout(const iact_scene& sc, int ns, bool sort, int grid) {
  const int nf = sc.facets.n_facets, M = sc.facets.n_samples;
  TreeLayout T;
  memset(&T, 0, sizeof(T));
  T.n_top = (M + kTopSamples - 1) / kTopSamples;
  T.n_patch = (M + 63) / 64;
  T.n_leaf = (M + 15) / 16;
  const size_t nodes = (size_t)nf * (T.n_top + T.n_patch + T.n_leaf);
  // two records of padding after the table (the trace prefetches one ahead)
  size_t o = align256((size_t)IACT_REC_WORDS * ((size_t)nf * M + 2) * sizeof(float));
  T.nodes = o;
  o += nodes * IACT_NODE_WORDS * sizeof(float);
  T.balls = o;
  o = align256(o + nodes * 4 * sizeof(float));
  T.frame = o;
  o += 256;
  T.table = o;
  if (sc.sensor.kind == IACT_SENSOR_HEX)
    o += (size_t)(sc.sensor.table_q + 4) * (sc.sensor.table_r + 4) * sizeof(int16_t);
  o = align256(o);
  T.sort = sort;
  if (sort) {
    T.sws = o;
    o = align256(o + sort_workspace_bytes(ns, 1));
    T.perm = o;
    o = align256(o + (size_t)ns * sizeof(int32_t));
    T.src = o;
    o = align256(o + (size_t)ns * 3 * sizeof(double));
    T.val = o;
    o = align256(o + (size_t)ns * sizeof(float));
  }
  T.sums = o;
  // the blocks' partial images, or the facets' torques
  const size_t img = (size_t)grid * sc.sensor.n_pixels * sizeof(float);
  const size_t tq = (size_t)3 * nf * sizeof(double);
  T.end = o + (img > tq ? img : tq);
  return T;
}

// Blocks of a full grid (24 waves per CU: more than registers admit of some
// kernels, whose last blocks then find the queue empty).
int tree_max_grid(const DevInfo& dev) { return dev.n_cu * (24 / kWaves); }

bool tree_serves(const TraceArgs& A, int mode, int n_acc, const DevInfo& dev, LaunchShape& shp) {
  if (A.layout != 2 || A.per_ray || A.S.splat || A.n_stages > 0 || A.det || A.nf <= 0 || A.ns <= 0) return false;
  if (A.S.n_pixels > 32767) return false;
  const int n_ob = n_obstructions(A.ob);
  if (n_ob > 65535) return false;
  // Fewer sources leave a block's lanes idle: gradients of 875 x 1000 samples x
  // 100 sources behind masts, 1630 us in the tree, 1180 ray by ray.
  if (A.ns < 128) return false;
  // Without shadows to save, the preparation and the tests (some 0.2 ns per sample
  // and top) and the tails of few items have to be repaid by runs on one pixel,
  // which rough mirrors and near sources have few of.  Images of 2e8 rays: 12 m
  // dish, 382 x 512 x 1024, mirrors of 24 arcsec, 430 us against 354; 28 m dish,
  // smooth, far, 875 x 1024 x 300: 344 against 468; gradients of 8.75e8 rays 2730
  // against 2560, rough; 6.4e9 smooth ones 1020 against 3680.
  if (n_ob == 0 && (double)A.nf * A.M * A.ns < 1.5e9) return false;
  const int tw = table_words(A.S);
  const size_t lds = mode == 0   ? tree_lds_bytes<0>(A.S.n_pixels, tw, n_ob, 0)
                     : mode == 1 ? tree_lds_bytes<1>(A.S.n_pixels, tw, n_ob, 0)
                                 : tree_lds_bytes<2>(A.S.n_pixels, tw, n_ob, n_acc);
  if (lds > 65536) return false;
  // k_tree_nodes has 256 threads per (facet, top), and a grid of 2^32 threads wraps
  const long long tops = (long long)A.nf * ((A.M + kTopSamples - 1) / kTopSamples);
  if (tops >= (1ll << 24)) return false;
  const long long items = tops * (((long long)A.ns + kTreeSources - 1) / kTreeSources);
  if (items >= (1ll << 27)) return false;
  // the rows (An, Au, Av) must be invertible (they are for a rotation)
  const f3 n = A.S.An, u = A.S.Au, v = A.S.Av;
  const double det = (double)n.x * ((double)u.y * v.z - (double)u.z * v.y) -
                     (double)n.y * ((double)u.x * v.z - (double)u.z * v.x) +
                     (double)n.z * ((double)u.x * v.y - (double)u.y * v.x);
  const double size = sqrt((double)u.x * u.x + (double)u.y * u.y + (double)u.z * u.z) *
                      sqrt((double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z);
  if (!(fabs(det) > 1e-2 * size) || !isfinite(size) || !(size > 0.0)) return false;
  // as many blocks as the CUs' LDS holds (160 KB each)
  const int held = (int)fmin(24.0 / kWaves, floor(163840.0 / (double)lds));
  long long grid = (long long)dev.n_cu * held;
  shp.threads = 64 * kWaves;
  shp.lds = lds;
  shp.full_grid = (int)grid;
  // (items may be split into up to 16 parts)
  shp.grid = (int)(16 * items < grid ? 16 * items : grid);
  return true;
}

static TreeParams tree_args(TraceArgs& A, const TreeLayout& T, void* workspace, int full_grid) {
  char* ws = (char*)workspace;
  TreeParams K;
  A.recs = (const float*)ws;
  K.nodes = (const float*)(ws + T.nodes);
  K.balls = (const float*)(ws + T.balls);
  K.frame = (const float*)(ws + T.frame);
  K.table = (const int16_t*)(ws + T.table);
  K.n_top = T.n_top;
  K.n_patch = T.n_patch;
  K.n_leaf = T.n_leaf;
  K.per_facet = T.n_top + T.n_patch + T.n_leaf;
  K.n_sb = (uint32_t)((A.ns + kTreeSources - 1) / kTreeSources);
  // Items cost up to some 400 us (a block of sources on the camera against
  // 1024 samples), so a launch of few of them is split by patches until every
  // block has six: an iteration over 5 pointings of 1000 sources against 875
  // facets of 1024 samples (1750 items per launch) takes 7.16 ms with whole
  // tops and 6.92 ms in parts.  Parts repeat the top's tests, so no more.
  const uint32_t whole = (uint32_t)A.nf * (uint32_t)T.n_top * K.n_sb;
  const int most = T.n_patch < 16 ? T.n_patch : 16;
  K.n_part = 1;
  while (2 * K.n_part <= (uint32_t)most && (uint64_t)whole * K.n_part < 6ull * (uint64_t)full_grid)
    K.n_part *= 2;
  K.items = whole * K.n_part;
  K.d_sb = make_fastdiv(K.n_sb);
  K.d_part = make_fastdiv(K.n_part);
  K.d_top = make_fastdiv((uint32_t)T.n_top);
  const double r[3][3] = {{A.S.An.x, A.S.An.y, A.S.An.z},
                          {A.S.Au.x, A.S.Au.y, A.S.Au.z},
                          {A.S.Av.x, A.S.Av.y, A.S.Av.z}};
  double c[3][3];  // cofactors: inverse = transpose(c) / det
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
      c[i][j] = r[i1][j1] * r[i2][j2] - r[i1][j2] * r[i2][j1];
    }
  const double det = r[0][0] * c[0][0] + r[0][1] * c[0][1] + r[0][2] * c[0][2];
  for (int j = 0; j < 3; ++j) {
    K.b0[j] = (float)(c[0][j] / det);
    K.b1[j] = (float)(c[1][j] / det);
    K.b2[j] = (float)(c[2][j] / det);
  }
  K.n_au = (float)sqrt(r[1][0] * r[1][0] + r[1][1] * r[1][1] + r[1][2] * r[1][2]);
  K.n_av = (float)sqrt(r[2][0] * r[2][0] + r[2][1] * r[2][1] + r[2][2] * r[2][2]);
  if (A.S.kind == IACT_SENSOR_SQUARE) {
    K.hu = 0.5f - (A.S.edge ? A.S.edge_width * A.S.inv_dx : 0.f);
    K.hv = 0.5f - (A.S.edge ? A.S.edge_width * A.S.inv_dy : 0.f);
  } else {
    K.hu = K.hv = A.S.edge ? fminf(A.S.edge_thr, 1.f) : 1.f;
  }
  return K;
}

template <int SRC, int KIND>
static const void* pick_tree(const TraceArgs& A, int mode) {
  const bool ob = has_obstructions(A.ob);
  switch (mode) {
    case 0:
      return ob ? (const void*)k_tree<SRC, KIND, 1, 0> : (const void*)k_tree<SRC, KIND, 0, 0>;
    case 1:
      return ob ? (const void*)k_tree<SRC, KIND, 1, 1> : (const void*)k_tree<SRC, KIND, 0, 1>;
    default:
      return ob ? (const void*)k_tree<SRC, KIND, 1, 2> : (const void*)k_tree<SRC, KIND, 0, 2>;
  }
}

// The whole trace: sorted sources in obstructed scenes (an item's sources then
// bound a narrow bundle), frame, records, nodes, walk.  built: an image launch
// of the same scene, sources and stream has just left all of it but the walk in
// the workspace.
int launch_tree(AdjArgs& B, const TreeLayout& T, void* workspace, const LaunchShape& shp,
                int source_type, int mode, int n_acc, bool built, hipStream_t st) {
  TraceArgs& A = B.T;
  char* ws = (char*)workspace;
  TreeParams K = tree_args(A, T, workspace, shp.full_grid);
  K.n_acc = n_acc;
  hipError_t e;
  const bool hex = A.S.kind == IACT_SENSOR_HEX;
  if (T.sort) {
    int32_t* pm = (int32_t*)(ws + T.perm);
    double* so = (double*)(ws + T.src);
    float* vo = (float*)(ws + T.val);
    if (!built) {
      e = launch_sort_sources(A.sources, A.values, A.ns, nullptr, 1, source_type, ws + T.sws, pm,
                              so, vo, st);
      if (e != hipSuccess) return hip_error(e, "source sort");
    }
    A.sources = so;
    A.values = vo;
    B.src_perm = pm;
  }
  if (!built) {
    e = launch_records(A, (float*)workspace, st);
    if (e != hipSuccess) return hip_error(e, "k_sample_records");
    const int tw = table_words(A.S);
    hipLaunchKernelGGL(k_tree_frame, dim3(1 + (tw + 1023) / 1024), dim3(1024), 0, st, A.sources,
                       A.ns, source_type, A.S, (float*)(ws + T.frame), (int16_t*)(ws + T.table));
    e = hipGetLastError();
    if (e != hipSuccess) return hip_error(e, "k_tree_frame");
    const dim3 ng(A.nf * T.n_top);
    if (hex)
      hipLaunchKernelGGL(k_tree_nodes<IACT_SENSOR_HEX>, ng, dim3(256), 0, st, A, K,
                         (float*)(ws + T.nodes), (float*)(ws + T.balls));
    else
      hipLaunchKernelGGL(k_tree_nodes<IACT_SENSOR_SQUARE>, ng, dim3(256), 0, st, A, K,
                         (float*)(ws + T.nodes), (float*)(ws + T.balls));
    e = hipGetLastError();
    if (e != hipSuccess) return hip_error(e, "k_tree_nodes");
  }
  const void* k =
      source_type == IACT_SOURCE_POINT
          ? (hex ? pick_tree<IACT_SOURCE_POINT, IACT_SENSOR_HEX>(A, mode)
                 : pick_tree<IACT_SOURCE_POINT, IACT_SENSOR_SQUARE>(A, mode))
          : (hex ? pick_tree<IACT_SOURCE_PARALLEL, IACT_SENSOR_HEX>(A, mode)
                 : pick_tree<IACT_SOURCE_PARALLEL, IACT_SENSOR_SQUARE>(A, mode));
  AdjArgs b = B;
  void* args[] = {&b, &K};
  const int grid = (int)min((uint32_t)shp.grid, K.items);
  e = hipLaunchKernel(k, dim3(grid), dim3(shp.threads), args, shp.lds, st);
  if (e != hipSuccess) return hip_error(e, "k_tree");
  if (mode == 0) {
    hipLaunchKernelGGL(k_sum_partials, dim3((A.S.n_pixels + 63) / 64), dim3(1024), 0, st,
                       A.partials, grid, A.S.n_pixels, A.out, (uint32_t*)(ws + T.frame) + 4);
    e = hipGetLastError();
    if (e != hipSuccess) return hip_error(e, "k_sum_partials");
  }
  return IACT_OK;
}

}  // namespace iact
