// nb_cycle.hip -- the rest of one compute cycle on gfx950: FP64 reference-order force, pair sort,
// elastic collision resolution, FP64 update, source-stream maintenance, diagnostics.
//
// Compiled with -ffp-contract=off: every FP64 expression below is evaluated as written, one
// correctly rounded IEEE operation at a time (gfx950's FP64 divide and square root are correctly
// rounded), which is what makes the FP64 path bit-identical to the reference's arithmetic.
#include <cfloat>
#include <cmath>

#include <algorithm>

#include "nb_internal.hpp"

namespace nb {

typedef const __attribute__((address_space(4))) double *cdp;
typedef const __attribute__((address_space(4))) int32_t *cip;

__device__ __forceinline__ bool active_f(uint8_t f) {
  return (f & NB_F_EXISTS) && !(f & NB_F_FRAGMENTING);
}
__device__ __forceinline__ bool collide_b(int32_t b) {
  return b == NB_CB_ELASTIC || b == NB_CB_FRAGMENT;
}

// ---------------------------------------------------------------------------------------------
// FP64 force in the reference's operation order, sources added in index order.
//   eps == 0 && cutoff: calcForceFrom (body.go:214-225)
//       dist = sqrt(dx*dx+dy*dy+dz*dz); if dist > Ri+Rj: force = G*mi*mj/(dist*dist);
//       fx += force*dx/dist
//   otherwise: directForce (octree.go:314-325) with optional gate on the unsoftened distance
//       distSq = d2 + eps*eps; dist = sqrt(distSq); force = G*mi*mj/distSq; fx += force*dx/dist
// Pairs are emitted from the lower index (Collided, body.go:192-208).
// ---------------------------------------------------------------------------------------------
// Three quotients by one divisor, bit-identical to three divisions.  A correctly rounded FP64
// division n / d is v_div_scale of both operands, v_rcp, two Newton steps, the quotient, its
// residual, v_div_fmas and v_div_fixup; with d in [2^-400, 2^400] and |n| in [2^-400, 2^300] the
// scalings and the fix-up are identities, so the steps that depend on d alone are done once.  Zero
// numerators (a body on a coordinate plane of the other) take the division, like everything else
// outside that range.
// need: lanes whose quotients are used (the others may hold anything).
__device__ __forceinline__ void three_quotients(const double n[3], double d, bool need,
                                                double q[3]) {
  double y = __builtin_amdgcn_rcp(d);
  y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
  int ok = (int)(d >= 0x1p-400) & (int)(d <= 0x1p400);
#pragma unroll
  for (int c = 0; c < 3; c++) ok &= (int)(fabs(n[c]) >= 0x1p-400) & (int)(fabs(n[c]) <= 0x1p300);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const double v = n[c] * y;
    q[c] = __builtin_fma(__builtin_fma(-d, v, n[c]), y, v);
  }
  if (__builtin_amdgcn_ballot_w64(need && !ok)) {
    __asm__ volatile("");  // a real branch: these divisions are rare
    if (!ok) {
#pragma unroll
      for (int c = 0; c < 3; c++) q[c] = n[c] / d;
    }
  }
}

// A target's terms are computed by many lanes and added by one, in index order.
// A workgroup owns TL targets.  Its 13 term waves take the next 13 * 64 / TL sources of a round
// (lane = target + TL * source; UN passes per round), and write the three components of each term
// to LDS; a skipped pair (self, inactive, behind the gate) writes +0.0, which leaves the sum's
// bits alone: a sum that starts at +0.0 is never -0.0.  Meanwhile its 3 sum waves, one per
// component, add the previous round's terms in index order.  The buffers alternate, so there is
// one barrier per round.
// One lane per target (sources staged in LDS) left most of the chip idle below 65,536 bodies, each
// lane in a serial chain of square roots and divisions: 0.413 ms at n = 1,000, 6.69 at 16,384,
// 26.6 at 65,536, 283 at 262,144.  This form, same bits: 0.018, 1.22, 17.1 and 263 ms.  What bounds
// it now is FP64 issue (about 110 VALU instructions a pair), and for small n the serial additions.
constexpr int kF64Term = 13, kF64Sum = 3;
template <int TL, int UN>
__global__ __launch_bounds__(64 * (kF64Term + kF64Sum)) __attribute__((amdgpu_waves_per_eu(8)))
void k_force_f64(Force64Args a) {
  constexpr int SL = 64 / TL;            // sources per wave
  constexpr int C = kF64Term * SL;       // sources per pass of the term waves
  __shared__ double terms[2][3][C * UN][TL];
  __shared__ PairBuf<192> found;  // (two workgroups' LDS just fits a CU with TL = 64)
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = blockIdx.x * TL + (lane & (TL - 1));
  const int rounds = (a.n + C * UN - 1) / (C * UN);
  if (threadIdx.x == 0) found.clear();
  __syncthreads();
  if (wave >= kF64Term) {  // a component's sums
    const int c = wave - kF64Term;
    double f = 0;
    for (int r = 0; r <= rounds; r++) {
      if (r > 0 && lane < TL) {
        const double *t = &terms[(r - 1) & 1][c][0][lane];
#pragma unroll 13
        for (int e = 0; e < C * UN; e++) f += t[e * TL];
      }
      __syncthreads();
    }
    if (lane < TL && i < a.npad) a.acc[(size_t)c * a.npad + i] = f;
  } else {
    const bool ai = i < a.n && active_f(a.flags[i]);
    const double xi = ai ? a.x[i] : 0, yi = ai ? a.y[i] : 0, zi = ai ? a.z[i] : 0;
    const double mi = ai ? a.m[i] : 0, ri = ai ? a.r[i] : 0;
    const int32_t bi = ai ? a.beh[i] : NB_CB_NONE;
    const bool ci = ai && a.collisions && nb_may_pair(bi, a.events);
    const double Gm = a.G * mi, eps2 = a.eps * a.eps;
    const bool ref = a.eps == 0.0 && a.cutoff;
    const bool need_d0 = ref || a.cutoff || a.collisions;
    // a source's words are requested one pass ahead, so no term waits for memory
    double sx, sy, sz, sm, sr;
    int sf;
    const int j0 = wave * SL + lane / TL;
    auto fetch = [&](int j) {
      const int q = min(j, a.n - 1);
      sx = a.x[q];
      sy = a.y[q];
      sz = a.z[q];
      sm = a.m[q];
      sr = a.r[q];
      sf = a.flags[q];
    };
    fetch(j0);
    for (int r = 0; r <= rounds; r++) {
      if (r < rounds) {
#pragma unroll
        for (int u = 0; u < UN; u++) {
          const int j = (r * UN + u) * C + j0;
          const double dx = sx - xi, dy = sy - yi, dz = sz - zi, mj = sm, rj = sr;
          const bool valid = j < a.n && j != i && ai && active_f((uint8_t)sf);
          fetch(j + C);
          const double d2 = dx * dx + dy * dy + dz * dz;
          const double rs = ri + rj;
          const double dist0 = need_d0 ? __builtin_sqrt(d2) : 0.0;
          const bool overlap = need_d0 && !(dist0 > rs);
          // eps == 0 with the gate divides by the rounded distance's square (body.go:221),
          // otherwise by the squared distance itself (octree.go:317-319)
          const double distSq = ref ? dist0 * dist0 : d2 + eps2;
          const double dist = ref ? dist0 : __builtin_sqrt(distSq);
          const double force = Gm * mj / distSq;
          const double n[3] = {force * dx, force * dy, force * dz};
          double q[3];
          three_quotients(n, dist, valid, q);
          const bool adds = valid && !(a.cutoff && overlap);
          const int e = u * C + j0;
#pragma unroll
          for (int c = 0; c < 3; c++) terms[r & 1][c][e][lane & (TL - 1)] = adds ? q[c] : 0.0;
          if (valid && overlap && i < j && ci &&
              nb_pair_event(bi, a.beh[j], ri, rj, dist0, a.events))
            found.add(a.pairs, a.ctr, a.pair_cap, i, j);
        }
      }
      __syncthreads();
    }
  }
  found.flush(a.pairs, a.ctr, a.pair_cap);
}

hipError_t launch_force_f64(const Force64Args &a, hipStream_t st) {
  // Targets per workgroup: the busiest of the 256 CUs takes k = ceil(n / (256 TL)) workgroups, and
  // the time measured from n = 200 to 40,000 is n (a + b k): a one round's latency, b the work of
  // TL targets, in units of 0.1 us per 1,000 sources.  Small TL spreads few targets over the chip,
  // large TL reads each source for more of them.
  const struct { int tl, a, b; } cost[] = {{64, 207, 559}, {32, 110, 336}, {16, 65, 169},
                                           {8, 43, 103}, {4, 75, 69}};
  int tl = 64;
  int64_t best = INT64_MAX;
  for (const auto &q : cost) {
    const int64_t k = ((int64_t)a.n + 256 * q.tl - 1) / (256 * q.tl), v = q.a + q.b * k;
    if (v < best) best = v, tl = q.tl;
  }
  const dim3 grid((unsigned)(a.npad / tl)), block(64 * (kF64Term + kF64Sum));
  switch (tl) {
    case 64: hipLaunchKernelGGL((k_force_f64<64, 2>), grid, block, 0, st, a); break;
    case 32: hipLaunchKernelGGL((k_force_f64<32, 1>), grid, block, 0, st, a); break;
    case 16: hipLaunchKernelGGL((k_force_f64<16, 1>), grid, block, 0, st, a); break;
    case 8: hipLaunchKernelGGL((k_force_f64<8, 1>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((k_force_f64<4, 1>), grid, block, 0, st, a); break;
  }
  return hipGetLastError();
}

// FP64 accelerations for a sample of targets (error reference for the FP32 path).
__global__ __launch_bounds__(256) void k_accel_f64(Accel64Args a) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= a.nidx) return;
  const int64_t i = a.idx[k];
  double ax = 0, ay = 0, az = 0;
  if (i >= 0 && i < a.n && active_f(a.flags[i])) {
    const double xi = a.x[i], yi = a.y[i], zi = a.z[i], ri = a.r[i];
    const double eps2 = a.eps * a.eps;
    for (int j = 0; j < a.n; j++) {
      if (j == i || !active_f(a.flags[j])) continue;
      const double dx = a.x[j] - xi, dy = a.y[j] - yi, dz = a.z[j] - zi;
      const double d2 = dx * dx + dy * dy + dz * dz;
      if (a.cutoff && !(__builtin_sqrt(d2) > ri + a.r[j])) continue;
      const double ds = d2 + eps2;
      const double w = a.G * a.m[j] / (ds * __builtin_sqrt(ds));
      ax += w * dx;
      ay += w * dy;
      az += w * dz;
    }
  }
  a.out[k] = ax;
  a.out[a.nidx + k] = ay;
  a.out[2 * a.nidx + k] = az;
}

hipError_t launch_accel_f64(const Accel64Args &a, hipStream_t st) {
  if (a.nidx <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_accel_f64, dim3((unsigned)((a.nidx + 255) / 256)), dim3(256), 0, st, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Elastic collision resolution (ProcessMods, body_collection.go:212-233), one thread walking the
// sorted pair list: each unordered pair is resolved once, as lo.ResolveCollision(hi) when lo is
// Elastic, else hi.ResolveCollision(lo) (only an Elastic first body resolves, body.go:252-253).
// ---------------------------------------------------------------------------------------------
struct Elastic {
  double v1[3], v2[3], cm[3];
};

// calcElasticCollision, cmd/body/collisioncalc.go:42-186 (coll3d), in two parts: what depends on
// the two positions and radii alone, which a pass evaluates for all its pairs at once, and the
// rest.  The operations and their order are the reference's.
struct ElasticGeom {
  double d, r12, st, ct, sp, cp;
};

__device__ static ElasticGeom elastic_geom(const ResolveArgs &a, int b, int o) {
  const double r1 = a.r[b], r2 = a.r[o];
  const double x1 = a.x[b], y1 = a.y[b], z1 = a.z[b];
  const double x21 = a.x[o] - x1, y21 = a.y[o] - y1, z21 = a.z[o] - z1;
  ElasticGeom g;
  g.r12 = r1 + r2;
  g.d = sqrt(x21 * x21 + y21 * y21 + z21 * z21);
  const double theta2 = acos(z21 / g.d);
  double phi2;
  if (x21 == 0 && y21 == 0)
    phi2 = 0;
  else
    phi2 = atan2(y21, x21);
  g.st = sin(theta2);
  g.ct = cos(theta2);
  g.sp = sin(phi2);
  g.cp = cos(phi2);
  return g;
}

__device__ static bool elastic(const ResolveArgs &a, int b, int o, const ElasticGeom &g,
                               Elastic &res) {
  double m21, v, st, ct, sp, cp, vx1r, vy1r, vz1r, fvz1r, thetav, phiv, dr, alpha, beta, sbeta,
      cbeta, aa, dvz2, vx2r, vy2r, vz2r, vx21, vy21, vz21, vx_cm, vy_cm, vz_cm;
  const double m1 = a.m[b], m2 = a.m[o];
  double vx1 = a.vx[b], vy1 = a.vy[b], vz1 = a.vz[b];
  const double vx2 = a.vx[o], vy2 = a.vy[o], vz2 = a.vz[o];

  m21 = m2 / m1;
  vx21 = vx2 - vx1;
  vy21 = vy2 - vy1;
  vz21 = vz2 - vz1;

  vx_cm = (m1 * vx1 + m2 * vx2) / (m1 + m2);
  vy_cm = (m1 * vy1 + m2 * vy2) / (m1 + m2);
  vz_cm = (m1 * vz1 + m2 * vz2) / (m1 + m2);

  v = sqrt(vx21 * vx21 + vy21 * vy21 + vz21 * vz21);
  if (v == 0) return false;

  vx1 = -vx21;
  vy1 = -vy21;
  vz1 = -vz21;

  st = g.st;
  ct = g.ct;
  sp = g.sp;
  cp = g.cp;

  vx1r = ct * cp * vx1 + ct * sp * vy1 - st * vz1;
  vy1r = cp * vy1 - sp * vx1;
  vz1r = st * cp * vx1 + st * sp * vy1 + ct * vz1;
  fvz1r = vz1r / v;
  if (fvz1r > 1)
    fvz1r = 1;
  else if (fvz1r < -1)
    fvz1r = -1;
  // separating (thetav > pi / 2 below) is settled before any angle: acos(x) is pi / 2 - x near 0,
  // so at -1e-14 it exceeds M_PI / 2 by 45 of its ulps
  if (fvz1r < -1e-14) return false;
  thetav = acos(fvz1r);
  if (vx1r == 0 && vy1r == 0)
    phiv = 0;
  else
    phiv = atan2(vy1r, vx1r);

  dr = g.d * sin(thetav) / g.r12;
  if (thetav > M_PI / 2 || fabs(dr) > 1) return false;

  alpha = asin(-dr);
  beta = phiv;
  sbeta = sin(beta);
  cbeta = cos(beta);

  aa = tan(thetav + alpha);
  dvz2 = 2 * (vz1r + aa * (cbeta * vx1r + sbeta * vy1r)) / ((1 + aa * aa) * (1 + m21));

  vz2r = dvz2;
  vx2r = aa * cbeta * dvz2;
  vy2r = aa * sbeta * dvz2;
  vz1r = vz1r - m21 * vz2r;
  vx1r = vx1r - m21 * vx2r;
  vy1r = vy1r - m21 * vy2r;

  res.v1[0] = ct * cp * vx1r - sp * vy1r + st * cp * vz1r + vx2;
  res.v1[1] = ct * sp * vx1r + cp * vy1r + st * sp * vz1r + vy2;
  res.v1[2] = ct * vz1r - st * vx1r + vz2;
  res.v2[0] = ct * cp * vx2r - sp * vy2r + st * cp * vz2r + vx2;
  res.v2[1] = ct * sp * vx2r + cp * vy2r + st * sp * vz2r + vy2;
  res.v2[2] = ct * vz2r - st * vx2r + vz2;
  res.cm[0] = vx_cm;
  res.cm[1] = vy_cm;
  res.cm[2] = vz_cm;
  return true;
}

// shouldFragment (fragcalc.go:24-49); the factors go to doFragment.
__device__ static bool should_fragment(const ResolveArgs &a, int b, int o, const Elastic &e,
                                       double *tf, double *of) {
  if (!(a.beh[b] == NB_CB_FRAGMENT || a.beh[o] == NB_CB_FRAGMENT)) return false;
  const double br = a.rest[b];
  const double vThis = a.vx[b] + a.vy[b] + a.vz[b];
  const double dvThis = fabs(a.vx[b] - ((e.v1[0] - e.cm[0]) * br + e.cm[0])) +
                        fabs(a.vy[b] - ((e.v1[1] - e.cm[1]) * br + e.cm[1])) +
                        fabs(a.vz[b] - ((e.v1[2] - e.cm[2]) * br + e.cm[2]));
  const double thisFactor = dvThis / fabs(vThis);
  const double vOther = a.vx[o] + a.vy[o] + a.vz[o];
  const double dvOther = fabs(a.vx[o] - ((e.v2[0] - e.cm[0]) * br + e.cm[0])) +
                         fabs(a.vy[o] - ((e.v2[1] - e.cm[1]) * br + e.cm[1])) +
                         fabs(a.vz[o] - ((e.v2[2] - e.cm[2]) * br + e.cm[2]));
  const double otherFactor = dvOther / fabs(vOther);
  const double fb = a.frag[b], fo = a.frag[o];
  *tf = thisFactor;
  *of = otherFactor;
  return (a.beh[b] == NB_CB_FRAGMENT && thisFactor > fb) ||
         (a.beh[o] == NB_CB_FRAGMENT && otherFactor > fo);
}

// initiateFragmentation (fragcalc.go:65-83): fragDelta, the fragment count Min(delta * FragStep,
// 2000), and fragInfo.  The body keeps this cycle's force while it fragments.
__device__ static void initiate_fragmentation(const ResolveArgs &a, int b, double factor,
                                              uint64_t *started, uint64_t *inactive) {
  const double fragDelta = a.frag[b] > 10 ? 10.0 : factor - a.frag[b];
  const double prod = fragDelta * a.fstep[b];
  const double fragments = isnan(prod) ? prod : (prod < 2000.0 ? prod : 2000.0);  // math.Min
  if (fragments <= 1) {
    a.beh[b] = NB_CB_FRAGMENT;
    return;
  }
  const uint8_t f = a.flags[b];
  if (!(f & NB_F_FRAGMENTING)) {
    (*started)++;
    if (f & NB_F_EXISTS) (*inactive)++;
  }
  a.flags[b] = (uint8_t)(f | NB_F_FRAGMENTING);
  FragState st;
  double fx = 0, fy = 0, fz = 0;
  for (int sl = 0; sl < a.split; sl++) {
    const double *o = a.acc + (size_t)sl * 3 * a.npad;
    fx += o[b];
    fy += o[a.npad + b];
    fz += o[2 * a.npad + b];
  }
  st.fx = fx;
  st.fy = fy;
  st.fz = fz;
  st.mass = a.m[b] / fragments;
  st.radius = a.r[b];
  st.px = a.x[b];
  st.py = a.y[b];
  st.pz = a.z[b];
  // int(fragments): truncation; NaN converts to the most negative int64 on amd64
  st.left = isnan(fragments) ? INT64_MIN : (int64_t)fragments;
  st.made = 0;
  st.id = (int64_t)(a.ctr->frag_seq++);
  a.fst[b] = st;
}

// Tallies of one resolution pass.
struct ResolveTally {
  uint64_t resolved = 0, fragreq = 0, subsumed = 0, started = 0, inactive = 0;
};

// Whether the pair (lo, hi) can change anything when events are off: an Elastic first body
// (body.go:252-253) and both bodies existing (:249-251).  With events off nothing in the pass
// changes behaviours or flags, so this is decided once per pass.  b receives the first body.
__device__ static bool elastic_pair(const ResolveArgs &a, int lo, int hi, int *b, int *o) {
  if (a.beh[lo] == NB_CB_ELASTIC && collide_b(a.beh[hi])) {
    *b = lo;
    *o = hi;
  } else if (a.beh[hi] == NB_CB_ELASTIC && collide_b(a.beh[lo])) {
    *b = hi;
    *o = lo;
  } else {
    return false;
  }
  return (a.flags[*b] & NB_F_EXISTS) && (a.flags[*o] & NB_F_EXISTS);
}

// A pair that can act, b resolving (ResolveCollision, body.go:248-264).
__device__ static void resolve_elastic(const ResolveArgs &a, int b, int o, const ElasticGeom &g,
                                       ResolveTally &t) {
  Elastic e;
  if (!elastic(a, b, o, g, e)) return;
  t.resolved++;
  double tf = 0, of = 0;
  if (should_fragment(a, b, o, e, &tf, &of)) {
    t.fragreq++;
    if (a.events) {  // doFragment (fragcalc.go:54-63)
      if (a.beh[b] == NB_CB_FRAGMENT && tf > a.frag[b])
        initiate_fragmentation(a, b, tf, &t.started, &t.inactive);
      if (a.beh[o] == NB_CB_FRAGMENT && of > a.frag[o])
        initiate_fragmentation(a, o, of, &t.started, &t.inactive);
    }
    return;
  }
  // doElastic (collisioncalc.go:26-35): restitution of the first body.
  const double rr = a.rest[b];
  a.vx[b] = (e.v1[0] - e.cm[0]) * rr + e.cm[0];
  a.vy[b] = (e.v1[1] - e.cm[1]) * rr + e.cm[1];
  a.vz[b] = (e.v1[2] - e.cm[2]) * rr + e.cm[2];
  a.vx[o] = (e.v2[0] - e.cm[0]) * rr + e.cm[0];
  a.vy[o] = (e.v2[1] - e.cm[1]) * rr + e.cm[1];
  a.vz[o] = (e.v2[2] - e.cm[2]) * rr + e.cm[2];
  a.collided[b] = 1;
  a.collided[o] = 1;
}

// One canonical pair, as ProcessMods handles its event (body_collection.go:212-233).
__device__ static void resolve_pair(const ResolveArgs &a, int lo, int hi, ResolveTally &t) {
  if (a.events && !(collide_b(a.beh[lo]) && collide_b(a.beh[hi]))) {
    // a subsume pair: ResolveSubsume (body.go:228-244) by the larger body, no existence check
    const int b = a.r[lo] > a.r[hi] ? lo : hi, o = b == lo ? hi : lo;
    a.m[b] = a.m[b] + a.m[o];
    const uint8_t fo = a.flags[o];
    if ((fo & NB_F_EXISTS) && !(fo & NB_F_FRAGMENTING)) t.inactive++;
    a.flags[o] = (uint8_t)(fo & ~NB_F_EXISTS);  // SetNotExists (body.go:93-96)
    a.m[o] = 0.0;
    t.subsumed++;
    return;
  }
  int b, o;
  if (!elastic_pair(a, lo, hi, &b, &o)) return;
  resolve_elastic(a, b, o, elastic_geom(a, b, o), t);
}

__device__ static void add_tally(DevCounters *ctr, uint32_t found, const ResolveTally &t) {
  ctr->pairs_total += found;
  ctr->pairs_last = found;
  ctr->resolved_total += t.resolved;
  ctr->fragment_requests += t.fragreq;
  ctr->subsumed_total += t.subsumed;
  ctr->frag_started += t.started;
  ctr->inactive_events += t.inactive;
}

// The pass one pair at a time, in canonical order, on one lane: the ordering reference, and the
// pass used with events on (subsumes and fragmentation ids depend on the order across pairs).
__global__ __launch_bounds__(64) void k_resolve(ResolveArgs a) {
  if (threadIdx.x != 0) return;
  const uint32_t found = a.ctr->pair_count;
  const int64_t cnt = min((int64_t)found, a.pair_cap);
  ResolveTally t;
  for (int64_t k = 0; k < cnt; k++) {
    const uint64_t key = a.pairs[k];
    resolve_pair(a, (int)(key >> 32), (int)(key & 0xffffffffu), t);
  }
  add_tally(a.ctr, found, t);
}

// ---------------------------------------------------------------------------------------------
// The pair list in canonical order, and the pairs' chains.
//
// The force phase leaves the pairs (lo << 32 | hi) in any order.  They are counted per body, twice:
// as lo's (a body's own pairs) and as hi's (the pairs that reach it); prefix sums of the two counts
// place each pair in its body's two lists, and its rank among the list's partners gives its place
// in order.  Own lists one after another, partners ascending, are the canonical order.  A list is
// as long as its body's pairs, so ranking costs a few reads per pair; nothing depends on the list's
// capacity, only on the bodies and the pairs there are.  Where a list may be long (a body that
// overlaps thousands, a scene where all overlap) that would be its length squared: lists of more than
// kPairLong pairs are then put in order by a bit per body, and a pair finds its rank by bisection.
//
// With events off, pairs that share no body resolve together.  A pair reads and writes only its two
// bodies, and nothing in the pass changes which pairs act, so the state is bit-identical to the
// one-by-one pass as long as every pair sees both its bodies exactly as the pairs before it in
// canonical order left them.  The pairs touching one body form a chain in canonical order: the
// pairs (x, b) that reach it, x ascending, then its own pairs (b, y), y ascending.  A pair waits for
// at most two predecessors (the previous pair on each of its bodies) and releases at most two
// successors.  One workgroup resolves the ready pairs round by round.
//
// Up to kPairSmallN bodies one workgroup does all of it in one launch, the counts in LDS; above, or
// when the last count read is more than kPairSmallPairs (or a scene's first is still to come), the
// list takes five launches, the chains and the rounds one each (one workgroup / seven launches, reference scene: 0.020 / 0.033 ms with 63
// pairs, 0.045 / 0.057 with 1,074, 0.072 / 0.074 with 2,439, 0.184 / 0.114 with 6,998).
// A sort of the keys, one of the swapped keys and binary searches took 11 to 23 launches.
//
// A round costs one coll3d of latency (FP64 transcendentals): the half of it that depends on
// positions alone is evaluated beforehand for all pairs, and 512 threads leave it the registers it
// needs.  List and rounds together, before and now: 0.103 -> 0.019 ms at n = 1,000 (63 pairs, 3
// rounds), 0.63 -> 0.11 at 10,007 (6,998 pairs, 16 rounds), 1.30 -> 0.24 at 16,384 (18,696 pairs,
// 40 rounds).
// ---------------------------------------------------------------------------------------------
constexpr int kPairThreads = 512;         // coll3d keeps its 140 VGPRs (1,024 threads would spill)
constexpr int kPairLdsPend = 128 * 1024;  // pairs whose predecessor counts fit in LDS, one byte each

__device__ __forceinline__ int64_t pair_total(const PairArgs &a) {
  return min((int64_t)a.ctr->pair_count, a.cap);
}

// The next place in body i's list.  In memory, the lanes that share the first one's body take theirs
// with one atomic (2 million pairs among 2,000 bodies: 0.63 ms with one each, 0.32 so); in LDS, where
// the pairs are few, that costs more than it saves.
template <bool LDS, class P>
__device__ __forceinline__ int next_place(P counts, int i) {
  if (LDS) return atomicAdd(&counts[i], 1);
  const bool same = i == __builtin_amdgcn_readfirstlane(i);
  const uint64_t peers = __builtin_amdgcn_ballot_w64(same);
  const int rank = (int)__builtin_amdgcn_mbcnt_hi(
      (uint32_t)(peers >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)peers, 0));
  int at = 0;
  if (!same || rank == 0) at = atomicAdd(&counts[i], same ? __builtin_popcountll(peers) : 1);
  const int base = __builtin_amdgcn_readlane(at, __builtin_ctzll(peers));
  return same ? base + rank : at;
}

// A pair's place in its two bodies' lists, in arrival order.
template <bool LDS, class P>
__device__ __forceinline__ void pair_count(const PairArgs &a, int64_t cnt, P own, P reach,
                                           int64_t k0, int64_t step) {
  for (int64_t k = k0; k < cnt; k += step) {
    const uint64_t key = a.raw[k];
    a.slot_own[k] = next_place<LDS>(own, (int)(key >> 32));
    a.slot_reach[k] = next_place<LDS>(reach, (int)(key & 0xffffffffu));
  }
}

template <class P>
__device__ __forceinline__ void pair_fill(const PairArgs &a, int64_t cnt, P own, P reach,
                                          int64_t k0, int64_t step) {
  for (int64_t k = k0; k < cnt; k += step) {
    const uint64_t key = a.raw[k];
    const int lo = (int)(key >> 32), hi = (int)(key & 0xffffffffu);
    a.list_own[own[lo] + a.slot_own[k]] = hi;
    a.list_reach[reach[hi] + a.slot_reach[k]] = lo;
  }
}

// How many of list[u0 .. u1) are below v.
__device__ __forceinline__ int list_below(const int32_t *list, int u0, int u1, int v) {
  int n = 0, e = u0;
  for (; e + 8 <= u1; e += 8) {  // eight loads in flight
    int w[8];
#pragma unroll
    for (int q = 0; q < 8; q++) w[q] = list[e + q];
#pragma unroll
    for (int q = 0; q < 8; q++) n += w[q] < v ? 1 : 0;
  }
  for (; e < u1; e++) n += list[e] < v ? 1 : 0;
  return n;
}
__device__ __forceinline__ int sorted_below(const int32_t *list, int u0, int u1, int v) {
  int lo = u0, hi = u1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (list[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  return lo - u0;
}

// Ranks: the pair's canonical index, and the index by place in hi's list.  SORTED: k_pair_long has
// left the long lists in order where the slots were.
template <bool SORTED, class P>
__device__ __forceinline__ void pair_rank(const PairArgs &a, int64_t cnt, P own, P reach,
                                          int64_t k0, int64_t step) {
  for (int64_t k = k0; k < cnt; k += step) {
    const uint64_t key = a.raw[k];
    const int lo = (int)(key >> 32), hi = (int)(key & 0xffffffffu);
    const int u0 = own[lo], u1 = own[lo + 1], l0 = reach[hi], l1 = reach[hi + 1];
    const int p = u0 + (SORTED && u1 - u0 > kPairLong ? sorted_below(a.slot_own, u0, u1, hi)
                                                      : list_below(a.list_own, u0, u1, hi));
    const int q = l0 + (SORTED && l1 - l0 > kPairLong ? sorted_below(a.slot_reach, l0, l1, lo)
                                                      : list_below(a.list_reach, l0, l1, lo));
    a.keys[p] = key;
    a.by_hi[q] = p;
    a.place[p] = q;
  }
}

// Chains, roles and positions' half of coll3d of the sorted pairs.
template <class P>
__device__ __forceinline__ void pair_link(const PairArgs &a, const ResolveArgs &r, int64_t cnt,
                                          P own, P reach, int64_t k0, int64_t step) {
  for (int64_t k = k0; k < cnt; k += step) {
    const uint64_t key = a.keys[k];
    const int lo = (int)(key >> 32), hi = (int)(key & 0xffffffffu);
    const int q = a.place[k];
    // lo's chain: its own pairs in order, after the pairs that reach it
    int pend = (int)k > own[lo] || reach[lo + 1] > reach[lo] ? 1 : 0;
    int2 succ;
    succ.x = (int)k + 1 < own[lo + 1] ? (int)k + 1 : -1;
    // hi's chain: the pairs that reach it in order, then its own
    pend += q > reach[hi] ? 1 : 0;
    succ.y = q + 1 < reach[hi + 1] ? a.by_hi[q + 1] : own[hi] < own[hi + 1] ? own[hi] : -1;
    a.succ[k] = succ;
    a.pend[k] = pend;
    int b, o;
    const bool acts = elastic_pair(r, lo, hi, &b, &o);
    a.role[k] = acts ? make_int2(b, o) : make_int2(-1, -1);
    if (acts && k < a.geom_cap) {
      const ElasticGeom g = elastic_geom(r, b, o);
      double *w = a.geom + k * 6;
      w[0] = g.d;
      w[1] = g.r12;
      w[2] = g.st;
      w[3] = g.ct;
      w[4] = g.sp;
      w[5] = g.cp;
    }
  }
}

// The rounds, by one workgroup.  pend8: kPairLdsPend bytes of LDS (predecessor counts).
__device__ static void pair_rounds(const PairArgs &a, const ResolveArgs &r, int cnt,
                                   uint32_t *pend8, int *s_len, unsigned long long *s_tally) {
  const int tid = threadIdx.x, nt = blockDim.x;
  const bool lds = cnt <= kPairLdsPend;
  if (tid == 0) *s_len = 0, s_tally[0] = s_tally[1] = 0;
  __syncthreads();
  int32_t *cur = a.list_own, *nxt = a.list_reach;  // (the lists have done their work)
  for (int w = tid; w * 4 < cnt; w += nt) {
    uint32_t v = 0;
    for (int e = 0; e < 4 && w * 4 + e < cnt; e++) {
      const int p = a.pend[w * 4 + e];
      v |= (uint32_t)p << (8 * e);
      if (p == 0) cur[atomicAdd(s_len, 1)] = w * 4 + e;
    }
    if (lds) pend8[w] = v;
  }
  __syncthreads();
  int m = *s_len;
  ResolveTally t;
  while (m > 0) {
    __syncthreads();  // every thread has read s_len
    if (tid == 0) *s_len = 0;
    __syncthreads();
    for (int q = tid; q < m; q += nt) {
      const int k = cur[q];
      const int2 role = a.role[k], succ = a.succ[k];
      if (role.x >= 0) {
        ElasticGeom g;
        if (k < a.geom_cap) {
          const double *w = a.geom + (int64_t)k * 6;
          g.d = w[0];
          g.r12 = w[1];
          g.st = w[2];
          g.ct = w[3];
          g.sp = w[4];
          g.cp = w[5];
        } else {
          g = elastic_geom(r, role.x, role.y);
        }
        resolve_elastic(r, role.x, role.y, g, t);
      }
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int sk = e ? succ.y : succ.x;
        if (sk < 0) continue;
        bool ready;
        if (lds) {
          const int sh = 8 * (sk & 3);
          ready = (atomicSub(&pend8[sk >> 2], 1u << sh) >> sh & 255u) == 1u;
        } else {
          ready = atomicSub(&a.pend[sk], 1) == 1;
        }
        if (ready) nxt[atomicAdd(s_len, 1)] = sk;
      }
    }
    __syncthreads();  // the workgroup's writes are seen by its next reads
    m = *s_len;
    int32_t *sw = cur;
    cur = nxt;
    nxt = sw;
  }
  atomicAdd(&s_tally[0], (unsigned long long)t.resolved);
  atomicAdd(&s_tally[1], (unsigned long long)t.fragreq);
  __syncthreads();
  if (tid == 0) {
    ResolveTally all;
    all.resolved = s_tally[0];
    all.fragreq = s_tally[1];
    add_tally(a.ctr, a.ctr->pair_count, all);
  }
}

// Exclusive prefix sums of each thread's pair of values over the workgroup; total gets the sums.
__device__ static int2 block_scan2(int2 v, int2 *waves, int2 *total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int2 s = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int x = __shfl_up(s.x, d, 64), y = __shfl_up(s.y, d, 64);
    if (lane >= d) s.x += x, s.y += y;
  }
  if (lane == 63) waves[w] = s;
  __syncthreads();
  int2 base = make_int2(0, 0), all = make_int2(0, 0);
  for (int q = 0; q < nw; q++) {
    const int2 u = waves[q];
    if (q < w) base.x += u.x, base.y += u.y;
    all.x += u.x;
    all.y += u.y;
  }
  __syncthreads();
  *total = all;
  return make_int2(base.x + s.x - v.x, base.y + s.y - v.y);
}

// One workgroup, one launch: list (mode 0), or list and rounds (mode 1).
__global__ __launch_bounds__(kPairThreads) void k_pairs_small(PairArgs a, ResolveArgs r, int mode) {
  __shared__ int counts[2 * (kPairSmallN + 1)];
  __shared__ int2 waves[16];
  __shared__ int s_len;
  __shared__ unsigned long long s_tally[2];
  static_assert(kPairLdsPend <= sizeof(counts), "the predecessor counts reuse the count arrays");
  int *own = counts, *reach = counts + kPairSmallN + 1;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int cnt = (int)pair_total(a);
  if (cnt == 0) {
    if (mode == 1 && tid == 0) add_tally(a.ctr, 0, ResolveTally{});
    return;
  }
  for (int i = tid; i <= a.n; i += nt) own[i] = reach[i] = 0;
  __syncthreads();
  pair_count<true>(a, cnt, own, reach, tid, nt);
  __syncthreads();
  const int per = (a.n + nt - 1) / nt, i0 = min(tid * per, a.n), i1 = min(i0 + per, a.n);
  int2 v = make_int2(0, 0), total;
  for (int i = i0; i < i1; i++) v.x += own[i], v.y += reach[i];
  int2 at = block_scan2(v, waves, &total);
  for (int i = i0; i < i1; i++) {
    const int x = own[i], y = reach[i];
    own[i] = at.x;
    reach[i] = at.y;
    at.x += x;
    at.y += y;
  }
  if (tid == 0) own[a.n] = total.x, reach[a.n] = total.y;
  __syncthreads();
  pair_fill(a, cnt, own, reach, tid, nt);
  __syncthreads();
  pair_rank<false>(a, cnt, own, reach, tid, nt);
  if (mode == 0) return;
  __syncthreads();
  pair_link(a, r, cnt, own, reach, tid, nt);
  __syncthreads();
  pair_rounds(a, r, cnt, reinterpret_cast<uint32_t *>(counts), &s_len, s_tally);
}

// The same over the whole chip.  The counts are zero between uses.
__global__ __launch_bounds__(256) void k_pair_count(PairArgs a) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.nlong = 0;
  pair_count<false>(a, pair_total(a), a.own, a.reach, (int64_t)blockIdx.x * 256 + threadIdx.x,
             (int64_t)gridDim.x * 256);
}

constexpr int kPairScan = 4096;  // bodies per workgroup of the prefix sums, four per thread
__global__ __launch_bounds__(1024) void k_pair_sums(PairArgs a) {
  __shared__ int2 waves[16];
  if (pair_total(a) == 0) return;
  const int i0 = blockIdx.x * kPairScan + (int)threadIdx.x * 4;
  int2 v = make_int2(0, 0), total;
  for (int e = 0; e < 4; e++)
    if (i0 + e < a.n) v.x += a.own[i0 + e], v.y += a.reach[i0 + e];
  block_scan2(v, waves, &total);
  if (threadIdx.x == 0) a.bsum[blockIdx.x] = total;
}

__global__ __launch_bounds__(1024) void k_pair_offsets(PairArgs a) {
  __shared__ int2 waves[16];
  if (pair_total(a) == 0) return;
  int2 before = make_int2(0, 0), base, total;
  for (int q = threadIdx.x; q < (int)blockIdx.x; q += 1024)
    before.x += a.bsum[q].x, before.y += a.bsum[q].y;
  block_scan2(before, waves, &base);  // the sums of the workgroups before this one
  const int i0 = blockIdx.x * kPairScan + (int)threadIdx.x * 4;
  int2 c[4], v = make_int2(0, 0);
  for (int e = 0; e < 4; e++) {
    c[e] = i0 + e < a.n ? make_int2(a.own[i0 + e], a.reach[i0 + e]) : make_int2(0, 0);
    v.x += c[e].x;
    v.y += c[e].y;
  }
  int2 at = block_scan2(v, waves, &total);
  at.x += base.x;
  at.y += base.y;
  for (int e = 0; e < 4; e++) {
    if (i0 + e < a.n) {
      a.own[i0 + e] = a.reach[i0 + e] = 0;  // as the next use expects them
      a.own_off[i0 + e] = at.x;
      a.reach_off[i0 + e] = at.y;
      if (c[e].x > kPairLong) a.longs[atomicAdd(a.nlong, 1u)] = (uint32_t)(i0 + e) * 2;
      if (c[e].y > kPairLong) a.longs[atomicAdd(a.nlong, 1u)] = (uint32_t)(i0 + e) * 2 + 1;
    }
    at.x += c[e].x;
    at.y += c[e].y;
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
    a.own_off[a.n] = base.x + total.x;
    a.reach_off[a.n] = base.y + total.y;
  }
}

__global__ __launch_bounds__(256) void k_pair_fill(PairArgs a) {
  pair_fill(a, pair_total(a), a.own_off, a.reach_off, (int64_t)blockIdx.x * 256 + threadIdx.x,
            (int64_t)gridDim.x * 256);
}

// The long lists in order, a workgroup each: their bodies' bits are set in LDS, a window of kLongBits
// bodies at a time, and read off in order.
constexpr int kLongBits = 1 << 20;
__global__ __launch_bounds__(kPairThreads) void k_pair_long(PairArgs a) {
  __shared__ uint32_t bits[kLongBits / 32];
  __shared__ int first[kLongBits / 256];  // bodies in blocks of 256, then those before each block
  __shared__ int2 waves[16];
  const int tid = threadIdx.x, nt = blockDim.x, nl = (int)*a.nlong;
  for (int q = blockIdx.x; q < nl; q += gridDim.x) {
    const uint32_t e = a.longs[q];
    const int body = (int)(e >> 1);
    const int32_t *list = e & 1 ? a.list_reach : a.list_own;
    int32_t *sorted = e & 1 ? a.slot_reach : a.slot_own;
    const int32_t *off = e & 1 ? a.reach_off : a.own_off;
    const int u0 = off[body], u1 = off[body + 1];
    int out = u0;
    for (int64_t w0 = 0; w0 < a.n; w0 += kLongBits) {
      const int span = (int)min((int64_t)kLongBits, a.n - w0), blocks = (span + 255) / 256;
      __syncthreads();  // the last window has been read off
      for (int i = tid; i < blocks * 8; i += nt) bits[i] = 0;
      __syncthreads();
      for (int i = u0 + tid; i < u1; i += nt) {
        const int64_t v = list[i] - w0;
        if (v >= 0 && v < span) atomicOr(&bits[v >> 5], 1u << (v & 31));
      }
      __syncthreads();
      for (int b = tid; b < blocks; b += nt) {
        int s = 0;
        for (int i = 0; i < 8; i++) s += __builtin_popcount(bits[b * 8 + i]);
        first[b] = s;
      }
      __syncthreads();
      const int per = (blocks + nt - 1) / nt, b0 = min(tid * per, blocks), b1 = min(b0 + per, blocks);
      int2 v = make_int2(0, 0), total;
      for (int b = b0; b < b1; b++) v.x += first[b];
      int at = block_scan2(v, waves, &total).x;
      for (int b = b0; b < b1; b++) {
        const int s = first[b];
        first[b] = at;
        at += s;
      }
      __syncthreads();
      for (int i = tid; i < blocks * 8; i += nt) {  // a word each
        int o = out + first[i >> 3];
        for (int p = i & ~7; p < i; p++) o += __builtin_popcount(bits[p]);
        for (uint32_t m = bits[i]; m; m &= m - 1)
          if (o < u1) sorted[o++] = (int32_t)w0 + i * 32 + __builtin_ctz(m);
      }
      out += total.x;
    }
  }
}

template <bool SORTED>
__global__ __launch_bounds__(256) void k_pair_rank(PairArgs a) {
  pair_rank<SORTED>(a, pair_total(a), a.own_off, a.reach_off,
                    (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256);
}
__global__ __launch_bounds__(256) void k_pair_link(PairArgs a, ResolveArgs r) {
  pair_link(a, r, pair_total(a), a.own_off, a.reach_off,
            (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256);
}
__global__ __launch_bounds__(kPairThreads) void k_pair_rounds(PairArgs a, ResolveArgs r) {
  __shared__ uint32_t pend8[kPairLdsPend / 4];
  __shared__ int s_len;
  __shared__ unsigned long long s_tally[2];
  const int cnt = (int)pair_total(a);
  if (cnt == 0) {
    if (threadIdx.x == 0) add_tally(a.ctr, 0, ResolveTally{});
    return;
  }
  pair_rounds(a, r, cnt, pend8, &s_len, s_tally);
}

// Pairs up to which no list is worth the launch that puts long ones in order.
constexpr int64_t kPairMany = 8192;

hipError_t launch_pairs(const PairArgs &a, const ResolveArgs *r, int64_t expect, hipStream_t st) {
  const bool together = r && !r->events && !r->serial;
  if (a.n <= kPairSmallN && expect <= kPairSmallPairs) {
    hipLaunchKernelGGL(k_pairs_small, dim3(1), dim3(kPairThreads), 0, st, a, r ? *r : ResolveArgs{},
                       together ? 1 : 0);
  } else {
    const unsigned g = (unsigned)std::min<int64_t>(1024, (a.cap + 255) / 256);
    const unsigned gs = (unsigned)((a.n + kPairScan - 1) / kPairScan);
    hipLaunchKernelGGL(k_pair_count, dim3(g), dim3(256), 0, st, a);
    hipLaunchKernelGGL(k_pair_sums, dim3(gs), dim3(1024), 0, st, a);
    hipLaunchKernelGGL(k_pair_offsets, dim3(gs), dim3(1024), 0, st, a);
    hipLaunchKernelGGL(k_pair_fill, dim3(g), dim3(256), 0, st, a);
    if (expect > kPairMany) {
      hipLaunchKernelGGL(k_pair_long, dim3(256), dim3(kPairThreads), 0, st, a);
      hipLaunchKernelGGL(k_pair_rank<true>, dim3(g), dim3(256), 0, st, a);
    } else {
      hipLaunchKernelGGL(k_pair_rank<false>, dim3(g), dim3(256), 0, st, a);
    }
    if (together) {
      hipLaunchKernelGGL(k_pair_link, dim3(g), dim3(256), 0, st, a, *r);
      hipLaunchKernelGGL(k_pair_rounds, dim3(1), dim3(kPairThreads), 0, st, a, *r);
    }
  }
  if (r && !together) hipLaunchKernelGGL(k_resolve, dim3(1), dim3(64), 0, st, *r);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Update: Body.Update (body.go:114-139) + rewrite of the FP32 source stream.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ float4 stream_entry(bool act, double x, double y, double z, double m) {
  return act ? make_float4((float)x, (float)y, (float)z, (float)m)
             : make_float4(kSentinel, kSentinel, kSentinel, 0.f);
}

__global__ __launch_bounds__(256) void k_update(UpdateArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.npad) return;
  if (i >= a.n) {
    a.js[i] = stream_entry(false, 0, 0, 0, 0);
    return;
  }
  uint8_t f = a.flags[i];
  if (!(f & NB_F_EXISTS)) {
    a.js[i] = stream_entry(false, 0, 0, 0, 0);
    return;
  }
  const double dt = a.dt;
  double vx = a.vx[i], vy = a.vy[i], vz = a.vz[i];
  if (!a.collided[i]) {
    const double mi = a.m[i];
    double fx = 0, fy = 0, fz = 0;
    if (a.fst && (f & NB_F_FRAGMENTING)) {  // the force Body.fx kept from its last Compute
      fx = a.fst[i].fx;
      fy = a.fst[i].fy;
      fz = a.fst[i].fz;
    } else {
      for (int s = 0; s < a.split; s++) {
        const double *o = a.acc + (size_t)s * 3 * a.npad;
        fx += o[i];
        fy += o[a.npad + i];
        fz += o[2 * a.npad + i];
      }
    }
    if (a.force_mode == 1) {
      // FP64 path: acc holds the force; Vx += timeScaling * fx / Mass (body.go:120-122).
      vx += dt * fx / mi;
      vy += dt * fy / mi;
      vz += dt * fz / mi;
    } else {
      // FP32 path: acc holds sum mj dx / r^3; the kick is dt * G * a.  A massless body gets the
      // reference's 0/0 (its force G*0*mj/d^2 is zero), which the NaN guard below removes.
      if (mi == 0.0) {
        vx = vy = vz = __builtin_nan("");
      } else {
        vx += dt * (a.G * fx);
        vy += dt * (a.G * fy);
        vz += dt * (a.G * fz);
      }
    }
    a.vx[i] = vx;
    a.vy[i] = vy;
    a.vz[i] = vz;
  }
  const double x = a.x[i] + dt * vx;
  const double y = a.y[i] + dt * vy;
  const double z = a.z[i] + dt * vz;
  a.x[i] = x;
  a.y[i] = y;
  a.z[i] = z;
  a.collided[i] = 0;
  a.rest[i] = a.R;
  if (isnan(x) || isnan(y) || isnan(z)) {
    f &= (uint8_t)~NB_F_EXISTS;
    a.flags[i] = f;
    atomicAdd((unsigned long long *)&a.ctr->removed_total, 1ull);
  }
  a.js[i] = stream_entry(active_f(f), x, y, z, a.m[i]);
}

hipError_t launch_update(const UpdateArgs &a, hipStream_t st) {
  hipLaunchKernelGGL(k_update, dim3((unsigned)(a.npad / 256)), dim3(256), 0, st, a);
  return hipGetLastError();
}

__global__ void k_write_stream(const double *x, const double *y, const double *z,
                               const double *m, const uint8_t *flags, float4 *js, int n,
                               int npad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npad) return;
  js[i] = i < n ? stream_entry(active_f(flags[i]), x[i], y[i], z[i], m[i])
                : stream_entry(false, 0, 0, 0, 0);
}

hipError_t launch_write_stream(const double *x, const double *y, const double *z,
                               const double *m, const uint8_t *flags, float4 *js, int n,
                               int npad, hipStream_t st) {
  hipLaunchKernelGGL(k_write_stream, dim3((unsigned)(npad / 256)), dim3(256), 0, st, x, y, z, m,
                     flags, js, n, npad);
  return hipGetLastError();
}

// Per-tile max radius over active bodies, rounded up to the next float.
__global__ __launch_bounds__(256) void k_rmax_tile(const double *r, const uint8_t *flags, int n,
                                                   int tile_j, float *out) {
  __shared__ double sh[256];
  const int t = blockIdx.x;
  double mx = 0;
  for (int q = threadIdx.x; q < tile_j; q += blockDim.x) {
    const int j = t * tile_j + q;
    if (j < n && active_f(flags[j])) mx = fmax(mx, r[j]);
  }
  sh[threadIdx.x] = mx;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    float f = (float)sh[0];
    if ((double)f < sh[0]) f = __uint_as_float(__float_as_uint(f) + 1u);
    out[t] = f;
  }
}

hipError_t launch_rmax_tile(const double *r, const uint8_t *flags, int n, int tile_j, int tiles,
                            float *out, hipStream_t st) {
  hipLaunchKernelGGL(k_rmax_tile, dim3((unsigned)tiles), dim3(256), 0, st, r, flags, n, tile_j,
                     out);
  return hipGetLastError();
}

__global__ void k_zero_counters(DevCounters *c, int full) {
  if (threadIdx.x != 0) return;
  if (full) {
    DevCounters z{};
    *c = z;
  } else {
    c->pair_count = 0;
    c->rec_count = 0;
  }
}

hipError_t launch_zero_counters(DevCounters *ctr, int full, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, st, ctr, full);
  return hipGetLastError();
}

// Force per body (Body.fx/fy/fz) from the per-slice accumulators.
__global__ void k_combine_force(const double *acc, int split, int npad, int n, const double *m,
                                double G, int force_mode, double *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double f[3] = {0, 0, 0};
  for (int s = 0; s < split; s++)
    for (int c = 0; c < 3; c++) f[c] += acc[((size_t)s * 3 + c) * npad + i];
  for (int c = 0; c < 3; c++)
    out[(size_t)c * n + i] = force_mode == 1 ? f[c] : m[i] * (G * f[c]);
}

hipError_t launch_combine_force(const double *acc, int split, int npad, int n, const double *m,
                                double G, int force_mode, double *out, hipStream_t st) {
  hipLaunchKernelGGL(k_combine_force, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, acc,
                     split, npad, n, m, G, force_mode, out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Diagnostics: per-body FP64 terms then a fixed-order tree reduction (deterministic).
// scratch layout: [0, 8*n) per-body terms (ke, pe, px, py, pz, m, active, 0), then the result.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_diag_terms(const double *x, const double *y,
                                                    const double *z, const double *vx,
                                                    const double *vy, const double *vz,
                                                    const double *m, const uint8_t *flags, int n,
                                                    double eps, double *t) {
  // sources staged 256 at a time in LDS; each body sums its pair terms in ascending j
  __shared__ double sx[256], sy[256], sz[256], sm[256];
  __shared__ uint8_t se[256];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < n;
  const bool ex = valid && (flags[i] & NB_F_EXISTS);
  double ke = 0, pe = 0, px = 0, py = 0, pz = 0, mm = 0, act = 0;
  double xi = 0, yi = 0, zi = 0, mi = 0;
  if (ex) {
    mi = m[i];
    xi = x[i];
    yi = y[i];
    zi = z[i];
    ke = 0.5 * mi * (vx[i] * vx[i] + vy[i] * vy[i] + vz[i] * vz[i]);
    px = mi * vx[i];
    py = mi * vy[i];
    pz = mi * vz[i];
    mm = mi;
    act = 1;
  }
  const double eps2 = eps * eps;
  for (int j0 = 0; j0 < n; j0 += 256) {
    __syncthreads();
    const int jl = j0 + (int)threadIdx.x;
    if (jl < n) {
      sx[threadIdx.x] = x[jl];
      sy[threadIdx.x] = y[jl];
      sz[threadIdx.x] = z[jl];
      sm[threadIdx.x] = m[jl];
      se[threadIdx.x] = (flags[jl] & NB_F_EXISTS) ? 1 : 0;
    }
    __syncthreads();
    if (!ex) continue;
    const int cnt = min(256, n - j0);
    for (int jj = 0; jj < cnt; jj++) {
      if (j0 + jj == i || !se[jj]) continue;
      const double dx = sx[jj] - xi, dy = sy[jj] - yi, dz = sz[jj] - zi;
      const double d2 = dx * dx + dy * dy + dz * dz + eps2;
      if (d2 > 0) pe -= mi * sm[jj] / __builtin_sqrt(d2);
    }
  }
  if (!valid) return;
  pe *= 0.5;
  double *o = t + (size_t)i * 8;
  o[0] = ke;
  o[1] = pe;
  o[2] = px;
  o[3] = py;
  o[4] = pz;
  o[5] = mm;
  o[6] = act;
  o[7] = 0;
}

__global__ __launch_bounds__(256) void k_diag_reduce(const double *t, int n, double G,
                                                     double *out) {
  __shared__ double sh[256][8];
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  // Fixed assignment of bodies to threads and a fixed tree: the result does not depend on
  // scheduling.
  for (int i = threadIdx.x; i < n; i += blockDim.x)
    for (int c = 0; c < 8; c++) acc[c] += t[(size_t)i * 8 + c];
  for (int c = 0; c < 8; c++) sh[threadIdx.x][c] = acc[c];
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int c = 0; c < 8; c++) sh[threadIdx.x][c] += sh[threadIdx.x + w][c];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    for (int c = 0; c < 8; c++) out[c] = sh[0][c];
    out[1] = sh[0][1] * G;
  }
}

hipError_t launch_diag(const double *x, const double *y, const double *z, const double *vx,
                       const double *vy, const double *vz, const double *m, const uint8_t *flags,
                       int n, double G, double eps, double *scratch, int64_t scratch_len,
                       hipStream_t st) {
  if (scratch_len < (int64_t)n * 8 + 8) return hipErrorInvalidValue;
  if (n > 0)
    hipLaunchKernelGGL(k_diag_terms, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, y,
                       z, vx, vy, vz, m, flags, n, eps, scratch);
  hipLaunchKernelGGL(k_diag_reduce, dim3(1), dim3(256), 0, st, scratch, n, G,
                     scratch + (size_t)n * 8);
  return hipGetLastError();
}

__global__ void k_render(const double *x, const double *y, const double *z, const uint8_t *flags,
                         int n, float *xyz, uint8_t *exists) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const bool e = flags[i] & NB_F_EXISTS;
  // NewRenderable (renderable.go:22-40): float32 positions; zero for a non-existent body.
  exists[i] = e ? 1 : 0;
  xyz[3 * (size_t)i] = e ? (float)x[i] : 0.f;
  xyz[3 * (size_t)i + 1] = e ? (float)y[i] : 0.f;
  xyz[3 * (size_t)i + 2] = e ? (float)z[i] : 0.f;
}

hipError_t launch_render(const double *x, const double *y, const double *z, const uint8_t *flags,
                         int n, float *xyz, uint8_t *exists, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_render, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, y, z,
                     flags, n, xyz, exists);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Collection lifecycle on the device: compaction (BodyCollection.Cycle) and removals
// (ComputationRunner.processDeletes).
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_keep_count(const uint8_t *flags, int n, int run,
                                                    int32_t *part) {
  __shared__ int sh[4];
  const int64_t r0 = (int64_t)blockIdx.x * run, r1 = min(r0 + run, (int64_t)n);
  int v = 0;
  for (int64_t i = r0 + threadIdx.x; i < r1; i += 256) v += (flags[i] & NB_F_EXISTS) ? 1 : 0;
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

// Survivors to their places and zeros behind them up to the capacity: one pass over the two sets (a
// scan of the keep flags, 13 clears of whole arrays and the move apart were 145 us of kernels and
// 17 launches at 1,048,576 bodies; this and the count take 34).  A workgroup has a run of
// bodies, and the counts of the runs before it give its first place.
__global__ __launch_bounds__(256) void k_compact(CompactArgs a) {
  __shared__ int base_s[4], sum_s[4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t r0 = (int64_t)blockIdx.x * a.run;
  if (r0 < a.n) {  // uniform
    int before = 0;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += 256) before += a.part[b];
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
    if (lane == 0) base_s[w] = before;
    __syncthreads();
    int base = base_s[0] + base_s[1] + base_s[2] + base_s[3];
    for (int q = 0; q < a.run; q += 256) {  // 256 neighbours at a time, in order
      const int64_t i = r0 + q + threadIdx.x;
      const uint8_t f = i < a.n ? a.flags_src[i] : 0;
      const bool keep = f & NB_F_EXISTS;
      const uint64_t bal = __builtin_amdgcn_ballot_w64(keep);
      if (lane == 0) sum_s[w] = __builtin_popcountll(bal);
      __syncthreads();
      int p = base + __builtin_popcountll(bal & ((1ull << lane) - 1));
      for (int v = 0; v < 4; v++) {
        if (v < w) p += sum_s[v];
        base += sum_s[v];
      }
      __syncthreads();
      if (!keep) continue;
#pragma unroll
      for (int k = 0; k < 10; k++) a.dst[k][p] = a.src[k][i];
      a.beh_dst[p] = a.beh_src[i];
      a.flags_dst[p] = f;
      a.collided_dst[p] = 0;
      if (a.fstep_dst) a.fstep_dst[p] = a.fstep_src[i];
      if (a.fst_dst) a.fst_dst[p] = a.fst_src[i];
    }
  }
  for (int q = 0; q < a.run; q += 256) {
    const int64_t p = r0 + q + threadIdx.x;
    if (p < a.kept || p >= a.cap) continue;
#pragma unroll
    for (int k = 0; k < 10; k++) a.dst[k][p] = 0.0;
    a.beh_dst[p] = 0;
    a.flags_dst[p] = 0;
    a.collided_dst[p] = 0;
    if (a.fstep_dst) a.fstep_dst[p] = 0.0;
    if (a.fst_dst) a.fst_dst[p] = FragState{};
  }
}

hipError_t launch_compact(const CompactArgs &a, hipStream_t st) {
  const int64_t len = std::max<int64_t>(a.n, a.cap);
  if (len <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_compact, dim3((unsigned)((len + a.run - 1) / a.run)), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_keep_count(const uint8_t *flags, int n, int run, int32_t *part, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_keep_count, dim3((unsigned)(((int64_t)n + run - 1) / run)), dim3(256), 0, st,
                     flags, n, run, part);
  return hipGetLastError();
}

// processDeletes (computation-runner.go:176-216) without its sequential walk: the walk sets
// shouldRemove at every index that is a multiple of step and clears it at the first existing,
// unpinned body at or after that point.  So the removed bodies are, for each stride point p, the
// first such body in [p, p + step) -- or, if there is none, the one the next stride point finds
// (the flag is still set when the walk gets there).  One thread per stride point scans its own
// interval; the last one scans to the end.  all: the -1 request, every existing body.
__global__ void k_remove_walk(uint8_t *flags, double *m, int n, int step, int npoints, int all,
                              unsigned long long *removed) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= npoints) return;
  int lo, hi;
  if (all) {
    lo = k;
    hi = k + 1;
  } else {
    lo = k * step;
    hi = (k == npoints - 1) ? n : min(n, lo + step);
  }
  for (int i = lo; i < hi; i++) {
    const uint8_t f = flags[i];
    if ((f & NB_F_EXISTS) && (all || !(f & NB_F_PINNED))) {
      flags[i] = (uint8_t)(f & ~NB_F_EXISTS);  // SetNotExists (body.go:93-96)
      m[i] = 0.0;
      atomicAdd(&removed[0], 1ull);
      if (!(f & NB_F_FRAGMENTING)) atomicAdd(&removed[1], 1ull);
      break;
    }
  }
}

hipError_t launch_remove_walk(uint8_t *flags, double *m, int n, int step, int npoints, int all,
                              unsigned long long *removed, hipStream_t st) {
  if (npoints <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_remove_walk, dim3((unsigned)((npoints + 255) / 256)), dim3(256), 0, st,
                     flags, m, n, step, npoints, all, removed);
  return hipGetLastError();
}

// Largest radius over active bodies, as the bits of a non-negative double (their unsigned order
// is the numeric order), for the exact value the host computes when it loads the bodies.
__global__ __launch_bounds__(256) void k_rmax_active(const double *r, const uint8_t *flags, int n,
                                                     unsigned long long *out) {
  __shared__ unsigned long long sh[4];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long v = 0;
  if (i < n && active_f(flags[i]) && r[i] > 0.0) v = (unsigned long long)__double_as_longlong(r[i]);
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long w = __shfl_xor(v, o);
    v = w > v ? w : v;
  }
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 4; k++) v = sh[k] > v ? sh[k] : v;
    if (v) atomicMax(out, v);
  }
}

hipError_t launch_rmax_active(const double *r, const uint8_t *flags, int n,
                              unsigned long long *out, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_rmax_active, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, r, flags,
                     n, out);
  return hipGetLastError();
}

}  // namespace nb
