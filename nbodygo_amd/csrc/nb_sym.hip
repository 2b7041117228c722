// nb_sym.hip -- FP32 pairwise gravity with every unordered pair evaluated once.
//
// The force of nb_force.hip (a_i = sum_j m_j (x_j - x_i) / (|x_j - x_i|^2 + eps^2)^(3/2), the
// softened form of Body.Compute's loop, body.go:156-170) for eps > 0 without the overlap gate.
// nb_force.hip computes each pair twice, once from either side: 12 VALU ops and one v_rsq_f32 per
// ordered pair.  Here one evaluation of the differences, r^2, v_rsq_f32 and its cube serves both
// bodies: 16 VALU ops and one v_rsq_f32 per unordered pair, 8 and a half per ordered one.
//
// Split: bodies are cut into blocks of B = 64 IPL W.  A workgroup of W waves holds one block as
// targets (IPL per lane) and walks 64-body tiles of other blocks.  Within a tile lane l takes
// body (l + step) mod 64 at each of 64 steps; its position comes from LDS (the tile is stored
// twice in a row, so the address is the lane's base plus an immediate), and the three sums of the
// tile's bodies move with them, one lane per step, by the DPP wave rotate folded into the addition
// that ends the step.  So neither side needs a reduction across lanes.
// Block r meets the blocks r + 1 .. r + D (mod nb) with D = (nb - 1) / 2, and for even nb the first
// half of the blocks meets r + nb / 2 as well: every unordered pair of blocks once, the same work
// per row.  A block meets itself one-sided.
//
// Sums: a target keeps plain FP32 sums within a tile (64 sources) and adds them to FP64 sums in
// LDS; a tile body keeps plain FP32 sums over its 64 IPL partners per wave, the W waves are added
// in wave order, and the block's contribution is one FP32 triple per (block distance, body).
// k_sym_fold adds the target slices and the distances in FP64, in fixed order, so results do not
// depend on scheduling.  The tile bodies' sums are the ones in fewest bits: FP32 without compensation
// over up to 1,024 partners (64 steps of 4 in a chain, then 4 waves), as the one-sided kernel's are
// over the 512 of its tile.  Against FP64 the error is the one-sided kernel's or less, global / 99 of
// 100 bodies: 6.7e-8 / 2.1e-7 (one-sided 7.0e-8 / 2.2e-7) for a Plummer sphere of 262,144, 1.5e-7 /
// 4.7e-7 (1.5e-7 / 4.7e-7) of 65,536, 3.3e-7 / 9.6e-7 (3.6e-7 / 9.9e-7) of 4,096; and with masses far
// apart, where those sums matter most, at 65,536: lognormal with sigma 3 6.1e-7 / 8.4e-7 (7.4e-7 /
// 1.4e-6), one body with all of the mass 1.9e-7 / 3.1e-7 (the same), every seventh 64 bodies 1e5 times
// the others 3.8e-7 / 9.4e-7 (4.9e-7 / 1.9e-6).
//
// What bounds it: FP32 VALU issue.  gfx950 issues two independent FP32 instructions at a time, and
// the compiler's own order of a step (chains one target after another) leaves every second slot
// empty: 4,700 G interactions/s at N = 262,144.  With the step written as rows of independent
// instructions and the rows kept apart by scheduling barriers it is 5,560 to 5,650, against a ceiling
// of 5,790 from the measured issue rates of the instructions alone (at 2.4 GHz; the card holds 2.34).
// The one-sided kernel does 3,600 to 3,660 there.  Per force phase in a long run: 19.1 -> 12.2 to 12.4
// ms at N = 262,144, 1.18 -> 0.83 at 65,536, 0.30 -> 0.25 at 32,768; with detection 20.2 -> 12.8, 1.29
// -> 0.86 and 0.37 -> 0.26, 0.084 -> 0.050 at 10,000.  The first launches after an idle card are
// slower: 14.5, 12.8, 12.25 ms at 262,144, 0.95 to 1.0 for some thirty at 65,536.
//
// Detection: as nb_force.hip's bound on the tile's smallest r^2, evaluated from the target's side
// only (r^2 is symmetric); a flagged (target, tile) is re-tested at once in FP64 by the whole wave,
// one source per lane, with the reference's test (body.go:196-202).
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "nb_internal.hpp"

namespace nb {

__device__ __forceinline__ float rup_sym(double v) {  // smallest float >= v (v >= 0)
  float f = (float)v;
  if ((double)f < v) f = __uint_as_float(__float_as_uint(f) + 1u);
  return f;
}

// The neighbour's value: lane l receives lane l + 1's (lane 63 lane 0's).
__device__ __forceinline__ float from_next_lane(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x134 /* wave_rol:1 */, 0xf, 0xf, false));
}

// The reference's overlap test of target i against the 64 bodies of tile t, one per lane; `own`:
// the tile lies in the target's own block, where each pair is met from both sides.
template <class Buf>
__device__ __forceinline__ void exact_tile(const SymArgs &a, Buf &found, int i, int t, bool own) {
  const int j = t * 64 + (int)(threadIdx.x & 63);
  if (j >= a.n || j == i || (own && j < i)) return;
  const uint8_t fj = a.flags[j];
  if (!(fj & NB_F_EXISTS) || (fj & NB_F_FRAGMENTING)) return;
  const int32_t bi = a.beh[i];
  if (!nb_may_pair(bi, a.events)) return;
  const double dx = a.x[j] - a.x[i], dy = a.y[j] - a.y[i], dz = a.z[j] - a.z[i];
  const double d = __builtin_sqrt(dx * dx + dy * dy + dz * dz);
  const double ri = a.r[i], rj = a.r[j];
  if (d > ri + rj || !nb_pair_event(bi, a.beh[j], ri, rj, d, a.events)) return;
  found.add(a.pairs, a.ctr, a.pair_cap, min(i, j), max(i, j));
}

template <int IPL, int W, bool DETECT>
struct SymLds {
  float4 sh[2][128];
  float red[2][W][3][64];
  double sums[W][IPL][3][64];  // the targets' sums over the tiles so far
  PairBuf<DETECT ? 256 : 1> found;
};

// What one workgroup does: block `row` of a set of bodies against tiles u0 .. u1 - 1 of its list,
// which starts at tile `first` and wraps at ntiles.
struct SymWork {
  const float4 *js;  // the set's bodies
  int ntiles, nb, row, first, u0, u1;
  int slot0;         // distance d's sums go to layer slot d - slot0
  int limit;         // bodies a target's sums are written for
  size_t stride;     // words between components in acc and layer
  double *acc;
  float *layer;
};

template <int IPL, int W, bool DETECT>
__device__ __forceinline__ void sym_block(const SymWork &w, float eps2_s, const SymArgs &a,
                                          SymLds<IPL, W, DETECT> &lds) {
  constexpr int T = IPL * W;  // tiles per block
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = w.row, nb = w.nb, ntiles = w.ntiles, u0 = w.u0, u1 = w.u1;
  float xi[IPL], yi[IPL], zi[IPL], mi[IPL];
  float ri[IPL], amax[IPL];
  int live = 0;
#pragma unroll
  for (int k = 0; k < IPL; k++) {
    const int i = (row * T + wave * IPL + k) * 64 + lane;
    const float4 b = i < w.limit ? w.js[i] : make_float4(kSentinel, kSentinel, kSentinel, 0.f);
    xi[k] = b.x;
    yi[k] = b.y;
    zi[k] = b.z;
    mi[k] = b.w;
#pragma unroll
    for (int c = 0; c < 3; c++) lds.sums[wave][k][c][lane] = 0.0;
    if (DETECT) {
      const uint8_t f = i < a.n ? a.flags[i] : 0;
      if ((f & NB_F_EXISTS) && !(f & NB_F_FRAGMENTING)) live |= 1 << k;
      ri[k] = i < a.n ? rup_sym(a.r[i]) : 0.f;
      amax[k] = fmaxf(fabsf(b.x), fmaxf(fabsf(b.y), fabsf(b.z)));
    }
  }
  const float eps2 = to_vgpr(eps2_s);
  // The cube of 1/r is formed once for both bodies where it cannot leave FP32's normal range:
  // eps^2 >= 1e-24 and coordinates within 2.8e11 (r^2 < 1e24).  Elsewhere the masses are multiplied
  // in before the cube, as nb_force.hip does (one multiplication more per pair).  Sentinels need
  // neither: their terms are zero either way.
  auto tile_range = [](const float4 b) -> bool {
    const float m = fmaxf(fabsf(b.x), fmaxf(fabsf(b.y), fabsf(b.z)));
    const bool sentinel = b.x == kSentinel && b.y == kSentinel && b.z == kSentinel && b.w == 0.f;
    return __ballot(!(m <= 2.8e11f) && !sentinel) == 0;
  };
  bool near_range = eps2_s >= 1e-24f;
#pragma unroll
  for (int k = 0; k < IPL; k++)
    near_range = near_range && tile_range(make_float4(xi[k], yi[k], zi[k], mi[k]));

  int t = w.first + u0;
  if (t >= ntiles) t -= ntiles;
  if (DETECT && threadIdx.x == 0) lds.found.clear();
  if (u0 < u1 && wave == 0) {
    const float4 b = w.js[(size_t)t * 64 + lane];
    lds.sh[0][lane] = b;
    lds.sh[0][64 + lane] = b;
  }
  __syncthreads();
  for (int u = u0; u < u1; u++) {
    const int buf = (u - u0) & 1;
    int tn = t + 1;
    if (tn >= ntiles) tn -= ntiles;
    float4 next;
    const bool fetch = wave == 0 && u + 1 < u1;
    if (fetch) next = w.js[(size_t)tn * 64 + lane];
    const int blk = t / T;
    const int d = blk >= row ? blk - row : blk - row + nb;
    float px[IPL], py[IPL], pz[IPL], rmin[IPL];
#pragma unroll
    for (int k = 0; k < IPL; k++) px[k] = py[k] = pz[k] = 0.f, rmin[k] = FLT_MAX;
    const float4 *tl = &lds.sh[buf][lane];
    if (d != 0) {
      float qx = 0.f, qy = 0.f, qz = 0.f;
      // One step, written phase by phase over the targets with the order pinned: neighbouring
      // instructions are then independent, which is what lets gfx950 issue two at a time.
      auto step = [&](const float4 b, auto wide) {
        float dx[IPL], dy[IPL], dz[IPL], r2[IPL], inv[IPL], i2[IPL], gj[IPL], gi[IPL];
#pragma unroll
        for (int k = 0; k < IPL; k++) dx[k] = b.x - xi[k];
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) dy[k] = b.y - yi[k];
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) r2[k] = __builtin_fmaf(dx[k], dx[k], eps2);
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) dz[k] = b.z - zi[k];
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) r2[k] = __builtin_fmaf(dy[k], dy[k], r2[k]);
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) r2[k] = __builtin_fmaf(dz[k], dz[k], r2[k]);
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) {
          inv[k] = __builtin_amdgcn_rsqf(r2[k]);
          if (DETECT) rmin[k] = __builtin_fminf(rmin[k], r2[k]);
        }
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) i2[k] = inv[k] * inv[k];
        NB_ROW
        if constexpr (decltype(wide)::value) {
#pragma unroll
          for (int k = 0; k < IPL; k++) {
            gj[k] = b.w * inv[k] * i2[k];
            gi[k] = mi[k] * inv[k] * i2[k];
          }
        } else {
#pragma unroll
          for (int k = 0; k < IPL; k++) inv[k] *= i2[k];
          NB_ROW
#pragma unroll
          for (int k = 0; k < IPL; k++) gi[k] = mi[k] * inv[k];
          NB_ROW
#pragma unroll
          for (int k = 0; k < IPL; k++) gj[k] = b.w * inv[k];
        }
        NB_ROW
        float tx = dx[0] * gi[0], ty = dy[0] * gi[0], tz = dz[0] * gi[0];
#pragma unroll
        for (int k = 0; k < IPL; k++) {
          NB_ROW
          px[k] = __builtin_fmaf(dx[k], gj[k], px[k]);
          py[k] = __builtin_fmaf(dy[k], gj[k], py[k]);
          pz[k] = __builtin_fmaf(dz[k], gj[k], pz[k]);
          if (k + 1 < IPL) {
            NB_ROW
            tx = __builtin_fmaf(dx[k + 1], gi[k + 1], tx);
            ty = __builtin_fmaf(dy[k + 1], gi[k + 1], ty);
            tz = __builtin_fmaf(dz[k + 1], gi[k + 1], tz);
          }
        }
        NB_ROW
        // the sums of body (lane + s): so far one lane up (it took this body at step s - 1)
        qx = from_next_lane(qx) + tx;
        qy = from_next_lane(qy) + ty;
        qz = from_next_lane(qz) + tz;
      };
      float4 b = tl[0];
      if (tile_range(b) && near_range) {
#pragma unroll 4
        for (int s = 0; s < 64; s++) {
          const float4 bn = tl[s + 1];  // (step 63 reads entry lane + 64 <= 127)
          step(b, std::false_type{});
          b = bn;
        }
      } else {
        for (int s = 0; s < 64; s++) step(tl[s], std::true_type{});
      }
      // after step 63 lane l holds body (l + 63) mod 64: one more rotation brings it home
      lds.red[buf][wave][0][lane] = -from_next_lane(qx);
      lds.red[buf][wave][1][lane] = -from_next_lane(qy);
      lds.red[buf][wave][2][lane] = -from_next_lane(qz);
    } else {
      // the block against itself, one-sided; a target's own entry is met at step 0 of its own tile
      // (it adds exactly zero, but must not count as a candidate)
      float4 b = tl[0];
#pragma unroll 2
      for (int s = 0; s < 64; s++) {
        const float4 bn = tl[s + 1];
        float dx[IPL], dy[IPL], dz[IPL], r2[IPL], gj[IPL];
#pragma unroll
        for (int k = 0; k < IPL; k++) dx[k] = b.x - xi[k];
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) dy[k] = b.y - yi[k];
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) r2[k] = __builtin_fmaf(dx[k], dx[k], eps2);
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) dz[k] = b.z - zi[k];
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) r2[k] = __builtin_fmaf(dy[k], dy[k], r2[k]);
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) r2[k] = __builtin_fmaf(dz[k], dz[k], r2[k]);
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) {
          gj[k] = __builtin_amdgcn_rsqf(r2[k]);
          if (DETECT && !(s == 0 && t == row * T + wave * IPL + k))
            rmin[k] = __builtin_fminf(rmin[k], r2[k]);
        }
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) r2[k] = b.w * gj[k];
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) gj[k] = gj[k] * gj[k];
        NB_ROW
#pragma unroll
        for (int k = 0; k < IPL; k++) gj[k] = r2[k] * gj[k];
#pragma unroll
        for (int k = 0; k < IPL; k++) {
          NB_ROW
          px[k] = __builtin_fmaf(dx[k], gj[k], px[k]);
          py[k] = __builtin_fmaf(dy[k], gj[k], py[k]);
          pz[k] = __builtin_fmaf(dz[k], gj[k], pz[k]);
        }
        NB_ROW
        b = bn;
      }
    }
    if (fetch) {
      lds.sh[buf ^ 1][lane] = next;
      lds.sh[buf ^ 1][64 + lane] = next;
    }
#pragma unroll
    for (int k = 0; k < IPL; k++) {
      lds.sums[wave][k][0][lane] += (double)px[k];
      lds.sums[wave][k][1][lane] += (double)py[k];
      lds.sums[wave][k][2][lane] += (double)pz[k];
    }
    if (DETECT) {
      const float rmax = a.rmax_tile[t];
#pragma unroll
      for (int k = 0; k < IPL; k++) {
        // the bound of nb_force.hip's tile_end
        const float rs = ri[k] + rmax;
        const float e = 4.76837158e-7f * (amax[k] + rs);
        const float rse = rs + e;
        const float thr = __builtin_fmaf(rse, rse, eps2) * 1.0000039f;
        uint64_t hit = __ballot(rmin[k] <= thr && (live >> k & 1));
        if (hit && lane == 0)
          atomicAdd(&lds.found.tiles, (uint32_t)__builtin_popcountll(hit));
        while (hit) {
          const int l = __builtin_ctzll(hit);
          hit &= hit - 1;
          exact_tile(a, lds.found, (row * T + wave * IPL + k) * 64 + l, t, d == 0);
        }
      }
    }
    // one barrier per tile: the next tile is staged, every wave's sums are in lds.red[buf] (which is
    // written again two tiles on, after the next barrier)
    __syncthreads();
    if (d != 0) {
      for (int q = threadIdx.x; q < 192; q += 64 * W) {
        const int c = q >> 6, l = q & 63;
        float s = lds.red[buf][0][c][l];
#pragma unroll
        for (int v = 1; v < W; v++) s += lds.red[buf][v][c][l];
        w.layer[((size_t)(d - w.slot0) * 3 + c) * w.stride + t * 64 + l] = s;
      }
    }
    t = tn;
  }
  double *o = w.acc;
#pragma unroll
  for (int k = 0; k < IPL; k++) {
    const int i = (row * T + wave * IPL + k) * 64 + lane;
    if (i >= w.limit) continue;
    o[i] = lds.sums[wave][k][0][lane];
    o[w.stride + i] = lds.sums[wave][k][1][lane];
    o[2 * w.stride + i] = lds.sums[wave][k][2][lane];
  }
  if (DETECT) lds.found.flush(a.pairs, a.ctr, a.pair_cap);
}

template <int IPL, int W, bool DETECT>
__global__ __launch_bounds__(64 * W)
__attribute__((amdgpu_waves_per_eu(IPL == 1 ? 8 : IPL == 2 ? 6 : 4)))
void k_force_sym(SymArgs a) {
  constexpr int T = IPL * W;
  __shared__ SymLds<IPL, W, DETECT> lds;
  if (a.run_flag && *a.run_flag == 0u) return;  // conditional launch (surrogate fallback)
  const int row = blockIdx.x, slice = blockIdx.y;
  // the row's tiles: its own block's (first panel only), then those of blocks row + d0 .. row + d1
  const int nb = a.nb, ntiles = a.ntiles;
  const int dmax = (nb - 1) / 2 + ((nb & 1) == 0 && row < nb / 2 ? 1 : 0);
  const int d1 = min(a.d1, dmax);
  auto tiles_upto = [&](int b) { return min(b * T, ntiles); };  // b in [0, nb]
  int len = 0;
  if (d1 >= a.d0) {
    const int b0 = row + a.d0, b1 = row + d1 + 1;  // blocks [b0, b1), possibly past nb
    const int lo = b0 >= nb ? ntiles + tiles_upto(b0 - nb) : tiles_upto(b0);
    const int hi = b1 > nb ? ntiles + tiles_upto(b1 - nb) : tiles_upto(b1);
    len = hi - lo;
  }
  SymWork w;
  w.js = a.js;
  w.ntiles = ntiles;
  w.nb = nb;
  w.row = row;
  w.first = (row + a.d0) % nb * T;
  w.u0 = (int)((int64_t)len * slice / a.slices);
  w.u1 = (int)((int64_t)len * (slice + 1) / a.slices);
  w.slot0 = a.d0 == 0 ? 1 : a.d0;
  w.limit = a.npad;
  w.stride = (size_t)a.npad;
  w.acc = a.acc + (size_t)slice * 3 * a.npad;
  w.layer = a.layer;
  sym_block<IPL, W, DETECT>(w, a.eps2, a, lds);
}

// Many sets of bodies (batched simulations) in one persistent launch: items are (simulation, block,
// range of its tiles), longest first, taken from a device queue until it is exhausted.
// 512 simulations of 256 to 8,192 bodies: 2.7 ms a step, 4,500 G interactions/s, FP32 VALU issue
// (a simulation's blocks against themselves, a fifth of the tiles at 8,192 bodies, are one-sided);
// the one-sided kernel of nb_batch.hip takes 4.3 ms in its default shape, 3.45 in its tuned one.
// 8 simulations of 64 to 128 bodies: 0.041 -> 0.019 ms; 64 of 500 to 4,000: 0.29 -> 0.15 (tuned
// 0.16).  Blocks of two waves or one: 2.73 and 2.70 ms for the first, 0.16 and 0.20 for the last.
__global__ __launch_bounds__(64 * kBatchSymW) __attribute__((amdgpu_waves_per_eu(4)))
void k_batch_sym(BatchSymArgs b) {
  constexpr int W = kBatchSymW;
  __shared__ __attribute__((aligned(16))) char raw[sizeof(SymLds<4, W, false>)];
  __shared__ int cur;
  SymArgs none{};
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) cur = (int)atomicAdd(b.next, 1u);
    __syncthreads();
    const int q = cur;
    if (q >= b.nitems) break;
    const BatchSymItem it = b.items[q];
    SymWork w;
    w.js = b.js + it.p0;
    w.ntiles = it.ntiles;
    w.nb = it.nb;
    w.row = it.row;
    w.first = it.row * it.ipl * W;
    w.u0 = it.u0;
    w.u1 = it.u1;
    w.slot0 = 1;
    w.limit = it.ntiles * 64;
    w.stride = (size_t)b.npad;
    w.acc = b.acc + (size_t)it.slice * 3 * b.npad + it.p0;
    w.layer = b.layer + it.p0;
    if (it.ipl == 4)
      sym_block<4, W, false>(w, b.eps2, none, reinterpret_cast<SymLds<4, W, false> &>(raw));
    else if (it.ipl == 2)
      sym_block<2, W, false>(w, b.eps2, none, reinterpret_cast<SymLds<2, W, false> &>(raw));
    else
      sym_block<1, W, false>(w, b.eps2, none, reinterpret_cast<SymLds<1, W, false> &>(raw));
  }
}

// The batch's k_sym_fold: a body's slices and distances follow from its simulation.
__global__ __launch_bounds__(256) void k_batch_sym_fold(BatchSymArgs b, double *out) {
  const int c = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;  // npad is a multiple of 256
  const int64_t g = (int64_t)c * b.npad + i;
  const int sim = b.tile_sim[i >> 6];
  if (sim < 0) {
    out[g] = 0.0;
    return;
  }
  const BatchSymSim s = b.sims[sim];
  const size_t st = (size_t)3 * b.npad;
  double v = 0.0;
  for (int q = 0; q < s.slices; q++) v += b.acc[q * st + g];
  const int blk = (i - s.p0) / (s.ipl * 64 * kBatchSymW);
  const int cnt = (s.nb - 1) / 2 + ((s.nb & 1) == 0 && blk >= s.nb / 2 ? 1 : 0);
  const float *p = b.layer + (size_t)c * b.npad + i;
  for (int q = 0; q < cnt; q++) v += p[(size_t)q * st];
  out[g] = v;
}

hipError_t launch_batch_sym(const BatchSymArgs &b, double *out, int cus, hipStream_t st) {
  // 16 waves per CU are resident at once
  hipLaunchKernelGGL(k_batch_sym, dim3((unsigned)std::min(b.nitems, cus * 16 / kBatchSymW)),
                     dim3(64 * kBatchSymW), 0, st, b);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_batch_sym_fold, dim3((unsigned)(b.npad / 256), 3), dim3(256), 0, st, b,
                     out);
  return hipGetLastError();
}

// out = (first panel: 0, later: out) + the target slices + the distances that reached the body's
// block, in FP64 and in this order; one thread per word.
__global__ __launch_bounds__(256) void k_sym_fold(SymArgs a, int T, double *out) {
  if (a.run_flag && *a.run_flag == 0u) return;
  const int c = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;  // npad is a multiple of 256
  const int64_t g = (int64_t)c * a.npad + i;
  const size_t st = (size_t)3 * a.npad;
  double s = a.d0 == 0 ? 0.0 : out[g];
  for (int q = 0; q < a.slices; q++) s += a.acc[q * st + g];
  if (i >> 6 < a.ntiles) {
    // for even nb the largest distance reached only the blocks of the second half
    const int nb = a.nb, blk = (i >> 6) / T, lo = a.d0 == 0 ? 1 : a.d0;
    const int dmax = (nb - 1) / 2 + ((nb & 1) == 0 && blk >= nb / 2 ? 1 : 0);
    const int cnt = min(a.d1, dmax) - lo + 1;
    const float *p = a.layer + (size_t)c * a.npad + i;
    int q = 0;
    for (; q + 8 <= cnt; q += 8) {  // eight loads in flight
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] = p[(size_t)(q + e) * st];
#pragma unroll
      for (int e = 0; e < 8; e++) s += v[e];
    }
    for (; q < cnt; q++) s += p[(size_t)q * st];
  }
  out[g] = s;
}

template <int IPL, int W>
static hipError_t launch_sym_t(const SymArgs &a, int nb, bool detect, hipStream_t st) {
  const dim3 grid((unsigned)nb, (unsigned)a.slices), block(64 * W);
  if (detect)
    hipLaunchKernelGGL((k_force_sym<IPL, W, true>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((k_force_sym<IPL, W, false>), grid, block, 0, st, a);
  return hipGetLastError();
}

hipError_t launch_force_sym(const ForceShape &s, SymArgs a, double *out, int64_t layer_words,
                            bool detect, hipStream_t st) {
  const int W = s.block / 64, T = W * s.ipl;
  a.ntiles = (a.n + 63) / 64;
  a.nb = (a.ntiles + T - 1) / T;
  a.slices = s.jsplit;
  if (a.ntiles < 1 || a.ntiles * 64 > a.npad || s.jsplit < 1 || s.jsplit > kMaxSplit)
    return hipErrorInvalidValue;
  const int dall = a.nb / 2;  // the largest distance any row takes
  const int64_t per = (int64_t)3 * a.npad;
  const int fit = (int)(layer_words / per < dall ? layer_words / per : dall);
  if (fit < 1 && dall > 0) return hipErrorInvalidValue;
  // panels of block distances whose layers fit the workspace (one panel unless n is very large)
  for (int d = 0; d <= dall;) {
    a.d0 = d;
    a.d1 = d == 0 ? fit : (d + fit - 1 < dall ? d + fit - 1 : dall);
    hipError_t e;
    switch (s.ipl * 100 + W) {
      case 104: e = launch_sym_t<1, 4>(a, a.nb, detect, st); break;
      case 204: e = launch_sym_t<2, 4>(a, a.nb, detect, st); break;
      case 404: e = launch_sym_t<4, 4>(a, a.nb, detect, st); break;
      default: return hipErrorInvalidValue;
    }
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_sym_fold, dim3((unsigned)(a.npad / 256), 3), dim3(256), 0, st, a, T,
                       out);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    d = a.d1 + 1;
  }
  return hipSuccess;
}

}  // namespace nb
