// nb_bh.hip -- the reference's Barnes-Hut octree (cmd/body/octree.go) on the device, with Build
// wired into BuildTree (the reference only allocates an empty tree, body_collection.go:298-300,
// so its default mode computes no gravity).  FP64 throughout, with the reference's arithmetic
// for every interaction.
//
// Build, every force phase:
//   box     min/max over existing, non-fragmenting bodies; the root's centre and half exactly as
//           Build computes them (octree.go:136-194)
//   keys    each body descends from the root with the reference's centre arithmetic (octantOf,
//           childCenter: octree.go:55-88), one octal digit per level, max_depth levels
//   sort    stable radix sort of the keys: every node's bodies are one contiguous run, and a
//           bucket's bodies (the depth limit) stay in array order
//   nodes   from how many digits neighbours in key order share, every node's first body and depth;
//           then each node splits its run into its eight octant runs by binary
//           search on that level's digit.  Runs of two or more bodies become nodes, single
//           bodies leaves -- the tree that leaf-capacity-1 insertion builds (insert, subdivide:
//           octree.go:198-231): same topology, node centres, halves and leaf depths.
//   mass    bottom-up, deepest first.  A leaf's mass and centre of mass are updateMass's from zero,
//           (0 + x*m) / (0 + m) (octree.go:91-97); a node sums its children in octant order.
//           (The reference folds bodies into each node one at a time in array order, so a
//           node's centre of mass can differ from it in the last bits; leaves are identical.)
//           A bucket folds its bodies in array order as updateMass does.
// Links, after the masses: each live child slot gets the slot to visit when the walk opens it
// (its first live child) and the one to visit when it is accepted or done (its next live
// sibling, else its parent's), so a depth-first walk needs no stack.
// Force (accumForce, octree.go:276-309): one lane per body, bodies in key order.  Each lane walks
// the tree on its own by those links: it accepts or opens a node by its own test
// (2*half/dist) < theta, and children come in octant order, so every body's sum has the
// reference's terms in the reference's order.  Suns sum directly over all bodies in array order
// (CalcForce, octree.go:252-267).
// Collisions: a second walk opens every node whose box lies within R_i + R_max of the body and
// applies the reference's test at the leaves (Collided, body.go:192-208); pairs go to the same
// canonical list as the direct path.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>

#include <rocprim/rocprim.hpp>

#include "nb_internal.hpp"

namespace nb {

constexpr int kBhLevels = 21;        // octal digits in a 64-bit key
constexpr int kBhStack = 160;        // collision walk: per-wave stack entries (bound 7 * 20 + 8)
constexpr int32_t kBucket = INT32_MIN;
constexpr int kSunChunk = 64;

struct BhCounters {
  int32_t M;                         // bodies in the tree
  int32_t depth_max;                 // deepest leaf
  int32_t nodes;                     // nodes of two or more bodies
  uint32_t nsun;
  uint32_t buckets;
  uint32_t stack_overflow;
  uint32_t node_overflow;
  int32_t root_first;                // the root's first live child slot (-1: none)
  unsigned long long interactions;   // accepted nodes + leaf and direct terms, all targets
};

// A child as the force walk needs it, eight per node: centre of mass and mass (a leaf's from
// updateMass from zero), the child's code (-1 empty, <= -2 the leaf of sorted body -2 - code,
// else a node), the walk's links: `first` (slot of its first live child, for a node that is
// opened) and `skip` (slot visited next once this subtree is done; -1 ends the walk), and `dep`:
// a node's depth (its half is the root's halved dep times, exactly as the build halves it), -1
// for a bucket, 0 for a leaf or an empty slot.  A slot is live when its code is not -1 and its
// mass is > 0.  48 bytes: three 16-byte loads per visit instead of four, the half coming from
// a per-depth table.
struct alignas(16) BhSlot {
  double x, y, z, m;
  int32_t code, first, skip, dep;
};
static_assert(sizeof(BhSlot) == 48, "three 16-byte words");

// 2 half of each depth (the root's half, halved once per level: exact, as in the build), for
// d = 0..kBhLevels, into a workgroup's LDS table.
__device__ __forceinline__ void bh_half2_table(const double4 *nbox, double *h2s) {
  if (threadIdx.x <= kBhLevels) {
    double h = nbox[0].w;
    for (int d = 0; d < (int)threadIdx.x; d++) h = h / 2;
    h2s[threadIdx.x] = 2 * h;
  }
  __syncthreads();
}

struct Bh {
  nb_bh_params p{};
  int64_t cap = 0, node_cap = 0;
  uint64_t *keys_in = nullptr, *keys = nullptr;
  int32_t *perm_in = nullptr, *perm = nullptr;
  double *sx = nullptr, *sy = nullptr, *sz = nullptr, *sm = nullptr;
  double *lcx = nullptr, *lcy = nullptr, *lcz = nullptr;
  int32_t *depth = nullptr, *suns = nullptr;
  double4 *nbox = nullptr, *nmc = nullptr;
  int32_t *nchild = nullptr;
  BhSlot *slots = nullptr;
  int32_t *pslot = nullptr;  // each node's slot in its parent
  int2 *nrange = nullptr;    // each node's bodies
  int2 *nstart = nullptr;    // each node's first body and depth
  int32_t *first = nullptr;  // the first node that a body or a later one starts
  int32_t *npart = nullptr, *cross = nullptr;
  uint8_t *live = nullptr;
  double *bpart = nullptr;
  void *sort_tmp = nullptr;
  size_t sort_bytes = 0;
  BhCounters *cnt = nullptr;
  int64_t builds = 0;
  int cus = 256;  // compute units of the device
};

template <class T>
static hipError_t balloc(T **p, size_t count) {
  if (*p) {
    (void)hipFree(*p);
    *p = nullptr;
  }
  return hipMalloc((void **)p, std::max<size_t>(count, 1) * sizeof(T));
}

__device__ __forceinline__ bool bh_active(uint8_t f) {
  return (f & NB_F_EXISTS) && !(f & NB_F_FRAGMENTING);
}

__device__ __forceinline__ void bh_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// ---- box ---------------------------------------------------------------------------------------
// Partial min/max (x, y, z) and count over existing, non-fragmenting bodies: 7 values per block.
__global__ __launch_bounds__(256) void k_bh_box_part(const double *x, const double *y,
                                                     const double *z, const uint8_t *flags, int n,
                                                     double *part) {
  __shared__ double sh[7][256];
  double v[7] = {DBL_MAX, DBL_MAX, DBL_MAX, -DBL_MAX, -DBL_MAX, -DBL_MAX, 0.0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    if (!bh_active(flags[i])) continue;
    const double px = x[i], py = y[i], pz = z[i];
    v[0] = px < v[0] ? px : v[0];
    v[1] = py < v[1] ? py : v[1];
    v[2] = pz < v[2] ? pz : v[2];
    v[3] = px > v[3] ? px : v[3];
    v[4] = py > v[4] ? py : v[4];
    v[5] = pz > v[5] ? pz : v[5];
    v[6] += 1.0;
  }
  for (int q = 0; q < 7; q++) sh[q][threadIdx.x] = v[q];
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      const int o = threadIdx.x + s;
      for (int q = 0; q < 3; q++) {
        const double a = sh[q][threadIdx.x], b = sh[q][o];
        sh[q][threadIdx.x] = b < a ? b : a;
      }
      for (int q = 3; q < 6; q++) {
        const double a = sh[q][threadIdx.x], b = sh[q][o];
        sh[q][threadIdx.x] = b > a ? b : a;
      }
      sh[6][threadIdx.x] += sh[6][o];
    }
    __syncthreads();
  }
  if (threadIdx.x < 7) part[blockIdx.x * 8 + threadIdx.x] = sh[threadIdx.x][0];
}

// The root cell (Build: cx = (minX + maxX) / 2, half = max extent / 2 * 1.05) and the level
// bookkeeping.  One block of 256: the partials are folded per thread, then in LDS (min, max and
// sums of whole numbers are exact in any order).
__global__ __launch_bounds__(256) void k_bh_root(const double *part, int nparts,
                                                 BhCounters *cnt, double4 *nbox,
                                                 int32_t *nchild) {
  __shared__ double sh[7][256];
  double v[7] = {DBL_MAX, DBL_MAX, DBL_MAX, -DBL_MAX, -DBL_MAX, -DBL_MAX, 0.0};
  for (int b = threadIdx.x; b < nparts; b += blockDim.x) {
    const double *p = part + b * 8;
    for (int q = 0; q < 3; q++) v[q] = p[q] < v[q] ? p[q] : v[q];
    for (int q = 3; q < 6; q++) v[q] = p[q] > v[q] ? p[q] : v[q];
    v[6] += p[6];
  }
  for (int q = 0; q < 7; q++) sh[q][threadIdx.x] = v[q];
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) {
      const int o = threadIdx.x + st;
      for (int q = 0; q < 3; q++) {
        const double a = sh[q][threadIdx.x], b = sh[q][o];
        sh[q][threadIdx.x] = b < a ? b : a;
      }
      for (int q = 3; q < 6; q++) {
        const double a = sh[q][threadIdx.x], b = sh[q][o];
        sh[q][threadIdx.x] = b > a ? b : a;
      }
      sh[6][threadIdx.x] += sh[6][o];
    }
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  for (int q = 0; q < 7; q++) v[q] = sh[q][0];
  const int M = (int)v[6];
  cnt->M = M;
  cnt->depth_max = 0;
  cnt->nodes = 0;
  cnt->nsun = 0;
  cnt->buckets = 0;
  cnt->stack_overflow = 0;
  cnt->node_overflow = 0;
  cnt->interactions = 0;
  if (M == 0) return;
  const double ex = v[3] - v[0], ey = v[4] - v[1], ez = v[5] - v[2];
  const double mx = ey > ez ? ey : ez;  // math.Max on finite values
  const double half = (ex > mx ? ex : mx) / 2 * 1.05;
  nbox[0] = make_double4((v[0] + v[3]) / 2, (v[1] + v[4]) / 2, (v[2] + v[5]) / 2, half);
  for (int c = 0; c < 8; c++) nchild[c] = -1;
}

// Octant path of each body from the root, octantOf / childCenter op by op; D digits,
// left-aligned in 63 bits.  Bodies outside the tree get the largest key.
__global__ __launch_bounds__(256) void k_bh_keys(const double *x, const double *y,
                                                 const double *z, const uint8_t *flags, int n,
                                                 const double4 *nbox, int D, uint64_t *keys,
                                                 int32_t *perm, int32_t *depth) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  perm[i] = i;
  depth[i] = -1;
  if (!bh_active(flags[i])) {
    keys[i] = ~0ull;
    return;
  }
  const double4 r = nbox[0];
  double cx = r.x, cy = r.y, cz = r.z, half = r.w;
  const double px = x[i], py = y[i], pz = z[i];
  uint64_t key = 0;
  for (int l = 0; l < D; l++) {
    const int o = (px >= cx ? 1 : 0) | (py >= cy ? 2 : 0) | (pz >= cz ? 4 : 0);
    key = (key << 3) | (uint64_t)o;
    const double q = half / 2;
    cx = (o & 1) ? cx + q : cx - q;
    cy = (o & 2) ? cy + q : cy - q;
    cz = (o & 4) ? cz + q : cz - q;
    half = half / 2;
  }
  keys[i] = key << (3 * (kBhLevels - D));
}

// Sorted copies of position and mass, and each body's leaf centre of mass (updateMass from
// zero: (0*0 + x*m) / (0 + m)).
__global__ __launch_bounds__(256) void k_bh_gather(const int32_t *perm, const double *x,
                                                   const double *y, const double *z,
                                                   const double *m, const BhCounters *cnt,
                                                   double *sx, double *sy, double *sz,
                                                   double *sm, double *lcx, double *lcy,
                                                   double *lcz) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= cnt->M) return;
  const int i = perm[s];
  const double px = x[i], py = y[i], pz = z[i], mm = m[i];
  const double zero = 0.0;
  const double tot = zero + mm;
  sx[s] = px;
  sy[s] = py;
  sz[s] = pz;
  sm[s] = mm;
  lcx[s] = (zero * zero + px * mm) / tot;
  lcy[s] = (zero * zero + py * mm) / tot;
  lcz[s] = (zero * zero + pz * mm) / tot;
}

// ---- nodes -------------------------------------------------------------------------------------
// The tree follows from how many leading digits neighbours in key order share.  Let L(j) be that
// number for bodies j - 1 and j (at most D; -1 before the first body and after the last).  A node of
// depth d is a run of two or more bodies with d digits in common, so body j starts one for every d
// with L(j) < d <= L(j + 1), and nodes numbered by their first body, then by depth, are in
// depth-first order with the root first.  All of them can then be made at once (a launch per level,
// 21 of them, was 380 us at 262,144 bodies, mostly launches and one counter of the next level's
// nodes; these three take 34).
__device__ __forceinline__ int bh_shared(const uint64_t *keys, int j, int M, int D) {
  if (j <= 0 || j >= M) return -1;
  const uint64_t x = keys[j - 1] ^ keys[j];
  return x ? (__builtin_clzll(x) - 1) / 3 : D;  // keys use bits 0..62
}

constexpr int kBhRun = 1024;  // bodies per workgroup of the next two: four to a thread

// Nodes started in each run of kBhRun bodies; every body's leaf depth.
__global__ __launch_bounds__(256) void k_bh_count(const uint64_t *keys, const int32_t *perm, int D,
                                                  BhCounters *cnt, int32_t *part,
                                                  int32_t *depth) {
  __shared__ int red[3][4];
  const int M = cnt->M, j0 = blockIdx.x * kBhRun + threadIdx.x * 4;
  int n = 0, buckets = 0, deep = 0;
  int l = bh_shared(keys, j0, M, D);
  for (int j = j0; j < min(j0 + 4, M); j++) {
    const int l1 = bh_shared(keys, j + 1, M, D);
    n += max(0, l1 - l);
    buckets += l < D && l1 == D;
    const int dep = min(max(l, l1) + 1, D);
    depth[perm[j]] = dep;
    deep = max(deep, dep);
    l = l1;
  }
  for (int o = 32; o > 0; o >>= 1) {
    n += __shfl_xor(n, o);
    buckets += __shfl_xor(buckets, o);
    deep = max(deep, __shfl_xor(deep, o));
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = n;
    red[1][threadIdx.x >> 6] = buckets;
    red[2][threadIdx.x >> 6] = deep;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  part[blockIdx.x] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
  buckets = red[1][0] + red[1][1] + red[1][2] + red[1][3];
  deep = max(max(red[2][0], red[2][1]), max(red[2][2], red[2][3]));
  if (buckets) atomicAdd(&cnt->buckets, (uint32_t)buckets);
  if (deep > 0) atomicMax(&cnt->depth_max, deep);
}

// first[j]: the first node that body j or a later one starts (first[M]: the number of nodes);
// nstart[node] = (first body, depth).
__global__ __launch_bounds__(256) void k_bh_starts(const uint64_t *keys, int D, BhCounters *cnt,
                                                   const int32_t *part, int64_t node_cap,
                                                   int32_t *first, int2 *nstart) {
  __shared__ int wsum[4], base_s[4];
  const int M = cnt->M, j0 = blockIdx.x * kBhRun + threadIdx.x * 4;
  if ((int)(blockIdx.x * kBhRun) >= M) return;  // uniform
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int before = 0;
  for (int b = threadIdx.x; b < (int)blockIdx.x; b += 256) before += part[b];
  int l[5], n = 0;
  for (int q = 0; q < 5; q++) l[q] = bh_shared(keys, j0 + q, M, D);
  for (int q = 0; q < 4; q++) n += max(0, l[q + 1] - l[q]);
  int scan = n;
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(scan, o);
    if (lane >= o) scan += v;
  }
  for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
  if (lane == 63) {
    wsum[w] = scan;
    base_s[w] = before;
  }
  __syncthreads();
  int id = base_s[0] + base_s[1] + base_s[2] + base_s[3] + scan - n;
  for (int v = 0; v < w; v++) id += wsum[v];
  for (int q = 0; q < 4 && j0 + q < M; q++) {
    first[j0 + q] = id;
    for (int d = l[q] + 1; d <= l[q + 1]; d++, id++)
      if (id < node_cap) nstart[id] = make_int2(j0 + q, d);
    if (j0 + q == M - 1) {
      first[M] = id;
      cnt->nodes = id;
      if (id > node_cap) cnt->node_overflow = 1;
    }
  }
}

__device__ __forceinline__ int bh_nodes(const BhCounters *cnt, int64_t node_cap) {
  return (int)min((int64_t)cnt->nodes, node_cap);
}

struct BhNodeArgs {
  const uint64_t *keys;
  const BhCounters *cnt;
  const int32_t *first;
  const int2 *nstart;
  double4 *nbox;
  int2 *nrange;
  int32_t *nchild, *pslot;
  int64_t node_cap;
  int D;
};

// Eight lanes per node.  The run's end by an eight-way search upwards from its start; then lane c
// (1..7) finds by binary search the first body whose digit d is >= c, the boundaries go round by
// shuffles, and lane c makes child c's code.  A child of two or more bodies is the node after this
// one if it starts with it, else the first that its own first body starts.
__global__ __launch_bounds__(256) void k_bh_nodes(BhNodeArgs a) {
  const int nodes = bh_nodes(a.cnt, a.node_cap), M = a.cnt->M, D = a.D;
  const int c = threadIdx.x & 7, gsh = threadIdx.x & 56;
  const int groups = gridDim.x * (blockDim.x >> 3);
  const int mine = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 3);
  // every lane runs the same number of iterations, so ballots and shuffles see full groups
  for (int k0 = 0; k0 < nodes; k0 += groups) {
    const int k = mine + k0;
    const bool live = k < nodes;
    const int2 st = live ? a.nstart[k] : make_int2(0, 0);
    const int lo = st.x, d = st.y, sh = 63 - 3 * d;
    const uint64_t pre = live ? a.keys[lo] >> sh : 0;
    auto inside = [&](int t) { return live && t < M && (a.keys[t] >> sh) == pre; };
    auto count = [&](bool in) {  // of the group's lanes; those inside come first
      return __builtin_popcount((uint32_t)(__builtin_amdgcn_ballot_w64(in) >> gsh) & 255u);
    };
    // the bodies lo + 2, lo + 8, lo + 32, ...; then the range between the last inside (b0) and the
    // first outside (b1) cut in nine, until they are neighbours
    int n = count(inside(lo + (2 << (2 * c))));
    int b0 = n ? lo + (2 << (2 * (n - 1))) : lo + 1;
    int b1 = n < 8 ? min(M, lo + (2 << (2 * n))) : M;
    if (!live) b1 = b0;
    while (__builtin_amdgcn_ballot_w64(b1 - b0 > 1)) {
      const int span = b1 - b0;
      auto at = [&](int q) { return span <= 9 ? b0 + q + 1 : b0 + (int)((int64_t)span * (q + 1) / 9); };
      const int t = at(c);
      n = count(t < b1 && inside(t));
      const int n0 = n ? at(n - 1) : b0, n1 = n < 8 ? min(b1, at(n)) : b1;
      b0 = n0;
      b1 = n1;
    }
    const int hi = b1;
    const bool bucket = d == D;
    int lb = lo;
    if (live && !bucket && c > 0) {
      const int dsh = 60 - 3 * d;
      int p = lo, q = hi;
      while (p < q) {
        const int mid = (p + q) >> 1;
        if ((int)((a.keys[mid] >> dsh) & 7) < c)
          p = mid + 1;
        else
          q = mid;
      }
      lb = p;
    }
    int ub = __shfl_down(lb, 1, 8);
    if (c == 7) ub = hi;
    if (!live) continue;
    int32_t code = -1;
    if (bucket) {  // depth limit: a bucket of bodies in array order
      code = c == 0 ? kBucket : c == 1 ? lo : c == 2 ? hi - lo : -1;
    } else if (ub - lb == 1) {
      code = -2 - lb;
    } else if (ub - lb >= 2) {
      const int id = lb == lo ? k + 1 : a.first[lb];
      if (id < a.node_cap) {
        code = id;
        a.pslot[id] = k * 8 + c;
      }
    }
    a.nchild[(size_t)k * 8 + c] = code;
    if (c != 0) continue;
    a.nrange[k] = make_int2(lo, hi);
    if (k == 0) continue;  // the root's box is there
    // centre and half from the root's, a digit at a time, as the keys were made
    double4 bx = a.nbox[0];
    const uint64_t key = a.keys[lo];
    for (int e = 0; e < d; e++) {
      const int o = (int)((key >> (60 - 3 * e)) & 7);
      const double q = bx.w / 2;
      bx.x = (o & 1) ? bx.x + q : bx.x - q;
      bx.y = (o & 2) ? bx.y + q : bx.y - q;
      bx.z = (o & 4) ? bx.z + q : bx.z - q;
      bx.w = bx.w / 2;
    }
    a.nbox[k] = bx;
  }
}

// ---- masses and links --------------------------------------------------------------------------
// Bottom-up: mass and centre of mass of a node from its children (or, for a bucket, its bodies
// folded in array order by updateMass), its children's slots, and which of them are live.
struct BhMassArgs {
  const BhCounters *cnt;
  const int32_t *nchild, *first;
  const int2 *nstart, *nrange;
  double4 *nmc;
  BhSlot *slots;
  uint8_t *live;  // bit c: slot c of the node is live
  int32_t *cross;
  const double *sx, *sy, *sz, *sm, *lcx, *lcy, *lcz;
  int64_t node_cap;
  int D, blocks;
};

__device__ __forceinline__ void bh_mass_node(const BhMassArgs &a, int k, int d) {
  const int4 *cw = reinterpret_cast<const int4 *>(a.nchild + (size_t)k * 8);
  const int4 c0 = cw[0], c1 = cw[1];
  if (d == a.D) {
    double mt = 0, cx = 0, cy = 0, cz = 0;
    for (int s = c0.y; s < c0.y + c0.z; s++) {
      const double mm = a.sm[s];
      const double nt = mt + mm;
      cx = (cx * mt + a.sx[s] * mm) / nt;
      cy = (cy * mt + a.sy[s] * mm) / nt;
      cz = (cz * mt + a.sz[s] * mm) / nt;
      mt = nt;
    }
    a.nmc[k] = make_double4(cx, cy, cz, mt);
    a.live[k] = 0;
    return;
  }
  const int32_t code[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  double x[8], y[8], z[8], m[8];
  uint8_t cl[8];
  // all of the children's loads at once (an empty slot reads its own node's words, unused)
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const bool leaf = code[c] <= -2;
    const int s = leaf ? -2 - code[c] : 0, id = code[c] >= 0 ? code[c] : 0;
    const double *v = reinterpret_cast<const double *>(a.nmc + id);
    x[c] = *(leaf ? a.lcx + s : v);
    y[c] = *(leaf ? a.lcy + s : v + 1);
    z[c] = *(leaf ? a.lcz + s : v + 2);
    m[c] = *(leaf ? a.sm + s : v + 3);
    cl[c] = a.live[id];
  }
  double mt = 0, wx = 0, wy = 0, wz = 0;
  uint32_t live = 0;
#pragma unroll
  for (int c = 0; c < 8; c++) {
    if (code[c] == -1) {
      x[c] = y[c] = z[c] = m[c] = 0.0;
      continue;
    }
    if (code[c] <= -2) m[c] = 0.0 + m[c];
    mt += m[c];
    wx += x[c] * m[c];
    wy += y[c] * m[c];
    wz += z[c] * m[c];
    live |= (m[c] > 0 ? 1u : 0u) << c;
  }
  BhSlot *sl = a.slots + (size_t)k * 8;
#pragma unroll
  for (int c = 0; c < 8; c++) {
    BhSlot o;
    o.x = x[c];
    o.y = y[c];
    o.z = z[c];
    o.m = m[c];
    o.code = code[c];
    o.dep = code[c] >= 0 ? (d + 1 == a.D ? -1 : d + 1) : 0;
    const bool on = (live >> c) & 1;
    o.first = on && o.code >= 0 && o.dep >= 0 && cl[c] ? o.code * 8 + __builtin_ctz(cl[c]) : -1;
    // the next live sibling; the last one's comes from an ancestor, in k_bh_links
    const uint32_t rest = live >> (c + 1);
    o.skip = on && rest ? k * 8 + c + 1 + __builtin_ctz(rest) : -1;
    sl[c] = o;
  }
  a.nmc[k] = make_double4(wx / mt, wy / mt, wz / mt, mt);
  a.live[k] = (uint8_t)live;
}

// Nodes whose run lies within one block of kBhBlock bodies, a workgroup per block, deepest first;
// their numbers are in one range and so is everything below them.  A node that crosses the block's
// end is noted by depth (at most one each) for k_bh_mass_top.  (A launch per depth, 22 of them, was
// 215 us at 262,144 bodies; these two take 42 + 77, at 100,003 35 + 46.  Each is a chain of loads
// and stores per depth: blocks of 512 38 + 115 and 32 + 61, of 2,048 52 + 55 and 50 + 38, but 20
// more at 5,000.)
constexpr int kBhBlock = 1024;
constexpr int kBhBlockNodes = kBhBlock / 2 * (kBhLevels + 1) + kBhLevels + 1;
__global__ __launch_bounds__(256) void k_bh_mass(BhMassArgs a) {
  __shared__ int count[kBhLevels + 2], at[kBhLevels + 2];
  __shared__ uint16_t order[kBhBlockNodes];
  const int M = a.cnt->M, j0 = blockIdx.x * kBhBlock, tid = threadIdx.x;
  if (j0 >= M) return;  // uniform
  const int j1 = min(M, j0 + kBhBlock);
  const int k0 = min(a.first[j0], bh_nodes(a.cnt, a.node_cap));
  const int k1 = min(a.first[j1], bh_nodes(a.cnt, a.node_cap));
  int32_t *cross = a.cross + (size_t)blockIdx.x * (kBhLevels + 1);
  if (tid <= kBhLevels) {
    count[tid] = 0;
    cross[tid] = -1;
  }
  __syncthreads();
  for (int k = k0 + tid; k < k1; k += 256) {
    const int d = a.nstart[k].y;
    if (a.nrange[k].y <= j1) atomicAdd(&count[d], 1);
    else cross[d] = k;
  }
  __syncthreads();
  if (tid == 0) {
    int s = 0;
    for (int d = 0; d <= kBhLevels; d++) {
      at[d] = s;
      s += count[d];
    }
  }
  __syncthreads();
  for (int k = k0 + tid; k < k1; k += 256)
    if (a.nrange[k].y <= j1) order[atomicAdd(&at[a.nstart[k].y], 1)] = (uint16_t)(k - k0);
  __syncthreads();
  for (int d = a.D; d >= 0; d--) {  // at[d] is now the end of depth d's part
    const int n = count[d];
    if (n == 0) continue;  // uniform
    for (int i = tid; i < n; i += 256) bh_mass_node(a, k0 + order[at[d] - n + i], d);
    __syncthreads();
  }
}

__global__ __launch_bounds__(1024) void k_bh_mass_top(BhMassArgs a) {
  __shared__ uint32_t depths;
  const int M = a.cnt->M, nb = min(a.blocks, (M + kBhBlock - 1) / kBhBlock), tid = threadIdx.x;
  if (tid == 0) depths = 0;
  __syncthreads();
  uint32_t has = 0;
  for (int i = tid; i < nb * (kBhLevels + 1); i += 1024)
    if (a.cross[i] >= 0) has |= 1u << (i % (kBhLevels + 1));
  if (has) atomicOr(&depths, has);
  __syncthreads();
  for (int d = a.D; d >= 0; d--) {
    if (!((depths >> d) & 1)) continue;  // uniform
    for (int b = tid; b < nb; b += 1024) {
      const int k = a.cross[(size_t)b * (kBhLevels + 1) + d];
      if (k >= 0) bh_mass_node(a, k, d);
    }
    __syncthreads();
  }
}

// The slot after each node's last live child: the next live sibling of the nearest ancestor that
// has one.  The root's first live child goes to the counters.
__global__ __launch_bounds__(256) void k_bh_links(BhCounters *cnt, const int32_t *pslot,
                                                  const uint8_t *live, int64_t node_cap,
                                                  BhSlot *slots) {
  const int nodes = bh_nodes(cnt, node_cap);
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nodes; k += gridDim.x * blockDim.x) {
    const uint32_t on = live[k];
    if (k == 0) cnt->root_first = on ? __builtin_ctz(on) : -1;
    if (on == 0) continue;
    int skip = -1;
    for (int node = k; node != 0;) {
      const int up = pslot[node];
      node = up >> 3;
      const uint32_t rest = (uint32_t)live[node] >> ((up & 7) + 1);
      if (rest) {
        skip = up + 1 + __builtin_ctz(rest);
        break;
      }
    }
    slots[(size_t)k * 8 + (31 - __builtin_clz(on))].skip = skip;
  }
}

// ---- force -------------------------------------------------------------------------------------
struct BhForceArgs {
  const BhCounters *cnt;
  BhCounters *cnt_w;
  const int32_t *perm;
  const uint64_t *keys;  // sorted keys (fast mode's group cut)
  const uint8_t *flags;
  const double *sx, *sy, *sz, *sm;
  const double4 *nbox, *nmc;
  const int32_t *nchild;
  const BhSlot *slots;
  double *acc;
  int npad;
  int gsz;  // bodies per wave (lanes gsz..63 idle)
  double G, theta, soft2;
  double theta2;  // RN(theta^2) when it is a normal number, else NaN (exact test always)
  int64_t node_cap;
};

// The reference's opening test RN(2 half / RN(sqrt(distSq))) < theta (octree.go:299-306),
// decided from squares where it is clear-cut.  Let a = RN((2h)^2) and b = RN(RN(theta^2)
// distSq), with RN(theta^2) normal (the host passes NaN otherwise) and b in [2^-1000, 2^1000].
// Then each rounding (a when normal, theta^2, b, the margin product) and the square root's is
// within 2^-53 relative, so a < b (1 - 2^-40) gives 2h / dist < theta (1 - 2^-43), below
// theta's predecessor, and a > b (1 + 2^-40) gives 2h / dist > theta (1 + 2^-44), above its
// successor: the rounded quotient lands on the same side of theta as the exact one.  a needs
// no range check: below the normal range its absolute error (2^-1075) is 2^-74 of b, and an
// infinite a exceeds any such b.  Anything else (within 2^-40 of the boundary, b out of range,
// NaN) is left undecided for the reference's own expression.
__device__ __forceinline__ void bh_quick_test(double h2, double distSq, double theta2,
                                              bool &yes, bool &no) {
  const double a = h2 * h2, b = theta2 * distSq;
  const bool normal = b >= 0x1p-1000 && b <= 0x1p1000;
  yes = normal && a < b * (1.0 - 0x1p-40);
  no = normal && a > b * (1.0 + 0x1p-40);
}

// One interaction, op for op as accumForce / directForce (octree.go:292-298, 314-325).
__device__ __forceinline__ void bh_term(double dx, double dy, double dz, double distSq,
                                        double dist, double Gm, double pm, double &fx, double &fy,
                                        double &fz) {
  const double force = Gm * pm / distSq;
  fx += force * dx / dist;
  fy += force * dy / dist;
  fz += force * dz / dist;
}

// The same interaction with the three divisions by dist sharing one reciprocal.  A correctly
// rounded FP64 division n / d compiles to: d' = v_div_scale(d, d, n); y = v_rcp(d'); two Newton
// steps y = fma(y, fma(-d', y, 1), y); n' = v_div_scale(n, d, n); q = n' y; r = fma(-d', q, n');
// q = v_div_fmas(r, y, q); v_div_fixup(q, d, n).  With d in [2^-400, 2^400] and |n| in
// [2^-400, 2^300] both scalings return their operand unchanged and clear VCC (no zero operand, no
// denormal d, 1/d or n/d, exponent gap below 768, n not tiny), v_div_fmas is then a plain fma
// and v_div_fixup returns q with the sign of n / d, which q already has.  So within that range
// the steps that depend on d alone are computed once and each quotient takes three
// instructions, bit-identical to the division; any operand outside it takes the division.
// (The conditions are combined in int, as one lane mask rather than a chain of branches.)
__device__ __forceinline__ int bh_div_range(double n) {
  return (int)(fabs(n) >= 0x1p-400) & (int)(fabs(n) <= 0x1p300);
}

__device__ __forceinline__ void bh_term_shared(double dx, double dy, double dz, double distSq,
                                               double dist, double Gm, double pm, double &fx,
                                               double &fy, double &fz) {
  // the reciprocal does not wait for the numerators: it runs beside the first division
  double y = __builtin_amdgcn_rcp(dist);
  y = __builtin_fma(y, __builtin_fma(-dist, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-dist, y, 1.0), y);
  const double force = Gm * pm / distSq;
  const double nx = force * dx, ny = force * dy, nz = force * dz;
  const int shared = (int)(dist >= 0x1p-400) & (int)(dist <= 0x1p400) & bh_div_range(nx) &
                     bh_div_range(ny) & bh_div_range(nz);
  if (shared) {
    auto quot = [&](double n) {
      const double q = n * y;
      return __builtin_fma(__builtin_fma(-dist, q, n), y, q);
    };
    fx += quot(nx);
    fy += quot(ny);
    fz += quot(nz);
  } else {
    fx += nx / dist;
    fy += ny / dist;
    fz += nz / dist;
  }
}

// The exact walk: one lane per body, bodies in key order.  Each step decides its slot (a leaf
// is taken unless it is the body itself; a node by the opening test from squares, with the
// reference's expression behind a wave-uniform branch only near the boundary), requests the
// next slot and only then computes the taken slot's term, so the term's square root and
// divisions run while the load is in flight.  Terms and their order are the reference's.
// SHARED selects the term with one reciprocal for its three divisions: fewer instructions, a
// longer step (measured on one box: 10.63 against 10.94 ms at N = 262,144, four waves per SIMD;
// 3.31 against 3.14 ms at N = 65,536, one wave per SIMD).
template <bool SHARED>
__global__ __launch_bounds__(256) void k_bh_force(BhForceArgs a) {
  const int M = a.cnt->M;
  if (M < 2) return;  // a lone body feels nothing; forces were zeroed
  __shared__ double h2s[kBhLevels + 1];
  bh_half2_table(a.nbox, h2s);
  const int lane = threadIdx.x & 63;
  const int s = (blockIdx.x * 4 + (int)(threadIdx.x >> 6)) * a.gsz + lane;
  bool act = lane < a.gsz && s < M;
  int i = -1;
  if (act) {
    i = a.perm[s];
    act = !(a.flags[i] & NB_F_SUN);  // suns sum directly
  }
  const unsigned long long nact = __builtin_amdgcn_ballot_w64(act);
  double fx = 0, fy = 0, fz = 0;
  unsigned long long nint = 0;
  if (act) {
    const double xi = a.sx[s], yi = a.sy[s], zi = a.sz[s], Gm = a.G * a.sm[s];
    const double soft2 = a.soft2, theta = a.theta, theta2 = a.theta2;
    const double4 root = a.nmc[0];
    int q = -1;
    if (root.w != 0.0) {  // accumForce: n.totalMass == 0 returns
      const double dx = root.x - xi, dy = root.y - yi, dz = root.z - zi;
      const double distSq = dx * dx + dy * dy + dz * dz + soft2;
      const double dist = __builtin_sqrt(distSq);
      if ((2 * a.nbox[0].w / dist) < theta) {
        bh_term(dx, dy, dz, distSq, dist, Gm, root.w, fx, fy, fz);
        nint++;
      } else {
        const int f = a.cnt->root_first;
        q = f < 0 ? -1 : f;
      }
    }
    int4 w0, w1, w2;
    auto fetch = [&](int slot) {
      const int4 *w = reinterpret_cast<const int4 *>(a.slots + slot);
      w0 = w[0];
      w1 = w[1];
      w2 = w[2];
    };
    // Every step requests a slot, slot 0 (node 0's first slot, always allocated) once the walk is
    // done: an unconditional load lands straight in the registers the next step reads, where a
    // conditional one is copied there and waited for before the term.
    fetch(max(q, 0));
    uint32_t nterm = 0;  // fewer than 2^32: one per visited slot
    while (q >= 0) {
      BhSlot sl;
      __builtin_memcpy(&sl, &w0, 16);
      __builtin_memcpy(reinterpret_cast<char *>(&sl) + 16, &w1, 16);
      __builtin_memcpy(reinterpret_cast<char *>(&sl) + 32, &w2, 16);
      const bool leaf = sl.code <= -2;
      if (!leaf && sl.dep < 0) {  // depth limit: the bucket's bodies one by one (directForce)
        const int32_t *ch = a.nchild + (size_t)sl.code * 8;
        const int b0 = ch[1], bn = ch[2];
        for (int s2 = b0; s2 < b0 + bn; s2++) {
          if (s2 == s) continue;
          const double ex = a.sx[s2] - xi, ey = a.sy[s2] - yi, ez = a.sz[s2] - zi;
          const double d2 = ex * ex + ey * ey + ez * ez + soft2;
          bh_term(ex, ey, ez, d2, __builtin_sqrt(d2), Gm, a.sm[s2], fx, fy, fz);
          nint++;
        }
        q = sl.skip;
        fetch(max(q, 0));
        continue;
      }
      const double dx = sl.x - xi, dy = sl.y - yi, dz = sl.z - zi;
      const double distSq = dx * dx + dy * dy + dz * dz + soft2;
      const double h2 = h2s[leaf ? 0 : sl.dep];
      bool yes, no;
      bh_quick_test(h2, distSq, theta2, yes, no);
      const bool other = -2 - sl.code != s;
      bool take = (leaf & other) | (!leaf & yes);
      const bool und = !leaf & !yes & !no;
      if (__builtin_amdgcn_ballot_w64(und)) {
        __asm__ volatile("");  // a real branch: this division is rare
        if (und) take = (h2 / __builtin_sqrt(distSq)) < theta;
      }
      q = (leaf | take) ? sl.skip : sl.first;
      fetch(max(q, 0));
      if (take) {
        if constexpr (SHARED)
          bh_term_shared(dx, dy, dz, distSq, __builtin_sqrt(distSq), Gm, sl.m, fx, fy, fz);
        else
          bh_term(dx, dy, dz, distSq, __builtin_sqrt(distSq), Gm, sl.m, fx, fy, fz);
        nterm++;
      }
    }
    nint += nterm;
    a.acc[i] = fx;
    a.acc[a.npad + i] = fy;
    a.acc[2 * a.npad + i] = fz;
  }
  if (nact == 0) return;
  for (int o = 32; o > 0; o >>= 1) nint += __shfl_xor(nint, o);
  if (lane == 0) atomicAdd(&a.cnt_w->interactions, nint);
}

// ---- fast mode: one walk per group of bodies, FP32 terms ------------------------------------------
// The 64 bodies of a wave (consecutive in key order) are cut into groups at tree-cell boundaries:
// a run whose smallest enclosing cell holds kBhGroupSpan or more bodies on either side of the run
// is split between that cell's children, and again, until every run lies in a cell of fewer than
// 64 + 2 kBhGroupSpan bodies (or is one body, or one bucket).  Each group shares one traversal.
// Without the cut, a run that straddles two large cells takes a box spanning both and opens
// everything inside it to the leaves (on a Plummer sphere one such wave met 261,464 of the
// 262,144 bodies and set the kernel's duration).  A node is accepted for the whole group when
// 2 half < theta * sqrt(d_box^2 + soft^2), d_box being its centre of mass's distance to the
// group's bounding box: every body of the group is then at least that far away, so each would
// accept it by the reference's own test (octree.go:299-309); otherwise the node is opened.
// A workgroup has the 64 bodies.  Its first wave walks: each step pops up to 8 nodes from an LDS
// stack and the 64 lanes examine their 64 child slots at once; accepted nodes and leaves go to an
// LDS list of terms, opened nodes back to the stack, and the next slots are requested before the
// terms are listed.  The other three waves evaluate the list, 64 terms in a row each, a body per
// lane, like the direct FP32 kernel (sources broadcast from LDS, coordinates relative to the
// group's centre, r^-3 from v_rsq_f32), while the first fills another.  Each 64 terms' sums are
// added into FP64 per lane; the self term is skipped by body index.  The walk is about a quarter of
// the instructions and a chain of dependent loads; terms are 10,000 a body at theta 0.3 and want
// all the issue slots.  One wave doing both, 64 bodies to each, left the longest of four waves a
// SIMD 1.5 times over the mean: 2.35 ms for 262,144 bodies in a Plummer sphere (2.09 with the
// terms' rows pinned and the slots requested ahead) against 1.65 now, and a step of 100,003 bodies
// 1.99 ms against 1.17.  Two evaluating waves 2.55 ms a step of 262,144, three 2.36, four 2.42.
constexpr int kBhGroupSpan = 512;   // see the group cut above
// Stack entries.  The stack stays sorted by depth (each step pops the deepest entries
// and pushes their children on top), so entries of depth d can only be pushed by a step that
// popped every deeper-or-equal entry: at most 64 entries per depth, 21 depths below the root.
constexpr int kBhFastStack = 64 * kBhLevels;
constexpr int kBhFastEval = 3;      // waves of a workgroup that evaluate terms (one lists them)
constexpr int kBhFastOut = 64 * kBhFastEval;        // terms handed over at a time
constexpr int kBhFastList = kBhFastOut + 64;  // < 64 kept + up to 64 added per step

// A list of terms on its way from the listing wave to the others.
struct BhFastSet {
  float4 term[kBhFastList];
  int32_t tidx[kBhFastList];  // body (sorted index) of a leaf term, -1 for a node
  int32_t len, ga, gb, last;  // terms, the group's lanes, whether this is the workgroup's last list
};
struct BhFastLds {
  BhFastSet set[2];
  int32_t stack[kBhFastStack];
};

__device__ __forceinline__ void fast_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// This lane's place among the lanes set in `bal`.
__device__ __forceinline__ int lanes_below(unsigned long long bal) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
}

// Listed terms j .. j + T - 1 against the lane's body.  Four at a time they go row by row with the
// order pinned (neighbouring instructions are then independent, which is what lets gfx950 issue two
// at a time); the sums take them in order.  OWN: one of them may be the body itself.
template <int T, bool OWN>
__device__ __forceinline__ void fast_terms(const BhFastSet &L, int j, float tx, float ty, float tz,
                                           float sf, int s, float &px, float &py, float &pz) {
  float4 e[T];
  float dx[T], dy[T], dz[T], r2[T], inv[T], w[T];
#define NB_T _Pragma("unroll") for (int k = 0; k < T; k++)
  NB_T e[k] = L.term[j + k];
  NB_ROW
  NB_T dx[k] = e[k].x - tx;
  NB_ROW
  NB_T dy[k] = e[k].y - ty;
  NB_ROW
  NB_T r2[k] = __builtin_fmaf(dx[k], dx[k], sf);
  NB_ROW
  NB_T dz[k] = e[k].z - tz;
  NB_ROW
  NB_T r2[k] = __builtin_fmaf(dy[k], dy[k], r2[k]);
  NB_ROW
  NB_T r2[k] = __builtin_fmaf(dz[k], dz[k], r2[k]);
  NB_ROW
  NB_T inv[k] = __builtin_amdgcn_rsqf(r2[k]);
  NB_ROW
  NB_T w[k] = e[k].w * inv[k];
  NB_ROW
  NB_T inv[k] *= inv[k];
  NB_ROW
  NB_T w[k] *= inv[k];
  if (OWN) {
    NB_T w[k] = L.tidx[j + k] == s ? 0.f : w[k];
  }
  NB_T {
    NB_ROW
    px = __builtin_fmaf(dx[k], w[k], px);
    py = __builtin_fmaf(dy[k], w[k], py);
    pz = __builtin_fmaf(dz[k], w[k], pz);
  }
  NB_ROW
#undef NB_T
}

// Listed terms j0 .. j0 + cnt - 1 (64, fewer at a group's end) against the lane's body: one FP32
// partial sum each.
__device__ __forceinline__ void fast_chunk(const BhFastSet &L, int j0, int cnt, float tx, float ty,
                                           float tz, float sf, int s, int g0, int g1, float &px,
                                           float &py, float &pz) {
  const int lane = threadIdx.x & 63;
  const int id = lane < cnt ? L.tidx[j0 + lane] : -1;
  const int c4 = j0 + (cnt & ~3), c1 = j0 + cnt;
  if (__builtin_amdgcn_ballot_w64(id >= g0 && id < g1)) {  // the group's own bodies are rare
    for (int j = j0; j < c4; j += 4) fast_terms<4, true>(L, j, tx, ty, tz, sf, s, px, py, pz);
    for (int j = c4; j < c1; j++) fast_terms<1, true>(L, j, tx, ty, tz, sf, s, px, py, pz);
  } else {
    for (int j = j0; j < c4; j += 4) fast_terms<4, false>(L, j, tx, ty, tz, sf, s, px, py, pz);
    for (int j = c4; j < c1; j++) fast_terms<1, false>(L, j, tx, ty, tz, sf, s, px, py, pz);
  }
}

// The box of the lanes of a group: centre and half extents (FP64), the same on every lane.
struct BhBox {
  double cx, cy, cz, hx, hy, hz;
};
__device__ __forceinline__ BhBox fast_box(bool mine, double px, double py, double pz) {
  double glo[3] = {mine ? px : DBL_MAX, mine ? py : DBL_MAX, mine ? pz : DBL_MAX};
  double ghi[3] = {mine ? px : -DBL_MAX, mine ? py : -DBL_MAX, mine ? pz : -DBL_MAX};
  for (int o = 32; o > 0; o >>= 1)
    for (int d = 0; d < 3; d++) {
      glo[d] = fmin(glo[d], __shfl_xor(glo[d], o));
      ghi[d] = fmax(ghi[d], __shfl_xor(ghi[d], o));
    }
  return BhBox{0.5 * (glo[0] + ghi[0]), 0.5 * (glo[1] + ghi[1]), 0.5 * (glo[2] + ghi[2]),
               0.5 * (ghi[0] - glo[0]), 0.5 * (ghi[1] - glo[1]), 0.5 * (ghi[2] - glo[2])};
}

__global__ __launch_bounds__(64 * (1 + kBhFastEval)) void k_bh_force_fast(BhForceArgs a) {
  __shared__ BhFastLds L;
  __shared__ double h2s[kBhLevels + 1];
  __shared__ double part[kBhFastEval][3][64];
  __shared__ unsigned long long nints[kBhFastEval];
  const int M = a.cnt->M;
  if (M < 2) return;
  bh_half2_table(a.nbox, h2s);
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = blockIdx.x * 64 + lane;
  bool act = s < M;
  int i = -1;
  if (act) {
    i = a.perm[s];
    act = !(a.flags[i] & NB_F_SUN);  // suns sum directly
  }
  if (__builtin_amdgcn_ballot_w64(act) == 0) return;  // the same in all four waves
  const double px = act ? a.sx[s] : 0, py = act ? a.sy[s] : 0, pz = act ? a.sz[s] : 0;
  // the group cut (wave-uniform): bit j of `starts` marks a group starting at lane j
  const int wbase = s - lane, nl = min(64, M - wbase);
  const uint64_t kl = lane < nl ? a.keys[s] : ~0ull;
  const uint64_t kprev = __shfl_up(kl, 1);
  unsigned long long starts = 1ull, fin = 0ull;
  for (;;) {
    const unsigned long long todo = starts & ~fin;
    if (todo == 0) break;
    const int ga = __builtin_ctzll(todo);
    const unsigned long long later = starts & ~((2ull << ga) - 1ull);
    const int gb = later ? __builtin_ctzll(later) : nl;
    const uint64_t ka = __shfl(kl, ga), kb = __shfl(kl, gb - 1);
    const uint64_t x = ka ^ kb;  // live keys use bits 0..62, so x < 2^63
    bool cut = false;
    if (gb - ga > 1 && x != 0) {
      // bits below the run's common prefix: whole octal digits down from the highest difference
      const int lb = 3 * ((63 - __builtin_clzll(x)) / 3 + 1);
      const uint64_t pre = ka >> lb;
      const int pa = wbase + ga - kBhGroupSpan, pb = wbase + gb - 1 + kBhGroupSpan;
      const bool big = (pa >= 0 && (a.keys[pa] >> lb) == pre) ||
                       (pb < M && (a.keys[pb] >> lb) == pre);
      if (big) {
        // cut where the next digit changes: the run's parts in the cell's children
        starts |= __builtin_amdgcn_ballot_w64(lane > ga && lane < gb &&
                                              ((kl ^ kprev) >> (lb - 3)) != 0);
        cut = true;
      }
    }
    if (!cut) fin |= 1ull << ga;
  }
  if (wv > 0) {  // evaluates the listed terms: 64 in a row to each of these waves in turn
    double ax = 0, ay = 0, az = 0;
    unsigned long long nint = 0;
    float tx = 0.f, ty = 0.f, tz = 0.f;
    bool mine = false;
    const float sf = to_vgpr((float)a.soft2);
    int ga = -1;
    for (int set = 0;; set ^= 1) {
      __syncthreads();
      const BhFastSet &S = L.set[set];
      const int len = S.len;
      if (len > 0) {
        const int gb = S.gb;
        if (S.ga != ga) {  // another group: its bodies about its box's centre
          ga = S.ga;
          mine = act && lane >= ga && lane < gb;
          const BhBox bx = fast_box(mine, px, py, pz);
          tx = (float)(px - bx.cx);
          ty = (float)(py - bx.cy);
          tz = (float)(pz - bx.cz);
        }
        for (int j0 = (wv - 1) * 64; j0 < len; j0 += 64 * kBhFastEval) {
          const int cnt = min(64, len - j0);
          float qx = 0.f, qy = 0.f, qz = 0.f;
          fast_chunk(S, j0, cnt, tx, ty, tz, sf, s, wbase + ga, wbase + gb, qx, qy, qz);
          if (mine) {
            ax += qx;
            ay += qy;
            az += qz;
            nint += (unsigned long long)cnt;
          }
        }
      }
      if (S.last) break;
    }
    part[wv - 1][0][lane] = ax;
    part[wv - 1][1][lane] = ay;
    part[wv - 1][2][lane] = az;
    for (int o = 32; o > 0; o >>= 1) nint += __shfl_xor(nint, o);
    if (lane == 0) nints[wv - 1] = nint;
    __syncthreads();
    return;
  }
  // the first wave walks the tree and lists the terms; the others wait for it
  const double th2 = a.theta * a.theta, soft2 = a.soft2;
  bool overflow = false;
  const int node_lim = (int)min(a.node_cap, (int64_t)INT32_MAX / 8);
  int set = 0, len = 0;  // the list being filled and its length
  int ga = 0, gb = 0;
  // The list goes to the evaluating waves, all of it at a group's end, else the whole rounds of 64;
  // what is left starts the other list.
  auto hand_over = [&](bool end, bool last) {
    BhFastSet &S = L.set[set], &N = L.set[set ^ 1];
    const int out = end ? len : kBhFastOut, rest = len - out;
    float4 mv = make_float4(0.f, 0.f, 0.f, 0.f);
    int mi = -1;
    if (lane < rest) {
      mv = S.term[out + lane];
      mi = S.tidx[out + lane];
    }
    if (lane == 0) {
      S.len = out;
      S.ga = ga;
      S.gb = gb;
      S.last = last;
    }
    __syncthreads();  // the others are done with the other list and start on this one
    if (lane < rest) {
      N.term[lane] = mv;
      N.tidx[lane] = mi;
    }
    set ^= 1;
    len = rest;
  };
  // One term per lane that has one, in lane order.
  auto append = [&](bool has, float4 t, int id) {
    const unsigned long long bal = __builtin_amdgcn_ballot_w64(has);
    if (has) {
      const int pos = len + lanes_below(bal);
      L.set[set].term[pos] = t;
      L.set[set].tidx[pos] = id;
    }
    len += __builtin_popcountll(bal);
    if (len >= kBhFastOut) hand_over(false, false);
  };
  for (unsigned long long segs = starts; segs;) {
    ga = __builtin_ctzll(segs);
    segs &= segs - 1;
    gb = segs ? __builtin_ctzll(segs) : nl;
    const bool mine = act && lane >= ga && lane < gb;
    if (__builtin_amdgcn_ballot_w64(mine) == 0) continue;
    const BhBox bx = fast_box(mine, px, py, pz);
    // a node accepted for the group: (2 half)^2 < theta^2 (d_box^2 + soft^2)
    auto accept = [&](double x, double y, double z, double half) {
      const double ex = fmax(fabs(x - bx.cx) - bx.hx, 0.0), ey = fmax(fabs(y - bx.cy) - bx.hy, 0.0),
                   ez = fmax(fabs(z - bx.cz) - bx.hz, 0.0);
      return 4.0 * half * half < th2 * (ex * ex + ey * ey + ez * ez + soft2);
    };
    int top = 0;
    const double4 root = a.nmc[0];
    if (root.w != 0.0) {
      if (accept(root.x, root.y, root.z, a.nbox[0].w)) {
        append(lane == 0, make_float4((float)(root.x - bx.cx), (float)(root.y - bx.cy),
                                      (float)(root.z - bx.cz), (float)root.w), -1);
      } else {
        if (lane == 0) L.stack[0] = 0;
        top = 1;
      }
    }
    // Pops up to 8 nodes and requests their child slots, one per lane.
    BhSlot sl;
    bool have = false;
    auto pop = [&]() {
      fast_sync();
      const int nn = min(8, top), k = lane >> 3;
      const int node = k < nn ? L.stack[top - nn + k] : -1;
      have = node >= 0 && node < node_lim;
      if (have) sl = a.slots[(size_t)node * 8 + (lane & 7)];
      top -= nn;
      fast_sync();
    };
    bool more = top > 0;
    if (more) pop();
    while (more) {
      bool term = false, open = false, bucket = false;
      float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
      int id = -1, code = -1;
      if (have) {
        code = sl.code;
        if (code != -1 && sl.m > 0) {
          if (code <= -2) {  // a leaf: the body's own centre of mass (x*m)/m and mass 0 + m
            term = true;
            id = -2 - code;
          } else if (sl.dep < 0) {
            bucket = code < node_lim;
          } else if (accept(sl.x, sl.y, sl.z, 0.5 * h2s[sl.dep])) {
            term = true;
          } else {
            open = code < node_lim;
          }
          if (term)
            t = make_float4((float)(sl.x - bx.cx), (float)(sl.y - bx.cy), (float)(sl.z - bx.cz),
                            (float)sl.m);
        }
      }
      // opened nodes onto the stack, and the next slots requested before the terms are listed
      const unsigned long long bo = __builtin_amdgcn_ballot_w64(open);
      const int nopen = __builtin_popcountll(bo);
      if (top + nopen > kBhFastStack) {
        overflow = true;
        break;
      }
      if (open) L.stack[top + lanes_below(bo)] = code;
      top += nopen;
      more = top > 0;
      if (more) pop();
      append(term, t, id);
      // buckets (the depth limit): their bodies one by one, 64 at a time
      unsigned long long bb = __builtin_amdgcn_ballot_w64(bucket);
      while (bb) {
        const int src = __builtin_ctzll(bb);
        bb &= bb - 1;
        const int bnode = __shfl(code, src);
        const int32_t *ch = a.nchild + (size_t)bnode * 8;
        const int b0 = ch[1], bn = ch[2];
        for (int q0 = 0; q0 < bn; q0 += 64) {
          const int q = b0 + q0 + lane;
          const bool h = q0 + lane < bn;
          float4 e = make_float4(0.f, 0.f, 0.f, 0.f);
          if (h)
            e = make_float4((float)(a.sx[q] - bx.cx), (float)(a.sy[q] - bx.cy),
                            (float)(a.sz[q] - bx.cz), (float)a.sm[q]);
          append(h, e, q);
        }
      }
    }
    hand_over(true, false);
  }
  hand_over(true, true);  // (empty)
  if (overflow && lane == 0) atomicOr(&a.cnt_w->stack_overflow, 1u);
  __syncthreads();
  if (lane == 0) {
    unsigned long long nint = 0;
    for (int v = 0; v < kBhFastEval; v++) nint += nints[v];
    atomicAdd(&a.cnt_w->interactions, nint);
  }
  if (act) {  // the evaluating waves' sums in wave order
    double f[3];
    for (int q = 0; q < 3; q++) {
      f[q] = part[0][q][lane];
      for (int v = 1; v < kBhFastEval; v++) f[q] += part[v][q][lane];
    }
    const double Gm = a.G * a.sm[s];
    a.acc[i] = Gm * f[0];
    a.acc[a.npad + i] = Gm * f[1];
    a.acc[2 * a.npad + i] = Gm * f[2];
  }
}

// Suns: directForce from every other existing, non-fragmenting body in array order.
__global__ __launch_bounds__(256) void k_bh_sun_list(const uint8_t *flags, int n, BhCounters *cnt,
                                                     int32_t *suns) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && bh_active(flags[i]) && (flags[i] & NB_F_SUN)) suns[atomicAdd(&cnt->nsun, 1u)] = i;
}

struct BhSunArgs {
  BhCounters *cnt;
  const int32_t *suns;
  const double *x, *y, *z, *m;
  const uint8_t *flags;
  double *acc;
  int n, npad;
  double G, soft2;
};

__global__ __launch_bounds__(64) void k_bh_sun(BhSunArgs a) {
  __shared__ double t[3][kSunChunk];
  __shared__ int valid[kSunChunk];
  if (a.cnt->M < 2) return;
  const int lane = threadIdx.x;
  const int nsun = (int)a.cnt->nsun;
  for (int k = blockIdx.x; k < nsun; k += gridDim.x) {
    const int b = a.suns[k];
    const double xb = a.x[b], yb = a.y[b], zb = a.z[b], Gm = a.G * a.m[b];
    double sum = 0;  // lane c < 3 accumulates component c
    unsigned long long nint = 0;
    for (int j0 = 0; j0 < a.n; j0 += kSunChunk) {
      const int j = j0 + lane;
      const bool v = j < a.n && j != b && bh_active(a.flags[j]);
      double tx = 0, ty = 0, tz = 0;
      if (v) {
        const double dx = a.x[j] - xb;
        const double dy = a.y[j] - yb;
        const double dz = a.z[j] - zb;
        const double distSq = dx * dx + dy * dy + dz * dz + a.soft2;
        const double dist = __builtin_sqrt(distSq);
        const double force = Gm * a.m[j] / distSq;
        tx = force * dx / dist;
        ty = force * dy / dist;
        tz = force * dz / dist;
        nint++;
      }
      t[0][lane] = tx;
      t[1][lane] = ty;
      t[2][lane] = tz;
      valid[lane] = v ? 1 : 0;
      bh_wave_sync();
      if (lane < 3)
        for (int q = 0; q < kSunChunk; q++)
          if (valid[q]) sum += t[lane][q];
      bh_wave_sync();
    }
    if (lane < 3) a.acc[(size_t)lane * a.npad + b] = sum;
    for (int o = 32; o > 0; o >>= 1) nint += __shfl_xor(nint, o);
    if (lane == 0) atomicAdd(&a.cnt->interactions, nint);
  }
}

// ---- collision pairs ---------------------------------------------------------------------------
struct BhDetectArgs {
  const BhCounters *cnt;
  const int32_t *perm;
  const double *x, *y, *z, *r;
  const int32_t *beh;
  const double4 *nbox;
  const int32_t *nchild;
  uint64_t *pairs;
  DevCounters *ctr;
  int64_t pair_cap;
  double rmax;
  int events;
};

__device__ __forceinline__ void bh_emit(const BhDetectArgs &a, int i, int j) {
  const uint32_t q = atomicAdd(&a.ctr->pair_count, 1u);
  if ((int64_t)q < a.pair_cap)
    a.pairs[q] = ((uint64_t)(uint32_t)i << 32) | (uint32_t)j;
  else
    atomicOr(&a.ctr->pair_overflow, 1u);
}

// Collided (body.go:192-208) from body i's side, pairs i < j, dispatched as Compute does.
__device__ __forceinline__ void bh_test_pair(const BhDetectArgs &a, int i, int32_t bi, double xi,
                                             double yi, double zi, double ri, int s2) {
  const int j = a.perm[s2];
  if (j <= i) return;
  const double dx = a.x[j] - xi;
  const double dy = a.y[j] - yi;
  const double dz = a.z[j] - zi;
  const double dist = __builtin_sqrt(dx * dx + dy * dy + dz * dz);
  const double rj = a.r[j];
  if (dist <= ri + rj && nb_pair_event(bi, a.beh[j], ri, rj, dist, a.events)) bh_emit(a, i, j);
}

__global__ __launch_bounds__(256) void k_bh_detect(BhDetectArgs a) {
  __shared__ int32_t stk_code[4][kBhStack];
  __shared__ unsigned long long stk_mask[4][kBhStack];
  const int M = a.cnt->M;
  if (M < 2) return;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  int i = -1;
  bool act = false;
  int32_t bi = NB_CB_NONE;
  double xi = 0, yi = 0, zi = 0, ri = 0, lim = 0;
  if (s < M) {
    i = a.perm[s];
    bi = a.beh[i];
    act = nb_may_pair(bi, a.events);
    xi = a.x[i];
    yi = a.y[i];
    zi = a.z[i];
    ri = a.r[i];
    // a box farther than R_i + R_max holds no partner; the slack covers the box test's rounding
    const double reach = ri + a.rmax;
    lim = reach + 1e-12 * (fabs(xi) + fabs(yi) + fabs(zi) + reach) + 1e-300;
  }
  const unsigned long long start = __builtin_amdgcn_ballot_w64(act);
  if (start == 0) return;
  if (lane == 0) {
    stk_code[w][0] = 0;
    stk_mask[w][0] = start;
  }
  int sp = 1;
  bh_wave_sync();
  while (sp > 0) {
    sp--;
    const int code = __builtin_amdgcn_readfirstlane(stk_code[w][sp]);
    const unsigned long long msk = stk_mask[w][sp];
    const bool on = (msk >> lane) & 1ull;
    if (code <= -2) {
      if (on) bh_test_pair(a, i, bi, xi, yi, zi, ri, -2 - code);
      continue;
    }
    const int32_t *ch = a.nchild + (size_t)code * 8;
    if (ch[0] == kBucket) {
      if (on)
        for (int s2 = ch[1]; s2 < ch[1] + ch[2]; s2++)
          if (s2 != s) bh_test_pair(a, i, bi, xi, yi, zi, ri, s2);
      continue;
    }
    const double4 bx = a.nbox[code];
    bool pass = false;
    if (on) {
      const double ex = fmax(fabs(xi - bx.x) - bx.w, 0.0);
      const double ey = fmax(fabs(yi - bx.y) - bx.w, 0.0);
      const double ez = fmax(fabs(zi - bx.z) - bx.w, 0.0);
      const double slack = 1e-12 * (fabs(bx.x) + fabs(bx.y) + fabs(bx.z) + bx.w);
      const double l = lim + slack;
      pass = ex * ex + ey * ey + ez * ez <= l * l;
    }
    const unsigned long long pm = __builtin_amdgcn_ballot_w64(pass);
    if (pm && sp + 8 <= kBhStack) {
      for (int c = 7; c >= 0; c--) {
        const int32_t cc = ch[c];
        if (cc == -1) continue;
        if (lane == 0) {
          stk_code[w][sp] = cc;
          stk_mask[w][sp] = pm;
        }
        sp++;
      }
    }
    bh_wave_sync();
  }
}

__global__ void k_bh_zero(double *acc, size_t len) {
  for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < len;
       k += (size_t)gridDim.x * blockDim.x)
    acc[k] = 0.0;
}

// ---- host --------------------------------------------------------------------------------------
static int nb256(int64_t n) { return (int)std::max<int64_t>(1, (n + 255) / 256); }

void bh_free(Bh *b) {
  if (!b) return;
  void *ps[] = {b->keys_in, b->keys, b->perm_in, b->perm, b->sx,     b->sy,     b->sz,
                b->sm,      b->lcx,  b->lcy,     b->lcz,  b->depth,  b->suns,   b->nbox,
                b->nmc,     b->nchild, b->nrange, b->bpart, b->sort_tmp, b->cnt, b->slots,
                b->pslot, b->nstart, b->first, b->npart, b->cross, b->live};
  for (void *p : ps)
    if (p) (void)hipFree(p);
  delete b;
}

static int bh_ensure(Ctx *c) {
  Bh *b = c->bh;
  if (!b->cnt) {
    NB_HIP(c, hipMalloc((void **)&b->cnt, sizeof(BhCounters)));
    NB_HIP(c, hipMemset(b->cnt, 0, sizeof(BhCounters)));
    NB_HIP(c, balloc(&b->bpart, 1024 * 8));
  }
  if (b->cap >= c->cap) return NB_OK;
  const size_t n = (size_t)c->cap;
  NB_HIP(c, balloc(&b->keys_in, n));
  NB_HIP(c, balloc(&b->keys, n));
  NB_HIP(c, balloc(&b->perm_in, n));
  NB_HIP(c, balloc(&b->perm, n));
  NB_HIP(c, balloc(&b->sx, n));
  NB_HIP(c, balloc(&b->sy, n));
  NB_HIP(c, balloc(&b->sz, n));
  NB_HIP(c, balloc(&b->sm, n));
  NB_HIP(c, balloc(&b->lcx, n));
  NB_HIP(c, balloc(&b->lcy, n));
  NB_HIP(c, balloc(&b->lcz, n));
  NB_HIP(c, balloc(&b->depth, n));
  NB_HIP(c, balloc(&b->suns, n));
  // every node holds 2+ bodies and the nodes of one level are disjoint: at most n/2 per level
  b->node_cap = (int64_t)(n / 2) * kBhLevels + 64;
  NB_HIP(c, balloc(&b->nbox, (size_t)b->node_cap));
  NB_HIP(c, balloc(&b->nmc, (size_t)b->node_cap));
  NB_HIP(c, balloc(&b->nchild, (size_t)b->node_cap * 8));
  NB_HIP(c, balloc(&b->slots, (size_t)b->node_cap * 8));
  NB_HIP(c, balloc(&b->pslot, (size_t)b->node_cap));
  NB_HIP(c, balloc(&b->nrange, (size_t)b->node_cap));
  NB_HIP(c, balloc(&b->nstart, (size_t)b->node_cap));
  NB_HIP(c, balloc(&b->live, (size_t)b->node_cap));
  NB_HIP(c, balloc(&b->first, n + 1));
  NB_HIP(c, balloc(&b->npart, (n + kBhRun - 1) / kBhRun));
  NB_HIP(c, balloc(&b->cross, (n + kBhBlock - 1) / kBhBlock * (kBhLevels + 1)));
  size_t bytes = 0;
  NB_HIP(c, rocprim::radix_sort_pairs(nullptr, bytes, b->keys_in, b->keys, b->perm_in, b->perm,
                                      n, 0, 64, c->stream));
  void *tmp = nullptr;
  NB_HIP(c, hipMalloc(&tmp, bytes ? bytes : 1));
  if (b->sort_tmp) (void)hipFree(b->sort_tmp);
  b->sort_tmp = tmp;
  b->sort_bytes = bytes;
  b->cap = c->cap;
  return NB_OK;
}

int bh_force_phase(Ctx *c, bool timed, int ev_slot) {
  Bh *b = c->bh;
  hipStream_t st = c->stream;
  NB_HIP(c, launch_zero_counters(c->ctr, 0, st));
  int rc = bh_ensure(c);
  if (rc) return rc;
  const int n = (int)c->n;
  const int D = b->p.max_depth;
  const size_t acc_len = (size_t)3 * c->npad;
  hipLaunchKernelGGL(k_bh_zero, dim3(nb256((int64_t)std::min<size_t>(acc_len, 1 << 20))),
                     dim3(256), 0, st, c->acc, acc_len);
  if (n == 0) return NB_OK;
  const int nparts = std::min(1024, nb256(n));
  hipLaunchKernelGGL(k_bh_box_part, dim3(nparts), dim3(256), 0, st, c->x, c->y, c->z, c->flags,
                     n, b->bpart);
  hipLaunchKernelGGL(k_bh_root, dim3(1), dim3(256), 0, st, b->bpart, nparts, b->cnt, b->nbox,
                     b->nchild);
  hipLaunchKernelGGL(k_bh_keys, dim3(nb256(n)), dim3(256), 0, st, c->x, c->y, c->z, c->flags, n,
                     b->nbox, D, b->keys_in, b->perm_in, b->depth);
  NB_HIP(c, hipGetLastError());
  size_t bytes = b->sort_bytes;
  NB_HIP(c, rocprim::radix_sort_pairs(b->sort_tmp, bytes, b->keys_in, b->keys, b->perm_in,
                                      b->perm, (size_t)n, 0, 64, st));
  hipLaunchKernelGGL(k_bh_gather, dim3(nb256(n)), dim3(256), 0, st, b->perm, c->x, c->y, c->z,
                     c->m, b->cnt, b->sx, b->sy, b->sz, b->sm, b->lcx, b->lcy, b->lcz);
  const unsigned runs = (unsigned)((n + kBhRun - 1) / kBhRun);
  hipLaunchKernelGGL(k_bh_count, dim3(runs), dim3(256), 0, st, b->keys, b->perm, D, b->cnt,
                     b->npart, b->depth);
  hipLaunchKernelGGL(k_bh_starts, dim3(runs), dim3(256), 0, st, b->keys, D, b->cnt, b->npart,
                     b->node_cap, b->first, b->nstart);
  BhNodeArgs na;
  na.keys = b->keys;
  na.cnt = b->cnt;
  na.first = b->first;
  na.nstart = b->nstart;
  na.nbox = b->nbox;
  na.nrange = b->nrange;
  na.nchild = b->nchild;
  na.pslot = b->pslot;
  na.node_cap = b->node_cap;
  na.D = D;
  // about half as many nodes as bodies: eight lanes for each
  hipLaunchKernelGGL(k_bh_nodes, dim3(nb256((int64_t)std::max(1, n / 2) * 8)), dim3(256), 0, st,
                     na);
  BhMassArgs ma;
  ma.cnt = b->cnt;
  ma.nchild = b->nchild;
  ma.first = b->first;
  ma.nstart = b->nstart;
  ma.nrange = b->nrange;
  ma.nmc = b->nmc;
  ma.slots = b->slots;
  ma.live = b->live;
  ma.cross = b->cross;
  ma.sx = b->sx; ma.sy = b->sy; ma.sz = b->sz; ma.sm = b->sm;
  ma.lcx = b->lcx; ma.lcy = b->lcy; ma.lcz = b->lcz;
  ma.node_cap = b->node_cap;
  ma.D = D;
  ma.blocks = (n + kBhBlock - 1) / kBhBlock;
  hipLaunchKernelGGL(k_bh_mass, dim3((unsigned)ma.blocks), dim3(256), 0, st, ma);
  hipLaunchKernelGGL(k_bh_mass_top, dim3(1), dim3(1024), 0, st, ma);
  hipLaunchKernelGGL(k_bh_links, dim3(nb256(n)), dim3(256), 0, st, b->cnt, b->pslot,
                     b->live, b->node_cap, b->slots);
  NB_HIP(c, hipGetLastError());
  BhForceArgs fa;
  fa.cnt = b->cnt;
  fa.cnt_w = b->cnt;
  fa.perm = b->perm;
  fa.keys = b->keys;
  fa.flags = c->flags;
  fa.sx = b->sx; fa.sy = b->sy; fa.sz = b->sz; fa.sm = b->sm;
  fa.nbox = b->nbox;
  fa.nmc = b->nmc;
  fa.nchild = b->nchild;
  fa.slots = b->slots;
  // 64 bodies per wave unless asked: smaller groups only repeat the shared part of the walk in
  // more waves (measured 6.9 / 8.4 / 10.7 ms at N = 65,536 for 64 / 32 / 16)
  fa.gsz = b->p.group ? b->p.group : 64;
  fa.node_cap = b->node_cap;
  fa.acc = c->acc;
  fa.npad = (int)c->npad;
  fa.G = c->p.G;
  fa.theta = b->p.theta;
  {
    const double t2 = b->p.theta * b->p.theta;
    fa.theta2 = (t2 >= 0x1p-1000 && t2 <= 0x1p1000) ? t2 : std::nan("");
  }
  fa.soft2 = b->p.softening * b->p.softening;
  if (timed) NB_HIP(c, hipEventRecord(c->ev[2 * ev_slot], st));
  if (b->p.mode == 1)
    hipLaunchKernelGGL(k_bh_force_fast, dim3((unsigned)((n + 63) / 64)),
                       dim3(64 * (1 + kBhFastEval)), 0, st, fa);
  else {
    // by default the shared-reciprocal term once the walk has four waves per SIMD (issue-bound)
    const int64_t waves = (n + fa.gsz - 1) / fa.gsz;
    const bool shared = b->p.term == 2 || (b->p.term == 0 && waves >= (int64_t)4 * 4 * b->cus);
    hipLaunchKernelGGL(shared ? k_bh_force<true> : k_bh_force<false>,
                       dim3((unsigned)((n + 4 * fa.gsz - 1) / (4 * fa.gsz))), dim3(256), 0, st,
                       fa);
  }
  hipLaunchKernelGGL(k_bh_sun_list, dim3(nb256(n)), dim3(256), 0, st, c->flags, n, b->cnt,
                     b->suns);
  BhSunArgs sa;
  sa.cnt = b->cnt;
  sa.suns = b->suns;
  sa.x = c->x; sa.y = c->y; sa.z = c->z; sa.m = c->m;
  sa.flags = c->flags;
  sa.acc = c->acc;
  sa.n = n;
  sa.npad = (int)c->npad;
  sa.G = c->p.G;
  sa.soft2 = fa.soft2;
  hipLaunchKernelGGL(k_bh_sun, dim3(64), dim3(64), 0, st, sa);
  if (timed) NB_HIP(c, hipEventRecord(c->ev[2 * ev_slot + 1], st));
  NB_HIP(c, hipGetLastError());
  if (c->p.collisions) {
    BhDetectArgs da;
    da.cnt = b->cnt;
    da.perm = b->perm;
    da.x = c->x; da.y = c->y; da.z = c->z; da.r = c->r;
    da.beh = c->beh;
    da.nbox = b->nbox;
    da.nchild = b->nchild;
    da.pairs = c->pairs;
    da.ctr = c->ctr;
    da.pair_cap = c->pair_cap;
    da.rmax = c->rmax;
    da.events = c->p.events;
    hipLaunchKernelGGL(k_bh_detect, dim3(nb256(n)), dim3(256), 0, st, da);
    NB_HIP(c, hipGetLastError());
  }
  b->builds++;
  return NB_OK;
}

}  // namespace nb

using namespace nb;

extern "C" {

int nb_bh_params_init(nb_bh_params *p) {
  if (!p) return NB_E_INVALID;
  memset(p, 0, sizeof *p);
  p->theta = 0.3;
  p->softening = 1e-4;
  p->max_depth = kBhLevels;
  return NB_OK;
}

int nb_bh_enable(nb_ctx *c, const nb_bh_params *p) {
  if (!c) return NB_E_INVALID;
  nb_bh_params q;
  if (p)
    q = *p;
  else
    nb_bh_params_init(&q);
  if (!(q.theta >= 0) || !std::isfinite(q.theta) || !(q.softening >= 0) ||
      !std::isfinite(q.softening) || q.max_depth < 1 || q.max_depth > kBhLevels ||
      !(q.group == 0 || q.group == 16 || q.group == 32 || q.group == 64) ||
      (q.mode != 0 && q.mode != 1) || q.term < 0 || q.term > 2)
    return fail_msg(c, NB_E_INVALID,
                    "nb_bh_enable: theta, softening >= 0, max_depth in [1, 21], group 0/16/32/64, "
                    "mode 0/1, term 0/1/2");
  if (c->p.precision != NB_PREC_FP64)
    return fail_msg(c, NB_E_UNSUPPORTED, "nb_bh_enable: the octree path is FP64 (precision fp64)");
  if (c->sur_on)
    return fail_msg(c, NB_E_UNSUPPORTED, "nb_bh_enable: the surrogate is on; disable it first");
  NB_HIP(c, hipSetDevice(c->device));
  if (!c->bh) {
    c->bh = new Bh();
    NB_HIP(c, hipDeviceGetAttribute(&c->bh->cus, hipDeviceAttributeMultiprocessorCount,
                                    c->device));
  }
  c->bh->p = q;
  c->bh_on = true;
  return NB_OK;
}

int nb_bh_disable(nb_ctx *c) {
  if (!c) return NB_E_INVALID;
  c->bh_on = false;
  return NB_OK;
}

int nb_bh_get_stats(nb_ctx *c, nb_bh_stats *out) {
  if (!c || !out) return NB_E_INVALID;
  memset(out, 0, sizeof *out);
  if (!c->bh || !c->bh->cnt) return NB_OK;
  NB_HIP(c, hipSetDevice(c->device));
  BhCounters h;
  NB_HIP(c, hipStreamSynchronize(c->stream));
  NB_HIP(c, hipMemcpy(&h, c->bh->cnt, sizeof h, hipMemcpyDeviceToHost));
  out->builds = c->bh->builds;
  out->bodies = h.M;
  out->nodes = h.nodes;
  out->buckets = h.buckets;
  out->interactions = (int64_t)h.interactions;
  out->depth_max = h.depth_max;
  out->overflow = (int32_t)(h.stack_overflow | h.node_overflow);
  return NB_OK;
}

int nb_bh_get_depths(nb_ctx *c, int32_t *depth) {
  if (!c || !depth) return NB_E_INVALID;
  if (!c->bh || !c->bh->depth || c->bh->builds == 0)
    return fail_msg(c, NB_E_STATE, "nb_bh_get_depths: no tree built yet");
  if (c->n == 0) return NB_OK;
  NB_HIP(c, hipSetDevice(c->device));
  NB_HIP(c, hipMemcpyAsync(depth, c->bh->depth, (size_t)c->n * sizeof(int32_t),
                           hipMemcpyDeviceToHost, c->stream));
  NB_HIP(c, hipStreamSynchronize(c->stream));
  return NB_OK;
}

}  // extern "C"
