// Broadphase: Verlet-skin refresh test, spatial re-sort of the particle
// storage by counting per cell, pair generation over the cells, and the merge
// that carries contact history across refreshes. Replaces
// InsertionSortCollider::run (InsertionSortCollider.cpp:386-613).
//
// Pair-set semantics kept from the reference:
//  * AABB of a sphere = centre -/+ (r*distFactor') -/+ verletDist, of a wall =
//    infinite except along its axis (Sphere.cpp:52-82, Wall.cpp:25-38,
//    Collision.cpp:125-162);
//  * refresh when any particle moved more than verletDist since the last one
//    (Collision.cpp:80-123);
//  * potential set after a refresh = {pairs whose enlarged AABBs overlap and that
//    mayCollide} U {real contacts}; a broken contact whose AABBs did not overlap
//    is dropped (InsertionSortCollider.hpp:213-218).
// The step kernels only need the pairs that can touch before the next refresh:
// the slots hold the AABB pairs whose centres are within r1+r2+2*verletDist
// (each particle moves at most verletDist until then), plus carried real
// contacts. The full potential set is regenerated on request (potential_pairs).
//
// Refresh: spheres are re-sorted by cell (storage order) and the particle arrays
// permuted; each sphere generates its pairs with the spheres after it over the 27
// neighbour cells (one pass, staged per sphere, then laid out in storage order);
// each old real contact finds its pair among the few generated by its lower
// sphere, or is appended, so that its history is carried; finally every
// particle's adjacency list is sorted by the other particle's user id, the
// canonical summation order.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <vector>

#include "wdg_internal.hpp"
#include "wdg_math.hpp"

namespace wdg {

// the cell grid of one scene of a batched context, over that scene's bounding box with cells
// as large as its own largest enlarged AABB; its cells are keys off .. off + nc0 nc1 nc2 - 1
struct SceneGrid {
  double org[3];
  double h;
  int nc[3];
  uint32_t off;
};
struct Grid {
  double org[3];
  double h[3];
  int nc[3];
  int periodic;
  double L[3];
  // sparse aperiodic scenes (a dense grid of the bounding box would need far more cells than
  // spheres): the key of a cell is a hash of its coordinates into hmask + 1 buckets, so the
  // cells keep their size however far the spheres spread
  int hashed;
  uint32_t hmask;
  // batched aperiodic scenes: one grid per scene (null: the grid above); the spheres are then
  // stored scene by scene
  const SceneGrid* sg;
  // dense grid whose keys are the Morton codes of the cells (coordinates' bits interleaved),
  // so that storage order keeps neighbouring cells near each other in all three directions
  int morton;
};

struct AabbParams {
  double vd;      // verletDist (absolute)
  double absDf;   // |distFactor|
  uint32_t loneMask;
  int periodic;
  double L[3];
};

// ------------------------------------------------------------------ helpers
__device__ __forceinline__ bool may_collide(uint32_t ma, uint32_t mb, uint32_t lone) {
  return (ma & mb) != 0u && (ma & mb & lone) == 0u;
}
// sphere AABB bounds along one axis, same operations as updateAabb
__device__ __forceinline__ void sph_bounds(double p, double hs, double vd, double& lo, double& hi) {
  lo = p - hs;
  hi = p + hs;
  if (vd > 0) {
    hi = hi + vd;
    lo = lo - vd;
  }
}
// nearest periodic image of B relative to A, from refresh positions
__device__ __forceinline__ int near_img(double pa, double pb, double L) {
  double d = (pb - pa) / L;
  return -(int)floor(d + 0.5);
}
// AABB overlap of spheres a (pA) and b (pB) with b shifted by cd; counts overlapping images when periodic
__device__ __forceinline__ bool sph_overlap(const double pa[3], double hsa, const double pb[3], double hsb,
                                            const AabbParams& P, double vd, int cd[3], int& nimg) {
  bool ok = true;
  nimg = 1;
  for (int k = 0; k < 3; k++) {
    double alo, ahi, blo, bhi;
    sph_bounds(pa[k], hsa, vd, alo, ahi);
    sph_bounds(pb[k], hsb, vd, blo, bhi);
    if (P.periodic) {
      cd[k] = near_img(pa[k], pb[k], P.L[k]);
      double s = P.L[k] * cd[k];
      if (!(alo <= bhi + s && ahi >= blo + s)) ok = false;
      int cnt = 0;
      for (int dd = -1; dd <= 1; dd++) {
        double s2 = P.L[k] * (cd[k] + dd);
        if (alo <= bhi + s2 && ahi >= blo + s2) cnt++;
      }
      nimg *= cnt;
    } else {
      cd[k] = 0;
      if (!(alo <= bhi + 0. && ahi >= blo + 0.)) ok = false;
    }
  }
  return ok;
}

// ------------------------------------------------------------------ refresh test
// the Verlet distance of particle i: its scene's (batched scenes with per-scene skins) or the
// context's
__device__ __forceinline__ double vd_at(const double* vdS, const uint32_t* scene, int64_t i, double vd) {
  return vdS ? vdS[scene[i]] : vd;
}
// largest squared speed of every scene's spheres (non-negative doubles order as their bits):
// a workgroup takes the maximum per scene in LDS first (its spheres belong to a few scenes),
// then makes one global atomic per scene it saw; beyond SV_LDS scenes straight to HBM
constexpr int SV_LDS = 1024;
__global__ __launch_bounds__(256) void k_scene_vmax(int64_t nW, int64_t n, int64_t nScenes,
                                                    const double* __restrict__ vx, const double* __restrict__ vy,
                                                    const double* __restrict__ vz, const uint32_t* __restrict__ scene,
                                                    unsigned long long* vmax) {
  __shared__ unsigned long long sm[SV_LDS];
  const bool inLds = nScenes <= SV_LDS;
  if (inLds)
    for (int k = threadIdx.x; k < nScenes; k += blockDim.x) sm[k] = 0ull;
  __syncthreads();
  const int64_t i = nW + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const unsigned long long v = (unsigned long long)__double_as_longlong(sqn3(mk3(vx[i], vy[i], vz[i])));
    if (inLds) atomicMax(&sm[scene[i]], v);
    else atomicMax(&vmax[scene[i]], v);
  }
  __syncthreads();
  if (inLds)
    for (int k = threadIdx.x; k < nScenes; k += blockDim.x)
      if (sm[k]) atomicMax(&vmax[k], sm[k]);
}
__global__ void k_dirty(int64_t n, const double* __restrict__ px, const double* __restrict__ py,
                        const double* __restrict__ pz, const double* __restrict__ lx, const double* __restrict__ ly,
                        const double* __restrict__ lz, double maxD2, const double* __restrict__ vdS,
                        const uint32_t* __restrict__ scene, uint32_t* dflags) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool dirty = false;
  if (i < n) {
    d3 d = sub3(mk3(lx[i], ly[i], lz[i]), mk3(px[i], py[i], pz[i]));
    double d2 = 0;
    d2 = fmax(d2, sqn3(d));
    double m2 = maxD2;
    if (vdS) {
      const double v = vdS[scene[i]];
      m2 = v * v;
    }
    dirty = d2 + 0. > m2;
  }
  if (__ballot(dirty) != 0ull && (threadIdx.x & 63) == 0) atomicOr(&dflags[0], 1u);
}

// order-preserving map of doubles to unsigned for atomic min/max
__device__ __forceinline__ unsigned long long ord_bits(double x) {
  unsigned long long b = (unsigned long long)__double_as_longlong(x);
  return (b >> 63) ? ~b : (b | (1ull << 63));
}
static inline double ord_to_double(unsigned long long b) {
  unsigned long long r = (b >> 63) ? (b & ~(1ull << 63)) : ~b;
  double d;
  std::memcpy(&d, &r, 8);
  return d;
}

// bounding box of the spheres: a grid-stride loop of few workgroups, each reducing in registers and
// across its wavefronts in LDS to six words; k_bbox_all takes those of all workgroups, to pinned
// memory: 4 + 2 us at 60,000 spheres (8 us with an atomic of every workgroup on one line, and two
// copies to set it up and read it back)
constexpr int BBOX_BLOCKS = 256;
__global__ __launch_bounds__(256) void k_bbox(int64_t s0, int64_t n, const double* __restrict__ px,
                                              const double* __restrict__ py, const double* __restrict__ pz,
                                              unsigned long long* out) {
  __shared__ unsigned long long sm[4][6];
  unsigned long long mn[3] = {~0ull, ~0ull, ~0ull}, mx[3] = {0, 0, 0};
  for (int64_t s = s0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < n; s += (int64_t)gridDim.x * blockDim.x) {
    const double p[3] = {px[s], py[s], pz[s]};
    for (int k = 0; k < 3; k++) {
      const unsigned long long b = ord_bits(p[k]);
      mn[k] = b < mn[k] ? b : mn[k];
      mx[k] = b > mx[k] ? b : mx[k];
    }
  }
  for (int k = 0; k < 3; k++) {
    for (int off = 32; off > 0; off >>= 1) {
      unsigned long long a = __shfl_xor(mn[k], off);
      unsigned long long b = __shfl_xor(mx[k], off);
      mn[k] = a < mn[k] ? a : mn[k];
      mx[k] = b > mx[k] ? b : mx[k];
    }
  }
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < 3; k++) {
      sm[wv][k] = mn[k];
      sm[wv][3 + k] = mx[k];
    }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    unsigned long long v = sm[0][k];
    for (int w = 1; w < 4; w++) v = k < 3 ? (sm[w][k] < v ? sm[w][k] : v) : (sm[w][k] > v ? sm[w][k] : v);
    out[6 * (int64_t)blockIdx.x + k] = v;
  }
}
// one wavefront per bound; the result in pinned host memory
__global__ __launch_bounds__(384) void k_bbox_all(int nb, const unsigned long long* __restrict__ part,
                                                  unsigned long long* out) {
  const int k = threadIdx.x >> 6, lane = threadIdx.x & 63;
  unsigned long long v = k < 3 ? ~0ull : 0ull;
  for (int b = lane; b < nb; b += 64) {
    const unsigned long long x = part[6 * b + k];
    v = k < 3 ? (x < v ? x : v) : (x > v ? x : v);
  }
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long x = __shfl_xor(v, off);
    v = k < 3 ? (x < v ? x : v) : (x > v ? x : v);
  }
  if (lane == 0) out[k] = v;
}

// bucket of cell (c0, c1, c2) in hashed mode: the coordinates packed into 63 bits and mixed
// (the finaliser of splitmix64), the high bits kept
__device__ __forceinline__ uint32_t cell_hash(int c0, int c1, int c2, uint32_t hmask) {
  uint64_t x = (uint64_t)(uint32_t)c0 | ((uint64_t)(uint32_t)c1 << 21) | ((uint64_t)(uint32_t)c2 << 42);
  x ^= x >> 30;
  x *= 0xbf58476d1ce4e5b9ull;
  x ^= x >> 27;
  x *= 0x94d049bb133111ebull;
  x ^= x >> 31;
  return (uint32_t)(x >> 32) & hmask;
}
// Morton code of cell (c0, c1, c2), each below 2^10: bit b of c_k at bit 3 b + k
__host__ __device__ inline uint32_t spread_bits3(uint32_t x) {
  x &= 0x3FFu;
  x = (x | (x << 16)) & 0x030000FFu;
  x = (x | (x << 8)) & 0x0300F00Fu;
  x = (x | (x << 4)) & 0x030C30C3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}
__host__ __device__ inline uint32_t gather_bits3(uint32_t x) {
  x &= 0x09249249u;
  x = (x | (x >> 2)) & 0x030C30C3u;
  x = (x | (x >> 4)) & 0x0300F00Fu;
  x = (x | (x >> 8)) & 0x030000FFu;
  x = (x | (x >> 16)) & 0x3FFu;
  return x;
}
__host__ __device__ inline uint32_t morton3(int c0, int c1, int c2) {
  return spread_bits3((uint32_t)c0) | (spread_bits3((uint32_t)c1) << 1) | (spread_bits3((uint32_t)c2) << 2);
}
__device__ __forceinline__ void cell_coords(const double p[3], const Grid& g, int c[3]) {
  for (int k = 0; k < 3; k++) {
    double x = p[k] - g.org[k];
    if (g.periodic) x = x - floor(x / g.L[k]) * g.L[k];
    int ci = (int)floor(x / g.h[k]);
    c[k] = min(max(ci, 0), g.nc[k] - 1);
  }
}
__device__ __forceinline__ uint32_t cell_key(const double p[3], const Grid& g) {
  int c[3];
  cell_coords(p, g, c);
  if (g.hashed) return cell_hash(c[0], c[1], c[2], g.hmask);
  if (g.morton) return morton3(c[0], c[1], c[2]);
  return (uint32_t)(((int64_t)c[2] * g.nc[1] + c[1]) * g.nc[0] + c[0]);
}

// cell of a position in a scene's grid
__device__ __forceinline__ void scene_cell(const double p[3], const SceneGrid& G, int c[3]) {
  for (int k = 0; k < 3; k++) {
    const int ci = (int)floor((p[k] - G.org[k]) / G.h);
    c[k] = min(max(ci, 0), G.nc[k] - 1);
  }
}
// cell key of every sphere (storage [s0,n)); value = current storage index
__global__ void k_keys(int64_t s0, int64_t n, const double* __restrict__ px, const double* __restrict__ py,
                       const double* __restrict__ pz, Grid g, const uint32_t* __restrict__ scene, uint32_t* key,
                       uint32_t* idx, uint32_t* cnt, uint32_t* rank) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t s = s0 + t;
  if (s >= n) return;
  double p[3] = {px[s], py[s], pz[s]};
  uint32_t k;
  if (g.sg) {
    const SceneGrid& G = g.sg[scene[s]];
    int c[3];
    scene_cell(p, G, c);
    k = G.off + (uint32_t)(((int64_t)c[2] * G.nc[1] + c[1]) * G.nc[0] + c[0]);
  } else {
    k = cell_key(p, g);
  }
  key[t] = k;
  if (cnt) rank[t] = atomicAdd(&cnt[k], 1u);
  else idx[t] = (uint32_t)s;
}

// Spheres in cell order by counting, with the spheres of a cell in their previous order (what a
// stable sort by cell gives). k_keys counts the spheres of each cell (a sphere's place in the
// count depends on the race), the counts are scanned, k_cell_place puts each sphere into its
// cell's range and k_cell_rank ranks it there among its cell's few by its previous place. The
// scanned counts are the cells' starts that the pair pass reads. Five launches, bound by latency;
// the radix passes it replaces (histogram, scan, scatter, each three times), the search for the
// cells' starts and the storage-index and record kernels took 190 us of a refresh of 150,000
// spheres, these with the permutation 60 us.
__global__ void k_cell_place(int64_t nSph, int64_t nW, const uint32_t* __restrict__ key,
                             const uint32_t* __restrict__ rank, const uint32_t* __restrict__ cbeg, uint32_t* placed) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < nSph) placed[cbeg[key[t]] - (uint32_t)nW + rank[t]] = (uint32_t)t;
}
// perm[new storage] = old storage, its inverse, and the key of each sphere in the new order;
// boundary bodies keep their place
__global__ void k_cell_rank(int64_t n, int64_t nW, const uint32_t* __restrict__ key,
                            const uint32_t* __restrict__ cbeg, const uint32_t* __restrict__ placed, uint32_t* perm,
                            uint32_t* invPerm, uint32_t* sortedKey) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (i < nW) {
    perm[i] = (uint32_t)i;
    invPerm[i] = (uint32_t)i;
    return;
  }
  const uint32_t w = (uint32_t)nW, v = placed[i - nW], k = key[v];
  const uint32_t b = cbeg[k], e = cbeg[k + 1];
  uint32_t s = b;
  for (uint32_t q = b; q < e; q++) s += placed[q - w] < v ? 1u : 0u;
  perm[s] = v + w;
  invPerm[v + w] = s;
  sortedKey[s - w] = k;
}

// bounding box and sphere count of every scene (ordered bits of the bounds, as k_bbox): per
// workgroup in LDS when the scenes are few, then one atomic per scene and bound
constexpr int SB_LDS = 512;
__global__ __launch_bounds__(256) void k_scene_bbox(int64_t nW, int64_t n, int64_t nScenes,
                                                    const double* __restrict__ px, const double* __restrict__ py,
                                                    const double* __restrict__ pz, const uint32_t* __restrict__ scene,
                                                    unsigned long long* out) {
  __shared__ unsigned long long sm[SB_LDS][7];
  const bool inLds = nScenes <= SB_LDS;
  if (inLds)
    for (int64_t k = threadIdx.x; k < nScenes; k += blockDim.x) {
      for (int q = 0; q < 3; q++) { sm[k][q] = ~0ull; sm[k][3 + q] = 0ull; }
      sm[k][6] = 0ull;
    }
  __syncthreads();
  const int64_t i = nW + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const uint32_t sc = scene[i];
    unsigned long long* o = inLds ? sm[sc] : out + 7 * (int64_t)sc;
    const double p[3] = {px[i], py[i], pz[i]};
    for (int q = 0; q < 3; q++) {
      const unsigned long long b = ord_bits(p[q]);
      atomicMin(&o[q], b);
      atomicMax(&o[3 + q], b);
    }
    atomicAdd(&o[6], 1ull);
  }
  __syncthreads();
  if (inLds)
    for (int64_t k = threadIdx.x; k < nScenes; k += blockDim.x) {
      if (!sm[k][6]) continue;
      for (int q = 0; q < 3; q++) {
        atomicMin(&out[7 * k + q], sm[k][q]);
        atomicMax(&out[7 * k + 3 + q], sm[k][3 + q]);
      }
      atomicAdd(&out[7 * k + 6], sm[k][6]);
    }
}

// perm[new storage] = old storage; walls keep their place
__global__ void k_build_perm(int64_t nW, int64_t n, const uint32_t* __restrict__ sorted, uint32_t* perm,
                             uint32_t* invPerm) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t o = i < nW ? (uint32_t)i : sorted[i - nW];
  perm[i] = o;
  invPerm[o] = (uint32_t)i;
}

struct PermArgs {
  int64_t n;
  const uint32_t* perm;
  const double* sd[NPD];
  double* dd[NPD];
  const uint32_t* su[NPU];
  uint32_t* du[NPU];
  // the refresh positions and the pair pass's float records, and the storage index of each user id
  Grid g;
  double absDf, vd0;
  const double* vdS;
  double *lx, *ly, *lz;
  float4* pf;
  uint32_t* sto;
};
// Every particle array in the new storage order; with the values in registers also the refresh
// positions, the user ids' storage index, and per particle the float record the pair kernel
// filters candidates with: position relative to the grid (wrapped into the cell when periodic) and
// the AABB half-size |distFactor|*r + verletDist. Bound by its 464 bytes per particle at the rate
// of a copy (1M: 95 us; as three kernels 116 us).
__global__ __launch_bounds__(256) void k_permute(PermArgs a) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const uint32_t o = a.perm[i];
  double d[NPD];
  uint32_t u[NPU];
#pragma unroll
  for (int k = 0; k < NPD; k++) d[k] = a.sd[k][o];
#pragma unroll
  for (int k = 0; k < NPU; k++) u[k] = a.su[k][o];
#pragma unroll
  for (int k = 0; k < NPD; k++) a.dd[k][i] = d[k];
#pragma unroll
  for (int k = 0; k < NPU; k++) a.du[k][i] = u[k];
  // the order of the arrays: pos first, radius last; flags, mask, uid, mat, scene
  a.sto[u[2]] = (uint32_t)i;
  a.lx[i] = d[0];
  a.ly[i] = d[1];
  a.lz[i] = d[2];
  float f[3];
  // relative to the origin of the sphere's grid (its scene's, with scene grids; the boundary
  // bodies' records are not read)
  const double* org = a.g.org;
  if (a.g.sg && !((u[0] >> F_SHAPE_SHIFT) & 3u)) org = a.g.sg[u[4]].org;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double x = d[k] - org[k];
    if (a.g.periodic) x = x - floor(x / a.g.L[k]) * a.g.L[k];
    f[k] = (float)x;
  }
  const double vd = a.vdS ? a.vdS[u[4]] : a.vd0;  // the scene's Verlet distance (vd_at)
  a.pf[i] = make_float4(f[0], f[1], f[2], (float)(a.absDf * d[NPD - 1] + vd));
}

// enlarged AABB of every boundary body from its refresh position: Bo1_Wall_Aabb
// (Wall.cpp:25-38), Bo1_Facet_Aabb (Facet.cpp:275-298, aperiodic), updateAabb's Verlet
// enlargement (Collision.cpp:150-160)
__global__ void k_bnd_bounds(int64_t nW, const double* __restrict__ lx, const double* __restrict__ ly,
                             const double* __restrict__ lz, const uint32_t* __restrict__ flags,
                             const double* __restrict__ fgeo, double vd0, const double* __restrict__ vdS,
                             const uint32_t* __restrict__ scene, double* bnd) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= nW) return;
  const double vd = vd_at(vdS, scene, w, vd0);
  const uint32_t fl = flags[w];
  double lo[3], hi[3];
  if (flag_shape(fl) == WDG_FACET) {
    const double* g = fgeo + (int64_t)FGEO * w;
    const double ht = g[12];
    for (int k = 0; k < 3; k++) {
      lo[k] = g[k] - ht;
      hi[k] = g[k] + ht;
    }
    for (int i = 1; i < 3; i++)
      for (int k = 0; k < 3; k++) {
        lo[k] = fmin(lo[k], g[3 * i + k] - ht);
        hi[k] = fmax(hi[k], g[3 * i + k] + ht);
      }
  } else {
    const int ax = flag_axis(fl);
    const double p[3] = {lx[w], ly[w], lz[w]};
    for (int k = 0; k < 3; k++) {
      lo[k] = -INFINITY;
      hi[k] = INFINITY;
    }
    lo[ax] = hi[ax] = p[ax];
  }
  if (vd > 0)
    for (int k = 0; k < 3; k++) {
      hi[k] = hi[k] + vd;
      lo[k] = lo[k] - vd;
    }
  for (int k = 0; k < 3; k++) {
    bnd[6 * w + k] = lo[k];
    bnd[6 * w + 3 + k] = hi[k];
  }
}

// cbeg[k] = storage index of the first sphere whose cell key is k or larger (s0 + nSph when
// none), for k in [0, ncells]: the spheres of cells [k0, k1] are storage [cbeg[k0], cbeg[k1 + 1]).
// One thread per cell, a binary search over the sorted keys.
__global__ void k_cell_begin(int64_t nSph, int64_t s0, const uint32_t* __restrict__ key, int64_t ncells,
                             uint32_t* cbeg) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k > ncells) return;
  int64_t lo = 0, hi = nSph;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)key[mid] < k) lo = mid + 1;
    else hi = mid;
  }
  cbeg[k] = (uint32_t)(s0 + lo);
}

enum { MODE_NEAR = 0, MODE_AABB = 1 };
// what k_pairs produces: counts only; counts plus the first PAIR_STAGE partners of each
// sphere in a staging area; slots written at given offsets; user-id keys at given offsets
enum { OUT_COUNT = 0, OUT_STAGE = 1, OUT_SLOTS = 2, OUT_KEYS = 3 };
constexpr int PAIR_STAGE = 24;  // staged pairs per generating sphere, at first (Ctx::pairStage)
constexpr int NB_STAGE = 48;    // staged neighbours per sphere (both directions), at first (Ctx::nbStage)

struct PairArgs {
  int64_t nW, n;
  const uint32_t* key;  // cell key of storage nW+t
  const double *px, *py, *pz;  // refresh positions (lastPos), storage order
  const double* rad;
  const uint32_t *mask, *uid, *flags;
  const uint32_t* scene;  // batched scenes: pairs only within a scene (else null)
  // batched scenes: the boundary bodies of scene k are sceneBody[sceneBodyOff[k] ..
  // sceneBodyOff[k+1]) (else null: the workgroup's list of bodies)
  const uint32_t *sceneBodyOff, *sceneBody;
  const uint32_t* cbeg;  // k_cell_begin
  const double* bnd;  // enlarged AABB of every boundary body (min3, max3), k_bnd_bounds
  const float4* pf;  // float candidate records (k_permute)
  const double* vdS;  // per-scene Verlet distances (batched scenes with per-scene skins), else null
  int stage;          // OUT_STAGE: staged pairs per sphere
  int nbStage;        // OUT_STAGE: staged neighbours per sphere
  float margin;      // added to the float reach so that the float test never rejects a pair
  Grid g;
  AabbParams P;
  int brute;
  int64_t nSph;
  // outputs
  uint32_t* count;
  uint32_t* deg;      // OUT_STAGE: neighbours of every sphere, both directions and walls
  uint32_t* nb;       // OUT_STAGE: the neighbours, NB_STAGE per sphere, neighbour-major
  const uint32_t* off;
  uint32_t *sA, *sB, *sInfo, *sCarry;  // OUT_SLOTS: slot arrays; OUT_STAGE: sA = partner, sInfo
  uint64_t* sDist;
  uint64_t* pkey;    // OUT_KEYS: (uidA<<32)|uidB
  uint64_t* pdist;
  uint32_t* bmax;    // OUT_STAGE: per workgroup, the largest pair count and neighbour count
  uint32_t* dflags;
};

// boundary bodies a workgroup's spheres can meet, found once per workgroup
constexpr int BLIST = 256;

// Pairs generated by sphere s: spheres j > s (storage order) of the 27 neighbour cells,
// and every wall. Each pair is emitted once, by its sphere of lower storage index. With
// OUT_STAGE the sphere also records every neighbour (j < s too, with the same test, whose
// arithmetic follows the canonical pA/pB roles and so gives the same answer from either
// side), which is its adjacency list. A float test on the grid-relative positions decides most
// candidates; its margin keeps it from rejecting any pair or accepting anything else.
//
// G lanes share a sphere: each walks a part of its candidates and queues those that pass the
// float test; the queues are worked off by the whole wavefront together, a group's finds placed
// one after the other by ballots (a fixed order: rounds of the queue, lanes within a round).
// Bound by the latency of the loads and of the instructions between them (a sphere has about 70
// candidates in 27 cells, some 5,000 instructions): one lane a sphere left 2 wavefronts a SIMD
// at 150,000 spheres and less below; before, each lane loaded one candidate at a time and tested
// every queued one in FP64: 72 us for 300 spheres, 60 us for 20,000, 107 us for 150,000, 293 us
// for 1M. pair_lanes gives the figures now.
constexpr int PAIR_Q = 12;  // candidates queued per lane
constexpr int PAIR_B = 4;   // candidates read together
constexpr uint32_t PAIR_SURE = 0x80000000u;  // queued candidate: a pair for certain
// the cells of the spheres: none (all pairs), rows along x (one grid or a grid per scene), Morton
// codes, hashed
enum { CELL_NONE = 0, CELL_ROWS = 1, CELL_MORTON = 2, CELL_HASHED = 3 };

template <int OUT, int MODE, int KIND, int G>
__global__ __launch_bounds__(256) void k_pairs(PairArgs a) {
  __shared__ uint32_t sq[PAIR_Q][256];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = threadIdx.x & (G - 1);
  // consecutive workgroups on one XCD: a sphere's neighbour cells are mostly in its own XCD's L2
  const int64_t s = a.nW + ((int64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x) / G;
  const bool live = s < a.n;
  const int64_t sl = live ? s : a.n - 1;  // a sphere to read for the lanes past the end
  const int64_t t = sl - a.nW;
  uint32_t cnt = 0, ndeg = 0;  // pairs and neighbours of the sphere so far (the same in its lanes)
  const double ps[3] = {a.px[sl], a.py[sl], a.pz[sl]};
  const double rs = a.rad[sl];
  const uint32_t ms = a.mask[sl], us = a.uid[sl];
  const uint32_t scs = a.scene ? a.scene[sl] : 0u;
  const float4 fs = a.pf[sl];
  // this sphere's Verlet distance (its scene's; the pairs never cross scenes)
  const double vds = vd_at(a.vdS, a.scene, sl, a.P.vd);
  // enlarged AABB of the wavefront's and the workgroup's spheres: the workgroup lists the boundary
  // bodies its box meets (in body order), each wavefront skips those its own box misses, each
  // sphere tests the rest
  __shared__ uint32_t blist[BLIST];
  __shared__ uint32_t bwc[4];
  __shared__ double bbox[4][6];
  __shared__ int bcount;
  int nb = 0;
  bool bfull = false;
  if (a.nW > 0 && !a.sceneBodyOff) {
    double wlo[3], whi[3];
    for (int k = 0; k < 3; k++) {
      sph_bounds(ps[k], a.P.absDf * rs, vds, wlo[k], whi[k]);
      for (int off = 32; off > 0; off >>= 1) {
        wlo[k] = fmin(wlo[k], __shfl_xor(wlo[k], off));
        whi[k] = fmax(whi[k], __shfl_xor(whi[k], off));
      }
    }
    if (lane == 0)
      for (int k = 0; k < 3; k++) {
        bbox[wv][k] = wlo[k];
        bbox[wv][3 + k] = whi[k];
      }
    if (threadIdx.x == 0) bcount = 0;
    __syncthreads();
    double glo[3], ghi[3];
    for (int k = 0; k < 3; k++) {
      glo[k] = fmin(fmin(bbox[0][k], bbox[1][k]), fmin(bbox[2][k], bbox[3][k]));
      ghi[k] = fmax(fmax(bbox[0][3 + k], bbox[1][3 + k]), fmax(bbox[2][3 + k], bbox[3][3 + k]));
    }
    for (int64_t w0 = 0; w0 < a.nW; w0 += blockDim.x) {
      const int64_t w = w0 + threadIdx.x;
      bool hit = false;
      if (w < a.nW) {
        const double* b = a.bnd + 6 * w;
        hit = b[0] <= ghi[0] && b[3] >= glo[0] && b[1] <= ghi[1] && b[4] >= glo[1] && b[2] <= ghi[2] &&
              b[5] >= glo[2];
      }
      const unsigned long long m = __ballot(hit);
      if (lane == 0) bwc[wv] = (uint32_t)__popcll(m);
      __syncthreads();
      int base = bcount;
      for (int q = 0; q < wv; q++) base += (int)bwc[q];
      const unsigned long long lt = lane ? (~0ull >> (64 - lane)) : 0ull;
      const int pos = base + __popcll(m & lt);
      if (hit && pos < BLIST) blist[pos] = (uint32_t)w;
      __syncthreads();
      if (threadIdx.x == 0) bcount += (int)(bwc[0] + bwc[1] + bwc[2] + bwc[3]);
      __syncthreads();
    }
    nb = bcount;
    bfull = nb > BLIST;  // too many for the list: every body is tested
  }
  const int64_t o = (OUT == OUT_SLOTS || OUT == OUT_KEYS) ? (int64_t)a.off[t] : t;
  const unsigned long long gmask = (G == 64 ? ~0ull : ((1ull << G) - 1ull)) << (lane & ~(G - 1));
  const unsigned long long below = gmask & ((1ull << lane) - 1ull);
  // One find of each lane (hit): neighbour j, and with gen the pair itself. Every lane of the
  // wavefront calls it. Staged arrays are neighbour-major: entry q of sphere t at q * nSph + t.
  auto emit = [&](bool hit, bool gen, uint32_t partner, uint32_t lo, uint32_t hi, uint32_t info, uint64_t cd,
                  uint64_t ukey) {
    const unsigned long long H = __ballot(hit), P = __ballot(hit && gen);
    if (hit && OUT == OUT_STAGE) {
      const uint32_t d = ndeg + (uint32_t)__popcll(H & below);
      if (d < (uint32_t)a.nbStage) a.nb[(int64_t)d * a.nSph + t] = partner;
    }
    if (hit && gen) {
      const uint32_t c = cnt + (uint32_t)__popcll(P & below);
      if (OUT == OUT_STAGE) {
        if (c < (uint32_t)a.stage) {
          const int64_t e = (int64_t)c * a.nSph + o;
          a.sA[e] = partner;
          a.sInfo[e] = info;
          if (a.P.periodic) a.sDist[e] = cd;
        }
      } else if (OUT == OUT_SLOTS) {
        a.sA[o + c] = lo;
        a.sB[o + c] = hi;
        a.sInfo[o + c] = info;
        a.sCarry[o + c] = 0u;
        if (a.P.periodic) a.sDist[o + c] = cd;
      } else if (OUT == OUT_KEYS) {
        a.pkey[o + c] = ukey;
        if (a.P.periodic) a.pdist[o + c] = cd;
      }
    }
    ndeg += (uint32_t)__popcll(H & gmask);
    cnt += (uint32_t)__popcll(P & gmask);
  };
  // the exact test of a candidate that the float test left open (the periodic image is found
  // again in FP64 by sph_overlap)
  auto exact = [&](int64_t j, bool sIsA, const double (&pj)[3], uint64_t& pcd) {
    const double rj = a.rad[j];
    // canonical roles: the smaller user id is pA
    const double* pa = sIsA ? ps : pj;
    const double* pb = sIsA ? pj : ps;
    const double ra = sIsA ? rs : rj, rb = sIsA ? rj : rs;
    int cd[3], nimg;
    if (!sph_overlap(pa, a.P.absDf * ra, pb, a.P.absDf * rb, a.P, vds, cd, nimg)) return false;
    if (a.P.periodic && nimg > 1) {
      atomicOr(&a.dflags[1], ERR_DOUBLE_IMAGE);
      return false;
    }
    if (MODE == MODE_NEAR) {
      // centres within reach before the next refresh
      d3 d = mk3(pb[0] + a.P.L[0] * cd[0] * a.P.periodic - pa[0], pb[1] + a.P.L[1] * cd[1] * a.P.periodic - pa[1],
                 pb[2] + a.P.L[2] * cd[2] * a.P.periodic - pa[2]);
      double reach = a.P.absDf * (ra + rb) + 2 * vds;
      if (sqn3(d) > reach * reach * (1 + 1e-9)) return false;
    }
    pcd = a.P.periodic ? pack_cd(cd[0], cd[1], cd[2]) : 0ull;
    return true;
  };
  int nq = 0;
  // Works off the queues. A candidate that the float test accepted for certain needs its periodic
  // image only: the pair is far nearer than half a period on every axis, so the nearest integer is
  // that of near_img.
  auto flush = [&]() {
    for (int k = 0; __any(k < nq); k++) {
      bool hit = k < nq;
      const uint32_t e = hit ? sq[k][threadIdx.x] : (uint32_t)sl;
      const uint32_t j = e & ~PAIR_SURE;
      const uint32_t uj = a.uid[j];
      const bool sIsA = us < uj;
      hit = hit && may_collide(ms, a.mask[j], a.P.loneMask) && (!a.scene || a.scene[j] == scs);
      uint64_t pcd = 0ull;
      if (hit && (a.P.periodic || !(e & PAIR_SURE))) {
        const double pj[3] = {a.px[j], a.py[j], a.pz[j]};
        if (!(e & PAIR_SURE)) {
          hit = exact((int64_t)j, sIsA, pj, pcd);
        } else {
          int cd[3];
#pragma unroll
          for (int d = 0; d < 3; d++) {
            const int c = (int)rint((pj[d] - ps[d]) / a.P.L[d]);
            cd[d] = sIsA ? -c : c;
          }
          pcd = pack_cd(cd[0], cd[1], cd[2]);
        }
      }
      emit(hit, (int64_t)j > s, j, (uint32_t)s, j, (uint32_t)CT_SS | CI_NEAR | (sIsA ? 0u : CI_SWAP), pcd,
           sIsA ? (((uint64_t)us << 32) | uj) : (((uint64_t)uj << 32) | us));
    }
    nq = 0;
  };
  // The float test of candidate j with the periodic shift of its cell. Its margin covers the
  // rounding of the float positions many times over, so a candidate beyond reach plus margin is
  // no pair, one within reach minus margin is one, and only those between need the exact test.
  auto consider = [&](int64_t j, const float4& fj, float sx, float sy, float sz) {
    if (OUT == OUT_STAGE ? j == s : j <= s) return;
    if (KIND == CELL_NONE && a.P.periodic) {
      const float d[3] = {fj.x - fs.x, fj.y - fs.y, fj.z - fs.z};
      sx = -(float)a.P.L[0] * rintf(d[0] / (float)a.P.L[0]);
      sy = -(float)a.P.L[1] * rintf(d[1] / (float)a.P.L[1]);
      sz = -(float)a.P.L[2] * rintf(d[2] / (float)a.P.L[2]);
    }
    const float dx = (fj.x + sx) - fs.x, dy = (fj.y + sy) - fs.y, dz = (fj.z + sz) - fs.z;
    const float R = (fs.w + fj.w) + a.margin;
    const float mx = fmaxf(fmaxf(fabsf(dx), fabsf(dy)), fabsf(dz));
    if (mx > R) return;
    const float d2 = (dx * dx + dy * dy) + dz * dz;
    // the centre-distance test must not hide a pair whose AABBs overlap through two
    // periodic images (an error below); that needs fewer than 3 cells along an axis,
    // which is the all-pairs path
    if (MODE == MODE_NEAR && KIND != CELL_NONE && d2 > R * R) return;
    const float Ri = R - 2.f * a.margin;
    const bool sure = KIND != CELL_NONE && Ri > 0.f && (MODE == MODE_NEAR ? d2 < Ri * Ri : mx < Ri);
    sq[nq++][threadIdx.x] = (uint32_t)j | (sure ? PAIR_SURE : 0u);
  };
  // The candidates as M storage ranges [t0, t1), each with the periodic shift of its cells; the
  // lane takes ranges m0 .. m1 - 1 (all pairs: a part of the one range).
  struct Range {
    uint32_t t0, t1;
    float sx, sy, sz;
  };
  int M = G;
  int c[3] = {0, 0, 0}, nc[3] = {a.g.nc[0], a.g.nc[1], a.g.nc[2]};
  uint32_t kbase = 0u;
  int xlo = 0, xhi = 0, xw = -1;
  float xwsh = 0.f;
  if (KIND == CELL_HASHED) {
    cell_coords(ps, a.g, c);
    M = 27;
  } else if (KIND == CELL_MORTON) {
    const uint32_t k = a.key[t];
    for (int d = 0; d < 3; d++) c[d] = (int)gather_bits3(k >> d);
    M = 27;
  } else if (KIND == CELL_ROWS) {
    // the sphere's grid: its scene's (keys from the scene's offset), or the one grid
    uint32_t k = a.key[t];
    if (a.g.sg) {
      const SceneGrid& S = a.g.sg[scs];
      kbase = S.off;
      for (int d = 0; d < 3; d++) nc[d] = S.nc[d];
      k -= kbase;
    }
    c[0] = (int)(k % (uint32_t)nc[0]);
    c[1] = (int)((k / (uint32_t)nc[0]) % (uint32_t)nc[1]);
    c[2] = (int)(k / ((uint32_t)nc[0] * (uint32_t)nc[1]));
    xlo = c[0] > 0 ? c[0] - 1 : 0;
    xhi = c[0] + 1 < nc[0] ? c[0] + 1 : nc[0] - 1;
    if (a.g.periodic && c[0] == 0) { xw = nc[0] - 1; xwsh = -(float)a.g.L[0]; }
    if (a.g.periodic && c[0] == nc[0] - 1) { xw = 0; xwsh = (float)a.g.L[0]; }
    M = a.g.periodic ? 18 : 9;
  }
  const int m1 = live ? (g + 1) * M / G : 0;
  auto range = [&](int m) {
    Range r{0u, 0u, 0.f, 0.f, 0.f};
    if (m >= m1) return r;
    if (KIND == CELL_NONE) {
      r.t0 = (uint32_t)(a.nW + a.nSph * m / G);
      r.t1 = (uint32_t)(a.nW + a.nSph * (m + 1) / G);
      return r;
    }
    // The 27 neighbour cells one by one where their keys are not consecutive (Morton, hashed).
    // Else as 9 rows along x: cells x-1..x+1 of a row are consecutive keys, so their spheres are
    // one storage range; across a periodic x boundary the wrapped cell is a second range.
    const bool rows = KIND == CELL_ROWS;
    const bool wrap = rows && a.g.periodic && (m & 1);
    const int row = rows ? (a.g.periodic ? m >> 1 : m) : m / 3;
    int q[3] = {rows ? 0 : c[0] + m % 3 - 1, c[1] + row % 3 - 1, c[2] + row / 3 - 1};
    // a cell across a periodic boundary is its image, one period away on this side (every axis
    // has at least 3 cells, so the 27 are distinct)
    float sh[3] = {0.f, 0.f, 0.f};
    bool ok = !wrap || xw >= 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const bool lo = q[d] < 0, hi = q[d] >= nc[d];
      ok = ok && (!(lo || hi) || a.g.periodic);
      sh[d] = lo ? -(float)a.g.L[d] : (hi ? (float)a.g.L[d] : 0.f);
      q[d] += lo ? nc[d] : (hi ? -nc[d] : 0);
    }
    if (!ok) return r;
    uint32_t b0, b1;
    if (KIND == CELL_HASHED) {
      b0 = cell_hash(q[0], q[1], q[2], a.g.hmask);
      // a bucket shared by two of the cells (a hash collision) is walked once, at the first; a
      // sphere of a far cell in a walked bucket fails the float test
      for (int m2 = 0; m2 < m; m2++) {
        const int r0 = c[0] + m2 % 3 - 1, r1 = c[1] + (m2 / 3) % 3 - 1, r2 = c[2] + m2 / 9 - 1;
        if (r0 < 0 || r1 < 0 || r2 < 0 || r0 >= nc[0] || r1 >= nc[1] || r2 >= nc[2]) continue;
        if (cell_hash(r0, r1, r2, a.g.hmask) == b0) return r;
      }
      b1 = b0;
    } else if (KIND == CELL_MORTON) {
      b0 = b1 = morton3(q[0], q[1], q[2]);
    } else {
      const uint32_t rb = kbase + (uint32_t)(((int64_t)q[2] * nc[1] + q[1]) * nc[0]);
      b0 = rb + (uint32_t)(wrap ? xw : xlo);
      b1 = rb + (uint32_t)(wrap ? xw : xhi);
      sh[0] = wrap ? xwsh : 0.f;
    }
    r = Range{a.cbeg[b0], a.cbeg[b1 + 1], sh[0], sh[1], sh[2]};
    return r;
  };
  // One batch of PAIR_B candidates a turn, every lane in its own ranges, the bounds of the next
  // range loaded while the current one is walked
  {
    int m = g * M / G;
    Range ra = range(m), rb = range(m + 1);
    uint32_t tt = ra.t0;
    while (__any(m < m1)) {
      if (__any(nq > PAIR_Q - PAIR_B)) flush();
      float4 f[PAIR_B];
#pragma unroll
      for (int q = 0; q < PAIR_B; q++) f[q] = a.pf[tt + q < ra.t1 ? (int64_t)(tt + q) : sl];
#pragma unroll
      for (int q = 0; q < PAIR_B; q++)
        if (tt + q < ra.t1) consider(tt + q, f[q], ra.sx, ra.sy, ra.sz);
      tt += PAIR_B;
      if (tt >= ra.t1) {
        m++;
        ra = rb;
        tt = ra.t0;
        rb = range(m + 1);
      }
    }
  }
  flush();
  // boundary bodies (storage [0,nW): walls, facets) against every sphere, the body as pA:
  // AABB overlap (InsertionSortCollider.cpp:67-73) of the body's enlarged AABB and the
  // sphere's. The AABB of a wall is infinite except along its axis (Wall.cpp:25-38).
  // batched scenes: the sphere's own scene's bodies; else the workgroup's list; the lanes of a
  // sphere take them in turn
  if (a.nW > 0) {
    const bool own = a.sceneBodyOff != nullptr;
    const double* wb = bbox[wv];  // the wavefront's box
    double slo[3], shi[3];
    for (int k = 0; k < 3; k++) sph_bounds(ps[k], a.P.absDf * rs, vds, slo[k], shi[k]);
    const int64_t q0 = own ? (int64_t)a.sceneBodyOff[scs] : 0;
    const int64_t q1 = !live ? 0 : (own ? (int64_t)a.sceneBodyOff[scs + 1] : (bfull ? a.nW : nb));
    for (int64_t q = q0 + g; __any(q < q1); q += G) {
      bool hit = q < q1;
      int64_t w = 0;
      if (hit) {
        w = own ? (int64_t)a.sceneBody[q] : (bfull ? q : (int64_t)blist[q]);
        const double* b = a.bnd + 6 * w;
        hit = own || (b[0] <= wb[3] && b[3] >= wb[0] && b[1] <= wb[4] && b[4] >= wb[1] && b[2] <= wb[5] &&
                      b[5] >= wb[2]);
        hit = hit && b[0] <= shi[0] && b[3] >= slo[0] && b[1] <= shi[1] && b[4] >= slo[1] && b[2] <= shi[2] &&
              b[5] >= slo[2];
        hit = hit && may_collide(a.mask[w], ms, a.P.loneMask) && (!a.scene || a.scene[w] == scs);
      }
      const uint32_t type = hit && flag_shape(a.flags[w]) == WDG_FACET ? CT_FS : CT_WS;
      emit(hit, true, (uint32_t)w, (uint32_t)w, (uint32_t)s, type | CI_NEAR, pack_cd(0, 0, 0),
           hit ? (((uint64_t)a.uid[w] << 32) | us) : 0ull);
    }
  }
  if (live && g == 0) {
    if (OUT == OUT_COUNT || OUT == OUT_STAGE) a.count[t] = cnt;
    if (OUT == OUT_STAGE) a.deg[t] = ndeg;
  }
  if (OUT == OUT_STAGE) {
    // largest counts, for the staging-capacity check: one pair of words per workgroup
    // (reduced by k_block_max; device-wide atomics on one line would serialise)
    __shared__ uint32_t wm[4][2];
    uint32_t mc = cnt, md = ndeg;
    for (int off = 32; off > 0; off >>= 1) {
      mc = max(mc, (uint32_t)__shfl_xor(mc, off));
      md = max(md, (uint32_t)__shfl_xor(md, off));
    }
    if ((threadIdx.x & 63) == 0) {
      wm[threadIdx.x >> 6][0] = mc;
      wm[threadIdx.x >> 6][1] = md;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
      const int k = threadIdx.x;
      a.bmax[2 * blockIdx.x + k] = max(max(wm[0][k], wm[1][k]), max(wm[2][k], wm[3][k]));
    }
  }
}

// Lanes per sphere: as many as fill the chip's 1,024 SIMDs with a few wavefronts. Measured (us, with 1 / 2
// / 4 / 8 lanes): all pairs of 300 spheres 73 / 46 / 34 / 24, 2,000 in cells 46 / 30 / 19 / 15, 20,000: 56 /
// 35 / 23 / 18, 150,000 dense: 94 / 92 / 85 / 92, 186,000 sparse in 64 scenes 36 / 46 / 59 / 80, 1M: 309 /
// 328 / 377 / 481 (the passes over queues and cells that more lanes repeat then cost more than the
// latency they hide, the more so the fewer candidates a sphere has). The density is not known before the
// pass, so one lane from 100,000 on: that gives up a tenth in a dense scene and four lanes would cost a
// sparse one two thirds.
static int pair_lanes(int64_t nSph) { return nSph <= 40000 ? 8 : (nSph <= 100000 ? 4 : 1); }
template <int OUT, int MODE, int G>
static void launch_pairs_g(Ctx& c, const PairArgs& a) {
  const dim3 grid(nblocks(a.nSph * G, 256)), block(256);
  if (a.brute) hipLaunchKernelGGL((k_pairs<OUT, MODE, CELL_NONE, G>), grid, block, 0, c.stream, a);
  else if (a.g.hashed) hipLaunchKernelGGL((k_pairs<OUT, MODE, CELL_HASHED, G>), grid, block, 0, c.stream, a);
  else if (a.g.morton) hipLaunchKernelGGL((k_pairs<OUT, MODE, CELL_MORTON, G>), grid, block, 0, c.stream, a);
  else hipLaunchKernelGGL((k_pairs<OUT, MODE, CELL_ROWS, G>), grid, block, 0, c.stream, a);
  WDG_LAUNCH_CHECK();
}
template <int OUT, int MODE>
static void launch_pairs(Ctx& c, const PairArgs& a) {
  // (the passes besides the refresh's own, which are rare, all take 4)
  const int G = OUT == OUT_STAGE ? pair_lanes(a.nSph) : 4;
  if (OUT == OUT_STAGE && G == 1) launch_pairs_g<OUT, MODE, OUT == OUT_STAGE ? 1 : 4>(c, a);
  else if (OUT == OUT_STAGE && G == 8) launch_pairs_g<OUT, MODE, OUT == OUT_STAGE ? 8 : 4>(c, a);
  else launch_pairs_g<OUT, MODE, 4>(c, a);
}

// largest of the per-workgroup maxima of k_pairs, one workgroup
// (and the number of pairs, dflags[4]: all three to the host's pinned words 4, 7 and 8; the merge's
// counter of extra slots is cleared on the way)
__global__ __launch_bounds__(1024) void k_block_max(int64_t nb, const uint32_t* __restrict__ bmax, uint32_t* dflags,
                                                     uint32_t* host) {
  __shared__ uint32_t sm[2][16];
  uint32_t m0 = 0, m1 = 0;
  for (int64_t i = threadIdx.x; i < nb; i += blockDim.x) {
    m0 = max(m0, bmax[2 * i]);
    m1 = max(m1, bmax[2 * i + 1]);
  }
  for (int off = 32; off > 0; off >>= 1) {
    m0 = max(m0, (uint32_t)__shfl_xor(m0, off));
    m1 = max(m1, (uint32_t)__shfl_xor(m1, off));
  }
  if ((threadIdx.x & 63) == 0) {
    sm[0][threadIdx.x >> 6] = m0;
    sm[1][threadIdx.x >> 6] = m1;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    uint32_t m = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) m = max(m, sm[threadIdx.x][w]);
    host[7 + threadIdx.x] = m;
  }
  if (threadIdx.x == 2) host[4] = dflags[4];
  if (threadIdx.x == 3) dflags[6] = 0u;
}

// staged pairs -> slot list. The 64 spheres of a wavefront write one contiguous range of slots:
// each lane takes every 64th slot of it, finds its sphere among the wavefront's offsets (LDS,
// binary search) and copies that staged entry, so every store is contiguous across the lanes.
constexpr int US_BS = 256;
__global__ __launch_bounds__(US_BS) void k_unstage(int64_t nW, int64_t nSph, const uint32_t* __restrict__ count,
                                                   const uint32_t* __restrict__ off,
                                                   const uint32_t* __restrict__ partner,
                                                   const uint32_t* __restrict__ pinfo,
                                                   const uint64_t* __restrict__ pdist, int periodic, uint32_t* A,
                                                   uint32_t* B, uint32_t* info, uint64_t* dist, uint32_t* carry) {
  __shared__ uint32_t so[US_BS / 64][65];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t tw = (int64_t)blockIdx.x * US_BS + w * 64;  // the wavefront's first sphere
  if (tw >= nSph) return;  // whole wavefront (uniform)
  const int64_t t = tw + lane;
  uint32_t o = 0, n = 0;
  if (t < nSph) {
    o = off[t];
    n = count[t];
  }
  const uint32_t ob = __shfl(o, 0);
  // end of the wavefront's range: the largest o + n of its valid lanes
  uint32_t end = t < nSph ? o + n : 0u;
  for (int d = 32; d > 0; d >>= 1) end = max(end, (uint32_t)__shfl_xor(end, d));
  so[w][lane] = (t < nSph ? o : end) - ob;
  if (lane == 0) so[w][64] = end - ob;
  wave_lds_sync();
  const uint32_t total = end - ob;
  for (uint32_t p = lane; p < total; p += 64) {
    // largest lane L with so[L] <= p
    int L = 0;
    for (int step = 32; step > 0; step >>= 1)
      if (L + step < 64 && so[w][L + step] <= p) L += step;
    const uint32_t q = p - so[w][L];
    const int64_t src = (int64_t)q * nSph + tw + L;
    const uint32_t s = (uint32_t)(nW + tw + L), j = partner[src], inf = pinfo[src];
    const bool ws = (inf & CI_TYPE_MASK) != CT_SS;  // a boundary body (storage below nW) is A
    const int64_t d = (int64_t)ob + p;
    A[d] = ws ? j : s;
    B[d] = ws ? s : j;
    info[d] = inf;
    carry[d] = 0u;
    if (periodic) dist[d] = pdist[src];
  }
}

// the slot among the n from g0 whose partner is p (0xFFFFFFFF: none), four read at a time so that
// the search costs one memory latency for most spheres instead of one per slot
__device__ __forceinline__ uint32_t find_partner(const uint32_t* __restrict__ B, uint32_t g0, uint32_t n, uint32_t p) {
  uint32_t slot = 0xFFFFFFFFu;
  for (uint32_t u = 0; u < n && slot == 0xFFFFFFFFu; u += 4) {
    uint32_t b[4];
#pragma unroll
    for (int q = 0; q < 4; q++) b[q] = B[g0 + (u + q < n ? u + q : u)];
#pragma unroll
    for (int q = 3; q >= 0; q--)
      if (u + q < n && b[q] == p) slot = g0 + u + q;
  }
  return slot;
}

struct MergeArgs {
  int64_t nOld, nW, nPairs;
  RealView ov;
  const uint32_t *oA, *oB, *oInfo;
  const uint64_t* oDist;
  const uint32_t* invPerm;
  const uint32_t *count, *off;  // per generating sphere
  int periodic;
  uint32_t *A, *B, *info, *carry;
  uint64_t* dist;
  uint32_t* nExtra;
};

// Each real contact of the old list finds its pair among the slots generated by its sphere
// of lower new storage index (a handful), or is appended behind the new pairs: a contact
// persists until its law breaks it, whether or not the pair is still near.
__global__ void k_merge(MergeArgs a) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= a.nOld || !rv_real(a.ov, (uint32_t)c)) return;
  const uint32_t oi = a.oInfo[c];
  const uint32_t x = a.invPerm[a.oA[c]], y = a.invPerm[a.oB[c]];
  const uint32_t lo = x < y ? x : y, hi = x < y ? y : x;
  const bool ws = (oi & CI_TYPE_MASK) != CT_SS;
  const uint32_t gen = ws ? hi : lo;  // the generating sphere (boundary bodies come first in storage)
  // its slots with spheres have it as A and a later sphere as B, those with boundary bodies the
  // other way round
  const uint32_t found = find_partner(ws ? a.A : a.B, a.off[gen - a.nW], a.count[gen - a.nW], ws ? lo : hi);
  if (found != 0xFFFFFFFFu) {
    a.carry[found] = (uint32_t)c + 1u;
    // the contact keeps the periodic image it was created in
    if (a.periodic) a.dist[found] = a.oDist[c];
    return;
  }
  const uint32_t t = (uint32_t)a.nPairs + atomicAdd(a.nExtra, 1u);
  // roles are fixed by user ids: find where the old pA went
  const uint32_t newPA = a.invPerm[(oi & CI_SWAP) ? a.oB[c] : a.oA[c]];
  a.A[t] = lo;
  a.B[t] = hi;
  a.info[t] = (oi & CI_TYPE_MASK) | (newPA == hi ? CI_SWAP : 0u);
  a.carry[t] = (uint32_t)c + 1u;
  if (a.periodic) a.dist[t] = a.oDist[c];
}

// contact state of the carried real contacts: old index -> new index
struct CarryArgs {
  int64_t n;
  const uint32_t* carry;
  RealView ov, nv;
  const double* o[10];
  double* d[10];
  const double* ogp;
  double* gp;
  const uint8_t* oE;  // material epochs (while more than one table is kept; else null)
  uint8_t* nE;
  const double* ogt;  // global phys torques (rolling resistance; else null)
  double* gt;
};
template <int PREC>
__global__ void k_carry_state(CarryArgs a) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= a.n) return;
  const uint32_t cy = a.carry[s];
  if (!cy) return;
  const uint32_t ko = rv_index(a.ov, cy - 1u), kn = rv_index(a.nv, (uint32_t)s);
  if (a.oE) a.nE[kn] = a.oE[ko];
  if (a.ogt)
    for (int q = 0; q < 3; q++) a.gt[(int64_t)3 * kn + q] = a.ogt[(int64_t)3 * ko + q];
  if (PREC == 32) {
#pragma unroll
    for (int q = 0; q < 10; q++) reinterpret_cast<float*>(a.d[q])[kn] = reinterpret_cast<const float*>(a.o[q])[ko];
    const float4* src = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(a.ogp) + (int64_t)GP32 * ko);
    float4* dst = reinterpret_cast<float4*>(reinterpret_cast<float*>(a.gp) + (int64_t)GP32 * kn);
#pragma unroll
    for (int q = 0; q < GP32 / 4; q++) dst[q] = src[q];
    return;
  }
#pragma unroll
  for (int q = 0; q < 10; q++) a.d[q][kn] = a.o[q][ko];
  const double2* src = reinterpret_cast<const double2*>(a.ogp + (int64_t)GP * ko);
  double2* dst = reinterpret_cast<double2*>(a.gp + (int64_t)GP * kn);
#pragma unroll
  for (int q = 0; q < GP / 2; q++) dst[q] = src[q];
}

// ------------------------------------------------------------------ adjacency
// entries per particle
__global__ void k_adj_deg(int64_t nc, const uint32_t* __restrict__ A, const uint32_t* __restrict__ B,
                          uint32_t* deg) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nc) return;
  atomicAdd(&deg[A[t]], 1u);
  atomicAdd(&deg[B[t]], 1u);
}
// entries (other user id << 32 | slot | ADJ_PA) in arbitrary order within each particle's
// range; deg counts down to zero
__global__ void k_adj_fill(int64_t nc, const uint32_t* __restrict__ A, const uint32_t* __restrict__ B,
                           const uint32_t* __restrict__ info, const uint32_t* __restrict__ uid,
                           const uint32_t* __restrict__ adjOff, uint32_t* deg, uint64_t* ent) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nc) return;
  const uint32_t lo = A[t], hi = B[t];
  const bool swap = (info[t] & CI_SWAP) != 0u;
  const uint32_t pl = atomicSub(&deg[lo], 1u) - 1u;
  ent[adjOff[lo] + pl] = ((uint64_t)uid[hi] << 32) | (uint32_t)t | (swap ? 0u : ADJ_PA);
  const uint32_t ph = atomicSub(&deg[hi], 1u) - 1u;
  ent[adjOff[hi] + ph] = ((uint64_t)uid[lo] << 32) | (uint32_t)t | (swap ? ADJ_PA : 0u);
}
// boundary bodies' list lengths from the slot list (their pairs have the body as A): counted
// per workgroup in LDS first when there are few bodies
constexpr int WD_LDS = 8192;
__global__ __launch_bounds__(256) void k_wall_deg(int64_t nc, int64_t nW, const uint32_t* __restrict__ A,
                                                  uint32_t* deg) {
  __shared__ uint32_t sh[WD_LDS];
  const bool inLds = nW <= WD_LDS;
  if (inLds)
    for (int64_t k = threadIdx.x; k < nW; k += blockDim.x) sh[k] = 0u;
  __syncthreads();
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < nc) {
    const uint32_t a = A[t];
    if (a < (uint32_t)nW) {
      if (inLds) atomicAdd(&sh[a], 1u);
      else atomicAdd(&deg[a], 1u);
    }
  }
  __syncthreads();
  if (inLds)
    for (int64_t k = threadIdx.x; k < nW; k += blockDim.x)
      if (sh[k]) atomicAdd(&deg[k], sh[k]);
}
__global__ void k_copy_deg(int64_t nSph, int64_t nW, const uint32_t* __restrict__ sdeg, uint32_t* deg) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < nSph) deg[nW + t] = sdeg[t];
}
// the boundary bodies' entries (other user id << 32 | slot | ADJ_PA) in arbitrary order within
// each body's range: a workgroup counts its entries per body in LDS, reserves one range per
// body with one atomic on the body's cursor (zeroed beforehand), and places them in it
__global__ __launch_bounds__(256) void k_wall_fill(int64_t nc, int64_t nW, const uint32_t* __restrict__ A,
                                                   const uint32_t* __restrict__ B, const uint32_t* __restrict__ info,
                                                   const uint32_t* __restrict__ uid,
                                                   const uint32_t* __restrict__ adjOff, uint32_t* cursor,
                                                   uint64_t* ent, int64_t n) {
  __shared__ uint32_t cnt[WD_LDS];
  if (adjOff[n] != (uint32_t)(2 * nc)) return;
  const bool inLds = nW <= WD_LDS;
  if (inLds)
    for (int64_t k = threadIdx.x; k < nW; k += blockDim.x) cnt[k] = 0u;
  __syncthreads();
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t lo = 0xFFFFFFFFu, loc = 0u;
  if (t < nc) {
    const uint32_t x = A[t];
    if (x < (uint32_t)nW) {
      lo = x;
      loc = inLds ? atomicAdd(&cnt[x], 1u) : atomicAdd(&cursor[x], 1u);
    }
  }
  __syncthreads();
  if (inLds)
    for (int64_t k = threadIdx.x; k < nW; k += blockDim.x)
      if (cnt[k]) cnt[k] = atomicAdd(&cursor[k], cnt[k]);
  __syncthreads();
  if (lo == 0xFFFFFFFFu) return;
  const uint32_t hi = B[t];
  const bool swap = (info[t] & CI_SWAP) != 0u;
  const uint32_t pos = (inLds ? cnt[lo] : 0u) + loc;
  ent[adjOff[lo] + pos] = ((uint64_t)uid[hi] << 32) | (uint32_t)t | (swap ? 0u : ADJ_PA);
}

// Each boundary body's entries sorted by the other particle's user id, in LDS by one workgroup
// (bitonic): lists up to WS_CAP entries; RW_LONGEST tells the host of longer ones. Instead of marks,
// scans, a gather, two to four radix passes and a scatter over all of them, with a wait for their
// number: 4 us for the walls of 2,000 spheres, 7 us for a floor under 60,000, against some 60.
constexpr int WS_BS = 512;
constexpr uint32_t WS_CAP = 4096;
__global__ __launch_bounds__(WS_BS) void k_wall_sort(const uint32_t* __restrict__ adjOff, int64_t n, uint32_t want,
                                                     const uint64_t* __restrict__ ent, uint32_t* __restrict__ adj) {
  __shared__ uint64_t key[WS_CAP];
  const uint32_t k0 = adjOff[blockIdx.x], m = adjOff[blockIdx.x + 1] - k0;
  if (adjOff[n] != want || m == 0u || m > WS_CAP) return;
  uint32_t P = 2u;
  while (P < m) P <<= 1;
  for (uint32_t t = threadIdx.x; t < P; t += WS_BS) key[t] = t < m ? ent[k0 + t] : ~0ull;
  __syncthreads();
  for (uint32_t size = 2u; size <= P; size <<= 1)
    for (uint32_t step = size >> 1; step > 0u; step >>= 1) {
      for (uint32_t t = threadIdx.x; t < (P >> 1); t += WS_BS) {
        const uint32_t a = 2u * t - (t & (step - 1u)), b = a + step;
        const bool up = (a & size) == 0u;
        const uint64_t x = key[a], y = key[b];
        if ((x > y) == up) {
          key[a] = y;
          key[b] = x;
        }
      }
      __syncthreads();
    }
  for (uint32_t t = threadIdx.x; t < m; t += WS_BS) adj[k0 + t] = (uint32_t)key[t];
}

// what the host needs of a finished refresh, to its pinned words; the displacement flag is cleared.
// staged: lists longer than k_wall_sort takes are not sorted yet (WALL_LONG stops k_ent_pos).
enum { RW_ENTRIES, RW_LONGEST, RW_GATHERED, RW_EXTRA, RW_ERR };
__global__ __launch_bounds__(256) void k_refresh_words(int64_t n, int64_t nW, int64_t nG,
                                                       const uint32_t* __restrict__ gbody,
                                                       const uint32_t* __restrict__ adjOff, int merged, int staged,
                                                       uint32_t* dflags, uint32_t* host) {
  __shared__ uint32_t wm[4][2];
  uint32_t all = 0u, ga = 0u;
  for (int64_t b = threadIdx.x; b < nW; b += 256) all = max(all, adjOff[b + 1] - adjOff[b]);
  for (int64_t q = threadIdx.x; q < nG; q += 256) ga = max(ga, adjOff[gbody[q] + 1] - adjOff[gbody[q]]);
  for (int off = 32; off > 0; off >>= 1) {
    all = max(all, (uint32_t)__shfl_xor(all, off));
    ga = max(ga, (uint32_t)__shfl_xor(ga, off));
  }
  if ((threadIdx.x & 63) == 0) {
    wm[threadIdx.x >> 6][0] = all;
    wm[threadIdx.x >> 6][1] = ga;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    all = max(max(wm[0][0], wm[1][0]), max(wm[2][0], wm[3][0]));
    ga = max(max(wm[0][1], wm[1][1]), max(wm[2][1], wm[3][1]));
    host[RW_ENTRIES] = adjOff[n];
    host[RW_LONGEST] = all;
    host[RW_GATHERED] = ga;
    host[RW_EXTRA] = merged ? dflags[6] : 0u;
    host[RW_ERR] = dflags[1];
    dflags[WALL_LONG] = staged && all > WS_CAP ? 1u : 0u;
    dflags[0] = 0u;
  }
}

// each particle's entries sorted by the other particle's user id (the order of
// Particle::contacts), then stripped to slot|ADJ_PA; lists longer than ADJ_INS (boundary
// bodies touching many spheres) are left to the radix-sort path below
constexpr uint32_t ADJ_INS = 64;
__global__ void k_adj_sort(int64_t n, uint32_t ins, const uint32_t* __restrict__ adjOff, uint64_t* ent, uint32_t* adj) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t k0 = adjOff[p], k1 = adjOff[p + 1];
  if (k1 - k0 > ins) return;
  for (uint32_t i = k0 + 1; i < k1; i++) {
    const uint64_t e = ent[i];
    uint32_t j = i;
    while (j > k0 && ent[j - 1] > e) {
      ent[j] = ent[j - 1];
      j--;
    }
    ent[j] = e;
  }
  for (uint32_t i = k0; i < k1; i++) adj[i] = (uint32_t)ent[i];
}

// long lists: their entries gathered into one array keyed (rank of the list, other user id),
// one radix sort, and scattered back; a list keeps its place, so the destination of sorted
// position i is that of unsorted position i
__global__ void k_big_mark(int64_t n, uint32_t ins, const uint32_t* __restrict__ adjOff, uint32_t* cnt,
                           uint32_t* flag) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t d = adjOff[p + 1] - adjOff[p];
  cnt[p] = d > ins ? d : 0u;
  flag[p] = d > ins ? 1u : 0u;
}
__global__ void k_big_list(int64_t n, uint32_t ins, const uint32_t* __restrict__ adjOff,
                           const uint32_t* __restrict__ bigRank, uint32_t* list) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n && adjOff[p + 1] - adjOff[p] > ins) list[bigRank[p]] = (uint32_t)p;
}
// one workgroup per long list
__global__ void k_big_gather(const uint32_t* __restrict__ list, const uint32_t* __restrict__ adjOff,
                             const uint32_t* __restrict__ bigOff, const uint64_t* __restrict__ ent, int uidBits,
                             uint64_t* key, uint32_t* val, uint32_t* dest) {
  const uint32_t p = list[blockIdx.x];
  const uint32_t k0 = adjOff[p], d = adjOff[p + 1] - k0;
  const uint32_t o = bigOff[p];
  const uint64_t r = (uint64_t)blockIdx.x << uidBits;
  for (uint32_t j = threadIdx.x; j < d; j += blockDim.x) {
    const uint64_t e = ent[k0 + j];
    key[o + j] = r | (e >> 32);
    val[o + j] = (uint32_t)e;
    dest[o + j] = k0 + j;
  }
}
__global__ void k_big_scatter(int64_t m, const uint32_t* __restrict__ val, const uint32_t* __restrict__ dest,
                              uint32_t* adj) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m) adj[dest[i]] = val[i];
}

// Adjacency of every sphere from its staged neighbours (no walls, no carried pairs that
// are not near): the slot of a neighbour after it is the next one the sphere generated;
// the slot of a neighbour before it is found among the few that neighbour generated.
// Entries are ranked by the other particle's user id (ids within a list are distinct).
struct AdjArgs {
  int64_t nSph, nW;
  const uint32_t *nb, *deg, *count, *off, *A, *B, *uid, *adjOff;
  uint64_t* ent;
  uint32_t* adj;
  uint32_t* dflags;
  uint32_t want;  // entries that the lists must hold
};
// Storage indices: boundary bodies [0, nW), spheres from nW; sphere t is storage nW + t and its
// generated pairs are off[t] .. off[t] + count[t]. Sphere p generated the pair with j when j is
// a boundary body or a sphere after it; its slots follow its neighbour order (the spheres
// above it, then the bodies).
__device__ __forceinline__ bool adj_generated(const AdjArgs& a, uint32_t p, uint32_t j) {
  return j > p || j < (uint32_t)a.nW;
}
// whether sphere p (user id up) is the contact's pA with neighbour j: a boundary body is always
// pA (the functor order Wall/Facet before Sphere), between spheres the smaller user id
__device__ __forceinline__ bool adj_is_pa(const AdjArgs& a, uint32_t up, uint32_t j, uint32_t uj) {
  return j >= (uint32_t)a.nW && up < uj;
}
// The entry of neighbour j of sphere p (storage): the slot of the pair (p's r-th generated one, or found
// among the pairs j generated), keyed by j's user id for the ranking. The slots lie in the order in which
// p staged its pairs, and so its neighbours, as long as one pass made both: a slot with another partner,
// like a pair found from one side only, is an error (bad), the entry kept in bounds. (The partner is
// compared last, so that its load is waited for together with the ids'.)
__device__ __forceinline__ uint64_t adj_entry(const AdjArgs& a, uint32_t p, uint32_t j, uint32_t r, bool& bad) {
  const bool own = adj_generated(a, p, j);
  uint32_t slot = own ? a.off[p - a.nW] + r : find_partner(a.B, a.off[j - a.nW], a.count[j - a.nW], p);
  const bool in = slot < a.want / 2u;
  if (!in) slot = 0u;
  const uint32_t partner = own ? (j < (uint32_t)a.nW ? a.A : a.B)[slot] : j;
  const uint32_t uj = a.uid[j], up = a.uid[p];
  const uint64_t e = ((uint64_t)uj << 32) | slot | (adj_is_pa(a, up, j, uj) ? ADJ_PA : 0u);
  bad = bad || !in || partner != j;
  return e;
}

// Each sphere's adjacency ranked by the neighbour's user id. The 64 spheres of a wavefront own
// one contiguous range of entries: the lanes take its entries in turn (every 64th), so a
// sphere with many neighbours does not hold up the others. Entry (sphere p, q-th neighbour j):
// the slot is generated by p when j > p (the next one after p's earlier neighbours above p),
// else found among j's generated pairs; the key (user id of j, slot) is ranked among p's
// keys in LDS. A wavefront with more than ADJ_CAP entries takes each sphere's list in one
// thread, through HBM (a.ent).
constexpr int ADJ_CAP = 640, ADJ_WAVES = 4;
__global__ __launch_bounds__(64 * ADJ_WAVES) void k_adj_sym(AdjArgs a) {
  __shared__ uint32_t so[ADJ_WAVES][65];
  __shared__ uint32_t sj[ADJ_WAVES][ADJ_CAP];
  __shared__ uint64_t se[ADJ_WAVES][ADJ_CAP];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // the wavefront's first sphere
  const int64_t tw = ((int64_t)xcd_block(blockIdx.x, gridDim.x) * ADJ_WAVES + w) * 64;
  if (tw >= a.nSph) return;  // whole wavefront; no workgroup barrier below
  if (a.adjOff[a.nW + a.nSph] != a.want) return;
  const int64_t t = tw + lane;
  const bool live = t < a.nSph;
  const uint32_t m = live ? a.deg[t] : 0u, k0 = live ? a.adjOff[a.nW + t] : 0u;
  const uint32_t kb = __shfl(k0, 0);
  uint32_t end = live ? k0 + m : 0u;
  for (int d = 32; d > 0; d >>= 1) end = max(end, (uint32_t)__shfl_xor(end, d));
  const uint32_t E = end - kb;
  so[w][lane] = (live ? k0 : end) - kb;
  if (lane == 0) so[w][64] = E;
  wave_lds_sync();
  // the sphere (lane L of the wavefront) owning entry e, and e's index q in its list
  auto owner = [&](uint32_t e, int& L, uint32_t& q) {
    L = 0;
    for (int step = 32; step > 0; step >>= 1)
      if (L + step < 64 && so[w][L + step] <= e) L += step;
    q = e - so[w][L];
  };
  // the wavefront's spheres in runs whose entries fit the LDS arrays; a sphere with more
  // entries than fit takes its list alone in one thread, through HBM (a.ent)
  bool bad = false;
  int L0 = 0;
  while (L0 < 64) {
    int L1 = L0 + 1;
    while (L1 < 64 && so[w][L1 + 1] - so[w][L0] <= (uint32_t)ADJ_CAP) L1++;
    const uint32_t E0 = so[w][L0], E1 = so[w][L1];
    if (E1 - E0 > (uint32_t)ADJ_CAP) {
      if (lane == L0) {
        const uint32_t p = (uint32_t)(a.nW + t);
        uint32_t gen = 0;
        for (uint32_t q = 0; q < m; q++) {
          const uint32_t j = a.nb[(int64_t)q * a.nSph + t];
          a.ent[k0 + q] = adj_entry(a, p, j, gen, bad);
          gen += adj_generated(a, p, j) ? 1u : 0u;
        }
        for (uint32_t q = 0; q < m; q++) {
          const uint64_t e = a.ent[k0 + q];
          uint32_t r = 0;
          for (uint32_t v = 0; v < m; v++) r += a.ent[k0 + v] < e ? 1u : 0u;
          a.adj[k0 + r] = (uint32_t)e;
        }
      }
      L0 = L1;
      continue;
    }
    // neighbours of the entries
    for (uint32_t e = E0 + lane; e < E1; e += 64) {
      int L;
      uint32_t q;
      owner(e, L, q);
      sj[w][e - E0] = a.nb[(int64_t)q * a.nSph + tw + L];
    }
    wave_lds_sync();
    // keys (user id of the neighbour, slot, role)
    for (uint32_t e = E0 + lane; e < E1; e += 64) {
      int L;
      uint32_t q;
      owner(e, L, q);
      const uint32_t p = (uint32_t)(a.nW + tw + L), j = sj[w][e - E0], b0 = so[w][L] - E0;
      uint32_t r = 0;
      if (adj_generated(a, p, j))
        for (uint32_t v = 0; v < q; v++) r += adj_generated(a, p, sj[w][b0 + v]) ? 1u : 0u;
      se[w][e - E0] = adj_entry(a, p, j, r, bad);
    }
    wave_lds_sync();
    // rank among the sphere's keys (distinct: one entry per neighbour)
    for (uint32_t e = E0 + lane; e < E1; e += 64) {
      int L;
      uint32_t q;
      owner(e, L, q);
      const uint32_t b0 = so[w][L] - E0, b1 = so[w][L + 1] - E0;
      const uint64_t key = se[w][e - E0];
      uint32_t r = 0;
      for (uint32_t v = b0; v < b1; v++) r += se[w][v] < key ? 1u : 0u;
      a.adj[kb + E0 + b0 + r] = (uint32_t)key;
    }
    // the next run overwrites the arrays
    wave_lds_sync();
    L0 = L1;
  }
  if (__any(bad) && lane == 0) atomicOr(&a.dflags[1], ERR_ADJ);
}

// the inverse of the adjacency: per slot the positions of its pA entry and its pB entry; every
// entry starts at NO_STATE, and the next filter writes those of every real slot
__global__ void k_ent_pos(int64_t nEnt, const uint32_t* __restrict__ adj, const uint32_t* __restrict__ total,
                          uint32_t* entPos, uint32_t* eidx, uint32_t* dflags) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (*total != (uint32_t)nEnt || dflags[WALL_LONG] != 0u) return;
  if (e == 0) dflags[EIDX_FULL] = 1u;
  if (e >= nEnt) return;
  const uint32_t v = adj[e];
  entPos[2 * (int64_t)(v & ~ADJ_PA) + ((v & ADJ_PA) ? 0 : 1)] = (uint32_t)e;
  eidx[e] = NO_STATE;
}

// ------------------------------------------------------------------ host side
static void check_device_errors(Ctx& c, uint32_t err) {
  if (err & ERR_DOUBLE_IMAGE)
    throw Error(WDG_E_GEOM, "InsertionSortCollider: a pair overlaps through two periodic images "
                            "(particle larger than half of the cell?)");
  if (err & ERR_NAN_FORCE) throw Error(WDG_E_NUMERIC, "NaN force in contact");
  if (err & ERR_CD_RANGE) throw Error(WDG_E_GEOM, "periodic cell distance out of range");
  if (err & ERR_ADJ) throw Error(WDG_E_STATE, "broadphase: a pair was found from one side only");
  if (err & ERR_FACET)
    throw Error(WDG_E_GEOM, "Cg2_Facet_Sphere_L6Geom: impossible sphere-facet intersection (degenerate facet?)");
  if (err & ERR_SNAP_IMAGE)
    throw Error(WDG_E_GEOM, "snapshot: a saved contact's periodic image differs from the refreshed pair's");
}

// error bits that the host has read (nothing is queued on the stream): cleared, in the leapfrog's pinned
// copy too, so that each is reported once, and raised
static void take_errors(Ctx& c, uint32_t err) {
  if (!err) return;
  WDG_HIP(hipMemsetAsync(c.dflags.p + 1, 0, sizeof(uint32_t), c.stream));
  c.hflags[HOST_ERR] = 0u;
  check_device_errors(c, err);
}

void check_errors(Ctx& c) { take_errors(c, read_u32(c, c.dflags.p + 1)); }

void drop_contacts(Ctx& c) {
  for (auto& s : c.C) {
    s.n = 0;
    s.ensure(0, c.n, c.field.periodic != 0);
    WDG_HIP(hipMemsetAsync(s.adjOff.p, 0, (c.n + 1) * sizeof(uint32_t), c.stream));
  }
  for (auto& r : c.R) {
    r.ensure(0);
    r.sidxValid = false;
    WDG_HIP(hipMemsetAsync(r.tpre.p, 0, sizeof(uint32_t), c.stream));
  }
  c.boundsValid = false;
  c.eidxValid = false;
  c.eidxClean = false;
  c.dirtyKnown = false;
  c.forcesPending = false;
  c.rollActive = false;
  c.grid.valid = false;
}

void clear_history(Ctx& c) {
  if (c.forcesPending) flush_forces(c);
  Contacts& C = c.con();
  Reals& R = c.reals();
  if (C.n > 0) {
    const int64_t g = ngroups(C.n);
    WDG_HIP(hipMemsetAsync(R.bits.p, 0, (size_t)g * (GROUP / 64) * sizeof(unsigned long long), c.stream));
    WDG_HIP(hipMemsetAsync(R.tpre.p, 0, (size_t)g * (GROUP / TILE) * sizeof(uint32_t), c.stream));
    WDG_HIP(hipMemsetAsync(R.gcnt.p, 0, (size_t)g * sizeof(uint32_t), c.stream));
  }
  R.sidxValid = false;
  // the per-entry real slots name contacts that are gone
  c.eidxValid = false;
  c.eidxClean = false;
}

static PairArgs pair_args(Ctx& c, const Grid& g, const AabbParams& P) {
  PairArgs pa{};
  pa.nW = c.nW; pa.n = c.n; pa.key = c.cellKey.p;
  pa.px = c.lastPos[0].p; pa.py = c.lastPos[1].p; pa.pz = c.lastPos[2].p; pa.rad = c.radius.p;
  pa.mask = c.mask.p; pa.uid = c.uid.p; pa.flags = c.flags.p;
  pa.scene = c.nScenes > 0 ? c.scene.p : nullptr;
  if (c.nScenes > 0 && c.nW > 0) {
    pa.sceneBodyOff = c.sceneBodyOff.p;
    pa.sceneBody = c.sceneBody.p;
  }
  pa.cbeg = c.cellStart.p; pa.g = g; pa.P = P; pa.brute = c.grid.brute;
  pa.count = c.scount.p; pa.off = c.soff.p; pa.dflags = c.dflags.p;
  pa.pf = c.posf.p;
  pa.bnd = c.bnd.p;
  pa.vdS = c.vdSceneActive ? c.vdScene.p : nullptr;
  pa.nSph = c.n - c.nW;
  // float positions are grid-relative, at most ext in magnitude; 1e-5*ext is ~80 float ulps
  double ext = 0;
  for (int k = 0; k < 3; k++) ext = std::max(ext, g.periodic ? g.L[k] : g.nc[k] * g.h[k]);
  pa.margin = (float)(1e-5 * ext + 1e-30);
  return pa;
}

static void sort_lists(Ctx& c, Contacts& N, int64_t np, uint32_t ins);
// general adjacency: entry counts and placement with atomics, then a sort of every list
static void build_adjacency_atomic(Ctx& c, Contacts& N, int64_t nNew) {
  const int64_t n = c.n;
  c.adjDeg.ensure(n + 1);
  WDG_HIP(hipMemsetAsync(c.adjDeg.p, 0, n * sizeof(uint32_t), c.stream));
  if (nNew > 0) {
    hipLaunchKernelGGL(k_adj_deg, dim3(nblocks(nNew, 256)), dim3(256), 0, c.stream, nNew, (const uint32_t*)N.A.p,
                       (const uint32_t*)N.B.p, c.adjDeg.p);
    WDG_LAUNCH_CHECK();
  }
  scan_exclusive(c, c.adjDeg.p, N.adjOff.p, n, N.adjOff.p + n);
  if (nNew > 0) {
    c.adjEnt.ensure(2 * nNew);
    hipLaunchKernelGGL(k_adj_fill, dim3(nblocks(nNew, 256)), dim3(256), 0, c.stream, nNew, (const uint32_t*)N.A.p,
                       (const uint32_t*)N.B.p, (const uint32_t*)N.info.p, (const uint32_t*)c.uid.p,
                       (const uint32_t*)N.adjOff.p, c.adjDeg.p, c.adjEnt.p);
    WDG_LAUNCH_CHECK();
    sort_lists(c, N, n, ADJ_INS);
  }
}

// the entries of particles [0, np) (in c.adjEnt, within N.adjOff) sorted into N.adj: lists of
// at most `ins` entries by insertion in one thread each, longer ones by one radix sort
static void sort_lists(Ctx& c, Contacts& N, int64_t np, uint32_t ins) {
  const int64_t n = np;
  {
    if (ins > 0) {
      hipLaunchKernelGGL(k_adj_sort, dim3(nblocks(n, 256)), dim3(256), 0, c.stream, n, ins,
                         (const uint32_t*)N.adjOff.p, c.adjEnt.p, N.adj.p);
      WDG_LAUNCH_CHECK();
    }
    // lists longer than ADJ_INS
    c.bigOff.ensure(n + 1);
    c.bigRank.ensure(n + 1);
    hipLaunchKernelGGL(k_big_mark, dim3(nblocks(n, 256)), dim3(256), 0, c.stream, n, ins, (const uint32_t*)N.adjOff.p,
                       c.adjDeg.p, c.bigRank.p);
    WDG_LAUNCH_CHECK();
    scan_exclusive(c, c.adjDeg.p, c.bigOff.p, n, c.dflags.p + 16);
    scan_exclusive(c, c.bigRank.p, c.bigRank.p, n, c.dflags.p + 17);
    WDG_HIP(hipMemcpyAsync(c.hflags + 16, c.dflags.p + 16, 2 * sizeof(uint32_t), hipMemcpyDeviceToHost, c.stream));
    WDG_HIP(hipStreamSynchronize(c.stream));
    const int64_t m = c.hflags[16], nBig = c.hflags[17];
    if (m > 0) {
      c.bigKey.ensure(m); c.bigKeyTmp.ensure(m);
      c.bigVal.ensure(m); c.bigValTmp.ensure(m); c.bigDest.ensure(m);
      // the key holds the other particle's user id: any particle of the context
      const int uidBits = bits_for((uint64_t)(c.n > 1 ? c.n - 1 : 1));
      const int rankBits = bits_for((uint64_t)(nBig > 1 ? nBig - 1 : 1));
      c.bigList.ensure(nBig);
      hipLaunchKernelGGL(k_big_list, dim3(nblocks(n, 256)), dim3(256), 0, c.stream, n, ins, (const uint32_t*)N.adjOff.p,
                         (const uint32_t*)c.bigRank.p, c.bigList.p);
      WDG_LAUNCH_CHECK();
      hipLaunchKernelGGL(k_big_gather, dim3((unsigned)nBig), dim3(256), 0, c.stream, (const uint32_t*)c.bigList.p,
                         (const uint32_t*)N.adjOff.p, (const uint32_t*)c.bigOff.p, (const uint64_t*)c.adjEnt.p,
                         uidBits, c.bigKey.p, c.bigVal.p, c.bigDest.p);
      WDG_LAUNCH_CHECK();
      radix_sort_pairs<uint64_t>(c, c.bigKey.p, c.bigVal.p, c.bigKeyTmp.p, c.bigValTmp.p, m, uidBits + rankBits);
      hipLaunchKernelGGL(k_big_scatter, dim3(nblocks(m, 256)), dim3(256), 0, c.stream, m, (const uint32_t*)c.bigVal.p,
                         (const uint32_t*)c.bigDest.p, N.adj.p);
      WDG_LAUNCH_CHECK();
    }
  }
}

static void refresh(Ctx& c) {
  const int64_t n = c.n, nW = c.nW, nSph = n - nW;
  c.gen++;
  if (c.maxScene >= std::max<int64_t>(c.nScenes, 1))
    throw Error(WDG_E_ARG, "a particle's scene index is not below the number of scenes (wdg_set_scenes)");
  const double vd = c.verletDist;
  const bool periodic = c.field.periodic != 0;
  if (periodic && c.nFacet > 0) throw Error(WDG_E_ARG, "facets in a periodic scene are not supported");
  c.nRefresh++;

  // per-scene skins (batched scenes, tuning.skinSteps > 0): each scene's Verlet distance
  // covers what its fastest sphere moves in skinSteps of its steps (speed now, plus gravity's
  // pull over that time), times 1.25, between the context's Verlet distance and rmin
  const bool perScene = c.nScenes > 0 && c.tune.skinSteps > 0 && nSph > 0 && vd > 0;
  double vdMax = vd;
  c.vdSceneActive = false;
  std::vector<double> vdHost;  // the per-scene skins on the host (empty: vd everywhere)
  if (perScene) {
    const int64_t ns = std::max<int64_t>(c.nScenes, c.maxScene + 1);
    c.vdScene.ensure((size_t)ns);
    c.sceneVmax.ensure((size_t)ns);
    unsigned long long* dv = reinterpret_cast<unsigned long long*>(c.sceneVmax.p);
    WDG_HIP(hipMemsetAsync(dv, 0, ns * sizeof(unsigned long long), c.stream));
    hipLaunchKernelGGL(k_scene_vmax, dim3(nblocks(nSph, 256)), dim3(256), 0, c.stream, nW, n, ns, c.vel[0].p,
                       c.vel[1].p, c.vel[2].p, c.scene.p, dv);
    WDG_LAUNCH_CHECK();
    std::vector<unsigned long long> hv((size_t)ns);
    std::vector<double> hdt((size_t)ns);
    WDG_HIP(hipMemcpyAsync(hv.data(), dv, ns * sizeof(unsigned long long), hipMemcpyDeviceToHost, c.stream));
    WDG_HIP(hipMemcpyAsync(hdt.data(), c.dtScene.p, ns * sizeof(double), hipMemcpyDeviceToHost, c.stream));
    WDG_HIP(hipStreamSynchronize(c.stream));
    const double gmag = std::sqrt(c.field.gravity[0] * c.field.gravity[0] + c.field.gravity[1] * c.field.gravity[1] +
                                  c.field.gravity[2] * c.field.gravity[2]);
    std::vector<double>& vs = vdHost;
    vs.assign((size_t)ns, vd);
    for (int64_t k = 0; k < ns; k++) {
      double v2;
      std::memcpy(&v2, &hv[k], sizeof(double));
      const double t = c.tune.skinSteps * hdt[k];
      const double d = 1.25 * (std::sqrt(v2) * t + 0.5 * gmag * t * t);
      vs[k] = std::min(std::max(d, vd), std::max(vd, 0.5 * c.rmin));
      vdMax = std::max(vdMax, vs[k]);
    }
    WDG_HIP(hipMemcpyAsync(c.vdScene.p, vs.data(), ns * sizeof(double), hipMemcpyHostToDevice, c.stream));
    WDG_HIP(hipStreamSynchronize(c.stream));
    c.vdSceneActive = true;
  }
  const double* vdS = c.vdSceneActive ? c.vdScene.p : nullptr;

  // grid: cell edge >= largest enlarged-AABB extent
  Grid g{};
  g.periodic = periodic;
  double absDf = std::fabs(c.field.distFactor);
  double ext = 2. * (absDf * c.rmax + vdMax);
  ext = ext * (1 + 1e-9) + 1e-300;
  bool brute = nSph < 512;
  if (periodic) {
    for (int k = 0; k < 3; k++) {
      g.L[k] = c.field.cell[k];
      g.nc[k] = (int)std::floor(g.L[k] / ext);
      if (g.nc[k] < 3) brute = true;
      g.nc[k] = std::max(g.nc[k], 1);
      g.h[k] = g.L[k] / g.nc[k];
      g.org[k] = 0;
    }
  } else if (nSph > 0) {
    const int nbb = (int)std::min<int64_t>(nblocks(nSph, 256), BBOX_BLOCKS);
    c.obsPart.ensure((size_t)6 * BBOX_BLOCKS);
    unsigned long long* dbb = reinterpret_cast<unsigned long long*>(c.obsPart.p);
    hipLaunchKernelGGL(k_bbox, dim3((unsigned)nbb), dim3(256), 0, c.stream, nW, n, c.pos[0].p, c.pos[1].p, c.pos[2].p,
                       dbb);
    WDG_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_bbox_all, dim3(1), dim3(384), 0, c.stream, nbb, (const unsigned long long*)dbb,
                       reinterpret_cast<unsigned long long*>(c.hresDev));
    WDG_LAUNCH_CHECK();
    WDG_HIP(hipStreamSynchronize(c.stream));
    unsigned long long hb[6];
    std::memcpy(hb, c.hres, sizeof(hb));
    double lo[3], hi[3];
    for (int k = 0; k < 3; k++) {
      lo[k] = ord_to_double(hb[k]);
      hi[k] = ord_to_double(hb[3 + k]);
    }
    // cells of the largest enlarged AABB; when the bounding box holds far more of them than
    // there are spheres (a spread-out scene), the cells are hashed into buckets instead of
    // growing (which would put more and more spheres into each cell)
    double h = ext;
    for (int k = 0; k < 3; k++)
      while (std::floor((hi[k] - lo[k]) / h) + 1 > 1e6) h *= 2;
    double cells = 1;
    for (int k = 0; k < 3; k++) {
      g.h[k] = h;
      g.nc[k] = (int)(std::floor((hi[k] - lo[k]) / h) + 1);
      cells *= g.nc[k];
    }
    if (cells > std::max(8.0 * nSph, 4096.0)) {
      g.hashed = 1;
      uint32_t m = 4096;
      while ((double)m < 2.0 * nSph && m < (1u << 30)) m <<= 1;
      g.hmask = m - 1;
    }
    for (int k = 0; k < 3; k++) g.org[k] = lo[k];
  }
  int64_t ncells = g.hashed ? (int64_t)g.hmask + 1 : (int64_t)g.nc[0] * g.nc[1] * g.nc[2];
  // batched aperiodic scenes: a grid per scene over its own bounding box, cells as large as its
  // own largest enlarged AABB (a dense grid of the whole layout would cover the gaps between
  // scenes and take the largest skin of all); keys scene by scene
  g.sg = nullptr;
  if (c.nScenes > 0 && !periodic && !brute && nSph > 0) {
    const int64_t ns = std::max<int64_t>(c.nScenes, c.maxScene + 1);
    std::vector<unsigned long long> hb((size_t)7 * ns);
    for (int64_t k = 0; k < ns; k++) {
      for (int q = 0; q < 3; q++) { hb[7 * k + q] = ~0ull; hb[7 * k + 3 + q] = 0ull; }
      hb[7 * k + 6] = 0ull;
    }
    c.sceneBox.ensure(hb.size());
    WDG_HIP(hipMemcpyAsync(c.sceneBox.p, hb.data(), hb.size() * 8, hipMemcpyHostToDevice, c.stream));
    hipLaunchKernelGGL(k_scene_bbox, dim3(nblocks(nSph, 256)), dim3(256), 0, c.stream, nW, n, ns, c.pos[0].p,
                       c.pos[1].p, c.pos[2].p, (const uint32_t*)c.scene.p, c.sceneBox.p);
    WDG_LAUNCH_CHECK();
    WDG_HIP(hipMemcpyAsync(hb.data(), c.sceneBox.p, hb.size() * 8, hipMemcpyDeviceToHost, c.stream));
    WDG_HIP(hipStreamSynchronize(c.stream));
    std::vector<SceneGrid> sgh((size_t)ns);
    int64_t total = 0;
    for (int64_t k = 0; k < ns; k++) {
      SceneGrid& G = sgh[k];
      const double cnt = (double)hb[7 * k + 6];
      const double vdk = vdHost.empty() ? vd : vdHost[k];
      double h = (2. * (absDf * c.rmax + vdk)) * (1 + 1e-9) + 1e-300;
      double lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
      if (cnt > 0)
        for (int q = 0; q < 3; q++) {
          lo[q] = ord_to_double(hb[7 * k + q]);
          hi[q] = ord_to_double(hb[7 * k + 3 + q]);
        }
      int64_t cells = 1;
      for (int it = 0; it < 200; it++) {
        double cl = 1;
        for (int q = 0; q < 3; q++) cl *= std::min(1e6, std::floor((hi[q] - lo[q]) / h) + 1);
        if (cl <= std::max(8.0 * cnt, 64.0)) {
          cells = (int64_t)cl;
          break;
        }
        h *= 1.25;
      }
      G.h = h;
      for (int q = 0; q < 3; q++) {
        G.org[q] = lo[q];
        G.nc[q] = (int)std::min(1e6, std::floor((hi[q] - lo[q]) / h) + 1);
      }
      cells = (int64_t)G.nc[0] * G.nc[1] * G.nc[2];
      G.off = (uint32_t)total;
      total += cells;
    }
    if (total < ((int64_t)1 << 31)) {
      c.sgrid.ensure(sgh.size() * sizeof(SceneGrid));
      WDG_HIP(hipMemcpyAsync(c.sgrid.p, sgh.data(), sgh.size() * sizeof(SceneGrid), hipMemcpyHostToDevice,
                             c.stream));
      g.sg = reinterpret_cast<const SceneGrid*>(c.sgrid.p);
      g.hashed = 0;
      ncells = total;
    }
  }

  // one dense grid: Morton keys when the code range stays within a few times the sphere count
  g.morton = 0;
  if (c.cellMorton && !g.hashed && !g.sg && !brute && nSph > 0) {
    int bits = 0;
    while ((1 << bits) < std::max(g.nc[0], std::max(g.nc[1], g.nc[2]))) bits++;
    if (bits <= 10 && g.nc[0] >= 3 && g.nc[1] >= 3 && g.nc[2] >= 3 &&
        ((int64_t)1 << (3 * bits)) <= std::max<int64_t>(16 * nSph, 4096)) {
      g.morton = 1;
      ncells = (int64_t)1 << (3 * bits);
    }
  }

  AabbParams P{};
  P.vd = vd;
  P.absDf = absDf;
  P.loneMask = c.field.loneMask;
  P.periodic = periodic;
  for (int k = 0; k < 3; k++) P.L[k] = c.field.cell[k];

  // 1. spatial order of the spheres and the permutation of all particle arrays
  c.cellKey.ensure(nSph + 1); c.sortIdx.ensure(nSph + 1);
  c.cellKeyTmp.ensure(nSph + 1); c.sortIdxTmp.ensure(nSph + 1);
  c.perm.ensure(n + 1); c.invPerm.ensure(n + 1);
  c.scount.ensure(nSph + 1); c.soff.ensure(nSph + 1);
  // by counting while the cells are no more than a few per sphere (a scan over them is then
  // cheaper than the passes of a sort), else by sorting the keys: a periodic cell that is nearly
  // empty. All-pairs keeps the order.
  const bool counting = !brute && nSph > 0 && ncells <= std::max<int64_t>(16 * nSph, 4096);
  if (nSph > 0) {
    Grid gk = g;
    if (brute) {
      for (int k = 0; k < 3; k++) { gk.nc[k] = 1; gk.h[k] = 1e300; gk.org[k] = 0; }
      gk.periodic = 0;
      gk.hashed = 0;
      gk.sg = nullptr;
    }
    uint32_t* cnt = nullptr;
    if (counting) {
      c.cellCnt.ensure(ncells + 1);  // and a zero after them, so that the scan also gives the end
      c.cellStart.ensure(ncells + 1);
      c.cellRank.ensure(nSph + 1);
      WDG_HIP(hipMemsetAsync(c.cellCnt.p, 0, (ncells + 1) * sizeof(uint32_t), c.stream));
      cnt = c.cellCnt.p;
    }
    uint32_t* key = counting ? c.cellKeyTmp.p : c.cellKey.p;
    hipLaunchKernelGGL(k_keys, dim3(nblocks(nSph, 256)), dim3(256), 0, c.stream, nW, n, c.pos[0].p, c.pos[1].p,
                       c.pos[2].p, gk, (const uint32_t*)c.scene.p, key, c.sortIdx.p, cnt, c.cellRank.p);
    WDG_LAUNCH_CHECK();
    if (counting) {
      scan_exclusive(c, c.cellCnt.p, c.cellStart.p, ncells + 1, c.dflags.p + 3, (uint32_t)nW);
      const uint32_t* cb = c.cellStart.p;
      hipLaunchKernelGGL(k_cell_place, dim3(nblocks(nSph, 256)), dim3(256), 0, c.stream, nSph, nW,
                         (const uint32_t*)key, (const uint32_t*)c.cellRank.p, cb, c.sortIdx.p);
      WDG_LAUNCH_CHECK();
      hipLaunchKernelGGL(k_cell_rank, dim3(nblocks(n, 256)), dim3(256), 0, c.stream, n, nW, (const uint32_t*)key, cb,
                         (const uint32_t*)c.sortIdx.p, c.perm.p, c.invPerm.p, c.cellKey.p);
      WDG_LAUNCH_CHECK();
    } else if (!brute) {
      radix_sort_pairs<uint32_t>(c, c.cellKey.p, c.sortIdx.p, c.cellKeyTmp.p, c.sortIdxTmp.p, nSph,
                                 bits_for((uint64_t)(ncells > 1 ? ncells - 1 : 1)));
    }
  }
  if (!counting) {
    hipLaunchKernelGGL(k_build_perm, dim3(nblocks(n, 256)), dim3(256), 0, c.stream, nW, n, c.sortIdx.p, c.perm.p,
                       c.invPerm.p);
    WDG_LAUNCH_CHECK();
  }
  {
    PermArgs pa{};
    pa.n = n;
    pa.perm = c.perm.p;
    DBuf<double>* d[NPD] = {&c.pos[0], &c.pos[1], &c.pos[2], &c.vel[0], &c.vel[1], &c.vel[2], &c.angVel[0],
                            &c.angVel[1], &c.angVel[2], &c.ori[0], &c.ori[1], &c.ori[2], &c.ori[3], &c.force[0],
                            &c.force[1], &c.force[2], &c.torque[0], &c.torque[1], &c.torque[2], &c.inertia[0],
                            &c.inertia[1], &c.inertia[2], &c.mass, &c.radius};
    DBuf<uint32_t>* u[NPU] = {&c.flags, &c.mask, &c.uid, reinterpret_cast<DBuf<uint32_t>*>(&c.mat), &c.scene};
    for (int k = 0; k < NPD; k++) {
      c.spareD[k].ensure(n + 1);
      pa.sd[k] = d[k]->p;
      pa.dd[k] = c.spareD[k].p;
    }
    for (int k = 0; k < NPU; k++) {
      c.spareU[k].ensure(n + 1);
      pa.su[k] = u[k]->p;
      pa.du[k] = c.spareU[k].p;
    }
    c.posf.ensure(n + 1);
    pa.g = g;
    pa.absDf = absDf;
    pa.vd0 = vd;
    pa.vdS = vdS;
    pa.lx = c.lastPos[0].p; pa.ly = c.lastPos[1].p; pa.lz = c.lastPos[2].p;
    pa.pf = c.posf.p;
    pa.sto = c.sto.p;
    hipLaunchKernelGGL(k_permute, dim3(nblocks(n, 256)), dim3(256), 0, c.stream, pa);
    WDG_LAUNCH_CHECK();
    for (int k = 0; k < NPD; k++) d[k]->swap(c.spareD[k]);
    for (int k = 0; k < NPU; k++) u[k]->swap(c.spareU[k]);
  }
  if (nW > 0) {
    c.bnd.ensure((size_t)6 * nW);
    hipLaunchKernelGGL(k_bnd_bounds, dim3(nblocks(nW, 256)), dim3(256), 0, c.stream, nW, c.lastPos[0].p,
                       c.lastPos[1].p, c.lastPos[2].p, c.flags.p, c.fgeo.p, vd, vdS, (const uint32_t*)c.scene.p,
                       c.bnd.p);
    WDG_LAUNCH_CHECK();
  }
  if (nSph > 0 && !brute && !counting) {
    c.cellStart.ensure(ncells + 1);
    hipLaunchKernelGGL(k_cell_begin, dim3(nblocks(ncells + 1, 256)), dim3(256), 0, c.stream, nSph, nW, c.cellKey.p,
                       ncells, c.cellStart.p);
    WDG_LAUNCH_CHECK();
  }
  for (int k = 0; k < 3; k++) {
    c.grid.org[k] = g.org[k]; c.grid.h[k] = g.h[k]; c.grid.L[k] = g.L[k]; c.grid.nc[k] = g.nc[k];
  }
  c.grid.periodic = periodic;
  c.grid.hashed = g.hashed;
  c.grid.hmask = g.hmask;
  c.grid.morton = g.morton;
  c.grid.sg = g.sg;
  c.grid.brute = brute;
  c.grid.valid = true;

  // 2. pairs that can touch before the next refresh, staged per generating sphere
  PairArgs pa = pair_args(c, g, P);
  int64_t nPairs = 0;
  bool overflow = false, nbFits = false;
  c.sdeg.ensure(nSph + 1);
  if (nSph > 0) {
    // a sphere that generated more pairs than staged makes the pair pass run again in place;
    // after that the next refreshes stage more (up to 96 per sphere)
    const int PS = c.pairStage;
    c.stPartner.ensure(nSph * PS);
    c.stInfo.ensure(nSph * PS);
    if (periodic) c.stDist.ensure(nSph * PS);
    pa.stage = PS;
    const int NS = c.nbStage;
    c.stNb.ensure(nSph * NS);
    pa.nbStage = NS;
    pa.sA = c.stPartner.p; pa.sInfo = c.stInfo.p; pa.sDist = c.stDist.p;
    pa.deg = c.sdeg.p; pa.nb = c.stNb.p;
    const int64_t npb = nblocks(nSph * pair_lanes(nSph), 256);
    c.pairMax.ensure(2 * npb);
    pa.bmax = c.pairMax.p;
    launch_pairs<OUT_STAGE, MODE_NEAR>(c, pa);
    scan_exclusive(c, c.scount.p, c.soff.p, nSph, c.dflags.p + 4);
    hipLaunchKernelGGL(k_block_max, dim3(1), dim3(1024), 0, c.stream, npb, (const uint32_t*)c.pairMax.p, c.dflags.p,
                       c.hflagsDev);
    WDG_LAUNCH_CHECK();
    WDG_HIP(hipStreamSynchronize(c.stream));
    nPairs = c.hflags[4];
    overflow = c.hflags[7] > (uint32_t)PS;
    if (overflow) c.pairStage = (int)std::min<uint32_t>(96u, (c.hflags[7] + 7u) / 8u * 8u);
    // (pairs generated again in place: the passes that stage and that do not work off their queues in
    // different rounds, so the staged neighbours do not tell the slots' order then, and k_adj_sym, which
    // takes a sphere's slots in that order, would give entries of other pairs)
    nbFits = !overflow && c.hflags[8] <= (uint32_t)NS;
    // a sphere with more neighbours than staged sends the adjacency to the general path; the
    // next refreshes stage more (up to 128)
    if (c.hflags[8] > (uint32_t)NS) c.nbStage = (int)std::min<uint32_t>(128u, (c.hflags[8] + 7u) / 8u * 8u);
  }
  Contacts& O = c.con();
  const int64_t nOld = O.n;
  Contacts& N = c.C[1 - c.cur];
  // room for the old real contacts that are no longer near (appended by the merge)
  N.ensure(nPairs + nOld, n, periodic);
  if (nPairs > 0) {
    if (!overflow) {
      hipLaunchKernelGGL(k_unstage, dim3(nblocks(nSph, US_BS)), dim3(US_BS), 0, c.stream, nW, nSph,
                         (const uint32_t*)c.scount.p, (const uint32_t*)c.soff.p, (const uint32_t*)c.stPartner.p,
                         (const uint32_t*)c.stInfo.p, (const uint64_t*)c.stDist.p, (int)periodic, N.A.p, N.B.p,
                         N.info.p, N.dist.p, N.carry.p);
    } else {
      // a sphere generated more pairs than the staging area holds: generate again, in place
      pa.sA = N.A.p; pa.sB = N.B.p; pa.sInfo = N.info.p; pa.sCarry = N.carry.p; pa.sDist = N.dist.p;
      launch_pairs<OUT_SLOTS, MODE_NEAR>(c, pa);
    }
    WDG_LAUNCH_CHECK();
  }
  // 3. merge with the old real contacts (history)
  const bool merged = nOld > 0 && nSph > 0;
  if (merged) {
    MergeArgs ma{};
    ma.nOld = nOld; ma.nW = nW; ma.nPairs = nPairs; ma.ov = c.rview();
    ma.oA = O.A.p; ma.oB = O.B.p; ma.oInfo = O.info.p; ma.oDist = O.dist.p; ma.invPerm = c.invPerm.p;
    ma.count = c.scount.p; ma.off = c.soff.p; ma.periodic = periodic;
    ma.A = N.A.p; ma.B = N.B.p; ma.info = N.info.p; ma.carry = N.carry.p; ma.dist = N.dist.p;
    ma.nExtra = c.dflags.p + 6;
    hipLaunchKernelGGL(k_merge, dim3(nblocks(nOld, 256)), dim3(256), 0, c.stream, ma);
    WDG_LAUNCH_CHECK();
  }
  const int rNew = 1 - c.rcur;
  // The rest is launched for a merge without extra slots (the old real contacts are all near, the
  // rule while the skin holds), and its counts are read in one wait at the end. Where the merge did
  // append some, the real set and the adjacency are made again with them.
  int64_t nNew = nPairs;
  const uint32_t* hw = c.hflags + HOST_REFRESH;
  for (int64_t nExtra = 0;;) {
    nNew = nPairs + nExtra;
    N.n = nNew;
    // real set of the new list: the carried contacts, with their state moved to the new indices
    reals_from_flags(c, N.carry.p, nNew, rNew);
    if (nNew > 0) {
      Reals &RO = c.R[c.rcur], &RN = c.R[rNew];
      CarryArgs ya{};
      ya.n = nNew; ya.carry = N.carry.p; ya.ov = c.rview(c.rcur); ya.nv = c.rview(rNew);
      DBuf<double>* so[10] = {&RO.hN[0], &RO.hN[1], &RO.hN[2], &RO.hY[0], &RO.hY[1],
                              &RO.hY[2], &RO.hF[0], &RO.hF[1], &RO.hF[2], &RO.huN};
      DBuf<double>* sn[10] = {&RN.hN[0], &RN.hN[1], &RN.hN[2], &RN.hY[0], &RN.hY[1],
                              &RN.hY[2], &RN.hF[0], &RN.hF[1], &RN.hF[2], &RN.huN};
      for (int q = 0; q < 10; q++) { ya.o[q] = so[q]->p; ya.d[q] = sn[q]->p; }
      ya.ogp = RO.gp.p; ya.gp = RN.gp.p;
      if (c.matEpochs > 1) { ya.oE = RO.hE.p; ya.nE = RN.hE.p; }
      if (c.rollActive) {
        RN.ensureRoll(nNew);
        ya.ogt = RO.gtq.p;
        ya.gt = RN.gtq.p;
      }
      hipLaunchKernelGGL(c.precision == 32 ? k_carry_state<32> : k_carry_state<64>, dim3(nblocks(nNew, 256)),
                         dim3(256), 0, c.stream, ya);
      WDG_LAUNCH_CHECK();
    }
    // 4. per-particle adjacency in canonical order (particle storage, other user id)
    const bool staged = nExtra == 0 && nbFits;
    if (staged) {
      // every slot is a near pair that its spheres staged: spheres' lists straight from the staged
      // neighbours (bodies included); the bodies' lists from the slot list
      if (nW > 0) {
        c.adjDeg.ensure(n + 1);
        WDG_HIP(hipMemsetAsync(c.adjDeg.p, 0, nW * sizeof(uint32_t), c.stream));
        if (nNew > 0) {
          hipLaunchKernelGGL(k_wall_deg, dim3(nblocks(nNew, 256)), dim3(256), 0, c.stream, nNew, nW,
                             (const uint32_t*)N.A.p, c.adjDeg.p);
          WDG_LAUNCH_CHECK();
        }
        if (nSph > 0) {
          hipLaunchKernelGGL(k_copy_deg, dim3(nblocks(nSph, 256)), dim3(256), 0, c.stream, nSph, nW,
                             (const uint32_t*)c.sdeg.p, c.adjDeg.p);
          WDG_LAUNCH_CHECK();
        }
        scan_exclusive(c, c.adjDeg.p, N.adjOff.p, n, N.adjOff.p + n);
      } else {
        scan_exclusive(c, c.sdeg.p, N.adjOff.p, n, N.adjOff.p + n);
      }
      // both ends of every pair listed it, so the lists hold two entries per slot: the kernels check
      // that themselves (and write nothing otherwise), the host at the end
      if (nNew > 0) {
        c.adjEnt.ensure(2 * nNew);
        AdjArgs aa{};
        aa.nSph = nSph; aa.nW = nW; aa.nb = c.stNb.p; aa.deg = c.sdeg.p; aa.count = c.scount.p; aa.off = c.soff.p;
        aa.A = N.A.p; aa.B = N.B.p; aa.uid = c.uid.p; aa.adjOff = N.adjOff.p; aa.ent = c.adjEnt.p; aa.adj = N.adj.p;
        aa.dflags = c.dflags.p;
        aa.want = (uint32_t)(2 * nNew);
        hipLaunchKernelGGL(k_adj_sym, dim3(nblocks(nSph, 64 * ADJ_WAVES)), dim3(64 * ADJ_WAVES), 0, c.stream, aa);
        WDG_LAUNCH_CHECK();
        if (nW > 0) {
          WDG_HIP(hipMemsetAsync(c.adjDeg.p, 0, nW * sizeof(uint32_t), c.stream));
          hipLaunchKernelGGL(k_wall_fill, dim3(nblocks(nNew, 256)), dim3(256), 0, c.stream, nNew, nW,
                             (const uint32_t*)N.A.p, (const uint32_t*)N.B.p, (const uint32_t*)N.info.p,
                             (const uint32_t*)c.uid.p, (const uint32_t*)N.adjOff.p, c.adjDeg.p, c.adjEnt.p, n);
          WDG_LAUNCH_CHECK();
          hipLaunchKernelGGL(k_wall_sort, dim3((unsigned)nW), dim3(WS_BS), 0, c.stream, (const uint32_t*)N.adjOff.p, n,
                             (uint32_t)(2 * nNew), (const uint64_t*)c.adjEnt.p, N.adj.p);
          WDG_LAUNCH_CHECK();
        }
      }
    } else {
      build_adjacency_atomic(c, N, nNew);
    }
    auto ent_pos = [&]() {
      if (nNew == 0) return;
      hipLaunchKernelGGL(k_ent_pos, dim3(nblocks(2 * nNew, 256)), dim3(256), 0, c.stream, 2 * nNew,
                         (const uint32_t*)N.adj.p, (const uint32_t*)(N.adjOff.p + n), N.entPos.p, N.eidx.p,
                         c.dflags.p);
      WDG_LAUNCH_CHECK();
    };
    hipLaunchKernelGGL(k_refresh_words, dim3(1), dim3(256), 0, c.stream, n, nW, c.nGBody, (const uint32_t*)c.gbody.p,
                       (const uint32_t*)N.adjOff.p, merged ? 1 : 0, staged ? 1 : 0, c.dflags.p,
                       c.hflagsDev + HOST_REFRESH);
    WDG_LAUNCH_CHECK();
    ent_pos();
    WDG_HIP(hipStreamSynchronize(c.stream));
    if (nExtra == 0 && hw[RW_EXTRA] > 0) {
      nExtra = hw[RW_EXTRA];
      continue;
    }
    if (hw[RW_ENTRIES] != 2 * (uint64_t)nNew) {
      drop_contacts(c);  // (the particles have moved in storage: the old list is of no use either)
      throw Error(WDG_E_STATE, "broadphase: neighbour lists disagree with the pair list (" +
                                   std::to_string(hw[RW_ENTRIES]) + " entries for " + std::to_string(nNew) + " pairs)");
    }
    if (staged && hw[RW_LONGEST] > WS_CAP) {
      // bodies with longer lists than a workgroup sorts: all by the radix sort
      sort_lists(c, N, nW, 0);
      WDG_HIP(hipMemsetAsync(c.dflags.p + WALL_LONG, 0, sizeof(uint32_t), c.stream));
      ent_pos();
    }
    break;
  }
  // the boundary-body gather cuts each list into parts of about 2048 entries
  if (c.nGBody > 0)
    c.bndParts = (int)std::min<uint32_t>(64u, std::max<uint32_t>(1u, (hw[RW_GATHERED] + 2047u) / 2048u));
  c.eidxValid = false;
  c.eidxClean = true;
  c.cur = 1 - c.cur;
  c.rcur = rNew;
  c.boundsValid = true;
  c.dirtyKnown = true;
  c.dirtyIdx = 0;
  // entries with wrong slots leave places of the slots' entries (entPos) unwritten, through which a
  // filter would store: nothing steps over such a list
  if (hw[RW_ERR] & ERR_ADJ) drop_contacts(c);
  take_errors(c, hw[RW_ERR]);
}

void collide(Ctx& c, const wdg_collide_params* p) {
  // the host mirror of the flag words is current only right after a graph batch
  bool fresh = c.hflagsFresh;
  c.hflagsFresh = false;
  if (c.n == 0) return;
  c.nCollide++;
  if (c.forcesPending) flush_forces(c);
  // Collision.cpp:164-184 setVerletDist: resolved once
  if (std::isnan(c.verletDist)) {
    double vd = p->verletDist;
    if (vd < 0) vd = std::isinf(c.rmin) ? 0. : std::fabs(vd) * c.rmin;
    c.verletDist = vd;
  }
  bool full = !c.boundsValid || p->forceInit;
  if (!full && c.verletDist == 0) full = true;
  if (!full) {
    if (!c.dirtyKnown) {
      WDG_HIP(hipMemsetAsync(c.dflags.p, 0, sizeof(uint32_t), c.stream));
      hipLaunchKernelGGL(k_dirty, dim3(nblocks(c.n, 256)), dim3(256), 0, c.stream, c.n, c.pos[0].p, c.pos[1].p,
                         c.pos[2].p, c.lastPos[0].p, c.lastPos[1].p, c.lastPos[2].p, c.verletDist * c.verletDist,
                         (const double*)(c.vdSceneActive ? c.vdScene.p : nullptr), (const uint32_t*)c.scene.p,
                         c.dflags.p);
      WDG_LAUNCH_CHECK();
      c.dirtyKnown = true;
      c.dirtyIdx = 0;
      fresh = false;
    }
    if (!fresh && c.hostWords && c.dirtyIdx >= DIRTY_PP) {
      // the leapfrog wrote its own answer to the pinned words
      WDG_HIP(hipStreamSynchronize(c.stream));
      c.hflags[1] = c.hflags[HOST_ERR];
      c.hflags[c.dirtyIdx] = c.hflags[HOST_DIRTY] == c.lfNumber ? 1u : 0u;
    } else if (!fresh) {
      WDG_HIP(hipMemcpyAsync(c.hflags, c.dflags.p, (DIRTY_PP + 2) * sizeof(uint32_t), hipMemcpyDeviceToHost,
                             c.stream));
      WDG_HIP(hipStreamSynchronize(c.stream));
    }
    take_errors(c, c.hflags[1]);
    if (c.hflags[c.dirtyIdx]) full = true;
  }
  if (full) {
    const auto t0 = std::chrono::steady_clock::now();
    refresh(c);
    c.refreshSec += std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  }
}

// potential set of the last refresh: enlarged-AABB pairs from the refresh positions
void potential_pairs(Ctx& c, std::vector<uint32_t>& ida, std::vector<uint32_t>& idb, std::vector<uint64_t>& cd) {
  ida.clear(); idb.clear(); cd.clear();
  const int64_t nSph = c.n - c.nW;
  if (!c.grid.valid || nSph <= 0) return;
  Grid g{};
  for (int k = 0; k < 3; k++) {
    g.org[k] = c.grid.org[k]; g.h[k] = c.grid.h[k]; g.L[k] = c.grid.L[k]; g.nc[k] = c.grid.nc[k];
  }
  g.periodic = c.grid.periodic;
  g.hashed = c.grid.hashed;
  g.hmask = c.grid.hmask;
  g.morton = c.grid.morton;
  g.sg = reinterpret_cast<const SceneGrid*>(c.grid.sg);
  AabbParams P{};
  P.vd = c.verletDist;
  P.absDf = std::fabs(c.field.distFactor);
  P.loneMask = c.field.loneMask;
  P.periodic = c.field.periodic;
  for (int k = 0; k < 3; k++) P.L[k] = c.field.cell[k];
  PairArgs pa = pair_args(c, g, P);
  launch_pairs<OUT_COUNT, MODE_AABB>(c, pa);
  scan_exclusive(c, c.scount.p, c.soff.p, nSph, c.dflags.p + 4);
  int64_t np = read_u32(c, c.dflags.p + 4);
  if (np == 0) return;
  DBuf<uint64_t> k, d;
  k.ensure(np);
  d.ensure(np);
  pa.pkey = k.p; pa.pdist = d.p;
  launch_pairs<OUT_KEYS, MODE_AABB>(c, pa);
  std::vector<uint64_t> hk((size_t)np), hd;
  WDG_HIP(hipMemcpyAsync(hk.data(), k.p, np * 8, hipMemcpyDeviceToHost, c.stream));
  if (c.field.periodic) {
    hd.resize((size_t)np);
    WDG_HIP(hipMemcpyAsync(hd.data(), d.p, np * 8, hipMemcpyDeviceToHost, c.stream));
  }
  WDG_HIP(hipStreamSynchronize(c.stream));
  k.release();
  d.release();
  for (int64_t i = 0; i < np; i++) {
    ida.push_back((uint32_t)(hk[i] >> 32));
    idb.push_back((uint32_t)(hk[i] & 0xFFFFFFFFu));
    cd.push_back(c.field.periodic ? hd[i] : 0);
  }
}

}  // namespace wdg
