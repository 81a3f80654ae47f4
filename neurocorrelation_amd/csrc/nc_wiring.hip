// The workload wiring built on the GPU: the network nc_net_generate builds on
// the host, bit for bit, from the same counter-based draws.  It replaces the
// reference's all-pairs scan (Neuron::makeConnections, src/NeuCor.cpp:418-444)
// for the distance rule of the benchmark workloads:
//   1. positions from Philox draws (one per draw index), their cells, and
//      the ids: draw order or the Morton order of the cells (radix sort);
//   2. a cell grid: in Morton order a cell's ids are a range, else a radix
//      sort of (cell, id);
//   3. work items of up to 64 targets of one cell; per item the ids of the 27
//      cells around it in ascending order -- in Morton order the 27 ranges in
//      order, else sorted in LDS -- and per target those within the radius:
//      counted, prefix-summed into the incoming rows, and, as they come out in
//      ascending source id (the order of Neuron::inSynapses,
//      src/NeuCor.h:212), written straight to their places, with
//   4. the delay from the distance and the weight and sign class from a draw
//      keyed by (source, target).
// What bounds it is the host: the arrays' first touch and copy.  On the device
// a thread per target (27 scattered ranges, twice) and a radix sort of all
// (target, source) pairs took 7.0 ms for 200 000 neurons and 1.9e7 synapses;
// a wave per cell, whose candidates are read once for all its targets, leaves
// 1.05 ms, and no pass over the synapses but the one that writes them (10 000
// neurons: 2.3 ms a call -> 0.92).
// Every float operation is written out with round-to-nearest intrinsics in
// the host builder's order, so no contraction or reassociation can differ.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <new>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "nc_common.h"
#include "nc_internal.h"

using nc::fail;

namespace {

#define NW_HIP(x)                                                          \
  do {                                                                     \
    hipError_t e_ = (x);                                                   \
    if (e_ != hipSuccess) return fail(NC_ERR_HIP, hipGetErrorString(e_)); \
  } while (0)

// Device buffers released together, allocated and freed in the order of the
// build's own stream (hipMallocAsync / hipFreeAsync), so that a build on one
// host thread does not wait for, or hold up, work on other streams.
struct Bufs {
  hipStream_t st;
  std::vector<void*> p;
  ~Bufs() {
    for (void* x : p) (void)hipFreeAsync(x, st);
  }
  template <class T>
  hipError_t alloc(T** out, size_t n) {
    void* q = nullptr;
    hipError_t e = hipMallocAsync(&q, (n ? n : 1) * sizeof(T), st);
    if (e == hipSuccess) p.push_back(q);
    *out = (T*)q;
    return e;
  }
};

// Arrays cut from one allocation, each at a multiple of 256 bytes.
struct Arena {
  std::vector<std::pair<void**, size_t>> a;  // where the pointer goes, its offset
  size_t bytes = 0;
  template <class T>
  void want(T** p, uint64_t n) {
    a.push_back({(void**)p, bytes});
    bytes += (n * sizeof(T) + 255) / 256 * 256;
  }
  hipError_t place(Bufs& B) {
    unsigned char* base = nullptr;
    const hipError_t e = B.alloc(&base, bytes);
    if (e == hipSuccess)
      for (auto& x : a) *x.first = base + x.second;
    return e;
  }
};

// The smallest float whose root, rounded, is not below the radius.
float d2_limit(float radius) {
  float x = (float)((double)radius * (double)radius);
  while (x > 0.0f && sqrtf(x) >= radius) x = nextafterf(x, 0.0f);
  while (x < INFINITY && sqrtf(x) < radius) x = nextafterf(x, INFINITY);
  return x;
}

dim3 grid_for(uint64_t n) { return dim3((uint32_t)std::min<uint64_t>((n + 255) / 256, 65535)); }

// 1. positions in draw order, their cells, and the id sort keys
__global__ __launch_bounds__(256) void k_wire_pos(uint64_t seed, uint32_t n, float side, int ncell,
                                                  uint32_t spatial, float* px, float* py, float* pz,
                                                  uint32_t* cell, uint64_t* key) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const nc_u32x4 r = nc_draw(seed, i, 0u, NC_STREAM_POS);
    const float x = __fmul_rn(nc_u01(r.v[0]), side);
    const float y = __fmul_rn(nc_u01(r.v[1]), side);
    const float z = __fmul_rn(nc_u01(r.v[2]), side);
    px[i] = x, py[i] = y, pz[i] = z;
    const uint32_t cx = (uint32_t)nc_cell_of(x, ncell, side), cy = (uint32_t)nc_cell_of(y, ncell, side),
                   cz = (uint32_t)nc_cell_of(z, ncell, side);
    cell[i] = (cz * (uint32_t)ncell + cy) * (uint32_t)ncell + cx;
    const uint64_t m = nc_part1by2(cx) | (nc_part1by2(cy) << 1) | (nc_part1by2(cz) << 2);
    key[i] = spatial ? ((m << 32) | i) : (uint64_t)i;
  }
}

// Positions and cells by id; (cell, id) keys for the grid.
__global__ __launch_bounds__(256) void k_wire_place(uint32_t n, const uint64_t* order, const float* px,
                                                    const float* py, const float* pz, const uint32_t* cell_d,
                                                    float* X, float* Y, float* Z, float* xyz, uint32_t* cell,
                                                    uint64_t* ckey) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t id = blockIdx.x * blockDim.x + threadIdx.x; id < n; id += stride) {
    const uint32_t d = (uint32_t)(order[id] & 0xffffffffu);
    X[id] = px[d], Y[id] = py[d], Z[id] = pz[d];
    xyz[3ull * id] = px[d], xyz[3ull * id + 1] = py[d], xyz[3ull * id + 2] = pz[d];
    cell[id] = cell_d[d];
    ckey[id] = ((uint64_t)cell_d[d] << 32) | id;
  }
}

// 2. the grid: members of each cell in ascending id (member k: id k in Morton
// order, else from the sorted keys), cells as ranges
__global__ __launch_bounds__(256) void k_wire_cells(uint32_t n, const uint32_t* cell, const uint64_t* ckey,
                                                    uint32_t* cmem, uint32_t* cstart, uint32_t* cend) {
  const uint32_t stride = gridDim.x * blockDim.x;
  auto cell_at = [&](uint32_t k) { return ckey ? (uint32_t)(ckey[k] >> 32) : cell[k]; };
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
    const uint32_t c = cell_at(k);
    cmem[k] = ckey ? (uint32_t)(ckey[k] & 0xffffffffu) : k;
    if (k == 0 || cell_at(k - 1) != c) cstart[c] = k;
    if (k + 1 == n || cell_at(k + 1) != c) cend[c] = k + 1;
  }
}

// 3. the work items: {first member, members}, up to kItem members of a cell
constexpr uint32_t kItem = 64;     // a lane per target
constexpr uint32_t kCand = 2048;   // candidate ids held in LDS at a time
constexpr uint32_t kItemWaves = 4;
__global__ __launch_bounds__(256) void k_wire_items(uint32_t n, const uint32_t* cell, const uint32_t* cmem,
                                                    const uint32_t* cstart, const uint32_t* cend, uint2* items,
                                                    uint32_t* n_items) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
    const uint32_t c = cell[cmem[k]];
    if ((k - cstart[c]) % kItem == 0) items[atomicAdd(n_items, 1u)] = make_uint2(k, min(kItem, cend[c] - k));
  }
}

// IEEE square root (round to nearest even) of a float: the approximation
// is moved to the neighbour on the other side of a rounding midpoint, the
// test done exactly in double (a midpoint between adjacent floats has 25
// significant bits, so its square is exact).
__device__ __forceinline__ float sqrt_rn(float x) {
  float r = sqrtf(x);
  if (!(x > 0.0f) || !(r < INFINITY)) return r;
  const double xd = (double)x;
  const float up = nextafterf(r, INFINITY), dn = nextafterf(r, 0.0f);
  const double mu = 0.5 * ((double)r + (double)up), md = 0.5 * ((double)r + (double)dn);
  if (xd >= mu * mu) r = up;
  else if (xd < md * md) r = dn;
  return r;
}

// The distance test of the host builder, operation by operation.
__device__ __forceinline__ float wire_dist(const float* X, const float* Y, const float* Z, uint32_t src,
                                           uint32_t tg) {
  const float ddx = __fsub_rn(X[src], X[tg]), ddy = __fsub_rn(Y[src], Y[tg]), ddz = __fsub_rn(Z[src], Z[tg]);
  float d2 = __fadd_rn(__fmul_rn(ddx, ddx), __fmul_rn(ddy, ddy));
  d2 = __fadd_rn(d2, __fmul_rn(ddz, ddz));
  return sqrt_rn(d2);
}

// The rows by a thread per target: the sources within the radius, in
// cell-visiting order, as (target, source) keys and distances.
__global__ __launch_bounds__(256) void k_wire_scan(uint32_t n, int ncell, float radius, const float* X,
                                                   const float* Y, const float* Z, const uint32_t* cell,
                                                   const uint32_t* cmem, const uint32_t* cstart,
                                                   const uint32_t* cend, const uint64_t* in_ptr, uint64_t* ekey,
                                                   float* edist) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t tg = blockIdx.x * blockDim.x + threadIdx.x; tg < n; tg += stride) {
    const uint32_t c0 = cell[tg];
    const int x0 = (int)(c0 % (uint32_t)ncell), y0 = (int)((c0 / (uint32_t)ncell) % (uint32_t)ncell),
              z0 = (int)(c0 / ((uint32_t)ncell * (uint32_t)ncell));
    uint64_t at = in_ptr[tg];
    for (int dz = -1; dz <= 1; ++dz) {
      const int zz = z0 + dz;
      if (zz < 0 || zz >= ncell) continue;
      for (int dy = -1; dy <= 1; ++dy) {
        const int yy = y0 + dy;
        if (yy < 0 || yy >= ncell) continue;
        for (int dx = -1; dx <= 1; ++dx) {
          const int xx = x0 + dx;
          if (xx < 0 || xx >= ncell) continue;
          const uint32_t c = ((uint32_t)zz * ncell + (uint32_t)yy) * ncell + (uint32_t)xx;
          const uint32_t b = cstart[c], e = cend[c];
          for (uint32_t q = b; q < e; ++q) {
            const uint32_t src = cmem[q];
            if (src == tg) continue;
            const float dist = wire_dist(X, Y, Z, src, tg);
            if (!(dist < radius)) continue;
            ekey[at] = ((uint64_t)tg << 32) | src;
            edist[at] = dist;
            ++at;
          }
        }
      }
    }
  }
}

// Per synapse of those, sorted: source, delay, weight, sign class.
__global__ __launch_bounds__(256) void k_wire_attr(uint64_t S, const uint64_t* ekey, const float* edist,
                                                   uint64_t seed, float radius, float fdmax, uint32_t dmin,
                                                   uint32_t dmax, float w_min, float wspan, float inhib,
                                                   uint32_t* in_src, float* w, uint8_t* delay, uint8_t* inh,
                                                   uint32_t* max_delay) {
  uint32_t seen = 0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < S; k += stride) {
    const uint32_t tg = (uint32_t)(ekey[k] >> 32), src = (uint32_t)(ekey[k] & 0xffffffffu);
    const float q = edist[k] / radius;  // IEEE division (HIP's default for float)
    const float dl = ceilf(__fmul_rn(q, fdmax));
    const uint32_t dd = dl < (float)dmin ? dmin : (dl > fdmax ? dmax : (uint32_t)dl);
    const nc_u32x4 r = nc_draw(seed, src, tg, NC_STREAM_WEIGHT);
    float wv = __fadd_rn(w_min, __fmul_rn(nc_u01(r.v[0]), wspan));
    const uint8_t ih = nc_u01(r.v[1]) < inhib ? 1 : 0;
    if (ih) wv = -wv;
    in_src[k] = src;
    w[k] = wv;
    delay[k] = (uint8_t)dd;
    inh[k] = ih;
    seen = max(seen, dd);
  }
  if (seen) atomicMax(max_delay, seen);
}

// The synapse attributes of a pair at distance dist, as k_wire_attr.
struct Attr {
  uint64_t seed;
  float radius, fdmax;
  uint32_t dmin, dmax;
  float w_min, wspan, inhib;
};

// 3. and 4.: a wave per work item.  FILL == false counts the rows (deg, and
// the longest in *max_deg, the most candidates of an item in *max_cand); FILL
// == true writes them.  d2lim is the smallest float whose root is not below
// the radius: d2 < d2lim exactly when the rounded distance is below it.
// SORTED: ids follow the cells' Morton order, so the 27 ranges in order of
// their starts hold the candidates in ascending id; else they are sorted in
// LDS (all of them at once: at most kCand).  The pairs found queue up in LDS
// and get their attributes 64 at a time.
template <bool FILL, bool SORTED>
__global__ __launch_bounds__(64 * kItemWaves) void k_wire_rows(const uint2* items, const uint32_t* n_items, int ncell,
                                                               float d2lim, const float* X, const float* Y,
                                                               const float* Z, const uint32_t* cell,
                                                               const uint32_t* cmem, const uint32_t* cstart,
                                                               const uint32_t* cend, uint64_t* deg,
                                                               uint32_t* max_deg, uint32_t* max_cand,
                                                               const uint64_t* in_ptr, Attr A, uint32_t* in_src,
                                                               float* w, uint8_t* delay, uint8_t* inh,
                                                               uint32_t* max_delay) {
  __shared__ uint32_t s_cand[kItemWaves][kCand];
  __shared__ uint4 s_que[FILL ? kItemWaves : 1][FILL ? 128 : 1];  // {place, source, target, d2}
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t* const cand = s_cand[wv];
  uint4* const que = s_que[FILL ? wv : 0];
  uint32_t qn = 0, top = 0, longest = 0, dmax_seen = 0;
  auto put = [&](uint32_t i) {
    const uint4 q = que[i];
    const float dist = sqrt_rn(__uint_as_float(q.w));
    const float dl = ceilf(__fmul_rn(dist / A.radius, A.fdmax));  // IEEE division (HIP's default for float)
    const uint32_t dd = dl < (float)A.dmin ? A.dmin : (dl > A.fdmax ? A.dmax : (uint32_t)dl);
    const nc_u32x4 r = nc_draw(A.seed, q.y, q.z, NC_STREAM_WEIGHT);
    float wv_ = __fadd_rn(A.w_min, __fmul_rn(nc_u01(r.v[0]), A.wspan));
    const uint8_t ih = nc_u01(r.v[1]) < A.inhib ? 1 : 0;
    if (ih) wv_ = -wv_;
    in_src[q.x] = q.y;
    w[q.x] = wv_;
    delay[q.x] = (uint8_t)dd;
    inh[q.x] = ih;
    dmax_seen = max(dmax_seen, dd);
  };
  const uint32_t ni = *n_items, nw = gridDim.x * kItemWaves;
  for (uint32_t it = blockIdx.x * kItemWaves + wv; it < ni; it += nw) {
    const uint2 item = items[it];
    const uint32_t c0 = cell[cmem[item.x]];
    const int x0 = (int)(c0 % (uint32_t)ncell), y0 = (int)((c0 / (uint32_t)ncell) % (uint32_t)ncell),
              z0 = (int)(c0 / ((uint32_t)ncell * (uint32_t)ncell));
    // lanes 0-26: the members around, and where they go among the candidates
    uint32_t start = 0, len = 0, off = 0, total = 0;
    if (lane < 27u) {
      const int xx = x0 + (int)(lane % 3u) - 1, yy = y0 + (int)(lane / 3u % 3u) - 1, zz = z0 + (int)(lane / 9u) - 1;
      if (xx >= 0 && xx < ncell && yy >= 0 && yy < ncell && zz >= 0 && zz < ncell) {
        const uint32_t c = ((uint32_t)zz * ncell + (uint32_t)yy) * ncell + (uint32_t)xx;
        start = cstart[c];
        len = cend[c] - start;
      }
    }
#pragma unroll
    for (uint32_t j = 0; j < 27u; ++j) {
      const uint32_t sj = __builtin_amdgcn_readlane(start, j), lj = __builtin_amdgcn_readlane(len, j);
      total += lj;
      if (SORTED ? (sj < start || (sj == start && j < lane)) : j < lane) off += lj;
    }
    longest = max(longest, total);
    const bool tgt = lane < item.y;
    const uint32_t id = tgt ? cmem[item.x + lane] : 0u;
    const float tx = X[id], ty = Y[id], tz = Z[id];
    uint32_t cur = FILL && tgt ? (uint32_t)in_ptr[id] : 0u;
    for (uint32_t base = 0; base < total; base += kCand) {
      const uint32_t m = min(kCand, total - base);
      for (uint32_t j = 0; j < 27u; ++j) {
        const uint32_t sj = __builtin_amdgcn_readlane(start, j), lj = __builtin_amdgcn_readlane(len, j),
                       oj = __builtin_amdgcn_readlane(off, j);
        for (uint32_t i = lane; i < lj; i += 64) {
          const uint32_t p = oj + i - base;  // wraps below base
          if (p < m) cand[p] = SORTED ? sj + i : cmem[sj + i];
        }
      }
      if (FILL && !SORTED) {
        uint32_t np = 64;
        while (np < m) np <<= 1;
        for (uint32_t i = m + lane; i < np; i += 64) cand[i] = ~0u;
        for (uint32_t k = 2; k <= np; k <<= 1)
          for (uint32_t d = k >> 1; d; d >>= 1) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            for (uint32_t i = lane; i < np / 2; i += 64) {
              const uint32_t lo = ((i & ~(d - 1u)) << 1) | (i & (d - 1u)), hi = lo + d;
              const uint32_t a = cand[lo], b = cand[hi];
              if ((a > b) == ((lo & k) == 0u)) {
                cand[lo] = b;
                cand[hi] = a;
              }
            }
          }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (uint32_t j0 = 0; j0 < m; j0 += 64) {
        const bool in = j0 + lane < m;
        const uint32_t src = in ? cand[j0 + lane] : 0u;
        const float sx = X[src], sy = Y[src], sz = Z[src];
        for (uint32_t t = 0; t < item.y; ++t) {
          const uint32_t tid = __builtin_amdgcn_readlane(id, t);
          const float ux = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(tx), t)),
                      uy = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ty), t)),
                      uz = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(tz), t));
          // the distance test of the host builder, operation by operation
          const float ddx = __fsub_rn(sx, ux), ddy = __fsub_rn(sy, uy), ddz = __fsub_rn(sz, uz);
          float d2 = __fadd_rn(__fmul_rn(ddx, ddx), __fmul_rn(ddy, ddy));
          d2 = __fadd_rn(d2, __fmul_rn(ddz, ddz));
          const bool ok = in && src != tid && d2 < d2lim;
          const unsigned long long mk = __ballot(ok);
          const uint32_t nf = (uint32_t)__builtin_popcountll(mk);
          if (FILL && mk) {
            const uint32_t below = (uint32_t)__builtin_popcountll(mk & ((1ull << lane) - 1ull));
            const uint32_t at = __builtin_amdgcn_readlane(cur, t);
            if (ok) que[qn + below] = make_uint4(at + below, src, tid, __float_as_uint(d2));
            qn += nf;
            if (qn >= 64u) {
              __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
              qn -= 64u;
              put(qn + lane);
            }
          }
          if (lane == t) cur += nf;
        }
      }
    }
    if (!FILL && tgt) {
      deg[id] = cur;
      top = max(top, cur);
    }
  }
  if (FILL) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < qn) put(lane);
    if (dmax_seen) atomicMax(max_delay, dmax_seen);
  } else {
    if (top) atomicMax(max_deg, top);
    if (lane == 0 && longest) atomicMax(max_cand, longest);
  }
}

template <class F>
nc_status with_temp(Bufs& B, F&& f) {
  size_t bytes = 0;
  NW_HIP(f(nullptr, bytes));
  void* tmp = nullptr;
  NW_HIP(B.alloc((unsigned char**)&tmp, bytes));
  NW_HIP(f(tmp, bytes));
  return NC_OK;
}

uint32_t bits_for(uint64_t v) {
  uint32_t b = 1;
  while (b < 64 && (v >> b)) ++b;
  return b;
}

}  // namespace

extern "C" nc_status nc_net_generate_device(const nc_wiring_spec* spec, int32_t device, nc_net** out) try {
  if (!spec || !out) return fail(NC_ERR_ARG, "null argument");
  *out = nullptr;
  const nc_wiring_spec s = *spec;
  {
    nc_status st = nc::check_wiring_spec(s);
    if (st != NC_OK) return st;
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(NC_ERR_NO_DEVICE, "no HIP device");
  if (device < 0 || device >= ndev) return fail(NC_ERR_RANGE, "device index out of range");
  NW_HIP(hipSetDevice(device));
  const uint32_t n = s.n_neurons;
  const int ncell = nc_cells_per_axis(s.side, s.radius);
  const uint64_t ncells = (uint64_t)ncell * ncell * ncell;
  hipStream_t st = nullptr;
  NW_HIP(nc::stream_take(device, &st));
  struct StreamGuard {
    int device;
    hipStream_t s;
    ~StreamGuard() { nc::stream_give(device, s); }  // waits for the buffers' frees, queued on it
  } sg{device, st};
  Bufs B{st, {}};
  float *px, *py, *pz, *X, *Y, *Z, *xyz;
  uint32_t *cell_d, *cell, *cmem, *cstart, *cend, *meta;
  uint64_t *key, *key2, *deg, *in_ptr;
  uint2* items;
  {
    // one allocation, cut into the arrays
    Arena R;
    R.want(&key, n), R.want(&key2, n), R.want(&deg, n), R.want(&in_ptr, n + 1ull), R.want(&items, n);
    R.want(&px, n), R.want(&py, n), R.want(&pz, n), R.want(&X, n), R.want(&Y, n), R.want(&Z, n);
    R.want(&xyz, 3ull * n), R.want(&cell_d, n), R.want(&cell, n), R.want(&cmem, n);
    R.want(&meta, 64), R.want(&cstart, ncells), R.want(&cend, ncells);
    NW_HIP(R.place(B));
  }
  uint32_t* const n_items = meta;       // work items
  uint32_t* const max_deg = meta + 1;   // longest row
  uint32_t* const max_cand = meta + 2;  // most candidates of an item
  uint32_t* const max_dly = meta + 3;   // longest delay
  const dim3 gn = grid_for(n);
  hipLaunchKernelGGL(k_wire_pos, gn, dim3(256), 0, st, s.seed, n, s.side, ncell, s.spatial_order, px, py, pz,
                     cell_d, key);
  NW_HIP(hipGetLastError());
  // the counters, then the cells' ranges
  NW_HIP(hipMemsetAsync(meta, 0, (char*)(cend + ncells) - (char*)meta, st));
  const uint64_t* order = key;
  if (s.spatial_order) {
    // by Morton code: stable, so equal codes stay in draw order
    nc_status r = with_temp(B, [&](void* t, size_t& b) {
      return rocprim::radix_sort_keys(t, b, key, key2, (size_t)n, 32u, 32u + 3u * bits_for(ncell - 1), st);
    });
    if (r != NC_OK) return r;
    order = key2;
  }
  // (the keys not in use by `order` take the grid's)
  uint64_t* const ckey = s.spatial_order ? key : key2;
  hipLaunchKernelGGL(k_wire_place, gn, dim3(256), 0, st, n, order, px, py, pz, cell_d, X, Y, Z, xyz, cell, ckey);
  NW_HIP(hipGetLastError());
  const uint64_t* grid_key = nullptr;
  if (!s.spatial_order) {
    nc_status r = with_temp(B, [&](void* t, size_t& b) {
      return rocprim::radix_sort_keys(t, b, ckey, key, (size_t)n, 32u, 32u + bits_for(ncells - 1), st);
    });
    if (r != NC_OK) return r;
    grid_key = key;
  }
  hipLaunchKernelGGL(k_wire_cells, gn, dim3(256), 0, st, n, cell, grid_key, cmem, cstart, cend);
  NW_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_wire_items, gn, dim3(256), 0, st, n, cell, cmem, cstart, cend, items, n_items);
  NW_HIP(hipGetLastError());
  const Attr A{s.seed, s.radius, (float)s.delay_max, s.delay_min, s.delay_max, s.w_min, s.w_max - s.w_min, s.inhib_frac};
  const float d2lim = d2_limit(s.radius);
  uint32_t* in_src = nullptr;
  float* w = nullptr;
  uint8_t *delay = nullptr, *inh = nullptr;
  // at most a wave per item (there are at most n), and several items a wave
  const dim3 gw((uint32_t)std::min<uint64_t>((n + kItemWaves - 1) / kItemWaves, 4096));
  auto rows = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, gw, dim3(64 * kItemWaves), 0, st, items, n_items, ncell, d2lim, X, Y, Z, cell, cmem,
                       cstart, cend, deg, max_deg, max_cand, in_ptr, A, in_src, w, delay, inh, max_dly);
    return hipGetLastError();
  };
  NW_HIP(rows(k_wire_rows<false, false>));  // counting needs no order
  NW_HIP(hipMemsetAsync(in_ptr, 0, 8, st));
  {
    nc_status r = with_temp(B, [&](void* t, size_t& b) {
      return rocprim::inclusive_scan(t, b, deg, in_ptr + 1, (size_t)n, rocprim::plus<uint64_t>(), st);
    });
    if (r != NC_OK) return r;
  }
  uint64_t S = 0;
  uint32_t seen[4] = {0, 0, 0, 0};
  NW_HIP(hipMemcpyAsync(&S, in_ptr + n, 8, hipMemcpyDeviceToHost, st));
  NW_HIP(hipMemcpyAsync(seen, meta, sizeof seen, hipMemcpyDeviceToHost, st));
  NW_HIP(hipStreamSynchronize(st));
  if (S >= (1ull << 32) - (1ull << 24)) return fail(NC_ERR_ARG, "too many synapses");
  {
    Arena R;
    R.want(&in_src, S), R.want(&w, S), R.want(&delay, S), R.want(&inh, S);
    NW_HIP(R.place(B));
  }
  if (S && s.spatial_order) {
    NW_HIP(rows(k_wire_rows<true, true>));
  } else if (S && seen[2] <= kCand) {
    NW_HIP(rows(k_wire_rows<true, false>));
  } else if (S) {
    // more candidates around a cell than its wave can sort in LDS: a thread
    // per target, then the pairs sorted by (target, source)
    uint64_t *ekey, *ekey2;
    float *edist, *edist2;
    NW_HIP(B.alloc(&ekey, S));
    NW_HIP(B.alloc(&ekey2, S));
    NW_HIP(B.alloc(&edist, S));
    NW_HIP(B.alloc(&edist2, S));
    hipLaunchKernelGGL(k_wire_scan, gn, dim3(256), 0, st, n, ncell, s.radius, X, Y, Z, cell, cmem, cstart, cend,
                       (const uint64_t*)in_ptr, ekey, edist);
    NW_HIP(hipGetLastError());
    const uint32_t hi = 32u + bits_for(n > 1 ? n - 1 : 1);
    nc_status r = with_temp(B, [&](void* t, size_t& b) {
      return rocprim::radix_sort_pairs(t, b, ekey, ekey2, edist, edist2, (size_t)S, 0u, hi, st);
    });
    if (r != NC_OK) return r;
    hipLaunchKernelGGL(k_wire_attr, grid_for(S), dim3(256), 0, st, S, ekey2, edist2, s.seed, s.radius,
                       (float)s.delay_max, s.delay_min, s.delay_max, s.w_min, s.w_max - s.w_min, s.inhib_frac,
                       in_src, w, delay, inh, max_dly);
    NW_HIP(hipGetLastError());
  }
  std::unique_ptr<nc_net> net(new (std::nothrow) nc_net());
  if (!net) return fail(NC_ERR_OOM, "host allocation failed");
  try {
    net->n = n;
    net->xyz.resize(3ull * n);
    net->in_ptr.resize(n + 1ull);
    net->in_src.resize(S);
    net->w.resize(S);
    net->delay.resize(S);
    net->inh.resize(S);
  } catch (const std::bad_alloc&) {
    return fail(NC_ERR_OOM, "host allocation failed");
  }
  const nc::Segment seg[] = {
      {net->in_src.data(), in_src, 4ull * S}, {net->w.data(), w, 4ull * S},
      {net->delay.data(), delay, S},          {net->inh.data(), inh, S},
      {net->xyz.data(), xyz, 12ull * n},      {net->in_ptr.data(), in_ptr, 8ull * (n + 1ull)},
      {seen, meta, sizeof seen}};
  hipError_t e = nc::download(device, st, seg, sizeof seg / sizeof seg[0]);
  if (e != hipSuccess) return fail(NC_ERR_HIP, hipGetErrorString(e));
  net->max_in_degree = seen[1];
  net->max_delay = seen[3];
  *out = net.release();
  return NC_OK;
}
NC_ABI_CATCH
