// Kernels between a network's device layout and the caller's orders (neuron
// ids; synapses by target id, then source): state read back, weights written,
// checkpoints packed and laid out again.
//
// What bounds the calls is the host: before, every call moved whole 16-byte
// slot records (with the layout's padding) across PCIe and put them in order
// in host loops, one scattered record at a time.  Here 16 lanes take a
// neuron's row -- two 128-byte chunks of records on the device's side, 16
// consecutive values on the caller's -- so that only the values asked for
// cross, in the caller's order.  A network of 20 000 neurons and 9e5
// synapses, before -> after (microseconds): spike state read 8498 -> 1746
// (11 MB into fresh pages), weights written 6305 -> 591, 64 of them edited
// 4898 -> 32; one of 1.1e6 synapses restored 23 944 -> 1272.
#pragma once
#include "nc_kernels.h"

#define NC_ROW_LANES 16u

// Tells the host that a kernel of a few workgroups has written its results to
// pinned memory, sooner than a stream synchronisation does (a read of 750
// neurons 12.0 -> 8.2 us with its launch; from about 40 workgroups on the
// fences cost more than it gains).  count: 0 between kernels; flag == null:
// nobody waits so.
struct nc_done {
  uint32_t *count, *flag, tag;
};
__device__ __forceinline__ void nc_tell(const nc_done& d) {
  if (!d.flag) return;
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (atomicAdd(d.count, 1u) + 1u != gridDim.x) return;
  *d.count = 0u;
  __threadfence_system();
  __hip_atomic_store(d.flag, d.tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A network on the device, for these kernels.
struct nc_place {
  nc_slot* slots;
  const uint32_t* slice_off;
  const uint2* ndw;
  const uint32_t *id_pos, *id_row;  // neuron id -> local position; its first synapse
  uint32_t pos0, q0, n;             // first position and slice; neurons
};

// A lane's share of a neuron's row: neuron `id`, in-slots k = sub, sub +
// NC_ROW_LANES, ...; synapse row + k sits in slot(k).
struct nc_row {
  uint32_t p, row, deg, sub, so;
  __device__ __forceinline__ uint32_t slot(uint32_t k) const { return nc_slot_of(so, p & 63u, k); }
};
__device__ __forceinline__ bool nc_row_of(const nc_place& N, uint32_t t, nc_row& r) {
  const uint32_t id = t / NC_ROW_LANES;
  if (id >= N.n) return false;
  r.sub = t % NC_ROW_LANES;
  r.p = N.id_pos[N.pos0 + id];
  r.row = N.id_row[N.pos0 + id];
  r.deg = N.ndw[N.pos0 + r.p].x & NC_DEG_MASK;
  r.so = N.slice_off[N.q0 + (r.p >> 6)];
  return true;
}

// One value per neuron, by id.
__global__ __launch_bounds__(256) void k_read_neurons(nc_place N, const uint32_t* v, uint32_t n, uint32_t* out,
                                                      nc_done done) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = v[N.pos0 + N.id_pos[N.pos0 + i]];
  nc_tell(done);
}

// The first n_syn synapses' weights.
__global__ __launch_bounds__(256) void k_read_weights(nc_place N, float* out, uint32_t n_syn, nc_done done) {
  nc_row r;
  if (nc_row_of(N, blockIdx.x * blockDim.x + threadIdx.x, r))
    for (uint32_t k = r.sub; k < r.deg && r.row + k < n_syn; k += NC_ROW_LANES)
      out[r.row + k] = N.slots[r.slot(k)].w;
  nc_tell(done);
}

// The first n_syn synapses' spike state at step s (a null array is not wanted):
// the arrival of the latched spike until its latch releases (Synapse::
// AP_fireTime), rel steps later, else 0; lastSpikeArrival -- the latched
// spike's arrival once it has arrived, else the one before it, which fan-out
// moved to last_arr, or one restored without a latched spike; the latched
// depolarisation.
__global__ __launch_bounds__(256) void k_read_spikes(nc_place N, int32_t s, int32_t rel, int32_t* arrival,
                                                     int32_t* last, float* depol, uint32_t n_syn, nc_done done) {
  nc_row r;
  if (nc_row_of(N, blockIdx.x * blockDim.x + threadIdx.x, r))
    for (uint32_t k = r.sub; k < r.deg && r.row + k < n_syn; k += NC_ROW_LANES) {
      const nc_slot x = N.slots[r.slot(k)];
      const int32_t a = x.arr_inh >> 1;
      if (arrival) arrival[r.row + k] = (a != NC_NEVER && s < a + rel) ? a : 0;
      if (last) last[r.row + k] = (a != NC_NEVER && a <= s) ? a : x.last_arr;
      if (depol) depol[r.row + k] = x.depol;
    }
  nc_tell(done);
}

// Synapse::setWeight (src/NeuCor.cpp:576-579): the weight and its sign class.
__device__ __forceinline__ void nc_set_weight(nc_slot* x, float w) {
  x->w = w;
  x->arr_inh = (x->arr_inh & ~1) | (w < 0.0f ? 1 : 0);
}

// The first n_syn synapses' weights.
__global__ __launch_bounds__(256) void k_write_weights(nc_place N, const float* w, uint32_t n_syn) {
  nc_row r;
  if (!nc_row_of(N, blockIdx.x * blockDim.x + threadIdx.x, r)) return;
  for (uint32_t k = r.sub; k < r.deg && r.row + k < n_syn; k += NC_ROW_LANES)
    nc_set_weight(&N.slots[r.slot(k)], w[r.row + k]);
}

// The weights of the synapses whose bits are set.
__global__ __launch_bounds__(256) void k_write_listed(nc_place N, const float* w, const uint32_t* listed) {
  nc_row r;
  if (!nc_row_of(N, blockIdx.x * blockDim.x + threadIdx.x, r)) return;
  for (uint32_t k = r.sub; k < r.deg; k += NC_ROW_LANES) {
    const uint32_t i = r.row + k;
    if ((listed[i >> 5] >> (i & 31u)) & 1u) nc_set_weight(&N.slots[r.slot(k)], w[i]);
  }
}

// Listed slots' weights: (slot, weight bits), every slot once.
__global__ __launch_bounds__(256) void k_set_weights(nc_slot* slots, const uint2* sw, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) nc_set_weight(&slots[sw[i].x], __uint_as_float(sw[i].y));
}

// A checkpoint's neurons (potential, last fire, firings by id) and synapses
// (weight, depolarisation, last arrival, arrival) as 4-byte words.
__global__ __launch_bounds__(256) void k_pack(nc_place N, const float* V, const int32_t* last_fire,
                                              const uint32_t* firings, int32_t s, uint32_t* out) {
  nc_row r;
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (!nc_row_of(N, t, r)) return;
  if (r.sub < 3u) {
    const uint32_t p = N.pos0 + r.p;
    out[t / NC_ROW_LANES * 3u + r.sub] =
        r.sub == 0u ? __float_as_uint(V[p]) : r.sub == 1u ? (uint32_t)last_fire[p] : firings[p];
  }
  uint32_t* const syn = out + 3ull * N.n;
  for (uint32_t k = r.sub; k < r.deg; k += NC_ROW_LANES) {
    const nc_slot x = N.slots[r.slot(k)];
    const int32_t a = x.arr_inh >> 1;
    uint32_t* const o = syn + 4ull * (r.row + k);
    o[0] = __float_as_uint(x.w);
    o[1] = __float_as_uint(x.depol);
    o[2] = (uint32_t)((a != NC_NEVER && a <= s) ? a : x.last_arr);
    o[3] = (uint32_t)a;
  }
}

// Step values a checkpoint may hold: NC_NEVER, or a step of the run so far
// (arrivals: up to the longest delay ahead); anything else would index the
// step tables out of range.  Ors into *bad: 1 last fires, 2 last arrivals, 4
// arrivals.
__global__ __launch_bounds__(256) void k_check_checkpoint(const uint32_t* in, uint32_t n, uint64_t n_syn, int32_t s,
                                                          uint32_t* bad) {
  auto past = [s](int32_t v) { return v == NC_NEVER || (v >= 1 && v <= s); };
  uint32_t b = 0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n + n_syn; i += stride) {
    if (i < n) {
      if (!past((int32_t)in[3 * i + 1])) b |= 1u;
    } else {
      const uint32_t* const e = in + 3ull * n + 4 * (i - n);
      const int32_t a = (int32_t)e[3];
      if (!past((int32_t)e[2])) b |= 2u;
      if (a != NC_NEVER && (a < 1 || a > s + 255)) b |= 4u;
    }
  }
  if (b) atomicOr(bad, b);
}

// A checkpoint into a network just added, at step s with a release window of
// rel steps: a lane per neuron lays out its neuron, its slot records and,
// from their arrivals, its active mask words and their summary, its cache of
// the first active slots and its spikes in flight (in the pending list of
// their window: their buckets are not theirs to fill in order).  The lists
// start empty: they hold the spikes of a checkpoint restored here before, if
// that one was taken before its first step.
__global__ __launch_bounds__(64) void k_unpack(nc_place N, const uint32_t* nid, const uint32_t* slice_moff,
                                               const uint32_t* in, int32_t s, int32_t rel, float* V,
                                               int32_t* last_fire, uint32_t* firings, uint32_t* amask, uint32_t* asum,
                                               uint4* acache, uint32_t* pend0, uint32_t* pend1, uint2* pend_cnt) {
  const uint32_t q = N.q0 + blockIdx.x, lane = threadIdx.x, pos = q * 64u + lane;
  const uint32_t dw = N.ndw[pos].x;
  if (lane == 0) pend_cnt[q] = make_uint2(0u, 0u);
  __threadfence();
  __syncthreads();
  if (!(dw & NC_DEG_VALID)) return;
  const uint32_t id = nid[pos], deg = dw & NC_DEG_MASK, row = N.id_row[N.pos0 + id], so = N.slice_off[q];
  V[pos] = __uint_as_float(in[3ull * id]);
  last_fire[pos] = (int32_t)in[3ull * id + 1];
  firings[pos] = in[3ull * id + 2];
  const uint32_t* const syn = in + 3ull * N.n + 4ull * row;
  const uint32_t nmw = (deg + 31u) / 32u, G = nmw <= 32u ? 1u : (nmw + 31u) / 32u;
  uint32_t c[4] = {0u, 0u, 0u, 0u}, nc = 0, sum = 0;
  static_assert(NC_ACACHE == 3, "three depolarisations and their arrivals' low bytes per 16-byte record");
  for (uint32_t w = 0; w < nmw; ++w) {
    uint32_t bits = 0;
    for (uint32_t k = 32u * w; k < min(deg, 32u * w + 32u); ++k) {
      nc_slot& x = N.slots[nc_slot_of(so, lane, k)];
      const uint32_t* const e = syn + 4ull * k;
      const uint32_t depol = e[1];
      const int32_t arr = (int32_t)e[3];
      x = nc_slot{__uint_as_float(e[0]), __uint_as_float(depol), (int32_t)e[2], arr * 2 + (x.arr_inh & 1)};
      if (arr == NC_NEVER) continue;
      if (arr > s) {
        const uint32_t list = ((uint32_t)arr >> NC_PEND_LOG_W) & 1u;
        const uint32_t at = atomicAdd(reinterpret_cast<uint32_t*>(&pend_cnt[q]) + list, 1u);
        (list ? pend1 : pend0)[so + at] = ((nc_slot_of(so, lane, k) - so) << 8) | ((uint32_t)arr & 255u);
      } else if (s < arr + rel) {
        bits |= 1u << (k & 31u);
        if (nc < NC_ACACHE) {
#pragma unroll
          for (uint32_t i = 0; i < NC_ACACHE; ++i)
            if (nc == i) c[i] = depol;
          c[3] |= ((uint32_t)arr & 255u) << (8u * nc++);
        }
      }
    }
    amask[slice_moff[q] + w * 64u + lane] = bits;
    if (bits) sum |= 1u << (w / G);
  }
  asum[pos] = sum;
  acache[pos] = make_uint4(c[0], c[1], c[2], c[3]);
}

// The source-side latch copies from the target records.
__global__ __launch_bounds__(256) void k_restore_latches(nc_edge* e, const nc_slot* slots, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    e[i].arr = slots[e[i].j].arr_inh >> 1;
}

// ---------------------------------------------------------------------------
// FNV-1a on the device: h <- (h ^ b) p for every byte b, p = 2^40 + 435.  The
// chain looks serial, but the low byte l of h has a chain of its own, l <-
// low8(435 (l ^ b)), and with it h ^ b = h + d, d = (l ^ b) - l, so that the
// rest is a sum: h_N = p^N h_0 + sum of p^(N - i) d_i.
//   k_fnv_maps   per segment of NC_FNV_SEG words, 256 threads run the chain
//                from each possible low byte, noting where it stands after
//                every piece of NC_FNV_PIECE words;
//   k_fnv_groups the same maps over NC_FNV_GROUP segments; k_fnv_starts the
//                low byte each group starts with;
//   k_fnv_sum    a thread per piece, its low byte now known, adds its terms.
// The host hashes a byte per four to five clocks, after copying the results:
// 18 ms of the server's loop for 24 jobs of 4.4e6 words in all, 4.8 so.
// A segment's chain is what k_fnv_maps takes for all but the largest results
// (those take the arithmetic, 256 chains): segments of 1024 words 71 us a job
// of that burst, of 256 words 26.
#define NC_FNV_PIECE 64u
#define NC_FNV_SEG 256u
#define NC_FNV_GROUP 64u
#define NC_FNV_P 1099511628211ull

// The words a result's digest covers: potentials by id, weights by synapse,
// firings by id; and the sum of the firings (sums[1]; sums[0] is cleared).
__global__ __launch_bounds__(256) void k_result_words(nc_place N, const float* V, const uint32_t* firings,
                                                      uint32_t n_syn, uint32_t* out, unsigned long long* spikes) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  nc_row r;
  const bool in = nc_row_of(N, t, r);
  unsigned long long f = 0;
  if (in) {
    const uint32_t id = t / NC_ROW_LANES, p = N.pos0 + r.p;
    if (r.sub == 0u) out[id] = __float_as_uint(V[p]);
    if (r.sub == 1u) {
      f = firings[p];
      out[N.n + n_syn + id] = (uint32_t)f;
    }
    for (uint32_t k = r.sub; k < r.deg; k += NC_ROW_LANES)
      out[N.n + r.row + k] = __float_as_uint(N.slots[r.slot(k)].w);
  }
  for (int o = 32; o > 0; o >>= 1) f += __shfl_xor(f, o);
  if ((threadIdx.x & 63u) == 0u && f) atomicAdd(spikes, f);
}

// maps[piece][l]: the low byte after the piece of a chain that entered the
// piece's segment with l.
__global__ __launch_bounds__(256) void k_fnv_maps(const uint32_t* __restrict__ words, uint32_t n, uint8_t* maps) {
  const uint32_t w0 = blockIdx.x * NC_FNV_SEG, w1 = min(n, w0 + NC_FNV_SEG);
  uint32_t l = threadIdx.x;  // only its low byte counts
  for (uint32_t p0 = w0; p0 < w1; p0 += NC_FNV_PIECE) {
    for (uint32_t i = p0; i < min(w1, p0 + NC_FNV_PIECE); ++i) {
      const uint32_t w = words[i];
#pragma unroll
      for (int b = 0; b < 32; b += 8) l = __umul24(l ^ ((w >> b) & 255u), 0xB3u);
    }
    maps[(size_t)(p0 / NC_FNV_PIECE) * 256u + threadIdx.x] = (uint8_t)l;
  }
}

// The maps of a group's segments (the row of each one's last piece) into LDS;
// returns how many.
__device__ __forceinline__ uint32_t nc_fnv_load(const uint8_t* maps, uint32_t n_pieces, uint32_t g, uint8_t* m) {
  constexpr uint32_t per = NC_FNV_SEG / NC_FNV_PIECE;
  const uint32_t s0 = g * NC_FNV_GROUP, n_seg = (n_pieces + per - 1) / per, ns = min(NC_FNV_GROUP, n_seg - s0);
  for (uint32_t i = threadIdx.x; i < ns * 64u; i += blockDim.x) {
    const uint32_t last = min((s0 + i / 64u + 1u) * per, n_pieces) - 1u;
    reinterpret_cast<uint32_t*>(m)[i] = reinterpret_cast<const uint32_t*>(maps)[(size_t)last * 64u + i % 64u];
  }
  __syncthreads();
  return ns;
}

__global__ __launch_bounds__(256) void k_fnv_groups(const uint8_t* maps, uint32_t n_pieces, uint8_t* groups) {
  __shared__ __align__(16) uint8_t m[NC_FNV_GROUP * 256u];
  const uint32_t ns = nc_fnv_load(maps, n_pieces, blockIdx.x, m);
  uint32_t l = threadIdx.x;
  for (uint32_t s = 0; s < ns; ++s) l = m[s * 256u + l];
  groups[blockIdx.x * 256u + threadIdx.x] = (uint8_t)l;
}

// starts[g]: the low byte group g's first segment starts with, from l0.
__global__ __launch_bounds__(256) void k_fnv_starts(const uint8_t* groups, uint32_t n_groups, uint32_t l0,
                                                    uint8_t* starts) {
  __shared__ __align__(16) uint8_t m[NC_FNV_GROUP * 256u];
  __shared__ uint32_t l;
  if (threadIdx.x == 0) l = l0;
  for (uint32_t g0 = 0; g0 < n_groups; g0 += NC_FNV_GROUP) {
    const uint32_t ng = min(NC_FNV_GROUP, n_groups - g0);
    for (uint32_t i = threadIdx.x; i < ng * 256u; i += 256u) m[i] = groups[(size_t)g0 * 256u + i];
    __syncthreads();
    if (threadIdx.x == 0)
      for (uint32_t g = 0; g < ng; ++g) {
        starts[g0 + g] = (uint8_t)l;
        l = m[g * 256u + l];
      }
    __syncthreads();
  }
}

// *sum += the terms of the pieces (64 of group blockIdx.x / 16 each) and, once,
// p^N h0.
__global__ __launch_bounds__(64) void k_fnv_sum(const uint32_t* words, uint32_t n, const uint8_t* maps,
                                                const uint8_t* starts, unsigned long long h0,
                                                unsigned long long* sum) {
  constexpr uint32_t per = NC_FNV_SEG / NC_FNV_PIECE;
  __shared__ __align__(16) uint8_t m[NC_FNV_GROUP * 256u];
  __shared__ uint8_t sl[NC_FNV_GROUP];
  const uint32_t n_pieces = (n + NC_FNV_PIECE - 1) / NC_FNV_PIECE;
  const uint32_t g = blockIdx.x / per, lane = threadIdx.x;
  const uint32_t ns = nc_fnv_load(maps, n_pieces, g, m);
  if (lane == 0) {
    uint32_t l = starts[g];
    for (uint32_t s = 0; s < ns; ++s) {
      sl[s] = (uint8_t)l;
      l = m[s * 256u + l];
    }
  }
  __syncthreads();
  const uint32_t piece = g * NC_FNV_GROUP * per + (blockIdx.x % per) * 64u + lane;
  unsigned long long c = 0;
  auto power = [](unsigned long long k) {
    unsigned long long r = 1, q = NC_FNV_P;
    for (; k; k >>= 1, q *= q)
      if (k & 1ull) r *= q;
    return r;
  };
  if (piece < n_pieces) {
    uint32_t l = sl[piece / per - g * NC_FNV_GROUP];
    if (piece % per) l = maps[(size_t)(piece - 1u) * 256u + l];
    const uint32_t w1 = min(n, (piece + 1u) * NC_FNV_PIECE);
    for (uint32_t i = piece * NC_FNV_PIECE; i < w1; ++i) {
      const uint32_t w = words[i];
#pragma unroll
      for (int b = 0; b < 32; b += 8) {
        const uint32_t x = l ^ ((w >> b) & 255u);
        c = (c + (unsigned long long)(long long)((int32_t)x - (int32_t)l)) * NC_FNV_P;
        l = (x * 0xB3u) & 255u;
      }
    }
    c *= power(4ull * (n - w1));
    if (piece == 0u) c += power(4ull * n) * h0;
  }
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (lane == 0) atomicAdd(sum, c);
}
