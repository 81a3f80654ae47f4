// The group forms of the step: a workgroup of several waves works on the
// slices of one group together.
//
//   k_neuron_wide  the neuron phase with a workgroup of W waves per slice
//                  (k_fanout follows as after k_neuron)
//   k_net_steps    a workgroup per network, for networks of up to NSL slices:
//                  every step of the call in one launch
//
// Both do what nc_neuron_slice does, in its order, with its results, for
// in-degrees up to 32 * NC_GW.  Wave i < slices owns slice i of the group: a
// lane per neuron, which sums the charge, decides the fire and writes the
// neuron's state.  What a wave of k_neuron does one fired lane and one batch
// of 64 arrivals after the other is shared by all waves through LDS:
//   post-side STDP  two fired lanes' rows per wave at a time, or four or
//                   eight when many fired
//   arrivals        a lane per bucket entry, whose record's weight was read
//                   while the owners summed the charge; mask bits and the new
//                   active slots go to their owner through LDS
// k_net_steps keeps the potentials, last fires, caches, active masks and the
// counts of the arrival buckets and pending lists in registers and LDS
// between the steps, so that a step reads only what is due in it, and a
// workgroup barrier takes the place of the kernel boundary.
//
// What bounds them, and what they measured (us per step):
//   k_neuron_wide: the chain of dependent reads (count and entries, masks,
//     records past the cache, rows) on a device that k_neuron's one wave per
//     slice leaves mostly idle, where each of a slice's 16 fired lanes and 6
//     batches of spikes added its own.  20 000 neurons, a quarter firing:
//     the neuron phase 50.4 -> 17.0, of which about 4 is the launch.  (With
//     the owner's masks read beside the entries, the entries' records in
//     flight over the charge and no barrier before it: 18.2 -> 17.0.)  For many
//     slices (19 200) it is the traffic of the fired lanes' rows: 301 -> 264.
//   k_net_steps: quiet networks the barrier and the LDS round trips of one
//     step (300 neurons: 6.9 -> 1.9); busy ones one compute unit's misses and
//     instructions (1000 neurons: 53 -> 23.6, of which the rows' records take
//     a quarter at about 12 bytes a clock).
#pragma once
#include "nc_kernels.h"

#define NC_GW 8       // active-mask words per lane: in-degrees up to 256
// arrivals of a lane and step kept for the next cache (more: read back from the records)
// (eight where waves wait for one another and the LDS holds them)
#define NC_GARR(w, res) ((res) || (w) == 1 ? 4 : 8)
#define NC_GREC 6     // slot records past the cache an owner lane reads together
#define NC_GTAB 2048  // trace-table entries k_net_steps stages in LDS, per table

// A network of k_net_steps: its slices are records act0 .. act0 + nq - 1.
struct nc_net_rec {
  uint32_t act0, nq, net, pad;
};

// A workgroup barrier for what its waves hand over in LDS: reads from memory
// stay in flight across it, and stores are not waited for.
__device__ __forceinline__ void nc_lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int NSL, int W, bool RES>
struct nc_gsh {
  uint32_t keepw[NSL][NC_GW][64];  // active-mask words
  uint32_t dirty[NSL][64];         // words that differ from memory's
  float trt[NSL][64];              // target trace at the step (0: none)
  int32_t lfo[RES ? NSL : 1][RES ? 64 : 1];  // last fire before the step
  uint32_t narr[NSL][64];          // arrivals of the step
  uint2 arr[NSL][64][NC_GARR(W, RES)];  // the first of them: {in-slot, depolarisation}
  uint32_t nrow[3];                // fired lanes, by the step modulo 3 (see below)
  uint32_t row[NSL * 64];          // fired lanes: slice << 6 | lane
  uint32_t rdeg[NSL * 64];         // their in-degrees
  uint32_t any[3];                 // the step has arrivals
  uint32_t soff[NSL];              // first slot of each slice
  unsigned long long fm;           // (one slice) its fired lanes
  uint2 rout[RES ? NSL * 64 : 1];  // fired lanes' out-rows
  uint32_t bcnt[RES ? NSL : 1][RES ? NC_NB : 1];
  uint32_t pcnt[RES ? NSL : 1][2];
  uint32_t que[RES ? W : 1][RES ? 320 : 1];  // per wave: edges to fire (at most 63 left over and 4 * 64 new)
  float tpre[RES ? NC_GTAB + 1 : 1], tpost[RES ? NC_GTAB : 1];
};

// A bucket entry of the step, its target's last fire, and its slot's weight
// (where the entry's may be stale) and sign class.
struct nc_gent {
  uint2 be;
  float w;
  uint32_t inh;
  int32_t lf;
  bool on, stale;
};
// Step of the fire behind an entry taken up at step s.
__device__ __forceinline__ int32_t nc_gent_fire(uint32_t x, int32_t s) { return s - (int32_t)(((x >> 24) & 63u) + 1u); }

__device__ __forceinline__ void nc_gent_slot(uint32_t rel, uint32_t& tl, uint32_t& k) {
  tl = (rel & (64u * NC_CHUNK - 1u)) >> NC_CHUNK_LOG;
  k = ((rel >> (6 + NC_CHUNK_LOG)) << NC_CHUNK_LOG) | (rel & (NC_CHUNK - 1u));
}

// One arrival at step s, taken up by any lane: pre-side STDP, the active bit
// and the new active slot for the lane that owns it.
template <int NSL, int W, bool RES>
__device__ __forceinline__ void nc_gtake(const nc_step_args& a, nc_gsh<NSL, W, RES>& sh, uint32_t sl, uint32_t tl,
                                         uint32_t k, float w, uint32_t inh, uint32_t depol, float pre_f, float post_f,
                                         float lr) {
  const float tr = sh.trt[sl][tl];
  if (tr != 0.0f) {
    const float wn = nc_stdp(w, inh, 0.0f, tr, pre_f, post_f, lr);
    if (__float_as_uint(wn) != __float_as_uint(w)) a.slots[nc_slot_of(sh.soff[sl], tl, k)].w = wn;
  }
  atomicOr(&sh.keepw[sl][k >> 5][tl], 1u << (k & 31u));
  if (!RES) atomicOr(&sh.dirty[sl][tl], 1u << (k >> 5));
  const uint32_t at = atomicAdd(&sh.narr[sl][tl], 1u);
  if (at < NC_GARR(W, RES)) sh.arr[sl][tl][at] = make_uint2(k, depol);
}

// What an owner lane keeps of its neuron.
struct nc_glane {
  uint2 nw, orow;
  float V;
  int32_t lf;
  uint32_t nid, pos, nmw, fires;
  uint4 cache;
  float V_in, tr;  // tr: the target trace at the step of a neuron that does not fire in it
  int32_t lf_in;
};

// The step s (step ci of the call) of the group's nsl slices.  gword: the
// owner lane's group-spike-train word; f_in, f_bg: its host-scheduled fires;
// rec_i, soff0, b_n0: the slice's place among the active ones, its first slot
// and its bucket's count (not resident).
template <int NSL, int W, bool RES, uint32_t BC>
__device__ __forceinline__ void nc_group_step(const nc_step_args& a, nc_gsh<NSL, W, RES>& sh, const nc_netdesc& nd,
                                              uint32_t nsl, uint32_t q0, uint32_t wv, uint32_t lane, int32_t s,
                                              int32_t ci, nc_glane& L, uint32_t sm, uint32_t* mrow,
                                              uint32_t pend_n, uint32_t gword, bool f_in, bool f_bg,
                                              const float* tpre, const float* tpost, uint32_t rec_i, uint32_t soff0,
                                              uint32_t b_n0) {
  const uint32_t par = (uint32_t)ci & 1u, ph = (uint32_t)ci % 3u;
  const bool owner = wv < nsl;
  // the waves of slice xs: xs, xs + nsl, ...; the owner takes the last share of
  // its entries, as it has the charge to sum
  const uint32_t xs = wv % nsl, nsub = (W - 1u - xs) / nsl + 1u, sub = wv < nsl ? nsub - 1u : wv / nsl - 1u;
  const uint32_t xq = q0 + xs;
  const size_t bi = (size_t)xq * NC_NB + ((uint32_t)s & (NC_NB - 1u));
  uint32_t* const pl = (((uint32_t)s >> NC_PEND_LOG_W) & 1u) ? a.pend1 : a.pend0;
  const float lr = nd.lr, pre_f = nd.pre_f, post_f = nd.post_f;
  const int32_t lf0 = L.lf;  // last fire before the step

  // The wave's first 64 entries of its slice's bucket.  A weight that may
  // have changed since the fire (the target fired since, or the host wrote
  // it) is read now, beside the owners' charge: what may still change it in
  // this step is the post-side STDP of a target that fires now, whose trace
  // is 0 and which does not use it.
  uint32_t b_n = b_n0;
  if constexpr (RES) b_n = sh.bcnt[xs][(uint32_t)s & (NC_NB - 1u)];
  const uint32_t b_take = min(b_n, BC);
  // (No branch around the reads: an entry whose record is not needed reads its
  // own place again.  They are first used after the fire.)
  auto place = [&](uint32_t i) { return a.bent + (bi * BC + min(i, BC - 1u)); };
  auto entry_of = [&](uint32_t i, uint2 be) {
    nc_gent g;
    const uint2* const own = place(i);
    g.on = i < b_take;
    g.be = be;
    uint32_t tl, k;
    nc_gent_slot(g.be.x & 0xFFFFFFu, tl, k);
    const int32_t sf = nc_gent_fire(g.be.x, s);
    if constexpr (RES) g.lf = sh.lfo[xs][tl];
    else if constexpr (W == 1) g.lf = __shfl(lf0, (int)tl);
    else g.lf = a.last_fire[xq * 64u + tl];
    // (with several waves, beside the last fire that says whether it is needed)
    constexpr bool late = !RES && W > 1;
    if constexpr (!late) g.stale = g.on && (g.lf > sf || sf < nd.whost);
    const bool rd = late ? g.on : g.stale;
    const nc_slot* const r = a.slots + nc_slot_of(RES ? sh.soff[xs] : soff0, tl, k);
    g.w = *(rd ? &r->w : reinterpret_cast<const float*>(&own->y));
    g.inh = g.be.x >> 31;
    if (g.on && sf < nd.whost) g.inh = (uint32_t)r->arr_inh & 1u;  // a host write may have changed it
    return g;
  };
  auto entry = [&](uint32_t i) { return entry_of(i, *place(i)); };
  constexpr bool kOne = !RES && W <= 2;  // every wave has a share of the bucket
  uint2 be0 = make_uint2(0u, 0u);
  if constexpr (kOne) be0 = *place(sub * 64u + lane);
  // The owner's mask words, read beside the entries.
  uint32_t mx[RES ? 1 : NC_GW];
  if constexpr (!RES) {
    if (owner) {
#pragma unroll
      for (uint32_t w = 0; w < NC_GW; ++w) mx[w] = ((sm >> w) & 1u) ? mrow[w * 64] : 0u;
    }
  }
  nc_gent g0;
  g0.on = false;
  // resident counts are at hand; else the entries are read beside the count
  if constexpr (kOne) g0 = entry_of(sub * 64u + lane, be0);
  else if (sub * 64u < (RES ? b_take : BC)) g0 = entry(sub * 64u + lane);

  static_assert(BC <= 128u, "at most two entries per lane of one wave");
  nc_gent g1;
  g1.on = false;
  if (RES && nsub == 1u && b_take > 64u) g1 = entry(64u + lane);

  // The owners: charge_insynapses, charge_passive, fires, AP waveform, as in
  // nc_neuron_slice (active slots past the cache are read four at a time:
  // here waves are few and the chain of reads is what counts).
  uint32_t nk[NC_ACACHE] = {0u, 0u, 0u}, nv[NC_ACACHE] = {0u, 0u, 0u}, ncnt = 0, smk = 0, dirty = 0;
  bool cache_dirty = false, fire = false;
  if (owner) {
    const uint32_t soff = RES ? sh.soff[wv] : soff0;
    const uint2 ac[NC_ACACHE] = {make_uint2(L.cache.x, (uint32_t)s - (((uint32_t)s - L.cache.w) & 255u)),
                                 make_uint2(L.cache.y, (uint32_t)s - (((uint32_t)s - (L.cache.w >> 8)) & 255u)),
                                 make_uint2(L.cache.z, (uint32_t)s - (((uint32_t)s - (L.cache.w >> 16)) & 255u))};
    float V = L.V;
    int32_t lf = L.lf;
    uint32_t idx = 0;
    if constexpr (!RES) {
#pragma unroll
      for (uint32_t w = 0; w < NC_GW; ++w) sh.keepw[wv][w][lane] = mx[w];
    }
    for (uint32_t w0 = 0; w0 < L.nmw; w0 += 2) {
      const uint32_t mw[2] = {sh.keepw[wv][w0][lane], sh.keepw[wv][w0 + 1][lane]};  // zero past the lane's words
      unsigned long long m = ((unsigned long long)mw[1] << 32) | mw[0];
      if (!__ballot(m != 0ull)) continue;
      uint32_t k0 = mw[0], k1 = mw[1];  // bits kept after the releases
      // the next active slot of these words, ascending
      auto pop = [&]() {
        const uint32_t p = (uint32_t)__builtin_ctzll(m);
        m &= m - 1;
        return p;
      };
      // kept slots come in ascending order: the next place of the cache
      auto charge = [&](uint32_t p, uint32_t depol, uint32_t arr) {
        const float inc = a.dt * __uint_as_float(depol);
        V = (float)((double)V + ((double)inc * a.c0) * a.e);
        const bool rel = s - (int32_t)arr >= a.r_rel;
        const uint32_t bit = rel ? 1u << (p & 31u) : 0u;
        if (p < 32u) k0 &= ~bit;
        else k1 &= ~bit;
        cache_dirty |= rel;
        const uint32_t key = (32u * w0 + p) | (arr << 24), at = rel ? NC_ACACHE : ncnt;
#pragma unroll
        for (int e = 0; e < NC_ACACHE; ++e) {
          nk[e] = at == (uint32_t)e ? key : nk[e];
          nv[e] = at == (uint32_t)e ? depol : nv[e];
        }
        ncnt += at < NC_ACACHE ? 1u : 0u;
      };
#pragma unroll
      for (int e = 0; e < NC_ACACHE; ++e)
        if (idx == (uint32_t)e && m) {
          charge(pop(), ac[e].x, ac[e].y);
          ++idx;
        }
      while (m) {
        uint32_t p[NC_GREC];
        uint2 dv[NC_GREC];
        uint32_t cnt = 0;
#pragma unroll
        for (int e = 0; e < NC_GREC; ++e) {
          p[e] = e ? p[0] : 0u;
          if (m) {
            p[e] = pop();
            cnt = e + 1;
          }
        }
        // no branch around the reads (the first slot again past the last)
#pragma unroll
        for (int e = 0; e < NC_GREC; ++e) {
          const nc_slot& r = a.slots[nc_slot_of(soff, lane, 32u * w0 + p[e])];
          dv[e] = make_uint2(__float_as_uint(r.depol), (uint32_t)(r.arr_inh >> 1));
        }
#pragma unroll
        for (int e = 0; e < NC_GREC; ++e)
          if ((uint32_t)e < cnt) charge(p[e], dv[e].x, dv[e].y);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const uint32_t w = w0 + u, kept = u ? k1 : k0;
        if (kept != mw[u]) {
          sh.keepw[wv][w][lane] = kept;
          dirty |= 1u << w;
        }
      }
    }
    V = (V - NC_BASELEVEL) * a.P + NC_BASELEVEL;

    const uint32_t dw = L.nw.x;
    const bool valid = (dw & NC_DEG_VALID) != 0;
    if (valid && (dw & NC_DEG_INPUT)) f_in |= ((gword >> (L.nw.y & 31u)) & 1u) != 0;
    if (valid && nd.bg_thr) {
      const uint64_t seed = ((uint64_t)nd.bg_hi << 32) | nd.bg_lo;
      f_bg |= nc_draw(seed, (uint32_t)s, L.nid, NC_STREAM_BG).v[0] < nd.bg_thr;
    }
    const int32_t since = s - lf;
    fire = valid && ((((NC_THRESHOLD < V) || f_bg) && since > a.d_ref) || f_in);
    if (b_take || pend_n) {
      sh.trt[wv][lane] = (!fire && (uint32_t)since < (uint32_t)a.len_post) ? (RES ? tpost[since] : L.tr) : 0.0f;
      sh.narr[wv][lane] = 0u;
      if (!RES) sh.dirty[wv][lane] = 0u;
      if (lane == 0) sh.any[ph] = 1u;
    }
    if (fire) lf = s;
    const int32_t dlf = s - lf;
    if (__ballot(dlf <= a.d_ref)) {
      if (a.d_ref < NC_WAP_K) {
        float v = a.w_ap_k[0];
#pragma unroll
        for (int k = 1; k < NC_WAP_K; ++k) v = (dlf == k) ? a.w_ap_k[k] : v;
        V = dlf <= a.d_ref ? v : V;
      } else if (dlf <= a.d_ref) {
        V = a.w_ap[dlf];
      }
    }
    L.V = V;
    L.lf = lf;
    L.fires += fire ? 1u : 0u;
    const unsigned long long fm = __ballot(fire);
    if (fm) {
      const uint32_t nfl = (uint32_t)__builtin_popcountll(fm);
      uint32_t at = 0;
      if constexpr (NSL == 1) {
        if (lane == 0) sh.nrow[ph] = nfl;
      } else {
        if (lane == 0) at = atomicAdd(&sh.nrow[ph], nfl);
        at = (uint32_t)__shfl((int)at, 0);
      }
      at += (uint32_t)__builtin_popcountll(fm & ((1ull << lane) - 1ull));
      if (fire) {
        sh.row[at] = (wv << 6) | lane;
        sh.rdeg[at] = dw & NC_DEG_MASK;
        if constexpr (RES) sh.rout[at] = L.orow;
      }
      if (!RES && lane == 0) sh.fm = fm;
      if (a.raster_cap) {
        const uint32_t rt = nc_wave_append(fire, a.raster_cnt);
        if (fire && rt < a.raster_cap) {
          a.raster[2ull * rt] = L.pos;
          a.raster[2ull * rt + 1] = (uint32_t)s;
        }
      }
    }
  }
  // Every store to memory of the step before is behind a full barrier of that
  // step (or of the kernel): only LDS is handed over here.
  nc_lds_barrier();
  const uint32_t nr = sh.nrow[ph];
  const bool any = sh.any[ph] != 0u;
  // The counts of the step after next, which were last read before this
  // barrier.  (The next step's are clear already: a wave that is ahead may
  // add to them before this store, as a quiet step has no other barrier.)
  if (threadIdx.x == 0) {
    const uint32_t p2 = ph ? ph - 1u : 2u;
    sh.nrow[p2] = 0u;
    sh.any[p2] = 0u;
  }

  // The slice's fan-out records, as k_neuron leaves them, by the last wave:
  // places now, records after the row passes.
  uint32_t f_n = 0, f_at = 0;
  if (!RES && nr && wv == W - 1u && lane == 0) {
    f_n = a.fsplit_od ? min(NC_FSPLIT, (nr * a.fsplit_od + 63u) >> 6) : 1u;
    // the list whose readers run on this workgroup's XCD: k_fanout's block of
    // four waves takes lists 4b .. 4b + 3 modulo 64, and blocks go round the
    // eight XCDs in turn; in XCD order, one of the XCD's eight
    const uint32_t b = a.xcd_lists ? 8u * (blockIdx.x & 7u) + ((blockIdx.x >> 3) & 7u)
                                   : 4u * (rec_i & 7u) + ((rec_i >> 3) & 3u) + (rec_i & 32u);
    f_at = b * a.fcap + atomicAdd(&a.fired_cnt[(par * NC_FLISTS + b) * NC_FCNT_STRIDE], f_n);
  }

  // Post-side STDP (Neuron::fire's inSynapses loop): two rows per wave, 128
  // slots of each in a round; or, when more lanes fired, 16 lanes per row:
  // four rows per wave, 64 slots of each in a round, while that covers the
  // rows, else eight rows per wave, 32 slots of each.
  const uint32_t lpr = nr <= 2u * W ? 6u : 4u, per = 64u >> lpr;
  const bool deep = W > 1 && lpr == 4u && nr <= 4u * W;
  if (nr) {
    const uint32_t step = 64u << lpr;  // slots between in-slots k and k + (1 << lpr) of a lane
    const uint32_t pass = deep ? 4u : 2u;  // slots of a row a lane takes in a round
    for (uint32_t r0 = wv; r0 < nr; r0 += 2u * W * per) {
      uint32_t j0[2], dg[2], kb[2];  // the lane's first slot of each row (deep: its first and third of one)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const uint32_t r = r0 + W * ((deep ? 0u : per * u) + (lane >> lpr)), rr = min(r, nr - 1u), code = sh.row[rr];
        kb[u] = deep ? 2u * u << lpr : 0u;
        j0[u] = nc_slot_of(sh.soff[code >> 6], code & 63u, lane & ((1u << lpr) - 1u)) + (deep ? 2u * u * step : 0u);
        dg[u] = r < nr ? sh.rdeg[rr] : 0u;
      }
      for (uint32_t k0 = lane & ((1u << lpr) - 1u); __ballot(k0 < max(dg[0], dg[1]));
           k0 += pass << lpr, j0[0] += pass * step, j0[1] += pass * step) {
        nc_slot x[4];
        uint32_t j[4];
        bool in[4];
        float tv[4];
        // no branch around the reads (slot 0 stands in past a row's end)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const uint32_t k = k0 + kb[u >> 1] + ((uint32_t)(u & 1) << lpr);
          in[u] = k < dg[u >> 1];
          // 16 or 64 slots on: whole chunks
          j[u] = in[u] ? j0[u >> 1] + ((u & 1) ? step : 0u) : 0u;
          x[u] = a.slots[j[u]];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int32_t ar = x[u].arr_inh >> 1;
          const int32_t la = (uint32_t)(ar - 1) < (uint32_t)(s - 1) ? ar : x[u].last_arr;
          const int32_t d = s - la;
          if constexpr (RES) {
            tv[u] = tpre[min((uint32_t)d, (uint32_t)a.len_pre)];  // a zero follows the table
          } else {
            tv[u] = tpre[min((uint32_t)d, (uint32_t)a.len_pre - 1u)];
            tv[u] = (uint32_t)d < (uint32_t)a.len_pre ? tv[u] : 0.0f;
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float wn = nc_stdp(x[u].w, (uint32_t)x[u].arr_inh & 1u, tv[u], 0.0f, pre_f, post_f, lr);
          if (in[u] && __float_as_uint(wn) != __float_as_uint(x[u].w)) a.slots[j[u]].w = wn;
        }
      }
    }
    // No barrier: the arrivals below write no weight of a lane that fired now,
    // and k_net_steps has one before its fan-out reads these.
  }

  if (!RES && f_n) {
    const unsigned long long fm = sh.fm;
    uint4 f = make_uint4((uint32_t)fm, (uint32_t)(fm >> 32), (uint32_t)s, xq | ((f_n - 1u) << 28));
    if (nr == 1u) {
      const uint2 o = a.out_row[xq * 64u + (uint32_t)__builtin_ctzll(fm)];
      f.x = o.x;
      f.y = o.y;
      f.w |= NC_FSINGLE;
    }
    for (uint32_t i = 0; i < f_n; ++i) a.fired[f_at + i] = make_uint4(f.x, f.y, f.z, f.w | (i << 24));
  }

  // Arrivals (Synapse::run): the buckets' entries, then the pending lists'.
  if (any) {
    for (uint32_t i = sub * 64u + lane; i - lane < b_take; i += nsub * 64u) {
      const nc_gent g = i == sub * 64u + lane ? g0 : RES ? g1 : entry(i);
      if (g.on) {
        uint32_t tl, k;
        nc_gent_slot(g.be.x & 0xFFFFFFu, tl, k);
        const int32_t sf = nc_gent_fire(g.be.x, s);
        const bool stale = (!RES && W > 1) ? g.lf > sf || sf < nd.whost : g.stale;
        nc_gtake<NSL, W, RES>(a, sh, xs, tl, k, stale ? g.w : __uint_as_float(g.be.y),
                              g.inh, __float_as_uint(a.depol_k * __uint_as_float(g.be.y)), pre_f, post_f, lr);
      }
    }
    if (owner && pend_n) {
      uint32_t* const p = pl + sh.soff[wv];
      uint32_t kept = 0;  // compacted in place: write index <= read index
      for (uint32_t t0 = 0; t0 < pend_n; t0 += 64) {
        const uint32_t t = t0 + lane, e = t < pend_n ? p[t] : 0u;
        const bool ev = t < pend_n && (e & 255u) == ((uint32_t)s & 255u);
        if (ev) {
          uint32_t tl, k;
          nc_gent_slot(e >> 8, tl, k);
          const nc_slot r = a.slots[nc_slot_of(sh.soff[wv], tl, k)];
          nc_gtake<NSL, W, RES>(a, sh, wv, tl, k, r.w, (uint32_t)r.arr_inh & 1u, __float_as_uint(r.depol), pre_f, post_f,
                             lr);
        }
        const bool keep = t < pend_n && !ev;
        const unsigned long long km = __ballot(keep);
        const uint32_t to = kept + (uint32_t)__builtin_popcountll(km & ((1ull << lane) - 1ull));
        if (keep && to != t) p[to] = e;
        kept += (uint32_t)__builtin_popcountll(km);
      }
      const uint32_t plist = ((uint32_t)s >> NC_PEND_LOG_W) & 1u;
      if (lane == 0) {
        if constexpr (RES) sh.pcnt[wv][plist] = kept;
        else reinterpret_cast<uint32_t*>(&a.pend_cnt[q0 + wv])[plist] = kept;
      }
    }
    // the weights written above are read in this kernel only where it goes on
    // to the next step
    if constexpr (RES) __syncthreads();
    else nc_lds_barrier();
  }

  // The owners: the next cache and, unless the group stays resident, the
  // changed mask words, their summary and the cache.
  if (owner) {
    const uint32_t na = (b_take || pend_n) ? sh.narr[wv][lane] : 0u;
    if (na) {
      cache_dirty = true;
      if (na <= NC_GARR(W, RES)) {
        for (uint32_t i = 0; i < na; i += 4u) {
          uint2 e[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) e[u] = sh.arr[wv][lane][i + u];
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (i + u < na) nc_push(nk, nv, ncnt, e[u].x, (uint32_t)s, e[u].y);
        }
      } else {
        // the first active slots (more arrived than the cache holds) from
        // their records, read together
        uint32_t k[NC_ACACHE];
        ncnt = 0;
        for (uint32_t w = 0; w < L.nmw && ncnt < NC_ACACHE; ++w)
          for (uint32_t m = sh.keepw[wv][w][lane]; m && ncnt < NC_ACACHE; m &= m - 1) {
            const uint32_t at = 32u * w + (uint32_t)__builtin_ctz(m);
#pragma unroll
            for (int e = 0; e < NC_ACACHE; ++e) k[e] = ncnt == (uint32_t)e || ncnt == 0u ? at : k[e];
            ++ncnt;
          }
        nc_slot r[NC_ACACHE];
#pragma unroll
        for (int e = 0; e < NC_ACACHE; ++e) r[e] = a.slots[nc_slot_of(sh.soff[wv], lane, k[e])];
#pragma unroll
        for (int e = 0; e < NC_ACACHE; ++e) {
          nk[e] = k[e] | ((uint32_t)(r[e].arr_inh >> 1) << 24);
          nv[e] = __float_as_uint(r[e].depol);
        }
      }
    }
    if (cache_dirty)
      L.cache = make_uint4(nv[0], nv[1], nv[2], (nk[0] >> 24) | ((nk[1] >> 24) << 8) | ((nk[2] >> 24) << 16));
    if constexpr (RES) {
      if (lane == 0 && b_n) sh.bcnt[wv][(uint32_t)s & (NC_NB - 1u)] = 0u;
      sh.lfo[wv][lane] = L.lf;
    } else {
      if (b_take || pend_n) dirty |= sh.dirty[wv][lane];
      uint32_t x[NC_GW];
#pragma unroll
      for (uint32_t w = 0; w < NC_GW; ++w) x[w] = sh.keepw[wv][w][lane];  // zero past the lane's words
#pragma unroll
      for (uint32_t w = 0; w < NC_GW; ++w) {
        if ((dirty >> w) & 1u) mrow[w * 64] = x[w];
        if (x[w]) smk |= 1u << w;
      }
      if (cache_dirty) a.acache[L.pos] = L.cache;
      if (smk != sm) a.asum[L.pos] = smk;
      if (lane == 0 && b_n) a.bcnt[bi] = 0u;
    }
  }

  // Synapse::fire on the fired lanes' out-edges: the latches in the same way
  // (most are taken: a synapse carries one spike at a time); the edges whose
  // latch is free queue up in LDS and are fired 64 at a time.
  if constexpr (RES) {
    if (nr) {
      __syncthreads();  // the buckets' counts were reset above
      uint32_t qn = 0;
      uint32_t* const que = sh.que[wv];
      auto fire_edge = [&](uint32_t e) {
        const nc_edge ed = a.edges[e];
        const nc_slot x = a.slots[ed.j];
        const uint32_t d = ed.tq_d & 0xffu, tq = ed.tq_d >> 8;
        const int32_t arr = s + (int32_t)d, prev = x.arr_inh >> 1;
        uint32_t at = BC;
        if (d <= NC_NB) at = atomicAdd(&sh.bcnt[tq - q0][(uint32_t)arr & (NC_NB - 1u)], 1u);
        nc_slot n;
        n.w = x.w;
        n.depol = a.depol_k * x.w;
        n.last_arr = prev != NC_NEVER ? prev : x.last_arr;
        n.arr_inh = arr * 2 + (x.arr_inh & 1);
        a.slots[ed.j] = n;
        a.edges[e].arr = arr;
        if (at < BC) {
          a.bent[((size_t)tq * NC_NB + ((uint32_t)arr & (NC_NB - 1u))) * BC + at] =
              make_uint2(ed.rel | ((d - 1u) << 24) | ((uint32_t)(x.arr_inh & 1) << 31), __float_as_uint(x.w));
        } else {
          const uint32_t plist = ((uint32_t)arr >> NC_PEND_LOG_W) & 1u;
          const uint32_t pt = atomicAdd(&sh.pcnt[tq - q0][plist], 1u);
          (plist ? a.pend1 : a.pend0)[ed.j - ed.rel + pt] = (ed.rel << 8) | ((uint32_t)arr & 255u);
        }
      };
      const uint32_t pass = deep ? 4u : 2u;
      for (uint32_t r0 = wv; r0 < nr; r0 += 2u * W * per) {
        uint2 o[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint32_t r = r0 + W * ((deep ? 0u : per * u) + (lane >> lpr));
          o[u] = sh.rout[min(r, nr - 1u)];
          if (r >= nr) o[u].y = 0u;
        }
        for (uint32_t i0 = lane & ((1u << lpr) - 1u); __ballot(i0 < max(o[0].y, o[1].y)); i0 += pass << lpr) {
          uint32_t e[4];
          bool in[4];
          int32_t lat[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const uint32_t i = i0 + ((deep ? (uint32_t)u : (uint32_t)(u & 1)) << lpr);
            in[u] = i < o[u >> 1].y;
            e[u] = in[u] ? o[u >> 1].x + i : 0u;
            lat[u] = a.edges[e[u]].arr;
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const bool acc = in[u] && lat[u] + a.r_rel <= s;
            const unsigned long long m = __ballot(acc);
            if (acc) que[qn + (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1ull))] = e[u];
            qn += (uint32_t)__builtin_popcountll(m);
          }
          __builtin_amdgcn_wave_barrier();
          while (qn >= 64u) {
            qn -= 64u;
            fire_edge(que[qn + lane]);
          }
        }
      }
      if (lane < qn) fire_edge(que[lane]);
      __syncthreads();
    }
  }
}

// The neuron phase of one step, a workgroup of W waves per active slice.
template <int W, uint32_t BC>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(6))) void k_neuron_wide(nc_step_args a) {
  __shared__ nc_gsh<1, W, false> sh;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t i = nc_block_id(a.xcd_swizzle + nc_have_neuron_args(a));
  const nc_slice_rec rec = a.active_slices[i];
  const uint32_t q = nc_slice_of(a, rec, i);
  nc_glane L;
  L.pos = q * 64u + lane;
  uint32_t sm = 0;
  uint2 pc = make_uint2(0u, 0u);
  if (wv == 0) {
    L.nw = a.ndw[L.pos];
    L.V = L.V_in = a.V[L.pos];
    L.lf = L.lf_in = a.last_fire[L.pos];
    L.cache = a.acache[L.pos];
    L.nid = a.nid[L.pos];
    sm = a.asum[L.pos];
    pc = a.pend_cnt[q];
  }
  const nc_netdesc nd = a.nets[nc_net_of(a, rec)];
  const int32_t ci = (int32_t)*a.chunk_off + a.chunk_i;
  const uint32_t par = (uint32_t)ci & 1u;
  const int32_t s = nd.base_step + ci + 1;
  const uint32_t b_n = a.bcnt[(size_t)q * NC_NB + ((uint32_t)s & (NC_NB - 1u))];
  // (after the uniform reads: a store before them would make them vector reads)
  if (i == 0 && threadIdx.x < NC_FLISTS) a.fired_cnt[((par ^ 1u) * NC_FLISTS + threadIdx.x) * NC_FCNT_STRIDE] = 0u;
  if (ci >= nd.remaining) return;  // the whole workgroup: one network
  uint32_t gword = 0;
  bool f_in = false, f_bg = false;
  L.fires = 0;
  if (wv == 0) {
    L.tr = a.t_post[min(max(s - L.lf, 0), a.len_post - 1)];
    L.nmw = ((L.nw.x & NC_DEG_MASK) + 31u) >> 5;
    gword = a.gfire[(size_t)((uint32_t)ci & (NC_GRING - 1u)) * a.gwords +
                    ((L.nw.x & NC_DEG_INPUT) ? (L.nw.y >> 5) : 0u)];
    if (a.use_forced) {
      const uint32_t wi = a.forced_in[L.pos >> 5], wb = a.forced_bg[L.pos >> 5];
      const bool valid = (L.nw.x & NC_DEG_VALID) != 0;
      f_in = valid && ((wi >> (L.pos & 31)) & 1u);
      f_bg = valid && ((wb >> (L.pos & 31)) & 1u);
      if ((L.pos & 31) == 0) {
        if (wi) a.forced_in[L.pos >> 5] = 0u;
        if (wb) a.forced_bg[L.pos >> 5] = 0u;
      }
    }
  }
  if (threadIdx.x == 0) {
    for (int i = 0; i < 3; ++i) sh.nrow[i] = sh.any[i] = 0u;
    sh.soff[0] = rec.slot_off;
  }
  // No barrier: before the step's first one, only wave 0 reads these (the
  // other waves have rec.slot_off itself).
  const uint32_t pend_n = (((uint32_t)s >> NC_PEND_LOG_W) & 1u) ? pc.y : pc.x;
  nc_group_step<1, W, false, BC>(a, sh, nd, 1u, q, wv, lane, s, ci, L, sm, a.amask + rec.mask_off + lane, pend_n, gword,
                             f_in, f_bg, a.t_pre, a.t_post, i, rec.slot_off, b_n);
  if (wv == 0 && (L.nw.x & NC_DEG_VALID)) {
    if (__float_as_uint(L.V) != __float_as_uint(L.V_in)) a.V[L.pos] = L.V;
    if (L.fires) {
      a.last_fire[L.pos] = L.lf;
      __hip_atomic_fetch_add(&a.firings[L.pos], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// Steps c0 .. c0 + len - 1 of the call for network blockIdx.x, whose slices
// the workgroup keeps.  ev_step: the step (0-based) of each host event of the
// call; a network's are events ev0 .. ev1 - 1 of its record, ascending (in one
// list by step for all networks every owner wave went through every network's:
// 256 networks of 300 neurons with 15 events a step each 114 us a step, 19 so).
template <int NSL, int W, uint32_t BC>
__global__ __launch_bounds__(64 * W) void k_net_steps(nc_step_args a, const nc_net_rec* nets, const uint32_t* ev_step,
                                                      uint32_t c0, uint32_t len) {
  extern __shared__ __align__(16) unsigned char sh_raw[];
  nc_gsh<NSL, W, true>& sh = *reinterpret_cast<nc_gsh<NSL, W, true>*>(sh_raw);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const nc_net_rec nr = nets[blockIdx.x];
  const nc_netdesc nd = a.nets[nr.net];
  const uint32_t end = min(c0 + len, (uint32_t)max(nd.remaining, 0));
  if (c0 >= end) return;  // the whole workgroup
  const uint32_t nsl = nr.nq;
  const nc_slice_rec rec = a.active_slices[nr.act0 + (wv < nsl ? wv : 0u)];
  const uint32_t q0 = a.active_slices[nr.act0].q;
  const bool owner = wv < nsl;
  uint32_t* const mrow = a.amask + rec.mask_off + lane;
  nc_glane L;
  L.pos = (q0 + (owner ? wv : 0u)) * 64u + lane;
  L.nw = a.ndw[L.pos];
  L.V = L.V_in = a.V[L.pos];
  L.lf = L.lf_in = a.last_fire[L.pos];
  L.cache = a.acache[L.pos];
  L.nid = a.nid[L.pos];
  L.orow = a.out_row[L.pos];
  L.fires = 0;
  L.nmw = ((L.nw.x & NC_DEG_MASK) + 31u) >> 5;
  if (owner) {
    const uint32_t sm = a.asum[L.pos];
    for (uint32_t w = 0; w < NC_GW; ++w)
      sh.keepw[wv][w][lane] = (w < L.nmw && ((sm >> w) & 1u)) ? mrow[w * 64] : 0u;
    sh.lfo[wv][lane] = L.lf;
    sh.bcnt[wv][lane] = a.bcnt[(size_t)(q0 + wv) * NC_NB + lane];
    if (lane == 0) {
      const uint2 pc = a.pend_cnt[q0 + wv];
      sh.pcnt[wv][0] = pc.x;
      sh.pcnt[wv][1] = pc.y;
      sh.soff[wv] = rec.slot_off;
    }
  }
  static_assert(NC_NB == 64u, "a lane per bucket count");
  for (uint32_t i = threadIdx.x; i <= (uint32_t)a.len_pre; i += 64 * W)
    sh.tpre[i] = i < (uint32_t)a.len_pre ? a.t_pre[i] : 0.0f;
  for (uint32_t i = threadIdx.x; i < (uint32_t)a.len_post; i += 64 * W) sh.tpost[i] = a.t_post[i];
  if (threadIdx.x == 0) for (int i = 0; i < 3; ++i) sh.nrow[i] = sh.any[i] = 0u;
  const uint32_t* const gw = a.gfire + ((L.nw.x & NC_DEG_INPUT) ? (L.nw.y >> 5) : 0u);
  auto train = [&](uint32_t c) { return owner ? gw[(size_t)(c & (NC_GRING - 1u)) * a.gwords] : 0u; };
  uint32_t next = train(c0);
  uint32_t ev = nd.ev0;  // the first event of the step or later
  if (owner && c0)
    for (uint32_t n = 64; n == 64u; ev += n) {
      n = (uint32_t)__builtin_popcountll(__ballot(ev + lane < nd.ev1 && ev_step[ev + lane] < c0));
    }
  __syncthreads();
  for (uint32_t c = c0; c < end; ++c) {
    const int32_t s = nd.base_step + (int32_t)c + 1;
    const uint32_t gword = next;
    if (c + 1 < end) next = train(c + 1);  // in flight over the step
    bool f_in = false, f_bg = false;
    if (owner) {
      while (ev < nd.ev1) {
        const uint32_t e = ev + lane;
        const bool due = e < nd.ev1 && ev_step[e] == c;
        const uint32_t pos = due ? a.ev_pos[e] : ~0u;
        const uint32_t kind = due ? a.ev_kind[e] : 0u;
        unsigned long long m = __ballot(due && (pos >> 6) == q0 + wv);
        ev += (uint32_t)__builtin_popcountll(__ballot(due));
        while (m) {
          const int l = __builtin_ctzll(m);
          m &= m - 1;
          const uint32_t p = (uint32_t)__shfl((int)pos, l), k = (uint32_t)__shfl((int)kind, l);
          if ((p & 63u) == lane) {
            if (k) f_bg = true;
            else f_in = true;
          }
        }
        if (!__shfl(due ? 1 : 0, 63)) break;
      }
    }
    const uint32_t pend_n = owner ? sh.pcnt[wv][((uint32_t)s >> NC_PEND_LOG_W) & 1u] : 0u;
    nc_group_step<NSL, W, true, BC>(a, sh, nd, nsl, q0, wv, lane, s, (int32_t)c, L, 0u, mrow, pend_n, gword, f_in, f_bg,
                                sh.tpre, sh.tpost, 0u, 0u, 0u);
  }
  __syncthreads();
  if (threadIdx.x == 0) nc_report(a, sh.nrow[(end - 1u) % 3u] >= NC_BUSY_LANES * nsl);
  if (owner) {
    uint32_t smk = 0;
    for (uint32_t w = 0; w < L.nmw; ++w) {
      const uint32_t x = sh.keepw[wv][w][lane];
      mrow[w * 64] = x;
      if (x) smk |= 1u << w;
    }
    a.asum[L.pos] = smk;
    a.acache[L.pos] = L.cache;
    a.bcnt[(size_t)(q0 + wv) * NC_NB + lane] = sh.bcnt[wv][lane];
    if (lane == 0) a.pend_cnt[q0 + wv] = make_uint2(sh.pcnt[wv][0], sh.pcnt[wv][1]);
    if (L.nw.x & NC_DEG_VALID) {
      a.V[L.pos] = L.V;
      a.last_fire[L.pos] = L.lf;
      if (L.fires) a.firings[L.pos] += L.fires;
    }
  }
}
