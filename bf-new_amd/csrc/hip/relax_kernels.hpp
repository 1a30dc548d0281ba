// relax_kernels.hpp -- the relaxation visits, the round loop and the
// relaxation kernels (persistent and one round per launch) as templates over
// block size, records per thread, instrumentation, wave bound and engine
// set; each relax_<engines>.hip instantiates one engine set, so the variants
// compile in parallel.
//
// Work unit: a slot s = (query q, selected tile T).  One workgroup visits one
// slot at a time.  The tile's edge records (pack, weight) are read once per
// visit, coalesced: the internal records (both ends in T) into registers,
// where they stay for the tile closure (thread t holds records t, t+B, ...),
// the boundary records streamed in chunks.  The distances the visit touches
// are staged in LDS and relaxed there with ds_min_u32 on the order-preserving
// u32 image of the fp32 distance (all distances are +0, finite positive or
// +inf, so unsigned order equals float order).
//
// Semantics (reference engines):
//   Jacobi pull   batched_jacobi.hip.cpp:466-694 -- two columns, round r reads
//                 column r&1 and writes column (r+1)&1:
//                 d'[v] = min(d[v], min over admitted in-edges fl(d[u] + w)).
//                 tile_sweeps = 1 is exactly that (same rounds as the
//                 reference); tile_sweeps = 0 additionally closes the tile's
//                 internal edges in LDS each round (block Jacobi: the same
//                 fixed point, fewer rounds).
//   dense push    batched_dense_chaotic_push.hip.cpp:392-627 -- one column,
//                 in place, atomicMin(d[dst], fl(d[src] + w)) over every
//                 admitted out-edge of a dirty tile.
//   frontier push batched_frontier_push.hip.cpp:710-906 -- as dense, but
//                 only from vertices whose label dropped below the label last
//                 pushed (column 1 holds that snapshot).
// Every schedule reaches the same bits: fl(x + w) is monotone in x, so the
// relaxation operator has one greatest fixed point.
//
// Admission: a neighbour tile that the query did not select is staged as
// +inf (pull) or has no slot (push), so edges from or to it never relax.
#pragma once

#include "bfn_internal.hpp"

namespace bfn {

// LDS carve-up (u32 words): [own | orig | work | table | flags], with
// `work` = staged neighbour slabs (pull), or the pushed snapshot followed by
// the boundary proposal slabs (push), and `table` = per-neighbour LDS offsets
// (pull) or neighbour slots, "pushed into" marks and proposal slab offsets
// (push).
struct Lds {
  std::uint32_t* own;
  std::uint32_t* orig;
  std::uint32_t* work;
  std::uint32_t* prop;   // push, proposals: the boundary proposal slabs
  std::uint32_t* bnd;    // push, direct: boundary record start per vertex
  std::uint32_t* list;   // push, direct: the visit's pushing vertices
  std::uint32_t* slots;  // per neighbour: its slot (push) / staged slab offset (pull)
  std::uint32_t* marks;  // per neighbour: pushed into during this visit
  std::uint32_t* offs;   // per neighbour: pool offset (two words) / proposal slab offset
  std::uint32_t* flags;
};

__device__ __forceinline__ Lds carve(std::uint32_t* base, std::uint32_t max_v,
                                     std::uint32_t work_words, std::uint32_t max_neighbor_tiles) {
  const std::uint32_t k = lds_table_entries(max_neighbor_tiles);
  Lds l;
  l.own = base;
  l.orig = base + max_v;
  l.work = base + 2 * max_v;
  l.prop = l.work + max_v;
  l.bnd = l.work + max_v;
  l.list = l.work + 2 * max_v;
  l.slots = l.work + work_words;
  l.marks = l.slots + k;
  l.offs = l.marks + k;
  l.flags = l.offs + 2 * k;
  return l;
}

// Boundary records per pushing vertex loaded together (one load, then one
// filter read, in flight per record).  Six covers a vertex of the tiled
// routing graphs (four intra-tile and six inter-tile edges per node) in one
// chunk, and at six the 256-thread push-only kernel fits 79 VGPRs: six
// workgroups per CU, where eight records per chunk needed 85 (five).
constexpr int kPushChunk = 6;
static_assert(kPushChunk % 2 == 0, "boundary records are loaded in pairs");

// Query q changed in round r, and whether it has work queued for r + 1.
// Every writer of a round stores the same value and later rounds store a
// larger one, so plain stores suffice (an atomic per visit would queue on
// the query's line).
__device__ __forceinline__ void mark_changed(const DevBatch& b, std::uint32_t q, std::uint32_t r,
                                             bool queued) {
  b.last_change[q] = r + 1;
  if (b.pending && queued) b.pending[q] = r + 2;
}

// Edge records in registers: thread t holds records t, t + B, t + 2B, ... of
// the range it loaded.
template <int B, int N>
struct RecordRegs {
  std::uint32_t pack[N];
  float w[N];
};

// Loads records [base, base + N*B) clipped to `end` (kNone past the end).
template <int B, int N>
__device__ __forceinline__ void load_records(RecordRegs<B, N>& r, const uint2* rec,
                                             std::uint32_t base, std::uint32_t end) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const std::uint32_t e = base + j * B + threadIdx.x;
    if (e < end) {
      const uint2 x = rec[e];
      r.pack[j] = x.x;
      r.w[j] = __uint_as_float(x.y);
    } else {
      r.pack[j] = kNone;
      r.w[j] = 0.0f;
    }
  }
}

// Boundary records per thread per streamed chunk (loads in flight per lane):
// more for the large blocks, fewer where registers bound the occupancy.
constexpr int stream_records(int block) { return block >= 512 ? 8 : 4; }

// Per-workgroup counters of the visits, compiled in for instrumented runs
// only (I = true; otherwise every counter is dead code).  Phase clocks are
// shader-clock cycles read by thread 0 at phase boundaries: 0 setup (tables,
// label staging), 1 internal records (pull: first pass), 2 tile closure,
// 3 boundary records, 4 write-back and enqueue.
template <bool I>
struct VisitStats {
  unsigned long long attempts = 0, successes = 0, bytes = 0, edges = 0, items = 0, sweeps = 0,
                     evals = 0;
  unsigned long long phase[kPhaseCount] = {};
  long long t = 0;
  __device__ __forceinline__ void start() {
    if constexpr (I) {
      if (threadIdx.x == 0) t = clock64();
    }
  }
  __device__ __forceinline__ void mark(int p) {
    if constexpr (I) {
      if (threadIdx.x == 0) {
        const long long now = clock64();
        phase[p] += static_cast<unsigned long long>(now - t);
        t = now;
      }
    }
  }
};

// Whether the workgroup takes a visit's slabs one after the other, four
// words per thread in flight, rather than `Slabs` slabs per wave and `Rows`
// 64-word rows of each: the form with fewer round trips (slabs are taken to
// be of the visited tile's size).  It is the one for large tiles with few
// neighbours, where most waves would have no slab.  Relaxation of 24 queries,
// slabs per wave / one after the other: point Jacobi on one tile of 4000
// vertices, 256 threads 421 / 316 us, 1024 threads 293 / 181; dense push
// through proposals on two tiles of 2000, 1024 threads 265 / 221; on 3x3
// tiles of 2000, 1024 threads 382 / 332.
template <int B, std::uint32_t Slabs, std::uint32_t Rows>
__device__ __forceinline__ bool slab_by_slab(std::uint32_t slabs, std::uint32_t words) {
  constexpr std::uint32_t kAtOnce = Slabs * (B / 64);
  // uniform values, said to be so: a branch on them without it cost 2 %
  slabs = __builtin_amdgcn_readfirstlane(slabs);
  words = __builtin_amdgcn_readfirstlane(words);
  return slabs * ((words + 4 * B - 1) / (4 * B)) <
         (words + 64 * Rows - 1) / (64 * Rows) * ((slabs + kAtOnce - 1) / kAtOnce);
}

__device__ __forceinline__ std::uint32_t pk_k(std::uint32_t p) { return p >> 24; }
__device__ __forceinline__ std::uint32_t pk_src(std::uint32_t p) { return (p >> 12) & kPackLocalMask; }
__device__ __forceinline__ std::uint32_t pk_dst(std::uint32_t p) { return p & kPackLocalMask; }

// ---------------------------------------------------------------------------
// Jacobi pull visit.
// ---------------------------------------------------------------------------
template <int B, int EPT, bool I>
__device__ __forceinline__ void visit_pull(const DevGraph& g, const DevBatch& b, const SlotDesc& d,
                           std::uint32_t r, const Lds& l, VisitStats<I>& st) {
  const std::uint32_t tid = threadIdx.x;
  st.start();
  const std::uint32_t q = d.query;
  const std::uint32_t npt = d.npt;
  const std::uint32_t nb0 = d.nbr0;
  const std::uint32_t K = d.nbr_count;
  const std::uint32_t rp = r & 1u;
  const std::uint32_t in_base = d.nbr_base;
  const unsigned long long dist = (static_cast<unsigned long long>(d.dist_hi) << 32) | d.dist_lo;

  // CSC block of T: internal records [e0, ei), boundary records [ei, e1).
  const std::uint32_t e0 = d.e0;
  const std::uint32_t e1 = d.e1;
  const std::uint32_t ei = d.ei;
  const bool resident = ei - e0 <= static_cast<std::uint32_t>(B * EPT);
  // Neighbour k's slab: LDS offset, size and pool offset of its read column,
  // looked up by thread k.  A visit is bound by the latency of its dependent
  // reads, so the table reads of all slabs travel together (two round trips
  // for the list).  Setup of a visit on 256-vertex tiles: 40.1k -> 9.6k
  // cycles; relaxation of 64 queries on 64x64x256 tiles (block Jacobi) 2928
  // -> 2298 us, of 32 point-Jacobi queries on 32x32x128 736 -> 580 us.
  // (Four rows in flight, or the internal records requested before the
  // slabs, take 12 to 26 more registers and measured 2 and 5 % slower.)
  for (std::uint32_t k = tid; k < K; k += B) {
    const std::uint32_t nt = g.in_nbr_tiles[nb0 + k];
    const std::uint32_t ns = b.slot_in[in_base + k];
    const std::uint32_t n = g.tile_vertex_offsets[nt + 1] - g.tile_vertex_offsets[nt];
    unsigned long long off = ~0ull;
    if (ns != kNone) {
      off = b.slot_dist[ns] + static_cast<unsigned long long>(rp) * n;
      st.bytes += 4ull * n;
    }
    l.slots[k] = g.in_nbr_stage[nb0 + k];
    l.marks[k] = n;
    l.offs[2 * k] = static_cast<std::uint32_t>(off);
    l.offs[2 * k + 1] = static_cast<std::uint32_t>(off >> 32);
  }
  __syncthreads();
  // Stage the read column of every in-neighbour slab (k = 0 is T itself).  A
  // wave takes four slabs at a time and keeps two 64-word rows of each in
  // flight, so 4 * B / 64 slabs of up to 128 words (16 at 256 threads) cost
  // one round trip.
  constexpr std::uint32_t kSlabs = 4, kRows = 2, kWaves = B / 64;
  const std::uint32_t lane = tid & 63u, wave = tid >> 6;
  const bool one_by_one = slab_by_slab<B, kSlabs, kRows>(K, npt);
  for (std::uint32_t k = one_by_one ? 0u : K; k < K; ++k) {
    const std::uint32_t n = l.marks[k], at = l.slots[k], hi = l.offs[2 * k + 1];
    const std::uint32_t* src = b.dist + ((static_cast<unsigned long long>(hi) << 32) | l.offs[2 * k]);
    for (std::uint32_t i0 = tid; i0 < n; i0 += 4 * B) {
      std::uint32_t x[4];
#pragma unroll
      for (std::uint32_t r = 0; r < 4; ++r) {
        x[r] = kInfBits;
        if (hi != kNone && i0 + r * B < n) x[r] = src[i0 + r * B];
      }
#pragma unroll
      for (std::uint32_t r = 0; r < 4; ++r)
        if (i0 + r * B < n) {
          l.work[at + i0 + r * B] = x[r];
          if (k == 0) l.own[i0 + r * B] = x[r];
        }
    }
  }
  for (std::uint32_t k0 = one_by_one ? K : wave; k0 < K; k0 += kSlabs * kWaves) {
    const std::uint32_t* src[kSlabs];
    std::uint32_t size[kSlabs], at[kSlabs], longest = 0;
#pragma unroll
    for (std::uint32_t j = 0; j < kSlabs; ++j) {
      const std::uint32_t k = k0 + j * kWaves;
      size[j] = at[j] = 0;
      src[j] = nullptr;
      if (k < K) {
        size[j] = __builtin_amdgcn_readfirstlane(l.marks[k]);
        at[j] = __builtin_amdgcn_readfirstlane(l.slots[k]);
        const std::uint32_t lo = __builtin_amdgcn_readfirstlane(l.offs[2 * k]);
        const std::uint32_t hi = __builtin_amdgcn_readfirstlane(l.offs[2 * k + 1]);
        if (hi != kNone) src[j] = b.dist + ((static_cast<unsigned long long>(hi) << 32) | lo);
        longest = max(longest, size[j]);
      }
    }
    for (std::uint32_t i0 = lane; i0 < longest; i0 += 64 * kRows) {
      std::uint32_t x[kSlabs][kRows];
#pragma unroll
      for (std::uint32_t j = 0; j < kSlabs; ++j)
#pragma unroll
        for (std::uint32_t r = 0; r < kRows; ++r) {
          x[j][r] = kInfBits;
          if (src[j] && i0 + 64 * r < size[j]) x[j][r] = src[j][i0 + 64 * r];
        }
#pragma unroll
      for (std::uint32_t j = 0; j < kSlabs; ++j)
#pragma unroll
        for (std::uint32_t r = 0; r < kRows; ++r)
          if (i0 + 64 * r < size[j]) {
            l.work[at[j] + i0 + 64 * r] = x[j][r];
            if (j == 0 && k0 == 0) l.own[i0 + 64 * r] = x[j][r];
          }
    }
  }
  __syncthreads();
  st.mark(0);

  if (tid == 0) {
    // edge records (pack + weight) once, the written column once
    st.bytes += 8ull * (e1 - e0) + 4ull * npt;
    st.edges += e1 - e0;
  }
  // Pass 1: every admitted in-edge reads the staged read column.
  auto relax_staged = [&](std::uint32_t p, float w) {
    if constexpr (I) ++st.evals;
    const std::uint32_t cb = as_bits(as_float(l.work[l.slots[pk_k(p)] + pk_src(p)]) + w);
    if (cb < l.own[pk_dst(p)]) atomicMin(&l.own[pk_dst(p)], cb);
  };
  // The internal records stay in registers through the tile closure when
  // they fit (resident), and are not kept across visits.  The first boundary
  // chunk travels with them.
  constexpr int kStream = stream_records(B);
  RecordRegs<B, EPT> internal;
  RecordRegs<B, kStream> chunk;
  load_records<B, kStream>(chunk, g.csc_rec, ei, e1);
  if (resident) load_records<B, EPT>(internal, g.csc_rec, e0, ei);
  for (std::uint32_t base = e0; base < ei; base += B * EPT) {
    if (!resident) load_records<B, EPT>(internal, g.csc_rec, base, ei);
#pragma unroll
    for (int j = 0; j < EPT; ++j)
      if (internal.pack[j] != kNone) relax_staged(internal.pack[j], internal.w[j]);
  }
  st.mark(1);
  for (std::uint32_t base = ei; base < e1; base += B * kStream) {
    if (base != ei) load_records<B, kStream>(chunk, g.csc_rec, base, e1);
#pragma unroll
    for (int j = 0; j < kStream; ++j)
      if (chunk.pack[j] != kNone) relax_staged(chunk.pack[j], chunk.w[j]);
  }
  __syncthreads();
  st.mark(3);
  if (b.tile_sweeps == 0) {
    // Close the tile's internal edges in place; the internal records stay in
    // registers when they fit.
    for (;;) {
      bool changed = false;
      for (std::uint32_t base = e0; base < ei; base += B * EPT) {
        if (!resident) load_records<B, EPT>(internal, g.csc_rec, base, ei);
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
          const std::uint32_t p = internal.pack[j];
          if (p == kNone) continue;
          if constexpr (I) ++st.evals;
          const std::uint32_t cb = as_bits(as_float(l.own[pk_src(p)]) + internal.w[j]);
          if (cb < l.own[pk_dst(p)]) {
            atomicMin(&l.own[pk_dst(p)], cb);
            changed = true;
          }
        }
      }
      ++st.sweeps;
      if (!__syncthreads_or(changed)) break;
    }
  }
  st.mark(2);

  std::uint32_t* out = b.dist + dist + static_cast<std::size_t>(rp ^ 1u) * npt;
  bool changed = false;
  for (std::uint32_t i = tid; i < npt; i += B) {
    const std::uint32_t v = l.own[i];
    out[i] = v;
    changed |= (v != l.work[i]);
  }
  if (__syncthreads_or(changed)) {
    if (tid == 0) mark_changed(b, q, r, true);
    // every selected out-neighbour (the tile itself first) reads the new
    // column next round
    for (std::uint32_t j = tid; j < d.out_count; j += B) {
      const std::uint32_t ns = b.slot_out[d.out_base + j];
      if (ns != kNone) enqueue(b, ns, r + 1);
    }
  }
  st.mark(4);
}

// ---------------------------------------------------------------------------
// Dense / frontier push visit.
// ---------------------------------------------------------------------------
template <int B, int EPT, bool I, int M>
__device__ __forceinline__ void visit_push(const DevGraph& g, const DevBatch& b, const SlotDesc& d,
                           std::uint32_t r, bool frontier, const Lds& l,
                           VisitStats<I>& st, std::uint32_t& queued_min) {
  const std::uint32_t tid = threadIdx.x;
  st.start();
  const std::uint32_t q = d.query;
  const std::uint32_t v0 = d.v0;
  const std::uint32_t npt = d.npt;
  const std::uint32_t ob0 = d.nbr0;
  const std::uint32_t KO = d.nbr_count;
  const std::uint32_t out_base = d.nbr_base;
  std::uint32_t* column = b.dist + ((static_cast<unsigned long long>(d.dist_hi) << 32) | d.dist_lo);
  std::uint32_t* snapshot = column + npt;
  // CSR block of T: internal records [e0, ei), boundary records [ei, e1).
  const std::uint32_t e0 = d.e0;
  const std::uint32_t e1 = d.e1;
  const std::uint32_t ei = d.ei;
  const bool resident = ei - e0 <= static_cast<std::uint32_t>(B * EPT);
  // The internal records are requested first, so that they travel together
  // with the label loads below (one round trip for both).  They live only
  // through the tile closure: kept in registers across visits of the same
  // tile they would stay live through the boundary phase too, and those 16
  // VGPRs cost the 256-thread push-only kernel two of its eight workgroups
  // per CU.
  RecordRegs<B, EPT> internal;
  if (resident) load_records<B, EPT>(internal, g.csr_rec, e0, ei);

  const bool proposals = M == kEnginesMixed ? b.boundary_mode == 0 : M == kEnginesPushLds;
  for (std::uint32_t k = tid; k < KO; k += B) {
    const std::uint32_t ns = b.slot_out[out_base + k];
    l.slots[k] = ns;
    l.marks[k] = kInfBits;
    if (proposals) {
      // the neighbour's proposal slab: size and LDS offset (an LDS offset is
      // below 2^16 words, a tile's size at most 2^12)
      const std::uint32_t nt = g.out_nbr_tiles[ob0 + k];
      const std::uint32_t n = k ? g.tile_vertex_offsets[nt + 1] - g.tile_vertex_offsets[nt] : 0u;
      l.offs[k] = (n << 16) | g.out_nbr_stage[ob0 + k];
    } else {
      // pool offset of the neighbour's labels, as two words
      const unsigned long long off =
          b.slot_out_off ? b.slot_out_off[out_base + k] : (ns != kNone ? b.slot_dist[ns] : ~0ull);
      l.offs[2 * k] = static_cast<std::uint32_t>(off);
      l.offs[2 * k + 1] = static_cast<std::uint32_t>(off >> 32);
    }
  }
  // Dense pushes every finite vertex: an infinite snapshot admits them all.
  if (((npt | v0) & 1u) == 0) {
    // Even tile size and first vertex: labels, snapshot and record starts
    // two per 8-byte load (pool offsets are sums of 2 npt, so all even).
    for (std::uint32_t i = 2 * tid; i < npt; i += 2 * B) {
      const unsigned long long x = __hip_atomic_load(
          reinterpret_cast<const unsigned long long*>(column + i), __ATOMIC_RELAXED,
          __HIP_MEMORY_SCOPE_AGENT);
      l.own[i] = l.orig[i] = static_cast<std::uint32_t>(x);
      l.own[i + 1] = l.orig[i + 1] = static_cast<std::uint32_t>(x >> 32);
      const uint2 sn = frontier ? *reinterpret_cast<const uint2*>(snapshot + i)
                                : make_uint2(kInfBits, kInfBits);
      l.work[i] = sn.x;
      l.work[i + 1] = sn.y;
      if (!proposals) {
        const uint2 bd = *reinterpret_cast<const uint2*>(g.csr_bnd + v0 + i);
        l.bnd[i] = bd.x;
        l.bnd[i + 1] = bd.y;
      }
    }
  } else {
    for (std::uint32_t i = tid; i < npt; i += B) {
      const std::uint32_t x = load_agent(column + i);
      l.own[i] = x;
      l.orig[i] = x;
      l.work[i] = frontier ? snapshot[i] : kInfBits;
      if (!proposals) l.bnd[i] = g.csr_bnd[v0 + i];
    }
  }
  if (tid == 0) l.flags[1] = 0;
  __syncthreads();
  if (proposals) {
    // Clear the proposal slabs: they are contiguous, and the tile closure's
    // barriers come before the first proposal.
    const std::uint32_t last = l.offs[KO - 1];
    const std::uint32_t words = (last & 0xFFFFu) + (last >> 16);
    for (std::uint32_t i = tid; i < words; i += B) l.prop[i] = kInfBits;
  }
  st.mark(0);

  if (tid == 0) {
    // internal records once, the column (and the snapshot for frontier)
    // once; proposals stream every boundary record, direct mode reads the
    // record starts and then only the pushing vertices' records
    st.bytes += 8ull * (ei - e0) + 4ull * npt * (frontier ? 2 : 1) +
                (proposals ? 8ull * (e1 - ei) : 4ull * npt);
    st.edges += (ei - e0) + (proposals ? e1 - ei : 0u);
  }
  st.mark(1);
  // Internal edges to the tile's local fixed point, from frontier sources.
  for (;;) {
    bool changed = false;
    for (std::uint32_t base = e0; base < ei; base += B * EPT) {
      if (!resident) load_records<B, EPT>(internal, g.csr_rec, base, ei);
#pragma unroll
      for (int j = 0; j < EPT; ++j) {
        const std::uint32_t p = internal.pack[j];
        if (p == kNone) continue;
        const std::uint32_t sv = l.own[pk_src(p)];
        if (!(sv < l.work[pk_src(p)])) continue;
        if constexpr (I) ++st.evals;
        const std::uint32_t cb = as_bits(as_float(sv) + internal.w[j]);
        if (cb < l.own[pk_dst(p)]) {
          atomicMin(&l.own[pk_dst(p)], cb);
          changed = true;
        }
      }
    }
    ++st.sweeps;
    if (!__syncthreads_or(changed)) break;
  }
  st.mark(2);
  // Boundary records, streamed once.  Labels only fall during a run, so an
  // ordinary (cacheable, possibly stale) load of a neighbour label is never
  // below the current label: comparing against it never drops a decrease, at
  // worst it issues an atomic or marks a neighbour that did not need it.
  unsigned long long att = 0, suc = 0;
  if (proposals) {
    // Gather the best candidate per destination in LDS, then compare each
    // neighbour slab once, coalesced, and issue one atomic per improvement.
    for (std::uint32_t base = ei; base < e1; base += B * stream_records(B)) {
      RecordRegs<B, stream_records(B)> chunk;
      load_records<B, stream_records(B)>(chunk, g.csr_rec, base, e1);
#pragma unroll
      for (int j = 0; j < stream_records(B); ++j) {
        const std::uint32_t p = chunk.pack[j];
        if (p == kNone) continue;
        const std::uint32_t sv = l.own[pk_src(p)];
        if (!(sv < l.work[pk_src(p)])) continue;
        if (l.slots[pk_k(p)] == kNone) continue;
        const std::uint32_t cb = as_bits(as_float(sv) + chunk.w[j]);
        std::uint32_t* slot = &l.prop[(l.offs[pk_k(p)] & 0xFFFFu) + pk_dst(p)];
        ++att;
        if (cb < *slot) atomicMin(slot, cb);
      }
    }
    __syncthreads();
    // A wave compares two slabs at a time, four 64-word rows of each in
    // flight.  (One slab after the other by the whole workgroup, each behind
    // its own table reads, was two thirds of a visit: 41 dense queries on
    // 45x37x301 tiles, relaxation 903 -> 545 us.)
    constexpr std::uint32_t kSlabs = 2, kRows = 4, kWaves = B / 64;
    const std::uint32_t lane = tid & 63u, wave = tid >> 6;
    const bool one_by_one = slab_by_slab<B, kSlabs, kRows>(KO - 1, npt);
    for (std::uint32_t k = one_by_one ? 1u : KO; k < KO; ++k) {
      const std::uint32_t ns = l.slots[k], at = l.offs[k] & 0xFFFFu, n = l.offs[k] >> 16;
      if (ns == kNone) continue;
      std::uint32_t* target = b.dist + (b.slot_out_off ? b.slot_out_off[out_base + k] : b.slot_dist[ns]);
      if (tid == 0) st.bytes += 4ull * n;  // the neighbour slab, read once
      std::uint32_t low = kInfBits;
      for (std::uint32_t i0 = tid; i0 < n; i0 += 4 * B) {
        std::uint32_t seen[4];
#pragma unroll
        for (std::uint32_t r4 = 0; r4 < 4; ++r4) seen[r4] = i0 + r4 * B < n ? target[i0 + r4 * B] : 0u;
#pragma unroll
        for (std::uint32_t r4 = 0; r4 < 4; ++r4) {
          if (i0 + r4 * B >= n) continue;
          const std::uint32_t pv = l.prop[at + i0 + r4 * B];
          if (pv < seen[r4]) {
            atomic_min_agent(target + i0 + r4 * B, pv);
            ++suc;
            low = min(low, pv);
          }
        }
      }
      if (low != kInfBits) atomicMin(&l.marks[k], low);
    }
    for (std::uint32_t k0 = one_by_one ? KO : 1 + wave; k0 < KO; k0 += kSlabs * kWaves) {
      std::uint32_t* target[kSlabs];
      std::uint32_t size[kSlabs], at[kSlabs], low[kSlabs], longest = 0;
#pragma unroll
      for (std::uint32_t j = 0; j < kSlabs; ++j) {
        const std::uint32_t k = k0 + j * kWaves;
        size[j] = at[j] = 0;
        low[j] = kInfBits;
        target[j] = nullptr;
        if (k < KO) {
          const std::uint32_t ns = __builtin_amdgcn_readfirstlane(l.slots[k]);
          const std::uint32_t slab = __builtin_amdgcn_readfirstlane(l.offs[k]);
          if (ns != kNone) {
            at[j] = slab & 0xFFFFu;
            size[j] = slab >> 16;
            target[j] = b.dist + (b.slot_out_off ? b.slot_out_off[out_base + k] : b.slot_dist[ns]);
            longest = max(longest, size[j]);
            if (lane == 0) st.bytes += 4ull * size[j];  // the neighbour slab, read once
          }
        }
      }
      for (std::uint32_t i0 = lane; i0 < longest; i0 += 64 * kRows) {
        std::uint32_t seen[kSlabs][kRows];
#pragma unroll
        for (std::uint32_t j = 0; j < kSlabs; ++j)
#pragma unroll
          for (std::uint32_t r4 = 0; r4 < kRows; ++r4) {
            const std::uint32_t i = i0 + 64 * r4;
            seen[j][r4] = i < size[j] ? target[j][i] : 0u;
          }
#pragma unroll
        for (std::uint32_t j = 0; j < kSlabs; ++j)
#pragma unroll
          for (std::uint32_t r4 = 0; r4 < kRows; ++r4) {
            const std::uint32_t i = i0 + 64 * r4;
            if (i >= size[j]) continue;
            const std::uint32_t pv = l.prop[at[j] + i];
            if (pv < seen[j][r4]) {  // an empty proposal is +inf: never below a label
              atomic_min_agent(target[j] + i, pv);
              ++suc;
              low[j] = min(low[j], pv);
            }
          }
      }
#pragma unroll
      for (std::uint32_t j = 0; j < kSlabs; ++j)
        if (low[j] != kInfBits) atomicMin(&l.marks[k0 + j * kWaves], low[j]);
    }
  } else {
    // Direct mode: only vertices that push (label below the snapshot;
    // dense: finite) read their boundary records.  They are listed in LDS
    // (one claim per wave) and taken one vertex per thread; a vertex's
    // boundary records are consecutive, loaded kPushChunk at a time, then
    // their filter reads are issued together, then one no-return atomic per
    // candidate that beats the label read.  The filter reads are ordinary
    // (cacheable, possibly stale) loads: labels only fall, so a stale label
    // is never below the true one and the filter never drops a decrease; a
    // neighbour is marked when its read label was above a candidate, which
    // covers every actual decrease.  (A returning atomic per candidate in
    // place of the read measured 1.6x slower on 128x128x512 tiles: device-
    // scope atomics are performed past the L2, at the memory side.)
    for (std::uint32_t base = 0; base < npt; base += B) {
      const std::uint32_t i = base + tid;
      const bool push = i < npt && l.own[i] < l.work[i];
      const unsigned long long m = __ballot(push);
      std::uint32_t at = 0;
      if ((tid & 63u) == 0 && m) at = atomicAdd(&l.flags[1], static_cast<std::uint32_t>(__popcll(m)));
      at = __shfl(at, 0);
      if (push) l.list[at + __popcll(m & ((1ull << (tid & 63u)) - 1ull))] = i;
    }
    __syncthreads();
    const std::uint32_t n_push = l.flags[1];
    unsigned long long loaded = 0;
    for (std::uint32_t j = tid; j < n_push; j += B) {
      const std::uint32_t i = l.list[j];
      const float sf = as_float(l.own[i]);
      const std::uint32_t rb = l.bnd[i];
      const std::uint32_t re = i + 1 < npt ? l.bnd[i + 1] : e1;
      loaded += re - rb;
      // Chunks start at even positions, so a lane's records arrive two per
      // 16-byte load (the stream holds one record to spare past its end).
      for (std::uint32_t r0 = rb & ~1u; r0 < re; r0 += kPushChunk) {
        std::uint32_t pk[kPushChunk];
        float w[kPushChunk];
#pragma unroll
        for (int c = 0; c < kPushChunk; c += 2) {
          uint4 x = make_uint4(kNone, 0u, kNone, 0u);
          if (r0 + c < re) x = *reinterpret_cast<const uint4*>(g.csr_rec + r0 + c);
          const bool in0 = r0 + c >= rb && r0 + c < re;
          const bool in1 = r0 + c + 1 >= rb && r0 + c + 1 < re;
          pk[c] = in0 ? x.x : kNone;
          w[c] = in0 ? as_float(x.y) : 0.0f;
          pk[c + 1] = in1 ? x.z : kNone;
          w[c + 1] = in1 ? as_float(x.w) : 0.0f;
        }
        auto target = [&](std::uint32_t p) -> std::uint32_t* {
          const unsigned long long off = (static_cast<unsigned long long>(l.offs[2 * pk_k(p) + 1]) << 32) |
                                         l.offs[2 * pk_k(p)];
          return b.dist + off + pk_dst(p);
        };
        std::uint32_t seen[kPushChunk];
#pragma unroll
        for (int c = 0; c < kPushChunk; ++c) {
          if (pk[c] != kNone && l.slots[pk_k(pk[c])] == kNone) pk[c] = kNone;  // not selected
          seen[c] = pk[c] != kNone ? *target(pk[c]) : 0u;
        }
#pragma unroll
        for (int c = 0; c < kPushChunk; ++c) {
          if (pk[c] == kNone) continue;
          ++att;
          const std::uint32_t cb = as_bits(sf + w[c]);
          if (cb < seen[c]) {
            atomic_min_agent(target(pk[c]), cb);
            ++suc;
            // read first: most candidates into one neighbour lose to its mark
            if (cb < l.marks[pk_k(pk[c])]) atomicMin(&l.marks[pk_k(pk[c])], cb);
          }
        }
      }
    }
    if (loaded) {
      st.edges += loaded;  // per-thread counters, summed at the end of the round
      st.bytes += 8ull * loaded;
    }
  }
  st.attempts += att;
  st.successes += suc;
  st.evals += att;
  // direct: a remote label read per attempt; both: read-modify-write per
  // atomic issued (proposal slabs read once, counted above)
  st.bytes += (proposals ? 0ull : 4ull * att) + 8ull * suc;
  st.mark(3);
  bool changed = false;
  for (std::uint32_t i = tid; i < npt; i += B) {
    const std::uint32_t v = l.own[i];
    if (v < l.orig[i]) {
      atomic_min_agent(column + i, v);
      changed = true;
    }
    if (frontier && v < l.work[i]) snapshot[i] = v;
  }
  const bool pushed_any = __syncthreads_or(changed);
  // A marked neighbour holds the smallest candidate pushed into it; with a
  // push window that candidate lowers the neighbour's priority.
  bool marked = false;
  for (std::uint32_t k = 1 + tid; k < KO; k += B) {
    const std::uint32_t low = l.marks[k];
    if (low == kInfBits) continue;
    marked = true;
    if (b.prio) {
      atomic_min_agent(&b.prio[l.slots[k]], low);
      queued_min = min(queued_min, low);
    }
    enqueue(b, l.slots[k], r + 1);
  }
  const bool queued_any = __syncthreads_or(marked);
  if (tid == 0 && (queued_any || pushed_any)) mark_changed(b, q, r, queued_any);
  st.mark(4);
}

// ---------------------------------------------------------------------------
// Round processing shared by the persistent and host-polled kernels.
// ---------------------------------------------------------------------------
// Round r's work list as wave 0 sees it: lane x holds the end of class x's
// entries in the round's flat order (class 0's entries first).  Wave 0 reads
// the 64 counts in one step; n is their total.
struct RoundQueue {
  std::uint32_t end;
  std::uint32_t n;
};
__device__ __forceinline__ RoundQueue load_round_queue(const DevBatch& b, std::uint32_t r) {
  const std::uint32_t lane = threadIdx.x & 63u;
  RoundQueue q;
  q.end = load_agent(list_count(b, r % 3, lane));
#pragma unroll
  for (std::uint32_t off = 1; off < 64; off <<= 1) {
    const std::uint32_t below = __shfl(q.end, static_cast<int>((lane - off) & 63u));
    if (lane >= off) q.end += below;
  }
  q.n = __shfl(q.end, 63);
  return q;
}
// Slot of flat position i < n (wave 0, i uniform).
__device__ __forceinline__ std::uint32_t queued_slot(const DevBatch& b, const RoundQueue& q,
                                                     std::uint32_t li, std::uint32_t i) {
  const std::uint32_t x = static_cast<std::uint32_t>(__popcll(__ballot(q.end <= i)));
  const std::uint32_t first = __shfl(q.end, static_cast<int>((x - 1u) & 63u));
  return b.lists[static_cast<std::size_t>(li) * b.slot_count + class_begin(b.slot_count, x) + i -
                 (x ? first : 0u)];
}

// Round r's share of one workgroup.  With a push window (b.prio set), a
// push slot whose priority is above `limit` is not visited: it keeps its
// priority and is queued again for round r + 1.  The smallest priority the
// workgroup leaves queued (deferred or pushed into) goes to the round's
// next_min counter of its XCD group.
template <int B, int EPT, bool I, int M>
__device__ __forceinline__ void process_round(const DevGraph& g, const DevBatch& b, std::uint32_t r,
                              const RoundQueue& queue, std::uint32_t limit, const Lds& l) {
  const std::uint32_t items = b.items_per_claim ? b.items_per_claim : 1u;
  VisitStats<I> st;
  std::uint32_t queued_min = kInfBits;
  if (threadIdx.x == 0) l.flags[4] = kInfBits;
  auto visit = [&](std::uint32_t s) {
    const SlotDesc d = load_slot_desc(g, b, s);
    bool run = true;
    // A variant without the slot's engine cannot visit it; seed_kernel flags
    // such a batch (the host picks the variant from the batch's
    // engines, so it does not happen).  Nothing is done here: any extra
    // global operation on this path costs the variant 18 VGPRs.
    if (d.engine == kJacobiPull) {
      if constexpr (holds_pull(M)) visit_pull<B, EPT, I>(g, b, d, r, l, st);
    } else if constexpr (holds_push(M)) {
      if (b.prio) {
        if (threadIdx.x == 0) {
          const std::uint32_t p = atomic_exch_agent(&b.prio[s], kInfBits);
          const bool defer = p != kInfBits && p > limit;
          if (defer) {
            atomic_min_agent(&b.prio[s], p);
            enqueue(b, s, r + 1);
            queued_min = min(queued_min, p);
          }
          l.flags[3] = defer ? 1u : 0u;
        }
        __syncthreads();
        run = l.flags[3] == 0u;
      }
      if (run)
        visit_push<B, EPT, I, M>(g, b, d, r, d.engine == kFrontierPush, l, st, queued_min);
    }
    if (run) ++st.items;
    __syncthreads();
  };
  if (b.ordered) {
    // Slot order: the round's list is cut into one segment per XCD group;
    // a workgroup claims from its own group's segment (blockIdx % 8: the
    // dispatcher places workgroups on the XCDs round-robin), then from the
    // others in turn.  Consecutive slots share a tile, so the slots of one
    // tile are visited by one XCD, close together in time, and a chunk of
    // them by one workgroup (the tile's records stay in that XCD's L2).
    // Thread 0 keeps the next claim in flight while a chunk is visited.
    DevControl* c = b.control;
    const std::uint32_t home = blockIdx.x % kBarrierGroups;
    std::uint32_t tried = 0;  // thread 0: segments exhausted so far
    std::uint32_t ahead = 0;  // thread 0: claim in flight on segment home + tried
    // Segment ends, read once into LDS (flags 8 .. 15): the claim counters
    // sit on lines of their own, which no plain load shares.
    std::uint32_t* seg_end = l.flags + 8;
    if (threadIdx.x == 0) {
      for (std::uint32_t x = 0; x < kBarrierGroups; ++x) seg_end[x] = c->seg_begin[x + 1];
      ahead = atomic_add_agent(&c->seg_claim[home * kBarrierStride], items);
    }
    for (;;) {
      if (threadIdx.x == 0) {
        std::uint32_t start = kNone, end = 0;
        while (tried < kBarrierGroups) {
          const std::uint32_t y = (home + tried) % kBarrierGroups;
          const std::uint32_t e = seg_end[y];
          if (ahead < e) {
            start = ahead;
            end = min(ahead + items, e);
            ahead = atomic_add_agent(&c->seg_claim[y * kBarrierStride], items);
            break;
          }
          if (++tried < kBarrierGroups)
            ahead = atomic_add_agent(&c->seg_claim[((home + tried) % kBarrierGroups) * kBarrierStride],
                                     items);
        }
        l.flags[0] = start;
        l.flags[2] = end;
      }
      __syncthreads();
      const std::uint32_t start = l.flags[0], end = l.flags[2];
      __syncthreads();
      if (start == kNone) break;
      for (std::uint32_t i = start; i < end; ++i) visit(b.lists[i]);
    }
  } else {
    // Chunks of the list are dealt to 64 groups of workgroups (blockIdx % 64)
    // in turn.  A workgroup's first chunk is its own index, with no claim;
    // chunks beyond the grid are claimed on the group's counter.  Wave 0
    // walks the list and hands each slot to the workgroup.  Measured with the
    // list classes (kQueueClasses) against one claim and one append counter,
    // relaxation per batch: 32 point-Jacobi lanes on 32x32x128 580 -> 270 us,
    // 64 queries on 64x64x256 block Jacobi 2298 -> 1722 us and frontier push
    // 1240 -> 946 us, 256 queries on 128x128x512 15.1 -> 13.8 ms.
    // A chunk is at most the list's share of a workgroup: with two items per
    // claim, a round of fewer items than twice the grid left workgroups idle
    // (64 queries on 64x64x256 935 -> 880 us, 256 on 128x128x512 13.61 ->
    // 13.46 ms).
    const std::uint32_t li = r % 3;
    const std::uint32_t chunk = max(1u, min(items, queue.n / gridDim.x));
    const std::uint32_t groups = min(gridDim.x, kQueueClasses);
    const std::uint32_t group = blockIdx.x % groups;
    const std::uint32_t dealt = group + groups * ((gridDim.x - group + groups - 1u) / groups);
    // Position of unit u's first item, kNone when it is past the list.
    auto begin = [&](unsigned long long u) {
      const unsigned long long at = u * chunk;
      return at < queue.n ? static_cast<std::uint32_t>(at) : kNone;
    };
    std::uint32_t i = begin(blockIdx.x);
    std::uint32_t left = chunk;
    for (;;) {
      if (threadIdx.x < 64) {
        if (left == 0) {
          i = begin(dealt);
          if (i != kNone) {
            std::uint32_t t = 0;
            if (threadIdx.x == 0) t = atomic_add_agent(list_claim(b, li, group), 1u);
            t = __builtin_amdgcn_readfirstlane(__shfl(t, 0));
            i = begin(dealt + static_cast<unsigned long long>(groups) * t);
          }
          left = chunk;
        }
        const std::uint32_t s = i < queue.n ? queued_slot(b, queue, li, i) : kNone;
        if (threadIdx.x == 0) l.flags[0] = s;
        i += i != kNone;
        --left;
      }
      __syncthreads();
      const std::uint32_t s = l.flags[0];
      if (s == kNone) break;
      visit(s);
    }
  }
  if (b.prio) {
    if (queued_min != kInfBits) atomicMin(&l.flags[4], queued_min);
    __syncthreads();
    if (threadIdx.x == 0 && l.flags[4] != kInfBits)
      atomic_min_agent(&b.control->next_min[(((r + 1) % 3) * kBarrierGroups + blockIdx.x % kBarrierGroups) *
                                            kBarrierStride],
                       l.flags[4]);
  }
  if constexpr (I) {
    // One add per thread keeps the counters off the hot path's critical lanes.
    DevControl* c = b.control;
    // Byte and record counts are per thread: tile-level terms are added by
    // thread 0 of the visit, per-record terms by the thread that did them.
    if (st.attempts) atomicAdd(&c->atomic_attempts, st.attempts);
    if (st.successes) atomicAdd(&c->atomic_successes, st.successes);
    if (st.bytes) atomicAdd(&c->algorithmic_bytes, st.bytes);
    if (st.edges) atomicAdd(&c->edges_relaxed, st.edges);
    if (st.evals) atomicAdd(&c->candidates, st.evals);
    if (threadIdx.x == 0) {
      if (st.items) atomicAdd(&c->items_processed, st.items);
      if (st.sweeps) atomicAdd(&c->closure_sweeps, st.sweeps);
      for (int p = 0; p < kPhaseCount; ++p)
        if (st.phase[p]) atomicAdd(&c->phase_cycles[p], st.phase[p]);
    }
  }
}

// One cooperative launch runs every round: process list r%3, grid barrier,
// repeat while the next list is non-empty and the round limit allows.
template <int B, int EPT, bool I, int MW, int M>
__global__ __launch_bounds__(B, MW) void relax_persistent_kernel(DevGraph g, DevBatch b,
                                                             std::uint32_t max_v,
                                                             std::uint32_t work_words) {
  extern __shared__ std::uint32_t lds_words[];
  const Lds l = carve(lds_words, max_v, work_words, g.max_neighbor_tiles);
  DevControl* c = b.control;
  if (b.probe) {  // co-residency probe: one short-bounded grid barrier
    grid_barrier_grouped(c, gridDim.x, kProbeSpinLimit);
    return;
  }
  std::uint32_t r = load_agent(&c->round);
  if (load_agent(&c->done)) return;
  std::uint32_t n = 0;
  std::uint32_t limit = b.prio ? load_agent(&c->window_limit) : 0u;
  for (;;) {
    RoundQueue queue{};
    if (threadIdx.x < 64) {
      queue = load_round_queue(b, r);
      if (threadIdx.x == 0) l.flags[5] = queue.n;
    }
    __syncthreads();
    n = l.flags[5];
    if (n == 0 || (b.maximum_rounds && r >= b.maximum_rounds)) break;
    if (blockIdx.x == 0 && threadIdx.x < kQueueClasses) {
      store_agent(list_count(b, (r + 2) % 3, threadIdx.x), 0u);
      store_agent(list_claim(b, (r + 2) % 3, threadIdx.x), 0u);
      if (threadIdx.x == 0) {
        // read after the barrier of round r - 2, written in round r + 1
        if (b.prio) reset_next_min(c, (r + 2) % 3);
        if (b.instrumentation) atomicMax(&c->max_list, static_cast<unsigned long long>(n));
      }
    }
    process_round<B, EPT, I, M>(g, b, r, queue, limit, l);
    if (!grid_barrier_grouped(c, gridDim.x)) return;  // error bits set; the host reports a device failure
    if (b.prio) limit = next_window_limit(c, b, r, limit);
    ++r;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    c->round = r;
    c->rounds_executed = r;
    c->done = 1;
    c->stop_reason = n == 0 ? kStopConverged : kStopMaximumRounds;
  }
}

// After round r, by one wave (lane x looks after class x of the lists):
// count the round, reset the list that the next round fills, stop on an
// empty list or the round limit.
__device__ __forceinline__ void advance_round(const DevBatch& b, std::uint32_t r) {
  static_assert(kQueueClasses == 64, "one lane per class");
  DevControl* c = b.control;
  const std::uint32_t lane = threadIdx.x & 63u;
  const bool any = __ballot(load_agent(list_count(b, (r + 1) % 3, lane)) != 0) != 0;
  if (b.instrumentation) {
    std::uint32_t n = load_agent(list_count(b, r % 3, lane));
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off);
    if (lane == 0 && n > c->max_list) c->max_list = n;
  }
  store_agent(list_count(b, (r + 2) % 3, lane), 0u);
  store_agent(list_claim(b, (r + 2) % 3, lane), 0u);
  if (lane != 0) return;
  if (b.prio) {
    c->window_limit = next_window_limit(c, b, r, c->window_limit);
    reset_next_min(c, (r + 2) % 3);
  }
  c->round = r + 1;
  c->rounds_executed = r + 1;
  if (!any) {
    c->done = 1;
    c->stop_reason = kStopConverged;
  } else if (b.maximum_rounds && r + 1 >= b.maximum_rounds) {
    c->done = 1;
    c->stop_reason = kStopMaximumRounds;
  }
}

// Host-polled control: one round per launch (ordinary grid); the workgroup
// that finishes last advances the round (jacobi_pull.hpp:153-220 shape).  A
// kernel of its own between the rounds cost 4.7 us and a launch gap per
// round.  Workgroups arrive on group counters first, as at the persistent
// grid's barrier: all on one counter would queue 11.4 ns each.
template <int B, int EPT, bool I, int MW, int M>
__global__ __launch_bounds__(B, MW) void relax_round_kernel(DevGraph g, DevBatch b,
                                                        std::uint32_t max_v,
                                                        std::uint32_t work_words) {
  extern __shared__ std::uint32_t lds_words[];
  const Lds l = carve(lds_words, max_v, work_words, g.max_neighbor_tiles);
  DevControl* c = b.control;
  if (load_agent(&c->done)) return;
  const std::uint32_t r = load_agent(&c->round);
  RoundQueue queue{};
  if (!b.ordered && threadIdx.x < 64) queue = load_round_queue(b, r);
  const std::uint32_t limit = b.prio ? load_agent(&c->window_limit) : 0u;
  process_round<B, EPT, I, M>(g, b, r, queue, limit, l);
  if (b.ordered) return;
  __builtin_amdgcn_s_waitcnt(0);  // every wave's atomics of the round are performed
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const bool last = threadIdx.x == 0 && arrive_last(c, gridDim.x);
  if (__ballot(last)) advance_round(b, r);
}

// ---------------------------------------------------------------------------
// Launch wrappers (host side).
// ---------------------------------------------------------------------------
template <int B, int EPT, bool I, int MW, int M>
hipError_t launch_relax(bool persistent, bool cooperative, std::uint32_t grid,
                        std::size_t lds_bytes, std::uint32_t max_v, std::uint32_t work_words,
                        const DevGraph& g, const DevBatch& b, hipStream_t stream) {
  if (persistent) {
    void* args[] = {const_cast<DevGraph*>(&g), const_cast<DevBatch*>(&b), &max_v, &work_words};
    const void* kernel = reinterpret_cast<const void*>(&relax_persistent_kernel<B, EPT, I, MW, M>);
    if (cooperative)
      return hipLaunchCooperativeKernel(kernel, dim3(grid), dim3(B), args,
                                        static_cast<unsigned>(lds_bytes), stream);
    return hipLaunchKernel(kernel, dim3(grid), dim3(B), args, lds_bytes, stream);
  }
  hipLaunchKernelGGL((relax_round_kernel<B, EPT, I, MW, M>), dim3(grid), dim3(B), lds_bytes, stream,
                     g, b, max_v, work_words);
  return hipGetLastError();
}

template <int B, int EPT, bool I, int MW, int M>
hipError_t occupancy_relax(bool persistent, std::size_t lds_bytes, int* blocks_per_cu) {
  const void* kernel =
      persistent ? reinterpret_cast<const void*>(&relax_persistent_kernel<B, EPT, I, MW, M>)
                 : reinterpret_cast<const void*>(&relax_round_kernel<B, EPT, I, MW, M>);
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, kernel, B, lds_bytes);
}

// Instantiated kernel variants.  Block sizes come with the registers per
// thread that hold a tile's internal records through its closure (B * EPT =
// 2048: 512-vertex tiles with four internal out-edges per vertex fit).
// The 256- and 512-thread blocks also come bounded to at least 6, 7 or 8 waves
// per SIMD (fewer registers per lane, more visits in flight); instrumented
// runs use the unbounded variant.
template <int B, int EPT, typename F>
hipError_t with_waves(bool instrumented, std::uint32_t min_waves, F& f) {
  if (instrumented) return f.template operator()<B, EPT, true, 1>();
  if constexpr (B == 256 || B == 512) {
    if (min_waves >= 8) return f.template operator()<B, EPT, false, 8>();
    if (min_waves >= 7) return f.template operator()<B, EPT, false, 7>();
    if (min_waves >= 6) return f.template operator()<B, EPT, false, 6>();
  }
  return f.template operator()<B, EPT, false, 1>();
}

template <typename F>
hipError_t with_shape(std::uint32_t block, bool instrumented, std::uint32_t min_waves, F&& f) {
  switch (block) {
    case 64: return with_waves<64, 32>(instrumented, min_waves, f);
    case 128: return with_waves<128, 16>(instrumented, min_waves, f);
    case 256: return with_waves<256, 8>(instrumented, min_waves, f);
    case 512: return with_waves<512, 4>(instrumented, min_waves, f);
    case 1024: return with_waves<1024, 2>(instrumented, min_waves, f);
    default: return hipErrorInvalidValue;
  }
}

// The variants of one engine set, for every block size and wave bound.
template <int M>
hipError_t relax_launch_engines(std::uint32_t block, bool persistent, bool cooperative,
                                std::uint32_t grid, std::size_t lds_bytes, std::uint32_t max_v,
                                std::uint32_t work_words, const DevGraph& g, const DevBatch& b,
                                hipStream_t stream) {
  return with_shape(block, b.instrumentation != 0, b.min_waves,
                    [&]<int B, int EPT, bool I, int MW>() {
                      return launch_relax<B, EPT, I, MW, M>(persistent, cooperative, grid, lds_bytes,
                                                            max_v, work_words, g, b, stream);
                    });
}

template <int M>
hipError_t relax_occupancy_engines(std::uint32_t block, bool persistent, bool instrumented,
                                   std::uint32_t min_waves, std::size_t lds_bytes,
                                   int* blocks_per_cu) {
  return with_shape(block, instrumented, min_waves, [&]<int B, int EPT, bool I, int MW>() {
    return occupancy_relax<B, EPT, I, MW, M>(persistent, lds_bytes, blocks_per_cu);
  });
}

}  // namespace bfn
