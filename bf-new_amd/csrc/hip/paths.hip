// paths.hip -- result extraction: compact paths, predecessors, distances,
// per-query finalisation, occupancy and negotiated-cost weight updates.
//
// Compact paths follow compact_paths.cpp:117-206 (and the device version
// compact_path_results.hip.cpp:169-249): from each target, walk tight
// admitted incoming edges (d[u] + w == d[v], u selected and finite) in
// stable-EdgeId order, skipping vertices already on the path, backtracking
// when a vertex has no untried candidate, until a source is reached.  A
// workgroup owns a query and a wave one target: its 64 lanes scan a vertex's
// incoming edges together and a wave min-reduction picks the smallest
// EdgeId, so a step costs one pass over the in-edges instead of a sort.
//
// Where every tight edge lowers the label (no zero-weight plateau), the walk
// never meets its own path and never runs dry, so it is a chain of smallest
// EdgeIds: walk_descending.  It is bound by the latency of a step's dependent
// reads, so the winning lane hands over all that the next step needs (slot,
// label, column bounds) and a step is four dependent reads; looking the
// vertex up in its query's tiles three times per step made it about thirty.
// The first pass keeps each path in the frame scratch, so the second only
// copies it out.  A whole routing pass, before and after: one net on 64x64x256
// tiles 491 -> 384 us, 41 queries with 123 targets on 45x37x301 1168 -> 905
// us, 256 queries on 128x128x512 14.35 -> 13.97 ms.  A target whose walk meets a plateau, a dead end or the end
// of its frame space is walked again by walk_backtracking, the general rule:
// a frame stores its vertex and the last EdgeId tried from it; resuming a
// frame asks for the smallest candidate above that EdgeId, which visits
// candidates in exactly the reference's cursor order.
#include "bfn_internal.hpp"

#include <algorithm>

namespace bfn {


__device__ __forceinline__ std::uint32_t column_of(const DevBatch& b, std::uint32_t q,
                                                   std::uint32_t jacobi_copy) {
  return b.engine[q] == kJacobiPull ? jacobi_copy : 0u;
}

// Label of global vertex v for query q (+inf when its tile is not selected).
__device__ std::uint32_t label_of(const DevGraph& g, const DevBatch& b, std::uint32_t q,
                                  std::uint32_t v, std::uint32_t jacobi_copy,
                                  unsigned long long* pool_index) {
  const std::uint32_t T = g.owner_tiles[v];
  const std::uint32_t s = find_slot(b, q, T);
  if (s == kNone) {
    if (pool_index) *pool_index = ~0ull;
    return kInfBits;
  }
  const std::uint32_t v0 = g.tile_vertex_offsets[T];
  const std::uint32_t npt = g.tile_vertex_offsets[T + 1] - v0;
  const unsigned long long base = b.slot_dist[s] + (v - v0);
  if (pool_index) *pool_index = base;
  return b.dist[base + static_cast<unsigned long long>(column_of(b, q, jacobi_copy)) * npt];
}

__device__ __forceinline__ bool is_source(const DevBatch& b, std::uint32_t q, std::uint32_t v) {
  return find_sorted(b.sources, b.source_offsets[q], b.source_offsets[q + 1], v) != kNone;
}

// The lanes of this wave meet, and their global stores are visible to its own
// later loads (in uniform control flow).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_s_waitcnt(0);
  __threadfence_block();
  (void)__ballot(1);
}

__device__ __forceinline__ unsigned long long wave_min_u64(unsigned long long x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const std::uint32_t lo = __shfl_xor(static_cast<std::uint32_t>(x), off, 64);
    const std::uint32_t hi = __shfl_xor(static_cast<std::uint32_t>(x >> 32), off, 64);
    const unsigned long long y = (static_cast<unsigned long long>(hi) << 32) | lo;
    x = y < x ? y : x;
  }
  return x;
}

// Pool offset of slot s's final labels.
__device__ __forceinline__ unsigned long long labels_of_slot(const DevGraph& g, const DevBatch& b,
                                                             std::uint32_t s, std::uint32_t col) {
  if (b.slot_desc) {
    const unsigned long long at = (static_cast<unsigned long long>(b.slot_desc[s].dist_hi) << 32) |
                                  b.slot_desc[s].dist_lo;
    return at + static_cast<unsigned long long>(col) * b.slot_desc[s].npt;
  }
  unsigned long long at = b.slot_dist[s];
  if (col) {
    const std::uint32_t T = b.tiles[s];
    at += g.tile_vertex_offsets[T + 1] - g.tile_vertex_offsets[T];
  }
  return at;
}

// Frames [fb, fb + room) hold the walk: vertex, the edge it was reached by,
// and its label.  Returns the number of edges, or -1 when the target needs
// walk_backtracking.  Wave-uniform arguments and result.
__device__ std::int32_t walk_descending(const PathArgs& a, std::uint32_t q, std::uint32_t target,
                                        std::uint32_t col, unsigned long long fb,
                                        unsigned long long room) {
  const DevGraph& g = a.g;
  const DevBatch& b = a.b;
  const std::uint32_t lane = threadIdx.x & 63u;
  const std::uint32_t T = g.owner_tiles[target];
  const std::uint32_t s = find_slot(b, q, T);
  std::uint32_t v = target;
  std::uint32_t dv = b.dist[labels_of_slot(g, b, s, col) + (target - g.tile_vertex_offsets[T])];
  std::uint32_t c0 = g.column_offsets[v], c1 = g.column_offsets[v + 1], in_base = b.slot_in_base[s];
  if (lane == 0) {
    a.frame_vertex[fb] = v;
    a.frame_via[fb] = kNone;
    a.frame_last[fb] = dv;
  }
  for (std::int32_t top = 0;; ++top) {
    if (dv == 0u && is_source(b, q, v)) return top;
    if (static_cast<unsigned long long>(top) + 1 >= room) return -1;
    std::uint32_t eid = kNone, u = 0, du = 0, u0 = 0, u1 = 0, u_base = 0;
    bool plateau = false;
    for (std::uint32_t e = c0 + lane; e < c1; e += 64) {
      const std::uint32_t id = g.in_edge_ids[e];
      const std::uint32_t p = g.csc_pack[e];
      const std::uint32_t from = g.sources[e];
      const float w = g.in_weights[e];
      const std::uint32_t ns = b.slot_in[in_base + (p >> 24)];
      if (ns == kNone) continue;
      // what the next step needs of this candidate travels with its label
      const std::uint32_t n0 = g.column_offsets[from], n1 = g.column_offsets[from + 1];
      const std::uint32_t n_base = b.slot_in_base[ns];
      const std::uint32_t d = b.dist[labels_of_slot(g, b, ns, col) + ((p >> 12) & kPackLocalMask)];
      if (d == kInfBits || as_bits(as_float(d) + w) != dv) continue;
      plateau |= d == dv;
      if (id < eid) {
        eid = id;
        u = from;
        du = d;
        u0 = n0;
        u1 = n1;
        u_base = n_base;
      }
    }
    std::uint32_t best = eid;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) best = min(best, __shfl_xor(best, off));
    if (best == kNone || __ballot(plateau)) return -1;
    const unsigned long long m = __ballot(eid == best);
    const int winner = __popcll((m - 1ull) & ~m);  // an edge has one id: one lane holds it
    v = __shfl(u, winner);
    dv = __shfl(du, winner);
    c0 = __shfl(u0, winner);
    c1 = __shfl(u1, winner);
    in_base = __shfl(u_base, winner);
    if (lane == 0) {
      a.frame_vertex[fb + top + 1] = v;
      a.frame_via[fb + top + 1] = best;
      a.frame_last[fb + top + 1] = dv;
    }
  }
}

// The general walk of one target by one wave, in the query's whole frame
// space and with its own stamp on the vertices of its path.  Returns the
// number of edges, or -1 when no tight path reaches a source.
__device__ std::int32_t walk_backtracking(const PathArgs& a, std::uint32_t q, std::uint32_t target,
                                          std::uint32_t stamp, std::uint32_t copy,
                                          unsigned long long fb) {
  const DevGraph& g = a.g;
  const DevBatch& b = a.b;
  const std::uint32_t lane = threadIdx.x & 63u;
  unsigned long long target_pool;
  label_of(g, b, q, target, copy, &target_pool);
  std::int32_t top = 0;
  std::uint32_t v = target;
  std::uint32_t last = kNone;  // EdgeId last tried from the top frame
  if (lane == 0) {
    a.frame_vertex[fb] = target;
    a.frame_via[fb] = kNone;
    a.onpath[target_pool] = stamp;
  }
  for (;;) {
    if (is_source(b, q, v)) return top;
    const std::uint32_t T = g.owner_tiles[v];
    const std::uint32_t s = find_slot(b, q, T);
    const std::uint32_t dv = label_of(g, b, q, v, copy, nullptr);
    const std::uint32_t in0 = g.in_nbr_offsets[T];
    unsigned long long best = ~0ull;
    for (std::uint32_t e = g.column_offsets[v] + lane; e < g.column_offsets[v + 1]; e += 64) {
      const std::uint32_t eid = g.in_edge_ids[e];
      if (last != kNone && eid <= last) continue;
      const std::uint32_t p = g.csc_pack[e];
      const std::uint32_t k = p >> 24;
      const std::uint32_t ns = b.slot_in[b.slot_in_base[s] + k];
      if (ns == kNone) continue;
      const std::uint32_t nt = g.in_nbr_tiles[in0 + k];
      const std::uint32_t nn = g.tile_vertex_offsets[nt + 1] - g.tile_vertex_offsets[nt];
      const unsigned long long pool = b.slot_dist[ns] + ((p >> 12) & kPackLocalMask);
      const std::uint32_t du =
          b.dist[pool + static_cast<unsigned long long>(column_of(b, q, copy)) * nn];
      if (du == kInfBits) continue;
      if (as_bits(as_float(du) + g.in_weights[e]) != dv) continue;
      if (a.onpath[pool] == stamp) continue;
      const unsigned long long key =
          (static_cast<unsigned long long>(eid) << 32) | g.sources[e];
      best = key < best ? key : best;
    }
    best = wave_min_u64(best);
    if (best != ~0ull) {
      const std::uint32_t eid = static_cast<std::uint32_t>(best >> 32);
      const std::uint32_t u = static_cast<std::uint32_t>(best);
      unsigned long long upool;
      label_of(g, b, q, u, copy, &upool);
      if (lane == 0) {
        a.frame_last[fb + top] = eid;
        a.frame_vertex[fb + top + 1] = u;
        a.frame_via[fb + top + 1] = eid;
        a.onpath[upool] = stamp;
      }
      ++top;
      v = u;
      last = kNone;
    } else {
      unsigned long long vpool;
      label_of(g, b, q, v, copy, &vpool);
      if (lane == 0) a.onpath[vpool] = 0;
      --top;
      if (top < 0) return -1;
      wave_fence();
      v = a.frame_vertex[fb + top];
      last = a.frame_last[fb + top];
    }
    wave_fence();
  }
}

// One workgroup per query, wave w walks (pass 1) or copies out (pass 2) its
// targets w, w + waves, ...; wave 0 then takes those that need backtracking.
__global__ __launch_bounds__(512) void compact_paths_kernel(PathArgs a) {
  const std::uint32_t q = a.query_list ? a.query_list[blockIdx.x] : blockIdx.x;
  const DevGraph& g = a.g;
  const DevBatch& b = a.b;
  const std::uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const std::uint32_t copy =
      a.jacobi_copy_from_control ? (b.control->round & 1u) : a.jacobi_copy;
  const std::uint32_t col = column_of(b, q, copy);
  const std::uint32_t t0 = b.target_offsets[q], t1 = b.target_offsets[q + 1];
  const unsigned long long fb = a.frame_base[q];
  const unsigned long long space =
      a.frame_slab ? static_cast<unsigned long long>(b.tile_end[q] - b.tile_begin[q]) * a.frame_slab
                   : (q + 1 < b.query_count ? a.frame_base[q + 1] : a.frame_words) - fb;
  const unsigned long long room = space / (t1 - t0);  // frames of one target's descending walk
  const std::uint32_t state = a.query_clean[q];
  auto summarise = [&](std::uint32_t t, std::uint32_t target, std::uint32_t dt, std::int32_t top,
                       unsigned long long frames) {
    if (lane != 0) return;
    std::uint32_t* sum = a.summaries + static_cast<std::size_t>(t) * 7;
    const bool reached = dt != kInfBits && (state & kPathClean);
    const bool found = reached && top >= 0;
    sum[0] = target;
    sum[1] = found ? a.frame_vertex[frames + top] : 0u;
    sum[2] = reached ? dt : kInfBits;
    sum[3] = found ? static_cast<std::uint32_t>(top) : 0u;
    sum[4] = reached;
    // complete, query terminal failure, unreachable, no tight path
    sum[5] = found ? 0u : !(state & kPathClean) ? 2u : dt == kInfBits ? 1u : 3u;
    sum[6] = found;
    a.lengths[t] = found ? static_cast<unsigned long long>(top) + 1 : 0ull;
  };
  // Edges share the vertex offsets; a path of L edges leaves slot L unused.
  auto copy_out = [&](std::uint32_t t, std::int32_t top, unsigned long long frames, bool labels) {
    const unsigned long long out = a.offsets[t];
    for (std::int32_t i = static_cast<std::int32_t>(lane); i <= top; i += 64) {
      const unsigned long long from = frames + static_cast<std::uint32_t>(top - i);
      const std::uint32_t vert = a.frame_vertex[from];
      const std::uint32_t label = labels ? a.frame_last[from] : label_of(g, b, q, vert, copy, nullptr);
      const std::uint32_t edge = i < top ? a.frame_via[from] : kNone;
      a.arena_vertices[out + i] = vert;
      a.arena_labels[out + i] = label;
      a.arena_edges[out + i] = edge;
      if (a.host_vertices) {
        a.host_vertices[out + i] = vert;
        a.host_labels[out + i] = label;
        a.host_edges[out + i] = edge;
      }
    }
  };
  const bool emit = a.pass == 2;
  if (emit && a.arena_capacity != ~0ull && a.offsets[a.target_total] > a.arena_capacity)
    return;  // the host retries with room for them
  if (emit && a.host_left && (state & kPathGeneral)) {
    if (threadIdx.x == 0) *a.host_left = 1u;
    return;
  }
  __shared__ std::uint32_t general;  // targets for walk_backtracking
  if (threadIdx.x == 0) general = 0;
  __syncthreads();
  if (!emit || !(state & kPathGeneral)) {
    for (std::uint32_t t = t0 + wave; t < t1; t += waves) {
      const std::uint32_t target = b.targets[t];
      const unsigned long long frames = fb + room * (t - t0);
      if (emit) {
        const std::int32_t n = static_cast<std::int32_t>(a.lengths[t]);
        if (n) copy_out(t, n - 1, frames, !(state & kPathKept));
        continue;
      }
      const std::uint32_t dt = label_of(g, b, q, target, copy, nullptr);
      std::int32_t top = -1;
      if (dt != kInfBits && (state & kPathClean)) {
        top = room ? walk_descending(a, q, target, col, frames, room) : -1;
        if (top < 0) {
          if (lane == 0) {
            atomicAdd(&general, 1u);
            a.lengths[t] = ~0ull;
          }
          continue;
        }
      }
      wave_fence();
      summarise(t, target, dt, top, frames);
    }
    wave_fence();
    __syncthreads();
    if (emit) return;
    const std::uint32_t again = general == 0 ? 0u : t1 - t0 == 1 ? kPathKept : kPathGeneral;
    const std::uint32_t marked = (state & kPathClean) | again;
    if (threadIdx.x == 0 && marked != state) a.query_clean[q] = marked;
    if (general == 0) return;
  }
  if (wave != 0) return;
  for (std::uint32_t t = t0; t < t1; ++t) {
    const std::uint32_t target = b.targets[t];
    if (a.lengths[t] != (emit ? a.lengths[t] : ~0ull) || a.lengths[t] == 0) continue;
    const std::int32_t top = walk_backtracking(a, q, target, a.stamp_base + t + 1, copy, fb);
    wave_fence();
    if (emit) {
      if (top >= 0) copy_out(t, top, fb, false);
    } else {
      summarise(t, target, label_of(g, b, q, target, copy, nullptr), top, fb);
    }
    wave_fence();
  }
}

// Where the image of a query's region holds its position i, tile T: at
// offsets[i], or, where the tiles are one run (no offsets), as far from the
// first tile as in the graph.
__device__ __forceinline__ unsigned long long region_at(const DevGraph& g, const DevBatch& b, std::uint32_t q,
                                                        const unsigned long long* offsets, std::uint32_t i,
                                                        std::uint32_t T) {
  if (offsets) return offsets[i];
  return g.tile_vertex_offsets[T] - g.tile_vertex_offsets[b.tiles[slot_at(b, b.tile_begin[q])]];
}

// Smallest-EdgeId tight admitted predecessor of each vertex of query q, tile
// by tile in the order of its sorted selected tiles.
__global__ void predecessors_kernel(DevGraph g, DevBatch b, std::uint32_t q,
                                    std::uint32_t jacobi_copy, const unsigned long long* offsets,
                                    std::uint32_t* out) {
  const std::uint32_t pos = b.tile_begin[q] + blockIdx.x;
  if (pos >= b.tile_end[q]) return;
  const std::uint32_t s = slot_at(b, pos);
  const std::uint32_t T = b.tiles[s];
  const std::uint32_t v0 = g.tile_vertex_offsets[T];
  const std::uint32_t npt = g.tile_vertex_offsets[T + 1] - v0;
  const unsigned long long at = region_at(g, b, q, offsets, blockIdx.x, T);
  const std::uint32_t in0 = g.in_nbr_offsets[T];
  const std::uint32_t col = column_of(b, q, jacobi_copy);
  for (std::uint32_t i = threadIdx.x; i < npt; i += blockDim.x) {
    const std::uint32_t v = v0 + i;
    std::uint32_t best_eid = kNone, best_u = kNone;
    const std::uint32_t dv = b.dist[b.slot_dist[s] + static_cast<unsigned long long>(col) * npt + i];
    if (dv != kInfBits && !is_source(b, q, v)) {
      for (std::uint32_t e = g.column_offsets[v]; e < g.column_offsets[v + 1]; ++e) {
        const std::uint32_t p = g.csc_pack[e];
        const std::uint32_t k = p >> 24;
        const std::uint32_t ns = b.slot_in[b.slot_in_base[s] + k];
        if (ns == kNone) continue;
        const std::uint32_t nt = g.in_nbr_tiles[in0 + k];
        const std::uint32_t nn = g.tile_vertex_offsets[nt + 1] - g.tile_vertex_offsets[nt];
        const std::uint32_t du = b.dist[b.slot_dist[ns] + static_cast<unsigned long long>(col) * nn +
                                        ((p >> 12) & kPackLocalMask)];
        if (du == kInfBits || as_bits(as_float(du) + g.in_weights[e]) != dv) continue;
        const std::uint32_t eid = g.in_edge_ids[e];
        if (eid < best_eid) {
          best_eid = eid;
          best_u = g.sources[e];
        }
      }
    }
    out[at + i] = best_u;
  }
}

__global__ void finalize_kernel(DevGraph g, DevBatch b, const unsigned long long* relaxations,
                                QueryStatusDev* out, std::uint32_t* path_state) {
  const std::uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= b.query_count) return;
  const DevControl* c = b.control;
  // Round r writes Jacobi column (r+1)&1; unvisited tiles hold equal columns.
  const std::uint32_t jacobi_copy = c->rounds_executed & 1u;
  const std::uint32_t executed = c->rounds_executed;
  const std::uint32_t lc = b.last_change[q];
  const bool clean = c->error_bits == 0;
  // A query converged once a round after its last decrease found no change.
  const bool converged = clean && (lc < executed || c->stop_reason == kStopConverged);
  bool reached = true;
  for (std::uint32_t i = b.target_offsets[q]; i < b.target_offsets[q + 1]; ++i)
    reached &= label_of(g, b, q, b.targets[i], jacobi_copy, nullptr) != kInfBits;
  QueryStatusDev st;
  st.rounds = converged ? static_cast<unsigned long long>(lc) + 1 : executed;
  st.relaxations = relaxations ? relaxations[q] : 0;
  st.converged = converged;
  st.reached = converged && reached;
  st.miss = converged && !reached;
  st.stop_reason = !clean ? kStopDeviceFailure : (converged ? kStopConverged : c->stop_reason);
  st.error_bits = c->error_bits;
  st.engine = b.engine[q];
  out[q] = st;
  if (path_state) path_state[q] = converged ? kPathClean : 0u;  // what the path passes start from
}

// Work-normalised relaxation count: admitted out-edges of reached vertices.
__global__ void relaxation_count_kernel(DevGraph g, DevBatch b, unsigned long long* out) {
  const std::uint32_t jacobi_copy = b.control->rounds_executed & 1u;
  const std::uint32_t s = blockIdx.x;
  if (s >= b.slot_count) return;
  const std::uint32_t q = b.slot_query[s];
  const std::uint32_t T = b.tiles[s];
  const std::uint32_t v0 = g.tile_vertex_offsets[T];
  const std::uint32_t npt = g.tile_vertex_offsets[T + 1] - v0;
  const std::uint32_t col = column_of(b, q, jacobi_copy);
  unsigned long long count = 0;
  for (std::uint32_t i = threadIdx.x; i < npt; i += blockDim.x) {
    if (b.dist[b.slot_dist[s] + static_cast<unsigned long long>(col) * npt + i] == kInfBits) continue;
    const std::uint32_t v = v0 + i;
    for (std::uint32_t e = g.row_offsets[v]; e < g.row_offsets[v + 1]; ++e)
      count += b.slot_out[b.slot_out_base[s] + (g.csr_pack[e] >> 24)] != kNone;
  }
  if (count) atomicAdd(&out[q], count);
}

__global__ void occupancy_kernel(const std::uint32_t* arena_vertices, unsigned long long n,
                                 int* occupancy) {
  const unsigned long long stride = static_cast<unsigned long long>(gridDim.x) * blockDim.x;
  for (unsigned long long i = static_cast<unsigned long long>(blockIdx.x) * blockDim.x +
                              threadIdx.x;
       i < n; i += stride)
    atomicAdd(&occupancy[arena_vertices[i]], 1);
}

// w(u -> v) = base[v] * (1 + 0.5 * occ[v]) in this fp32 order.
__device__ __forceinline__ float node_cost(const float* base, const int* occupancy, std::uint32_t v) {
  const float occ = occupancy ? static_cast<float>(occupancy[v]) : 0.0f;
  const float scale = 1.0f + 0.5f * occ;
  return base[v] * scale;
}

__global__ void node_cost_kernel(const float* base, const int* occupancy, std::uint32_t n, float* cost) {
  const std::uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < n) cost[v] = node_cost(base, occupancy, v);
}

// The weights of both orientations, one thread per edge so that the arrays
// are written in whole lines: the first `csr_blocks` workgroups take the CSR
// edges (their destination's cost), the others 256 columns of the CSC each
// (found by a search of their offsets in LDS).  (One thread per node wrote
// ten edges apart from its neighbours' and read two arrays per edge: 1137 us
// for 84M edges.)
__global__ __launch_bounds__(256) void edge_cost_kernel(DevGraph g, const float* base, const int* occupancy,
                                                        std::uint32_t csr_blocks, float* csr_weights,
                                                        float* csc_weights) {
  const std::uint32_t tid = threadIdx.x;
  if (blockIdx.x < csr_blocks) {
    for (unsigned long long e = blockIdx.x * 256ull + tid; e < g.edge_count; e += csr_blocks * 256ull)
      csr_weights[e] = node_cost(base, occupancy, g.destinations[e]);
    return;
  }
  __shared__ std::uint32_t ends[256];
  __shared__ float costs[256];
  const std::uint32_t v0 = (blockIdx.x - csr_blocks) * 256u;
  const std::uint32_t count = min(256u, g.vertex_count - v0);
  const std::uint32_t begin = g.column_offsets[v0], end = g.column_offsets[v0 + count];
  ends[tid] = tid < count ? g.column_offsets[v0 + tid + 1] : end;
  costs[tid] = tid < count ? node_cost(base, occupancy, v0 + tid) : 0.0f;
  __syncthreads();
  for (unsigned long long e = static_cast<unsigned long long>(begin) + tid; e < end; e += 256) {
    std::uint32_t c = 0;  // columns that end at or before e
#pragma unroll
    for (std::uint32_t step = 128; step > 0; step >>= 1)
      if (ends[c + step - 1] <= e) c += step;
    csc_weights[e] = costs[c];
  }
}

// Whether every cost is finite and nonnegative; bad[0] is raised otherwise.
__global__ void check_costs_kernel(const float* base, std::uint32_t n, std::uint32_t* bad) {
  const std::uint32_t stride = gridDim.x * blockDim.x;
  bool fine = true;
  for (unsigned long long v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride)
    fine &= base[v] >= 0.0f && base[v] <= 3.4e38f;
  if (!fine) atomicOr(bad, 1u);
}

__global__ void scan_u64_kernel(const unsigned long long* in, unsigned long long* out,
                                std::uint32_t n) {
  __shared__ unsigned long long buf[1024];
  __shared__ unsigned long long carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (std::uint32_t base = 0; base < n; base += 1024) {
    const std::uint32_t i = base + threadIdx.x;
    const unsigned long long x = i < n ? in[i] : 0;
    buf[threadIdx.x] = x;
    __syncthreads();
    for (std::uint32_t off = 1; off < 1024; off <<= 1) {
      const unsigned long long y = threadIdx.x >= off ? buf[threadIdx.x - off] : 0;
      __syncthreads();
      buf[threadIdx.x] += y;
      __syncthreads();
    }
    if (i < n) out[i] = carry + buf[threadIdx.x] - x;
    __syncthreads();
    if (threadIdx.x == 1023) carry += buf[1023];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[n] = carry;
}

// ---- launch wrappers ------------------------------------------------------
// A wave per target up to eight (the walks of a query's targets are chains of
// their own; more waves per workgroup than targets would only exit).
hipError_t paths_launch(const PathArgs& a, std::uint32_t query_count, hipStream_t stream) {
  const std::uint32_t waves = a.most_targets < 1 ? 1u : a.most_targets > 8 ? 8u : a.most_targets;
  hipLaunchKernelGGL(compact_paths_kernel, dim3(query_count), dim3(64 * waves), 0, stream, a);
  return hipGetLastError();
}

hipError_t scan_u64_launch(const unsigned long long* in, unsigned long long* out, std::uint32_t n,
                           hipStream_t stream) {
  hipLaunchKernelGGL(scan_u64_kernel, dim3(1), dim3(1024), 0, stream, in, out, n);
  return hipGetLastError();
}

hipError_t predecessors_launch(const DevGraph& g, const DevBatch& b, std::uint32_t q,
                               std::uint32_t slots, std::uint32_t copy,
                               const unsigned long long* offsets, std::uint32_t* out,
                               hipStream_t stream) {
  if (slots)
    hipLaunchKernelGGL(predecessors_kernel, dim3(slots), dim3(256), 0, stream, g, b, q, copy, offsets, out);
  return hipGetLastError();
}

// Copies query q's final labels tile by tile, in the order of its sorted
// selected tiles, tile by tile.
__global__ void gather_region_kernel(DevGraph g, DevBatch b, std::uint32_t q,
                                     std::uint32_t jacobi_copy, const unsigned long long* offsets,
                                     std::uint32_t* out) {
  const std::uint32_t i = blockIdx.x;
  const std::uint32_t pos = b.tile_begin[q] + i;
  if (pos >= b.tile_end[q]) return;
  const std::uint32_t s = slot_at(b, pos);
  const std::uint32_t T = b.tiles[s];
  const std::uint32_t npt = g.tile_vertex_offsets[T + 1] - g.tile_vertex_offsets[T];
  const std::uint32_t* src =
      b.dist + b.slot_dist[s] + static_cast<unsigned long long>(column_of(b, q, jacobi_copy)) * npt;
  std::uint32_t* dst = out + region_at(g, b, q, offsets, i, T);
  for (std::uint32_t k = threadIdx.x; k < npt; k += blockDim.x) dst[k] = src[k];
}

hipError_t gather_region_launch(const DevGraph& g, const DevBatch& b, std::uint32_t q,
                                std::uint32_t slots, std::uint32_t copy,
                                const unsigned long long* offsets, std::uint32_t* out,
                                hipStream_t stream) {
  if (slots)
    hipLaunchKernelGGL(gather_region_kernel, dim3(slots), dim3(256), 0, stream, g, b, q, copy,
                       offsets, out);
  return hipGetLastError();
}

hipError_t finalize_launch(const DevGraph& g, const DevBatch& b,
                           const unsigned long long* relaxations, void* out,
                           std::uint32_t* path_state, hipStream_t stream) {
  hipLaunchKernelGGL(finalize_kernel, dim3((b.query_count + 127) / 128), dim3(128), 0, stream, g,
                     b, relaxations, static_cast<QueryStatusDev*>(out), path_state);
  return hipGetLastError();
}

hipError_t relaxation_count_launch(const DevGraph& g, const DevBatch& b,
                                   unsigned long long* out, hipStream_t stream) {
  if (b.slot_count)
    hipLaunchKernelGGL(relaxation_count_kernel, dim3(b.slot_count), dim3(256), 0, stream, g, b,
                       out);
  return hipGetLastError();
}

hipError_t occupancy_launch(const std::uint32_t* arena, unsigned long long n, int* occ,
                            hipStream_t stream) {
  if (n) hipLaunchKernelGGL(occupancy_kernel, dim3(1024), dim3(256), 0, stream, arena, n, occ);
  return hipGetLastError();
}

hipError_t node_cost_launch(const DevGraph& g, const float* base, const int* occ, float* cost,
                            float* csr_w, float* csc_w, hipStream_t stream) {
  const std::uint32_t V = g.vertex_count, columns = (V + 255u) / 256u;
  if (V == 0) return hipSuccess;
  if (cost) hipLaunchKernelGGL(node_cost_kernel, dim3(columns), dim3(256), 0, stream, base, occ, V, cost);
  const std::uint32_t csr_blocks = std::min(8192u, (g.edge_count + 255u) / 256u);
  hipLaunchKernelGGL(edge_cost_kernel, dim3(csr_blocks + columns), dim3(256), 0, stream, g, cost ? cost : base,
                     cost ? nullptr : occ, csr_blocks, csr_w, csc_w);
  return hipGetLastError();
}

hipError_t check_costs_launch(const float* base, std::uint32_t n, std::uint32_t* bad, hipStream_t stream) {
  hipLaunchKernelGGL(check_costs_kernel, dim3(std::min(1024u, (n + 255u) / 256u)), dim3(256), 0, stream, base,
                     n, bad);
  return hipGetLastError();
}

}  // namespace bfn
