// relax.hip -- control of the relaxation engines: the compaction between
// slot-order rounds, batch preparation (control reset, label fill,
// slot tables, seeds) and the launch dispatch to the kernel variant of a
// batch's engine set (relax_kernels.hpp, instantiated by relax_mixed.hip,
// relax_push.hip, relax_push_lds.hip and relax_pull.hip).
#include "bfn_launch.hpp"

#include <algorithm>
#include <mutex>

namespace bfn {

// Between rounds in slot order (one workgroup): count the round as
// advance_round does, then compact the queued bits into lists[0, n)
// and clear them.  Slots are taken in groups of 64 (two bit words); group k
// belongs to segment k % 8, and the list holds segment 0's groups in order,
// then segment 1's, ..., so each segment is in slot order.  first = 1 (after
// seeding) compacts only.
constexpr std::uint32_t kCompactGroupsPerThread = 8;

__global__ __launch_bounds__(1024) void ordered_advance_kernel(DevBatch b, std::uint32_t first) {
  __shared__ std::uint32_t scan[1024];
  __shared__ std::uint32_t seg_start[kBarrierGroups];
  DevControl* c = b.control;
  if (c->done) return;
  const std::uint32_t tid = threadIdx.x;
  const std::uint32_t W = (b.slot_count + 31u) / 32u;
  const std::uint32_t NG = (W + 1u) / 2u;
  // Groups of segment x: x, x + 8, ...; its first position in the virtual
  // order (segment 0's groups first) is vstart[x].
  std::uint32_t vstart[kBarrierGroups + 1];
  vstart[0] = 0;
#pragma unroll
  for (std::uint32_t x = 0; x < kBarrierGroups; ++x)
    vstart[x + 1] = vstart[x] + (NG > x ? (NG - 1u - x) / kBarrierGroups + 1u : 0u);
  if (tid < kBarrierGroups) seg_start[tid] = kNone;
  std::uint32_t carry = 0;
  for (std::uint32_t base = 0; base < NG; base += 1024u * kCompactGroupsPerThread) {
    const std::uint32_t v0 = base + tid * kCompactGroupsPerThread;
    std::uint32_t w0[kCompactGroupsPerThread], w1[kCompactGroupsPerThread],
        grp[kCompactGroupsPerThread], seg[kCompactGroupsPerThread];
    std::uint32_t total = 0;
#pragma unroll
    for (std::uint32_t j = 0; j < kCompactGroupsPerThread; ++j) {
      const std::uint32_t v = v0 + j;
      w0[j] = w1[j] = 0;
      grp[j] = kNone;
      seg[j] = 0;
      if (v < NG) {
        std::uint32_t x = 0;
        while (v >= vstart[x + 1]) ++x;
        seg[j] = x;
        grp[j] = x + kBarrierGroups * (v - vstart[x]);
        w0[j] = b.active[2 * grp[j]];
        if (2 * grp[j] + 1 < W) w1[j] = b.active[2 * grp[j] + 1];
      }
    }
#pragma unroll
    for (std::uint32_t j = 0; j < kCompactGroupsPerThread; ++j) total += __popc(w0[j]) + __popc(w1[j]);
    scan[tid] = total;
    __syncthreads();
    for (std::uint32_t off = 1; off < 1024; off <<= 1) {
      const std::uint32_t add = tid >= off ? scan[tid - off] : 0u;
      __syncthreads();
      scan[tid] += add;
      __syncthreads();
    }
    std::uint32_t pos = carry + scan[tid] - total;
    const std::uint32_t chunk_total = scan[1023];
#pragma unroll
    for (std::uint32_t j = 0; j < kCompactGroupsPerThread; ++j) {
      if (grp[j] == kNone) continue;
      if (v0 + j == vstart[seg[j]]) seg_start[seg[j]] = pos;
      const std::uint32_t s0 = 64u * grp[j];
      for (std::uint32_t m = w0[j]; m; m &= m - 1u) b.lists[pos++] = s0 + __ffs(m) - 1u;
      for (std::uint32_t m = w1[j]; m; m &= m - 1u) b.lists[pos++] = s0 + 32u + __ffs(m) - 1u;
      if (w0[j]) b.active[2 * grp[j]] = 0;
      if (w1[j]) b.active[2 * grp[j] + 1] = 0;
    }
    carry += chunk_total;
    __syncthreads();
  }
  __syncthreads();
  if (tid == 0) {
    const std::uint32_t n = carry;
    // Segments without groups (NG < 8) are empty and sit at the end.
    for (std::uint32_t x = 0; x < kBarrierGroups; ++x) {
      const std::uint32_t at = seg_start[x] == kNone ? n : seg_start[x];
      c->seg_begin[x] = at;
      c->seg_claim[x * kBarrierStride] = at;
    }
    c->seg_begin[kBarrierGroups] = n;
    if (b.instrumentation && n > c->max_list) c->max_list = n;
    if (!first) {
      const std::uint32_t r = c->round;
      if (b.prio) {
        c->window_limit = next_window_limit(c, b, r, c->window_limit);
        reset_next_min(c, (r + 2) % 3);
      }
      c->round = r + 1;
      c->rounds_executed = r + 1;
      if (n == 0) {
        c->done = 1;
        c->stop_reason = kStopConverged;
      } else if (b.maximum_rounds && r + 1 >= b.maximum_rounds) {
        c->done = 1;
        c->stop_reason = kStopMaximumRounds;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Batch preparation.
// ---------------------------------------------------------------------------
// Control block and list counters of a run, by one workgroup.
__device__ __forceinline__ void reset_control(DevControl* c, std::uint32_t* queue, std::uint32_t window) {
  std::uint32_t* words = reinterpret_cast<std::uint32_t*>(c);
  for (std::uint32_t i = threadIdx.x; i < sizeof(DevControl) / 4; i += blockDim.x) words[i] = 0;
  if (queue)
    for (std::uint32_t i = threadIdx.x; i < kQueueWords / kBarrierStride; i += blockDim.x)
      queue[i * kBarrierStride] = 0;
  __syncthreads();
  for (std::uint32_t i = threadIdx.x; i < 3 * kBarrierGroups * kBarrierStride; i += blockDim.x)
    c->next_min[i] = kInfBits;
  if (threadIdx.x == 0) c->window_limit = window;  // round 0 visits the sources' slots (priority 0)
}

__global__ __launch_bounds__(1024) void reset_control_kernel(DevControl* c, std::uint32_t* queue,
                                                             std::uint32_t window) {
  reset_control(c, queue, window);
}

__global__ void fill_u32_kernel(std::uint32_t* p, unsigned long long n, std::uint32_t v) {
  const unsigned long long stride = static_cast<unsigned long long>(gridDim.x) * blockDim.x;
  for (unsigned long long i = static_cast<unsigned long long>(blockIdx.x) * blockDim.x +
                              threadIdx.x;
       i < n; i += stride)
    p[i] = v;
}

// Preparation of a run, one launch: the first `fill_blocks` workgroups set
// every label to +inf, the next `slot_blocks` the slots' queue stamps and
// window priorities, the last one the control block and each query's last
// change.  With `structure` (the first run of a batch) the slot workgroups
// also resolve each slot's in- and out-neighbour tiles to the query's slots
// and write its descriptor: they depend only on the batch and the graph's
// tile directory, so the reruns of a batch keep them.  A neighbour is a
// binary search of dependent reads, so kSlotLanes lanes share a slot's
// lists; one thread per slot took 27 us for 36 slots and 181 us for 213k.
constexpr std::uint32_t kSlotLanes = 16;

__global__ __launch_bounds__(256) void prepare_kernel(DevGraph g, DevBatch b, unsigned long long pool_words,
                                                      std::uint32_t fill_blocks, std::uint32_t slot_blocks,
                                                      std::uint32_t structure) {
  const std::uint32_t tid = threadIdx.x;
  if (blockIdx.x < fill_blocks) {
    const uint4 inf = make_uint4(kInfBits, kInfBits, kInfBits, kInfBits);
    const unsigned long long quads = pool_words / 4;
    const unsigned long long stride = static_cast<unsigned long long>(fill_blocks) * 256;
    for (unsigned long long i = static_cast<unsigned long long>(blockIdx.x) * 256 + tid; i < quads; i += stride)
      reinterpret_cast<uint4*>(b.dist)[i] = inf;
    if (blockIdx.x == 0 && tid < pool_words % 4) b.dist[4 * quads + tid] = kInfBits;
    return;
  }
  if (blockIdx.x >= fill_blocks + slot_blocks) {
    reset_control(b.control, b.queue, b.window);
    for (std::uint32_t q = tid; q < b.query_count; q += 256) b.last_change[q] = 0;
    return;
  }
  const std::uint32_t lanes = structure ? kSlotLanes : 1u;
  const std::uint32_t s = (blockIdx.x - fill_blocks) * (256u / lanes) + tid / lanes;
  const std::uint32_t lane = tid % lanes;
  if (s >= b.slot_count) return;
  if (lane == 0) {
    b.stamp[s] = 0;  // also every queue-bit word of slot-order claims (ceil(S/32) <= S)
    if (b.prio) b.prio[s] = kInfBits;
  }
  if (!structure) return;
  const std::uint32_t q = b.slot_query[s], T = b.tiles[s];
  const std::uint32_t in0 = g.in_nbr_offsets[T], in1 = g.in_nbr_offsets[T + 1];
  const std::uint32_t o0 = g.out_nbr_offsets[T], o1 = g.out_nbr_offsets[T + 1];
  const std::uint32_t in_base = b.slot_in_base[s], out_base = b.slot_out_base[s];
  for (std::uint32_t k = lane; k < max(in1 - in0, o1 - o0); k += kSlotLanes) {
    if (k < in1 - in0) b.slot_in[in_base + k] = find_slot(b, q, g.in_nbr_tiles[in0 + k]);
    if (k < o1 - o0) {
      const std::uint32_t ns = find_slot(b, q, g.out_nbr_tiles[o0 + k]);
      b.slot_out[out_base + k] = ns;
      if (b.slot_out_off) b.slot_out_off[out_base + k] = ns == kNone ? ~0ull : b.slot_dist[ns];
    }
  }
  if (lane == kSlotLanes - 1 && b.slot_desc) const_cast<SlotDesc*>(b.slot_desc)[s] = make_slot_desc(g, b, s);
}

// Zero the sources and queue round 0: Jacobi queues the source tiles and
// every tile they feed; push engines queue the source tiles.  One wave per
// query; its lanes share the fed tiles of a source (Jacobi) or the sources
// (push: 20000 sources one after the other took 40 ms, 1 ms by lanes).
__global__ __launch_bounds__(64) void seed_kernel(DevGraph g, DevBatch b) {
  const std::uint32_t q = blockIdx.x, lane = threadIdx.x;
  const bool jacobi = b.engine[q] == kJacobiPull;
  // the relaxation kernel variant must hold the engine of every query
  if (lane == 0 && (jacobi ? !holds_pull(b.engines) : !holds_push(b.engines)))
    atomicOr(&b.control->error_bits, 4u);
  const std::uint32_t first = jacobi ? 0u : lane, step = jacobi ? 1u : 64u;
  const bool mine = !jacobi || lane == 0;
  for (std::uint32_t i = b.source_offsets[q] + first; i < b.source_offsets[q + 1]; i += step) {
    const std::uint32_t u = b.sources[i];
    const std::uint32_t T = g.owner_tiles[u];
    const std::uint32_t s = find_slot(b, q, T);
    if (s == kNone) {
      if (mine) atomicOr(&b.control->error_bits, 4u);  // device_failure: host validated this
      continue;
    }
    if (mine) {
      const std::uint32_t v0 = g.tile_vertex_offsets[T];
      const std::uint32_t npt = g.tile_vertex_offsets[T + 1] - v0;
      std::uint32_t* column = b.dist + b.slot_dist[s];
      column[u - v0] = 0u;
      if (jacobi) column[npt + (u - v0)] = 0u;
      if (b.prio && !jacobi) atomic_min_agent(&b.prio[s], 0u);
      enqueue(b, s, 0);
    }
    if (jacobi) {
      const std::uint32_t ob = b.slot_out_base[s];
      const std::uint32_t KO = g.out_nbr_offsets[T + 1] - g.out_nbr_offsets[T];
      for (std::uint32_t k = lane; k < KO; k += 64) {
        const std::uint32_t ns = b.slot_out[ob + k];
        if (ns != kNone) enqueue(b, ns, 0);
      }
    }
  }
}

// Relaxation launch: the kernel variant of the batch's engine set, and for
// slot-order claims the compaction between rounds.
hipError_t relax_launch(std::uint32_t block, bool persistent, bool cooperative,
                        std::uint32_t grid, std::size_t lds_bytes, std::uint32_t max_v,
                        std::uint32_t work_words, const DevGraph& g, const DevBatch& b,
                        hipStream_t stream) {
  hipError_t e;
  switch (b.engines) {
    case kEnginesPush:
      e = relax_launch_push(block, persistent, cooperative, grid, lds_bytes, max_v, work_words, g, b, stream);
      break;
    case kEnginesPushLds:
      e = relax_launch_push_lds(block, persistent, cooperative, grid, lds_bytes, max_v, work_words, g, b, stream);
      break;
    case kEnginesPull:
      e = relax_launch_pull(block, persistent, cooperative, grid, lds_bytes, max_v, work_words, g, b, stream);
      break;
    default:
      e = relax_launch_mixed(block, persistent, cooperative, grid, lds_bytes, max_v, work_words, g, b, stream);
  }
  if (e != hipSuccess || persistent) return e;
  if (b.ordered) hipLaunchKernelGGL(ordered_advance_kernel, dim3(1), dim3(1024), 0, stream, b, 0u);
  return hipGetLastError();
}

hipError_t relax_occupancy(std::uint32_t engines, std::uint32_t block, bool persistent,
                           bool instrumented, std::uint32_t min_waves, std::size_t lds_bytes,
                           int* blocks_per_cu) {
  switch (engines) {
    case kEnginesPush:
      return relax_occupancy_push(block, persistent, instrumented, min_waves, lds_bytes, blocks_per_cu);
    case kEnginesPushLds:
      return relax_occupancy_push_lds(block, persistent, instrumented, min_waves, lds_bytes, blocks_per_cu);
    case kEnginesPull:
      return relax_occupancy_pull(block, persistent, instrumented, min_waves, lds_bytes, blocks_per_cu);
    default:
      return relax_occupancy_mixed(block, persistent, instrumented, min_waves, lds_bytes, blocks_per_cu);
  }
}

// Workgroups per CU of a persistent grid that the device places at once.
// The grid's workgroups wait for each other at every grid barrier, so all of
// them must be resident together; the occupancy query has promised more than
// the device places (on MI355X: 7 per CU for the 256-thread Jacobi-only
// kernel, whose grid then never passed its first barrier).  So the count is
// checked by a probe launch of the same kernel variant with the same LDS:
// every workgroup passes one grid barrier with a short bounded wait and
// exits; a timeout lowers the count by one.  Results are kept per device,
// variant and LDS size in a fixed table (no allocation).
namespace {
struct ProbeResult {
  int device;
  std::uint32_t engines, block, min_waves, instrumented;
  std::size_t lds_bytes;
  int promised, placed;
};
constexpr int kProbeTable = 64;
ProbeResult g_probe[kProbeTable];
int g_probe_count = 0;
std::mutex g_probe_mutex;
}  // namespace

hipError_t coresident_per_cu(int device, int promised, std::uint32_t cus, std::size_t lds_bytes,
                             std::uint32_t max_v, std::uint32_t work_words, const DevGraph& g,
                             const DevBatch& b, hipStream_t stream, std::uint32_t block,
                             int* placed) {
  std::lock_guard<std::mutex> lock(g_probe_mutex);
  for (int i = 0; i < g_probe_count; ++i) {
    const ProbeResult& p = g_probe[i];
    if (p.device == device && p.engines == b.engines && p.block == block &&
        p.min_waves == b.min_waves && p.instrumented == (b.instrumentation != 0) &&
        p.lds_bytes == lds_bytes && p.promised == promised) {
      *placed = p.placed;
      return hipSuccess;
    }
  }
  DevBatch probe{};
  probe.engines = b.engines;
  probe.min_waves = b.min_waves;
  probe.instrumentation = b.instrumentation;
  probe.control = b.control;
  probe.probe = 1;
  int per_cu = promised;
  for (; per_cu >= 1; --per_cu) {
    hipLaunchKernelGGL(reset_control_kernel, dim3(1), dim3(1024), 0, stream, b.control, nullptr, 0u);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
      e = relax_launch(block, true, true, static_cast<std::uint32_t>(per_cu) * cus, lds_bytes, max_v,
                       work_words, g, probe, stream);
    std::uint32_t bits = 0;
    if (e == hipSuccess)
      e = hipMemcpyAsync(&bits, &b.control->error_bits, sizeof bits, hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return e;
    if ((bits & kErrorBarrierTimeout) == 0) break;
  }
  if (g_probe_count < kProbeTable)
    g_probe[g_probe_count++] = ProbeResult{device, b.engines, block, b.min_waves,
                                           b.instrumentation != 0u, lds_bytes, promised, per_cu};
  *placed = per_cu;
  return hipSuccess;
}

hipError_t prep_launch(const DevGraph& g, const DevBatch& b, std::uint64_t pool_words,
                       hipStream_t stream, bool structure) {
  const std::uint32_t fill_blocks =
      static_cast<std::uint32_t>(std::min<std::uint64_t>(4096, (pool_words + 4095) / 4096));
  const std::uint32_t per_block = 256u / (structure ? kSlotLanes : 1u);
  const std::uint32_t slot_blocks = (b.slot_count + per_block - 1) / per_block;
  hipLaunchKernelGGL(prepare_kernel, dim3(fill_blocks + slot_blocks + 1), dim3(256), 0, stream, g, b,
                     static_cast<unsigned long long>(pool_words), fill_blocks, slot_blocks,
                     structure ? 1u : 0u);
  if (b.query_count) hipLaunchKernelGGL(seed_kernel, dim3(b.query_count), dim3(64), 0, stream, g, b);
  if (b.ordered) hipLaunchKernelGGL(ordered_advance_kernel, dim3(1), dim3(1024), 0, stream, b, 1u);
  return hipGetLastError();
}

}  // namespace bfn

namespace bfn {
hipError_t fill_launch(std::uint32_t* p, unsigned long long n, std::uint32_t value,
                       hipStream_t stream) {
  if (n) hipLaunchKernelGGL(fill_u32_kernel, dim3(2048), dim3(256), 0, stream, p, n, value);
  return hipGetLastError();
}
}  // namespace bfn
