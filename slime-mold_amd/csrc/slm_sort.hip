// slm_sort.hip - periodic spatial re-sort of the agents (no counterpart in the
// reference, whose agents keep their creation order, src/main.rs:263-282).
//
// Agents are bucketed by the Morton (Z-order) code of the 2^k x 2^k cell bin
// they stand in, then scattered bin by bin into the other agent buffer, so a
// wave's lanes sense and deposit in nearby cells and share L2 lines.  Each
// instance of a pool owns a contiguous range of bins, so agents stay inside
// their instance's slot range.  The slot -> original index table id[] moves
// with them.  The order inside a bin comes from atomics and is not fixed,
// which is harmless: an agent's update depends only on its own state, its
// original index and the step-start trail, and the deposit marks commute, so
// any permutation gives the same result.
#include <type_traits>

#include "slm_internal.h"

namespace slm {
namespace {

constexpr int kScanBlock = 256;
constexpr int kScanPerThread = 4;
constexpr uint32_t kScanTile = kScanBlock * kScanPerThread;  // entries per scan block

__device__ inline uint32_t spread_bits(uint32_t v) {  // 16 bits -> even positions
  v &= 0xffffu;
  v = (v | (v << 8)) & 0x00ff00ffu;
  v = (v | (v << 4)) & 0x0f0f0f0fu;
  v = (v | (v << 2)) & 0x33333333u;
  v = (v | (v << 1)) & 0x55555555u;
  return v;
}

// float -> u32 of a value that may lie below 0 or beyond 2^32 (clamped).
__device__ inline uint32_t clamp_u32(float v) {
  v = __builtin_fmaxf(v, 0.0f);
  v = __builtin_fminf(v, 4294967040.0f);
  return static_cast<uint32_t>(v);
}

// The re-sort key of an agent at (x, y) with heading th: the Morton code of
// its 2^cell_log2 bin - with SLM_SORT_AT_SENSOR the bin holding the point its
// centre sensor reads, (x, y) + sensor_dist * (cos th, sin th) - followed by
// k = sort_key & SLM_SORT_HEADING_MASK bits of heading class.  The point only
// has to be near the true one, so it comes from the hardware sin/cos
// (v_sin/v_cos_f32, argument in revolutions).  The count and scatter kernels
// evaluate this function on the same loaded values, so they agree on every
// key.
__device__ inline uint32_t key_of(float x, float y, float th, const Instance& in,
                                  const DevParams& p, uint32_t cell_log2, uint32_t sort_key) {
  const uint32_t hl = sort_key & SLM_SORT_HEADING_MASK;
  const float rev = th * 0.159154943f;
  if (sort_key & SLM_SORT_AT_SENSOR) {
    x = __builtin_fmaf(p.sensor_dist, __builtin_amdgcn_cosf(rev), x);
    y = __builtin_fmaf(p.sensor_dist, __builtin_amdgcn_sinf(rev), y);
  }
  uint32_t bx = clamp_u32(x) >> cell_log2;  // x in [0, width] without the sensor offset
  uint32_t by = clamp_u32(y) >> cell_log2;
  bx = bx < in.nbx ? bx : in.nbx - 1u;
  by = by < in.nby ? by : in.nby - 1u;
  const uint32_t m = spread_bits(bx) | (spread_bits(by) << 1);
  const uint32_t h = clamp_u32(rev * static_cast<float>(1u << hl)) & ((1u << hl) - 1u);
  return in.bin_off + ((m << hl) | h);
}

__global__ void zero_u32_kernel(uint32_t* p, uint32_t n) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// A workgroup of the count and scatter kernels takes kSortPer x 256 consecutive
// slots, each thread kSortPer of them (slots q*256 + threadIdx.x of the range).
// Agents re-sorted earlier arrive grouped by bin, so these usually stand in a few
// neighbouring bins, which the workgroup counts in LDS: one global atomic per
// distinct bin of the workgroup.  (Dense instances put ~10^4 agents in one bin; a
// global atomic per wave and bin serialised ~10^2 times more.)  A bin's entry there
// is its key mod kLocalBins: the Morton codes of any 32 x 32 bins differ in their low
// 10 bits, also where the region straddles an edge of a large aligned square and
// its codes lie far apart (a table by distance from the lowest code refuses those,
// a quarter of the workgroups or more).  Where two bins meet in an entry one of them
// has it, and the other's agents take atomics on the global counters (all agents of
// such a workgroup did: where one instance's last agents wrap to its first bins, beside
// the next one's, 350 instances of 40 x 300 with 2.1 * 10^6 agents counted in 25 us).
constexpr uint32_t kLocalBins = 1024;  // LDS for 5 workgroups a CU (2048: 4, up to 7% slower)
constexpr int kSortPer = 4;
constexpr uint32_t kSortSlots = kSortPer * kAgentBlock;

// The tables of a re-sort kernel's launch.
struct SortArgs {
  const Instance* insts;
  const DevParams* params;
  const uint32_t* block_inst;  // per kAgentBlock slots
  uint32_t ninst, total, cell_log2, sort_key;
  int xcd_remap;
};

// XCD-contiguous workgroups: neighbouring slots, their bins' counters and their
// output ranges stay with one XCD's L2 (the re-sort of the 256-instance mix
// measured 10% faster).
__device__ inline uint32_t sort_base(const SortArgs& g) {
  return (g.xcd_remap ? xcd_logical_block(blockIdx.x, gridDim.x) : blockIdx.x) * kSortSlots;
}

// Slot q of this thread, and whether there is one (a 64-bit test: near the 2^32 - 256
// agent limit the last workgroup's slots wrap).
__device__ inline bool sort_slot(const SortArgs& g, uint32_t base, int q, uint32_t& j) {
  j = base + q * kAgentBlock + threadIdx.x;
  return uint64_t(base) + q * kAgentBlock + threadIdx.x < g.total;
}

// The keys of the workgroup's agents, whether their bin has its entry, with the bin's
// agents here in `s_cnt` and its key in `s_tag`, and then their ranks among them.
struct Keys {
  uint32_t k[kSortPer], r[kSortPer];
  bool act[kSortPer], own[kSortPer];
  __device__ uint32_t entry(int q) const { return k[q] & (kLocalBins - 1u); }
};
__device__ inline Keys block_keys(const SortArgs& g, uint32_t base, const float (&x)[kSortPer],
                                  const float (&y)[kSortPer], const float (&th)[kSortPer],
                                  uint32_t* s_cnt, uint32_t* s_tag) {
  for (uint32_t i = threadIdx.x; i < kLocalBins; i += kAgentBlock) s_cnt[i] = 0u;
  Keys t;
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    uint32_t j;
    t.act[q] = sort_slot(g, base, q, j);
    t.own[q] = false;
    t.k[q] = t.r[q] = 0;
  }
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    if (uint64_t(base) + q * kAgentBlock >= g.total) break;  // uniform; no block_inst entry
    const uint32_t first = base + q * kAgentBlock;
    const uint32_t last = min(first + kAgentBlock, g.total) - 1u;
    const uint32_t j = first + threadIdx.x;
    for (uint32_t ii = g.block_inst[first / kAgentBlock];; ii++) {  // block-uniform walk
      const Instance in = g.insts[ii];
      const uint32_t end = in.agent_off + in.agent_count;
      if (t.act[q] && j >= in.agent_off && j < end)
        t.k[q] = key_of(x[q], y[q], th[q], in, g.params[ii], g.cell_log2, g.sort_key);
      if (last < end || ii + 1u >= g.ninst) break;
    }
  }
#pragma unroll
  for (int q = 0; q < kSortPer; q++)
    if (t.act[q]) s_tag[t.entry(q)] = t.k[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kSortPer; q++)
    if (t.act[q] && s_tag[t.entry(q)] == t.k[q]) {
      t.own[q] = true;
      t.r[q] = atomicAdd(&s_cnt[t.entry(q)], 1u);
    }
  __syncthreads();
  return t;
}

// s_tag[entry] = add(bin, its agents) for each bin that has its entry: entry by entry, so
// that neighbouring bins' counters are reached by neighbouring lanes, and all in flight
// before one is used.  (One lane per bin wherever its first agent stood: count and
// scatter of 2^24 agents on 4096^2 230 us instead of 209, on 256^2 with 8 * 10^6
// agents 129 instead of 112.)
template <class Add>
__device__ inline void each_bin(const uint32_t* s_cnt, uint32_t* s_tag, Add&& add) {
  constexpr uint32_t kPer = kLocalBins / kAgentBlock;
  uint32_t n[kPer], old[kPer];
#pragma unroll
  for (uint32_t i = 0; i < kPer; i++) {
    const uint32_t e = i * kAgentBlock + threadIdx.x;
    n[i] = s_cnt[e];
    old[i] = n[i] ? add(s_tag[e], n[i]) : 0u;
  }
#pragma unroll
  for (uint32_t i = 0; i < kPer; i++)
    if (n[i]) s_tag[i * kAgentBlock + threadIdx.x] = old[i];
}

// The agents without an entry: old = add(bin, n) by one lane for n lanes of a wave in
// the bin, then use(q, old, rank among them) by each.  The first few distinct bins of a wave are
// taken together (agents that crowd a few distant bins), the others lane by lane
// (agents in any order, as before the first re-sort, share almost none).
constexpr int kWaveBins = 4;
template <class Add, class Use>
__device__ inline void each_wave_bin(const Keys& t, Add&& add, Use&& use) {
  const int lane = static_cast<int>(threadIdx.x & 63u);
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    bool todo = t.act[q] && !t.own[q];
    for (int n = 0; n < kWaveBins; n++) {
      const uint64_t pending = __ballot(todo);
      if (!pending) break;
      const int leader = __builtin_ctzll(pending);
      const bool mine = todo && t.k[q] == static_cast<uint32_t>(__shfl(t.k[q], leader));
      const uint64_t same = __ballot(mine);
      uint32_t old = 0;
      if (lane == leader) old = add(t.k[q], static_cast<uint32_t>(__popcll(same)));
      old = __shfl(old, leader);
      if (mine) use(q, old, static_cast<uint32_t>(__popcll(same & ((uint64_t(1) << lane) - 1u))));
      todo = todo && !mine;
    }
    if (todo) use(q, add(t.k[q], 1u), 0u);
  }
}

// count[bin] += the bin's agents; kRank: rank[slot] = the agent's rank in its bin.  All
// of a thread's agents are loaded before any is used: with one agent per thread the
// chain of load, barrier and atomic per block set the kernel's time, not the bandwidth.
template <bool kRank>
__global__ __launch_bounds__(kAgentBlock) void count_kernel(SortArgs g, AgentSoA a, int pos64,
                                                            uint32_t* count, uint32_t* rank) {
  __shared__ uint32_t s_cnt[kLocalBins], s_tag[kLocalBins];
  const uint32_t base = sort_base(g);
  float px[kSortPer], py[kSortPer], pth[kSortPer];
  // the heading only enters refined keys: the plain key loads positions only
  const bool heading = g.sort_key != 0u;
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    uint32_t j;
    px[q] = py[q] = pth[q] = 0.0f;
    if (sort_slot(g, base, q, j)) {
      px[q] = pos64 ? static_cast<float>(a.x64[j]) : a.x[j];
      py[q] = pos64 ? static_cast<float>(a.y64[j]) : a.y[j];
      if (heading) pth[q] = a.th[j];
    }
  }
  const Keys t = block_keys(g, base, px, py, pth, s_cnt, s_tag);
  auto add = [&](uint32_t k, uint32_t n) { return atomicAdd(count + k, n); };
  each_bin(s_cnt, s_tag, add);
  each_wave_bin(t, add, [&](int q, uint32_t first, uint32_t r) {
    if constexpr (kRank) rank[base + q * kAgentBlock + threadIdx.x] = first + r;
  });
  if constexpr (kRank) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kSortPer; q++)
      if (t.own[q]) rank[base + q * kAgentBlock + threadIdx.x] = s_tag[t.entry(q)] + t.r[q];
  }
}

// Exclusive scan of one tile of `in` into `out` (in place allowed); writes
// the tile total to sums[tile].
__global__ __launch_bounds__(kScanBlock) void scan_tile_kernel(const uint32_t* in, uint32_t n,
                                                               uint32_t* out, uint32_t* sums) {
  __shared__ uint32_t sh[kScanBlock];
  uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanPerThread;
  uint32_t v[kScanPerThread];
  uint32_t local = 0;
#pragma unroll
  for (int k = 0; k < kScanPerThread; k++) {
    v[k] = base + k < n ? in[base + k] : 0u;
    local += v[k];
  }
  sh[threadIdx.x] = local;
  __syncthreads();
  for (int off = 1; off < kScanBlock; off <<= 1) {  // inclusive Hillis-Steele
    uint32_t t = threadIdx.x >= static_cast<unsigned>(off) ? sh[threadIdx.x - off] : 0u;
    __syncthreads();
    sh[threadIdx.x] += t;
    __syncthreads();
  }
  uint32_t run = sh[threadIdx.x] - local;
#pragma unroll
  for (int k = 0; k < kScanPerThread; k++) {
    if (base + k < n) out[base + k] = run;
    run += v[k];
  }
  if (threadIdx.x == kScanBlock - 1) sums[blockIdx.x] = sh[threadIdx.x];
}

// out[i] += prefix[tile of i] (the exclusively scanned tile totals).
__global__ __launch_bounds__(kScanBlock) void scan_add_kernel(uint32_t* out, uint32_t n,
                                                              const uint32_t* prefix) {
  uint32_t add = prefix[blockIdx.x];
  uint32_t base = blockIdx.x * kScanTile;
  for (uint32_t k = threadIdx.x; k < kScanTile; k += kScanBlock)
    if (base + k < n) out[base + k] += add;
}

// Moves each agent into its bin's range of slots, [offset[bin], offset[bin] +
// count[bin]), from the end of the range down: count[bin] is the part of it that is
// still free.  Bins are recomputed from the positions, by the count kernel's
// arithmetic.
//
// The vector L1 takes a divergent store one lane a cycle, so writing each agent
// where it goes costs 64 accesses per array and wave (count and scatter of 2^24
// agents, f32: 111 + 214 us).  The workgroup orders its agents by bin in LDS
// instead (each bin's agents are reserved one run of slots) and writes the runs:
// 50 + 151 us; 8192^2 bf16 with f64 positions and 2^26 agents 398 + 831 -> 282 + 701;
// 64 instances of 256^2 to 2048^2 with 5 * 10^7 agents 480 + 692 -> 134 + 449.
// Bound by the LDS passes and the reservation's round trip.
template <bool P64>
__global__ __launch_bounds__(kAgentBlock) void scatter_kernel(SortArgs g, AgentSoA src,
                                                              AgentSoA dst, uint32_t* count,
                                                              const uint32_t* offset) {

  __shared__ uint32_t s_cnt[kLocalBins];   // agents per bin, then the bin's first position
  __shared__ uint32_t s_base[kLocalBins];  // the bin's first slot
  // s_dst: the waves' sums, then each position's slot
  __shared__ uint32_t s_dst[kSortSlots], s_th[kSortSlots], s_v[kSortSlots], s_id[kSortSlots];
  using pos = std::conditional_t<P64, double, float>;
  __shared__ pos s_x[kSortSlots], s_y[kSortSlots];
  const pos *sx, *sy;
  pos *dx, *dy;
  if constexpr (P64) {
    sx = src.x64, sy = src.y64, dx = dst.x64, dy = dst.y64;
  } else {
    sx = src.x, sy = src.y, dx = dst.x, dy = dst.y;
  }
  const uint32_t base = sort_base(g);
  pos x[kSortPer], y[kSortPer];
  float fx[kSortPer], fy[kSortPer], th[kSortPer], v[kSortPer];
  uint32_t id[kSortPer];
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    uint32_t j;
    x[q] = y[q] = 0;
    th[q] = v[q] = 0.0f;
    id[q] = 0;
    if (sort_slot(g, base, q, j)) {
      x[q] = sx[j];
      y[q] = sy[j];
      th[q] = src.th[j];
      v[q] = src.v[j];
      id[q] = src.id[j];
    }
    fx[q] = static_cast<float>(x[q]);
    fy[q] = static_cast<float>(y[q]);
  }
  const Keys t = block_keys(g, base, fx, fy, th, s_cnt, s_base);
  // the first of n slots for agents of bin k
  auto reserve = [&](uint32_t k, uint32_t n) { return offset[k] + atomicSub(count + k, n) - n; };
  each_bin(s_cnt, s_base, reserve);
  each_wave_bin(t, reserve, [&](int q, uint32_t first, uint32_t rank) {
    const uint32_t d = first + rank;
    if (d >= g.total) return;  // unreachable: the count kernel's bins
    dx[d] = x[q];
    dy[d] = y[q];
    dst.th[d] = th[q];
    dst.v[d] = v[q];
    dst.id[d] = id[q];
  });
  // each bin's first position: thread i scans kPer consecutive bins
  constexpr uint32_t kPer = kLocalBins / kAgentBlock;
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t c[kPer], sum = 0;
#pragma unroll
  for (uint32_t i = 0; i < kPer; i++) {
    c[i] = s_cnt[threadIdx.x * kPer + i];
    sum += c[i];
  }
  uint32_t run = sum;  // inclusive, over the wave
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t n = __shfl_up(run, off);
    if (lane >= static_cast<uint32_t>(off)) run += n;
  }
  if (lane == 63u) s_dst[threadIdx.x >> 6] = run;
  __syncthreads();
  run -= sum;
  uint32_t placed = 0;  // the workgroup's agents with an entry
#pragma unroll
  for (uint32_t i = 0; i < kAgentBlock / 64; i++) {
    if (i < threadIdx.x >> 6) run += s_dst[i];
    placed += s_dst[i];
  }
#pragma unroll
  for (uint32_t i = 0; i < kPer; i++) {
    s_cnt[threadIdx.x * kPer + i] = run;
    run += c[i];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kSortPer; q++)
    if (t.own[q]) {
      const uint32_t p = s_cnt[t.entry(q)] + t.r[q];
      s_dst[p] = s_base[t.entry(q)] + t.r[q];
      s_x[p] = x[q];
      s_y[p] = y[q];
      s_th[p] = __float_as_uint(th[q]);
      s_v[p] = __float_as_uint(v[q]);
      s_id[p] = id[q];
    }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    const uint32_t p = q * kAgentBlock + threadIdx.x;
    if (p >= placed) continue;
    const uint32_t d = s_dst[p];
    if (d >= g.total) continue;  // unreachable: the count kernel's bins
    dx[d] = s_x[p];
    dy[d] = s_y[p];
    dst.th[d] = __uint_as_float(s_th[p]);
    dst.v[d] = __uint_as_float(s_v[p]);
    dst.id[d] = s_id[p];
  }
}

// The scatter of pools up to ranked_agents: each agent straight to offset[bin] + rank,
// its bin recomputed by the count kernel's arithmetic.  No barrier and no atomic: a load
// and a store, in workgroups of kAgentBlock slots.  (Speed and index are loaded where they
// are stored: loaded with the others, 2^22 agents on 256^2 take 58.5 us instead of 57.5.)
template <bool P64>
__global__ __launch_bounds__(kAgentBlock) void scatter_ranked_kernel(
    SortArgs g, AgentSoA src, AgentSoA dst, const uint32_t* rank, const uint32_t* offset) {
  const uint32_t blk = g.xcd_remap ? xcd_logical_block(blockIdx.x, gridDim.x) : blockIdx.x;
  const uint32_t first = blk * kAgentBlock, last = min(first + kAgentBlock, g.total) - 1u;
  const uint32_t j = first + threadIdx.x;
  const bool act = j < g.total;
  double x64 = 0.0, y64 = 0.0;
  float x = 0.0f, y = 0.0f, th = 0.0f;
  uint32_t r = 0;
  if (act) {
    if constexpr (P64) {
      x64 = src.x64[j];
      y64 = src.y64[j];
      x = static_cast<float>(x64);
      y = static_cast<float>(y64);
    } else {
      x = src.x[j];
      y = src.y[j];
    }
    th = src.th[j];
    r = rank[j];
  }
  uint32_t k = 0;
  for (uint32_t ii = g.block_inst[blk];; ii++) {  // block-uniform walk
    const Instance in = g.insts[ii];
    const uint32_t end = in.agent_off + in.agent_count;
    if (act && j >= in.agent_off && j < end)
      k = key_of(x, y, th, in, g.params[ii], g.cell_log2, g.sort_key);
    if (last < end || ii + 1u >= g.ninst) break;
  }
  if (!act) return;
  const uint32_t d = offset[k] + r;
  if (d >= g.total) return;  // unreachable: the count kernel's bins
  if constexpr (P64) {
    dst.x64[d] = x64;
    dst.y64[d] = y64;
  } else {
    dst.x[d] = x;
    dst.y[d] = y;
  }
  dst.th[d] = th;
  dst.v[d] = src.v[j];
  dst.id[d] = src.id[j];
}

__global__ __launch_bounds__(kAgentBlock) void canonical_copy_kernel(
    AgentSoA src, AgentSoA dst, const Instance* insts, const uint32_t* block_inst, uint32_t total,
    int pos64) {
  uint32_t j = blockIdx.x * kAgentBlock + threadIdx.x;
  if (j >= total) return;
  uint32_t ii = block_inst[blockIdx.x];
  while (j >= insts[ii].agent_off + insts[ii].agent_count) ii++;  // ends: j < total
  uint32_t off = insts[ii].agent_off;
  uint32_t local = src.id ? src.id[j] : j - off;
  uint32_t d = off + local;
  if (pos64) {
    dst.x64[d] = src.x64[j];
    dst.y64[d] = src.y64[j];
  } else {
    dst.x[d] = src.x[j];
    dst.y[d] = src.y[j];
  }
  dst.th[d] = src.th[j];
  dst.v[d] = src.v[j];
  if (dst.id) dst.id[d] = local;
}

// Work items of a tile of n agents, cut into equal parts of about kItemAgents.
__device__ inline uint32_t items_of(uint32_t n) {
  return n == 0u ? 0u : max(1u, (n + kItemAgents / 2u) / kItemAgents);
}

// Work items of each tile, 0 for an empty one.
__global__ void tile_count_kernel(const Instance* insts, const uint32_t* tile_inst,
                                  uint32_t ntiles, uint32_t cell_log2, const uint32_t* offset,
                                  uint32_t* tile_items, WorkItem* items, uint32_t max_items) {
  uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  // every entry starts empty; tile_items_kernel fills those there are
  for (uint32_t i = g; i < max_items; i += gridDim.x * blockDim.x) items[i] = WorkItem{0, 0, 0, 0};
  if (g >= ntiles) return;
  const Instance in = insts[tile_inst[g]];
  uint32_t t = g - in.tile_off;
  uint32_t per = 1u << (2u * (in.tile_log2 - cell_log2));  // bins per tile
  uint32_t b0 = in.bin_off + t * per;
  uint32_t n = offset[b0 + per] - offset[b0];
  tile_items[g] = items_of(n);
}

// Writes each tile's work items.  Item k of the list goes to the entry of the
// block that takes logical block k of a launch over the items there are, so
// that every XCD works on one contiguous run of tiles and none is left without:
// a map over the whole list, whose empty end the last XCDs would get, left
// three of the eight idle.
__global__ void tile_items_kernel(const Instance* insts, const uint32_t* tile_inst,
                                  uint32_t ntiles, uint32_t cell_log2, const uint32_t* offset,
                                  const uint32_t* item_off, int xcd_remap, WorkItem* items) {
  uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ntiles) return;
  auto range = [&](uint32_t tile, uint32_t& ii, uint32_t& t, uint32_t& begin, uint32_t& end) {
    ii = tile_inst[tile];
    const Instance in = insts[ii];
    t = tile - in.tile_off;
    uint32_t per = 1u << (2u * (in.tile_log2 - cell_log2));
    uint32_t b0 = in.bin_off + t * per;
    begin = offset[b0];
    end = offset[b0 + per];
  };
  uint32_t ii, t, begin, end;
  range(ntiles - 1u, ii, t, begin, end);
  const uint32_t total = item_off[ntiles - 1u] + items_of(end - begin);
  range(g, ii, t, begin, end);
  const uint32_t n = items_of(end - begin);
  auto cut = [&](uint32_t i) {
    return begin + static_cast<uint32_t>(static_cast<uint64_t>(end - begin) * i / n);
  };
  for (uint32_t i = 0; i < n; i++) {
    const uint32_t k = item_off[g] + i;
    items[xcd_remap ? xcd_block_of(k, total) : k] = WorkItem{ii, t, cut(i), cut(i + 1u)};
  }
}

inline uint32_t next_pow2(uint32_t v) {
  uint32_t p = 1;
  while (p < v) p <<= 1;
  return p;
}

// Exclusive scan of in[0..n) into out, using the levels from `level` on.
void scan(const SortScratch& s, const uint32_t* in, uint32_t n, uint32_t* out, int level,
          hipStream_t stream) {
  uint32_t tiles = blocks_for(n, kScanTile);
  scan_tile_kernel<<<tiles, kScanBlock, 0, stream>>>(in, n, out, s.level[level]);
  if (tiles > 1) {
    scan(s, s.level[level], tiles, s.level[level], level + 1, stream);
    scan_add_kernel<<<tiles, kScanBlock, 0, stream>>>(out, n, s.level[level]);
  }
}

}  // namespace

uint64_t plan_bins(Instance& in, uint32_t cell_log2) {
  uint32_t side = 1u << cell_log2;
  in.nbx = (in.width + side - 1) / side;
  in.nby = (in.height + side - 1) / side;
  uint64_t p = next_pow2(in.nbx > in.nby ? in.nbx : in.nby);
  // a wide grid with small bins can need 2^32 or more; the caller rejects
  // counts beyond its limit (2^30), below which bin coordinates fit the
  // 16-bit Morton code
  in.nbins = static_cast<uint32_t>(std::min<uint64_t>(p * p, 0x80000000ull));
  return p * p;
}

uint32_t plan_scan(SortScratch& s, uint32_t nbins) {
  uint32_t n = nbins, total = 0;
  s.levels = 0;
  for (int k = 0; k < 3; k++) {
    n = blocks_for(n, kScanTile);
    s.level_len[k] = n;
    total += n;
    s.levels = k + 1;
    if (n <= 1) break;
  }
  return total;
}

void plan_tiles(Instance& in, uint32_t cell_log2, uint32_t tile_log2) {
  in.tile_log2 = tile_log2 > cell_log2 ? tile_log2 : cell_log2;
  in.tiles = in.nbins >> (2u * (in.tile_log2 - cell_log2));
  if (in.tiles == 0) {  // a whole grid smaller than one tile: one tile of all bins
    in.tile_log2 = cell_log2;
    while ((1u << (2u * (in.tile_log2 - cell_log2))) < in.nbins) in.tile_log2++;
    in.tiles = 1;
  }
}

void launch_morton_sort(const Pool& pool, const AgentSoA& src, const AgentSoA& dst,
                        const SortScratch& s, hipStream_t stream) {
  if (pool.total_agents == 0) return;
  zero_u32_kernel<<<blocks_for(pool.total_bins, 256), 256, 0, stream>>>(s.count, pool.total_bins);
  const SortArgs g{pool.inst,          pool.params,   pool.agent_block_inst, pool.count,
                   pool.total_agents,  pool.sort_cell_log2, pool.sort_key,   pool.xcd_remap};
  const uint32_t nb = blocks_for(pool.total_agents, kSortSlots);
  if (s.rank)
    count_kernel<true><<<nb, kAgentBlock, 0, stream>>>(g, src, pool.pos64, s.count, s.rank);
  else
    count_kernel<false><<<nb, kAgentBlock, 0, stream>>>(g, src, pool.pos64, s.count, nullptr);
  scan(s, s.count, pool.total_bins, s.offset, 0, stream);
  if (s.rank) {
    const uint32_t na = blocks_for(pool.total_agents, kAgentBlock);
    if (pool.pos64)
      scatter_ranked_kernel<true><<<na, kAgentBlock, 0, stream>>>(g, src, dst, s.rank, s.offset);
    else
      scatter_ranked_kernel<false><<<na, kAgentBlock, 0, stream>>>(g, src, dst, s.rank, s.offset);
  } else if (pool.pos64)
    scatter_kernel<true><<<nb, kAgentBlock, 0, stream>>>(g, src, dst, s.count, s.offset);
  else
    scatter_kernel<false><<<nb, kAgentBlock, 0, stream>>>(g, src, dst, s.count, s.offset);
  if (pool.items) {  // work list of the tiled agent pass
    uint32_t nt = pool.total_tiles;
    tile_count_kernel<<<blocks_for(nt, 256), 256, 0, stream>>>(
        pool.inst, pool.tile_inst, nt, pool.sort_cell_log2, s.offset, s.tile_items, pool.items,
        pool.max_items);
    scan(s, s.tile_items, nt, s.tile_items, 0, stream);
    tile_items_kernel<<<blocks_for(nt, 256), 256, 0, stream>>>(
        pool.inst, pool.tile_inst, nt, pool.sort_cell_log2, s.offset, s.tile_items,
        pool.xcd_remap, pool.items);
  }
}

void launch_canonical_copy(const Pool& pool, const AgentSoA& src, const AgentSoA& dst,
                           hipStream_t stream) {
  if (pool.total_agents == 0) return;
  canonical_copy_kernel<<<blocks_for(pool.total_agents, kAgentBlock), kAgentBlock, 0, stream>>>(
      src, dst, pool.inst, pool.agent_block_inst, pool.total_agents, pool.pos64);
}

}  // namespace slm
