// kernels.hip -- the step of a batch of runs as gfx950 kernels.
//
// One step of every active run is, in stream order:
//   k_transport      liquid transport of all runs      (implScalar.cpp:250-264);
//                    its last block lays out the step's tiles: the tile -> run
//                    table (k_layout alone at commit)
//   k_particle<M>    fused per-particle pass: model update + division requests
//                    + contribution scatter + move test + leave
//                    (model_kernel.hpp:163-268, contribution_kernel.hpp:144-186,
//                     move_kernel.hpp:209-273,347-437,586-648)
//   k_resolve<M>     neighbour pick + exit test of the particles that left their
//                    compartment; division acceptance in slot order over the
//                    run, mother halving, daughters written to [n, n + births)
//                    (particles_container.hpp:559-599); its last block keeps the
//                    books: counters, removal decision (particles_container.hpp:539-557)
//   k_remove_runs, or k_gap_count and k_gap_fill for large runs
//                    removal of Exit/Dead slots by gap filling over [0, n + births)
//                    (particles_container.hpp:292-385,735-796), when a particle
//                    can become inactive
// Every kernel reads particle counts from device memory, so the sequence can
// be replayed without host round trips.  The model-dependent kernels
// (k_transport, k_particle, k_resolve, k_properties) are templates in
// step_kernels.hpp; this file instantiates them for the built-in models and
// holds the others.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "step_kernels.hpp"

namespace mcst {

// ------------------------------------------------------------------ removal
// Over the slots [0, n_end) of every compacting run: gaps are the non-Idle
// slots below n_keep (ascending); fillers the Idle slots in [n_keep, n_end)
// (descending), the step's newborns among them.  The i-th gap receives the
// i-th filler (while both last, should the inactive count be wrong).
//
// The removal is launched with every step of a batch in which particles can
// leave, and does nothing in most of them (a run compacts when a hundredth of
// it is inactive), so what it costs is its launches, about 4.5 us each between
// two others: it used to be four.  Runs of up to REMOVE_RUN_TILES tiles are
// compacted by one block each, in one launch; above, the status bytes are
// counted per tile by the whole grid, whose last block adds up the tiles, and
// a second launch fills the gaps.  A single block compacts 250 000 slots of 8
// states (1 % of them gaps) in 90 us, in every 50th step or fewer of the
// lattice tanks: under 2 us a step against the second launch's 4.5; the time
// grows with the slots, so the line lies at twice that size.  (Launches of a
// step: 100 000 particles of a ring 26 -> 21 us a step, 250 000 of a lattice
// 50 -> 44 us, both with four launches before.)
__device__ __forceinline__ void move_particle(const BatchDev& b, uint32_t n_var, uint64_t dst, uint64_t src) {
  // every load of a group before its stores: the arrays may alias as far as
  // the compiler knows, and a load behind each store is a round trip each
  const uint32_t pos = b.pos[src], ch = b.clk_hyd[src], cd = b.clk_div[src];
  const double ah = b.age_hyd[src], ad = b.age_div[src];
  for (uint32_t v0 = 0; v0 < n_var; v0 += 4) {
    double x[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) x[j] = v0 + j < n_var ? b.state[(uint64_t)(v0 + j) * b.P + src] : 0.0;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
      if (v0 + j < n_var) b.state[(uint64_t)(v0 + j) * b.P + dst] = x[j];
  }
  b.pos[dst] = pos;
  b.status[dst] = IDLE;
  b.age_hyd[dst] = ah;
  b.age_div[dst] = ad;
  b.clk_hyd[dst] = ch;
  b.clk_div[dst] = cd;
}

// One block per run: the gaps from the front, listed in LDS until the next
// 8192 slots' may not fit (they are sparse: a hundredth of a run fits whole),
// and the fillers from the back, 4096 slots at a time (nearly all of them),
// matched as far as the shorter list goes.  (4096 slots of gaps at a time,
// moved before the next were read, took 335 us for 250 000 slots of 8 states,
// a round trip per 41 gaps.)
constexpr uint32_t REMOVE_THREADS = 1024, GAP_LIST = 8 * REMOVE_THREADS, FILL_LIST = 4 * REMOVE_THREADS;
__global__ void __launch_bounds__(REMOVE_THREADS) k_remove_runs(BatchDev b, uint32_t n_var) {
  constexpr uint32_t NWV = REMOVE_THREADS / 64;
  __shared__ uint32_t s_gap[GAP_LIST], s_fill[FILL_LIST];
  __shared__ uint32_t s_w[NWV];
  const uint32_t r = blockIdx.x;
  const RunState* rs = b.rs + r;
  if (rs->compact != 1u) return;
  const uint32_t n_end = rs->n_end, n_keep = rs->n_keep;
  const uint64_t p0 = b.runs[r].p_off;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  // Idle flags of the thread's 4 slots from s0 on that are in [lo, hi)
  auto idle4 = [&](uint32_t w, uint32_t s0, uint32_t lo, uint32_t hi, bool idle) -> uint32_t {
    uint32_t f = 0;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const bool hit = s0 + j >= lo && s0 + j < hi && ((((w >> (8 * j)) & 0xFFu) == IDLE) == idle);
      f |= (hit ? 1u : 0u) << j;
    }
    return f;
  };
  // block-wide: flags before this thread's, and their total
  auto scan = [&](uint32_t c, uint32_t& tot) -> uint32_t {
    const uint32_t inc = wave_incl_scan(c, lane);
    __syncthreads();  // earlier readers of s_w and of the lists are done
    if (lane == 63) s_w[wave] = inc;
    __syncthreads();
    uint32_t at = inc - c;
    tot = 0;
    for (uint32_t k = 0; k < NWV; ++k) {
      if (k < wave) at += s_w[k];
      tot += s_w[k];
    }
    return at;
  };
  const uint32_t* status = (const uint32_t*)(b.status + p0);  // a run starts on a tile: whole words
  uint32_t g_next = 0, f_next = n_end ? ((n_end - 1u) / FILL_LIST + 1u) * FILL_LIST : 0u;  // slots not yet listed
  uint32_t ng = 0, gi = 0, nf = 0, fi = 0;
  for (;;) {  // block-uniform
    if (gi == ng) {
      gi = ng = 0;
      while (g_next < n_keep) {
        const uint32_t s0 = g_next + 8u * tid;
        const uint32_t w0 = s0 < n_keep ? status[s0 / 4] : 0u, w1 = s0 + 4 < n_keep ? status[s0 / 4 + 1] : 0u;
        const uint32_t f = idle4(w0, s0, 0u, n_keep, false) | (idle4(w1, s0 + 4, 0u, n_keep, false) << 4);
        uint32_t tot;
        uint32_t at = ng + scan((uint32_t)__popc(f), tot);
        if (ng + tot > GAP_LIST) break;  // these with the next list
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j)
          if (f & (1u << j)) s_gap[at++] = s0 + j;
        ng += tot;
        g_next += GAP_LIST;
      }
    }
    while (fi == nf && f_next > n_keep) {
      f_next -= FILL_LIST;
      const uint32_t s0 = f_next + 4u * tid;
      const uint32_t f = idle4(s0 < n_end ? status[s0 / 4] : 0u, s0, n_keep, n_end, true);
      uint32_t tot;
      uint32_t at = scan((uint32_t)__popc(f), tot);
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j)
        if (f & (1u << j)) s_fill[tot - 1u - at++] = s0 + j;
      nf = tot;
      fi = 0;
    }
    if (gi == ng || fi == nf) return;
    __syncthreads();  // the lists are written
    const uint32_t m = ng - gi < nf - fi ? ng - gi : nf - fi;
    for (uint32_t k = tid; k < m; k += REMOVE_THREADS) move_particle(b, n_var, p0 + s_gap[gi + k], p0 + s_fill[fi + k]);
    gi += m;
    fi += m;
  }
}

// A tile's gaps (low 32 bits) and fillers (high) over the tiles of the removal
// layout (rm_tile_off, written by the bookkeeping); the grid's last block
// turns them into sums before each tile, tile_pre[0..T].  The counts cross
// blocks, so they are stored and read at device scope.
__global__ void __launch_bounds__(BLOCK) k_gap_count(BatchDev b) {
  __shared__ unsigned long long s_c[WAVES];
  __shared__ uint32_t s_last;
  const uint32_t* off = b.rm_tile_off;
  const uint32_t T = off[b.R];
  const uint32_t nb = T < gridDim.x ? T : gridDim.x;  // blocks with a tile
  if (blockIdx.x >= nb) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  for (uint32_t t = blockIdx.x; t < T; t += gridDim.x) {
    const uint32_t r = find_run(off, b.R, t);
    const RunState* rs = b.rs + r;
    const uint32_t s0 = (t - off[r]) * TILE + 4u * tid;
    const uint32_t n_end = rs->n_end, n_keep = rs->n_keep;
    const uint32_t w = s0 < n_end ? *(const uint32_t*)(b.status + b.runs[r].p_off + s0) : 0u;
    uint32_t ng = 0, nf = 0;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const bool live = ((w >> (8 * j)) & 0xFFu) == IDLE;
      const uint32_t s = s0 + j;
      ng += (s < n_keep && !live) ? 1u : 0u;
      nf += (s >= n_keep && s < n_end && live) ? 1u : 0u;
    }
    ng = wave_sum(ng);
    nf = wave_sum(nf);
    if (lane == 0) s_c[wave] = (unsigned long long)ng | ((unsigned long long)nf << 32);
    __syncthreads();
    if (tid == 0)
      __hip_atomic_store(b.tile_cnt + t, s_c[0] + s_c[1] + s_c[2] + s_c[3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
  }
  static_assert(WAVES == 4 && TILE == 4 * BLOCK, "four waves, four slots per thread");
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  uint32_t* ticket = b.ticket + (1u + RESOLVE_TICKETS) * TICKET_STRIDE;
  if (tid == 0) s_last = atomicAdd(ticket, 1u) == nb - 1u ? 1u : 0u;
  __syncthreads();
  if (!s_last) return;
  if (tid == 0) *ticket = 0u;
  // sums before each tile: RB consecutive tiles per thread and round
  constexpr uint32_t RB = 16;
  unsigned long long carry = 0;
  for (uint32_t base = 0; base < T; base += RB * BLOCK) {
    unsigned long long v[RB], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < RB; ++j) {
      const uint32_t t = base + tid * RB + j;
      v[j] = t < T ? __hip_atomic_load(b.tile_cnt + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
    }
#pragma unroll
    for (uint32_t j = 0; j < RB; ++j) sum += v[j];
    unsigned long long inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned long long x = __shfl_up(inc, d, 64);
      if (lane >= (uint32_t)d) inc += x;
    }
    __syncthreads();  // earlier readers of s_c are done
    if (lane == 63) s_c[wave] = inc;
    __syncthreads();
    unsigned long long run = carry + inc - sum;
    for (uint32_t k = 0; k < wave; ++k) run += s_c[k];
#pragma unroll
    for (uint32_t j = 0; j < RB; ++j) {
      const uint32_t t = base + tid * RB + j;
      if (t < T) b.tile_pre[t] = run;
      run += v[j];
    }
    carry += s_c[0] + s_c[1] + s_c[2] + s_c[3];
  }
  if (tid == 0) b.tile_pre[T] = carry;
}

// rank of this thread's flagged slots among the flagged slots of the tile,
// in ascending slot order (slot = k*BLOCK + tid); returns the tile total.
__device__ __forceinline__ uint32_t tile_ranks(const bool (&f)[PPT], uint32_t (&rank)[PPT],
                                               uint32_t (*s_cnt)[WAVES], uint32_t lane, uint32_t wave) {
  uint64_t mk[PPT];
#pragma unroll
  for (uint32_t k = 0; k < PPT; ++k) {
    mk[k] = __ballot(f[k]);
    if (lane == 0) s_cnt[k][wave] = (uint32_t)__popcll(mk[k]);
  }
  __syncthreads();
  uint32_t before = 0;
#pragma unroll
  for (uint32_t k = 0; k < PPT; ++k) {
    uint32_t rk = before + (uint32_t)__popcll(mk[k] & lanemask_lt(lane));
#pragma unroll
    for (uint32_t wv = 0; wv < WAVES; ++wv) {
      rk += (wv < wave) ? s_cnt[k][wv] : 0u;
      before += s_cnt[k][wv];
    }
    rank[k] = rk;
  }
  __syncthreads();
  return before;
}

// Fills the gaps of a tile: its gaps' ranks [go, go + ng) in the run name the
// fillers of descending rank [go, go + ng), which sit in one or a few
// consecutive tiles; the block lists those in LDS, then moves them.
__global__ void __launch_bounds__(BLOCK) k_gap_fill(BatchDev b, uint32_t n_var) {
  __shared__ uint32_t s_cnt[PPT][WAVES];
  __shared__ uint32_t s_src[TILE];
  const uint32_t* off = b.rm_tile_off;
  const uint32_t T = off[b.R];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  for (uint32_t t = blockIdx.x; t < T; t += gridDim.x) {
    const uint32_t ng = (uint32_t)b.tile_pre[t + 1] - (uint32_t)b.tile_pre[t];
    if (ng == 0) continue;
    const uint32_t r = find_run(off, b.R, t);
    const RunState* rs = b.rs + r;
    const uint64_t p0 = b.runs[r].p_off;
    const uint32_t t0 = off[r], t1 = off[r + 1];
    const unsigned long long pre0 = b.tile_pre[t0];
    const uint32_t f0 = (uint32_t)(pre0 >> 32);
    const uint32_t F = (uint32_t)(b.tile_pre[t1] >> 32) - f0;  // the run's fillers
    const uint32_t go = (uint32_t)b.tile_pre[t] - (uint32_t)pre0;
    const uint32_t n_end = rs->n_end, n_keep = rs->n_keep;
    // ascending ranks [qa, qb) of the fillers wanted (fewer than ng when they run out)
    const uint32_t qb = F > go ? F - go : 0u, qa = F > go + ng ? F - go - ng : 0u;
    if (qa >= qb) continue;
    // the last tile whose fillers start at or before rank qa
    uint32_t lo = t0, hi = t1;
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if ((uint32_t)(b.tile_pre[mid] >> 32) - f0 <= qa) lo = mid; else hi = mid;
    }
    for (uint32_t ft = lo; ft < t1; ++ft) {
      const uint32_t fb = (uint32_t)(b.tile_pre[ft] >> 32) - f0;  // rank of the tile's first filler
      if (fb >= qb) break;
      bool f[PPT];
      uint32_t rank[PPT];
#pragma unroll
      for (uint32_t k = 0; k < PPT; ++k) {
        const uint32_t s = (ft - t0) * TILE + k * BLOCK + tid;
        f[k] = s < n_end && s >= n_keep && b.status[p0 + s] == IDLE;
      }
      tile_ranks(f, rank, s_cnt, lane, wave);
#pragma unroll
      for (uint32_t k = 0; k < PPT; ++k) {
        const uint32_t q = fb + rank[k];
        if (f[k] && q >= qa && q < qb) s_src[q - qa] = (ft - t0) * TILE + k * BLOCK + tid;
      }
    }
    const uint32_t slot0 = (t - t0) * TILE;
    bool f[PPT];
    uint32_t rank[PPT];
#pragma unroll
    for (uint32_t k = 0; k < PPT; ++k) {
      const uint32_t s = slot0 + k * BLOCK + tid;
      f[k] = s < n_keep && b.status[p0 + s] != IDLE;
    }
    tile_ranks(f, rank, s_cnt, lane, wave);  // its barriers also put s_src before its readers
#pragma unroll
    for (uint32_t k = 0; k < PPT; ++k) {
      if (!f[k] || rank[k] >= qb - qa) continue;
      move_particle(b, n_var, p0 + slot0 + k * BLOCK + tid, p0 + s_src[qb - 1u - rank[k] - qa]);
    }
    __syncthreads();  // s_src is read before the next tile's list
  }
}

__global__ void __launch_bounds__(SCAN_THREADS) k_layout(BatchDev b) { layout_pass<SCAN_THREADS>(b); }

// ------------------------------------------------------------------ histogram
// Idle particles per compartment of run r (getRepartition, unit.cpp:190-230).
// As k_properties: a block counts a contiguous range of slots in LDS (`win`
// compartments; block row y the y-th window) and adds its nonzero counts, and
// a wave in one compartment counts itself once.  One global atomic per
// particle took 546 us for 1.5e6 particles in 500 compartments, now 15 us.
__global__ void __launch_bounds__(EXPORT_THREADS) k_repartition(BatchDev b, uint32_t r, unsigned long long* hist,
                                                                uint32_t win, uint32_t y0) {
  constexpr uint32_t NT = EXPORT_THREADS;
  extern __shared__ uint32_t s_cnt[];
  const RunDev& rd = b.runs[r];
  const uint32_t n = b.rs[r].n, n_c = rd.n_c;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t c0 = (y0 + blockIdx.y) * win, w = n_c - c0 < win ? n_c - c0 : win;
  const uint64_t even = ((uint64_t)n + gridDim.x - 1) / gridDim.x;
  const uint64_t per = even < EXPORT_MIN_SLOTS ? EXPORT_MIN_SLOTS : even;
  const uint64_t i0 = blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
  if (i0 >= i1) return;  // the whole block
  for (uint32_t i = tid; i < w; i += NT) s_cnt[i] = 0u;
  __syncthreads();
  for (uint64_t base = i0; base < i1; base += NT) {
    const uint64_t s = base + tid;
    const uint64_t g = rd.p_off + (s < i1 ? s : i0);
    const uint32_t k = b.pos[g] - c0;  // wraps above the window when below it
    const bool in = s < i1 && b.status[g] == IDLE && k < w;
    const uint64_t mask = __ballot(in);
    if (!mask) continue;
    const uint32_t lead = (uint32_t)__ffsll((long long)mask) - 1u;
    const uint32_t k0 = (uint32_t)__shfl((int)k, (int)lead, 64);
    if (__ballot(in && k == k0) == mask) {
      if (lane == lead) atomicAdd(s_cnt + k0, (uint32_t)__popcll(mask));
    } else if (in) {
      atomicAdd(s_cnt + k, 1u);
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < w; i += NT)
    if (s_cnt[i]) atomicAdd(hist + c0 + i, (unsigned long long)s_cnt[i]);
}

// Clears n counters (a kernel rather than a memset node, so that a caller
// may capture it in a graph).
__global__ void __launch_bounds__(256) k_clear_u64(unsigned long long* p, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = 0ull;
}

// ------------------------------------------------------------------ launchers
const ModelOps* builtin_model_ops(int model_id) {
  static const ModelOps ops[] = {model_ops<MonodMass>(), model_ops<DualMonod>(), model_ops<Monod>(),
                                 model_ops<FixedLength>(), model_ops<SimpleAcetate>(), model_ops<QuadMonod>()};
  static_assert(MonodMass::ID == 0 && DualMonod::ID == 1 && Monod::ID == 2 && FixedLength::ID == 3 &&
                    SimpleAcetate::ID == 4 && QuadMonod::ID == 5,
                "built-in model ids index the table");
  if (model_id < 0 || model_id >= (int)(sizeof(ops) / sizeof(ops[0]))) return nullptr;
  return &ops[model_id];
}

void launch_removal(const BatchDev& b, uint32_t n_var, int grid, uint32_t max_tiles, hipStream_t s) {
  if (max_tiles <= REMOVE_RUN_TILES) {
    hipLaunchKernelGGL(k_remove_runs, dim3(b.R), dim3(REMOVE_THREADS), 0, s, b, n_var);
    return;
  }
  hipLaunchKernelGGL(k_gap_count, dim3(grid), dim3(BLOCK), 0, s, b);
  hipLaunchKernelGGL(k_gap_fill, dim3(grid), dim3(BLOCK), 0, s, b, n_var);
}

void launch_layout(const BatchDev& b, hipStream_t s) {
  hipLaunchKernelGGL(k_layout, dim3(1), dim3(SCAN_THREADS), 0, s, b);
}

void launch_clear_u64(unsigned long long* p, uint64_t n, hipStream_t s) {
  const uint64_t blocks = std::min<uint64_t>((n + 255) / 256, 1024);
  hipLaunchKernelGGL(k_clear_u64, dim3((unsigned)std::max<uint64_t>(blocks, 1)), dim3(256), 0, s, p, n);
}

void launch_repartition(const BatchDev& b, uint32_t run, uint32_t n_c, unsigned long long* hist, hipStream_t s) {
  const uint32_t cells = EXPORT_LDS / sizeof(uint32_t);
  const uint32_t win = n_c < cells ? n_c : cells;
  const uint32_t n_win = (uint32_t)(((uint64_t)n_c + win - 1) / win);
  for (uint32_t y = 0; y < n_win; y += EXPORT_MAX_ROWS)
    hipLaunchKernelGGL(k_repartition, dim3(EXPORT_MAX_BLOCKS, std::min(n_win - y, EXPORT_MAX_ROWS)),
                       dim3(EXPORT_THREADS), (size_t)win * sizeof(uint32_t), s, b, run, hist, win, y);
}

}  // namespace mcst
