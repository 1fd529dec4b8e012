// step_kernels.hpp -- the model-dependent kernels of the step (k_transport,
// k_particle, k_resolve, k_properties) as templates over the model, and the
// ModelOps table that launches them.  kernels.hip instantiates them for the
// built-in models; udf_plugin.hip for a model compiled into a plugin and
// loaded at run time (mcst_model_load).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "models.hpp"

namespace mcst {

namespace {

// Pointers read from the run tables are generic; tell the compiler they point
// to global memory so it emits global_* rather than flat_* accesses.
#define GLOBAL_AS __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ GLOBAL_AS T* gp(T* p) {
  return (GLOBAL_AS T*)p;
}

// A value every lane of the wave holds identically, moved to scalar registers.
template <class T>
__device__ __forceinline__ T uniform(T v) {
  static_assert(sizeof(T) % 4 == 0, "uniform() works on whole dwords");
  union {
    T t;
    uint32_t w[sizeof(T) / 4];
  } u;
  u.t = v;
#pragma unroll
  for (unsigned i = 0; i < sizeof(T) / 4; ++i) u.w[i] = __builtin_amdgcn_readfirstlane(u.w[i]);
  return u.t;
}

// Streaming accesses to the particle arrays: non-temporal, so the particle
// stream does not evict the flowmap and compartment tables from L2.
template <class T>
__device__ __forceinline__ T ld_stream(const GLOBAL_AS T* p) {
  return __builtin_nontemporal_load(p);
}
template <class T>
__device__ __forceinline__ void st_stream(GLOBAL_AS T* p, T v) {
  __builtin_nontemporal_store(v, p);
}

__device__ __forceinline__ uint64_t lanemask_lt(uint32_t lane) { return lane ? (~0ull >> (64u - lane)) : 0ull; }

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v, uint32_t lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t t = __shfl_up(v, d, 64);
    if (lane >= (uint32_t)d) v += t;
  }
  return v;
}

// largest r in [0, R) with off[r] <= t, given off[0] = 0 <= t < off[R]
__device__ __forceinline__ uint32_t find_run(const uint32_t* off, uint32_t R, uint32_t t) {
  uint32_t lo = 0, hi = R;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (off[mid] <= t)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

constexpr uint32_t SCAN_THREADS = 1024;

}  // namespace

// ------------------------------------------------------------------ transport
// m += dt*(C*M - C*diag(sink) + S + F);  C = m*diag(1/V)  for every
// compartment of every active run, one thread each, all species at once (the
// flow matrix entries are read once for all of them); also refreshes the
// per-compartment record {M::record(C), p_move, q_exit} the particle pass
// gathers.  The extra last block lays out the step's tiles
// (layout_pass), which needs only the counts of the previous step.
template <uint32_t NT>
__device__ void layout_pass(const BatchDev& b);

// sum_i C[s][i] * M(i, j) over column j of a transport matrix stored by
// destination column, for every species, in entry order.  The transport is a
// chain of dependent loads on the critical path of a step, so it is cut where
// it can be: start() requests the first group of entries before the caller's
// other loads, and finish() requests each next group with the concentrations of
// the one before (a column holds the degree plus the diagonal, mostly 7 or 8).
// With the terms beside the inflow loaded before it and scalar run fields, the
// resolve kernel of 345 679 particles in 777 compartments takes 9.0 us instead
// of 10.1, of 250 003 in 1989 of 4 species 9.9 instead of 13.2.
template <int NS>
struct ColumnInflow {
  static constexpr uint32_t EG = NS >= 4 ? 2u : 4u;  // entries in a group: fewer for many species (registers)
  const GLOBAL_AS uint32_t* src;
  const GLOBAL_AS double* val;
  uint32_t e, e1;
  uint32_t i[EG];
  double v[EG];
  __device__ __forceinline__ void request(uint32_t (&ni)[EG], double (&nv)[EG], uint32_t from) const {
#pragma unroll
    for (uint32_t k = 0; k < EG; ++k) {
      const uint32_t ek = from + k < e1 ? from + k : e1 - 1u;
      ni[k] = src[ek];
      nv[k] = val[ek];
    }
  }
  __device__ __forceinline__ void start(const uint32_t* col_ptr, const uint32_t* s, const double* w, uint32_t j) {
    e = gp(col_ptr)[j];
    e1 = gp(col_ptr)[j + 1];
    src = gp(s);
    val = gp(w);
    if (e < e1) request(i, v, e);
  }
  __device__ __forceinline__ void finish(const GLOBAL_AS double* c, uint32_t n_c, double (&acc)[NS]) {
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = 0.0;
    while (e < e1) {
      double cv[EG][NS];
#pragma unroll
      for (uint32_t k = 0; k < EG; ++k)
#pragma unroll
        for (int s = 0; s < NS; ++s) cv[k][s] = c[(size_t)s * n_c + i[k]];
      uint32_t ni[EG];
      double nv[EG];
      if (e + EG < e1) request(ni, nv, e + EG);
#pragma unroll
      for (uint32_t k = 0; k < EG; ++k)
        if (e + k < e1)
#pragma unroll
          for (int s = 0; s < NS; ++s) acc[s] += cv[k][s] * v[k];
#pragma unroll
      for (uint32_t k = 0; k < EG; ++k) {
        i[k] = ni[k];
        v[k] = nv[k];
      }
      e += EG;
    }
  }
};

// The transport of compartment j of run r for the step `ahead` steps after its
// run's current one (0: the step about to run; 1: the next one, computed
// during this step's resolve kernel).  It reads C and the contributions of
// the last pass, from S or (TAKE > 0) from the TAKE accumulators the pass has
// just filled, which it clears, and writes the other C buffer, m and the record
// table of its step's parity; the resolve kernel reads none of these but the
// other record table.  The copies' loads are issued first and summed where the
// sum is used, behind the flow columns' chain of loads (a lane per copy and a
// sum by shuffles before that chain cost the resolve kernel 2 us).  TAKE
// without a next step of this call or of the run (`ahead` 0, or the run's step
// target): the sums go to S, so that S holds the step's contributions
// whenever the host can read it.  TAKE_ROWS: the contributions are `given`,
// summed from the rows by the caller.
//
// Every load of a run without a gas phase comes before the first store (the
// arrays may alias as far as the compiler knows: a store in between made it read
// the run's and the flowmap's fields again, a round trip each); with one, the
// gas is stored first, which spares its registers to the liquid's inflow.
constexpr int TAKE_ROWS = -1;
template <class M, int TAKE>
__device__ __forceinline__ void transport_one(const BatchDev& b, const RunDev* __restrict__ runs,
                                              const MapDev* __restrict__ maps, uint32_t r, uint32_t j, uint32_t ahead,
                                              const double* given = nullptr) {
  constexpr int NS = M::NS;
  constexpr int NR = record_terms<M>();
  constexpr uint32_t KM = TAKE > 0 ? (uint32_t)TAKE : 1u;
  const RunDev& rd = runs[r];
  // the step being prepared; the run's activity is recomputed here rather
  // than read from the layout, which other blocks write concurrently
  const uint32_t step = b.rs[r].step + ahead;
  if (step - ahead >= rd.step_target) return;  // the run did not take (or does not take) this step
  const uint32_t n_c = rd.n_c;
  // the contributions of the last pass
  double sp[KM][NS];
  GLOBAL_AS double* const from = gp(TAKE ? rd.Sp : rd.S) + j;
#pragma unroll
  for (uint32_t k = 0; k < KM; ++k)
#pragma unroll
    for (int s = 0; s < NS; ++s) sp[k][s] = TAKE == TAKE_ROWS ? given[s] : from[((size_t)k * NS + s) * n_c];
  auto source = [&](int s) -> double {
    double t = sp[0][s];
#pragma unroll
    for (uint32_t k = 1; k < KM; ++k) t += sp[k][s];
    return t;
  };
  auto clear = [&]() {
    if constexpr (TAKE <= 0) return;
#pragma unroll
    for (uint32_t k = 0; k < KM; ++k)
#pragma unroll
      for (int s = 0; s < NS; ++s) from[((size_t)k * NS + s) * n_c] = 0.0;
  };
  if (TAKE && (!ahead || step >= rd.step_target)) {
    GLOBAL_AS double* const S = gp(rd.S) + j;
#pragma unroll
    for (int s = 0; s < NS; ++s) S[(size_t)s * n_c] = source(s);
    clear();
    return;
  }
  const MapDev& mp = maps[rd.map_base + (step / rd.steps_per_map) % rd.n_maps];
  const bool flow = (b.stages & STAGE_TRANSPORT) != 0;
  ColumnInflow<NS> in;
  if (flow) in.start(mp.col_ptr, mp.src, mp.val, j);
  const GLOBAL_AS double* c = gp(rd.C[step & 1u]);
  double cn[NS], mn[NS];  // new concentrations and masses
#pragma unroll
  for (int s = 0; s < NS; ++s) cn[s] = c[(size_t)s * n_c + j];
  const double p_move = gp(mp.p_move)[j];
  double qx = gp(mp.q_exit)[j];
  const double* const vf = rd.vf_q + (size_t)(step % VF_ROWS) * rd.vf_w;  // this step's flows (n_vf > 0)
  if (rd.n_vf && rd.vx_slot[j] >= 0) qx = vf[rd.n_vf + (uint32_t)rd.vx_slot[j]];
  const bool gas = rd.Cg[0] != nullptr;
  if (flow) {
    double sink = gp(rd.sink)[j];
    const double inv_v = gp(mp.inv_v)[j];
    double fv[NS], fvg[NS];  // time-dependent feeds of this compartment, in feed order
    double sink_g = gas ? gp(rd.sink_g)[j] : 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      fv[s] = fvg[s] = 0.0;
      mn[s] = gp(rd.m)[(size_t)s * n_c + j];
    }
    if (rd.n_vf) {
      for (uint32_t q = rd.vf_sink_ptr[j]; q < rd.vf_sink_ptr[j + 1]; ++q) {
        const uint32_t k = rd.vf_sink_k[q];
        if (k & VF_GAS)
          sink_g = sink_g + vf[k & ~VF_GAS];
        else
          sink = sink + vf[k];
      }
      for (uint32_t q = rd.vf_src_ptr[j]; q < rd.vf_src_ptr[j + 1]; ++q) {
        const double add = vf[rd.vf_src_k[q]] * rd.vf_src_c[q];
        const uint32_t sp = rd.vf_src_s[q];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          if ((uint32_t)s == sp) fv[s] += add;
          if (((uint32_t)s | VF_GAS) == sp) fvg[s] += add;
        }
      }
    }
    // the terms beside the inflow
    double src_f[NS], out[NS], mtr[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      src_f[s] = source(s) + (gp(rd.F)[(size_t)s * n_c + j] + fv[s]);
      out[s] = cn[s] * sink;
      mtr[s] = 0.0;
    }
    double acc[NS];
    if (gas) {
      // two-phase step (SimulationUnit::ode_step, simulation.model.cpp:131-150):
      // mtr = kla*(H*C_gas - C)*V from the old concentrations, the gas
      // step with -mtr and the liquid step with +mtr (performStepGL,
      // implScalar.cpp:228-248), then clearNegs on the liquid
      // (implScalar.cpp:266-297): a value in (-1e-4*5e-3, 0) becomes 0
      const GLOBAL_AS double* cg = gp(rd.Cg[step & 1u]);
      ColumnInflow<NS> in_g;
      in_g.start(mp.g_col_ptr, mp.g_src, mp.g_val, j);
      in_g.finish(cg, n_c, acc);
      const double inv_vg = gp(mp.g_inv_v)[j];
      double cgn[NS], mgn[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const size_t o = (size_t)s * n_c + j;
        const double cgs = cg[o];
        mtr[s] = (gp(mp.g_kla)[o] * ((cgs * rd.henry[s]) - cn[s])) * gp(mp.vol)[j];
        const double dg = ((acc[s] - cgs * sink_g) + (gp(rd.Fg)[o] + fvg[s])) - mtr[s];
        mgn[s] = gp(rd.mg)[o] + rd.dt * dg;
        cgn[s] = mgn[s] * inv_vg;
      }
      GLOBAL_AS double* const Cgn = gp(rd.Cg[(step + 1u) & 1u]) + j;
      GLOBAL_AS double* const mg_out = gp(rd.mg) + j;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        Cgn[(size_t)s * n_c] = cgn[s];
        mg_out[(size_t)s * n_c] = mgn[s];
      }
    } else if (rd.kla) {  // gas-liquid transfer from a fixed gas phase: kla*(C* - C)*V
      const double vol = gp(mp.vol)[j];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const size_t o = (size_t)s * n_c + j;
        mtr[s] = (gp(rd.kla)[o] * (gp(rd.cstar)[o] - cn[s])) * vol;
      }
    }
    in.finish(c, n_c, acc);
    const double tol = 1e-4 * 5e-3;
    const bool transfer = gas || rd.kla;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      double dmdt = (acc[s] - out[s]) + src_f[s];
      if (transfer) dmdt = dmdt + mtr[s];
      mn[s] = mn[s] + rd.dt * dmdt;
      double cl = mn[s] * inv_v;
      if (gas && cl < 0.0 && fabs(cl) < tol) cl = 0.0;
      cn[s] = cl;
    }
  }
  double rt[NR];
  M::record(rd.params, cn, rt);
  GLOBAL_AS double* const rec = gp(rd.rec) + ((size_t)(step & 1u) * n_c + j) * rd.rec_w;
  GLOBAL_AS double* const Cn = gp(rd.C[(step + 1u) & 1u]) + j;
  GLOBAL_AS double* const m_out = gp(rd.m) + j;
#pragma unroll
  for (int k = 0; k < NR; ++k) rec[k] = rt[k];
  rec[NR] = p_move;
  rec[NR + 1] = qx;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const size_t o = (size_t)s * n_c;
    Cn[o] = cn[s];
    if (flow) m_out[o] = mn[s];
  }
  clear();
}

// The transport (or, TAKE, what becomes of the pass's contributions) of every
// active run's compartments, by blocks `blk` of `n_blk`.
template <class M, int TAKE>
__device__ void transport_compartments(const BatchDev& b, const RunDev* __restrict__ runs,
                                       const MapDev* __restrict__ maps, uint32_t blk, uint32_t n_blk, uint32_t ahead) {
  // a wave takes 64 compartments of one run (comp_off counts such chunks), so
  // that the run's and the flowmap's fields are scalars
  const uint32_t wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63u, wpb = blockDim.x >> 6;
  for (uint32_t q = blk * wpb + wave; q < b.n_chunk_total; q += n_blk * wpb) {
    const uint32_t r = find_run(b.comp_off, b.R, q);
    const uint32_t j = (q - b.comp_off[r]) * 64u + lane;
    if (j < runs[r].n_c) transport_one<M, TAKE>(b, runs, maps, r, j, ahead);
  }
}

// With contribution rows: as transport_compartments, a block taking 64
// compartments.  Each of its waves sums (and clears) a quarter of the rows, 8 in
// flight, and the first adds the waves' sums in turn: the order is the rows' alone.
template <class M>
__device__ void sum_rows(const BatchDev& b, const RunDev* __restrict__ runs, const MapDev* __restrict__ maps,
                         uint32_t blk, uint32_t n_blk, uint32_t ahead) {
  constexpr int NS = M::NS;
  constexpr uint32_t NWV = 256 / 64;
  __shared__ double s_sum[NWV][NS][64];
  const uint32_t wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63u;
  for (uint32_t q = blk; q < b.n_chunk_total; q += n_blk) {
    const uint32_t r = find_run(b.comp_off, b.R, q);
    const uint32_t n_c = runs[r].n_c, j = (q - b.comp_off[r]) * 64u + lane;
    if (b.rs[r].step >= runs[r].step_target) continue;  // the run took no step
    double t[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) t[s] = 0.0;
    if (j < n_c) {
      GLOBAL_AS double* const part = gp(runs[r].Sp) + j;
      constexpr uint32_t RG = 8;
      for (uint32_t row = wave; row < b.rows; row += RG * NWV) {
        double x[RG][NS];
#pragma unroll
        for (uint32_t k = 0; k < RG; ++k)
#pragma unroll
          for (int s = 0; s < NS; ++s)
            x[k][s] = row + k * NWV < b.rows ? part[((size_t)(row + k * NWV) * NS + s) * n_c] : 0.0;
#pragma unroll
        for (uint32_t k = 0; k < RG; ++k)
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            t[s] += x[k][s];
            if (row + k * NWV < b.rows) part[((size_t)(row + k * NWV) * NS + s) * n_c] = 0.0;
          }
      }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) s_sum[wave][s][lane] = t[s];
    __syncthreads();
    if (wave == 0 && j < n_c) {
#pragma unroll
      for (uint32_t w = 1; w < NWV; ++w)
#pragma unroll
        for (int s = 0; s < NS; ++s) t[s] += s_sum[w][s][lane];
      transport_one<M, TAKE_ROWS>(b, runs, maps, r, j, ahead, t);
    }
    __syncthreads();  // read before the next compartments' sums
  }
}

template <class M>
__global__ void __launch_bounds__(256) k_transport(BatchDev b, const RunDev* __restrict__ runs,
                                                  const MapDev* __restrict__ maps) {
  if (blockIdx.x == gridDim.x - 1) {
    layout_pass<256>(b);
    return;
  }
  transport_compartments<M, 0>(b, runs, maps, blockIdx.x, gridDim.x - 1, 0u);
}

// ------------------------------------------------------------------ particles
// This block's counter shard of run r.
__device__ __forceinline__ RunShard* run_shard(const BatchDev& b, uint32_t r) {
  return b.shards + (size_t)r * b.n_shard + (blockIdx.x & (b.n_shard - 1u));
}

// Two counts of a run in one word of its shard (no atomic for none).
__device__ __forceinline__ void add_pair(unsigned long long* w, uint32_t lo, uint32_t hi) {
  if (lo | hi) atomicAdd(w, (unsigned long long)lo | ((unsigned long long)hi << 32));
}

// Adds a block's LDS contribution accumulator, [n_s][win] for compartments
// [w0, w0 + win) of a run with n_c compartments, to S, and clears it: one
// atomic per nonzero entry.
template <int BLK>
__device__ __forceinline__ void flush_window(double* s_acc, GLOBAL_AS double* S, uint32_t ns, uint32_t win,
                                             uint32_t n_c, uint32_t w0, uint32_t tid) {
  const uint32_t len = ns * win;
  if (win == n_c) {  // the whole run: the layouts coincide
    for (uint32_t i = tid; i < len; i += BLK) {
      const double v = s_acc[i];
      if (v != 0.0) {
        unsafeAtomicAdd((double*)(S + i), v);
        s_acc[i] = 0.0;
      }
    }
    return;
  }
  for (uint32_t i = tid; i < len; i += BLK) {
    const double v = s_acc[i];
    if (v != 0.0) {
      const uint32_t q = i / win;
      unsafeAtomicAdd((double*)(S + (size_t)q * n_c + w0 + (i - q * win)), v);
      s_acc[i] = 0.0;
    }
  }
}

// First column of a cumulative row with cp[c] >= u, clamped to m-1: for a
// non-decreasing row this is #{c < m-1 : cp[c] < u}, the result of the
// reference's bisection (move_kernel.hpp:89-102).  The count runs over chunks
// of 8 independent loads, one memory round trip each, and stops at the first
// chunk holding a column with cp[c] >= u: in a non-decreasing row no later
// column can count.  Most rows end within the first chunk.
__device__ __forceinline__ uint32_t cdf_column(const GLOBAL_AS double* cp, uint32_t m, double u) {
  constexpr int CH = 8;
  uint32_t left = 0;
  const int last = (int)m - 1;
  for (int c0 = 0; c0 < last; c0 += CH) {
    double v[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) v[j] = (c0 + j < last) ? cp[c0 + j] : 2.0;
    uint32_t k = 0;
#pragma unroll
    for (int j = 0; j < CH; ++j) k += (u > v[j]) ? 1u : 0u;
    left += k;
    if (k < (uint32_t)CH) break;
  }
  return left;
}

// Where a particle that leaves compartment `pos` goes: the first column of its
// cumulative row at or above u (move_kernel.hpp:61-103).
__device__ __forceinline__ uint32_t next_place(const MapDev& mp, uint32_t pos, double u);

// Loads and stores of the NL consecutive slots of one lane: 8-byte fields
// move in 16-byte accesses per lane when NL > 1 (aligned: every run's slots
// start on a tile boundary), 4-byte fields in one access of 4*NL bytes.
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int NL>
__device__ __forceinline__ void ld_lane(const GLOBAL_AS double* p, double (&o)[NL]) {
  if constexpr (NL == 1) {
    o[0] = ld_stream(p);
  } else {
#pragma unroll
    for (int h = 0; h < NL / 2; ++h) {
      const f64x2 v = ld_stream((const GLOBAL_AS f64x2*)p + h);
      o[2 * h] = v[0];
      o[2 * h + 1] = v[1];
    }
  }
}
template <int NL>
__device__ __forceinline__ void ld_lane(const GLOBAL_AS uint32_t* p, uint32_t (&o)[NL]) {
  if constexpr (NL == 1) {
    o[0] = ld_stream(p);
  } else if constexpr (NL == 2) {
    const u32x2 v = ld_stream((const GLOBAL_AS u32x2*)p);
    o[0] = v[0];
    o[1] = v[1];
  } else {
    const u32x4 v = ld_stream((const GLOBAL_AS u32x4*)p);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = v[j];
  }
}
template <int NL>
__device__ __forceinline__ uint32_t ld_lane(const GLOBAL_AS uint8_t* p) {  // NL status bytes
  if constexpr (NL == 1)
    return ld_stream(p);
  else if constexpr (NL == 2)
    return ld_stream((const GLOBAL_AS uint16_t*)p);
  else
    return ld_stream((const GLOBAL_AS uint32_t*)p);
}
template <int NL>
__device__ __forceinline__ void st_lane(GLOBAL_AS double* p, const double (&v)[NL]) {
  if constexpr (NL == 1) {
    st_stream(p, v[0]);
  } else {
#pragma unroll
    for (int h = 0; h < NL / 2; ++h) {
      f64x2 w;
      w[0] = v[2 * h];
      w[1] = v[2 * h + 1];
      st_stream((GLOBAL_AS f64x2*)p + h, w);
    }
  }
}
template <int NL>
__device__ __forceinline__ void st_status(GLOBAL_AS uint8_t* p, uint32_t v) {
  if constexpr (NL == 1)
    *p = (uint8_t)v;
  else if constexpr (NL == 2)
    *(GLOBAL_AS uint16_t*)p = (uint16_t)v;
  else
    *(GLOBAL_AS uint32_t*)p = v;
}

__device__ __forceinline__ uint32_t next_place(const MapDev& mp, uint32_t pos, double u) {
  if (mp.move_row) {  // the compartment's 64-byte record: 5 cdf columns, 6 neighbours
    const GLOBAL_AS u32x4* rw = (const GLOBAL_AS u32x4*)(gp(mp.move_row) + (size_t)pos * 16);
    const u32x4 q0 = rw[0], q1 = rw[1], q2 = rw[2], q3 = rw[3];
    const uint32_t col = (u > __hiloint2double((int)q0.y, (int)q0.x) ? 1u : 0u) +
                         (u > __hiloint2double((int)q0.w, (int)q0.z) ? 1u : 0u) +
                         (u > __hiloint2double((int)q1.y, (int)q1.x) ? 1u : 0u) +
                         (u > __hiloint2double((int)q1.w, (int)q1.z) ? 1u : 0u) +
                         (u > __hiloint2double((int)q2.y, (int)q2.x) ? 1u : 0u);
    return col == 0 ? q2.z : col == 1 ? q2.w : col == 2 ? q3.x : col == 3 ? q3.y : col == 4 ? q3.z : q3.w;
  }
  const uint32_t m = mp.m;
  const uint32_t col = cdf_column(gp(mp.cdf) + (size_t)pos * m, m, u);
  return gp(mp.nbr)[(size_t)pos * m + col];
}

// The particle pass.  The unit of work is a sub-chunk of SUB = 64*NL slots;
// lane l holds the slots j*64 + l (ILV: every field access of the wave is a
// contiguous 64-slot run) or NL*l + j (16-byte accesses per lane).  A
// sub-chunk lists its movers and its division requests in its own segment of
// the tile's lists, so sub-chunks are independent: the block's waves take
// the sub-chunks of one group (one per wave) and groups are dealt to blocks G
// at a time (b.tile_group; 0: one contiguous range per block).  Which
// requests the run accepts (the first min(cap - n, div_cap) in slot order)
// is decided after the pass (k_resolve).  With PRIV the block accumulates the
// contributions of one run in LDS (ds_add_f64), switching runs only between
// groups; sub-chunks of another run add to S directly.
//
// Memory pipeline of a wave, per sub-chunk: issue the next sub-chunk's loads;
// compute on the current one with its compartment records (gathered one step
// earlier); gather the records of the next sub-chunk; store the current one.
// Every load is issued for every lane (slots past the count read valid
// memory of the tile and are masked where used), so the waits the compiler
// places for a load's operands do not depend on the data.
//
// LV: some run of the batch has a leaving flow.  Without one (LV false) the
// pass issues no load or store of hydraulic ages and gathers no exit
// threshold: the loads a run without an outlet would issue anyway, to a
// single address, took 3 % of the pass on the 1e7-particle network, and a
// run-time branch around them cost more than it saved.
template <class M, int BLK, int NL, bool ILV, bool PRIV, bool PROBE, bool WIN, bool LV>
__global__ void __launch_bounds__(BLK)
    k_particle(BatchDev b, const RunDev* __restrict__ runs, const RunState* __restrict__ rsr,
               const uint32_t* __restrict__ tile_off) {
  constexpr int NV = M::NV, NS = M::NS, NR = record_terms<M>(), REC = rec_stride(NR);
  constexpr int NQ = NR + 2;             // record fields: M::record terms r_0..r_{NR-1}, p_move, q_exit
  constexpr int NG = LV ? NQ : NQ - 1;   // fields gathered (q_exit only when some run leaves)
  constexpr int NP = M::NP > 0 ? M::NP : 1;
  constexpr uint32_t WPB = BLK / 64;     // waves per block = sub-chunks per group
  constexpr uint32_t SUB = 64 * NL;       // slots per sub-chunk
  static_assert(NL == 1 || NL == 2 || NL == 4, "1, 2 or 4 slots per lane");
  static_assert(NR >= 1 && NR + 2 <= 16, "1..14 record terms");
  constexpr uint32_t NSUB = TILE / SUB;  // sub-chunks per tile (b.nsub is set to the same)
  extern __shared__ double s_acc[];      // [n_s][acc_win] of run acc_run (PRIV)
  __shared__ uint32_t s_w0;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = uniform(tid >> 6);  // wave-uniform: scalar bookkeeping
  const uint32_t stages = b.stages;
  const uint64_t P = b.P;
  const uint32_t R = b.R;
  const uint32_t T = tile_off[R];
  const uint32_t n_sc = T * NSUB;        // sub-chunks of the pass
  const uint32_t n_groups = (n_sc + WPB - 1) / WPB;
  // a turn is at most a block's share of the groups, so that every block has
  // one (8 served runs of 6e5 particles: 12.0 us a pass, 17 with turns of 4)
  const uint32_t chunk = (n_groups + gridDim.x - 1) / gridDim.x;
  const uint32_t G = b.tile_group && b.tile_group < chunk ? b.tile_group : (chunk ? chunk : 1u);
  uint32_t grp = blockIdx.x * G;
  if (grp >= n_groups) return;  // the whole block
  const uint32_t copy = blockIdx.x & (b.n_copies - 1u);  // of each run's accumulator
  auto next_group = [&](uint32_t g) -> uint32_t {
    const uint32_t g0 = g - g % G;
    return (g + 1 < g0 + G) ? g + 1 : g0 + gridDim.x * G;
  };
  const bool do_model = (stages & STAGE_MODEL) != 0;
  const bool do_contrib = (stages & STAGE_CONTRIB) != 0;

  // one sub-chunk as the wave sees it; sc >= n_sc is a phantom: no slots,
  // no stores.  cnt counts the sub-chunk's slots below the run's count.
  struct SubRef {
    uint32_t sc, t, r, slot0, cnt;  // slot0: run-relative slot of the sub-chunk's first slot
    uint64_t base;                   // its batch-wide slot
    const double* rec;               // the run's record table of its current step
  };
  auto sub_ref = [&](uint32_t sc) -> SubRef {
    SubRef q{sc, 0u, 0u, 0u, 0u, 0ull, nullptr};
    // a phantom stands at the first slot of the pass's last tile: the run of
    // that tile is live, so the loads of the phantom (particle arrays, the
    // run's compartment record) stay inside memory the run owns; the run of
    // index 0 may have been retired and its arrays freed
    const uint32_t t = sc < n_sc ? sc / NSUB : T - 1u;
    q.t = t;
    q.r = find_run(tile_off, R, t);
    q.slot0 = (t - tile_off[q.r]) * TILE + (sc < n_sc ? (sc % NSUB) * SUB : 0u);
    if (sc < n_sc) {
      const uint32_t n = rsr[q.r].n;
      q.cnt = n > q.slot0 ? (n - q.slot0 < SUB ? n - q.slot0 : SUB) : 0u;
    }
    q.base = runs[q.r].p_off + q.slot0;
    q.rec = runs[q.r].rec + ((rsr[q.r].step & 1u) ? (size_t)runs[q.r].n_c * runs[q.r].rec_w : (size_t)0);
    return q;
  };
  // sub-chunk-relative slot of the lane's j-th slot: interleaved (64 apart,
  // every field access a contiguous 64-lane run) or NL consecutive slots
  auto off = [&](int j) -> uint32_t { return ILV ? (uint32_t)j * 64u + lane : NL * lane + (uint32_t)j; };
  // the NL slots of a lane in one sub-chunk, as loaded
  struct Sub {
    uint32_t st;       // NL status bytes
    uint32_t pos[NL];
    double x[NV][NL];
  };
  auto load_sub = [&](const SubRef& q, Sub& a) {
    if constexpr (ILV) {
      uint32_t st = 0;
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const uint64_t ij = q.base + (q.cnt ? off(j) : 0u);  // an empty sub-chunk reads its first slot
        st |= (uint32_t)ld_stream(gp(b.status) + ij) << (8 * j);
        a.pos[j] = ld_stream(gp(b.pos) + ij);
#pragma unroll
        for (int v = 0; v < NV; ++v) a.x[v][j] = reads_var<M>(v) ? ld_stream(gp(b.state) + (uint64_t)v * P + ij) : 0.0;
      }
      a.st = st;
    } else {
      const uint64_t i0 = q.base + (q.cnt ? NL * lane : 0u);
      a.st = ld_lane<NL>(gp(b.status) + i0);
      ld_lane<NL>(gp(b.pos) + i0, a.pos);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        if (reads_var<M>(v))
          ld_lane<NL>(gp(b.state) + (uint64_t)v * P + i0, a.x[v]);
        else
          for (int j = 0; j < NL; ++j) a.x[v][j] = 0.0;
      }
    }
  };
  auto gather = [&](const SubRef& q, const Sub& a, double (&rr)[NL][NQ]) {
    const GLOBAL_AS double* __restrict__ rec = gp(q.rec);
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      // slots past the count hold no particle: their position may be anything
      const uint32_t pj = off(j) < q.cnt ? a.pos[j] : 0u;
      const GLOBAL_AS double* rp = rec + (size_t)pj * REC;
#pragma unroll
      for (int f = 0; f < NG; ++f) rr[j][f] = rp[f];
      if constexpr (!LV) rr[j][NQ - 1] = 1.0;  // no exit test without a leaving flow
    }
  };

  // the wave's exits and deaths of the run cnt_run, added to its shard when
  // the wave changes runs (its movers and requests are counted from their
  // lists by k_resolve, a wave's count there being a block's of 8 to 16 waves)
  uint32_t cnt_exits = 0, cnt_deaths = 0;
  uint32_t cnt_run = 0xFFFFFFFFu;
  auto flush_counts = [&]() {
    if (cnt_run != 0xFFFFFFFFu && lane == 0) add_pair(&run_shard(b, cnt_run)->exits_deaths, cnt_exits, cnt_deaths);
    cnt_exits = cnt_deaths = 0;
  };
  // the wave's division requests summed per block of each level of the
  // request counts (div_l1/2/3: blocks of 2^6, 2^12, 2^18 sub-chunks),
  // added with one atomic when the wave leaves the block: its sub-chunks
  // come in increasing order.  An atomic per sub-chunk with requests put
  // most of a step's atomics on the few top-level entries when a tenth of
  // the cells divide together (the lattice tank: 1e6 requests per step)
  uint32_t dv_i[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, dv_n[3] = {0u, 0u, 0u};
  auto flush_requests = [&](int lvl) {
    if (dv_n[lvl] && lane == 0) {
      uint32_t* const base = lvl == 0 ? b.div_l1 : lvl == 1 ? b.div_l2 : b.div_l3;
      atomicAdd(base + dv_i[lvl], dv_n[lvl]);
    }
    dv_n[lvl] = 0u;
  };
  // the LDS accumulator holds compartments [acc_w0, acc_w0 + acc_win) of run
  // acc_run: the whole run when it fits (acc_win = n_c), else a window
  // centred on the block's first slot of the run (particles are stored in
  // compartment order, so a block's slots see few compartments); particles
  // outside the window add to S directly
  uint32_t acc_run = 0xFFFFFFFFu;
  GLOBAL_AS double* acc_S = nullptr;
  uint32_t acc_ns = 0, acc_nc = 0, acc_win = 0, acc_w0 = 0;

  SubRef cur = sub_ref(grp * WPB + wave);
  Sub A;
  double rr[NL][NQ];
  load_sub(cur, A);
  gather(cur, A, rr);
  // Later sub-chunks enter with their slots copied from the prefetch and
  // their records in flight; taking the first one's registers through empty
  // asm statements makes the entry path match.
  asm volatile("" : "+v"(A.st));
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    asm volatile("" : "+v"(A.pos[j]));
#pragma unroll
    for (int v = 0; v < NV; ++v)
      if (reads_var<M>(v)) asm volatile("" : "+v"(A.x[v][j]));
#pragma unroll
    for (int f = 0; f < NQ; ++f) asm volatile("" : "+v"(rr[j][f]));
  }

  for (;;) {
    // ---- block-uniform: the run whose contributions the LDS accumulates
    if (PRIV) {
      const uint32_t r0 = find_run(tile_off, R, (grp * WPB) / NSUB);
      if (r0 != acc_run) {
        __syncthreads();
        flush_window<BLK>(s_acc, acc_S, acc_ns, acc_win, acc_nc, acc_w0, tid);
        acc_run = r0;
        acc_S = gp(runs[r0].Sp) + (size_t)copy * runs[r0].n_s * runs[r0].n_c;
        acc_ns = runs[r0].n_s;
        acc_nc = runs[r0].n_c;
        acc_win = acc_nc;
        if constexpr (WIN) {
          acc_win = b.acc_w < acc_nc ? b.acc_w : acc_nc;
          if (tid == 0) {
            // wave 0 holds the group's first sub-chunk; its lane 0 the first slot
            s_w0 = window_at(cur.cnt ? A.pos[0] : 0u, acc_win, acc_nc);
          }
          __syncthreads();
          acc_w0 = s_w0;
        }
        for (uint32_t i = tid; i < acc_ns * acc_win; i += BLK) s_acc[i] = 0.0;
        __syncthreads();
      } else if constexpr (WIN) {
        // the window follows the block's slots, looked at where a turn of one
        // group begins, or every other group of a longer one (two block
        // barriers each time): flushed where it moves
        if (acc_win < acc_nc && (G == 1 || (grp & 1u) == 0)) {
          if (tid == 0) s_w0 = cur.cnt ? window_next(A.pos[0], acc_w0, acc_win, acc_nc) : acc_w0;
          __syncthreads();
          const uint32_t w0 = s_w0;
          __syncthreads();  // every wave has read s_w0
          if (w0 != acc_w0) {
            flush_window<BLK>(s_acc, acc_S, acc_ns, acc_win, acc_nc, acc_w0, tid);
            acc_w0 = w0;
            __syncthreads();  // the flush has cleared every entry
          }
        }
      }
    }
    // ---- the wave's sub-chunk of this group
    const uint32_t sc = cur.sc;
    const uint32_t r = cur.r;
    const RunDev& rd = runs[r];
    if (cur.cnt && r != cnt_run) {  // wave moves to another run
      flush_counts();
      cnt_run = r;
    }
    const uint32_t step = rsr[r].step;
    // the run's age clocks: the division clock of this step (after its tick
    // when the model runs), the hydraulic clock before this step's tick and
    // after it
    const uint32_t clk_d = rsr[r].clock_div + (do_model ? 1u : 0u);
    const uint32_t clk_h0 = rsr[r].clock_hyd;
    const double dt = rd.dt;
    const double w = rd.weight;
    const uint32_t n_c = rd.n_c;
    const uint64_t seed = rd.seed;
    GLOBAL_AS double* __restrict__ S = gp(rd.Sp) + (size_t)copy * NS * n_c;  // contributions outside LDS
    const bool to_lds = PRIV && r == acc_run;
    double p[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) p[q] = rd.params[q];
    const bool do_move = rd.enable_move && (stages & STAGE_MOVE);
    const bool do_leave = LV && rd.enable_leave && (stages & STAGE_LEAVE);
    const uint32_t clk_h = clk_h0 + (do_leave ? 1u : 0u);
    const uint32_t g_next = next_group(grp);

    // ---- prefetch: the wave's sub-chunk of the next group (a phantom past
    // the last group)
    const SubRef nxt = sub_ref(g_next < n_groups ? g_next * WPB + wave : n_sc);
    __builtin_amdgcn_sched_barrier(0);
    Sub B;
    load_sub(nxt, B);
    __builtin_amdgcn_sched_barrier(0);

    // ---- per-particle work: arithmetic only
    const uint32_t i0 = NL * lane;  // contiguous layout: sub-chunk-relative slot of j = 0
    const bool pair_valid = i0 < cur.cnt;
    bool valid[NL], idle[NL], updated[NL], want[NL], mover[NL], exited[NL], dead[NL];
    double x[NL][NV];
    double contrib[NL][NS];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const uint32_t stj = (A.st >> (8 * j)) & 0xFFu;
      valid[j] = off(j) < cur.cnt;
      idle[j] = valid[j] && stj == IDLE;
      updated[j] = idle[j] && do_model;  // its state changes
      want[j] = mover[j] = exited[j] = dead[j] = false;
#pragma unroll
      for (int v = 0; v < NV; ++v) x[j][v] = A.x[v][j];
#pragma unroll
      for (int q = 0; q < NS; ++q) contrib[j][q] = 0.0;
      if (!valid[j]) continue;
      if (idle[j]) {  // its division age ticks with the run's clock
        int code = IDLE;
        if (do_model) code = M::update(p, dt, x[j], rr[j], contrib[j]);
        if constexpr (M::CAN_DIE) dead[j] = code == DEAD;  // stops contributing and leaving
        want[j] = code == DIVISION;
      }
      // every slot below the count takes the move test, whatever its status
      // (move_kernel.hpp:209-273: Exit and Dead slots waiting for removal
      // keep moving); a particle that leaves its compartment (dt*Q/V > u,
      // probability_leaving.hpp:33-46) is listed, and k_resolve finds its
      // neighbour and, for an Idle one, runs its exit test there
      const U4 u = draw4(seed, cur.slot0 + off(j), step, TAG_TRANSPORT, 0u);
      mover[j] = do_move && rr[j][NR] > u01(u.x);
      if (do_leave && idle[j] && !dead[j]) {  // its hydraulic age ticks with the run's clock
        const double qx = rr[j][NR + 1];
        if (!mover[j] && qx < 1.0 && u01(u.z) > qx) {  // u > exp(-dt*Q/V)  <=>  dt*Q > -ln(u)*V
          if constexpr (PROBE) {
            if (rd.probe_exit) {
              const uint64_t g = cur.base + off(j);
              const double age = clock_age(gp(b.age_hyd)[g], clk_h, gp(b.clk_hyd)[g], dt);
              const unsigned long long e = atomicAdd(&b.rs[r].probe_exit_n, 1ull);
              if (e < rd.probe_cap) rd.probe_exit[e] = age;
            }
          }
          exited[j] = true;
        }
      }
    }
    // contributions of the Idle particles (a dead cell contributes nothing)
    if (do_contrib) {
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        if (!idle[j] || dead[j]) continue;
#pragma unroll
        for (int q = 0; q < NS; ++q) {
          const double c = w * contrib[j][q];
          if constexpr (WIN) {
            const uint32_t k = A.pos[j] - acc_w0;  // wraps above the window when below it
            if (to_lds && k < acc_win)
              atomicAdd(s_acc + q * acc_win + k, c);
            else
              unsafeAtomicAdd((double*)(S + (size_t)q * n_c + A.pos[j]), c);
          } else {
            if (to_lds)
              atomicAdd(s_acc + q * n_c + A.pos[j], c);
            else
              unsafeAtomicAdd((double*)(S + (size_t)q * n_c + A.pos[j]), c);
          }
        }
      }
    }

    // ---- the records of the next sub-chunk (its positions have arrived)
    double rn[NL][NQ];
    gather(nxt, B, rn);

    // ---- ranks of the sub-chunk's movers and division requests in slot order
    const uint64_t lt = lanemask_lt(lane);
    const uint64_t seg = (uint64_t)sc * SUB;  // the sub-chunk's list segment
    const uint32_t slot_t = cur.slot0 % TILE;  // tile-relative slot of the sub-chunk's first slot
    uint32_t n_mov = 0, n_div = 0;
    uint32_t rm[NL], rd_[NL];  // rank of slot off(j) among the flagged slots of the sub-chunk
    {
      uint64_t mv[NL], wd[NL];
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        mv[j] = __ballot(mover[j]);
        wd[j] = __ballot(want[j]);
      }
      if constexpr (ILV) {
        uint32_t am = 0, adv = 0;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
          rm[j] = am + (uint32_t)__popcll(mv[j] & lt);
          rd_[j] = adv + (uint32_t)__popcll(wd[j] & lt);
          am += (uint32_t)__popcll(mv[j]);
          adv += (uint32_t)__popcll(wd[j]);
        }
        n_mov = am;
        n_div = adv;
      } else {
        uint32_t bm = 0, bd = 0;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
          bm += (uint32_t)__popcll(mv[j] & lt);
          bd += (uint32_t)__popcll(wd[j] & lt);
          n_mov += (uint32_t)__popcll(mv[j]);
          n_div += (uint32_t)__popcll(wd[j]);
        }
#pragma unroll
        for (int j = 0; j < NL; ++j) {
          rm[j] = bm;
          rd_[j] = bd;
          bm += mover[j] ? 1u : 0u;
          bd += want[j] ? 1u : 0u;
        }
      }
    }
    // ---- divisions in registers (rare): the first DIV_STAGE requests of the
    // sub-chunk are divided here, where the mother's state is at hand.  Her
    // state before division is staged, one contiguous record per request; the
    // halved mother is stored below with everything else.  k_resolve decides
    // acceptance: an accepted request writes the daughter (M::division of the
    // staged state again: the same draws, so the same daughter) and restarts
    // the mother's division age, a refused one restores the mother from the
    // stage.  Later requests of a crowded sub-chunk are divided by k_resolve
    // from the stored state.
    if (n_div) {
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        if (!(want[j] && rd_[j] < DIV_STAGE)) continue;
        GLOBAL_AS double* stg = gp(b.div_stage) + ((uint64_t)sc * DIV_STAGE + rd_[j]) * NV;
        GLOBAL_AS double* const sj = gp(b.state) + cur.base + off(j);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          if (!reads_var<M>(v) && !writes_var<M>(v)) x[j][v] = sj[(uint64_t)v * P];
          stg[v] = x[j][v];
        }
        double xd[NV];
        M::division(p, x[j], xd, RngKey{seed, cur.slot0 + off(j), step});
#pragma unroll
        for (int v = 0; v < NV; ++v)
          if (!writes_var<M>(v)) sj[(uint64_t)v * P] = x[j][v];
      }
    }

    // ---- stores: the lane's final state, status changes, and the
    // sub-chunk's movers and division requests
    const uint64_t gi = cur.base + i0;
    if constexpr (ILV) {
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        if (!updated[j]) continue;
        const uint64_t gj = cur.base + off(j);
#pragma unroll
        for (int v = 0; v < NV; ++v)
          if (writes_var<M>(v)) st_stream(gp(b.state) + (uint64_t)v * P + gj, x[j][v]);
      }
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const uint64_t gj = cur.base + off(j);
        if (exited[j] || dead[j]) gp(b.status)[gj] = dead[j] ? (uint8_t)DEAD : (uint8_t)EXIT;
      }
    } else {
      bool all = true;
#pragma unroll
      for (int j = 0; j < NL; ++j) all = all && updated[j];
      if (all) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          if (!writes_var<M>(v)) continue;
          double xv[NL];
#pragma unroll
          for (int j = 0; j < NL; ++j) xv[j] = x[j][v];
          st_lane<NL>(gp(b.state) + (uint64_t)v * P + gi, xv);
        }
      } else {
#pragma unroll
        for (int j = 0; j < NL; ++j) {
          if (!updated[j]) continue;
#pragma unroll
          for (int v = 0; v < NV; ++v)
            if (writes_var<M>(v)) st_stream(gp(b.state) + (uint64_t)v * P + gi + (uint32_t)j, x[j][v]);
        }
      }
      uint32_t stn = A.st;
      bool changed = false;
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const uint32_t nv = dead[j] ? (uint32_t)DEAD : exited[j] ? (uint32_t)EXIT : ((A.st >> (8 * j)) & 0xFFu);
        stn = (stn & ~(0xFFu << (8 * j))) | (nv << (8 * j));
        changed = changed || exited[j] || dead[j];
      }
      if (changed && pair_valid) st_status<NL>(gp(b.status) + gi, stn);
    }
    // a slot that stops being Idle keeps its ages from now on: the hydraulic
    // age (0 after an exit; a dead cell's without this step's tick) and, in
    // clk_hyd, the division clock it stopped at (rare)
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      if (!(exited[j] || dead[j])) continue;
      const uint64_t g = cur.base + off(j);
      GLOBAL_AS double* a_h = gp(b.age_hyd) + g;
      GLOBAL_AS uint32_t* c_h = gp(b.clk_hyd) + g;
      *a_h = dead[j] ? clock_age(*a_h, clk_h0, *c_h, dt) : 0.0;
      *c_h = clk_d;
    }
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      if (mover[j]) {
        const bool leaves = idle[j] && !dead[j];
        const uint32_t pv = A.pos[j] < LIST_POS_FAR ? A.pos[j] : LIST_POS_FAR;
        gp(b.move_rec)[seg + rm[j]] = (slot_t + off(j)) | (leaves ? 0u : MOVER_INACTIVE) | (pv << LIST_POS_SHIFT);
      }
      if (n_div && want[j]) {  // rare
        const uint32_t pv = A.pos[j] < LIST_POS_FAR ? A.pos[j] : LIST_POS_FAR;
        gp(b.div_rec)[seg + rd_[j]] = (slot_t + off(j)) | (pv << LIST_POS_SHIFT);
        gp(b.div_pos)[seg + rd_[j]] = A.pos[j];
      }
    }
    if (lane == 0 && sc < n_sc) {
      gp(b.sub_moves)[sc] = n_mov;
      gp(b.sub_divs)[sc] = n_div;
    }
    if (n_div) {  // the block counts the resolve kernel's prefixes start from
#pragma unroll
      for (int lvl = 0; lvl < 3; ++lvl) {
        const uint32_t i = sc >> (6 * (lvl + 1));
        if (i != dv_i[lvl]) {
          flush_requests(lvl);
          dv_i[lvl] = i;
        }
        dv_n[lvl] += n_div;
      }
    }
    // ---- counters of the sub-chunk (wave-uniform)
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      if constexpr (LV) cnt_exits += (uint32_t)__popcll(__ballot(exited[j]));
      if constexpr (M::CAN_DIE) cnt_deaths += (uint32_t)__popcll(__ballot(dead[j]));
    }

    __builtin_amdgcn_sched_barrier(0);
    cur = nxt;
    A = B;
#pragma unroll
    for (int j = 0; j < NL; ++j)
#pragma unroll
      for (int f = 0; f < NQ; ++f) rr[j][f] = rn[j][f];
    grp = g_next;
    if (grp >= n_groups) break;
  }
  if (PRIV) {
    __syncthreads();
    flush_window<BLK>(s_acc, acc_S, acc_ns, acc_win, acc_nc, acc_w0, tid);
  }
  flush_counts();
#pragma unroll
  for (int lvl = 0; lvl < 3; ++lvl) flush_requests(lvl);
}

// The particle pass of a small batch (b.moved; small_tiles).  Such a pass is
// not bound by memory but by the length of one wave's work from the launch to
// its last store, so it is cut shorter, not wider: one
// slot per lane (a sub-chunk is 64 slots; with 4 the model and the draws of a
// wave took 2 us and the contributions of a wave up to 2.5), no pipeline across
// sub-chunks (a wave mostly has one), and a mover is moved here instead of in
// k_resolve, whose group scan, list and chain of loads took 3.8 us more: its
// row is requested before the model's arithmetic.  Plain loads and stores: the
// state stays in cache from step to step.  Pass and resolve of 100 000 particles
// of 2 states in 64 compartments 8.7 and 7.9 us before, 5.6 and 6.6 now.
template <class M, int BLK, bool LV>
__global__ void __launch_bounds__(BLK)
    k_particle_small(BatchDev b, const RunDev* __restrict__ runs, const RunState* __restrict__ rsr,
                     const MapDev* __restrict__ maps, const uint32_t* __restrict__ tile_off) {
  constexpr int NV = M::NV, NS = M::NS, NR = record_terms<M>(), REC = rec_stride(NR);
  constexpr int NQ = NR + 2, NG = LV ? NQ : NQ - 1;
  constexpr int NP = M::NP > 0 ? M::NP : 1;
  constexpr uint32_t WPB = BLK / 64, SUB = 64, NSUB = TILE / SUB;
  extern __shared__ double s_acc[];  // [n_s][n_c] of run acc_run
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = uniform(tid >> 6);
  const uint32_t stages = b.stages, R = b.R;
  const uint64_t P = b.P;
  const uint32_t n_sc = tile_off[R] * NSUB;
  const uint32_t n_groups = (n_sc + WPB - 1) / WPB;
  // groups dealt to the blocks one at a time, or one range per block
  const uint32_t chunk = (n_groups + gridDim.x - 1) / gridDim.x;
  const bool deal = b.tile_group == 1u;
  const uint32_t g_first = deal ? blockIdx.x : blockIdx.x * chunk, g_step = deal ? gridDim.x : 1u;
  const uint32_t g_end = deal || n_groups - g_first < chunk ? n_groups : g_first + chunk;
  if (g_first >= n_groups) return;
  const uint32_t copy = blockIdx.x & (b.n_copies - 1u);
  const bool do_model = (stages & STAGE_MODEL) != 0;
  const bool do_contrib = (stages & STAGE_CONTRIB) != 0;
  uint32_t acc_run = 0xFFFFFFFFu, acc_ns = 0, acc_nc = 0;
  GLOBAL_AS double* acc_S = nullptr;
  for (uint32_t grp = g_first; grp < g_end; grp += g_step) {
    // ---- the wave's sub-chunk; none past the last (every wave meets the
    // block's barriers)
    const uint32_t sc = grp * WPB + wave;
    const bool on = sc < n_sc;
    const uint32_t t = on ? sc / NSUB : 0u;
    const uint32_t r = on ? find_run(tile_off, R, t) : 0u;
    const RunDev& rd = runs[r];
    const uint32_t slot0 = on ? (t - tile_off[r]) * TILE + (sc % NSUB) * SUB : 0u;
    const uint32_t n = on ? rsr[r].n : 0u;
    const bool valid = slot0 + lane < n;  // its lane's slot holds a particle
    const uint32_t slot = valid ? slot0 + lane : 0u;
    const uint64_t g = rd.p_off + slot;
    uint32_t st = EXIT, pos = 0;
    double x[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) x[v] = 0.0;
    if (valid) {
      st = gp(b.status)[g];
      pos = gp(b.pos)[g];
#pragma unroll
      for (int v = 0; v < NV; ++v)
        if (reads_var<M>(v)) x[v] = gp(b.state)[(uint64_t)v * P + g];
    }
    // ---- block-uniform: the run whose contributions the LDS accumulates
    const uint32_t r0 = find_run(tile_off, R, (grp * WPB) / NSUB);
    if (r0 != acc_run) {
      __syncthreads();
      flush_window<BLK>(s_acc, acc_S, acc_ns, acc_nc, acc_nc, 0u, tid);
      acc_run = r0;
      acc_ns = runs[r0].n_s;
      acc_nc = runs[r0].n_c;
      acc_S = gp(runs[r0].Sp) + (size_t)copy * acc_ns * acc_nc;
      for (uint32_t i = tid; i < acc_ns * acc_nc; i += BLK) s_acc[i] = 0.0;
      __syncthreads();
    }
    if (!on) continue;
    const uint32_t step = rsr[r].step;
    const uint32_t n_c = rd.n_c;
    const double dt = rd.dt, w = rd.weight;
    const bool do_move = rd.enable_move && (stages & STAGE_MOVE);
    const bool do_leave = LV && rd.enable_leave && (stages & STAGE_LEAVE);
    const uint32_t clk_d = rsr[r].clock_div + (do_model ? 1u : 0u);
    const uint32_t clk_h0 = rsr[r].clock_hyd;
    const MapDev& mp = maps[rd.map_base + (step / rd.steps_per_map) % rd.n_maps];
    const GLOBAL_AS double* const rec = gp(rd.rec) + ((step & 1u) ? (size_t)n_c * REC : (size_t)0);
    double rr[NQ];
#pragma unroll
    for (int f = 0; f < NG; ++f) rr[f] = valid ? rec[(size_t)pos * REC + f] : 0.0;
    if constexpr (!LV) rr[NQ - 1] = 1.0;
    double p[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) p[q] = rd.params[q];

    // ---- the particle: draws, move, model
    const U4 u = draw4(rd.seed, slot, step, TAG_TRANSPORT, 0u);
    const bool idle = valid && st == IDLE;
    const bool mover = valid && do_move && rr[NR] > u01(u.x);  // whatever its status
    uint32_t to = pos;
    if (mover) to = next_place(mp, pos, u01(u.y));
    bool want = false, dead = false, exited = false;
    double contrib[NS];
#pragma unroll
    for (int q = 0; q < NS; ++q) contrib[q] = 0.0;
    if (idle && do_model) {
      const int code = M::update(p, dt, x, rr, contrib);
      if constexpr (M::CAN_DIE) dead = code == DEAD;
      want = code == DIVISION;
    }
    if (do_contrib && idle && !dead) {
#pragma unroll
      for (int q = 0; q < NS; ++q) {
        const double c = w * contrib[q];
        if (r == acc_run)
          atomicAdd(s_acc + q * n_c + pos, c);
        else
          unsafeAtomicAdd((double*)(gp(rd.Sp) + ((size_t)copy * NS + q) * n_c + pos), c);
      }
    }
    if (do_leave && idle && !dead) {  // the exit test in the compartment it is in now
      const double qx = mover ? rec[(size_t)to * REC + NR + 1] : rr[NR + 1];
      exited = qx < 1.0 && u01(u.z) > qx;
    }
    // ---- division requests of the sub-chunk, as in k_particle
    const uint64_t wd = __ballot(want), mv = __ballot(mover);
    const uint32_t n_div = (uint32_t)__popcll(wd);
    const uint32_t rk = (uint32_t)__popcll(wd & lanemask_lt(lane));
    if (n_div) {
      const uint64_t seg = (uint64_t)sc * SUB;
      if (want) {
        if (rk < DIV_STAGE) {
          GLOBAL_AS double* stg = gp(b.div_stage) + ((uint64_t)sc * DIV_STAGE + rk) * NV;
          GLOBAL_AS double* const sg = gp(b.state) + g;
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            if (!reads_var<M>(v) && !writes_var<M>(v)) x[v] = sg[(uint64_t)v * P];
            stg[v] = x[v];
          }
          double xd[NV];
          M::division(p, x, xd, RngKey{rd.seed, slot, step});
#pragma unroll
          for (int v = 0; v < NV; ++v)
            if (!writes_var<M>(v)) sg[(uint64_t)v * P] = x[v];
        }
        const uint32_t pv = pos < LIST_POS_FAR ? pos : LIST_POS_FAR;
        gp(b.div_rec)[seg + rk] = (slot % TILE) | (pv << LIST_POS_SHIFT);
        gp(b.div_pos)[seg + rk] = pos;
      }
      // of the block counts, those of 64 sub-chunks alone (request_prefix): with
      // an atomic per sub-chunk on a count of 4096 as well, 8e5 cells in a full
      // container, a quarter of them asking in every step, had a pass of 106 us,
      // nearly all of it those atomics one after another; now 49
      // (the index in a vector register: for an address that it knows to be the
      // wave's the compiler puts a reduction over the wave before the atomic)
      uint32_t i1 = sc >> 6;
      asm volatile("" : "+v"(i1));
      if (lane == 0) atomicAdd(b.div_l1 + i1, n_div);
    }
    // ---- stores
    if (idle && do_model) {
#pragma unroll
      for (int v = 0; v < NV; ++v)
        if (writes_var<M>(v)) gp(b.state)[(uint64_t)v * P + g] = x[v];
    }
    if (mover) gp(b.pos)[g] = to;
    if (exited || dead) {
      gp(b.status)[g] = dead ? (uint8_t)DEAD : (uint8_t)EXIT;
      GLOBAL_AS double* a_h = gp(b.age_hyd) + g;
      GLOBAL_AS uint32_t* c_h = gp(b.clk_hyd) + g;
      *a_h = dead ? clock_age(*a_h, clk_h0, *c_h, dt) : 0.0;
      *c_h = clk_d;
    }
    const uint32_t n_exit = LV ? (uint32_t)__popcll(__ballot(exited)) : 0u;
    const uint32_t n_dead = M::CAN_DIE ? (uint32_t)__popcll(__ballot(dead)) : 0u;
    if (lane == 0) {
      gp(b.sub_moves)[sc] = (uint32_t)__popcll(mv);
      gp(b.sub_divs)[sc] = n_div;
      add_pair(&run_shard(b, r)->exits_deaths, n_exit, n_dead);
    }
  }
  __syncthreads();
  flush_window<BLK>(s_acc, acc_S, acc_ns, acc_nc, acc_nc, 0u, tid);
}

// What the books read of a run, requested together (before its counter shards
// are, so that both round trips to memory overlap).
struct RunBooks {
  uint32_t n = 0, inactive = 0, step = 0, active = 0;
  uint32_t cap = 0, div_cap = 0, leave = 0, target = 0;
  uint64_t min_removal = 0;
  double ratio = 0.0;
  unsigned long long cnt[C_COUNT] = {};
};

__device__ __forceinline__ void read_books(const RunState* rs, const RunDev& rd, RunBooks& k) {
  k.n = rs->n;
  k.inactive = rs->inactive;
  k.step = rs->step;
  k.active = rs->active;
#pragma unroll
  for (int c = 0; c < C_COUNT; ++c) k.cnt[c] = rs->counters[c];
  k.cap = rd.cap;
  k.div_cap = rd.div_cap;
  k.leave = rd.enable_leave;
  k.target = rd.step_target;
  k.min_removal = rd.min_removal;
  k.ratio = rd.ratio;
}

// The books of one run after its step, from the step's counts (packed as in
// RunShard).  tiles: of [0, n_end) when the run compacts; tiles_l: of the next
// step's layout.
__device__ __forceinline__ void keep_books(const BatchDev& b, RunState* rs, RunBooks& k, unsigned long long mr,
                                           unsigned long long ed, bool layout, uint32_t& tiles, uint32_t& tiles_l) {
  uint32_t step_now = k.step, n_now = k.n;  // after this step's books
  if (k.active) {
    const uint32_t n = k.n;
    const unsigned long long moves = (uint32_t)mr, req = mr >> 32;
    const unsigned long long exits = (uint32_t)ed, deaths = ed >> 32;
    const unsigned long long processed = n - k.inactive;  // every Idle slot
    const uint32_t room = k.cap - n;
    const uint32_t budget = room < k.div_cap ? room : k.div_cap;
    const uint32_t births = req < budget ? (uint32_t)req : budget;
    k.cnt[C_BIRTHS] += births;
    k.cnt[C_EXITS] += exits;
    k.cnt[C_DEATHS] += deaths;
    k.cnt[C_MOVES] += moves;
    k.cnt[C_OVERFLOW] += req - births;
    k.cnt[C_PROCESSED] += processed;
    uint64_t inactive = (uint64_t)k.inactive + exits + deaths;
    const uint64_t thr_ratio = (uint64_t)((double)n * k.ratio);
    const uint64_t thr = k.min_removal > thr_ratio ? k.min_removal : thr_ratio;
    const uint32_t n_end = n + births;
    uint32_t n_keep = n_end, compact = 0;
    if ((b.stages & STAGE_REMOVE) && inactive > thr) {
      k.cnt[C_COMPACTIONS] += 1;
      if (inactive >= n_end) {
        n_keep = 0;
        compact = 2;  // everything removed, nothing to move
      } else {
        n_keep = n_end - (uint32_t)inactive;
        compact = 1;
        tiles = (n_end + TILE - 1u) / TILE;
      }
      inactive = 0;
    }
    // the age clocks tick with the stages the step ran
    if (b.stages & STAGE_MODEL) rs->clock_div += 1u;
    if (k.leave && (b.stages & STAGE_LEAVE)) rs->clock_hyd += 1u;
    step_now = k.step + 1u;
    n_now = n_keep;
    rs->n_end = n_end;
    rs->n_keep = n_keep;
    rs->compact = compact;
    rs->births = births;
    rs->inactive = (uint32_t)inactive;
    rs->n = n_keep;
    rs->step = step_now;
    k.cnt[C_STEPS] = step_now;
    k.cnt[C_N] = n_keep;
    k.cnt[C_INACTIVE] = (uint32_t)inactive;
#pragma unroll
    for (int c = 0; c < C_COUNT; ++c) rs->counters[c] = k.cnt[c];
  } else {
    rs->compact = 0;
  }
  if (layout) {  // layout_pass's table, from the values at hand
    const uint32_t act = step_now < k.target ? 1u : 0u;
    tiles_l = act ? (n_now + TILE - 1u) / TILE : 0u;
    rs->active = act;
    rs->n_tiles = tiles_l;
  }
}

// The books of every run after its step, kept by the last block of
// k_resolve: counters, births (the accepted requests), the removal decision
// of update_and_remove_inactive (particles_container.hpp:539-557, threshold
// from the pass's count) over [0, n_end) where the newborns already sit, and
// the removal's tile layout; then the request block counts are cleared for
// the next pass (n_sc: the sub-chunks of this step's layout).  With `layout`
// it also lays out the next step's tiles (layout_pass), from the counts it
// has just computed, in the other of two tables: a resolve block without a
// group is not waited for, so it may start after the books and must still find
// the step's own tile count, or it would take itself for a block with work.
__device__ void bookkeep_pass(const BatchDev& b, const RunDev* __restrict__ runs, uint32_t n_sc, bool layout) {
  constexpr uint32_t NT = 256, NWV = NT / 64;
  __shared__ uint32_t s_w[NWV], s_wl[NWV];
  __shared__ uint32_t s_carry, s_carry_l;
  __shared__ unsigned long long s_mr[NT], s_ed[NT];  // the counts of 256 runs, summed over their shards
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t nsh = b.n_shard;
  // read and reset with atomics: other blocks added to the shards with
  // atomics up to a moment ago.  One lane per shard, all in flight at once;
  // both halves of a sum stay below 2^32 (a run has fewer slots)
  auto take = [&](uint32_t i, uint32_t n, unsigned long long& mr, unsigned long long& ed) {
    mr = ed = 0;
    if (i < n) {
      mr = atomicExch(&b.shards[i].moves_requests, 0ull);
      ed = atomicExch(&b.shards[i].exits_deaths, 0ull);
    }
    for (uint32_t d = nsh >> 1; d; d >>= 1) {
      mr += __shfl_xor(mr, (int)d, 64);
      ed += __shfl_xor(ed, (int)d, 64);
    }
  };
  if (b.R == 1) {  // one run: no scan over runs, no barrier (1 us of a step)
    if (wave == 0) {
      RunBooks k;
      if (lane == 0) read_books(b.rs, runs[0], k);
      unsigned long long mr, ed;
      take(lane, nsh, mr, ed);
      if (lane == 0) {
        uint32_t tiles = 0, tiles_l = 0;
        keep_books(b, b.rs, k, mr, ed, layout, tiles, tiles_l);
        b.rm_tile_off[0] = 0u;
        b.rm_tile_off[1] = tiles;
        if (layout) {
          b.tile_off_next[0] = 0u;
          b.tile_off_next[1] = tiles_l;
          b.rs[0].tile_begin = 0u;
        }
      }
    }
  } else {
    if (tid == 0) s_carry = s_carry_l = 0;
    for (uint32_t r0 = 0; r0 < b.R; r0 += NT) {
      const uint32_t r = r0 + tid;
      RunBooks k;
      if (r < b.R) read_books(b.rs + r, runs[r], k);
      const uint32_t n_run = b.R - r0 < NT ? b.R - r0 : NT;
      for (uint32_t i0 = 0; i0 < n_run * nsh; i0 += NT) {
        const uint32_t i = i0 + tid;
        unsigned long long mr, ed;
        take(r0 * nsh + i, (r0 + n_run) * nsh, mr, ed);
        if (i < n_run * nsh && i % nsh == 0) {
          s_mr[i / nsh] = mr;
          s_ed[i / nsh] = ed;
        }
      }
      __syncthreads();
      uint32_t tiles = 0, tiles_l = 0;
      if (r < b.R) keep_books(b, b.rs + r, k, s_mr[tid], s_ed[tid], layout, tiles, tiles_l);
      const uint32_t inc = wave_incl_scan(tiles, lane);
      const uint32_t inc_l = layout ? wave_incl_scan(tiles_l, lane) : 0u;
      if (lane == 63) {
        s_w[wave] = inc;
        s_wl[wave] = inc_l;
      }
      __syncthreads();
      uint32_t wpre = 0, tot = 0, wpre_l = 0, tot_l = 0;
      for (uint32_t w = 0; w < NWV; ++w) {
        if (w < wave) {
          wpre += s_w[w];
          wpre_l += s_wl[w];
        }
        tot += s_w[w];
        tot_l += s_wl[w];
      }
      const uint32_t carry = s_carry, carry_l = s_carry_l;
      if (r < b.R) {
        b.rm_tile_off[r] = carry + wpre + inc - tiles;
        if (layout) {
          b.tile_off_next[r] = carry_l + wpre_l + inc_l - tiles_l;
          b.rs[r].tile_begin = carry_l + wpre_l + inc_l - tiles_l;
        }
      }
      __syncthreads();
      if (tid == 0) {
        s_carry = carry + tot;
        s_carry_l = carry_l + tot_l;
      }
      __syncthreads();
    }
    if (tid == 0) {
      b.rm_tile_off[b.R] = s_carry;
      if (layout) b.tile_off_next[b.R] = s_carry_l;
    }
  }
  for (uint32_t i = tid; i < (n_sc + 63u) >> 6; i += NT) b.div_l1[i] = 0u;
  for (uint32_t i = tid; i < (n_sc + 4095u) >> 12; i += NT) b.div_l2[i] = 0u;
  for (uint32_t i = tid; i <= (n_sc >> 18); i += NT) b.div_l3[i] = 0u;
  for (uint32_t i = tid; i <= RESOLVE_TICKETS; i += NT) b.ticket[i * TICKET_STRIDE] = 0u;
}

// After the particle pass, per group of 32 or 64 sub-chunks, 128 after the small
// pool's pass (one per thread of the block for the prefix sums): (1) the movers the pass listed take
// their neighbour, the first CDF column at or above u, and an Idle one runs
// the exit test in its new compartment (move_kernel.hpp:392-437, 586-648);
// (2) the division requests are accepted in slot order over the whole run:
// the k-th request of the step (k counted from the run's first slot)
// succeeds iff k < min(cap - n, div_cap), the reference's division buffer
// (particles_container.hpp:559-573) made deterministic; the daughter is
// written straight to slot n + k, where the reference's merge_buffer would
// append her (:575-599), from the mother's state the pass staged (the pass
// stored the halved mother; a refused request restores her) or, past the
// first DIV_STAGE requests of a sub-chunk, from the mother's slot (halved
// here, M::division).  k is the requests before the group (the per-block
// counts of the pass, summed over at most 64 entries per level) plus the
// requests before it in the group.
// Every mover and every request is independent, so the processing order is
// free.  (3) The last block to finish keeps the books of every run: counters,
// births, the removal decision (update_and_remove_inactive,
// particles_container.hpp:539-557) and the removal's tile layout.
constexpr uint32_t RES_SC = RESOLVE_GROUP_MAX;  // shared arrays; a group is GS <= RES_SC sub-chunks
static_assert(RES_SC <= 256 && 32 % NSUB_MAX == 0, "a group is at most one sub-chunk per thread, of whole tiles");

// Requests of the pass in sub-chunks [0, sc), summed by one wave from the
// block counts (div_l3, div_l2, div_l1: blocks of 2^18, 2^12 and 2^6
// sub-chunks; in a small pool div_l1 alone, 768 at most) and the sub-chunk
// counts of sc's own block of 64.
__device__ __forceinline__ uint32_t request_prefix(const BatchDev& b, uint32_t sc, uint32_t lane) {
  const uint32_t a3 = sc >> 18, a2 = sc >> 12, a1 = sc >> 6;
  uint32_t v = 0;
  for (uint32_t i = lane; i < a3; i += 64) v += b.div_l3[i];
  const uint32_t i2 = (a3 << 6) + lane, i1 = (b.moved ? 0u : a2 << 6) + lane, i0 = (a1 << 6) + lane;
  const uint32_t x2 = i2 < a2 ? b.div_l2[i2] : 0u;
  const uint32_t x0 = i0 < sc ? b.sub_divs[i0] : 0u;
  uint32_t x1 = i1 < a1 ? b.div_l1[i1] : 0u;
  if (b.moved && a1 > 64u)
    for (uint32_t i = i1 + 64u; i < a1; i += 256) {
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) x1 += i + 64 * k < a1 ? b.div_l1[i + 64 * k] : 0u;
    }
  return wave_sum(v + x2 + x1 + x0);
}

// The resolve kernel.  The grid's first tr_blocks blocks (dispatched first:
// their chain is the shorter) are aux blocks: they take the pass's
// contributions and, with `ahead`, transport the liquid
// (and gas) for the next step meanwhile: the two touch disjoint data (the
// records of the two steps are separate tables, the concentrations are
// double-buffered), and the block that keeps the books also lays out the next
// step's tiles, so the next step starts with its particle pass.  K: copies of
// the accumulators, or TAKE_ROWS (a variant each, as the copies' registers cost the others
// occupancy: one copy's taking turns of 8 copies' code made the resolve kernel
// of a 40-run batch 24 us instead of 20).
template <class M, int K>
__global__ void __launch_bounds__(256, M::NV <= 8 ? 4 : 1) k_resolve(BatchDev b, const RunDev* __restrict__ runs,
                                                 const MapDev* __restrict__ maps,
                                                 const uint32_t* __restrict__ tile_off, uint32_t tr_blocks,
                                                 uint32_t ahead) {
  constexpr int NV = M::NV;
  constexpr int NP = M::NP > 0 ? M::NP : 1;
  __shared__ uint32_t s_pre[RES_SC + 1];   // movers: prefix over the group's sub-chunks
  __shared__ uint32_t s_run[RES_SC];
  __shared__ uint32_t s_dpre[RES_SC + 1];  // division requests: prefix over the group's sub-chunks
  __shared__ uint32_t s_p0, s_pr0;         // requests before the group, before its first run
  __shared__ uint32_t s_wm[4], s_wd[4];    // movers and requests of each wave's sub-chunks
  __shared__ uint32_t s_last;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t R = b.R;
  const uint32_t nsub = b.nsub;          // sub-chunks per tile (divides the group)
  const uint32_t sub = TILE / nsub;      // slots per sub-chunk
  const uint32_t T = tile_off[R];
  const uint32_t n_sc = T * nsub;
  // groups of 32 sub-chunks while they fit the grid (one group per block:
  // shorter chains); with more sub-chunks, groups twice as large as long as
  // they still fill the grid, up to RES_SC: a mover takes a chain of
  // dependent loads, and a larger group keeps more of them in flight per
  // block, but one block works through all requests of its group, and where
  // newborns divide together (the end of the run) a large group's requests
  // become a long serial chain.  On the 50 000-compartment lattice at 1e8
  // particles groups of 64, 128 and 256 took 225, 227 and 266 us per step on
  // average.  Threads GS..255 hold no sub-chunk.
  const uint32_t n_res = gridDim.x - tr_blocks;  // blocks of the resolve work
  const bool tr_block = blockIdx.x < tr_blocks;
  const uint32_t rb = tr_block ? 0u : blockIdx.x - tr_blocks;  // index among the resolve blocks
  // A small batch's groups hold 128 sub-chunks of 64 slots, whose movers are done.
  uint32_t GS = nsub > 8 ? RES_SC : 32;
  while (GS < 64 && (n_sc + 2 * GS - 1) / (2 * GS) >= n_res) GS *= 2;
  const uint32_t n_groups = (n_sc + GS - 1) / GS;
  uint32_t ev_run = 0, ev_moves = 0, ev_req = 0;  // movers and requests of the block's groups (thread 0)
  const bool leave_stage = (b.stages & STAGE_LEAVE) != 0;
  if (tr_block) {
    if constexpr (K == TAKE_ROWS)
      sum_rows<M>(b, runs, maps, blockIdx.x, tr_blocks, ahead);
    else
      transport_compartments<M, K>(b, runs, maps, blockIdx.x, tr_blocks, ahead);
  }
  for (uint32_t grp = rb; !tr_block && grp < n_groups; grp += n_res) {
    const uint32_t sc0 = grp * GS;
    {  // the group's sub-chunks, one thread each: block-wide prefix sums
      const uint32_t sc = sc0 + tid;
      uint32_t cm = 0, cd = 0, r = 0;
      if (tid < GS && sc < n_sc) {
        cm = b.sub_moves[sc];
        cd = b.sub_divs[sc];
        r = find_run(tile_off, R, sc / nsub);
      }
      const uint32_t inc = wave_incl_scan(cm, lane);
      const uint32_t incd = wave_incl_scan(cd, lane);
      if (lane == 63) {
        s_wm[wave] = inc;
        s_wd[wave] = incd;
      }
      __syncthreads();
      uint32_t om = 0, od = 0;  // the earlier waves' totals
      for (uint32_t w = 0; w < wave; ++w) {
        om += s_wm[w];
        od += s_wd[w];
      }
      if (tid < GS) {
        s_pre[tid] = om + inc - cm;
        s_dpre[tid] = od + incd - cd;
        s_run[tid] = r;
      }
      if (tid == GS - 1) {
        s_pre[GS] = om + inc;
        s_dpre[GS] = od + incd;
      }
    }
    __syncthreads();
    // ---- movers
    const uint32_t total = s_pre[GS];
    const uint32_t to_move = b.moved ? 0u : total;
    // the step's moves and requests, from the lists: one atomic per block and
    // run, or per sub-chunk where the group holds several runs
    const uint32_t g_last = n_sc - sc0 < GS ? n_sc - sc0 - 1u : GS - 1u;
    if (s_run[0] == s_run[g_last]) {
      if (tid == 0) {
        if (s_run[0] != ev_run) {
          add_pair(&run_shard(b, ev_run)->moves_requests, ev_moves, ev_req);
          ev_run = s_run[0];
          ev_moves = ev_req = 0;
        }
        ev_moves += total;
        ev_req += s_dpre[GS];
      }
    } else if (tid <= g_last) {
      add_pair(&run_shard(b, s_run[tid])->moves_requests, s_pre[tid + 1] - s_pre[tid], s_dpre[tid + 1] - s_dpre[tid]);
    }
    for (uint32_t e = tid; e < to_move; e += blockDim.x) {
      uint32_t lo = 0, hi = GS;  // the sub-chunk j with s_pre[j] <= e < s_pre[j+1]
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_pre[mid] <= e) lo = mid; else hi = mid;
      }
      const uint32_t j = lo;
      const uint32_t sc = sc0 + j;
      const uint32_t t = sc / nsub;
      const uint32_t r = s_run[j];
      const RunDev& rd = runs[r];
      RunState* rs = b.rs + r;
      const uint64_t q = (uint64_t)sc * sub + (e - s_pre[j]);
      const uint32_t ms = b.move_rec[q];
      const uint32_t slot = (t - tile_off[r]) * TILE + (ms & (TILE - 1u));
      const uint64_t g = rd.p_off + slot;
      uint32_t pos = ms >> LIST_POS_SHIFT;
      if (pos == LIST_POS_FAR) pos = b.pos[g];  // a compartment id of 21 bits or more
      const uint32_t step = rs->step;
      const MapDev& mp = maps[rd.map_base + (step / rd.steps_per_map) % rd.n_maps];
      const U4 u = draw4(rd.seed, slot, step, TAG_TRANSPORT, 0u);
      pos = next_place(mp, pos, u01(u.y));
      b.pos[g] = pos;
      bool exits = false;
      if (rd.enable_leave && leave_stage && !(ms & MOVER_INACTIVE)) {
        const double qx = gp(rd.rec)[((size_t)(step & 1u) * rd.n_c + pos) * rd.rec_w + record_terms<M>() + 1];
        if (qx < 1.0 && u01(u.z) > qx) {
          if (rd.probe_exit) {  // its hydraulic age after this step's tick
            const double age = clock_age(b.age_hyd[g], rs->clock_hyd + 1u, b.clk_hyd[g], rd.dt);
            const unsigned long long k = atomicAdd(&rs->probe_exit_n, 1ull);
            if (k < rd.probe_cap) rd.probe_exit[k] = age;
          }
          // no longer Idle: hydraulic age 0, the division clock it stopped at
          b.age_hyd[g] = 0.0;
          b.clk_hyd[g] = rs->clock_div + ((b.stages & STAGE_MODEL) ? 1u : 0u);
          b.status[g] = EXIT;
          exits = true;
        }
      }
      // the exit counter takes one atomic per wave for the run of the wave's
      // first active lane (the wave's movers are in slot order: nearly always
      // one run), and one per exit of any other run; an atomic per exit
      // queued tens of thousands of them on one address per step
      const uint32_t r_lead = __builtin_amdgcn_readfirstlane(r);
      const uint64_t ex_lead = __ballot(exits && r == r_lead);
      if (exits && r != r_lead) add_pair(&run_shard(b, r)->exits_deaths, 1u, 0u);
      if (ex_lead && lane == (uint32_t)__ffsll((long long)ex_lead) - 1u)
        add_pair(&run_shard(b, r_lead)->exits_deaths, (uint32_t)__popcll(ex_lead), 0u);
    }
    // ---- divisions: every request of the group at once, one thread each
    const uint32_t n_req = s_dpre[GS];
    if (n_req) {
      // requests before the group and before the start of its first run
      if (wave == 0) {
        const uint32_t p0 = request_prefix(b, sc0, lane);
        if (lane == 0) s_p0 = p0;
      } else if (wave == 1) {
        const uint32_t s_r = tile_off[s_run[0]] * nsub;
        const uint32_t pr = request_prefix(b, s_r, lane);
        if (lane == 0) s_pr0 = pr;
      }
      __syncthreads();
      for (uint32_t f = tid; f < n_req; f += blockDim.x) {
        uint32_t lo = 0, hi = GS;  // the sub-chunk j with s_dpre[j] <= f < s_dpre[j+1]
        while (hi - lo > 1) {
          const uint32_t mid = (lo + hi) >> 1;
          if (s_dpre[mid] <= f) lo = mid; else hi = mid;
        }
        const uint32_t j = lo;
        const uint32_t sc = sc0 + j;
        const uint32_t t = sc / nsub;
        const uint32_t r = s_run[j];
        const RunDev& rd = runs[r];
        RunState* rs = b.rs + r;
        // rank of the request among the run's requests of the step, in slot order
        const uint32_t first = tile_off[r] * nsub;  // the run's first sub-chunk
        const uint32_t k = first <= sc0 ? s_p0 - s_pr0 + f : f - s_dpre[first - sc0];
        const uint32_t n = rs->n;
        const uint32_t room = rd.cap - n;
        const bool accepted = k < (room < rd.div_cap ? room : rd.div_cap);  // else refused: Overflow
        const uint32_t rk = f - s_dpre[j];  // rank of the request in its sub-chunk
        if (rk >= DIV_STAGE && !accepted) continue;
        const uint64_t q = (uint64_t)sc * sub + rk;
        const uint32_t dw = b.div_rec[q];
        const uint32_t slot = (t - tile_off[r]) * TILE + (dw & (TILE - 1u));
        const uint64_t g = rd.p_off + slot;
        double p[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) p[i] = rd.params[i];
        double x[NV], xd[NV];
        if (rk < DIV_STAGE) {
          // divided by the pass: the mother's slot holds her halved state, the
          // stage her state before division
          const double* stg = b.div_stage + ((uint64_t)sc * DIV_STAGE + rk) * NV;
#pragma unroll
          for (int v = 0; v < NV; ++v) x[v] = stg[v];
          if (!accepted) {  // the mother as she was before the pass divided her
#pragma unroll
            for (int v = 0; v < NV; ++v) b.state[(uint64_t)v * b.P + g] = x[v];
            continue;
          }
        } else {
#pragma unroll
          for (int v = 0; v < NV; ++v) x[v] = b.state[(uint64_t)v * b.P + g];
        }
        // requests come from the model stage: the division clock has ticked
        const uint32_t clk_d = rs->clock_div + 1u;
        if (rd.probe_div) {  // the mother's division age
          const uint32_t w = b.clk_div[g];
          const double age = div_age((w & CLK_FRESH) ? 0.0 : b.age_div[g], clk_d, w, rd.dt);
          const unsigned long long i = atomicAdd(&rs->probe_div_n, 1ull);
          if (i < rd.probe_cap) rd.probe_div[i] = age;
        }
        M::division(p, x, xd, RngKey{rd.seed, slot, rs->step});
        const uint64_t d = rd.p_off + n + k;
#pragma unroll
        for (int v = 0; v < NV; ++v) b.state[(uint64_t)v * b.P + d] = xd[v];
        if (rk >= DIV_STAGE) {  // the mother, divided here
#pragma unroll
          for (int v = 0; v < NV; ++v) b.state[(uint64_t)v * b.P + g] = x[v];
        }
        // the mother's division age restarts (one store: an origin word with
        // CLK_FRESH); the daughter's ages start at 0
        b.clk_div[g] = clk_d | CLK_FRESH;
        uint32_t dpos = dw >> LIST_POS_SHIFT;
        if (dpos == LIST_POS_FAR) dpos = b.div_pos[q];  // a compartment id of 21 bits or more
        b.pos[d] = dpos;
        b.status[d] = IDLE;
        b.age_hyd[d] = 0.0;
        b.clk_hyd[d] = rs->clock_hyd + ((rd.enable_leave && leave_stage) ? 1u : 0u);
        b.clk_div[d] = clk_d | CLK_FRESH;
      }
    }
    __syncthreads();
  }
  if (tid == 0) add_pair(&run_shard(b, ev_run)->moves_requests, ev_moves, ev_req);
  // ---- the last block to finish keeps the books.  The books read, of this
  // kernel's work, only the counter shards, which are updated by atomics:
  // every thread waits for its memory operations to complete before its
  // block counts itself done, and the last block reads the counters with
  // atomics.  No cache writeback is needed (an agent-scope fence per block
  // writes back this XCD's L2 each time: 60 us over a 2048-block grid).
  // Up to RESOLVE_TICKETS blocks count themselves done on one counter (under
  // 1 us of atomics one after another, about what a second level costs); more
  // on RESOLVE_TICKETS sub-counters (block b on b % RESOLVE_TICKETS), a line
  // each, and the last of each on the main counter, so no line takes more than
  // a few dozen atomics; resolve blocks without a group take no
  // part, transport blocks do (the books advance the step count they read).
  const uint32_t nb = n_groups < n_res ? n_groups : n_res;  // resolve blocks with work
  const uint32_t np = nb + tr_blocks;                       // blocks that count themselves done
  if (np == 0) {
    if (blockIdx.x == 0) bookkeep_pass(b, runs, n_sc, ahead != 0);
    return;
  }
  if (!tr_block && rb >= nb) return;
  const uint32_t id = tr_block ? blockIdx.x : tr_blocks + rb;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0) {
    uint32_t last = 0;
    if (np <= RESOLVE_TICKETS) {
      last = atomicAdd(b.ticket, 1u) == np - 1u ? 1u : 0u;
    } else {
      const uint32_t j = id % RESOLVE_TICKETS;
      const uint32_t in_j = (np - j + RESOLVE_TICKETS - 1u) / RESOLVE_TICKETS;  // blocks counting on sub-counter j
      if (atomicAdd(b.ticket + (1u + j) * TICKET_STRIDE, 1u) == in_j - 1u)
        last = atomicAdd(b.ticket, 1u) == RESOLVE_TICKETS - 1u ? 1u : 0u;
    }
    s_last = last;
  }
  __syncthreads();
  if (!s_last) return;
  bookkeep_pass(b, runs, n_sc, ahead != 0);
}

// ------------------------------------------------------------------ layout
// Tile -> run table of the next pass (the tiles of [0, n) of every active run).
template <uint32_t NT>
__device__ void layout_pass(const BatchDev& b) {
  constexpr uint32_t NWV = NT / 64;
  __shared__ uint32_t s_w[NWV];
  __shared__ uint32_t s_carry;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  if (tid == 0) s_carry = 0;
  __syncthreads();
  for (uint32_t r0 = 0; r0 < b.R; r0 += NT) {
    const uint32_t r = r0 + tid;
    uint32_t tiles = 0;
    if (r < b.R) {
      RunState* rs = b.rs + r;
      const RunDev& rd = b.runs[r];
      const uint32_t active = rs->step < rd.step_target ? 1u : 0u;
      rs->active = active;
      tiles = active ? (rs->n + TILE - 1u) / TILE : 0u;
      rs->n_tiles = tiles;
    }
    const uint32_t inc = wave_incl_scan(tiles, lane);
    if (lane == 63) s_w[wave] = inc;
    __syncthreads();
    uint32_t wpre = 0, tot = 0;
    for (uint32_t w = 0; w < NWV; ++w) {
      if (w < wave) wpre += s_w[w];
      tot += s_w[w];
    }
    const uint32_t carry = s_carry;
    if (r < b.R) {
      b.tile_off[r] = carry + wpre + inc - tiles;
      b.rs[r].tile_begin = carry + wpre + inc - tiles;
    }
    __syncthreads();
    if (tid == 0) s_carry = carry + tot;
    __syncthreads();
  }
  if (tid == 0) b.tile_off[b.R] = s_carry;
}


// ------------------------------------------------------------------ properties
// One wave's values of one variable added to an LDS accumulator: lanes `in`
// add x to acc[k].  A wave whose lanes all hold one compartment (particles in
// compartment order) sums first and adds once.
__device__ __forceinline__ void add_by_compartment(double* acc, bool in, uint32_t k, bool one, uint32_t k0,
                                                   uint32_t lane, double x) {
  if (one) {
    double t = in ? x : 0.0;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) t += __shfl_xor(t, d, 64);
    if (lane == 0) atomicAdd(acc + k0, t);
  } else if (in) {
    atomicAdd(acc + k, x);
  }
}

// Per-particle export values of run r (get_properties, post_process.hpp:54-98):
// for every Idle slot the model state and M::mass, row-major [n_var+1][n]
// (zero for inactive slots), and their sums per compartment [n_var+1][n_c].
// values may be null: the sums only.
//
// A block takes a contiguous range of slots and sums them in LDS, then adds
// its nonzero sums to the device's: with one global atomic per particle and
// variable instead, the particles of a compartment, which sit together, queued
// on one address (1.5e6 particles of 10 values in 500 compartments 1187 us, now
// 56 us; 1e5 of 3 in 64 compartments 234 us, now 17 us).  LDS holds `vg` variables of `win`
// compartments; block row y takes one such share (variables y % n_vg, window
// y / n_vg), reading the positions again for each.
constexpr uint32_t EXPORT_THREADS = 512;
constexpr uint32_t EXPORT_LDS = 64 * 1024;      // two blocks per CU
constexpr uint32_t EXPORT_MIN_SLOTS = 4096;     // per block: 8 rounds of its threads
constexpr uint32_t EXPORT_MAX_BLOCKS = 512;
constexpr uint32_t EXPORT_MAX_ROWS = 32768;     // block rows of one launch
template <class M>
__global__ void __launch_bounds__(EXPORT_THREADS) k_properties(BatchDev b, uint32_t r, uint64_t n, double* values,
                                                               double* spatial, uint32_t vg, uint32_t n_vg,
                                                               uint32_t win, uint32_t y0) {
  constexpr uint32_t NV = M::NV, NT = EXPORT_THREADS;
  extern __shared__ double s_acc[];  // [vg][w]
  const RunDev& rd = b.runs[r];
  const uint32_t n_c = rd.n_c;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t y = y0 + blockIdx.y;
  const uint32_t v0 = (y % n_vg) * vg, v1 = v0 + vg < NV + 1u ? v0 + vg : NV + 1u;
  const uint32_t c0 = (y / n_vg) * win, w = n_c - c0 < win ? n_c - c0 : win;
  const bool store = values && y < n_vg;  // the first window's blocks write the values
  const bool has_mass = v1 == NV + 1u;
  const uint64_t per = (n + gridDim.x - 1) / gridDim.x;
  const uint64_t i0 = blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
  for (uint32_t i = tid; i < (v1 - v0) * w; i += NT) s_acc[i] = 0.0;
  __syncthreads();
  double p[M::NP > 0 ? M::NP : 1];
#pragma unroll
  for (int q = 0; q < M::NP; ++q) p[q] = rd.params[q];
  for (uint64_t base = i0; base < i1; base += NT) {
    const uint64_t s = base + tid;
    const bool valid = s < i1;
    const uint64_t g = rd.p_off + (valid ? s : i0);
    const bool live = valid && b.status[g] == IDLE;
    const uint32_t k = b.pos[g] - c0;  // wraps above the window when below it
    const bool in = live && k < w;
    const uint64_t mask = __ballot(in);
    const uint32_t lead = mask ? (uint32_t)__ffsll((long long)mask) - 1u : 0u;
    const uint32_t k0 = (uint32_t)__shfl((int)k, (int)lead, 64);
    if (!mask && !store) continue;  // none of the wave's particles in this window
    const bool one = mask && __ballot(in && k == k0) == mask;
    const bool need = live && (in || store);  // a particle's values are read in its own window only
    double x[NV];
#pragma unroll
    for (uint32_t v = 0; v < NV; ++v)
      x[v] = (has_mass || (v >= v0 && v < v1)) && need ? b.state[(uint64_t)v * b.P + g] : 0.0;
#pragma unroll
    for (uint32_t v = 0; v < NV; ++v) {
      if (v < v0 || v >= v1) continue;
      if (store && valid) values[(uint64_t)v * n + s] = x[v];
      add_by_compartment(s_acc + (v - v0) * w, in, k, one, k0, lane, x[v]);
    }
    if (has_mass) {
      const double m = need ? M::mass(p, x) : 0.0;
      if (store && valid) values[(uint64_t)NV * n + s] = m;
      add_by_compartment(s_acc + (NV - v0) * w, in, k, one, k0, lane, m);
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < (v1 - v0) * w; i += NT) {
    const double t = s_acc[i];
    if (t != 0.0) {
      const uint32_t q = i / w;
      unsafeAtomicAdd(spatial + (size_t)(v0 + q) * n_c + c0 + (i - q * w), t);
    }
  }
}

// ------------------------------------------------------------------ launchers
template <class M, int BLK, bool PRIV, bool PROBE, bool WIN, bool LV>
static void launch_particle_t(const BatchDev& b, int grid, size_t lds, hipStream_t s) {
  hipLaunchKernelGGL((k_particle<M, BLK, M::NL, lane_interleave(M::NL), PRIV, PROBE, WIN, LV>), dim3(grid), dim3(BLK), lds, s,
                     b, b.runs, (const RunState*)b.rs, (const uint32_t*)b.tile_off);
}

// The variants: direct global atomics (256 threads); an LDS accumulator of
// whole runs or of a compartment window (256/512/1024 both); each with
// and without the leaving-flow work; and the 256-thread probe variants of
// each accumulator kind (with it).
template <class M, bool LV>
static const void* kernel_ptr_lv(int blk, bool priv, bool win) {
  if (!priv) return blk == 256 ? (const void*)&k_particle<M, 256, M::NL, lane_interleave(M::NL), false, false, false, LV> : nullptr;
  if (win) {
    if (blk == 256) return (const void*)&k_particle<M, 256, M::NL, lane_interleave(M::NL), true, false, true, LV>;
    if (blk == 512) return (const void*)&k_particle<M, 512, M::NL, lane_interleave(M::NL), true, false, true, LV>;
    if (blk == 1024) return (const void*)&k_particle<M, 1024, M::NL, lane_interleave(M::NL), true, false, true, LV>;
    return nullptr;
  }
  if (blk == 256) return (const void*)&k_particle<M, 256, M::NL, lane_interleave(M::NL), true, false, false, LV>;
  if (blk == 512) return (const void*)&k_particle<M, 512, M::NL, lane_interleave(M::NL), true, false, false, LV>;
  if (blk == 1024) return (const void*)&k_particle<M, 1024, M::NL, lane_interleave(M::NL), true, false, false, LV>;
  return nullptr;
}
template <class M, bool LV>
static const void* small_ptr(int blk) {
  return blk == 256   ? (const void*)&k_particle_small<M, 256, LV>
         : blk == 512 ? (const void*)&k_particle_small<M, 512, LV>
                      : (const void*)&k_particle_small<M, 1024, LV>;
}
template <class M, bool LV>
static void launch_small(const BatchDev& b, const ParticleLaunch& L, hipStream_t s) {
  const uint32_t* off = b.tile_off;
  const RunState* rs = b.rs;
  if (L.block == 256)
    hipLaunchKernelGGL((k_particle_small<M, 256, LV>), dim3(L.grid), dim3(256), L.lds, s, b, b.runs, rs, b.maps, off);
  else if (L.block == 512)
    hipLaunchKernelGGL((k_particle_small<M, 512, LV>), dim3(L.grid), dim3(512), L.lds, s, b, b.runs, rs, b.maps, off);
  else
    hipLaunchKernelGGL((k_particle_small<M, 1024, LV>), dim3(L.grid), dim3(1024), L.lds, s, b, b.runs, rs, b.maps, off);
}
template <class M>
static const void* kernel_ptr_t(int blk, bool priv, bool probe, bool win, bool leave, bool small) {
  if (small) return leave ? small_ptr<M, true>(blk) : small_ptr<M, false>(blk);
  if (probe) {
    if (!priv) return (const void*)&k_particle<M, 256, M::NL, lane_interleave(M::NL), false, true, false, true>;
    return win ? (const void*)&k_particle<M, 256, M::NL, lane_interleave(M::NL), true, true, true, true>
               : (const void*)&k_particle<M, 256, M::NL, lane_interleave(M::NL), true, true, false, true>;
  }
  return leave ? kernel_ptr_lv<M, true>(blk, priv, win) : kernel_ptr_lv<M, false>(blk, priv, win);
}

// Runs with probes take a 256-thread variant that records exit and division
// ages; the atomics it needs (with returned values) are kept out of the
// production variants, where they would make every wait for a load in the
// tile loop a wait for all outstanding memory operations.
template <class M, bool LV>
static void launch_lv(const BatchDev& b, const ParticleLaunch& L, hipStream_t s) {
  if (!L.priv) {
    launch_particle_t<M, 256, false, false, false, LV>(b, L.grid, 0, s);
  } else if (L.win) {
    if (L.block == 1024)
      launch_particle_t<M, 1024, true, false, true, LV>(b, L.grid, L.lds, s);
    else if (L.block == 512)
      launch_particle_t<M, 512, true, false, true, LV>(b, L.grid, L.lds, s);
    else
      launch_particle_t<M, 256, true, false, true, LV>(b, L.grid, L.lds, s);
  } else if (L.block == 256) {
    launch_particle_t<M, 256, true, false, false, LV>(b, L.grid, L.lds, s);
  } else if (L.block == 512) {
    launch_particle_t<M, 512, true, false, false, LV>(b, L.grid, L.lds, s);
  } else {
    launch_particle_t<M, 1024, true, false, false, LV>(b, L.grid, L.lds, s);
  }
}
template <class M>
static void launch_t(const BatchDev& b, const ParticleLaunch& L, hipStream_t s) {
  if (b.moved) {
    if (L.leave)
      launch_small<M, true>(b, L, s);
    else
      launch_small<M, false>(b, L, s);
  } else if (L.probe) {
    if (!L.priv)
      launch_particle_t<M, 256, false, true, false, true>(b, L.grid, 0, s);
    else if (L.win)
      launch_particle_t<M, 256, true, true, true, true>(b, L.grid, L.lds, s);
    else
      launch_particle_t<M, 256, true, true, false, true>(b, L.grid, L.lds, s);
  } else if (L.leave) {
    launch_lv<M, true>(b, L, s);
  } else {
    launch_lv<M, false>(b, L, s);
  }
}

template <class M>
void transport_t(const BatchDev& b, int grid, hipStream_t s) {
  hipLaunchKernelGGL(k_transport<M>, dim3(grid), dim3(256), 0, s, b, b.runs, b.maps);
}
template <class M, int K>
static void launch_resolve(const BatchDev& b, int grid, uint32_t aux, bool ahead, hipStream_t s) {
  hipLaunchKernelGGL((k_resolve<M, K>), dim3(grid + (int)aux), dim3(256), 0, s, b, b.runs, b.maps,
                     (const uint32_t*)b.tile_off, aux, ahead ? 1u : 0u);
}
template <class M>
void resolve_t(const BatchDev& b, int grid, uint32_t aux, bool ahead, hipStream_t s) {
  if (b.rows)
    launch_resolve<M, TAKE_ROWS>(b, grid, aux, ahead, s);
  else if (b.n_copies == 1)
    launch_resolve<M, 1>(b, grid, aux, ahead, s);
  else
    launch_resolve<M, (int)run_copies(M::NS)>(b, grid, aux, ahead, s);
}
template <class M>
const void* resolve_kernel_t(const BatchDev& b) {
  return b.rows            ? (const void*)&k_resolve<M, TAKE_ROWS>
         : b.n_copies == 1 ? (const void*)&k_resolve<M, 1>
                           : (const void*)&k_resolve<M, (int)run_copies(M::NS)>;
}
template <class M>
void properties_t(const BatchDev& b, uint32_t run, uint64_t n, uint32_t n_c, double* values, double* spatial,
                  hipStream_t s) {
  constexpr uint32_t NV1 = M::NV + 1;
  const uint32_t cells = EXPORT_LDS / sizeof(double);
  const uint32_t win = n_c < cells ? n_c : cells;                      // compartments in LDS
  const uint32_t vg = cells / win < NV1 ? cells / win : NV1;           // variables in LDS
  const uint32_t n_vg = (NV1 + vg - 1) / vg, n_win = (uint32_t)(((uint64_t)n_c + win - 1) / win);
  const uint64_t want = (n + EXPORT_MIN_SLOTS - 1) / EXPORT_MIN_SLOTS;
  const uint32_t grid = (uint32_t)(want < EXPORT_MAX_BLOCKS ? (want ? want : 1) : EXPORT_MAX_BLOCKS);
  for (uint32_t y = 0; y < n_vg * n_win; y += EXPORT_MAX_ROWS)
    hipLaunchKernelGGL(k_properties<M>, dim3(grid, std::min(n_vg * n_win - y, EXPORT_MAX_ROWS)), dim3(EXPORT_THREADS),
                       (size_t)vg * win * sizeof(double), s, b, run, n, values, spatial, vg, n_vg, win, y);
}

// The launchers of model M's kernels.
template <class M>
ModelOps model_ops() {
  static_assert(vars_declared_soundly<M>(),
                "a model that declares READS declares WRITES too, and each has a bit per state variable at most");
  return ModelOps{&transport_t<M>, &launch_t<M>, &kernel_ptr_t<M>, &resolve_t<M>, &resolve_kernel_t<M>,
                  &properties_t<M>};
}

}  // namespace mcst
