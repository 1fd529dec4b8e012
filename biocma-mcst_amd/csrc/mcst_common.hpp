// mcst_common.hpp -- layout of the device-resident batch of runs.
//
// A batch ("engine") holds R independent runs that share one particle model.
// Every run owns a region [p_off, p_off + cap) of the batch-wide particle SoA
// arrays, its own compartment network (flowmaps), liquid state and counters.
// Particles are processed in tiles of TILE consecutive slots of one run; the
// tile -> run map is a prefix table rebuilt on the device after every step,
// so a step never needs the host to know particle counts.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcst {

constexpr uint32_t BLOCK = 256;            // threads per particle block (4 wave64)
constexpr uint32_t PPT = 4;                // particles per thread per tile
constexpr uint32_t TILE = BLOCK * PPT;     // 1024 slots per tile (the reference's 1024 particles/team)
// Particle pass layout: with 4 slots per lane a lane's slots lie 64 apart
// (every access of a wave one contiguous 64-slot run); with 2 they are
// consecutive (16-byte accesses per lane).  Measured on MI355X: 64 apart is
// 3 % faster at 4 slots per lane (pair-wise 16-byte accesses, half the load
// instructions, were slower), consecutive 4 % faster at 2.
constexpr bool lane_interleave(int nl) { return nl >= 4; }
constexpr uint32_t NSUB_MAX = TILE / 64;   // sub-chunks (the pass's unit of work) per tile: TILE / (64 * M::NL), 16 in
                                           // a small batch's pass
constexpr uint32_t WAVES = BLOCK / 64;
constexpr uint32_t RESOLVE_GROUP_MAX = 128; // sub-chunks per group of the resolve kernel: 32 or 64, 128 of 64 slots
constexpr uint32_t RESOLVE_TICKETS = 64;    // sub-counters of the resolve kernel's done-count
constexpr uint32_t TICKET_STRIDE = 32;      // words between two of those counters (a line each)
constexpr uint32_t REMOVE_RUN_TILES = 512;  // largest capacity at which one block removes a run's inactive slots
constexpr uint32_t DIV_STAGE = 16;          // division requests per sub-chunk divided in the particle pass
constexpr int MAX_PARAMS = 16;
constexpr int MAX_VAR = 16;
constexpr int MAX_SPECIES = 8;

// Particle status byte (apps/libs/mc/public/mc/alias.hpp:124-130).
enum Status : uint8_t { IDLE = 0, DIVISION = 1, EXIT = 2, DEAD = 3 };
// An entry of the pass's lists (u32): the slot within its tile (bits 0-9),
// MOVER_INACTIVE in a mover entry for a slot that moves but does not leave
// (not Idle: no exit test), and a compartment (bits 11-31): a mover's before
// the move, a division request's (the newborn's); LIST_POS_FAR for an id that
// does not fit.  A mover's compartment is then read from the slot's position
// (only the mover's own thread writes it, after the read), a request's from
// div_pos.
constexpr uint32_t MOVER_INACTIVE = 1u << 10;
constexpr uint32_t LIST_POS_SHIFT = 11;
constexpr uint32_t LIST_POS_FAR = 0xFFFFFFFFu >> LIST_POS_SHIFT;
static_assert(TILE <= MOVER_INACTIVE, "a tile-local slot fits below the flag");

// Largest pool, in tiles, that the small batch's particle pass serves.  A step
// with the pipelined pass and with this one: 500 000 particles of 2, 3 and 8
// states (the last with 2 slots per lane) 25, 22.6, 32.9 us and 24, 22.2, 30.3;
// 1e6 29.4, 28.1, 42.0 and 30.6, 28.0, 41.0: the line.  Where the pipelined pass
// holds many states of 4 slots per lane its registers leave it few waves and the
// line lies further up: 6 states 1e6 34.5 and 34.7, 2e6 51.0 and 47.4, 3e6 64.2
// and 59.7, 5e6 91.9 and 91.9; 9 states (half as many again after their first
// steps) 1e6 50.6 and 47.0, 2e6 77.6 and 70-80, 3e6 107 and 138, which a pool of
// these tiles holds only when it is full (its slots are what is known here, and
// a run has twice its particles by default).
constexpr uint32_t small_tiles(int nv, int nl) { return nv * nl >= 24 ? 3072u : 1024u; }

// Stage mask of one step (values shared with the C ABI).
enum Stage : uint32_t {
  STAGE_TRANSPORT = 1u,
  STAGE_MODEL = 2u,
  STAGE_CONTRIB = 4u,
  STAGE_MOVE = 8u,
  STAGE_LEAVE = 16u,
  STAGE_REMOVE = 32u,
  STAGE_ALL = 63u
};

// Philox counter purpose tags (third counter word = tag << 16 | block).
enum RngTag : uint32_t { TAG_TRANSPORT = 0, TAG_UPDATE = 1, TAG_DIVISION = 2, TAG_INIT = 3 };

// Cumulative per-run counters (order shared with the C ABI).
enum Counter : int {
  C_STEPS = 0,
  C_BIRTHS,
  C_EXITS,
  C_DEATHS,
  C_MOVES,
  C_OVERFLOW,
  C_COMPACTIONS,
  C_N,
  C_INACTIVE,
  C_PROCESSED,  // particle-steps: Idle particles that entered a pass
  C_COUNT
};

// Tables of one flowmap of one run (device pointers).
struct MapDev {
  const double* p_move;     // [n_c]  dt*Q_out/V
  const double* q_exit;     // [n_c]  exp(-dt*Q_leave/V) at outlets, 2.0 elsewhere
  const double* cdf;        // [n_c][m] cumulative neighbour probabilities
  const uint32_t* nbr;      // [n_c][m] neighbour ids (padding repeats the last)
  const uint32_t* col_ptr;  // [n_c+1] transport matrix by destination column
  const uint32_t* src;      // [nnz]   source compartment of each column entry
  const double* val;        // [nnz]   F(i,j) off-diagonal, -Q_out(j) on the diagonal
  const double* inv_v;      // [n_c]
  const double* vol;        // [n_c]   liquid volumes V
  // gas side of the flowmap in a two-phase run (null otherwise)
  const uint32_t* g_col_ptr;  // [n_c+1] gas transport matrix by destination column
  const uint32_t* g_src;
  const double* g_val;
  const double* g_inv_v;    // [n_c]   1 / gas volume
  const double* g_kla;      // [n_s][n_c] kLa of the flowmap
  // rows of at most MOVE_ROW_M neighbours (m <= MOVE_ROW_M), else null: one
  // 64-byte record per compartment, cdf columns 0..4 (2.0 from column m-1
  // on) then neighbours 0..5 as u32 (the last repeated), so that a mover
  // reads one line where cdf and nbr take two
  const uint32_t* move_row;
  uint32_t m;
  uint32_t pad;
};
constexpr uint32_t MOVE_ROW_M = 6;

// Steps of time-dependent feeds the host prepares at once at most: their flows
// depend on the step number alone.  (Prepared before every step, they cost a wait for
// the stream and a copy each time, and kept the next step's transport out of
// the resolve kernel: 20 011 particles of a two-phase column 50 us a step, now
// 25.)
constexpr uint32_t VF_ROWS = 256;
// Rows to prepare from `step` on, for a call with `left` steps to take: those
// steps, or twice the rows of the last time, so that single steps are prepared
// in ever longer blocks and nobody pays for more than twice what they use (a row
// of many outlets is as many exponentials); none past the run's last step.
constexpr uint32_t feed_rows(uint32_t step, uint32_t target, uint64_t left, uint32_t last) {
  const uint64_t want = left > 2ull * last ? left : 2ull * last;
  const uint64_t most = target - step < VF_ROWS ? target - step : VF_ROWS;
  return (uint32_t)(want < most ? want : most);
}

// vf_src_s / vf_sink_k entries that belong to the gas phase
constexpr uint32_t VF_GAS = 0x80000000u;

// Immutable description of one run.
struct RunDev {
  uint64_t p_off;           // first slot of the run in the batch arrays
  uint64_t seed;
  double dt;
  double weight;            // numerical weight of every particle (unit.cpp:232-257)
  double ratio;             // removal threshold ratio (particles_container.hpp:548-551)
  uint64_t min_removal;
  double params[MAX_PARAMS];
  double* C[2];             // [n_s][n_c] concentrations, ping-pong by step parity
  double* m;                // [n_s][n_c] liquid mass
  double* S;                // [n_s][n_c] particle sources of the last step, as the host may read them
  double* Sp;               // [copies][n_s][n_c] the pass adds to these; zero but between a pass and
                            // its resolve kernel
  const double* F;          // [n_s][n_c] constant feed sources
  const double* sink;       // [n_c]      outlet flow per compartment
  const double* kla;        // [n_s][n_c] gas-liquid transfer coefficient (null: no transfer)
  const double* cstar;      // [n_s][n_c] saturation concentration set by the gas phase
  // gas phase of a two-phase run (Cg[0] null otherwise): concentrations
  // (ping-pong like C), mass, constant gas feed sources, gas outlet flows,
  // Henry constants (C* = H C_gas)
  double* Cg[2];
  double* mg;
  const double* Fg;         // [n_s][n_c]
  const double* sink_g;     // [n_c]
  double henry[MAX_SPECIES];
  // time-dependent (linear, exponential) feeds: row step % VF_ROWS of vf_q
  // holds a step's flows, then the exit thresholds of the outlets they lead
  // (vf_w values, written by the host ahead of the steps); sources and sinks by
  // compartment (CSR); vx_slot[j] >= 0 selects the threshold of outlet j from
  // the row's n_vf + slot
  const double* vf_q;
  const uint32_t* vf_src_ptr;  // [n_c+1]
  const uint32_t* vf_src_k;    // feed (index into vf_q) of each source entry
  const uint32_t* vf_src_s;    // its species (| VF_GAS for a gas feed)
  const double* vf_src_c;      // its concentration
  const uint32_t* vf_sink_ptr; // [n_c+1]
  const uint32_t* vf_sink_k;   // (| VF_GAS for a gas outlet)
  const int32_t* vx_slot;      // [n_c]
  uint32_t n_vf, vf_w;
  double* rec;              // [2][n_c][rec_w] per-compartment record read by the particle pass, the
                            // table of step k at k & 1 (the next step's transport may write its
                            // table while this step's resolve kernel reads the other)
  double* probe_exit;       // exit ages (residence times), may be null
  double* probe_div;        // division ages, may be null
  uint32_t cap;             // slots reserved for the run
  uint32_t n_c;
  uint32_t n_s;
  uint32_t rec_w;           // record stride in doubles: {M::record(C)_0..NR-1, p_move, q_exit, pad}
  uint32_t enable_move;     // n_c > 1                        (kernels.hpp:54-55)
  uint32_t enable_leave;    // at least one leaving flow      (kernels.hpp:56)
  uint32_t n_maps;
  uint32_t steps_per_map;
  uint32_t map_base;        // index of the run's first MapDev
  uint32_t div_cap;         // newborns per step at most (the reference's division buffer)
  uint32_t comp_off;        // first compartment of the run in the batch transport space
  uint32_t probe_cap;
  uint32_t step_target;     // the run stops stepping at this step count
};

// Mutable per-run state, updated by the device every step.
struct RunState {
  uint32_t n;               // used slots (Idle + inactive)
  uint32_t n_end;           // slots after the last step's newborns joined: the removal's range
  uint32_t n_keep;          // slots the removal keeps (n_end - inactive)
  uint32_t inactive;        // Exit/Dead slots below n
  uint32_t step;
  uint32_t compact;         // removal requested by the last bookkeeping
  uint32_t births;          // newborns of the last step
  uint32_t tile_begin;      // first global tile of the run in the current layout
  uint32_t n_tiles;         // tiles of the run in the current layout
  uint32_t active;          // 1 while step < step_target
  // age clocks: the steps so far in which the run's Idle particles aged
  // (division age: steps with the model stage; hydraulic age: steps with the
  // leave stage while the run has a leaving flow)
  uint32_t clock_div;
  uint32_t clock_hyd;
  uint32_t pad;
  unsigned long long counters[C_COUNT];
  unsigned long long probe_exit_n, probe_div_n;
};

// One of a run's counter shards: the events of the step under way, added by
// the blocks whose index falls on the shard and taken (and cleared) by the
// books.  A line each: atomics on one line are served one after another, about
// 10 ns each across the XCDs, so 2700 waves adding their moves and particles
// to two counters of one line took 25 us of a 345 679-particle pass of 41 us.
// Particles processed need no count: they are the run's Idle slots, n -
// inactive.
struct RunShard {
  unsigned long long moves_requests;  // moves in the low 32 bits, division requests in the high
  unsigned long long exits_deaths;    // exits low, deaths high
  unsigned long long pad[14];
};
// Shards per run: fewer where many runs spread the atomics anyway (a power of
// two, at most 16: the books sum a run's shards within 16 lanes).
constexpr uint32_t run_shards(uint32_t runs) { return runs <= 16 ? 16u : runs <= 256 ? 4u : 1u; }

// Everything a step's kernels receive.
struct BatchDev {
  // particles, batch-wide SoA
  uint32_t* pos;
  uint8_t* status;
  double* state;            // [n_var][P]
  // ages: an Idle slot's age is age_x + (clock_x - clk_x) * dt, with clock_x
  // its run's age clock, so a step writes them only when they restart;
  // a slot that is not Idle has hydraulic age age_hyd and division age
  // age_div + (clk_hyd - clk_div) * dt (clk_hyd holds the division clock at
  // which it stopped being Idle).  clk_div is an origin word (div_age): a
  // restart at 0 sets CLK_FRESH there and leaves age_div unread.
  double* age_hyd;
  double* age_div;
  uint32_t* clk_hyd;
  uint32_t* clk_div;
  uint64_t P;               // total slots
  // division requests of the pass per block of 2^6, 2^12 and 2^18
  // sub-chunks (global sub-chunk index of the layout); with sub_divs they
  // give the requests before any sub-chunk in 64 terms per level (128 at the
  // top level for pools of more than 2^31 slots)
  uint32_t* div_l1;
  uint32_t* div_l2;
  uint32_t* div_l3;
  uint32_t* ticket;         // [2 + RESOLVE_TICKETS][TICKET_STRIDE] resolve blocks that are done (the last keeps the books);
                            // the last row: the removal's counting blocks
  uint32_t* rm_tile_off;    // [R+1] removal layout: first global tile of each run's [0, n_end)
  // per-tile bookkeeping of the removal
  unsigned long long* tile_cnt;  // [T_max] gaps (low 32 bits) and fillers (high) of each tile
  unsigned long long* tile_pre;  // [T_max+1] their sums before each tile
  uint32_t* tile_off;       // [R+1] first global tile of each run in the step's layout
  // lists of the particle pass, one segment of TILE/nsub entries per sub-chunk
  uint32_t* move_rec;       // [T_max*TILE] particles leaving their compartment, one entry each
                            // (slot, flag and compartment in one word, so that the few movers of a
                            // sub-chunk share one line)
  uint32_t* div_rec;        // [T_max*TILE] division requests, one entry each
  uint32_t* div_pos;        // [T_max*TILE] their compartment (read for ids past the entry's field only)
  double* div_stage;        // [T_max*nsub*DIV_STAGE][n_var] the first DIV_STAGE requests of each
                            // sub-chunk, divided in the pass: the mother's state before division
                            // (to restore her if the request is refused)
  uint32_t* sub_moves;      // [T_max*nsub] entries of each sub-chunk's mover segment
  uint32_t* sub_divs;       // [T_max*nsub] entries of each sub-chunk's request segment
  // runs
  const RunDev* runs;
  RunState* rs;
  RunShard* shards;         // [R][n_shard]
  const MapDev* maps;
  const uint32_t* comp_off; // [R+1] 64-compartment chunks before each run (none of a run off the device)
  uint32_t R;
  uint32_t n_shard;
  uint32_t n_chunk_total;
  uint32_t ns_max;          // largest species count of the batch
  uint32_t T_max;
  uint32_t nsub;            // sub-chunks per tile of the particle pass in use
  uint32_t moved;           // the small batch's pass is in use: it moves its movers itself
  uint32_t tile_group;      // particle pass: groups per block turn at most (0: one range per block)
  uint32_t acc_w;           // particle pass: compartments per LDS contribution window (PRIV)
  uint32_t stages;
  // copies of each run's contribution accumulator in use (1 or run_copies): block
  // k of the particle pass adds to copy k % n_copies, and the resolve kernel
  // sums the copies
  uint32_t n_copies;
  // contribution rows (one live run whose whole [n_s][n_c] accumulator fits
  // LDS): a copy for every block of the particle pass (n_copies is a power of two
  // past them), so that each holds one block's sums, and the resolve kernel adds
  // these `rows` copies in a fixed order; 0: the copies above
  uint32_t rows;
  // the next step's tile_off, written by the books while blocks of the step may yet read tile_off
  uint32_t* tile_off_next;
};

// A pass ends with every block adding its LDS accumulator to the run's, a
// line's adds one after another; blocks are dealt to the XCDs in turn, so with
// 8 copies an XCD's blocks queue on their own lines only.  338 blocks of a
// 345 679-particle pass took 16.2 us with one copy, 13.9 with 4 and 12.2 with 8,
// 512 blocks of the 1e7-particle pass 126, 123 and 123 (the resolve kernel 11.0,
// 10.8 and 13.9 us: 8 copies of 2 species spill).  Copies cost their sum and their clearing, so
// they are kept to batches of at most S_COPY_ENTRIES values in all (the
// blocks of a larger batch or network meet on fewer of its lines).
constexpr uint32_t S_COPIES = 8, S_COPY_ENTRIES = 16384;
// ... of a model with ns species: fewer where the thread that sums a
// compartment's copies would hold more than 16 of them in registers
constexpr uint32_t run_copies(int ns) { return ns == 1 ? S_COPIES : ns == 2 ? S_COPIES / 2 : S_COPIES / 4; }

// The particle pass's compartment window: `win` of n_c compartments from the
// returned one on, centred on compartment c0 as far as the network reaches.
__host__ __device__ inline uint32_t window_at(uint32_t c0, uint32_t win, uint32_t n_c) {
  const uint32_t lo = c0 > win / 2 ? c0 - win / 2 : 0u;
  return lo + win <= n_c ? lo : n_c - win;
}
// ... at a turn that starts in c0, from the window at w0: centred anew once c0
// has left the window's middle half.  At the network's ends that may be where
// it is: a window that cannot move is not flushed (it was, in every turn that
// started near an end: the pass of 2e6 cells of 4 species at random places of
// 5500 compartments, one window of 5088, took 155 us, now 141; of 5150, 132 and
// 115)
__host__ __device__ inline uint32_t window_next(uint32_t c0, uint32_t w0, uint32_t win, uint32_t n_c) {
  return c0 - (w0 + win / 4) >= win / 2 ? window_at(c0, win, n_c) : w0;  // wraps when below
}

// Age of a slot from its base age, its origin on the age clock and the
// clock (the expression the host's conversion uses too).
__host__ __device__ inline double clock_age(double base, uint32_t clock, uint32_t origin, double dt) {
  return base + (double)(clock - origin) * dt;
}

// A division-age origin word: the origin on the division clock in its low 31
// bits (the age counts (clock - origin) mod 2^31 steps), and CLK_FRESH when
// the age restarted there from 0, so that a restart is one store (age_div is
// then not read).  Equal to clock_age for ages of fewer than 2^31 steps.
constexpr uint32_t CLK_FRESH = 1u << 31;
__host__ __device__ inline double div_age(double base, uint32_t clock, uint32_t word, double dt) {
  return ((word & CLK_FRESH) ? 0.0 : base) + (double)((clock - word) & ~CLK_FRESH) * dt;
}

}  // namespace mcst
