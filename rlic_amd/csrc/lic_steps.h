// Streamline step loops shared by the single-field and the batched kernels.
#pragma once

#include "lic_device.h"

namespace rlic {

// Kernel weights are read through a copy padded with kKernelPad zeros on
// each side, so a group of 8 taps can be loaded without bounds checks.
constexpr int32_t kKernelPad = 8;

// Move-code layout: a direction's steps are cut into chunks of 32 steps
// (4 words of 8 four-bit codes, the first step of a word in its top nibble:
// move_code); chunk c of pixel p (row-major index
// i * nx + j) is the 16-byte vector codes4[(c0 + c) * ny * nx + p], so one
// lane moves 32 steps of codes with one load or store, and the tracing and
// replay kernels may tile the image differently.
constexpr int32_t kChunkSteps = 32;

__host__ __device__ inline int32_t chunks_of(int32_t nsteps) {
  return (nsteps + kChunkSteps - 1) / kChunkSteps;
}

// One streamline direction of one pixel (src/lib.rs:304-362), starting from
// the vector (pu, pv) of the start cell, already loaded.  The position `row`
// is the cell's slot (cell_slot).  Returns the updated accumulator.  With REC, writes the move code of every step.
//
// The step is written without divergent branches: a lane whose line has
// ended (NaN vector) keeps executing with its position frozen and its
// accumulator untouched, and a lane with a zero vector keeps its position
// (src/lib.rs:242-244); steps run in groups of 8 (one code word, one batch
// of 8 weights) and a wave leaves the loop once all its lines have ended.
// With `short_path` (the field's velocities are not wide, velocity_wide),
// whole groups of the branchless rule run as fast_group.
//
// The cells form a guarded array (guarded_cells: (ny + 2) x (nx + 2)
// with a ring of guard cells around the image).
// A guard cell holds the values of the cell that a step onto it ends on by
// the boundary rule (src/lib.rs:83-95: the edge cell itself for a closed
// side, the opposite edge cell for a periodic one) and, in its pad slot,
// the jump in cells to that cell (0 in image cells): a step is one add of
// +-1 cell or +-1 row, the gather, and one shifted add of the jump.
//
// PAIRS: the array may be in row pairs (or plain rows, as `sg` says); without,
// it is in plain rows.
//
// LANE_DIR: the direction is the lane's own (forward where fwd_lane), one
// body for both (the paired trace, lic_trace_pair); FORWARD then names the
// weights the accumulator takes (the backward lanes' sum is not used).
// `sink(s, x)` sees each step's texture value (possibly more than once: the
// last call for a step counts), and `*live_steps`, if not null, receives the
// number of steps taken before the line ended.
struct NoSink {
  template <typename T>
  __device__ __forceinline__ void operator()(int32_t, T) const {}
};

// Eight steps of the default step rule on the short path: what trace_direction
// does in its full group, with the two divisions of a step replaced by one.
//
// The full rule divides twice (tx = n_x / |u|, ty = n_y / |v|, with n the
// remaining fraction of the cell along the axis), compares, and then uses
// only the smaller quotient.  Here the axis is picked by the sign of
// e = n_x |v| - n_y |u| (one product and one fused multiply-add), and only the
// picked quotient is formed.  Besides the division saved, the next cell's
// address no longer waits for a quotient: the gather is issued first and the
// division runs while it is in flight.
//
// Exactness.  The caller guarantees that every nonzero finite velocity of
// the field lies within VelocityRange (velocity_wide), so the products
// neither overflow nor lose bits to underflow.  With |e| > near_tie n_y |u|
// the two exact quotients differ by more than near_tie / 2 relatively, so
// their roundings compare as the exact ones do; otherwise (an exact or a near tie, both components zero, a NaN component:
// every one of them fails the comparison) the lane is reported.  The
// quotient is quotient_rn's, which needs a numerator that is zero or not tiny
// (numerator_key_min): smaller ones are reported too.  A time of zero (n = 0)
// compares below the other one only if that does not underflow to zero: in
// float, lanes with |e| below kProductMin are reported (0.7% of a trace); in
// double it cannot (VelocityRange).  A chunk in which a moving
// lane is reported is thrown away and done again by the full rule, so the
// results are the full rule's bit for bit.  A reported lane may pick a wrong
// axis until the chunk ends, but a step always leads from an image cell to
// an image cell or a guard cell and from there to an image cell, so its
// gathers stay inside the guarded array.
//
// Lanes that do not move (line ended, or a zero vector) take part with a
// zero step; the caller restores their sums and codes.  Returns the lane
// mask of reported lanes.
//
// What bounds it: VALU issue.  On gfx950 a wave instruction occupies its SIMD
// for 2 cycles (float add, multiply, fma; 32-bit add, subtract, and/or/xor,
// bitop3, arithmetic shift right) or 4 (compares, v_cndmask, min/max,
// shift-or, bfi, add with carry, every double operation), 8 for v_rcp_f32 and
// 16 for v_rcp_f64 (measured with streams of one instruction).  So choices are
// made with lane masks in VGPRs (sign words and v_bitop3) rather than with
// compares and v_cndmask.  A step is about 36 VALU instructions, 90 issue
// cycles per wave (the full rule's 57 took about 170); with that the L1 gather
// path is as busy (TD 97%, 29-34 cycles per wave gather on the CU's one
// path).  Trace launches, full rule in plain rows -> with this alone -> and
// row pairs (cell_slot): 4096^2 float L=129 with the record 2.47 -> 1.92 ->
// 1.86 ms, 2111x1500 float with holes L=201 775 -> 684 -> 603 us, 1021x1537
// double L=151 499 -> 447 -> 430 us, 16384^2 float polarization L=257 (plain
// rows) 72.2 -> 55.0 -> 54.5 ms, 8192^2 double polarization 30.1 -> 26.4 ->
// 26.4 ms, 256^2 double L=65 (paired lanes) 22.6 -> 19.3 -> 19.9 us.
template <typename T, bool FMA, int POL, bool FORWARD, int REC, bool BUF, bool PAIRS,
          bool LANE_DIR, typename Sink>
__device__ __forceinline__ uint64_t fast_group(
    T& acc, T& fx, T& fy, T& pu, T& pv, T& last_u, T& last_v, uint32_t& row, uint32_t& word,
    const T (&kw)[8], const CellGather<T, BUF>& cell, const StepGeom& sg, uint32_t lane_sign,
    int32_t s0, Sink& sink) {
  // masks of the sign of (pu, pv): a backward step's signs are the opposite
  constexpr bool kFlip = !FORWARD && !LANE_DIR;
  uint32_t apart = 0xFFFFFFFFu;  // sign bit: no near tie so far
  uint32_t low = 0xFFFFFFFFu;    // smallest numerator seen (numerator_key)
  T least = T(1);                // and |e| (float)
  uint32_t jump[8], jumped = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    if constexpr (POL != 0) {  // src/lib.rs:339-347, unfused dot product
      const T d1 = pu * last_u;
      const T d2 = pv * last_v;
      const T dot = (d1 + d2) + T(0);  // + 0: a sum of -0 does not flip
      pu = copy_sign_of(pu, dot);
      pv = copy_sign_of(pv, dot);
      last_u = pu;
      last_v = pv;
    }
    const T mu = LANE_DIR ? xor_sign(pu, lane_sign) : (FORWARD ? pu : -pu);
    const T mv = LANE_DIR ? xor_sign(pv, lane_sign) : (FORWARD ? pv : -pv);
    const uint32_t sx = sign_mask(LANE_DIR ? mu : pu), sy = sign_mask(LANE_DIR ? mv : pv);
    // the numerators of time_to_next_pixel (branchless rule): with the
    // sign bit set 0 * (0.5 - f) + f, else 2 * (0.5 - f) + f
    const T nx = macc<FMA>(T(2), keep_where<kFlip>(T(0.5) - fx, sx), fx);
    const T ny = macc<FMA>(T(2), keep_where<kFlip>(T(0.5) - fy, sy), fy);
    const T cy = ny * abs_t(mu);
    const T e = fma_t(nx, abs_t(mv), -cy);
    const uint32_t mx = sign_mask(e);  // step along x
    if constexpr (sizeof(T) == 4) least = min(least, abs_t(e));
    apart &= top_word(fma_t(near_tie(static_cast<T*>(nullptr)), cy, -abs_t(e)));
    // where the picked component is nonzero (or the lane is reported),
    // pos_x and pos_y of the full rule are the sign tests already made
    const uint32_t sp = pick(mx, sx, sy);
    uint32_t dist_y = sg.far_y;
    if constexpr (PAIRS) {
      const uint32_t far = bitop3<kFlip ? 0xEB : 0xBE>(0u - (row & 1u), sp, sg.all_far);
      dist_y = pick(far, sg.far_y, sg.near_y);
    }
    const uint32_t s = pick(mx, sg.step_x, dist_y);
    const uint32_t at = kFlip ? row + sp - (s ^ sp) : row - sp + (s ^ sp);
    const CellVal<T> cv = cell(at);
    const T n = pick(mx, nx, ny);
    const T t = quotient_rn(n, abs_t(pick(mx, mu, mv)));
    low = min(low, numerator_key(n));
    if (q & 1) {
      keep_in_step(apart);
      keep_in_step(low);
      if constexpr (sizeof(T) == 4) keep_in_step(least);
    }
    const T fy_after_x = macc<FMA>(t, mv, fy);
    const T fx_after_y = macc<FMA>(t, mu, fx);
    // on the edge just crossed: 1 after a step toward lower indices, else 0
    const T edge = edge_fraction<kFlip>(sp, static_cast<T*>(nullptr));
    fx = pick(mx, edge, fx_after_y);
    fy = pick(mx, fy_after_x, edge);
    jump[q] = pad_bits(cv.pad);
    jumped |= jump[q];
    row = at + jump[q];
    acc = macc<FMA>(kw[q], cv.x, acc);  // src/lib.rs:353-360
    sink(s0 + q, cv.x);
    pu = cv.u;
    pv = cv.v;
    if constexpr (REC != 0) {
      word = push_code<kFlip>(word, sp, mx);
      keep_in_step(word);
    }
    keep_in_step(acc);
  }
  if constexpr (REC != 0) {
    word &= 0x11111111u * (kMoveNeg | kMoveAxisY);
    if (__builtin_amdgcn_ballot_w64(jumped != 0u) != 0) {  // uniform: some line left the image
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        keep_in_step(jump[q]);  // compared here, not before the branch
        // a jump back to the cell the step came from (as long as the step:
        // a closed side, or the only column or row of a periodic one) stays
        const uint32_t far = min(jump[q], 0u - jump[q]);
        const bool stays = far == sg.step_x || far == sg.near_y || far == sg.far_y;
        const uint32_t low = 28 - 4 * q;
        word = jump[q] == 0u ? word
                             : (stays ? (word & ~(15u << low)) | (kMoveStay << low)
                                      : word | (kMoveEdge << low));
      }
      keep_in_step(word);  // a branch, not selects
    }
  }
  return __builtin_amdgcn_ballot_w64(static_cast<int32_t>(apart) >= 0) |
         __builtin_amdgcn_ballot_w64(low < numerator_key_min(static_cast<T*>(nullptr))) |
         __builtin_amdgcn_ballot_w64(least < T(kProductMin)) |
         __builtin_amdgcn_ballot_w64(__builtin_isunordered(fx, fy));
}

template <typename T, bool FMA, bool BRANCHLESS, int POL, bool FORWARD, int REC, bool BUF,
          bool PAIRS, bool LANE_DIR = false, typename Sink = NoSink>
__device__ __forceinline__ T trace_direction(T acc, T pu, T pv, uint32_t row,
                                             const CellGather<T, BUF>& cell,
                                             const T* __restrict__ kernel, int32_t kmid,
                                             int32_t nsteps, const StepGeom& sg,
                                             uint4* __restrict__ codes, int64_t np, int64_t p,
                                             int32_t c0, bool& short_path,
                                             bool fwd_lane = true, Sink sink = Sink{},
                                             int32_t* live_steps = nullptr) {
  constexpr bool pol = POL != 0, rec = REC != 0;
  const uint32_t lane_sign = fwd_lane ? 0u : 0x80000000u;  // LANE_DIR: negate on backward lanes
  T fx = T(0.5), fy = T(0.5);      // src/lib.rs:315-318
  T last_u = T(0), last_v = T(0);  // src/lib.rs:320-323
  bool alive = true;
  const uint32_t far_y = lane_copy(sg.far_y), near_y = lane_copy(sg.near_y);  // held in VGPRs
  const int32_t nchunks = chunks_of(nsteps);
  // Short path: whole groups of a chunk by fast_group; when a moving lane is
  // reported, the chunk is done again by the full rule.  Off for the rest of
  // the direction after a chunk that reports many lanes (a field of ties,
  // e.g. u = v everywhere) or a second chunk that reports any, so that such
  // a line costs little more than the full rule alone; many lanes turn it off
  // for the line's other direction too, and lines that start on a tie never
  // try it (u = v = 1 everywhere, 2048^2, L = 129: 727 -> 681 us).  (One saved state
  // per chunk: saving it for every group cost 2 VALU instructions per step.)
  bool fast = BRANCHLESS && short_path &&
              __popcll(__builtin_amdgcn_ballot_w64(abs_t(pu) == abs_t(pv) && pu != T(0))) < 8;
  int32_t misses = 0;
  bool live_now = false, moves_now = false;  // set before a chunk of the short path
  bool status_known = false;
  for (int32_t ch = 0; ch < nchunks; ++ch) {
    uint32_t words[4] = {kWordStay, kWordStay, kWordStay, kWordStay};
    bool any_alive = true;
    int g0 = 0;
    if (BRANCHLESS && fast) {  // uniform
      if (!status_known) {  // lanes that do not move never move again
        live_now = alive && !__builtin_isunordered(pu, pv);
        moves_now = live_now && (pu != T(0) || pv != T(0));
        status_known = true;
      }
      const uint64_t m_moves = __builtin_amdgcn_ballot_w64(moves_now);
      const StepGeom sl = {moves_now ? sg.step_x : 0u, moves_now ? near_y : 0u,
                           moves_now ? far_y : 0u, sg.all_far};
      // fractions outside what fast_group takes (the full rule can leave
      // some after a tie): this chunk by the full rule
      const bool usable = __builtin_amdgcn_ballot_w64(moves_now && !(fraction_usable(fx) &&
                                                                      fraction_usable(fy))) == 0;
      const int full = usable ? min(4, (nsteps - ch * kChunkSteps) >> 3) : 0;
      const T acc_0 = acc, fx_0 = fx, fy_0 = fy, pu_0 = pu, pv_0 = pv, lu_0 = last_u,
              lv_0 = last_v;
      const uint32_t row_0 = row;
      uint64_t reported = 0;
#pragma unroll 1
      for (; g0 < full; ++g0) {
        const int32_t s0 = ch * kChunkSteps + 8 * g0;
        T kw[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
          kw[q] = kernel[FORWARD ? kmid + 1 + s0 + q : kmid - 1 - s0 - q];
        uint32_t word = 0;
        reported = fast_group<T, FMA, POL, FORWARD, REC, BUF, PAIRS, LANE_DIR>(
                       acc, fx, fy, pu, pv, last_u, last_v, row, word, kw, cell, sl, lane_sign,
                       s0, sink) &
                   m_moves;
        if (reported != 0) break;  // uniform
        words[g0] = word;
      }
      if (reported == 0) {
        if (m_moves != __builtin_amdgcn_ballot_w64(true)) {  // uniform
          // a zero vector stays and has added its cell's value at
          // every step; an ended line adds nothing and records stops
          acc = live_now ? acc : acc_0;
          const uint32_t still = live_now ? kWordStay : 0x11111111u * kMoveStop;
#pragma unroll
          for (int g = 0; g < 4; ++g) words[g] = moves_now || g >= full ? words[g] : still;
        }
        if (full == 0) {
          status_known = false;  // the full rule runs next
        } else {
          alive = live_now;
          if (live_steps) *live_steps = live_now ? ch * kChunkSteps + 8 * full : *live_steps;
          any_alive = __builtin_amdgcn_ballot_w64(alive) != 0;
        }
      } else {
        const bool many = __popcll(reported) >= 8;
        fast = ++misses < 2 && !many;
        short_path = short_path && !many;
        status_known = false;
        acc = acc_0;
        fx = fx_0;
        fy = fy_0;
        pu = pu_0;
        pv = pv_0;
        last_u = lu_0;
        last_v = lv_0;
        row = row_0;
        g0 = 0;
      }
    }
#pragma unroll 1
    for (int g = g0; g < 4; ++g) {
      const int32_t s0 = ch * kChunkSteps + 8 * g;
      if (s0 >= nsteps || !any_alive) break;  // uniform
      T kw[8];
#pragma unroll
      for (int q = 0; q < 8; ++q)
        kw[q] = kernel[FORWARD ? kmid + 1 + s0 + q : kmid - 1 - s0 - q];
      uint32_t word = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (s0 + q >= nsteps) break;  // uniform: last group only
        // a NaN component ends the line (src/lib.rs:336-338)
        const bool ordered = !__builtin_isunordered(pu, pv);
        const bool live = alive && ordered;
        if constexpr (pol) {  // src/lib.rs:339-347, unfused dot product
          const T d1 = pu * last_u;
          const T d2 = pv * last_v;
          const bool flip = d1 + d2 < T(0);
          pu = flip ? -pu : pu;
          pv = flip ? -pv : pv;
          last_u = pu;
          last_v = pv;
        }
        // src/lib.rs:348-351
        const T mu = LANE_DIR ? xor_sign(pu, lane_sign) : (FORWARD ? pu : -pu);
        const T mv = LANE_DIR ? xor_sign(pv, lane_sign) : (FORWARD ? pv : -pv);
        // sign tests of mu, mv read pu, pv (negation flips the sign bit), so
        // that a backward step does not materialize -pu, -pv for them: the
        // divisions and products take the negation as a source modifier
        const bool neg_x = LANE_DIR  ? __builtin_signbit(mu)
                           : FORWARD ? __builtin_signbit(pu)
                                     : !__builtin_signbit(pu);
        const bool neg_y = LANE_DIR  ? __builtin_signbit(mv)
                           : FORWARD ? __builtin_signbit(pv)
                                     : !__builtin_signbit(pv);
        const T tx = time_to_next_pixel<T, FMA, BRANCHLESS>(mu, fx, neg_x);
        const T ty = time_to_next_pixel<T, FMA, BRANCHLESS>(mv, fy, neg_y);
        // x edge first when tx < ty; ties and NaN go to y (src/lib.rs:249-269)
        const bool xs = tx < ty;
        // no move when both components are +-0 (src/lib.rs:242-244)
        const bool moves = live && (mu != T(0) || mv != T(0));
        // update_state (src/lib.rs:208-233) for either axis, then keep one
        // pos_x only matters when the x edge comes first (tx < ty), which
        // needs a finite tx and so a nonzero, non-NaN mu: there it equals
        // mu >= 0 (src/lib.rs:217), and the sign test is the one the step
        // time already made.  pos_y is used for y steps, which also happen
        // with mv = -0 (tx and ty both infinite), so it stays mv >= 0.
        const bool pos_x = !neg_x;
        const bool pos_y = LANE_DIR ? mv >= T(0) : FORWARD ? pv >= T(0) : pv <= T(0);  // mv >= 0
        const T fy_after_x = macc<FMA>(tx, mv, fy);
        const T fx_after_y = macc<FMA>(ty, mu, fx);
        const T fx_new = xs ? (pos_x ? T(0) : T(1)) : fx_after_y;
        const T fy_new = xs ? fy_after_x : (pos_y ? T(0) : T(1));
        // The fractions need no "moves" gate: a lane that does not move
        // never moves again (an ended line stays on its NaN cell, a zero
        // vector stays on its cell, whose vector stays zero, polarization
        // flips included), so its fractions are never read again: they only
        // feed step times, whose results are masked out of its code bits and
        // its position update.
        fx = fx_new;
        fy = fy_new;
        // a y step leaves the row pair up from an odd row, down from an even one
        const bool odd = (row & 1u) != 0u;
        const uint32_t dist_y = !PAIRS || odd == pos_y || sg.all_far != 0u ? far_y : near_y;
        const uint32_t step = xs ? (pos_x ? sg.step_x : 0u - sg.step_x)
                                 : (pos_y ? dist_y : 0u - dist_y);
        const uint32_t from = row;
        const uint32_t at = moves ? row + step : row;
        const CellVal<T> cv = cell(at);
        const uint32_t jump = pad_bits(cv.pad);
        const bool edge = jump != 0u;  // the step left the image
        row = at + jump;
        const T next_acc = macc<FMA>(kw[q], cv.x, acc);  // src/lib.rs:353-360
        acc = live ? next_acc : acc;
        sink(s0 + q, cv.x);
        if (live_steps) *live_steps = live ? s0 + q + 1 : *live_steps;
        pu = cv.u;
        pv = cv.v;
        if constexpr (rec) {
          // The code's four bits (stay, negative direction, y axis, edge or
          // stop) are combined from the step's comparisons as wave lane
          // masks on the scalar unit, then shifted into the word one at a
          // time with an add-with-carry (word = 2 * word + bit), so the
          // group's first step ends in the top nibble (move_code).  A line
          // that has ended stays on its NaN cell, so it records the stop
          // code again at every later step; readers stop at the first one.
          const uint64_t m_stop = ~__builtin_amdgcn_ballot_w64(ordered);
          const uint64_t m_stay = __builtin_amdgcn_ballot_w64(row == from);
          const uint64_t m_x = __builtin_amdgcn_ballot_w64(xs);
          const uint64_t m_edge = __builtin_amdgcn_ballot_w64(edge);
          const uint64_t m_neg = ~((m_x & __builtin_amdgcn_ballot_w64(pos_x)) |
                                   (~m_x & __builtin_amdgcn_ballot_w64(pos_y)));
          word = carry_in_bit(word, m_stay);
          word = carry_in_bit(word, m_neg & ~m_stay);
          word = carry_in_bit(word, ~m_x & ~m_stay);
          word = carry_in_bit(word, (m_edge & ~m_stay) | m_stop);
        }
        alive = live;
      }
      // a last group of fewer than 8 steps: its first step to the top
      // nibble, "stay" codes after its last
      if (rec && nsteps - s0 < 8) {
        const int32_t spare = 4 * (8 - (nsteps - s0));
        word = (word << spare) | (kWordStay >> (32 - spare));
      }
      words[g] = word;
      any_alive = __builtin_amdgcn_ballot_w64(alive) != 0;
    }
    if (rec) codes[(c0 + ch) * np + p] = make_uint4(words[0], words[1], words[2], words[3]);
    if (!any_alive) break;  // every line of the wave ended
  }
  return acc;
}

// Replay of one direction from its move codes.  Chunks of 32 steps: the
// chunk after the current one is loaded before the current one is used, and
// within a chunk each group of 8 steps decodes its 8 positions through the
// delta table, issues the 8 texture gathers together and accumulates them
// in step order.  Codes are valid up to the step where the line ended (the
// tracing pass wrote the stop code there), so a lane stops reading codes
// once its line has ended and its later codes are taken as "stay".
template <typename T, bool FMA, bool FORWARD, bool BUF>
__device__ __forceinline__ T replay_direction(T acc, uint32_t pos,
                                              const ValueGather<T, BUF>& x,
                                              const T* __restrict__ kernel, int32_t kmid,
                                              int32_t nsteps, const uint32_t* delta,
                                              const uint4* __restrict__ codes, int64_t np,
                                              int64_t p, int32_t c0) {
  const int32_t nchunks = chunks_of(nsteps);
  bool alive = true;
  uint4 next = nchunks > 0 ? codes[c0 * np + p] : make_uint4(0u, 0u, 0u, 0u);
  for (int32_t ch = 0; ch < nchunks; ++ch) {
    const uint4 cur = next;
    if (ch + 1 < nchunks && alive) next = codes[(c0 + ch + 1) * np + p];
    const uint32_t words[4] = {cur.x, cur.y, cur.z, cur.w};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int32_t s0 = ch * kChunkSteps + 8 * g;
      if (s0 >= nsteps) break;  // uniform
      const uint32_t word = alive ? words[g] : kWordStay;
      T kw[8];
#pragma unroll
      for (int q = 0; q < 8; ++q)
        kw[q] = kernel[FORWARD ? kmid + 1 + s0 + q : kmid - 1 - s0 - q];
      uint32_t at[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        pos += delta[move_code(word, q)];
        at[q] = pos;
      }
      T xv[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) xv[q] = x(at[q]);
      const bool full = alive && !group_has_stop(word) && nsteps - s0 >= 8;
      if (__builtin_amdgcn_ballot_w64(!full) == 0) {
        // every lane accumulates all 8 steps (wave-uniform): no masks
#pragma unroll
        for (int q = 0; q < 8; ++q) acc = macc<FMA>(kw[q], xv[q], acc);
      } else {
        // no break for the last group: a break lets the compiler sink the
        // gathers past it and wait for each one in turn; steps past the end
        // read "stay" codes (position unchanged, weight from the padding)
        const int32_t valid = alive ? steps_before_stop(word) : 0;
        const int32_t lim = min(valid, nsteps - s0);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const T next_acc = macc<FMA>(kw[q], xv[q], acc);
          acc = q < lim ? next_acc : acc;
        }
        alive = valid == 8;
      }
    }
    if (__builtin_amdgcn_ballot_w64(alive) == 0) break;
  }
  return acc;
}

}  // namespace rlic
