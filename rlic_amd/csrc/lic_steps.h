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
// is the cell's slot (cell_slot).  Returns the updated accumulator.  With REC,
// writes the move code of every step.
//
// Steps run in groups of 8 (one code word) without divergent branches, and a
// wave leaves the loop once all its lines have ended: whole groups by
// fast_group while `short_path` holds, others by full_group.
// NARROW: the branchless rule, and a field that is not wide (velocity_wide).
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

// Whether a step of `jump` slots on from a guard cell leads back to the cell it
// came from: a jump as long as a step (a closed side, or the only column or
// row of a periodic one).
__device__ __forceinline__ bool jump_stays(uint32_t jump, const StepGeom& sg) {
  const uint32_t far = min(jump, 0u - jump);
  return far == sg.step_x || far == sg.near_y || far == sg.far_y;
}

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
// their roundings compare as the exact ones do; otherwise (an exact or a near
// tie, both components zero, a NaN component: every one of them fails the
// comparison) the lane is reported.  The quotient is quotient_rn's, which needs a numerator that is zero or not tiny
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
// cycles per wave (the full rule's 57 took about 170).  The texture data unit's
// busy counter reads 94 to 97% beside it, but it does so in every variant, at
// 48 and at 63 cycles a gather of equal accesses, so it counts waiting and shows
// no bound.  Trace launches, full rule in plain rows -> with this alone -> and
// row pairs (cell_slot): 4096^2 float L=129 with the record 2.47 -> 1.92 ->
// 1.86 ms, 2111x1500 float with holes L=201 775 -> 684 -> 603 us, 1021x1537
// double L=151 499 -> 447 -> 430 us, 16384^2 float polarization L=257 (plain
// rows) 72.2 -> 55.0 -> 54.5 ms, 8192^2 double polarization 30.1 -> 26.4 ->
// 26.4 ms, 256^2 double L=65 (paired lanes) 22.6 -> 19.3 -> 19.9 us.  With the
// full rule as it is now beside it, the first and the last of these in one run:
// 2.50 and 1.87 ms, 789 and 627 us, 501 and 418 us; paired 21.5 and 19.2 us.  Row
// pairs alone cost the paired lanes 3% and are kept there because a field has
// one layout for every kernel.
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
    word &= kWordMoves;
    if (__builtin_amdgcn_ballot_w64(jumped != 0u) != 0) {  // uniform: some line left the image
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        keep_in_step(jump[q]);  // compared here, not before the branch
        const uint32_t low = 28 - 4 * q;
        const uint32_t left = jump_stays(jump[q], sg) ? (word & ~(15u << low)) | (kMoveStay << low)
                                                      : word | (kMoveEdge << low);
        word = jump[q] == 0u ? word : left;
      }
      keep_in_step(word);  // a branch, not selects
    }
  }
  return __builtin_amdgcn_ballot_w64(static_cast<int32_t>(apart) >= 0) |
         __builtin_amdgcn_ballot_w64(low < numerator_key_min(static_cast<T*>(nullptr))) |
         __builtin_amdgcn_ballot_w64(least < T(kProductMin)) |
         __builtin_amdgcn_ballot_w64(__builtin_isunordered(fx, fy));
}

// A lane's state at the start of a chunk, for doing the chunk again: kept in
// registers, or (SavedLds) in its kWords values of LDS.  The vector is not
// kept: it is gathered again.
template <typename T>
struct SavedRegisters {
  T a, x, y, u, v;
  __device__ __forceinline__ void put(T acc, T fx, T fy, T lu, T lv) {
    a = acc;
    x = fx;
    y = fy;
    u = lu;
    v = lv;
  }
  __device__ __forceinline__ T acc() const { return a; }
  __device__ __forceinline__ void get(T& acc, T& fx, T& fy, T& lu, T& lv) const {
    acc = a;
    fx = x;
    fy = y;
    lu = u;
    lv = v;
  }
};
template <typename T, bool POL>
struct SavedLds {
  static constexpr int32_t kWords = POL ? 5 : 3;
  // volatile: stored, not carried along in registers
  typedef volatile T __attribute__((address_space(3))) lds_t;
  lds_t* at;
  __device__ __forceinline__ void put(T acc, T fx, T fy, T lu, T lv) {
    at[0] = acc;
    at[1] = fx;
    at[2] = fy;
    if constexpr (POL) {
      at[3] = lu;
      at[4] = lv;
    }
  }
  __device__ __forceinline__ T acc() const { return at[0]; }
  __device__ __forceinline__ void get(T& acc, T& fx, T& fy, T& lu, T& lv) const {
    acc = at[0];
    fx = at[1];
    fy = at[2];
    if constexpr (POL) {
      lu = at[3];
      lv = at[4];
    }
  }
};

// A group of up to 8 steps by the full rule (src/lib.rs:304-362), for lanes in
// any state: a lane whose line has ended (NaN vector) keeps executing with its
// position frozen and its accumulator untouched, a lane with a zero vector
// keeps its position (src/lib.rs:242-244).  `m_live` receives the lanes whose
// line had not ended before the last step.
//
// QUICK (float, branchless rule, velocities within VelocityRange): the step
// times by quotient_rn, which is what the division gives but for tiny
// numerators; a step in which a moving lane has one is done again with the
// division (in double the tests cost what the shorter quotient saves).
//
// What bounds it: VALU issue, and the chain from a cell's vector to the next
// address.  So selections are bit operations on lane masks, as in fast_group,
// rare cases are tested behind the gather's issue (before it, the test's
// branch cost 8%), and eight steps are one block of straight code (a branch out
// of it for a short last group made the compiler copy the state at each step).
// A step is 51 VALU instructions, with the record 57, QUICK 47 and 53; 49 and 54
// before row pairs and the short path existed, 57 and 69 with them at first.
// 2048^2, L = 129, a field with one component out of range, us a call then, at
// first, now: float 601, 638, 606, double 1015, 1043, 990; with the record (L =
// 65, two passes) 426, 478, 420 and 662, 702, 649.
template <typename T, bool FMA, bool BRANCHLESS, int POL, bool FORWARD, int REC, bool BUF,
          bool PAIRS, bool LANE_DIR, bool QUICK, typename Sink>
__device__ __forceinline__ void full_group(T& acc, T& fx, T& fy, T& pu, T& pv, T& last_u,
                                           T& last_v, uint32_t& row, uint64_t& m_live,
                                           uint32_t& word, const T* __restrict__ taps,
                                           const CellGather<T, BUF>& cell, const StepGeom& sg,
                                           uint32_t lane_sign, int32_t s0, int32_t steps,
                                           Sink& sink, int32_t* live_steps) {
  constexpr bool kFlip = !FORWARD && !LANE_DIR;
  uint32_t marks = 0, moved = 0;  // codes of steps that left the image; steps that moved
  auto one = [&](int32_t q) {
    const T weight = taps[FORWARD ? q : -q];
    // a NaN component ends the line (src/lib.rs:336-338), which stays on its cell
    const bool live = !__builtin_isunordered(pu, pv);
    m_live = __builtin_amdgcn_ballot_w64(live);
    if constexpr (POL != 0) {  // src/lib.rs:339-347, unfused dot product
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
    // masks of the sign bits of mu, mv, read off pu, pv (kFlip: the opposite),
    // so that a backward step does not materialize -pu, -pv for them: the
    // divisions and products take the negation as a modifier
    const uint32_t sx = sign_mask(LANE_DIR ? mu : pu), sy = sign_mask(LANE_DIR ? mv : pv);
    // no move when both components are +-0 (src/lib.rs:242-244)
    const bool moves = live & ((mu != T(0)) | (mv != T(0)));
    T tx, ty;
    uint32_t mx, sp, at;
    auto step_to = [&](uint32_t neg_y) {
      // x edge first when tx < ty; ties and NaN go to y (src/lib.rs:249-269)
      mx = tx < ty ? ~0u : 0u;
      sp = pick(mx, sx, neg_y);  // toward lower indices (kFlip: higher)
      uint32_t dist_y = sg.far_y;
      if constexpr (PAIRS)  // up from an odd row, down from an even one: another pair
        dist_y = pick(bitop3<kFlip ? 0xEB : 0xBE>(0u - (row & 1u), sp, sg.all_far), sg.far_y,
                      sg.near_y);
      const uint32_t step = moves ? pick(mx, sg.step_x, dist_y) : 0u;
      at = kFlip ? row + sp - (step ^ sp) : row - sp + (step ^ sp);
    };
    auto divide = [&]() {
      if constexpr (BRANCHLESS) {
        tx = abs_t(div_rn(step_numerator<T, FMA, kFlip>(fx, sx), mu));
        ty = abs_t(div_rn(step_numerator<T, FMA, kFlip>(fy, sy), mv));
      } else {
        tx = time_to_next_pixel(mu, fx);
        ty = time_to_next_pixel(mv, fy);
      }
    };
    uint64_t tiny = 0;
    if constexpr (QUICK) {
      const T nx = step_numerator<T, FMA, kFlip>(fx, sx);
      const T ny = step_numerator<T, FMA, kFlip>(fy, sy);
      tx = abs_t(quotient_rn(nx, abs_t(mu)));
      // beside any other time, one over a component of 0 is as good as infinite
      ty = abs_t(quotient_rn(ny, positive_divisor(mv)));
      tiny = tiny_numerators(nx) | tiny_numerators(ny);
    } else {
      divide();
    }
    step_to(sy);
    CellVal<T> cv = cell(at);
    // Tested while the cell is on its way.  Toward lower indices is mu < 0, mv
    // < 0 (src/lib.rs:217): the sign bit, but for y steps with mv = -0 (ty
    // infinite or NaN).
    const uint64_t m_mv = __builtin_amdgcn_ballot_w64(mv != T(0));
    const uint64_t level = ~m_mv & ~__builtin_amdgcn_ballot_w64(tx < ty);
    if ((m_live & (m_mv | __builtin_amdgcn_ballot_w64(mu != T(0))) & (level | tiny)) != 0) {
      if constexpr (QUICK) divide();  // uniform
      step_to(mv == T(0) ? (kFlip ? ~0u : 0u) : sy);
      cv = cell(at);
    }
    // update_state (src/lib.rs:208-233) for either axis, keeping one.  The
    // fractions need no "moves" gate: a lane that does not move never moves
    // again (an ended line stays on its NaN cell, a zero vector stays on its
    // cell, whose vector stays zero, polarization flips included), so its
    // fractions are never read again: they only feed step times, whose
    // results are masked out of its codes and its position update.
    const T fy_after_x = macc<FMA>(tx, mv, fy);
    const T fx_after_y = macc<FMA>(ty, mu, fx);
    const T edge = edge_fraction<kFlip>(sp, static_cast<T*>(nullptr));
    fx = pick(mx, edge, fx_after_y);
    fy = pick(mx, fy_after_x, edge);
    const uint32_t jump = pad_bits(cv.pad);  // not 0: the step left the image
    row = at + jump;
    const T next_acc = macc<FMA>(weight, cv.x, acc);  // src/lib.rs:353-360
    acc = live ? next_acc : acc;
    keep_in_step(acc);
    sink(s0 + q, cv.x);
    if (live_steps) *live_steps = live ? s0 + q + 1 : *live_steps;
    pu = cv.u;
    pv = cv.v;
    if constexpr (REC != 0) {
      word = push_code<kFlip>(word, sp, mx);
      keep_in_step(word);
      moved += moves ? 1u : 0u;
      if (__builtin_amdgcn_ballot_w64(jump != 0u) != 0) {  // uniform
        uint32_t code = jump_stays(jump, sg) ? kMoveStay : kMoveEdge;
        keep_in_step(code);  // shifted after: the select's constants stay inline
        marks |= jump != 0u ? code << (28 - 4 * q) : 0u;
        keep_in_step(marks);  // a branch, not selects
      }
    }
  };
  if (!LANE_DIR && steps == 8) {  // uniform
#pragma unroll
    for (int32_t q = 0; q < 8; ++q) one(q);
  } else {
#pragma unroll 1
    for (int32_t q = 0; q < steps; ++q) one(q);
  }
  if constexpr (REC != 0) {
    // a last group of fewer than 8 steps: its first step to the top nibble
    if (steps < 8) word <<= 4 * (8 - steps);
    const uint32_t stays = marks & kWordStay;
    word = (word & kWordMoves & ~(stays >> 1 | stays >> 2)) | marks;
    if (steps < 8 || __builtin_amdgcn_ballot_w64(moved < 8) != 0) {  // uniform
      // A lane that stops moving stays so: "stay" from there on, or "stop" on
      // a NaN cell (readers stop at the first one).
      const bool ended = moved < static_cast<uint32_t>(steps) && __builtin_isunordered(pu, pv);
      const uint32_t still = ended ? 0x11111111u * kMoveStop : kWordStay;
      word = moved < 8 ? (word & ~(~0u >> (4 * moved))) | (still >> (4 * moved)) : word;
    }
  }
}

template <typename T, bool FMA, bool BRANCHLESS, int POL, bool FORWARD, int REC, bool BUF,
          bool PAIRS, bool NARROW, bool LANE_DIR = false, typename Saved, typename Sink = NoSink>
__device__ __forceinline__ T trace_direction(T acc, T pu, T pv, uint32_t row,
                                             const CellGather<T, BUF>& cell,
                                             const T* __restrict__ kernel, int32_t kmid,
                                             int32_t nsteps, const StepGeom& sg,
                                             uint4* __restrict__ codes, int64_t np, int64_t p,
                                             int32_t c0, bool& short_path, Saved& saved,
                                             bool fwd_lane = true, Sink sink = Sink{},
                                             int32_t* live_steps = nullptr) {
  constexpr bool rec = REC != 0;
  const uint32_t lane_sign = fwd_lane ? 0u : 0x80000000u;  // LANE_DIR: negate on backward lanes
  T fx = T(0.5), fy = T(0.5);      // src/lib.rs:315-318
  T last_u = T(0), last_v = T(0);  // src/lib.rs:320-323
  // held in VGPRs
  const StepGeom sl = {sg.step_x, lane_copy(sg.near_y), lane_copy(sg.far_y), sg.all_far};
  const int32_t nchunks = chunks_of(nsteps);
  // Short path: whole groups of a chunk by fast_group; when a moving lane is
  // reported, the chunk is done again by the full rule (one saved state per
  // chunk: saving it for every group cost 2 VALU instructions per step; the
  // paired trace in float is apart, below).  What
  // is thrown away costs a group at least, so the path is left for the rest of
  // the line and for its other direction where more reports are likely: after
  // one of many lanes, one in a chunk's first two groups, or a second one; in
  // double, where a step saves 1/6 (float: 1/4), after any, and it is not tried
  // where lanes of the wave start on a tie or only some of them move.
  // 2048^2, L = 129, us a call before this path existed, with two tries in each
  // direction, now: float 1% of cells NaN 596, 720, 582, 10% zero 577, 644, 535,
  // whole numbers (ties and zeros) 583, 654, 587, u = v 579, 635, 524; double
  // 991, 1202, 1027, then 970, 998, 890, then 922, 1020, 955, then 939, 989, 941.
  const uint64_t m_tie = __builtin_amdgcn_ballot_w64(abs_t(pu) == abs_t(pv)) &
                         __builtin_amdgcn_ballot_w64(pu != T(0));
  bool fast = NARROW && short_path;
  if constexpr (sizeof(T) == 4) {
    fast = fast && __popcll(m_tie) < 8;
  } else {
    const uint64_t m_rest = __builtin_amdgcn_ballot_w64(__builtin_isunordered(pu, pv)) |
                            (__builtin_amdgcn_ballot_w64(pu == T(0)) &
                             __builtin_amdgcn_ballot_w64(pv == T(0)));
    fast = fast && m_tie == 0 && (m_rest == 0 || m_rest == __builtin_amdgcn_ballot_w64(true));
  }
  int32_t misses = 0;
  bool live_now = false, moves_now = false;  // set before a chunk of the short path
  bool status_known = false;
  if constexpr (LANE_DIR && sizeof(T) == 4) {
    // So few waves that the longest one sets the launch's time, and in float one
    // of them nearly always has a report: so only the reported group is done
    // again.  A launch before the short path existed, with whole chunks done
    // again (and 8 times the reports: near_tie), now: 256^2 L = 65 17.9, 22.3,
    // 16.7 us, L = 33 11.9, 13.8, 12.0, 362^2 L = 65 23.9, 25.5, 20.4; without
    // any report 64^2 L = 65 13.6, 11.1, 11.6.  In double, where reports are
    // rare, whole chunks are 1 to 3% faster.
    StepGeom sm = sl;
    uint64_t m_moves = 0;
    bool all_move = false;
    for (int32_t ch = 0; ch < nchunks; ++ch) {
      uint32_t words[4] = {kWordStay, kWordStay, kWordStay, kWordStay};
      bool any_alive = true;
#pragma unroll 1
      for (int g = 0; g < 4; ++g) {
        const int32_t s0 = ch * kChunkSteps + 8 * g;
        if (s0 >= nsteps || !any_alive) break;  // uniform
        uint32_t word = 0;
        if (NARROW && fast && s0 + 8 <= nsteps && !status_known) {  // uniform
          live_now = !__builtin_isunordered(pu, pv);
          moves_now = live_now && (pu != T(0) || pv != T(0));
          sm = {moves_now ? sl.step_x : 0u, moves_now ? sl.near_y : 0u,
                moves_now ? sl.far_y : 0u, sl.all_far};
          m_moves = __builtin_amdgcn_ballot_w64(moves_now);
          all_move = m_moves == __builtin_amdgcn_ballot_w64(true);
          status_known = __builtin_amdgcn_ballot_w64(
                             moves_now && !(fraction_usable(fx) && fraction_usable(fy))) == 0;
        }
        if (NARROW && fast && s0 + 8 <= nsteps && status_known) {  // uniform
          const uint32_t row_0 = row;
          saved.put(acc, fx, fy, last_u, last_v);
          T kw[8];
#pragma unroll
          for (int q = 0; q < 8; ++q)
            kw[q] = kernel[FORWARD ? kmid + 1 + s0 + q : kmid - 1 - s0 - q];
          const uint64_t reported =
              fast_group<T, FMA, POL, FORWARD, REC, BUF, PAIRS, LANE_DIR>(
                  acc, fx, fy, pu, pv, last_u, last_v, row, word, kw, cell, sm, lane_sign, s0,
                  sink) &
              m_moves;
          if (reported == 0) {  // uniform
            if (all_move) {  // uniform
              if (live_steps) *live_steps = s0 + 8;
            } else {
              if (!live_now) acc = saved.acc();
              const uint32_t still = live_now ? kWordStay : 0x11111111u * kMoveStop;
              word = moves_now ? word : still;
              if (live_steps) *live_steps = live_now ? s0 + 8 : *live_steps;
              any_alive = __builtin_amdgcn_ballot_w64(live_now) != 0;
            }
            words[g] = word;
            continue;
          }
          fast = ++misses < 3 && __popcll(reported) < 8;
          saved.get(acc, fx, fy, last_u, last_v);
          row = row_0;
          const CellVal<T> cv = cell(row);
          pu = cv.u;
          pv = cv.v;
          word = 0;
        }
        status_known = false;
        uint64_t m_live = 0;
        full_group<T, FMA, BRANCHLESS, POL, FORWARD, REC, BUF, PAIRS, LANE_DIR,
                   NARROW && sizeof(T) == 4>(
            acc, fx, fy, pu, pv, last_u, last_v, row, m_live, word,
            kernel + (FORWARD ? kmid + 1 + s0 : kmid - 1 - s0), cell, sl, lane_sign, s0,
            min(8, nsteps - s0), sink, live_steps);
        words[g] = word;
        any_alive = m_live != 0;
      }
      if (rec) codes[(c0 + ch) * np + p] = make_uint4(words[0], words[1], words[2], words[3]);
      if (!any_alive) break;
    }
    return acc;
  }
  for (int32_t ch = 0; ch < nchunks; ++ch) {
    uint32_t words[4] = {kWordStay, kWordStay, kWordStay, kWordStay};
    bool any_alive = true;
    int g0 = 0;
    if (NARROW && fast) {  // uniform
      if (!status_known) {  // lanes that do not move never move again
        live_now = !__builtin_isunordered(pu, pv);
        moves_now = live_now && (pu != T(0) || pv != T(0));
        status_known = true;
      }
      const uint64_t m_moves = __builtin_amdgcn_ballot_w64(moves_now);
      const StepGeom sm = {moves_now ? sl.step_x : 0u, moves_now ? sl.near_y : 0u,
                           moves_now ? sl.far_y : 0u, sl.all_far};
      // fractions outside what fast_group takes (the full rule can leave
      // some after a tie): this chunk by the full rule
      const bool usable = __builtin_amdgcn_ballot_w64(moves_now && !(fraction_usable(fx) &&
                                                                      fraction_usable(fy))) == 0;
      const int full = usable ? min(4, (nsteps - ch * kChunkSteps) >> 3) : 0;
      const uint32_t row_0 = row;
      saved.put(acc, fx, fy, last_u, last_v);
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
                       acc, fx, fy, pu, pv, last_u, last_v, row, word, kw, cell, sm, lane_sign,
                       s0, sink) &
                   m_moves;
        if (reported != 0) break;  // uniform
        words[g0] = word;
      }
      if (reported == 0) {
        if (m_moves != __builtin_amdgcn_ballot_w64(true)) {  // uniform
          // a zero vector stays and has added its cell's value at
          // every step; an ended line adds nothing and records stops
          if (!live_now) acc = saved.acc();
          const uint32_t still = live_now ? kWordStay : 0x11111111u * kMoveStop;
#pragma unroll
          for (int g = 0; g < 4; ++g) words[g] = moves_now || g >= full ? words[g] : still;
        }
        if (full == 0) {
          status_known = false;  // the full rule runs next
        } else {
          if (live_steps) *live_steps = live_now ? ch * kChunkSteps + 8 * full : *live_steps;
          any_alive = __builtin_amdgcn_ballot_w64(live_now) != 0;
        }
      } else {
        fast = sizeof(T) == 4 && g0 >= 2 && ++misses < 2 && __popcll(reported) < 8;
        short_path = short_path && fast;
        status_known = false;
        saved.get(acc, fx, fy, last_u, last_v);
        row = row_0;
        const CellVal<T> cv = cell(row);  // the vector there, not kept for this
        pu = cv.u;
        pv = cv.v;
        g0 = 0;
      }
    }
#pragma unroll 1
    for (int g = g0; g < 4; ++g) {
      const int32_t s0 = ch * kChunkSteps + 8 * g;
      if (s0 >= nsteps || !any_alive) break;  // uniform
      uint32_t word = 0;
      uint64_t m_live = 0;
      full_group<T, FMA, BRANCHLESS, POL, FORWARD, REC, BUF, PAIRS, LANE_DIR,
                 NARROW && sizeof(T) == 4>(
          acc, fx, fy, pu, pv, last_u, last_v, row, m_live, word,
          kernel + (FORWARD ? kmid + 1 + s0 : kmid - 1 - s0), cell, sl, lane_sign, s0,
          min(8, nsteps - s0), sink, live_steps);
      words[g] = word;
      any_alive = m_live != 0;
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
