// LDS replay over boxes cut to the lines (gfx950).
//
// A replay pass gathers one texture value per recorded move.  A block takes
// a tile of 32 x 32 pixels, a line per lane, and stages in LDS, for either
// direction, the rectangle that the tile's lines visit (in unwrapped
// coordinates: a periodic edge is just crossed), then walks them there.  The
// rectangles are known from the moves: the first replay of a record reads it
// twice, once to find them, and stores them (32 bytes a tile) for the later
// passes.
//
// Lines of a tile follow one flow, so the rectangle is far smaller than the
// tile grown by the half length on all sides: at 4096^2, L = 129, on average
// 4,700 cells for a direction (25,600 the other way), at L = 201 5,200-8,600
// (53,800, which fits no LDS).  So long kernels replay from LDS too, and two
// blocks of 70 KB fit a CU: one stages while the other walks.  Both
// directions' boxes are staged at once if they fit together (L = 129: 83% of
// the tiles), else one after the other.  Where a direction's box does not fit
// (lines that part: 10% of the tiles at L = 201, 45% in double at 2048^2, L =
// 151), the box of as many waves as fit is staged and the others gather from
// the image beside them: a wave's 64 lines part far less than the tile's.
// Against a tile gathering from the image as a whole: 4096^2 L = 201 969 ->
// 684 us, L = 401 4610 -> 2714; 2048^2 double L = 151 323 -> 218.
//
// What bounds it: at 4096^2, L = 129, 360 us a later pass (whole boxes in
// lic_replay_lds: 486), of which reading the record alone takes 228 (64 bytes
// a pixel); VALU and scalar issue are each about 60% busy, LDS 45%.  The first
// pass takes 220 us more, the moves' dot products and a second chain of loads.
// Tried (against the 342 us a later pass took in those runs): two lines per
// lane in three blocks of 50 KB (528 us; fewer boxes fit), bounds per chunk of
// 32 steps with runs of chunks that fit (registers spilled), bounds kept by the
// tracing pass (12% longer there), up to four boxes one after the other for the
// waves left (L = 257 1076 -> 897 us, but 32 spilled registers: L = 129 342 ->
// 392), the first pass's record held in registers (no faster: the second read
// comes from the caches).
#include <algorithm>
#include <type_traits>

#include "lic_device.h"
#include "lic_launch.h"
#include "lic_lds.h"
#include "lic_steps.h"

namespace rlic {

namespace {

constexpr int32_t kBoxTile = 32;
constexpr int32_t kBoxThreads = kBoxTile * kBoxTile;  // a line per lane
constexpr int32_t kBoxWaves = kBoxThreads / 64;
// Steps per direction: bounds are 16-bit, and two boxes' sizes sum in 32 bits.
constexpr int32_t kBoxMaxSteps = 8000;
// Dynamic LDS of a block: with the static part two blocks take 160 KB.
constexpr int32_t kBoxLdsBytes = 70 * 1024;

// A word of a line that has ended (stops move like stays).
constexpr uint32_t kWordStop = 0x11111111u * kMoveStop;

// Row stride of a box of w columns, == 8 (mod 32) elements: the 64 lanes of an
// 8 x 8 square of pixels read from distinct banks.
__device__ __forceinline__ int32_t box_stride(int32_t w) { return w + ((8 - w) & 31); }

// Two 16-bit integers: x = row, y = column, relative to a tile's origin.
typedef int16_t Pair __attribute__((ext_vector_type(2)));
__device__ __forceinline__ Pair pair_of(int32_t bits) { return __builtin_bit_cast(Pair, bits); }
__device__ __forceinline__ int32_t bits_of(Pair p) { return __builtin_bit_cast(int32_t, p); }

// Smallest and largest row and column visited (ReplayBounds).
struct Bounds {
  Pair lo, hi;
};
__device__ __forceinline__ Bounds no_bounds() {
  return {pair_of(0x7FFF7FFF), pair_of(static_cast<int32_t>(0x80008000u))};
}
__device__ __forceinline__ Bounds unite(const Bounds& a, const Bounds& b) {
  return {__builtin_elementwise_min(a.lo, b.lo), __builtin_elementwise_max(a.hi, b.hi)};
}

// United over each row of 16 lanes, by rotations within it (all lanes active).
template <int N>
__device__ __forceinline__ Bounds rotated(const Bounds& b) {
  return {pair_of(__builtin_amdgcn_mov_dpp(bits_of(b.lo), 0x120 + N, 15, 15, false)),
          pair_of(__builtin_amdgcn_mov_dpp(bits_of(b.hi), 0x120 + N, 15, 15, false))};
}
__device__ __forceinline__ Bounds unite_rows(Bounds b) {
  b = unite(b, rotated<8>(b));
  b = unite(b, rotated<4>(b));
  b = unite(b, rotated<2>(b));
  return unite(b, rotated<1>(b));
}

// A line's bounds in one direction, in quarter pixels: of its positions after
// every word of 8 steps (and of its start).  Between two of them it strays at
// most 4 pixels further.  Stay and stop codes do not move, and an edge step
// moves on (unwrapped coordinates).
struct LineBounds {
  int32_t row4, column4;  // 4 times the position
  Bounds b;
  __device__ __forceinline__ LineBounds(int32_t row, int32_t column)
      : row4(4 * row), column4(4 * column) {
    b.lo.x = b.hi.x = static_cast<int16_t>(row4);
    b.lo.y = b.hi.y = static_cast<int16_t>(column4);
  }
  // A word's moves along an axis are one dot product of 8 signed nibbles:
  // 1 where the step goes along it, times -4 or 4.
  __device__ __forceinline__ void walk(uint32_t word) {
    const uint32_t moved = ~(word >> 3) & 0x11111111u, axis_y = word >> 1;
    const int32_t sign4 = static_cast<int32_t>(((word << 1) & 0x88888888u) | 0x44444444u);
    row4 = __builtin_amdgcn_sdot8(static_cast<int32_t>(moved & axis_y), sign4, row4, false);
    column4 = __builtin_amdgcn_sdot8(static_cast<int32_t>(moved & ~axis_y), sign4, column4, false);
    const Pair at = pair_of(static_cast<int32_t>(__builtin_amdgcn_perm(
        static_cast<uint32_t>(column4), static_cast<uint32_t>(row4), 0x05040100u)));
    b = unite(b, {at, at});
  }
};

// at + the sign-extended lower or upper half of d, in one instruction.
__device__ __forceinline__ uint32_t add_low(uint32_t at, uint32_t d) {
  uint32_t r;
  asm("v_add_u32_sdwa %0, %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD "
      "src1_sel:WORD_0"
      : "=v"(r)
      : "v"(at), "v"(d));
  return r;
}
__device__ __forceinline__ uint32_t add_high(uint32_t at, uint32_t d) {
  uint32_t r;
  asm("v_add_u32_sdwa %0, %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD "
      "src1_sel:WORD_1"
      : "=v"(r)
      : "v"(at), "v"(d));
  return r;
}

// The four LDS byte deltas of a box as 16-bit entries for v_perm_b32: entry
// k at byte 2 k, picked by the code 2 k (kMoveXPlus, kMoveYPlus, kMoveXMinus,
// kMoveYMinus); the stay code 8 picks the sign bytes of the first two, zero.
struct MoveTable {
  uint32_t plus, minus;
  __device__ __forceinline__ MoveTable(int32_t elem, int32_t row_bytes)
      : plus(lane_copy(static_cast<uint32_t>(elem) | (static_cast<uint32_t>(row_bytes) << 16))),
        minus(lane_copy((static_cast<uint32_t>(-elem) & 0xFFFFu) |
                        (static_cast<uint32_t>(-row_bytes) << 16))) {}
};

// The 8 positions of a word's steps from `at`, which moves on to the last.
// Decoding on the VALU (9 issue cycles a step) instead of by a table in LDS
// leaves the LDS pipe, which bounds the walk, to the gathers.
__device__ __forceinline__ void decode_word(uint32_t word, const MoveTable& t, uint32_t& at,
                                            uint32_t (&pos)[8]) {
  static_assert(kMoveXPlus == 0 && kMoveYPlus == 2 && kMoveXMinus == 4 && kMoveYMinus == 6 &&
                    kMoveStay == 8 && kMoveStop == (kMoveStay | kMoveEdge),
                "selectors of MoveTable");
  const uint32_t even = (word >> 4) & 0x0E0E0E0Eu;  // steps 0, 2, 4, 6 in bytes 3 .. 0
  const uint32_t odd = word & 0x0E0E0E0Eu;          // steps 1, 3, 5, 7
  const uint32_t even1 = even | 0x01010101u, odd1 = odd | 0x01010101u;
  // selectors (low byte, high byte) of two steps, then their two deltas
  const uint32_t d02 = __builtin_amdgcn_perm(t.minus, t.plus,
                                             __builtin_amdgcn_perm(even1, even, 0x06020703u));
  const uint32_t d13 = __builtin_amdgcn_perm(t.minus, t.plus,
                                             __builtin_amdgcn_perm(odd1, odd, 0x06020703u));
  const uint32_t d46 = __builtin_amdgcn_perm(t.minus, t.plus,
                                             __builtin_amdgcn_perm(even1, even, 0x04000501u));
  const uint32_t d57 = __builtin_amdgcn_perm(t.minus, t.plus,
                                             __builtin_amdgcn_perm(odd1, odd, 0x04000501u));
  pos[0] = add_low(at, d02);
  pos[1] = add_low(pos[0], d13);
  pos[2] = add_high(pos[1], d02);
  pos[3] = add_high(pos[2], d13);
  pos[4] = add_low(pos[3], d46);
  pos[5] = add_low(pos[4], d57);
  pos[6] = add_high(pos[5], d46);
  pos[7] = add_high(pos[6], d57);
  at = pos[7];
}

template <typename T>
__device__ __forceinline__ T lds_at(uint32_t address) {
  typedef const T __attribute__((address_space(3))) lds_t;
  return *reinterpret_cast<lds_t*>(address);
}

// move_delta without branches (the steps outside the LDS are unrolled).
__device__ __forceinline__ uint32_t image_delta(uint32_t code, const FieldGeom& g, uint32_t elem) {
  const bool y = (code & kMoveAxisY) != 0;
  const uint32_t unit = y ? static_cast<uint32_t>(g.nx) * elem : elem;
  const uint32_t span = static_cast<uint32_t>(y ? 1 - g.ny : 1 - g.nx) * unit;
  const uint32_t d = (code & kMoveEdge) != 0 ? span : unit;
  return (code & kMoveStay) != 0 ? 0u : (code & kMoveNeg) != 0 ? 0u - d : d;
}

// Direct loads of 16 or 4 bytes per lane from `at` + `row` (uniform) in a
// buffer to consecutive LDS from `lds` (uniform).
typedef void __attribute__((address_space(3))) lds_void;
__device__ __forceinline__ void quads_to_lds(__amdgpu_buffer_rsrc_t rsrc, unsigned char* lds,
                                             uint32_t at) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)lds, 16, at, 0, 0, 0);
}
__device__ __forceinline__ void dwords_to_lds(__amdgpu_buffer_rsrc_t rsrc, unsigned char* lds,
                                              uint32_t at, uint32_t row) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)lds, 4, at, row, 0, 0);
}

// A box of lines in one direction: its origin relative to the
// tile, its size, and the row stride it is staged with, in elements.
struct Box {
  int32_t r_lo, c_lo, rows, columns, stride;
  __device__ __forceinline__ explicit Box(const Bounds& b)
      : r_lo(b.lo.x), c_lo(b.lo.y), rows(b.hi.x - b.lo.x + 1), columns(b.hi.y - b.lo.y + 1),
        stride(box_stride(columns)) {}
  __device__ __forceinline__ int32_t elems() const { return rows * stride; }
};

// What a tile stages for its lines of one direction: a box and the waves that
// it holds all lines of.
struct Staged {
  Bounds b;
  uint32_t waves;
};

}  // namespace

// A tile's boxes in memory: of its forward, then of its backward lines; with
// FIRST the block finds and stores them.
template <typename T, bool FMA, bool FIRST>
__global__ __launch_bounds__(kBoxThreads, 8) void lic_replay_box(
    const T* __restrict__ x, const T* __restrict__ kernel, int32_t klen, FieldGeom g, TileMap m,
    T* __restrict__ out, const uint4* __restrict__ codes,
    ReplayBounds* __restrict__ bounds) {
  constexpr int32_t elem = static_cast<int32_t>(sizeof(T));
  constexpr int32_t box_elems = kBoxLdsBytes / elem;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ ReplayBounds of_waves[FIRST ? kBoxWaves : 1][2];
  const int32_t tid = threadIdx.x, lane = tid & 63;
  const int32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int32_t ty, tx;
  tile_of_block(blockIdx.x, m, ty, tx);
  // a wave takes an 8 x 8 square of the tile
  const int32_t py = ((wave >> 2) << 3) | (lane >> 3), px = ((wave & 3) << 3) | (lane & 7);
  const int32_t i_tile = ty * kBoxTile, j_tile = tx * kBoxTile;
  const int64_t np = static_cast<int64_t>(g.ny) * g.nx;
  const int32_t kmid = klen / 2;
  const int32_t n_fwd = klen - 1 - kmid, n_bwd = kmid;  // n_fwd <= n_bwd
  const int32_t ch_fwd = chunks_of(n_fwd), ch_all = ch_fwd + chunks_of(n_bwd);
  const bool inside = i_tile + py < g.ny && j_tile + px < g.nx;
  // a lane past the image reads pixel 0's record and drops what it gets
  const int64_t p = inside ? static_cast<int64_t>(i_tile + py) * g.nx + (j_tile + px) : 0;
  T acc = macc<FMA>(kernel[kmid], x[p], T(0));
  if (ch_all == 0) {  // uniform: a kernel of one tap has no record
    if (inside) out[p] = acc;
    return;
  }
  ReplayBounds* const tile = bounds + 2 * (static_cast<int64_t>(ty) * m.tiles_x + tx);
  Staged tiles[2];
  if constexpr (FIRST) {
    const uint4* record = codes + p;
    for (int32_t dir = 0; dir < 2; ++dir) {
      LineBounds line(py, px);
      bool alive = inside;
      for (int32_t ch = dir ? ch_all - ch_fwd : ch_fwd; ch > 0; ch -= 2) {  // two loads in flight
        const uint4 c[2] = {record[0], record[ch > 1 ? np : 0]};
        record += ch > 1 ? 2 * np : np;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          if (k == 4 && ch == 1) break;  // uniform
          const uint4& w = c[k / 4];
          const uint32_t word = k % 4 == 0 ? w.x : k % 4 == 1 ? w.y : k % 4 == 2 ? w.z : w.w;
          line.walk(alive ? word : kWordStay);
          alive = alive && !group_has_stop(word);
        }
      }
      Bounds b = inside ? line.b : no_bounds();
      b = unite_rows(b);
#pragma unroll
      for (int off = 32; off > 8; off >>= 1)
        b = unite(b, {pair_of(__shfl_xor(bits_of(b.lo), off)),
                      pair_of(__shfl_xor(bits_of(b.hi), off))});
      if (lane == 0) of_waves[wave][dir] = ReplayBounds{bits_of(b.lo), bits_of(b.hi), 0, 0};
    }
    __syncthreads();
    // lanes 0..15 the waves' forward bounds, 16..31 the backward ones
    static_assert(kBoxWaves == 16, "a row of lanes");
    const ReplayBounds mine = of_waves[lane & 15][lane >> 4 & 1];
    const Bounds in_rows = unite_rows({pair_of(mine.lo), pair_of(mine.hi)});
    // to pixels, grown by 4 (LineBounds), to 16-byte aligned columns (stage)
    auto in_pixels = [](Bounds b) {
      b.lo = (b.lo >> static_cast<int16_t>(2)) - static_cast<int16_t>(4);
      b.hi = (b.hi >> static_cast<int16_t>(2)) + static_cast<int16_t>(4);
      b.lo.y &= ~3;
      return b;
    };
    auto in_lane = [](const Bounds& b, int32_t l) {
      return Bounds{pair_of(__builtin_amdgcn_readlane(bits_of(b.lo), l)),
                    pair_of(__builtin_amdgcn_readlane(bits_of(b.hi), l))};
    };
    tiles[0] = {in_pixels(in_lane(in_rows, 0)), (1u << kBoxWaves) - 1};
    tiles[1] = {in_pixels(in_lane(in_rows, 16)), (1u << kBoxWaves) - 1};
    const bool fits[2] = {Box(tiles[0].b).elems() <= box_elems,
                          Box(tiles[1].b).elems() <= box_elems};
    if (!fits[0] || !fits[1]) {  // uniform
      // A direction whose box does not fit: the waves taken one after the
      // other if they still fit, each lane of a row in an order of its own
      // (by the wave's number xor the lane's); the order that takes most.
      Bounds some = no_bounds();
      uint32_t waves = 0;
      for (int32_t k = 0; k < kBoxWaves; ++k) {
        const int32_t w = k ^ (lane & 15);
        const ReplayBounds r = of_waves[w][lane >> 4 & 1];
        const Bounds wider = unite(some, {pair_of(r.lo), pair_of(r.hi)});
        const bool take = r.hi != bits_of(no_bounds().hi) &&
                          Box(in_pixels(wider)).elems() <= box_elems;
        some = take ? wider : some;
        waves |= take ? 1u << w : 0u;
      }
      const int32_t key = __builtin_popcount(waves) * 16 + (lane & 15);
      int32_t best = max(key, __builtin_amdgcn_mov_dpp(key, 0x128, 15, 15, false));
      best = max(best, __builtin_amdgcn_mov_dpp(best, 0x124, 15, 15, false));
      best = max(best, __builtin_amdgcn_mov_dpp(best, 0x122, 15, 15, false));
      best = max(best, __builtin_amdgcn_mov_dpp(best, 0x121, 15, 15, false));
#pragma unroll
      for (int dir = 0; dir < 2; ++dir) {
        if (fits[dir]) continue;
        const int32_t l = 16 * dir + (__builtin_amdgcn_readlane(best, 16 * dir) & 15);
        tiles[dir].waves =
            static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int32_t>(waves), l));
        // no wave fits: nothing is staged, whatever the bounds
        tiles[dir].b = in_pixels(
            tiles[dir].waves ? in_lane(some, l)
                             : in_lane({pair_of(mine.lo), pair_of(mine.hi)}, 16 * dir));
      }
    }
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
      if (tid == 0)
        tile[dir] = ReplayBounds{bits_of(tiles[dir].b.lo), bits_of(tiles[dir].b.hi),
                                 tiles[dir].waves, 0};
    }
  } else {
#pragma unroll
    for (int dir = 0; dir < 2; ++dir)
      tiles[dir] = {{pair_of(__builtin_amdgcn_readfirstlane(tile[dir].lo)),
                     pair_of(__builtin_amdgcn_readfirstlane(tile[dir].hi))},
                    static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(tile[dir].waves))};
  }
  // Stages a box at element `first` of the dynamic LDS with direct memory ->
  // LDS loads, wrapped modulo the image size (one add or subtract where the
  // box lies within one image size of the image).  With x 16-byte aligned
  // and nx a multiple of 16 bytes (a box then starts at such a column, and
  // quads of elements do not straddle the wrap), 16 bytes a lane, the box's
  // quads dealt over the block: a lane finds its quad's row by the
  // reciprocal of the quads per row (exact for fewer than 2^20 quads).
  // Otherwise a wave copies rows of 64 dwords, the row on the scalar unit.
  constexpr int32_t kQuad = 16 / elem;
  const bool quads = (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && g.nx % kQuad == 0;
  const ImageWalk<T> image(x, np);
  auto stage = [&](const Box& box, int32_t first) {
    const int32_t i_box = i_tile + box.r_lo, j_box = j_tile + box.c_lo;
    const bool once = i_box >= -g.ny && int64_t{i_box} + box.rows <= 2 * int64_t{g.ny} &&
                      j_box >= -g.nx && int64_t{j_box} + box.stride <= 2 * int64_t{g.nx};
    auto wrap = [&](int32_t c, int32_t n) {  // `once` is uniform
      return once ? (c < 0 ? c + n : (c >= n ? c - n : c)) : wrap_index(c, n);
    };
    const int32_t row_quads = box.stride / kQuad, count = box.rows * row_quads;
    const float inverse = 1.0f / static_cast<float>(row_quads);
    if (quads && i_box >= 0 && i_box + box.rows <= g.ny && j_box >= 0 &&
        j_box + box.stride <= g.nx) {
      // within the image: element offset of quad n = its place in the box plus
      // what the rows above skip
      const uint32_t base = (static_cast<uint32_t>(i_box) * static_cast<uint32_t>(g.nx) +
                             static_cast<uint32_t>(j_box)) * elem;
      const uint32_t skip = static_cast<uint32_t>(g.nx - box.stride) * elem;
      for (int32_t k = wave * 64; k < count; k += kBoxThreads) {
        const int32_t n = k + lane;
        const uint32_t a = static_cast<uint32_t>((static_cast<float>(n) + 0.5f) * inverse);
        if (n < count)
          quads_to_lds(image.rsrc, smem + first * elem + k * 16,
                       base + static_cast<uint32_t>(n) * 16 + a * skip);
      }
    } else if (quads) {
      for (int32_t k = wave * 64; k < count; k += kBoxThreads) {
        const int32_t n = k + lane;
        const int32_t a = static_cast<int32_t>((static_cast<float>(n) + 0.5f) * inverse);
        const int32_t i = wrap(i_box + a, g.ny);
        const int32_t j = wrap(j_box + (n - a * row_quads) * kQuad, g.nx);
        if (n < count)
          quads_to_lds(image.rsrc, smem + first * elem + k * 16,
                       (static_cast<uint32_t>(i) * static_cast<uint32_t>(g.nx) +
                        static_cast<uint32_t>(j)) * elem);
      }
    } else {
      constexpr int32_t kDw = elem / 4;        // dwords per element
      constexpr int32_t kSegElems = 64 / kDw;  // elements per copy
      for (int32_t s = 0; s < box.columns; s += kSegElems) {
        const int32_t e = s + lane / kDw;  // element of the box row
        const uint32_t column =
            static_cast<uint32_t>(wrap(j_box + e, g.nx)) * elem + 4 * (lane % kDw);
        if (e < box.columns)
          for (int32_t a = wave; a < box.rows; a += kBoxWaves)
            dwords_to_lds(image.rsrc, smem + (first + a * box.stride + s) * elem, column,
                          static_cast<uint32_t>(wrap(i_box + a, g.ny)) *
                              static_cast<uint32_t>(g.nx) * elem);
      }
    }
  };
  auto staged = [&]() {
    __builtin_amdgcn_s_waitcnt(0);  // this wave's copies have landed
    __syncthreads();
  };
  // Walks the line through a direction of nsteps >= 1 steps, whose first
  // chunk `next` is at `record`: from LDS address `at` in a staged box with
  // rows of row_bytes (in_lds: std::true_type), or from byte `at` of the image.
  auto walk = [&](auto forward, auto in_lds, int32_t nsteps, const uint4* record, uint4 next,
                  uint32_t at, int32_t row_bytes) {
    constexpr bool kForward = decltype(forward)::value, kLds = decltype(in_lds)::value;
    bool alive = inside;
    // in the constant address space: scalar loads
    typedef const T __attribute__((address_space(4))) const_t;
    const_t* taps = (const_t*)(kernel + (kForward ? kmid + 1 : kmid - 8));
    const MoveTable table(elem, row_bytes);
    for (int32_t left = nsteps; left > 0;) {
      uint4 words = next;
      if (left > kChunkSteps) next = *(record += np);
#pragma unroll(kLds ? 4 : 1)
      for (int k = 0; k < 4; ++k) {
        if (left <= 0) break;  // uniform
        // the weights of the 8 steps, in ascending order
        T kw[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) kw[kForward ? q : 7 - q] = taps[q];
        taps += kForward ? 8 : -8;
        const uint32_t word = alive ? words.x : kWordStop;
        words = make_uint4(words.y, words.z, words.w, 0);
        T xv[8];
        if constexpr (kLds) {
          uint32_t pos[8];
          decode_word(word, table, at, pos);
#pragma unroll
          for (int q = 0; q < 8; ++q) xv[q] = lds_at<T>(pos[q]);
        } else {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            at += image_delta(move_code(word, q), g, elem);
            xv[q] = image(at);
          }
        }
        if (left >= 8 && __builtin_amdgcn_ballot_w64(group_has_stop(word)) == 0) {
#pragma unroll
          for (int q = 0; q < 8; ++q) acc = macc<FMA>(kw[q], xv[q], acc);
        } else {
          const int32_t valid = steps_before_stop(word), lim = min(valid, left);
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const T next_acc = macc<FMA>(kw[q], xv[q], acc);
            acc = q < lim ? next_acc : acc;
          }
          alive = valid == 8;
        }
        left -= 8;
      }
    }
  };
  auto direction = [&](auto forward, int32_t nsteps, const uint4* record, uint4 next,
                       const Box& box, bool fits, uint32_t lds) {
    if (fits) {  // uniform in the wave; a lane past the image stays at the box's first element
      const int32_t start = (py - box.r_lo) * box.stride + (px - box.c_lo);
      walk(forward, std::true_type{}, nsteps, record, next,
           lds + static_cast<uint32_t>(inside ? start * elem : 0), box.stride * elem);
    } else {
      walk(forward, std::false_type{}, nsteps, record, next, static_cast<uint32_t>(p * elem), 0);
    }
  };

  const Box fwd(tiles[0].b), bwd(tiles[1].b);
  const bool stage_fwd = n_fwd > 0 && tiles[0].waves != 0, stage_bwd = tiles[1].waves != 0;
  const int32_t need_fwd = stage_fwd ? fwd.elems() : 0, need_bwd = stage_bwd ? bwd.elems() : 0;
  typedef unsigned char __attribute__((address_space(3))) lds_bytes;
  const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_bytes*)smem));
  const uint4* const rec_fwd = codes + p;
  const uint4* const rec_bwd = rec_fwd + static_cast<int64_t>(ch_fwd) * np;
  // Both directions' boxes at once (one wait, one barrier) if they fit
  // together, else one after the other.
  const bool both = need_fwd + need_bwd <= box_elems;
  const uint4 next_fwd = *rec_fwd, next_bwd = *rec_bwd;
  if (n_fwd > 0) {
    if (stage_fwd) stage(fwd, 0);
    if (both && stage_bwd) stage(bwd, need_fwd);
    staged();
    direction(std::true_type{}, n_fwd, rec_fwd, next_fwd, fwd,
              (tiles[0].waves >> wave & 1) != 0, lds);
    if (!both) __syncthreads();  // the LDS is staged again next
  }
  if (!(both && n_fwd > 0)) {
    if (stage_bwd) stage(bwd, 0);
    staged();
  }
  direction(std::false_type{}, n_bwd, rec_bwd, next_bwd, bwd, (tiles[1].waves >> wave & 1) != 0,
            lds + static_cast<uint32_t>((both ? need_fwd : 0) * elem));
  if (inside) out[p] = acc;
}

size_t replay_bounds_bytes(const FieldGeom& g) {
  const int64_t tiles = ((int64_t{g.ny} + kBoxTile - 1) / kBoxTile) *
                        ((int64_t{g.nx} + kBoxTile - 1) / kBoxTile);
  return 2 * sizeof(ReplayBounds) * static_cast<size_t>(tiles);
}

template <typename T>
bool box_replay_fits(int32_t klen, const FieldGeom& g) {
  return klen / 2 <= kBoxMaxSteps &&
         fits_buffer(static_cast<int64_t>(g.ny) * g.nx * static_cast<int64_t>(sizeof(T))) &&
         kBoxLdsBytes + 1024 <= lds_replay_limit_bytes();
}

template <typename T>
hipError_t launch_replay_box(const T* x, const T* kernel, int32_t klen, const FieldGeom& g,
                             int profile, T* out, const uint4* codes, ReplayBounds* bounds,
                             bool first, hipStream_t stream) {
  if (!bounds || !box_replay_fits<T>(klen, g)) return hipErrorInvalidValue;
  TileMap m;
  m.wave_w_log2 = 3;
  m.tiles_x = (g.nx + kBoxTile - 1) / kBoxTile;
  m.tiles_y = (g.ny + kBoxTile - 1) / kBoxTile;
  m.n_tiles = m.tiles_x * m.tiles_y;
  m.per_xcd = m.n_tiles / kXcds;
  m.rem_xcd = m.n_tiles % kXcds;
  m.band = 8;
  const bool fma = (profile & 1) != 0;
  auto* fn = first ? (fma ? &lic_replay_box<T, true, true> : &lic_replay_box<T, false, true>)
                   : (fma ? &lic_replay_box<T, true, false> : &lic_replay_box<T, false, false>);
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kBoxLdsBytes);
  (void)hipGetLastError();  // the attribute is advisory on this target
  hipLaunchKernelGGL(fn, dim3(m.n_tiles), dim3(kBoxThreads), kBoxLdsBytes, stream, x, kernel, klen,
                     g, m, out, codes, bounds);
  return hipGetLastError();
}

#define RLIC_BOX_INSTANTIATE(T)                                                                  \
  template bool box_replay_fits<T>(int32_t, const FieldGeom&);                                   \
  template hipError_t launch_replay_box<T>(const T*, const T*, int32_t, const FieldGeom&, int,   \
                                           T*, const uint4*, ReplayBounds*, bool, hipStream_t);

RLIC_BOX_INSTANTIATE(float)
RLIC_BOX_INSTANTIATE(double)

}  // namespace rlic
