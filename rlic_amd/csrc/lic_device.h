// Device-side building blocks of the streamline kernels (gfx950 / CDNA4).
//
// Semantics follow the reference's per-step rule (src/lib.rs:157-273,
// 304-362) exactly; the arithmetic is literal so that results are
// bit-identical to the reference's CPU arithmetic:
//   * fused multiply-add only where the reference calls `mul_add`
//     (src/lib.rs:177, 231, 359, 382), selected by the FMA template flag;
//   * every other product is a separate rounded multiply (the library is
//     compiled with -ffp-contract=off);
//   * divisions are IEEE correctly rounded (hipcc's default fp32 division
//     and the fp64 div_scale/div_fmas/div_fixup sequence), denormals kept.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rlic {

// One packed field cell: the vector (u, v) at the cell and the texture
// value x.  A streamline step reads the texture at the cell it enters and,
// on the next step, the vector at that same cell, so packing the three
// values turns three gathers per step into one 16-byte (fp32) or two
// adjacent 16-byte (fp64) loads from a single cache line.
template <typename T>
struct Cell;

template <>
struct __align__(16) Cell<float> {
  float u, v, x, pad;
};

template <>
struct __align__(32) Cell<double> {
  double u, v, x, pad;
};

template <typename T>
struct CellVal {
  T u, v, x;
  T pad;  // a guarded array's jump (see pad_bits)
};

// The jump in cells that a guarded cell array keeps in a cell's pad slot
// (low 32 bits of its bit pattern; 0 in image cells).
__device__ __forceinline__ uint32_t pad_bits(float pad) { return __builtin_bit_cast(uint32_t, pad); }
__device__ __forceinline__ uint32_t pad_bits(double pad) {
  return static_cast<uint32_t>(__builtin_bit_cast(uint64_t, pad));
}
__host__ __device__ inline float jump_pad(int32_t jump, float*) {
  return __builtin_bit_cast(float, jump);
}
__host__ __device__ inline double jump_pad(int32_t jump, double*) {
  return __builtin_bit_cast(double, static_cast<uint64_t>(static_cast<uint32_t>(jump)));
}

__device__ __forceinline__ CellVal<float> load_cell(const Cell<float>* __restrict__ p,
                                                    uint32_t idx) {
  const float4 c = *reinterpret_cast<const float4*>(p + idx);
  return {c.x, c.y, c.z, c.w};
}

__device__ __forceinline__ CellVal<double> load_cell(const Cell<double>* __restrict__ p,
                                                     uint32_t idx) {
  const double2* q = reinterpret_cast<const double2*>(p + idx);
  const double2 a = q[0];
  const double2 b = q[1];
  return {a.x, a.y, b.x, b.y};
}

// ---------------------------------------------------------------------------
// Gathers.  With BUF, arrays are addressed through a raw buffer resource and
// a 32-bit byte offset (one VALU add per address, hardware range check: an
// out-of-range read returns 0 instead of faulting); usable when the array
// spans fewer than 2^32 bytes.  Otherwise 64-bit global addresses are used.
// ---------------------------------------------------------------------------
// gfx9 raw-buffer descriptor word 3 (no swizzle, dword data format).
constexpr int32_t kBufferWord3 = 0x00020000;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                           kBufferWord3);
}

__device__ __forceinline__ float buf_load(const __amdgpu_buffer_rsrc_t r, uint32_t off, float*) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ double buf_load(const __amdgpu_buffer_rsrc_t r, uint32_t off,
                                           double*) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}

// The b64/b128 builtins return GCC vector_size vectors of unsigned int;
// they are bit-cast whole (bit-casting a subscripted lane miscompiles).
// Structured buffer load of 16 bytes at `offset` of element `index` (an LLVM
// intrinsic that has no builtin of its own).
typedef uint32_t Quad __attribute__((ext_vector_type(4)));
__device__ Quad struct_buffer_load(__amdgpu_buffer_rsrc_t r, int32_t index, int32_t offset,
                                   int32_t soffset,
                                   int32_t aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.v4i32");
__device__ __forceinline__ CellVal<float> buf_load_cell(const __amdgpu_buffer_rsrc_t r,
                                                        uint32_t index, float*) {
  const float4 c = __builtin_bit_cast(float4, struct_buffer_load(r, index, 0, 0, 0));
  return {c.x, c.y, c.z, c.w};
}
__device__ __forceinline__ CellVal<double> buf_load_cell(const __amdgpu_buffer_rsrc_t r,
                                                         uint32_t index, double*) {
  const double2 uv = __builtin_bit_cast(double2, struct_buffer_load(r, index, 0, 0, 0));
  const double2 xp = __builtin_bit_cast(double2, struct_buffer_load(r, index, 16, 0, 0));
  return {uv.x, uv.y, xp.x, xp.y};
}

// Cell gather at the cell index `pos`.  With BUF the buffer is a structured
// one (its stride the cell size, its range counted in cells), so the address
// unit multiplies the index: positions, steps and jumps are plain slot
// counts, and a jump is one 2-cycle add instead of a 4-cycle shift-add.
template <typename T, bool BUF>
struct CellGather {
  const Cell<T>* base;
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ CellGather(const Cell<T>* p, int64_t n) : base(p) {
    if constexpr (BUF)
      rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<Cell<T>*>(p), (short)sizeof(Cell<T>),
                                               static_cast<int>(n), kBufferWord3);
  }
  static constexpr uint32_t unit = 1u;
  __device__ __forceinline__ CellVal<T> operator()(uint32_t pos) const {
    if constexpr (BUF) {
      return buf_load_cell(rsrc, pos, static_cast<T*>(nullptr));
    } else {
      return load_cell(base, pos);
    }
  }
};

// Texture gather at `pos`: a byte offset (BUF) or an element index (global).
template <typename T, bool BUF>
struct ValueGather {
  const T* base;
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ ValueGather(const T* p, int64_t n) : base(p) {
    if constexpr (BUF) rsrc = make_rsrc(p, static_cast<uint32_t>(n * sizeof(T)));
  }
  static constexpr uint32_t unit = BUF ? static_cast<uint32_t>(sizeof(T)) : 1u;
  __device__ __forceinline__ T operator()(uint32_t pos) const {
    if constexpr (BUF) {
      return buf_load(rsrc, pos, static_cast<T*>(nullptr));
    } else {
      return base[pos];
    }
  }
};

// A copy of a (wave-uniform) value that the compiler must treat as
// lane-varying: loop-invariant select operands kept this way live in VGPRs,
// so each select is one v_cndmask instead of a scalar-to-vector move (a
// VALU instruction reads at most one scalar register) or a branch.
__device__ __forceinline__ uint32_t lane_copy(uint32_t x) {
  uint32_t r;
  asm("v_mov_b32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

// Keeps the computation of x where it is written: without it the compiler
// moves a group's sums past the group's closing branch, and with them (global
// loads) a second load of each cell for its texture value, or (masks of the
// move codes) the registers that hold what they are made from.
template <typename T>
__device__ __forceinline__ void keep_in_step(T& x) {
  asm volatile("" : "+v"(x));
}

// x with its sign bit xor-ed with `sign` (0 or 0x80000000; for double it
// applies to the top word): -x when the bit is set, bit for bit the
// negation, as one integer instruction.
__device__ __forceinline__ float xor_sign(float x, uint32_t sign) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) ^ sign);
}
__device__ __forceinline__ double xor_sign(double x, uint32_t sign) {
  return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, x) ^ (uint64_t{sign} << 32));
}

__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float abs_t(float a) { return __builtin_fabsf(a); }
__device__ __forceinline__ double abs_t(double a) { return __builtin_fabs(a); }
__device__ __forceinline__ bool isnan_t(float a) { return __builtin_isnan(a); }
__device__ __forceinline__ bool isnan_t(double a) { return __builtin_isnan(a); }

template <typename T>
__device__ __forceinline__ T inf_t() {
  return static_cast<T>(__builtin_huge_valf());
}

// `a.mul_add(b, c)` with the fma feature, else `c += a * b` (two roundings).
template <bool FMA, typename T>
__device__ __forceinline__ T macc(T a, T b, T c) {
  if constexpr (FMA) {
    return fma_t(a, b, c);
  } else {
    const T prod = a * b;
    return c + prod;
  }
}

// Lane masks (0 or all ones) in VGPRs, and selections by them: v_bitop3
// issues in half the cycles of v_cndmask and v_bfi, and written as builtins
// they are not turned back into compares and selects.
__device__ __forceinline__ uint32_t sign_mask(float x) {
  return static_cast<uint32_t>(__builtin_bit_cast(int32_t, x) >> 31);
}
__device__ __forceinline__ uint32_t sign_mask(double x) {
  return static_cast<uint32_t>(static_cast<int32_t>(__builtin_bit_cast(uint64_t, x) >> 32) >> 31);
}
template <uint32_t TABLE>
__device__ __forceinline__ uint32_t bitop3(uint32_t a, uint32_t b, uint32_t c) {
  return static_cast<uint32_t>(__builtin_amdgcn_bitop3_b32(a, b, c, TABLE));
}
// where the mask is set a, else b
__device__ __forceinline__ uint32_t pick(uint32_t m, uint32_t a, uint32_t b) {
  return bitop3<0xCA>(m, a, b);
}
struct Words {
  uint32_t lo, hi;
};
__device__ __forceinline__ float pick(uint32_t m, float a, float b) {
  return __builtin_bit_cast(float, pick(m, __builtin_bit_cast(uint32_t, a),
                                        __builtin_bit_cast(uint32_t, b)));
}
__device__ __forceinline__ double pick(uint32_t m, double a, double b) {
  const Words x = __builtin_bit_cast(Words, a), y = __builtin_bit_cast(Words, b);
  return __builtin_bit_cast(double, Words{pick(m, x.lo, y.lo), pick(m, x.hi, y.hi)});
}
// 2 where the mask is clear (FLIP: set), else +0
template <bool FLIP>
__device__ __forceinline__ float two_where(uint32_t m, float*) {
  return __builtin_bit_cast(float, bitop3<FLIP ? 0xC0 : 0x30>(0x40000000u, m, m));
}
template <bool FLIP>
__device__ __forceinline__ double two_where(uint32_t m, double*) {
  return __builtin_bit_cast(double, Words{0u, bitop3<FLIP ? 0xC0 : 0x30>(0x40000000u, m, m)});
}
// x where the mask is clear (FLIP: set), else +0
template <bool FLIP>
__device__ __forceinline__ uint32_t keep_bits(uint32_t x, uint32_t m) {
  return bitop3<FLIP ? 0xC0 : 0x30>(x, m, m);
}
template <bool FLIP>
__device__ __forceinline__ float keep_where(float x, uint32_t m) {
  return __builtin_bit_cast(float, keep_bits<FLIP>(__builtin_bit_cast(uint32_t, x), m));
}
template <bool FLIP>
__device__ __forceinline__ double keep_where(double x, uint32_t m) {
  const Words w = __builtin_bit_cast(Words, x);
  return __builtin_bit_cast(double, Words{keep_bits<FLIP>(w.lo, m), keep_bits<FLIP>(w.hi, m)});
}
// 1 where the mask `neg` is set (FLIP: clear), else 0
template <bool FLIP>
__device__ __forceinline__ float edge_fraction(uint32_t neg, float*) {
  const uint32_t one = 0x3F800000u;
  return __builtin_bit_cast(float, bitop3<FLIP ? 0x0C : 0xC0>(neg, one, one));
}
template <bool FLIP>
__device__ __forceinline__ double edge_fraction(uint32_t neg, double*) {
  const uint32_t one = 0x3FF00000u;
  return __builtin_bit_cast(double, Words{0u, bitop3<FLIP ? 0x0C : 0xC0>(neg, one, one)});
}
// Time to reach the next cell edge along one axis (src/lib.rs:157-180).
// Correctly rounded division (IEEE round-to-nearest-even, denormals kept):
// hipcc's float and double division (v_div_scale / v_rcp / v_div_fmas /
// v_div_fixup).  A float quotient formed in double from a Newton-refined
// reciprocal and rounded once is also exact (8 instructions instead of 11)
// but measured slower on gfx950 (trace 3.54 ms vs 3.10 ms at 4096^2, L=129):
// the double-precision operations cost more issue cycles.
__device__ __forceinline__ float div_rn(float a, float b) { return a / b; }
__device__ __forceinline__ double div_rn(double a, double b) { return a / b; }

// `velocity` is never NaN here: NaN vectors end the streamline first
// (src/lib.rs:336-338).
template <typename T>
__device__ __forceinline__ T time_to_next_pixel(T velocity, T frac) {
  if (velocity > T(0)) return div_rn(T(1) - frac, velocity);
  if (velocity < T(0)) return -div_rn(frac, velocity);
  return inf_t<T>();
}

// The branchless rule divides this by the velocity: 1 + signum(velocity) is 0
// when the sign bit is set (also -0.0), else 2.  `sign` is the mask of that
// bit (FLIP: the opposite), which the caller uses otherwise too.
template <typename T, bool FMA, bool FLIP>
__device__ __forceinline__ T step_numerator(T frac, uint32_t sign) {
  return macc<FMA>(two_where<FLIP>(sign, static_cast<T*>(nullptr)), T(0.5) - frac, frac);
}

// Ranges of the step's short path (fast_group) and quick quotient
// (full_group).  A field is "wide" when a velocity component is infinite or
// nonzero below kMin / above kMax in magnitude (float: 2^-60 = 8.7e-19 to 2^40 =
// 1.1e12); the packing kernels look at every component and mark such a field
// (wide_mark), whose lines then take the divisions throughout: a limit on speed,
// not on results.
// Within these ranges and with numerators of at least numerator_key_min (or
// zero) the quotient and its remainder are normal numbers or exact, so no
// scaling is needed, and so are the products n |w| compared in fast_group
// wherever they are not below kProductMin.
template <typename T>
struct VelocityRange;
template <>
struct VelocityRange<float> {
  static constexpr float kMin = 0x1p-60f, kMax = 0x1p40f;
};
template <>
struct VelocityRange<double> {
  // With numerators of at least 2^-300 the times taken are at least 2^-450,
  // what they add to a fraction at least 2^-750 and a multiple of 2^-802, and
  // so are numerators: no quotient of one by up to 2^150 underflows.
  static constexpr double kMin = 0x1p-300, kMax = 0x1p150;
};

template <typename T>
__device__ __forceinline__ bool velocity_wide(T w) {
  const T a = abs_t(w);
  return a > VelocityRange<T>::kMax || (a < VelocityRange<T>::kMin && a != T(0));
}

// The mark of a wide field: the first word of its guarded array's corner
// cell (0, 0), which no step reaches.  Each packing of a field has its own
// `epoch`; a packing thread that sees a wide component stores the epoch
// there, so the word needs no clearing before (a stale word that happens to
// equal the epoch only costs the short path).
// In a captured graph the arguments are the same at every replay, so there the
// epoch is counted in the corner cell itself (argument kCountedEpoch): packing
// takes word 1 plus one and keeps it in word 2 for the traces, which compare
// with that and copy it back to word 1 (count_epoch).  No word is written in a
// launch that reads it, whatever they held before.  A launch that clears the
// mark instead took 5 us of a replay of 256^2 double, L = 65 (27 -> 33 us).
constexpr uint32_t kCountedEpoch = 0;

__device__ __forceinline__ uint32_t packing_epoch(const uint32_t* corner, uint32_t epoch) {
  return epoch != kCountedEpoch ? epoch : corner[1] + 1;
}

template <typename T>
__device__ __forceinline__ bool wide_mark(const Cell<T>* cells, uint32_t epoch) {
  const uint32_t* corner = reinterpret_cast<const uint32_t*>(cells);
  return corner[0] == (epoch != kCountedEpoch ? epoch : corner[2]);
}

// In a trace, `corner` null but for kCountedEpoch.
__device__ __forceinline__ void count_epoch(uint32_t* corner) {
  if (corner && blockIdx.x == 0 && threadIdx.x == 0) corner[1] = corner[2];
}

// The products n_x |v| and n_y |u| tell the order of the step times where they
// differ by more than this share of the second.  In float, with r = 2^-24: their
// difference is off by r at most; the times' roundings differ if the times do by
// 2 r; and the fractions stay in [0, 1] (fraction_usable) if the times differ by
// 4 r, what the roundings of the numerator, the time and the product add up to.
// 8 r leaves 7.  A closer pair is reported, and costs the steps done again: with
// 64 r, 1.6% of the chunks of a trace (4096^2, L = 129: 1.87 -> 1.83 ms).
__device__ __forceinline__ float near_tie(float*) { return 0x1p-21f; }
__device__ __forceinline__ double near_tie(double*) { return 0x1p-40; }

// Key of a numerator n >= 0 that puts zero last: below numerator_key_min
// for 0 < n < 2^-60 (float), 2^-300 (double).  A double key reads the top
// word only: fractions, and with them numerators, that start at zero or at
// least 2^-300 (fraction_usable) stay multiples of 2^-802 (VelocityRange).
__device__ __forceinline__ uint32_t numerator_key(float n) {
  return __builtin_bit_cast(uint32_t, n) - 1u;
}
__device__ __forceinline__ uint32_t numerator_key(double n) {
  return static_cast<uint32_t>(__builtin_bit_cast(uint64_t, n) >> 32) - 1u;
}
// |w|, or for a zero w far less than any other divisor: numerators that are not
// tiny over it exceed every quotient by a |w| within VelocityRange.
__device__ __forceinline__ float positive_divisor(float w) {
  return __builtin_amdgcn_fmed3f(abs_t(w), 0x1p-125f, inf_t<float>());
}
// The lanes with a nonzero numerator below what quotient_rn takes.
__device__ __forceinline__ uint64_t tiny_numerators(float n) {
  return __builtin_amdgcn_ballot_w64(n != 0.0f) & __builtin_amdgcn_ballot_w64(abs_t(n) < 0x1p-60f);
}
__device__ __forceinline__ uint32_t numerator_key_min(float*) { return ((127u - 60u) << 23) - 1u; }
__device__ __forceinline__ uint32_t numerator_key_min(double*) {
  return ((1023u - 300u) << 20) - 1u;
}

// Float products n |w| from here on have quotients n / |w'| that do not round to
// zero, for every |w'| up to kMax: 2 kMax^2 times the smallest number.
constexpr float kProductMin = 0x1p-68f;

// Fractions the short path starts from: in [0, 1], zero or at least 2^-300.
// It keeps them in [0, 1]: away from ties the step ends before the other
// axis' edge, and rounding is monotone.
__device__ __forceinline__ bool fraction_usable(float f) { return f >= 0.0f && f <= 1.0f; }
__device__ __forceinline__ bool fraction_usable(double f) {
  return f == 0.0 || (f >= 0x1p-300 && f <= 1.0);
}

__device__ __forceinline__ uint32_t top_word(float x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ uint32_t top_word(double x) { return __builtin_bit_cast(Words, x).hi; }
// x with its sign bit xor-ed with that of s
__device__ __forceinline__ float copy_sign_of(float x, float s) {
  return __builtin_bit_cast(float, bitop3<0x78>(__builtin_bit_cast(uint32_t, x),
                                                __builtin_bit_cast(uint32_t, s), 0x80000000u));
}
__device__ __forceinline__ double copy_sign_of(double x, double s) {
  const Words a = __builtin_bit_cast(Words, x), b = __builtin_bit_cast(Words, s);
  return __builtin_bit_cast(double, Words{a.lo, bitop3<0x78>(a.hi, b.hi, 0x80000000u)});
}
// n / d correctly rounded, for n, d >= 0 within the ranges above and d > 0:
// the refinement steps of the IEEE division (reciprocal, Newton, quotient,
// exact remainder, correction: Markstein 1990) without its scaling and
// special cases.  In float one Newton step and one correction do: every pair
// of 23-bit mantissas was tried on gfx950 against the remainder test (2^46
// pairs, none wrong: tests/test_quotient.py); scaling by powers of two is exact
// in between.  In
// double these are the steps of hipcc's own division.
__device__ __forceinline__ float quotient_rn(float n, float d) {
  const float y0 = __builtin_amdgcn_rcpf(d);
  const float y = fma_t(fma_t(-d, y0, 1.0f), y0, y0);
  const float q = n * y;
  return fma_t(fma_t(-d, q, n), y, q);
}
__device__ __forceinline__ double quotient_rn(double n, double d) {
  double y = __builtin_amdgcn_rcp(d);
  y = fma_t(fma_t(-d, y, 1.0), y, y);
  y = fma_t(fma_t(-d, y, 1.0), y, y);
  const double q = n * y;
  return fma_t(fma_t(-d, q, n), y, q);
}

struct FieldGeom {
  int32_t ny, nx;
  int32_t x_left, x_right, y_left, y_right;  // 1 = periodic, 0 = closed
  int32_t linear = 0;  // guarded array in plain row order (see cell_slot)
};

// Cells of the guarded array of an ny x nx field: (ny + 2) x (nx + 2), the
// image's cell (i, j) at (i + 1, j + 1), a ring of guard cells around it.
__host__ __device__ inline int64_t guarded_cells(int64_t ny, int64_t nx) {
  return (ny + 2) * (nx + 2);
}

// Where cell (gi, gj) of the guarded array is stored.  Rows are stored in
// pairs, the two cells of a column next to each other, so that 2 x 2 cells
// are 64 (float) or 128 (double) consecutive bytes.  A wave's gather of 16
// bytes per lane takes one L1 cycle per distinct run of memory in each four
// consecutive lanes: with quads of lanes on 2 x 2 pixels (pixel_of_quads) and
// this order a gather cost 19.7 cycles, averaged over directions of flow,
// against 35.6 in row order with lanes along rows (32-byte cells: 42.4
// against 73.4), and the trace is bound by that path.  `linear` (row order)
// serves the sizes that the spare cells of an odd last row would not fit.
__host__ __device__ inline int64_t cell_slot(const FieldGeom& g, int32_t gi, int32_t gj) {
  const int64_t w = static_cast<int64_t>(g.nx) + 2;
  return g.linear ? gi * w + gj : (gi >> 1) * 2 * w + 2 * static_cast<int64_t>(gj) + (gi & 1);
}

// Slots of a field's guarded array (with the unused half of an odd last pair).
__host__ __device__ inline int64_t cell_slots(const FieldGeom& g) {
  const int64_t h = static_cast<int64_t>(g.ny) + 2, w = static_cast<int64_t>(g.nx) + 2;
  return (g.linear ? h : (h + 1) / 2 * 2) * w;
}

// Per-field constants of the incremental step rule on a guarded array: the
// slots from a cell to its neighbour along x, to the one along y in the other
// row of its pair (near_y) and in the next pair (far_y); up from an odd row
// and down from an even one leads to another pair, with all_far every y step.
struct StepGeom {
  uint32_t step_x, near_y, far_y, all_far;  // all_far: 0 or all ones
};

__host__ __device__ inline StepGeom make_step_geom(const FieldGeom& g) {
  const uint32_t w = static_cast<uint32_t>(g.nx + 2);
  return g.linear ? StepGeom{1u, w, w, 0xFFFFFFFFu} : StepGeom{2u, 1u, 2u * w - 1u, 0u};
}

// Image cell (ti, tj) whose values guard cell (gi, gj) of the guarded array
// holds: itself for an image cell, else the cell the boundary rule sends a
// step onto the guard cell to (src/lib.rs:83-95: the edge cell on a closed
// side, the opposite edge cell on a periodic one).  False for the four
// corners, which no step reaches (a step changes one coordinate).
__host__ __device__ inline bool guard_source(int32_t gi, int32_t gj, int32_t ny, int32_t nx,
                                             int32_t x_left, int32_t x_right, int32_t y_left,
                                             int32_t y_right, int32_t& ti, int32_t& tj) {
  ti = gi - 1;
  tj = gj - 1;
  const bool out_y = ti < 0 || ti >= ny, out_x = tj < 0 || tj >= nx;
  if (out_y && out_x) return false;
  if (tj < 0) tj = x_left ? nx - 1 : 0;
  if (tj >= nx) tj = x_right ? 0 : nx - 1;
  if (ti < 0) ti = y_left ? ny - 1 : 0;
  if (ti >= ny) ti = y_right ? 0 : ny - 1;
  return true;
}

// Cell (gi, gj) of a field's guarded array from its strided texture, u, v.
template <typename T>
__device__ __forceinline__ Cell<T> guarded_cell(const T* __restrict__ tex, int64_t tsy,
                                                int64_t tsx, const T* __restrict__ u,
                                                int64_t usy, int64_t usx,
                                                const T* __restrict__ v, int64_t vsy,
                                                int64_t vsx, const FieldGeom& g, int32_t gi,
                                                int32_t gj) {
  Cell<T> c;
  int32_t i, j;
  if (guard_source(gi, gj, g.ny, g.nx, g.x_left, g.x_right, g.y_left, g.y_right, i, j)) {
    c.u = u[i * usy + j * usx];
    c.v = v[i * vsy + j * vsx];
    c.x = tex[i * tsy + j * tsx];
    c.pad = jump_pad(static_cast<int32_t>(static_cast<uint32_t>(cell_slot(g, i + 1, j + 1)) -
                                          static_cast<uint32_t>(cell_slot(g, gi, gj))),
                     static_cast<T*>(nullptr));
  } else {
    c.u = T(0);
    c.v = T(0);
    c.x = T(0);
    c.pad = T(0);
  }
  return c;
}

// Thread of a packing block -> cell (di, dj) of the 4 x 64 cells it covers: a
// wave takes 32 columns of one row pair, whose slots are consecutive.
__device__ __forceinline__ void pack_cell_of_thread(int32_t tid, int32_t& di, int32_t& dj) {
  di = ((tid >> 7) << 1) | (tid & 1);
  dj = (tid >> 1) & 63;
}

// Kernels below this have no whole group of 8 steps in either direction and so
// no use for the short path, whose preparation takes a third of so short a trace:
// their fields are marked too.  2048^2 float, L = 3 and 9, us a launch before the
// short path existed, with it, marked: 33, 47, 36 and 54, 65, 59 (L = 17: 86,
// 73); double 38, 58, 43 and 75, 94, 84.  (A test of the length in the trace cost
// a 4096^2 one of L = 129 2.5%.)
constexpr int32_t kShortPathMinLen = 16;

// Stores guarded cell (gi, gj); marks a wide field (wide_mark) and one traced
// with fewer than kShortPathMinLen weights in corner (0, 0), its place.
template <typename T>
__device__ __forceinline__ void store_guarded_cell(Cell<T>* __restrict__ cells, int32_t gi,
                                                   int32_t gj, const FieldGeom& g,
                                                   const Cell<T>& c, uint32_t epoch,
                                                   int32_t klen) {
  uint32_t* corner = reinterpret_cast<uint32_t*>(cells);
  if (gi != 0 || gj != 0) {
    cells[cell_slot(g, gi, gj)] = c;
  } else {
    if (epoch == kCountedEpoch) corner[2] = packing_epoch(corner, epoch);
    if (klen < kShortPathMinLen) corner[0] = packing_epoch(corner, epoch);
  }
  if (velocity_wide(c.u) || velocity_wide(c.v)) corner[0] = packing_epoch(corner, epoch);
}

// Move codes recorded by the tracing pass (4 bits per step, 8 per word): a
// step to a neighbouring cell along x, or with kMoveAxisY along y (rows),
// toward higher indices or with kMoveNeg lower ones, with kMoveEdge when it
// left the image over a periodic side; kMoveStay for no move (a zero vector,
// or a step held at a closed side) and kMoveStop where the streamline ended
// on a NaN vector (src/lib.rs:336-338).  A code without its lowest bit is a
// byte selector of v_perm_b32: 0, 2, 4, 6 pick one of four 16-bit deltas, 8 the
// sign byte of the first, which is zero (replay_box).
enum : uint32_t {
  kMoveEdge = 1,
  kMoveAxisY = 2,
  kMoveNeg = 4,
  kMoveStay = 8,
  kMoveStop = 9,
  kMoveXPlus = 0,
  kMoveXMinus = kMoveNeg,
  kMoveYPlus = kMoveAxisY,
  kMoveYMinus = kMoveAxisY | kMoveNeg
};
constexpr uint32_t kWordStay = 0x11111111u * kMoveStay;
constexpr uint32_t kWordMoves = 0x11111111u * (kMoveNeg | kMoveAxisY);

// word * 16 + a step's code: kMoveAxisY where `mx` is clear, kMoveNeg where
// `neg` is set (with FLIP clear); the lowest and the highest bit of the code
// are left over from the masks.
template <bool FLIP>
__device__ __forceinline__ uint32_t push_code(uint32_t word, uint32_t neg, uint32_t mx) {
  static_assert(kMoveNeg == 4 && kMoveAxisY == 2, "bits 30 and 29 of the masks");
  const uint32_t bits = bitop3<FLIP ? 0x1B : 0xB1>(neg, mx, 1u << 30);
  return __builtin_amdgcn_alignbit(word, bits, 28);
}

// A word holds the codes of 8 consecutive steps, the first step in the top
// nibble: step q in bits 28 - 4q .. 31 - 4q.  (The tracing pass shifts
// each code bit in at the bottom of the word with one add-with-carry, so
// the first step's bits end on top.)
__host__ __device__ inline uint32_t move_code(uint32_t word, int q) {
  return (word >> (28 - 4 * q)) & 15u;
}

// Bit 4k set where nibble k of `word` is the stop code.
__host__ __device__ inline uint32_t stop_nibbles(uint32_t word) {
  return (word >> 3) & word & 0x11111111u;
}

// Steps of a word before its first stop code (8 when it has none): with
// the top stop bit at 4k (step 7 - k), (stops << 3) | 1 has its top bit at
// 4k + 3 (bit 0 without a stop), so (leading zeros + 1) / 4 = 7 - k (8);
// branch-free, and the argument of clz is never 0.
__host__ __device__ inline int32_t steps_before_stop(uint32_t word) {
  const uint32_t stops = stop_nibbles(word);
  return (__builtin_clz((stops << 3) | 1u) + 1) >> 2;
}

// Whether a word of 8 recorded steps holds a stop code.  The tracing pass
// records the stop code again at every step after a line has ended (the
// line stays on its NaN cell), so a word whose 8 steps were all recorded
// has one exactly when its last code (the bottom nibble) is the stop code.
__host__ __device__ inline bool group_has_stop(uint32_t word) {
  return (word & 15u) == kMoveStop;
}

// Position change of each move code in `unit`s, added modulo 2^32
// (positions are uint32_t).  `row` is the row length and `span_x`, `span_y`
// the distance between opposite edge cells, all in units; a periodic edge
// step jumps across the image.
__host__ __device__ inline uint32_t move_delta_units(uint32_t code, uint32_t unit, uint32_t row,
                                                     uint32_t span_x, uint32_t span_y) {
  switch (code) {
    case kMoveXPlus: return unit;
    case kMoveXMinus: return 0u - unit;
    case kMoveYPlus: return row;
    case kMoveYMinus: return 0u - row;
    case kMoveXPlus | kMoveEdge: return 0u - span_x;
    case kMoveXMinus | kMoveEdge: return span_x;
    case kMoveYPlus | kMoveEdge: return 0u - span_y;
    case kMoveYMinus | kMoveEdge: return span_y;
    default: return 0u;
  }
}

// Replay through the image itself: wraps jump across it.
__host__ __device__ inline uint32_t move_delta(uint32_t code, const FieldGeom& g, uint32_t unit) {
  const uint32_t row = static_cast<uint32_t>(g.nx) * unit;
  return move_delta_units(code, unit, row, static_cast<uint32_t>(g.nx - 1) * unit,
                          static_cast<uint32_t>(g.ny - 1) * row);
}

// Block -> pixel tile.  A block is 4 wave64s in a 2x2 arrangement; each wave
// covers a wave_w x (64 / wave_w) rectangle, so a block tile is
// (2 * wave_w) x (128 / wave_w).  Workgroups are dealt round-robin to the
// 8 XCDs; each XCD is given a contiguous run of logical tiles, and logical
// tiles run column-major inside horizontal strips `band` tiles tall, so the
// tiles resident on one XCD at a time form a compact patch whose streamline
// halo stays in that XCD's L2.
struct TileMap {
  int32_t tiles_x, tiles_y, n_tiles;
  int32_t per_xcd, rem_xcd;  // n_tiles = 8 * per_xcd + rem_xcd
  int32_t band;
  int32_t wave_w_log2;       // 3, 4 or 5 (wave tile 8x8, 16x4, 32x2)
};

constexpr int kBlock = 256;
constexpr int kXcds = 8;

__host__ __device__ inline int32_t tile_w(const TileMap& m) { return 2 << m.wave_w_log2; }
__host__ __device__ inline int32_t tile_h(const TileMap& m) { return 2 << (6 - m.wave_w_log2); }

__device__ __forceinline__ void tile_of_block(int32_t b, const TileMap& m, int32_t& ty,
                                              int32_t& tx) {
  const int32_t xcd = b & (kXcds - 1);
  const int32_t slot = b >> 3;
  const int32_t logical = xcd * m.per_xcd + min(xcd, m.rem_xcd) + slot;
  const int32_t strip_tiles = m.band * m.tiles_x;
  const int32_t strip = logical / strip_tiles;
  const int32_t within = logical - strip * strip_tiles;
  const int32_t h = min(m.band, m.tiles_y - strip * m.band);
  tx = within / h;
  ty = strip * m.band + (within - tx * h);
}

// Thread -> pixel (py, px) inside the block tile.
__device__ __forceinline__ void pixel_of_thread(int32_t tid, const TileMap& m, int32_t& py,
                                                int32_t& px) {
  const int32_t w = tid >> 6, l = tid & 63;
  const int32_t ww = m.wave_w_log2, wh = 6 - m.wave_w_log2;
  px = ((w & 1) << ww) | (l & ((1 << ww) - 1));
  py = ((w >> 1) << wh) | (l >> ww);
}

// The same for a tracing wave: four consecutive lanes on 2 x 2 pixels
// (cell_slot), the quads along the rows of the wave's rectangle.
__device__ __forceinline__ void pixel_of_quads(int32_t tid, const TileMap& m, int32_t& py,
                                               int32_t& px) {
  const int32_t w = tid >> 6, l = tid & 63, k = l >> 2;
  const int32_t ww = m.wave_w_log2, wh = 6 - m.wave_w_log2;
  px = ((w & 1) << ww) | ((k & ((1 << (ww - 1)) - 1)) << 1) | (l & 1);
  py = ((w >> 1) << wh) | ((k >> (ww - 1)) << 1) | ((l >> 1) & 1);
}

}  // namespace rlic
