// What the GEMM kernels of weight_only_linear share: MFMA wrappers, exact
// dequantisers, the parameters of a launch.  wol_linear_gemm.hip holds the
// kernels of up to 64 rows, the general one and the plans, wol_linear_wide.hip
// the tiles of 128 and 256 rows.
#pragma once

#include <atomic>
#include <climits>
#include <type_traits>

#include "wol_common.h"
#include "wol_dequant.h"

namespace wol {

// What one launch of the fast kernel works on.
struct DmaParams {
  const uint16_t* x;
  const uint8_t* codes;
  const uint16_t* bias;
  const uint16_t* scale;
  void* out;                    // T or fp32 [M, N]; with nsplit > 1 fp32 partial sums
                                // [nsplit][M][columns of the launch]
  int M, K, N;
  int out_f32;
  int strip_lo, strip_hi;       // the launch covers the 16-column strips [strip_lo, strip_hi)
  int nbx, nby;                 // output tiles of the launch
  int nsplit, tiles_per_split;  // K is cut into nsplit runs of k tiles, one workgroup each
  int xcd_rows;                 // row groups of the XCD grid (tile_of_block), 0 = plain order
  int act;                      // WOL_ACT_NONE or WOL_ACT_GELU, applied where the final sum is formed
  // Grouped launch (mixture of experts): row tile `by` of the launch is entry
  // `by` of this table -- {expert, first row, rows} -- written on the device by
  // moe_plan_kernel; an expert's rows use that expert's weights, scales and
  // bias (consecutive tensors, the strides below apart).  Null: one problem.
  const int* moe_table;
  int64_t moe_codes_stride;     // bytes between two experts' packed weights
  int moe_rows;                 // rows of the whole grouped problem (the partial sums' row count)
  // STAMP instantiation only: seven cycle counts and the number of k tiles of every wavefront, [workgroup][wavefront][8]
  // (see wol_prefill_phases)
  unsigned long long* stamps;
};

// One entry of the row-tile table of a grouped launch.
struct MoeTile {
  int expert;  // -1: the tile is not used
  int row0;    // first row of the tile in the permuted input
  int rows;    // rows of the tile that exist (1 .. tile height)
  int first;   // gemm_experts_kernel: first row tile of the tile's expert ...
  int count;   // ... and how many it has
  int pad[3];
};

// Where a tile of gemm_experts_kernel lies.
struct TilePlace {
  int bx;      // column tile of the launch
  int expert;  // the tile lies in this expert's rows
  int row0;    // the tile's first row in x and out
  int rows;    // rows of the tile that exist
};

// The tiles of 128 and 256 rows (wol_linear_wide.hip), compiled as one translation unit per element type.
enum class WideTile {
  kWhole,  // 256 x 256
  kHalf,   // 128 x 256
};
// group: 0, 64 or 128.  swi: 1 = swiglu of a gate | up projection in the epilogue (p.out is [M, N / 2], the strips are
// those of the gate half).
void launch_wide_bf16(const DmaParams& p, int bits, int group, WideTile tile, int swi, hipStream_t stream);
void launch_wide_f16(const DmaParams& p, int bits, int group, WideTile tile, int swi, hipStream_t stream);
// The grouped GEMM over experts on tiles of up to 256 rows x 256 columns (narrow: 128); p.moe_table is that of
// moe_plan_kernel<true>.  swiglu: of the product rounded to T, p.out is [rows, N / 2].
void launch_experts_bf16(const DmaParams& p, int bits, bool narrow, bool swiglu, unsigned blocks, hipStream_t stream);
void launch_experts_f16(const DmaParams& p, int bits, bool narrow, bool swiglu, unsigned blocks, hipStream_t stream);

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int DT>
__device__ inline f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if (DT == WOL_DTYPE_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

__device__ inline uint32_t pack_bf16_hi(float lo, float hi) {
  // both values are small integers, exact in bf16: keep the high halves
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

__device__ inline uint32_t f16x2_add(uint32_t v, uint32_t c) {
  const f16x2 r = __builtin_bit_cast(f16x2, v) + __builtin_bit_cast(f16x2, c);
  return __builtin_bit_cast(uint32_t, r);
}

// Codes of one k step (8 per lane) -> four dwords of T pairs holding the exact
// signed code.
template <int DT, int BITS>
struct DequantExact;

template <>
struct DequantExact<WOL_DTYPE_BF16, 8> {
  __device__ static inline float sbyte(uint32_t v, int i) {
    return static_cast<float>(static_cast<int>(static_cast<int8_t>((v >> (8 * i)) & 0xFFu)));
  }
  __device__ static inline u32x4 run(const uint32_t* w) {
    // stored byte = code + 128; flipping the top bit gives the two's complement code
    const uint32_t a = w[0] ^ 0x80808080u, b = w[1] ^ 0x80808080u;
    u32x4 o;
    o.x = pack_bf16_hi(sbyte(a, 0), sbyte(a, 1));
    o.y = pack_bf16_hi(sbyte(a, 2), sbyte(a, 3));
    o.z = pack_bf16_hi(sbyte(b, 0), sbyte(b, 1));
    o.w = pack_bf16_hi(sbyte(b, 2), sbyte(b, 3));
    return o;
  }
};

template <>
struct DequantExact<WOL_DTYPE_F16, 8> {
  __device__ static inline u32x4 run(const uint32_t* w) {
    u32x4 o;  // byte | 0x6400 = 1024 + byte, minus 1152 = code
    o.x = f16x2_add(__builtin_amdgcn_perm(w[0], 0x64646464u, 0x00050004u), 0xE480E480u);
    o.y = f16x2_add(__builtin_amdgcn_perm(w[0], 0x64646464u, 0x00070006u), 0xE480E480u);
    o.z = f16x2_add(__builtin_amdgcn_perm(w[1], 0x64646464u, 0x00050004u), 0xE480E480u);
    o.w = f16x2_add(__builtin_amdgcn_perm(w[1], 0x64646464u, 0x00070006u), 0xE480E480u);
    return o;
  }
};

template <>
struct DequantExact<WOL_DTYPE_F16, 4> {
  __device__ static inline u32x4 run(const uint32_t* w) {
    const uint32_t v = w[0];
    u32x4 o;  // nibble<<4 | 0x5400 = 64 + nibble, minus 72 = code
    o.x = f16x2_add(((v << 4) & 0x00F000F0u) | 0x54005400u, 0xD480D480u);
    o.y = f16x2_add((v & 0x00F000F0u) | 0x54005400u, 0xD480D480u);
    o.z = f16x2_add(((v >> 4) & 0x00F000F0u) | 0x54005400u, 0xD480D480u);
    o.w = f16x2_add(((v >> 8) & 0x00F000F0u) | 0x54005400u, 0xD480D480u);
    return o;
  }
};

template <>
struct DequantExact<WOL_DTYPE_BF16, 4> {
  __device__ static inline uint32_t fix(uint32_t pair) {
    // pair = two bf16 holding 136 + code; widen, subtract, narrow (all exact)
    const float lo = __uint_as_float(pair << 16) - 136.0f;
    const float hi = __uint_as_float(pair & 0xFFFF0000u) - 136.0f;
    return pack_bf16_hi(lo, hi);
  }
  __device__ static inline u32x4 run(const uint32_t* w) {
    const uint32_t v = w[0];
    u32x4 o;
    o.x = fix((v & 0x000F000Fu) | 0x43004300u);
    o.y = fix(((v >> 4) & 0x000F000Fu) | 0x43004300u);
    o.z = fix(((v >> 8) & 0x000F000Fu) | 0x43004300u);
    o.w = fix(((v >> 12) & 0x000F000Fu) | 0x43004300u);
    return o;
  }
};

// The same codes in 19 instructions per eight instead of 27: each nibble pair
// becomes two fp16 values 1024 + 16 * nibble (one and-or), a mixed-precision FMA
// takes the offset out and widens to fp32 in one instruction, and the high
// halves are the bf16 codes, every step exact.  Against the other form the small-M
// tiles are 1 to 2 % faster; gemm_kernel: per channel 2 to 4 % faster, group-wise
// up to 9 % slower (K = 4544: 65 rows), so it keeps the other there.
template <int DT, int BITS>
struct DequantExactFma : DequantExact<DT, BITS> {};

template <>
struct DequantExactFma<WOL_DTYPE_BF16, 4> {
  __device__ static inline uint32_t pair(uint32_t v) {
    const f16x2 h = __builtin_bit_cast(f16x2, (v & 0x00F000F0u) | 0x64006400u);
    return pack_bf16_hi(__builtin_fmaf(static_cast<float>(h.x), 0.0625f, -72.0f),
                        __builtin_fmaf(static_cast<float>(h.y), 0.0625f, -72.0f));
  }
  __device__ static inline u32x4 run(const uint32_t* w) {
    const uint32_t v = w[0];
    u32x4 o;
    o.x = pair(v << 4);
    o.y = pair(v);
    o.z = pair(v >> 4);
    o.w = pair(v >> 8);
    return o;
  }
};

// s_waitcnt that only bounds the number of outstanding vector-memory loads.
template <int N_>
__device__ inline void wait_vmcnt() {
  // gfx9 encoding: vmcnt = [15:14][3:0], expcnt = [6:4], lgkmcnt = [11:8]
  __builtin_amdgcn_s_waitcnt((N_ & 0xF) | ((N_ >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// XOR applied to the 16-byte piece index of an A row in LDS (C pieces per
// row).  A lane group reads the same piece of 16 consecutive rows; the XOR
// spreads those reads over the banks whether the LDS serves 8 or 16 lanes of
// a 128-bit read per cycle.
template <int C>
__device__ inline int a_swizzle(int row) {
  if (C == 8) return (row & 7) ^ ((row >> 3) & 1);  // 128-byte rows
  return row & (C - 1);                             // 256-byte rows
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int DT>
__device__ inline f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  if (DT == WOL_DTYPE_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Where position `pos` of a launch's tiles lies.  The sequence walks the tiles in bands of four row tiles or so, column
// by column within a band, and every XCD works on a piece of it that hangs together: its 32 CUs then share four row
// blocks and eight column blocks in their L2.  (A grid of XCDs that needs both tile counts to divide left ragged ones in
// plain order, where the 32 tiles of an XCD have 32 different column blocks.)
__device__ inline void tile_of_position(int pos, int nbx, int nby, int* bx, int* by) {
  const int bands = nby > 5 ? (nby + 2) / 4 : 1, base = nby / bands, extra = nby % bands;
  int rows = base + 1, lo = 0, w = pos;  // the first `extra` bands have a row tile more
  if (w >= extra * rows * nbx) {
    w -= extra * rows * nbx;
    lo = extra * rows;
    rows = base;
  }
  const int b = w / (rows * nbx);
  w -= b * rows * nbx;
  *by = lo + b * rows + w % rows;
  *bx = w / rows;
}

// Raises a kernel's dynamic LDS limit once per device (the attribute belongs to
// the device's copy of the function); safe to call from several threads.
inline void allow_lds(const void* kern, size_t lds, std::atomic<uint32_t>& done) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  const uint32_t bit = 1u << (dev & 31);
  if (done.load(std::memory_order_acquire) & bit) return;
  (void)hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
  done.fetch_or(bit, std::memory_order_release);
}

inline int num_cus() {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    return n;
  }();
  return cus;
}

}  // namespace

}  // namespace wol
