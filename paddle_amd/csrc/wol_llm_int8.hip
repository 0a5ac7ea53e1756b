// llm_int8_linear for gfx950: dynamic per-row int8 quantisation of the
// activations, an int8 x int8 -> int32 MFMA GEMM against the plain [N,K] int8
// weight that weight_quantize(algo="llm.int8") returns, the outlier columns in
// T x dequantised-weight arithmetic, and the merge of the two.
//
// Stages (paddle/phi/kernels/impl/llm_int8_matmul_kernel_impl.h:560-690 runs
// the same ones as separate kernels plus two library GEMMs and a device-to-host
// copy of the outlier count; here nothing returns to the host):
//   rowmax  : range[m] = max |x[m,k]| over the elements not above the
//             threshold; bit k set where any |x[m,k]| > threshold
//             (ReduceAbsMaxKernel, :221-268), per workgroup in LDS
//   mask    : ORs the workgroups' bits into the mask
//   quant   : qx = 0 in outlier columns, else clip(round(x * 127 * (1/range)))
//             (QuantActKernel :270-303, QuantFunc :153-164); one extra
//             workgroup turns the mask into an ascending list of columns
//             (up to eight rows: these three as one kernel)
//   outlier : sub = T(sum over the outlier columns of x * T(w * wscale)), fp32
//             sum in ascending column order; leaves at once without outliers
//   gemm    : acc = qx . w^T in int32 on v_mfma_i32_32x32x32_i8 (above 128 rows
//             16x16x64), both operands
//             through direct-to-LDS loads, two or three k tiles deep.  The
//             epilogue is DequantMergeKernel (:415-447): out = T( sub + T(acc *
//             range * wscale / 127) ), then T(out + bias).
//   merge   : only when K is cut into runs (few tiles): every run leaves its
//             int32 sums in a slab of its own and this kernel adds them (exact,
//             so the result does not depend on the cut) and applies the same
//             epilogue.
#include "wol_gemm_common.h"

namespace wol {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------
// activation side
// ---------------------------------------------------------------------------
// Row ranges and outlier bits.  A workgroup takes a run of rows, four at a time,
// and a thread the same columns of each (16-byte loads); the outlier bits of
// the run are ORed in an LDS mask and leave as the workgroup's own row of
// `part` -- no global atomics: device-wide atomics on one word serialise at
// 100-150 ns each across the XCDs, and outlier columns are the same in most
// rows (with them this kernel took 15 us for 2048 rows x 4096).  The mask
// kernel below ORs the rows of `part`.
constexpr int kRowChunk = 4;
constexpr int kMaxRowGroups = 512;

template <int DT>
__global__ __launch_bounds__(256) void llm_rowmax_kernel(const uint16_t* __restrict__ x, float threshold, int M,
                                                         int K, int rows_per_group, float* __restrict__ ranges,
                                                         uint32_t* __restrict__ part) {
  extern __shared__ uint32_t smask[];  // K / 32 words
  __shared__ float red[4][kRowChunk];
  const float thr = to_f32<DT>(from_f32_rne<DT>(threshold));  // the comparison is made in T
  const int nwords = K / 32;
  for (int w = threadIdx.x; w < nwords; w += 256) smask[w] = 0u;
  __syncthreads();
  const int m_begin = blockIdx.x * rows_per_group;
  const int m_end = m_begin + rows_per_group < M ? m_begin + rows_per_group : M;
  for (int m0 = m_begin; m0 < m_end; m0 += kRowChunk) {
    float mx[kRowChunk];
#pragma unroll
    for (int r = 0; r < kRowChunk; ++r) mx[r] = 0.0f;
    for (int k0 = threadIdx.x * 8; k0 < K; k0 += 256 * 8) {
      u32x4 v[kRowChunk];
#pragma unroll
      for (int r = 0; r < kRowChunk; ++r) {
        const int m = m0 + r < m_end ? m0 + r : m_end - 1;  // past the end: the last row again
        v[r] = *reinterpret_cast<const u32x4*>(x + static_cast<int64_t>(m) * K + k0);
      }
      uint32_t bits = 0;
#pragma unroll
      for (int r = 0; r < kRowChunk; ++r) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float a = fabsf(to_f32<DT>(static_cast<uint16_t>(v[r][i >> 1] >> (16 * (i & 1)))));
          if (a > thr) {
            bits |= 1u << i;
            a = 0.0f;
          }
          mx[r] = a > mx[r] ? a : mx[r];
        }
      }
      if (bits != 0) atomicOr(&smask[k0 >> 5], bits << (k0 & 31));
    }
#pragma unroll
    for (int r = 0; r < kRowChunk; ++r) {
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) {
        const float o = __shfl_xor(mx[r], d, 64);
        mx[r] = o > mx[r] ? o : mx[r];
      }
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][r] = mx[r];
    }
    __syncthreads();
    if (threadIdx.x < kRowChunk && m0 + threadIdx.x < m_end) {
      float r = red[0][threadIdx.x];
#pragma unroll
      for (int i = 1; i < 4; ++i) r = red[i][threadIdx.x] > r ? red[i][threadIdx.x] : r;
      ranges[m0 + threadIdx.x] = r;
    }
    __syncthreads();  // red is reused by the next four rows
  }
  for (int w = threadIdx.x; w < nwords; w += 256) part[static_cast<int64_t>(blockIdx.x) * nwords + w] = smask[w];
}

// QuantFunc (:153-164).  NaN (0 * inf in a row whose range is 0) becomes 0.
__device__ inline uint32_t quant_one(float xv, float inv) {
  float t = xv * 127.0f * inv;
  t = roundf(t);
  t = t > 127.0f ? 127.0f : (t < -127.0f ? -127.0f : t);
  if (t != t) t = 0.0f;
  return static_cast<uint32_t>(static_cast<int>(t)) & 0xFFu;
}

// The mask (nwords words, word w from word_at(w)) as an ascending list of
// outlier columns and their count.  Called by every thread of a workgroup (of
// at least 256 threads; the first 256 do the work); scan (256 ints) and base_s
// are LDS.
template <class F>
__device__ inline void build_list(int nwords, F word_at, int32_t* list, int32_t* count, int* scan, int* base_s) {
  const int tid = threadIdx.x;
  const bool worker = tid < 256;
  if (tid == 0) *base_s = 0;
  __syncthreads();
  for (int w0 = 0; w0 < nwords; w0 += 256) {
    uint32_t word = worker && w0 + tid < nwords ? word_at(w0 + tid) : 0u;
    const int c = __popc(word);
    if (worker) scan[tid] = c;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
      const int add = worker && tid >= d ? scan[tid - d] : 0;
      __syncthreads();
      if (worker) scan[tid] += add;
      __syncthreads();
    }
    const int base = *base_s;
    int o = worker ? base + scan[tid] - c : 0;
    while (word != 0) {
      const int b = __ffs(word) - 1;
      list[o++] = (w0 + tid) * 32 + b;
      word &= word - 1;
    }
    __syncthreads();
    if (tid == 0) *base_s = base + scan[255];
    __syncthreads();
  }
  if (tid == 0) *count = *base_s;
}

// Row ranges, outlier mask and list, activation codes of up to kSmallRows rows
// in one launch: the decode-sized case, where a launch costs more than the work.
// A workgroup per row, and one more for the list.  Which columns are outliers
// depends on every row, so each workgroup looks through all of them (a few dozen
// KiB out of L2) instead of waiting for the others, and finds its own row's
// range on the way.  The mask lives in LDS (K / 32 words, dynamic).
// Whole call, us, against three launches (one or two rows: one workgroup for
// everything), K = 4096, N = 11008, 3 outlier columns: 1 row 20.1 -> 18.5, 4 rows
// 23.4 -> 20.3, 8 rows 28.9 -> 26.8.  Every workgroup's look through all rows grows
// with M * K, so the gain shrinks: 8 rows K = 11008 31.7 -> 28.9, 28672 49.1 -> 48.3,
// 32768 55.9 -> 56.6, 65536 79.7 -> 82.1; 7 rows 53.9 -> 52.4 and 77.7 -> 76.0.  Hence
// eight rows up to K = 28672 and seven beyond.
constexpr int kSmallRows = 8;
constexpr int kSmallRowsMaxK = 28672;  // one row fewer beyond
constexpr int kSmallThreads = 1024;
constexpr int kSmallMaxK = 65536;

template <int DT>
__global__ __launch_bounds__(kSmallThreads) void llm_act_small_kernel(const uint16_t* __restrict__ x, float threshold,
                                                                      int M, int K, float* __restrict__ ranges,
                                                                      int32_t* __restrict__ mask,
                                                                      int8_t* __restrict__ qx,
                                                                      int32_t* __restrict__ count,
                                                                      int32_t* __restrict__ list) {
  extern __shared__ uint32_t smask[];
  __shared__ float part[kSmallThreads / 64];
  const int tid = threadIdx.x, row = blockIdx.x;
  const int nwords = K / 32, per = K / 8;
  const float thr = to_f32<DT>(from_f32_rne<DT>(threshold));
  for (int w = tid; w < nwords; w += kSmallThreads) smask[w] = 0u;
  __syncthreads();
  float mx = 0.0f;
  // 16 bytes of a row per thread, four in flight
  const int nvec = M * per;
  for (int v0 = tid; v0 < nvec; v0 += 4 * kSmallThreads) {
    u32x4 d[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int v = v0 + u * kSmallThreads;
      d[u] = *reinterpret_cast<const u32x4*>(x + static_cast<int64_t>(v < nvec ? v : v0) * 8);  // past the end: its first again
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int v = v0 + u * kSmallThreads;
      if (v >= nvec) break;
      const int m = v / per, k0 = (v - m * per) * 8;
      uint32_t bits = 0;
      float top = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float a = fabsf(to_f32<DT>(static_cast<uint16_t>(d[u][i >> 1] >> (16 * (i & 1)))));
        if (a > thr) {
          bits |= 1u << i;
          a = 0.0f;
        }
        top = a > top ? a : top;
      }
      mx = m == row && top > mx ? top : mx;
      if (bits != 0) atomicOr(&smask[k0 >> 5], bits << (k0 & 31));
    }
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const float o = __shfl_xor(mx, d, 64);
    mx = o > mx ? o : mx;
  }
  if ((tid & 63) == 0) part[tid >> 6] = mx;
  __syncthreads();
  if (row == M) {
    for (int w = tid; w < nwords; w += kSmallThreads) mask[w] = static_cast<int32_t>(smask[w]);  // for whoever inspects the stages
    if (tid >= 64) return;
    int n = 0;  // outlier columns so far
    for (int w0 = 0; w0 < nwords; w0 += 64) {
      uint32_t word = w0 + tid < nwords ? smask[w0 + tid] : 0u;
      const int c = __popc(word);
      int upto = c;  // of the words up to this lane's
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(upto, d, 64);
        upto += tid >= d ? o : 0;
      }
      for (int o = n + upto - c; word != 0; word &= word - 1) list[o++] = (w0 + tid) * 32 + __ffs(word) - 1;
      n += __shfl(upto, 63, 64);
    }
    if (tid == 0) *count = n;
    return;
  }
  float range = part[0];
#pragma unroll
  for (int i = 1; i < kSmallThreads / 64; ++i) range = part[i] > range ? part[i] : range;
  const float inv = 1.0f / range;
  const uint16_t* xrow = x + static_cast<int64_t>(row) * K;
  for (int v = tid; v < K / 16; v += kSmallThreads) {
    const int k = v * 16;
    const u32x4 lo = *reinterpret_cast<const u32x4*>(xrow + k);
    const u32x4 hi = *reinterpret_cast<const u32x4*>(xrow + k + 8);
    const uint32_t out_bits = smask[k >> 5] >> (k & 31);
    u32x4 q = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t word = i < 8 ? lo[(i & 7) >> 1] : hi[(i & 7) >> 1];
      const float xv = to_f32<DT>(static_cast<uint16_t>(word >> (16 * (i & 1))));
      const uint32_t c = (out_bits >> i) & 1u ? 0u : quant_one(xv, inv);
      q[i >> 2] |= c << (8 * (i & 3));
    }
    *reinterpret_cast<u32x4*>(qx + static_cast<int64_t>(row) * K + k) = q;
  }
  if (tid == 0) ranges[row] = range;
}

// ORs the row kernel's partial masks (groups rows of K / 32 words) into the
// mask.  A workgroup takes four words; 64 threads per word each take every
// 64th group and meet in LDS.
__global__ __launch_bounds__(256) void llm_mask_kernel(const uint32_t* __restrict__ part, int groups, int K,
                                                       int32_t* __restrict__ mask) {
  __shared__ uint32_t red[64][4];
  const int tid = threadIdx.x;
  const int nwords = K / 32;
  const int wl = tid & 3, sub = tid >> 2;
  const int w = blockIdx.x * 4 + wl;
  uint32_t v = 0u;
  if (w < nwords)
    for (int g = sub; g < groups; g += 64) v |= part[static_cast<int64_t>(g) * nwords + w];
  red[sub][wl] = v;
  __syncthreads();
  if (tid < 4 && w < nwords) {
    uint32_t o = 0u;
#pragma unroll
    for (int i = 0; i < 64; ++i) o |= red[i][tid];
    mask[w] = static_cast<int32_t>(o);
  }
}

// Activation codes; the last workgroup instead turns the mask into the
// ascending list of outlier columns.
template <int DT>
__global__ __launch_bounds__(256) void llm_quant_kernel(const uint16_t* __restrict__ x,
                                                        const float* __restrict__ ranges,
                                                        int32_t* mask, const uint32_t* __restrict__ part,
                                                        int groups, int M, int K, int8_t* __restrict__ qx,
                                                        int32_t* __restrict__ count, int32_t* __restrict__ list) {
  // groups > 0: the row kernel's few partial masks are ORed here (no mask
  // kernel ran); the list workgroup also leaves the combined mask in `mask`
  const int tid = threadIdx.x;
  const int nwords = K / 32;
  auto mask_word = [&](int w) {
    if (groups == 0) return static_cast<uint32_t>(mask[w]);
    uint32_t v = 0u;
    for (int g = 0; g < groups; ++g) v |= part[static_cast<int64_t>(g) * nwords + w];
    return v;
  };
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ int scan[256];
    __shared__ int base_s;
    build_list(nwords, [&](int w) {
      const uint32_t v = mask_word(w);
      if (groups != 0) mask[w] = static_cast<int32_t>(v);
      return v;
    }, list, count, scan, &base_s);
    return;
  }
  const int64_t stride = static_cast<int64_t>(gridDim.x - 1) * 256;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * 256 + tid;
  const int64_t nvec = static_cast<int64_t>(M) * K / 16;
  for (int64_t v = first; v < nvec; v += stride) {
    const int64_t e = v * 16;
    const int m = static_cast<int>(e / K);
    const int k = static_cast<int>(e - static_cast<int64_t>(m) * K);
    const u32x4 lo = *reinterpret_cast<const u32x4*>(x + e);
    const u32x4 hi = *reinterpret_cast<const u32x4*>(x + e + 8);
    const uint32_t out_bits = mask_word(k >> 5) >> (k & 31);
    const float inv = 1.0f / ranges[m];
    u32x4 q = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t word = i < 8 ? lo[(i & 7) >> 1] : hi[(i & 7) >> 1];
      const float xv = to_f32<DT>(static_cast<uint16_t>(word >> (16 * (i & 1))));
      const uint32_t c = (out_bits >> i) & 1u ? 0u : quant_one(xv, inv);
      q[i >> 2] |= c << (8 * (i & 3));
    }
    *reinterpret_cast<u32x4*>(qx + e) = q;
  }
}

// ---------------------------------------------------------------------------
// the epilogue arithmetic, shared by the GEMM and the merge kernel
// ---------------------------------------------------------------------------
struct Epi {
  const uint16_t* x;      // [M,K] T
  const int8_t* w;        // [N,K]
  const float* wscale;    // [N]
  const float* ranges;    // [M]
  const uint16_t* bias;   // [N] T or null
  const int32_t* count;
  const int32_t* list;
  uint16_t* out;          // [M,N] T
  int M, K, N;
  int pick;               // outlier columns, up to which the GEMM picks them out of x and w although cols is there
  // Few outlier columns, collected by the outlier kernel for the GEMM's epilogue (null: it picks them out of x and w):
  // [kOutCap][M rounded up to whole tiles] x of outlier column j, by row, and behind them [kOutCap][N rounded up]
  // T(w * wscale) of it, by output column.
  uint16_t* cols;
};
constexpr int kOutCap = 32;
__host__ __device__ constexpr int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }  // also whole tiles, of any height and width

// v / 127, correctly rounded, in four instructions instead of the dozen of the IEEE division sequence: q = v * RN(1/127),
// r = v - 127 q (exact in an FMA), q + r * RN(1/127), and v_div_fixup for v = -0 and infinities, where q is already the
// answer.  Equal to the division for every one of the 2^32 float inputs (checked exhaustively on the device).
__device__ inline float div127(float v) {
  const float y = 1.0f / 127.0f;
  const float q = v * y;
  const float r = __builtin_fmaf(-q, 127.0f, v);
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(r, y, q), 127.0f, v);
}

// DequantFunc (:172-176) and the two T additions that follow it.  The casts
// are the hardware's round-to-nearest-even conversions (the payload of a NaN
// result is unspecified).
template <int DT>
__device__ inline uint16_t merge_one(int acc, float sub, float range, float ws, bool has_bias, float bias) {
  const float dq = to_f32<DT>(cast_out<DT>(div127(static_cast<float>(acc) * range * ws)));
  const float o = to_f32<DT>(cast_out<DT>(sub + dq));  // sub is a T value
  return has_bias ? cast_out<DT>(o + bias) : cast_out<DT>(o);
}

// The same without outlier columns (sub = +0): T(0 + dq) is dq, -0 becoming +0.
template <int DT>
__device__ inline uint16_t merge_plain(int acc, float range, float ws, bool has_bias, float bias) {
  const uint16_t dq = cast_out<DT>(div127(static_cast<float>(acc) * range * ws));
  if (!has_bias) return dq == 0x8000u ? static_cast<uint16_t>(0) : dq;
  return cast_out<DT>(to_f32<DT>(dq) + 0.0f + bias);
}

// Eight neighbouring columns nn .. nn+7 of row m: the merge with the outlier
// columns' product (when there are any: out of LDS if xs is given, else as the
// outlier kernel left it in the output's own place) and one 16-byte store.  ws and bias hold the eight columns' values.
template <int DT>
__device__ inline void finish8(const Epi& e, int cnt, int m, int nn, float range, i32x4 s0, i32x4 s1,
                               const float* ws, const float* bias, const float* xs, int xs_stride,
                               const float* wd, int wd_stride) {
  u32x4 o;
  if (cnt == 0) {  // uniform: the count is one value for the whole launch
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const uint32_t lo = merge_plain<DT>(i < 4 ? s0[i] : s1[i - 4], range, ws[i], e.bias != nullptr, bias[i]);
      const uint32_t hi =
          merge_plain<DT>(i < 4 ? s0[i + 1] : s1[i - 3], range, ws[i + 1], e.bias != nullptr, bias[i + 1]);
      o[i >> 1] = lo | (hi << 16);
    }
    *reinterpret_cast<u32x4*>(e.out + static_cast<int64_t>(m) * e.N + nn) = o;
    return;
  }
  float sub[8];
  if (xs != nullptr) {
    // the workgroup holds this row's activations and these columns' dequantised
    // weights of every outlier column in LDS (xs[j * xs_stride], wd[j * wd_stride + i])
#pragma unroll
    for (int i = 0; i < 8; ++i) sub[i] = 0.0f;
#pragma unroll 1
    for (int j = 0; j < cnt; ++j) {
      const float xv = xs[j * xs_stride];
      const f32x4 w0 = *reinterpret_cast<const f32x4*>(wd + j * wd_stride);
      const f32x4 w1 = *reinterpret_cast<const f32x4*>(wd + j * wd_stride + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sub[i] += xv * w0[i];
        sub[4 + i] += xv * w1[i];
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) sub[i] = to_f32<DT>(cast_out<DT>(sub[i]));
  } else {
    const u32x4 sv = *reinterpret_cast<const u32x4*>(e.out + static_cast<int64_t>(m) * e.N + nn);
#pragma unroll
    for (int i = 0; i < 8; ++i) sub[i] = to_f32<DT>(static_cast<uint16_t>(sv[i >> 1] >> (16 * (i & 1))));
  }
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const uint32_t lo = merge_one<DT>(i < 4 ? s0[i] : s1[i - 4], sub[i], range, ws[i], e.bias != nullptr, bias[i]);
    const uint32_t hi =
        merge_one<DT>(i < 4 ? s0[i + 1] : s1[i - 3], sub[i + 1], range, ws[i + 1], e.bias != nullptr, bias[i + 1]);
    o[i >> 1] = lo | (hi << 16);
  }
  *reinterpret_cast<u32x4*>(e.out + static_cast<int64_t>(m) * e.N + nn) = o;
}

// The eight columns' scales and biases.
template <int DT>
__device__ inline void load_ws_bias8(const Epi& e, int nn, float* ws, float* bias) {
  const f32x4 w0 = *reinterpret_cast<const f32x4*>(e.wscale + nn);
  const f32x4 w1 = *reinterpret_cast<const f32x4*>(e.wscale + nn + 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    ws[i] = w0[i];
    ws[4 + i] = w1[i];
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) bias[i] = e.bias != nullptr ? to_f32<DT>(e.bias[nn + i]) : 0.0f;
}

// sub[m,n] = T( sum over the outlier columns k, ascending, of x[m,k] * T(w[n,k] *
// wscale[n]) ), fp32 sum: what the reference computes with SplitKernel and a
// library GEMM (:305-362, :593-640).  A workgroup takes 64 rows x 256 columns,
// a thread one column of them; the rows' activations of 32 outlier columns at
// a time wait in LDS.  Workgroups leave at once when there is no outlier or
// the GEMM's epilogue computes the product itself (up to fused_cap columns).
template <int DT>
__global__ __launch_bounds__(256) void llm_outlier_kernel(Epi e, int fused_cap) {
  uint16_t* sub = e.out;  // the product waits where the output will go: whoever merges element (m, n) reads it first
  const int per = e.M + e.N;  // elements of a collected column; kOutCap of them are below 2^30
  const int64_t first = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  // the first element's column, fetched beside the count: if there is no such column, what stands there is not used
  const bool may = e.cols != nullptr && first < static_cast<int64_t>(fused_cap) * per;
  int k = may ? e.list[static_cast<int>(first) / per] : 0;
  const int cnt = *e.count;
  if (cnt <= fused_cap) {
    if (e.cols == nullptr || cnt <= e.pick) return;  // the GEMM picks the columns itself
    for (int64_t i = first; i < static_cast<int64_t>(cnt) * per; i += static_cast<int64_t>(gridDim.x) * 256) {
      const int j = static_cast<int>(i) / per, r = static_cast<int>(i) - j * per;
      if (i != first) k = e.list[j];
      if (r < e.M) e.cols[j * align256(e.M) + r] = e.x[static_cast<int64_t>(r) * e.K + k];
      else
        e.cols[kOutCap * align256(e.M) + j * align256(e.N) + (r - e.M)] =
            cast_out<DT>(static_cast<float>(e.w[static_cast<int64_t>(r - e.M) * e.K + k]) * e.wscale[r - e.M]);
    }
    return;
  }
  __shared__ __attribute__((aligned(16))) float xs[32][64];
  const int tid = threadIdx.x;
  const int nbx = (e.N + 255) / 256;
  const int m0 = static_cast<int>(blockIdx.x / nbx) * 64;
  if (m0 >= e.M) return;  // launched to collect
  const int n = static_cast<int>(blockIdx.x % nbx) * 256 + tid;
  const int nn = n < e.N ? n : e.N - 1;
  const float ws = e.wscale[nn];
  const int8_t* wrow = e.w + static_cast<int64_t>(nn) * e.K;
  float acc[64];
#pragma unroll
  for (int r = 0; r < 64; ++r) acc[r] = 0.0f;
  for (int j0 = 0; j0 < cnt; j0 += 32) {
    __syncthreads();
    for (int i = tid; i < 64 * 32; i += 256) {
      const int r = i & 63, c = i >> 6;
      int m = m0 + r;
      m = m < e.M ? m : e.M - 1;
      xs[c][r] = j0 + c < cnt ? to_f32<DT>(e.x[static_cast<int64_t>(m) * e.K + e.list[j0 + c]]) : 0.0f;
    }
    __syncthreads();
    const int cn = cnt - j0 < 32 ? cnt - j0 : 32;
    // The list through the constant address space: the same element for all lanes, read by a scalar load.  Behind the
    // stores of the branch above the compiler would make it a vector load, one more full memory latency per outlier
    // column in front of the weight's: 9 x 4544 x 4096 with 20 columns, bf16, 48.9 us a call against 43.0.
    const auto* list = (const __attribute__((address_space(4))) int32_t*)e.list;
#pragma unroll 1
    for (int c = 0; c < cn; ++c) {
      const float wd = to_f32<DT>(cast_out<DT>(static_cast<float>(wrow[list[j0 + c]]) * ws));
#pragma unroll
      for (int r = 0; r < 64; r += 4) {
        const f32x4 xv = *reinterpret_cast<const f32x4*>(&xs[c][r]);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[r + i] += xv[i] * wd;
      }
    }
  }
  if (n < e.N) {
#pragma unroll
    for (int r = 0; r < 64; ++r)
      if (m0 + r < e.M) sub[static_cast<int64_t>(m0 + r) * e.N + n] = cast_out<DT>(acc[r]);
  }
}

// What the outlier kernel has collected for a tile of BM rows from m0 and BN
// columns from n0 on, as floats: xs [cnt][BM], wd [cnt][BN].
template <int DT, int BM, int BN, int THREADS>
__device__ inline void stage_outliers(const Epi& e, int cnt, int m0, int n0, int tid, float* xs, float* wd) {
  auto rows = [&](const uint16_t* src, int64_t ld, int len, float* dst) {
    for (int i = tid; i < cnt * len / 8; i += THREADS) {
      const int j = i / (len / 8), r = (i - j * (len / 8)) * 8;
      const u32x4 v = *reinterpret_cast<const u32x4*>(src + j * ld + r);
#pragma unroll
      for (int q = 0; q < 8; ++q) dst[j * len + r + q] = to_f32<DT>(static_cast<uint16_t>(v[q >> 1] >> (16 * (q & 1))));
    }
  };
  rows(e.cols + m0, align256(e.M), BM, xs);
  rows(e.cols + kOutCap * align256(e.M) + n0, align256(e.N), BN, wd);
}

// ---------------------------------------------------------------------------
// int8 GEMM
// ---------------------------------------------------------------------------
struct GemmParams {
  const int8_t* qx;  // [M,K]
  Epi e;
  int32_t* acc;      // [runs][M,N] int32, one slab per K run; only with K runs
  int8_t* ow;        // [kStash][N] weight bytes of up to kStash outlier columns, for llm_merge_few_kernel; else null
  int nbx, nby;      // tiles along N and M
  int n_lo, n_hi;    // columns [n_lo, n_hi) of the output belong to this launch
  int tiles_per_run; // k tiles per K run
  int cap;  // outlier columns the epilogue takes through LDS itself; more come from the outlier kernel
};

constexpr int kSlabInts = 32 * 40;  // a wavefront's slab of the GEMMs' epilogues

// XOR applied to the 16-byte piece index of a row in LDS (C pieces per row) so
// that the 16 rows a quarter of a wavefront reads hit distinct LDS banks,
// whether the LDS serves 8 or 16 lanes of a 128-bit read per cycle.
template <int C>
__device__ inline int row_swizzle(int row) {
  if (C == 8) return (row & 7) ^ ((row >> 3) & 1);                             // 128-byte rows
  return ((((row >> 1) ^ (row >> 3)) & 1) << 1) | ((row >> 2) & 1);            // 64-byte rows
}

// Outlier columns whose weight bytes the GEMM with K runs picks out of its own
// tiles as they pass through LDS and leaves in Workspace::ow for the merge kernel
// of up to kFewRows rows: the bytes of one k of w [N,K] lie K apart, for a K of a
// few KiB all behind the same memory channel, and cost far more as loads of that
// kernel's own.  Whole call, K = 4096, N = 11008, 4 rows, 3 outlier columns: 31.1
// -> 22.9 us (28.7 before that kernel's loads went out in batches); K = 8192, N =
// 4096, 3 rows, 20 of them: 66.6 -> 24.8.  (Without K runs the epilogue's gather
// stays: picking was 2 % faster with 8 outlier columns, 1 % slower with none.)
constexpr int kStash = 32;
constexpr int kFewRows = 4;
constexpr int stash_lds_bytes(int bn) { return 512 + kStash * bn; }  // list and count, then [kStash][bn] bytes

// WM x WN wavefronts, each TM x TN blocks of 32x32; k tiles of TK bytes per row
// (128: whole cache lines per row and load; 64 for a K that is not a multiple
// of 128), STAGES of them in LDS.  RUNS: K is cut into runs across workgroups,
// each leaving its sums in its slab of acc; otherwise the epilogue writes out.
// STASH (with RUNS): the outlier columns' weight bytes are picked out of the
// tiles for llm_merge_few_kernel.  An instantiation of its own: as a run-time
// switch it cost the launches without it 2 % (K = 4096, N = 11008, 65 rows, 3
// outlier columns: 38.4 against 37.3 us).
template <int DT, int WM, int WN, int TM, int TN, int TK, int STAGES, bool RUNS, bool STASH>
__global__ __launch_bounds__(WM* WN * 64) __attribute__((amdgpu_waves_per_eu(2))) void llm_gemm_kernel(GemmParams p) {
  constexpr int NW = WM * WN;
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
  constexpr int kTK = TK, kStages = STAGES, C = TK / 16;  // C: 16-byte pieces per row
  constexpr int kABytes = BM * kTK, kBBytes = BN * kTK, kStage = kABytes + kBBytes;
  constexpr int kABlocks = kABytes / 1024, kBBlocks = kBBytes / 1024;  // 1 KiB = one wavefront load
  constexpr int kALoads = (kABlocks + NW - 1) / NW, kBLoads = (kBBlocks + NW - 1) / NW;
  constexpr int kPerStage = kALoads + kBLoads;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int M = p.e.M, K = p.e.K, N = p.e.N;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int r32 = lane & 31, b = lane >> 5;

  // tile of this workgroup.  Consecutive workgroup ids go round the eight
  // XCDs; each XCD gets a band of column tiles with every row tile, so that
  // its L2 holds that band's weights once.
  const int ntiles = p.nbx * p.nby;
  const int run = blockIdx.x / ntiles;
  const int t = blockIdx.x - run * ntiles;
  int bx, by;
  if (p.nbx % 8 == 0) {
    const int xcd = t & 7, idx = t >> 3;
    bx = xcd * (p.nbx / 8) + idx / p.nby;
    by = idx % p.nby;
  } else {
    bx = t / p.nby;
    by = t % p.nby;
  }
  const int m0 = by * BM, n0 = p.n_lo + bx * BN;
  const int ktiles = K / kTK;
  const int t0 = run * p.tiles_per_run;
  const int niter = (ktiles - t0) < p.tiles_per_run ? (ktiles - t0) : p.tiles_per_run;

  // global sources of this lane's direct-to-LDS loads.  LDS piece q (16 bytes)
  // of a tile region is row q / C, slot q % C, and holds the row's logical
  // piece slot ^ swizzle(row).  Rows past M or N repeat the last valid row:
  // computed on valid data, never stored.  Where a region has fewer 1 KiB
  // blocks than there are wavefronts, some blocks are loaded twice.
  // (the casts at the load builtin are needed: with the array element passed as
  // it is, host compilation silently leaves out the kernel's stub and the
  // library does not link)
  const uint8_t* asrc[kALoads];
  int ablk[kALoads];
#pragma unroll
  for (int c = 0; c < kALoads; ++c) {
    ablk[c] = (c * NW + wave) % kABlocks;
    const int q = ablk[c] * 64 + lane;
    const int row = q / C, cc = (q % C) ^ row_swizzle<C>(row);
    int m = m0 + row;
    m = m < M ? m : M - 1;
    asrc[c] = reinterpret_cast<const uint8_t*>(p.qx) + static_cast<int64_t>(m) * K + static_cast<int64_t>(t0) * kTK + cc * 16;
  }
  const uint8_t* bsrc[kBLoads];
  int bblk[kBLoads];
#pragma unroll
  for (int c = 0; c < kBLoads; ++c) {
    bblk[c] = (c * NW + wave) % kBBlocks;
    const int q = bblk[c] * 64 + lane;
    const int row = q / C, cc = (q % C) ^ row_swizzle<C>(row);
    int n = n0 + row;
    n = n < N ? n : N - 1;
    bsrc[c] = reinterpret_cast<const uint8_t*>(p.e.w) + static_cast<int64_t>(n) * K + static_cast<int64_t>(t0) * kTK + cc * 16;
  }
  // tile `it` of this run into its stage; past the end of the run the last
  // tile again, into a spare stage, so that every iteration issues the same
  // number of loads
#define WOL_LLM_ISSUE(it_)                                                                           \
  do {                                                                                               \
    const int koff_ = ((it_) < niter ? (it_) : niter - 1) * kTK;                                      \
    unsigned char* stage_ = smem + ((it_) % kStages) * kStage;                                        \
    _Pragma("unroll") for (int c = 0; c < kALoads; ++c) __builtin_amdgcn_global_load_lds(             \
        reinterpret_cast<const uint8_t*>(asrc[c]) + koff_, (lds_ptr_t)(stage_ + ablk[c] * 1024), 16, 0, 0); \
    _Pragma("unroll") for (int c = 0; c < kBLoads; ++c) __builtin_amdgcn_global_load_lds(             \
        reinterpret_cast<const uint8_t*>(bsrc[c]) + koff_, (lds_ptr_t)(stage_ + kABytes + bblk[c] * 1024), \
        16, 0, 0);                                                                                   \
  } while (0)

  // the outlier list and count, ahead of the tiles in the same in-order stream
  unsigned char* const lds_list = smem + kStages * kStage;
  int8_t* const stash = reinterpret_cast<int8_t*>(lds_list + 512);
  if (STASH && wave == 0) {
    __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint8_t*>(p.e.list + lane), (lds_ptr_t)lds_list, 4, 0, 0);
    __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint8_t*>(p.e.count), (lds_ptr_t)(lds_list + 256), 4, 0, 0);
  }
  int my_k = INT_MAX;  // outlier column number `lane`

  i32x16 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int c = 0; c < TN; ++c)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][c][v] = 0;

  // byte offsets of this lane's fragments inside a stage, for k step 0; k step
  // 1 is the same with the piece index XOR 2
  const int swz = row_swizzle<C>(r32);  // rows are 32 * block + r32: the swizzle has period 16
  int aoff[TM], boff[TN];
#pragma unroll
  for (int a = 0; a < TM; ++a) aoff[a] = ((wm * TM + a) * 32 + r32) * kTK;
#pragma unroll
  for (int c = 0; c < TN; ++c) boff[c] = kABytes + ((wn * TN + c) * 32 + r32) * kTK;

  WOL_LLM_ISSUE(0);
  if (kStages == 3) WOL_LLM_ISSUE(1);
  for (int it = 0; it < niter; ++it) {
    // loads complete in order: all but the newest stage have landed.  A bare
    // s_barrier, not __syncthreads(): the fence of the latter makes the
    // compiler wait for every load in flight, the prefetched tile included.
    wait_vmcnt<(kStages - 2) * kPerStage>();
    __builtin_amdgcn_s_barrier();
    const unsigned char* stage = smem + (it % kStages) * kStage;
    // the fragments of k step ks + 1 are read while the MFMAs of step ks run;
    // those of step 0 while the next tile's loads are issued
    constexpr int KS = C / 2;
    i32x4 af[2][TM], bf[2][TN];
    {
      const int piece = (b ^ swz) * 16;
#pragma unroll
      for (int a = 0; a < TM; ++a) af[0][a] = *reinterpret_cast<const i32x4*>(stage + aoff[a] + piece);
#pragma unroll
      for (int c = 0; c < TN; ++c) bf[0][c] = *reinterpret_cast<const i32x4*>(stage + boff[c] + piece);
    }
    __builtin_amdgcn_sched_barrier(0);
    WOL_LLM_ISSUE(it + kStages - 1);  // into the stage every wavefront finished reading before the barrier
    __builtin_amdgcn_sched_barrier(0);
    if (STASH && it == 0) {  // landed with the first tile
      const int c = *reinterpret_cast<const int*>(lds_list + 256);
      if (c <= kStash && lane < c) my_k = *reinterpret_cast<const int*>(lds_list + lane * 4);
    }
    if (STASH) {
      const int kt = (t0 + it) * kTK;
      unsigned long long hit = __ballot(my_k >= kt && my_k < kt + kTK);
      while (hit != 0) {
        const int j = __builtin_ctzll(hit);
        hit &= hit - 1;
        const int kj = __builtin_amdgcn_readlane(my_k, j) - kt;
        for (int row = tid; row < BN; row += NW * 64)
          stash[j * BN + row] =
              static_cast<int8_t>(stage[kABytes + row * kTK + (((kj >> 4) ^ row_swizzle<C>(row)) << 4) + (kj & 15)]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + 1 < KS) {
        const int piece = (((ks + 1) * 2 + b) ^ swz) * 16;
#pragma unroll
        for (int a = 0; a < TM; ++a)
          af[(ks + 1) & 1][a] = *reinterpret_cast<const i32x4*>(stage + aoff[a] + piece);
#pragma unroll
        for (int c = 0; c < TN; ++c)
          bf[(ks + 1) & 1][c] = *reinterpret_cast<const i32x4*>(stage + boff[c] + piece);
      }
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int c = 0; c < TN; ++c)
          acc[a][c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[ks & 1][a], bf[ks & 1][c], acc[a][c], 0, 0, 0);
      // issue order: the LDS reads of the next step spread between this step's
      // MFMAs (left alone the scheduler reads one fragment, waits, and issues
      // the two MFMAs that use it)
      constexpr int kMfma = TM * TN, kRead = TM + TN;
#pragma unroll
      for (int i = 0; i < kMfma; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        const int reads = ks + 1 < KS ? kRead * (i + 1) / kMfma - kRead * i / kMfma : 0;
#pragma unroll
        for (int r = 0; r < reads; ++r) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);  // nothing moves between k steps
    }
  }
#undef WOL_LLM_ISSUE
  wait_vmcnt<0>();  // the spare-stage loads must have landed before the LDS is reused (or the workgroup ends)

  // accumulator v of a 32x32 block: row 8 * (v / 4) + 4 * (lane / 32) + v % 4, column lane % 32
  const Epi& e = p.e;
  // Each wavefront passes its blocks one at a time through a slab of LDS of its
  // own (32 rows of kSlabRow ints: with that stride the two halves of the
  // wavefront write to disjoint banks) and takes them back as rows: a lane
  // owns eight neighbouring columns of one row, so the output leaves as
  // 16-byte stores (with K runs: as two 16-byte stores into this run's slab of
  // int32 sums).  The loop over the rows is a real loop, which keeps the
  // epilogue's registers few.
  constexpr int kSlabRow = 40;
  __syncthreads();  // every wavefront is done with the stages
  int* slab = reinterpret_cast<int*>(smem) + wave * (32 * kSlabRow);
  const int cnt = RUNS ? 0 : *e.count;
  const int cgrp = (lane & 3) * 8;  // first of this lane's eight columns inside the block
  // few outlier columns: their activations (this tile's rows) and dequantised
  // weights (this tile's columns) go to LDS behind the slabs, as floats
  float* rng = reinterpret_cast<float*>(smem + NW * 32 * kSlabRow * 4);  // [BM]: the tile's row ranges
  float* xs = rng + BM;                                                  // [cnt][BM]
  float* wdl = xs + p.cap * BM;                                          // [cnt][BN]
  const bool fused = !RUNS && cnt > 0 && cnt <= p.cap;
  if (STASH) {
    const int lo = t0 * kTK, hi = (t0 + niter) * kTK;
    unsigned long long got = __ballot(my_k >= lo && my_k < hi);
    for (; got != 0; got &= got - 1) {
      const int j = __builtin_ctzll(got);
      for (int row = tid; row < BN; row += NW * 64)
        if (n0 + row < N) p.ow[static_cast<int64_t>(j) * N + n0 + row] = stash[j * BN + row];
    }
  }
  if (!RUNS) {
    // (read per row out of global memory inside the row loop they cost a
    // memory latency per row, sixteen in a row per wavefront)
    for (int i = tid; i < BM; i += NW * 64) rng[i] = e.ranges[m0 + i < M ? m0 + i : M - 1];
    if (!fused) __syncthreads();
  }
  if (fused) {
    if (e.cols != nullptr && cnt > e.pick) {
      stage_outliers<DT, BM, BN, NW * 64>(e, cnt, m0, n0, tid, xs, wdl);
    } else {  // one row tile, whose workgroup is the only one that needs its columns' weights, or one column
      for (int i = tid; i < cnt * BM; i += NW * 64) {
        const int j = i / BM, m = m0 + i % BM;
        xs[i] = to_f32<DT>(e.x[static_cast<int64_t>(m < M ? m : M - 1) * K + e.list[j]]);
      }
      for (int i = tid; i < cnt * BN; i += NW * 64) {
        const int j = i / BN, n = n0 + i % BN < N ? n0 + i % BN : N - 1;
        wdl[i] = to_f32<DT>(cast_out<DT>(static_cast<float>(e.w[static_cast<int64_t>(n) * K + e.list[j]]) * e.wscale[n]));
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int c = 0; c < TN; ++c) {
    const int n = n0 + (wn * TN + c) * 32 + cgrp;
    const bool n_ok = n < p.n_hi;  // a multiple of 16: eight columns are all inside or all outside
    const int nn = n_ok ? n : 0;
    float ws[8], bias[8];
    if (!RUNS) load_ws_bias8<DT>(e, nn, ws, bias);
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      __builtin_amdgcn_wave_barrier();  // the rows of the previous block have been read
#pragma unroll
      for (int v = 0; v < 16; ++v) slab[(8 * (v >> 2) + 4 * b + (v & 3)) * kSlabRow + r32] = acc[a][c][v];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 1
      for (int h = 0; h < 2; ++h) {
        const int row = h * 16 + (lane >> 2);
        const int m = m0 + (wm * TM + a) * 32 + row;
        if (m >= M || !n_ok) continue;
        const i32x4 s0 = *reinterpret_cast<const i32x4*>(slab + row * kSlabRow + cgrp);
        const i32x4 s1 = *reinterpret_cast<const i32x4*>(slab + row * kSlabRow + cgrp + 4);
        if (RUNS) {  // this run's sums, to be added by the merge kernel
          int32_t* dst = p.acc + (static_cast<int64_t>(run) * M + m) * N + nn;
          *reinterpret_cast<i32x4*>(dst) = s0;
          *reinterpret_cast<i32x4*>(dst + 4) = s1;
          continue;
        }
        finish8<DT>(e, cnt, m, nn, rng[(wm * TM + a) * 32 + row], s0, s1, ws, bias, fused ? xs + (wm * TM + a) * 32 + row : nullptr, BM,
                    wdl + (wn * TN + c) * 32 + cgrp, BN);
      }
    }
  }
}

// The product of more than 128 rows for a K of whole 128-byte k tiles: 256 x 256 or 128 x 256 tiles, a workgroup of two by
// four wavefronts of TM x 4 v_mfma_i32_16x16x64_i8 blocks each.
//
// What bounds it: as in the other large-tile GEMMs the matrix pipes and the power they draw, provided that nothing stands
// between two MFMAs.  Hence the order: the fragment of A block i is read again for the next k step right behind the four
// MFMAs that used it, the next step's B fragments arrive in a second set of registers, and the one workgroup barrier
// of a k tile (two steps of 64 k) sits a quarter into its second step, where the tile's last reads have long arrived; the
// next tile's first fragments are read behind it.  256 rows: two stages of 64 KiB, all loads of tile t + 2 go out right
// behind the barrier that frees their stage; 128 rows: three stages of 48 KiB, the loads spread from barrier to barrier.
// Whole call, us, against 32x32x32 blocks whose first fragments of a tile are read behind its barrier, with an epilogue
// that passes int32 sums through LDS and stores half cache lines: 8192 x 4096 x 12288 490 -> 398 (six rounds of tiles: 50
// in the k loop, 40 without its loads, and 11 in the epilogue each), 2048 x 4096 x 12288 132 -> 114, 300 x 4096 x 4096
// with 20 outlier columns 61.6 -> 49.0.
template <int TM>
constexpr int llm_wide_stages() { return TM == 8 ? 2 : 3; }
template <int TM>
constexpr size_t llm_wide_lds() { return static_cast<size_t>(llm_wide_stages<TM>()) * (TM * 32 + 256) * 128; }

template <int DT, int TM, bool RUNS>
__global__ __launch_bounds__(512) void llm_wide_kernel(GemmParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NW = 8, WN = 4, TN = 4;
  constexpr int BM = TM * 32, BN = 256;
  constexpr int kABytes = BM * 128, kStage = kABytes + BN * 128, kStages = llm_wide_stages<TM>();
  constexpr int kALoads = BM / 64, kLoads = kALoads + 4;  // loads of a tile, per wavefront (1 KiB = 8 rows each)
  constexpr int B0 = TM / 4, S = TM - B0;                 // slots of the second step in front of the barrier, behind it
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int M = p.e.M, K = p.e.K, N = p.e.N;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int lr = lane & 15, kb = lane >> 4;
  int bx, by, run;
  {  // consecutive workgroup ids go to the 8 XCDs in turn, and XCD x takes the x-th eighth of the sequence of (run, tile)
    constexpr int kXcd = 8;
    const int total = gridDim.x, x = blockIdx.x % kXcd, q = total / kXcd, r = total % kXcd;
    const int pos = x * q + (x < r ? x : r) + blockIdx.x / kXcd;
    run = pos / (p.nbx * p.nby);
    tile_of_position(pos - run * (p.nbx * p.nby), p.nbx, p.nby, &bx, &by);
  }
  const int m0 = by * BM, n0 = p.n_lo + bx * BN;
  const int t0 = run * p.tiles_per_run;  // this workgroup's run of k tiles
  const int nt = K / 128 - t0 < p.tiles_per_run ? K / 128 - t0 : p.tiles_per_run;

  // One descriptor per load, over the load's own eight rows as far as they exist: what lies past M or N arrives as zeros.
  __amdgpu_buffer_rsrc_t ra[kALoads], rb[4];
  auto rows_desc = [&](const int8_t* base, int row0, int rows) {
    const int nr = rows - row0 > 8 ? 8 : (rows > row0 ? rows - row0 : 0);
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(base + static_cast<int64_t>(nr > 0 ? row0 : 0) * K), 0, nr * K, 0x00020000);
  };
#pragma unroll
  for (int c = 0; c < kALoads; ++c) ra[c] = rows_desc(p.qx, m0 + (c * NW + wave) * 8, M);
#pragma unroll
  for (int c = 0; c < 4; ++c) rb[c] = rows_desc(p.e.w, n0 + (c * NW + wave) * 8, N);
  // rows of 128 bytes in LDS, the 16-byte piece XORed with row % 8
  const uint32_t off = static_cast<uint32_t>((lane / 8) * K + ((lane ^ (lane >> 3)) & 7) * 16);
  auto issue = [&](int t, int st, int i) {
    const int tt = t0 + (t < nt ? t : nt - 1);  // past the end: the last tile again, into a stage that nobody reads
    unsigned char* s = smem + st * kStage + (i < kALoads ? 0 : kABytes) + ((i < kALoads ? i : i - kALoads) * NW + wave) * 1024;
    if (i < kALoads) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra[i], (lds_ptr_t)s, 16, off, tt * 128, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rb[i - kALoads], (lds_ptr_t)s, 16, off, tt * 128, 0, 0);
  };

  i32x4 acc[TM][TN], af[TM], bf[2][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int c = 0; c < TN; ++c) acc[a][c] = i32x4{0, 0, 0, 0};
  const int swz = (kb ^ (lr & 7)) * 16;  // step 1's piece is four further on: XOR 64
  const int apos = (wm * TM * 16 + lr) * 128 + swz, bpos = kABytes + (wn * TN * 16 + lr) * 128 + swz;
  auto read_a = [&](const unsigned char* s, int h, int i) { af[i] = *reinterpret_cast<const i32x4*>(s + (h ? apos ^ 64 : apos) + i * 2048); };
  auto read_b = [&](const unsigned char* s, int h, int c) { bf[h][c] = *reinterpret_cast<const i32x4*>(s + (h ? bpos ^ 64 : bpos) + c * 2048); };
  auto mfmas = [&](int h, int a) {
#pragma unroll
    for (int c = 0; c < TN; ++c) acc[a][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bf[h][c], af[a], acc[a][c], 0, 0, 0);
  };

#pragma unroll
  for (int t = 0; t < kStages - 1; ++t)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) issue(t, t, i);
  // three stages: the part of tile 2 that the loop's first tile does not bring
  auto share = [&](int pos) { return kLoads * pos / (2 * TM); };
  constexpr int kFirst = kStages == 3 ? kLoads * S / (2 * TM) : kLoads;
#pragma unroll
  for (int i = 0; i < kFirst; ++i) issue(kStages - 1, kStages - 1, i);
  wait_vmcnt<(kStages - 2) * kLoads + kFirst>();  // tile 0 has landed
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int c = 0; c < TN; ++c) read_b(smem, 0, c);
#pragma unroll
  for (int a = 0; a < TM; ++a) read_a(smem, 0, a);

  int st = 0;
  for (int t = 0; t < nt; ++t) {
    const int st_n = st == kStages - 1 ? 0 : st + 1, st_p = st == 0 ? kStages - 1 : st - 1;
    const unsigned char* s = smem + st * kStage;
    const unsigned char* n = smem + st_n * kStage;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      mfmas(0, i);
      __builtin_amdgcn_sched_barrier(0);
      if (i < 2) {
        read_b(s, 1, 2 * i);
        read_b(s, 1, 2 * i + 1);
      }
      read_a(s, 1, i);
      if (kStages == 3) {
#pragma unroll
        for (int l = share(S + i); l < share(S + i + 1); ++l) issue(t + 2, st_p, l);
      }
    }
#pragma unroll
    for (int i = 0; i < B0; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      mfmas(1, i);
      if (kStages == 3) {
#pragma unroll
        for (int l = share(S + TM + i); l < share(S + TM + i + 1); ++l) issue(t + 2, st_p, l);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // lgkmcnt(0): this wavefront needs nothing more of the tile; tile t + 1 has landed
    __builtin_amdgcn_s_waitcnt(0x0070 | (kStages == 3 ? kLoads : 0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < S; ++i) {
      mfmas(1, B0 + i);
      __builtin_amdgcn_sched_barrier(0);
      if (i < 2) {
        read_b(n, 0, 2 * i);
        read_b(n, 0, 2 * i + 1);
      }
#pragma unroll
      for (int a = i > 0 ? TM * (i - 1) / (S - 1) : 0; a < TM * i / (S - 1); ++a) read_a(n, 0, a);
      if (kStages == 3) {
#pragma unroll
        for (int l = share(i); l < share(i + 1); ++l) issue(t + 3, st, l);
      } else {
#pragma unroll
        for (int l = kLoads * i / S; l < kLoads * (i + 1) / S; ++l) issue(t + 2, st, l);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    st = st_n;
  }
  __builtin_amdgcn_s_waitcnt(0x0070);
  __builtin_amdgcn_s_barrier();  // the spare loads are done and every wavefront has stopped reading

  // ---- epilogue.  The weight rows were the MFMA's first operand: element r of lane l is row l % 16 of x, column
  // 4 * (l / 16) + r of its block, so that a lane finishes four neighbouring columns, and 32 rows x 64 columns of T
  // leave through a slab of the wavefront's own as whole cache lines.
  const Epi& e = p.e;
  constexpr int kRow = 64 + 8;  // elements: the sixteen rows of a store to the slab lie in different banks
  static_assert(32 * kRow * 2 <= kSlabInts * 4, "fused_cap counts on slabs of kSlabInts");
  int etid = threadIdx.x;
  asm volatile("" : "+v"(etid));  // nothing of the epilogue's addresses is kept in registers during the loop
  const int el = etid & 63, er = el & 15, ec = (el >> 4) * 4;
  if constexpr (RUNS) {  // this run's sums, to be added by the merge kernel
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int c = 0; c < TN; ++c) {
        const int m = m0 + (wm * TM + a) * 16 + er, n = n0 + wn * 64 + c * 16 + ec;
        if (m < M && n < p.n_hi) *reinterpret_cast<i32x4*>(p.acc + (static_cast<int64_t>(run) * M + m) * N + n) = acc[a][c];
      }
    return;
  }
  uint16_t* slab = reinterpret_cast<uint16_t*>(smem) + wave * (32 * kRow);
  const int cnt = *e.count;
  float* rng = reinterpret_cast<float*>(smem + NW * kSlabInts * 4);  // [BM]: the tile's row ranges
  float* xs = rng + BM;                                              // [cnt][BM]
  float* wdl = xs + p.cap * BM;                                      // [cnt][BN]
  const bool fused = cnt > 0 && cnt <= p.cap;
  for (int i = etid; i < BM; i += NW * 64) rng[i] = e.ranges[m0 + i < M ? m0 + i : M - 1];
  if (fused) stage_outliers<DT, BM, BN, NW * 64>(e, cnt, m0, n0, etid, xs, wdl);
  const int nw = n0 + wn * 64;  // the wavefront's first column
  const bool has_bias = e.bias != nullptr;
  f32x4 ws[TN], bias[TN];
#pragma unroll
  for (int c = 0; c < TN; ++c) {
    const int n = nw + c * 16 < p.n_hi ? nw + c * 16 + ec : 0;
    ws[c] = *reinterpret_cast<const f32x4*>(e.wscale + n);
#pragma unroll
    for (int r = 0; r < 4; ++r) bias[c][r] = has_bias ? to_f32<DT>(e.bias[n + r]) : 0.0f;
  }
  __syncthreads();
  // piece q of the slab: eight columns of one row, the wavefront's 64 lanes on eight rows
  auto each_piece = [&](int a, auto&& f) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = q * 8 + (el >> 3), m = m0 + (wm * TM + a) * 16 + row, n = nw + (el & 7) * 8;
      if (m < M && n < p.n_hi)
        f(reinterpret_cast<u32x4*>(slab + row * kRow + (el & 7) * 8), reinterpret_cast<u32x4*>(e.out + static_cast<int64_t>(m) * N + n));
    }
  };
  auto settle = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto emit = [&](int a, int h, int c, auto&& one) {  // block (a + h, c): one(r) is its element r as T
    u32x2 o;
    o.x = static_cast<uint32_t>(one(0)) | (static_cast<uint32_t>(one(1)) << 16);
    o.y = static_cast<uint32_t>(one(2)) | (static_cast<uint32_t>(one(3)) << 16);
    *reinterpret_cast<u32x2*>(slab + (h * 16 + er) * kRow + c * 16 + ec) = o;
  };
#pragma unroll
  for (int a = 0; a < TM; a += 2) {
    const int row = (wm * TM + a) * 16 + er;  // of the tile; the second block's is 16 further on
    const float range[2] = {rng[row], rng[row + 16]};
    if (cnt == 0) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < TN; ++c)
          emit(a, h, c, [&](int r) { return merge_plain<DT>(acc[a + h][c][r], range[h], ws[c][r], has_bias, bias[c][r]); });
    } else {
      f32x4 sub[2][TN];  // the outlier columns' product
      if (fused) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int c = 0; c < TN; ++c) sub[h][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int j = 0; j < cnt; ++j) {
          const float xv[2] = {xs[j * BM + row], xs[j * BM + row + 16]};
#pragma unroll
          for (int c = 0; c < TN; ++c) {
            const f32x4 wd = *reinterpret_cast<const f32x4*>(wdl + j * BN + wn * 64 + c * 16 + ec);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int r = 0; r < 4; ++r) sub[h][c][r] += xv[h] * wd[r];
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int c = 0; c < TN; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) sub[h][c][r] = to_f32<DT>(cast_out<DT>(sub[h][c][r]));
      } else {  // as the outlier kernel left it in the output's own place
        each_piece(a, [&](u32x4* l, u32x4* g) { *l = *g; });
        settle();
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int c = 0; c < TN; ++c) {
            const u32x2 v = *reinterpret_cast<const u32x2*>(slab + (h * 16 + er) * kRow + c * 16 + ec);
#pragma unroll
            for (int r = 0; r < 4; ++r) sub[h][c][r] = to_f32<DT>(static_cast<uint16_t>(v[r >> 1] >> (16 * (r & 1))));
          }
        settle();
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < TN; ++c)
          emit(a, h, c, [&](int r) { return static_cast<uint16_t>(merge_one<DT>(acc[a + h][c][r], sub[h][c][r], range[h], ws[c][r], has_bias, bias[c][r])); });
    }
    settle();
    each_piece(a, [&](u32x4* l, u32x4* g) { *g = *l; });
    settle();  // the rows have been read
  }
#endif
}

// Adds the K runs' int32 sums and finishes; one thread per eight columns.
template <int DT>
__global__ __launch_bounds__(256) void llm_merge_kernel(const int32_t* __restrict__ acc, int runs, Epi e) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int groups = e.N / 8;
  if (i >= static_cast<int64_t>(e.M) * groups) return;
  const int m = static_cast<int>(i / groups);
  const int nn = static_cast<int>(i - static_cast<int64_t>(m) * groups) * 8;
  const int64_t slab = static_cast<int64_t>(e.M) * e.N;
  const int32_t* src = acc + static_cast<int64_t>(m) * e.N + nn;
  i32x4 s0 = {0, 0, 0, 0}, s1 = {0, 0, 0, 0};
  for (int r = 0; r < runs; ++r) {
    s0 += *reinterpret_cast<const i32x4*>(src + r * slab);
    s1 += *reinterpret_cast<const i32x4*>(src + r * slab + 4);
  }
  float ws[8], bias[8];
  load_ws_bias8<DT>(e, nn, ws, bias);
  finish8<DT>(e, *e.count, m, nn, e.ranges[m], s0, s1, ws, bias, nullptr, 0, nullptr, 0);
}

// The same for up to kFewRows rows, the outlier columns multiplied here (no
// outlier kernel ran).  Latency-bound: a thread takes one column of all rows, so
// that every weight byte is fetched once, eight of them in flight at a time.
template <int DT>
__global__ __launch_bounds__(64) void llm_merge_few_kernel(const int32_t* __restrict__ acc, int runs, Epi e,
                                                           const int8_t* __restrict__ ow) {
  const int n = blockIdx.x * 64 + threadIdx.x;
  if (n >= e.N) return;
  const int cnt = *e.count;
  const int64_t slab = static_cast<int64_t>(e.M) * e.N;
  int32_t sum[kFewRows] = {0, 0, 0, 0};
#pragma unroll 4
  for (int r = 0; r < runs; ++r)
#pragma unroll
    for (int m = 0; m < kFewRows; ++m)
      sum[m] += acc[r * slab + static_cast<int64_t>(m < e.M ? m : e.M - 1) * e.N + n];
  const float ws = e.wscale[n];
  const float bias = e.bias != nullptr ? to_f32<DT>(e.bias[n]) : 0.0f;
  const int8_t* wrow = e.w + static_cast<int64_t>(n) * e.K;
  float sub[kFewRows] = {0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int W = 8;
  const bool picked = cnt <= kStash;  // more than the GEMM picks: out of the weight itself
  for (int j0 = 0; j0 < cnt; j0 += W) {  // ascending k, as everywhere
    // every load of the batch under no condition (past the end: the last column, the last row again)
    int k[W];
    float w[W], xv[W][kFewRows];
#pragma unroll
    for (int u = 0; u < W; ++u) k[u] = e.list[j0 + u < cnt ? j0 + u : cnt - 1];
#pragma unroll
    for (int u = 0; u < W; ++u) {
      const int j = j0 + u < cnt ? j0 + u : cnt - 1;
      w[u] = static_cast<float>(picked ? ow[static_cast<int64_t>(j) * e.N + n] : wrow[k[u]]);
#pragma unroll
      for (int m = 0; m < kFewRows; ++m)
        xv[u][m] = to_f32<DT>(e.x[static_cast<int64_t>(m < e.M ? m : e.M - 1) * e.K + k[u]]);
    }
#pragma unroll
    for (int u = 0; u < W; ++u) {
      const float wd = to_f32<DT>(cast_out<DT>(w[u] * ws));
#pragma unroll
      for (int m = 0; m < kFewRows; ++m) sub[m] = j0 + u < cnt ? sub[m] + xv[u][m] * wd : sub[m];
    }
  }
#pragma unroll
  for (int m = 0; m < kFewRows; ++m)
    if (m < e.M)
      e.out[static_cast<int64_t>(m) * e.N + n] = static_cast<uint16_t>(
          merge_one<DT>(sum[m], to_f32<DT>(cast_out<DT>(sub[m])), e.ranges[m], ws, e.bias != nullptr, bias));
}

struct Plan {
  int bm, bn;     // tile
  int tk;         // k bytes per tile row
  int whole_cols; // many rows: the first whole_cols columns get 256x256 tiles, the rest 128x256
  int runs;       // K runs (1: the GEMM writes the output itself)
  int tiles_per_run;
};

// Up to 128 rows: one row tile of 32, 64 or 128 rows, 128 columns wide so that
// the column tiles spread over the CUs, and K cut into runs while CUs are
// still idle, every run keeps 256 k and the runs' int32 sums (written and read
// once each) stay below the weight bytes.
Plan make_plan(int64_t M, int64_t K, int64_t N) {
  Plan pl;
  pl.whole_cols = 0;
  const int tk = K % 128 == 0 ? 128 : 64;
  const int64_t ktiles = K / tk;
  int64_t runs = 1;
  if (M > 128) {
    // 128-deep tiles, eight wavefronts, one workgroup per CU: 256x256 with two
    // stages, or 128x256 with three where their rounds over the CUs come out
    // shorter (a half tile takes 0.55 of a whole one; 384 whole tiles on 256
    // CUs are two rounds, 768 half tiles three).  64-deep tiles (K not a
    // multiple of 128): 256x128, three stages, two workgroups of four per CU.
    pl.bm = 256;
    pl.bn = tk == 128 ? 256 : 128;
    if (tk == 128) {
      // a launch takes ceil(tiles / CUs) tile times: the columns are shared
      // out so that whole tiles fill whole rounds of the CUs
      const int64_t cus = num_cus();
      const int64_t cols = (N + 255) / 256, rows256 = (M + 255) / 256, rows128 = (M + 127) / 128;
      int64_t best_c = cols, best_t = INT64_MAX;
      for (int64_t c = cols; c >= 0; --c) {
        const int64_t t = 20 * ((c * rows256 + cus - 1) / cus) + 11 * (((cols - c) * rows128 + cus - 1) / cus);
        if (t < best_t) {
          best_t = t;
          best_c = c;
        }
      }
      pl.whole_cols = static_cast<int>(best_c * 256 < N ? best_c * 256 : N);
      if (best_c == 0) pl.bm = 128;
      // Few tiles leave CUs idle: half tiles with K cut into runs, by the estimate in us of a round (a k tile of a whole
      // tile takes 1.7, of a half one 1.0, their starts and ends 11 and 6, 4 with sums instead of results) and of the
      // merge launch with the sums' way through memory.  The 0.8: with runs the outlier columns' product is a pass of its
      // own, which the estimate cannot know; where it promises less (ten problems between 0.8 and 0.9) one run is 1 / 5 / 11 /
      // 19 % faster with 0 / 1 / 8 / 20 outlier columns.  Whole call, us, one run against this: 200 x 8192 x 3008
      // 56.0 -> 34.7, with 5 outlier columns 42.0; 1024 x 11008 x 4096 102 -> 79; 300 x 4096 x 4096 with 20 outlier
      // columns 49.0 -> 51.3.
      const double kt = static_cast<double>(ktiles);
      const double one = (best_c * rows256 + cus - 1) / cus * (1.7 * kt + 11) + ((cols - best_c) * rows128 + cus - 1) / cus * (1.0 * kt + 6);
      double best = 0.8 * one;
      int64_t best_r = 1;
      for (int64_t r = 2; r <= 8 && ktiles / r >= 4; ++r) {
        const int64_t per = (ktiles + r - 1) / r, eff = (ktiles + per - 1) / per;
        const double t = static_cast<double>((cols * rows128 * eff + cus - 1) / cus) * (1.0 * per + 4) + 4 +
                         static_cast<double>(M) * N * (8 * eff + 2) / 4.5e6;
        if (t < best) {
          best = t;
          best_r = eff;
        }
      }
      if (best_r > 1) {
        pl.bm = 128;
        pl.whole_cols = 0;
        runs = best_r;
      }
    }
  } else {
    pl.bm = M > 64 ? 128 : (M > 32 ? 64 : 32);
    pl.bn = 128;
    const int64_t tiles = (N + pl.bn - 1) / pl.bn;
    runs = 2 * num_cus() / tiles;  // two workgroups fit a CU: no second, nearly empty round
    if (runs > ktiles * tk / 256) runs = ktiles * tk / 256;  // at least 256 k per run
    if (runs > K / (8 * M)) runs = K / (8 * M);
    if (runs < 1) runs = 1;
  }
  int64_t per = (ktiles + runs - 1) / runs;
  runs = (ktiles + per - 1) / per;
  pl.tk = tk;
  pl.runs = static_cast<int>(runs);
  pl.tiles_per_run = static_cast<int>(per);
  return pl;
}

struct Workspace {
  float* ranges;
  int32_t* mask;
  uint32_t* part;
  int32_t* count;
  int32_t* list;
  int8_t* qx;
  int32_t* acc;
  int8_t* ow;
  uint16_t* cols;
  int64_t bytes;
};

Workspace carve(void* base, int64_t M, int64_t K, int64_t N, int runs) {
  if (runs <= 1) runs = 0;
  unsigned char* p = static_cast<unsigned char*>(base);
  int64_t off = 0;
  Workspace w;
  w.ranges = reinterpret_cast<float*>(p + off);
  off += align256(M * 4);
  w.mask = reinterpret_cast<int32_t*>(p + off);
  off += align256(K / 32 * 4);
  w.part = reinterpret_cast<uint32_t*>(p + off);
  off += align256(static_cast<int64_t>(kMaxRowGroups) * (K / 32) * 4);
  w.count = reinterpret_cast<int32_t*>(p + off);
  off += 256;
  w.list = reinterpret_cast<int32_t*>(p + off);
  off += align256(K * 4);
  w.qx = reinterpret_cast<int8_t*>(p + off);
  off += align256(M * K);
  w.acc = reinterpret_cast<int32_t*>(p + off);
  off += align256(M * N * 4 * runs);
  w.ow = reinterpret_cast<int8_t*>(p + off);
  if (runs > 1 && M <= kFewRows) off += align256(kStash * N);
  w.cols = reinterpret_cast<uint16_t*>(p + off);
  if (runs == 0) off += kOutCap * (align256(M) + align256(N)) * 2;
  w.bytes = off;
  return w;
}

template <int DT, int WM, int WN, int TM, int TN, int TK, int STAGES, bool RUNS, bool STASH = false>
int launch_gemm(const GemmParams& p, int runs, hipStream_t stream) {
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
  constexpr size_t stages = static_cast<size_t>(STAGES) * (BM + BN) * TK, lds = stages + (STASH ? stash_lds_bytes(BN) : 0);
  static_assert(stages >= static_cast<size_t>(WM * WN) * 32 * 40 * 4 + BM * 4,
                "the epilogue's slabs and row ranges must fit the stages");
  static std::atomic<uint32_t> done{0};
  auto kern = llm_gemm_kernel<DT, WM, WN, TM, TN, TK, STAGES, RUNS, STASH>;
  allow_lds(reinterpret_cast<const void*>(kern), lds, done);
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(p.nbx * p.nby * runs)), dim3(WM * WN * 64), lds, stream,
                     p);
  return check_launch();
}

template <int DT, int TM, bool RUNS>
int launch_wide(const GemmParams& p, int runs, hipStream_t stream) {
  static std::atomic<uint32_t> done{0};
  auto kern = llm_wide_kernel<DT, TM, RUNS>;
  allow_lds(reinterpret_cast<const void*>(kern), llm_wide_lds<TM>(), done);
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(p.nbx * p.nby * runs)), dim3(512), llm_wide_lds<TM>(), stream, p);
  return check_launch();
}

template <int DT, int TK, bool RUNS>
int launch_gemm_for(const GemmParams& p, const Plan& pl, hipStream_t stream) {
  switch (pl.bm) {
    case 256:
      if (RUNS) return WOL_ERR_BAD_SHAPE;  // make_plan cuts K only for tiles of at most 128 rows
      if (pl.bn == 256) return launch_wide<DT, 8, false>(p, 1, stream);
      return launch_gemm<DT, 2, 2, 4, 2, 64, 3, false>(p, pl.runs, stream);
    case 128:
      if (pl.bn == 256) {
        if (TK != 128) return WOL_ERR_BAD_SHAPE;  // make_plan: many rows, 128-deep tiles
        return launch_wide<DT, 4, RUNS>(p, pl.runs, stream);
      }
      return launch_gemm<DT, 1, 4, 4, 1, TK, 3, RUNS>(p, pl.runs, stream);
    case 64: return launch_gemm<DT, 1, 4, 2, 1, TK, 3, RUNS>(p, pl.runs, stream);
    default:
      if constexpr (RUNS)
        if (p.ow != nullptr) return launch_gemm<DT, 1, 4, 1, 1, TK, 3, true, true>(p, pl.runs, stream);
      return launch_gemm<DT, 1, 4, 1, 1, TK, 3, RUNS>(p, pl.runs, stream);
  }
}

template <int DT, bool RUNS>
int launch_gemm_tk(const GemmParams& p, const Plan& pl, hipStream_t stream) {
  return pl.tk == 128 ? launch_gemm_for<DT, 128, RUNS>(p, pl, stream) : launch_gemm_for<DT, 64, RUNS>(p, pl, stream);
}

// Outlier columns the GEMM's epilogue can hold in LDS behind its slabs (at most
// kOutCap): (rows + columns of the tile) floats each.
int fused_cap(const Plan& pl) {
  if (pl.runs > 1) return 0;  // the merge kernel reads the outlier kernel's product
  const bool eight = pl.bn == 256;  // the configurations of eight wavefronts
  const int64_t lds = static_cast<int64_t>(pl.bm == 256 && eight ? 2 : 3) * (pl.bm + pl.bn) * pl.tk;
  const int64_t room = lds - (eight ? 8 : 4) * kSlabInts * 4 - pl.bm * 4;  // slabs, row ranges
  const int64_t cap = room / ((pl.bm + pl.bn) * 4);
  return static_cast<int>(cap > kOutCap ? kOutCap : (cap < 0 ? 0 : cap));
}

template <int DT>
int run_llm_int8(const void* x, const void* weight, const void* bias, const float* wscale, float threshold,
                 int64_t M, int64_t K, int64_t N, void* out, void* workspace, hipStream_t stream) {
  const Plan pl = make_plan(M, K, N);
  const Workspace ws = carve(workspace, M, K, N, pl.runs);
  const uint16_t* xs = static_cast<const uint16_t*>(x);
  const bool small = M <= kSmallRows - (K > kSmallRowsMaxK ? 1 : 0) && K <= kSmallMaxK;
  if (small) {
    hipLaunchKernelGGL(llm_act_small_kernel<DT>, dim3(static_cast<unsigned>(M + 1)), dim3(kSmallThreads), static_cast<size_t>(K / 32 * 4), stream,
                       xs, threshold, static_cast<int>(M), static_cast<int>(K), ws.ranges, ws.mask, ws.qx, ws.count,
                       ws.list);
  }
  if (!small) {
    // at most kMaxRowGroups workgroups, each a whole number of four-row chunks
    int64_t rows_per_group = (M + kMaxRowGroups - 1) / kMaxRowGroups;
    rows_per_group = (rows_per_group + kRowChunk - 1) / kRowChunk * kRowChunk;
    const int groups = static_cast<int>((M + rows_per_group - 1) / rows_per_group);
    const size_t mask_lds = static_cast<size_t>(K / 32) * 4;
    hipLaunchKernelGGL(llm_rowmax_kernel<DT>, dim3(static_cast<unsigned>(groups)), dim3(256), mask_lds, stream, xs,
                       threshold, static_cast<int>(M), static_cast<int>(K), static_cast<int>(rows_per_group),
                       ws.ranges, ws.part);
    // up to four partial masks (16 rows) the quant kernel ORs itself: cheaper
    // than a launch (26.1 against 27.8 us at 8 rows; with 16 masks it loses 2 us)
    const bool or_in_quant = groups <= 4;
    if (!or_in_quant)
      hipLaunchKernelGGL(llm_mask_kernel, dim3(static_cast<unsigned>((K / 32 + 3) / 4)), dim3(256), 0, stream,
                         ws.part, groups, static_cast<int>(K), ws.mask);
    const int64_t nvec = M * K / 16;
    int64_t qblocks = (nvec + 255) / 256;
    if (qblocks > 8192) qblocks = 8192;
    hipLaunchKernelGGL(llm_quant_kernel<DT>, dim3(static_cast<unsigned>(qblocks + 1)), dim3(256), 0, stream, xs,
                       ws.ranges, ws.mask, ws.part, or_in_quant ? groups : 0, static_cast<int>(M),
                       static_cast<int>(K), ws.qx, ws.count, ws.list);
  }
  GemmParams p;
  p.qx = ws.qx;
  p.e = Epi{xs, static_cast<const int8_t*>(weight), wscale, ws.ranges, static_cast<const uint16_t*>(bias),
            ws.count, ws.list, static_cast<uint16_t*>(out), static_cast<int>(M), static_cast<int>(K),
            static_cast<int>(N), pl.bn == 256 ? 0 : 1, ws.cols};  // 256 columns: llm_wide_kernel, which cannot pick
  p.acc = ws.acc;
  p.ow = pl.runs > 1 && M <= kFewRows ? ws.ow : nullptr;
  p.n_lo = 0;
  p.n_hi = static_cast<int>(N);
  p.nbx = static_cast<int>((N + pl.bn - 1) / pl.bn);
  p.nby = static_cast<int>((M + pl.bm - 1) / pl.bm);
  p.tiles_per_run = pl.tiles_per_run;
  p.cap = fused_cap(pl);
  if (pl.runs == 1 && pl.bm == 256 && pl.bn == 256 && pl.whole_cols < N) {
    Plan half = pl;
    half.bm = 128;
    const int c = fused_cap(half);  // both launches and the outlier kernel go by one limit
    p.cap = c < p.cap ? c : p.cap;
  }
  // up to four rows with K runs the merge kernel multiplies the outlier columns
  // itself (a launch costs more than that work)
  const bool direct = pl.runs > 1 && M <= kFewRows;
  if (!direct) {
    // Few columns: collected once for all row tiles, by enough workgroups that no thread fetches many elements one after
    // the other (300 x 4544 -> 4096, fp16, 20 columns, 90.0 us a call when every tile picks, 81 so).  Up to 128 rows
    // there is one row tile, and the GEMM picks a column's weights exactly once (101 x 1024 -> 1024, bf16, 20 columns, us a
    // call: collected on the workgroups of the product 38.5, on enough of them 33.1, picked 32.9; 3 columns 25.1 / 24.0 /
    // 23.7).  Nor is a single column worth collecting for llm_gemm_kernel (Epi::pick): 129 x 2112 -> 12288, bf16, 39.4
    // collected, 38.7 picked, 256 rows 41.1 / 40.1; with 3 columns collecting is level (41.7 / 41.6) and gains from there.
    int64_t blocks = ((N + 255) / 256) * ((M + 63) / 64);  // one per 64 x 256 piece of the product
    if (M <= 128) p.e.cols = nullptr;
    const int64_t collect = p.e.cols != nullptr ? (p.cap * (M + N) + 255) / 256 : 0;
    if (blocks < collect) blocks = collect < 1024 ? collect : (blocks < 1024 ? 1024 : blocks);
    hipLaunchKernelGGL(llm_outlier_kernel<DT>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, p.e, p.cap);
  }
  if (check_launch() != WOL_OK) return WOL_ERR_HIP;
  if (pl.runs == 1 && pl.bm == 256 && pl.bn == 256 && pl.whole_cols < N) {
    // 256x256 tiles on the first columns, 128x256 tiles on the rest
    p.n_hi = pl.whole_cols;
    p.nbx = pl.whole_cols / 256;
    const int rc = launch_gemm_tk<DT, false>(p, pl, stream);
    if (rc != WOL_OK) return rc;
    Plan half = pl;
    half.bm = 128;
    p.n_lo = pl.whole_cols;
    p.n_hi = static_cast<int>(N);
    p.nbx = static_cast<int>((N - pl.whole_cols + 255) / 256);
    p.nby = static_cast<int>((M + 127) / 128);
    return launch_gemm_tk<DT, false>(p, half, stream);
  }
  if (pl.runs == 1) return launch_gemm_tk<DT, false>(p, pl, stream);
  const int rc = launch_gemm_tk<DT, true>(p, pl, stream);
  if (rc != WOL_OK) return rc;
  if (direct) {
    hipLaunchKernelGGL(llm_merge_few_kernel<DT>, dim3(static_cast<unsigned>((N + 63) / 64)), dim3(64), 0, stream,
                       ws.acc, pl.runs, p.e, ws.ow);
    return check_launch();
  }
  const int64_t total = M * (N / 8);
  hipLaunchKernelGGL(llm_merge_kernel<DT>, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, stream,
                     ws.acc, pl.runs, p.e);
  return check_launch();
}

}  // namespace

size_t llm_int8_workspace(int64_t M, int64_t K, int64_t N) {
  const Plan pl = make_plan(M, K, N);
  return static_cast<size_t>(carve(nullptr, M, K, N, pl.runs).bytes);
}

void llm_int8_workspace_offsets(int64_t M, int64_t K, int64_t N, int64_t* offsets) {
  const Plan pl = make_plan(M, K, N);
  const Workspace w = carve(nullptr, M, K, N, pl.runs);
  offsets[0] = reinterpret_cast<intptr_t>(w.ranges);
  offsets[1] = reinterpret_cast<intptr_t>(w.mask);
  offsets[2] = reinterpret_cast<intptr_t>(w.count);
  offsets[3] = reinterpret_cast<intptr_t>(w.list);
  offsets[4] = reinterpret_cast<intptr_t>(w.qx);
  offsets[5] = pl.runs > 1 ? reinterpret_cast<intptr_t>(w.acc) : -1;
  offsets[6] = pl.runs;
}

int launch_llm_int8_linear(const void* x, const void* weight, const void* bias, const float* wscale,
                           float threshold, int dtype, int64_t M, int64_t K, int64_t N, void* out,
                           void* workspace, hipStream_t stream) {
  if (dtype == WOL_DTYPE_BF16)
    return run_llm_int8<WOL_DTYPE_BF16>(x, weight, bias, wscale, threshold, M, K, N, out, workspace, stream);
  return run_llm_int8<WOL_DTYPE_F16>(x, weight, bias, wscale, threshold, M, K, N, out, workspace, stream);
}

}  // namespace wol
