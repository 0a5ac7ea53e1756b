// weight_only_linear for large M (prefill): MFMA GEMMs.
//
// For a K made of whole k tiles (64 k for int8, 128 k for int4) up to 64 rows run
// on gemm_dma_kernel: a workgroup of eight wavefronts side by side computes a BM
// x BN tile of the output from TM x TN blocks of v_mfma_f32_32x32x16 per
// wavefront; more rows on the tiles of wol_linear_wide.hip, planned here.  Both
// operands travel global -> LDS with direct-to-LDS loads; the packed weights
// land as they lie in memory and are dequantised in registers to exact signed
// bf16/fp16 integers on their way into the B operand; scales are applied to fp32
// accumulators -- in the epilogue (per-channel) or once per group -- so code *
// scale is never rounded to T.  For few rows K is cut into runs across
// workgroups whose fp32 partial sums reduce_partials_kernel adds.  Workgroups
// are numbered so that each XCD (one L2 each) works on a compact block of
// neighbouring tiles.
//
// gemm_kernel (v_mfma_f32_16x16x32, activations staged through registers into
// padded LDS rows, weights loaded straight into B-fragment order) takes the
// remaining K: those that end in a partial k tile.
#include "wol_gemm_common.h"

namespace wol {

// A GEMM call on its way from the entry points to the kernels of its element
// type, which are compiled as two translation units side by side: this file
// for bf16, and through wol_linear_gemm_f16.hip for fp16.
struct GemmArgs {
  const void* x; const void* codes; const void* bias; const void* scale; void* out;
  int M, K, N, gshift, out_f32;
  void* ws; size_t ws_bytes;  // scratch for split-K partial sums, may be null
  hipStream_t stream;
  int act;
};

// One product of moe_ffn (see MoeLaunch below).
struct MoeGemmArgs {
  const void* x; const int* table; int max_tiles, bm, ns; bool narrow; int64_t rows; float* partial; const int64_t* valid_rows;
  const void* codes; const void* bias; const void* scale; int64_t K, N; void* out; hipStream_t stream; bool swiglu;
};

void gemm_bf16(const GemmArgs& a, int bits);
void gemm_f16(const GemmArgs& a, int bits);
void swiglu_gemm_bf16(const GemmArgs& a, int bits);
void swiglu_gemm_f16(const GemmArgs& a, int bits);
void moe_gemm_bf16(const MoeGemmArgs& a, int bits);
void moe_gemm_f16(const MoeGemmArgs& a, int bits);

namespace {

#ifndef WOL_GEMM_DTYPE
#define WOL_GEMM_DTYPE WOL_DTYPE_BF16
#endif

// Workgroup -> output tile.  Hardware deals consecutive workgroup ids to the
// 8 XCDs in turn; give XCD x the ids that form a compact block of tiles so
// that its L2 sees every A row block and B column block of that block once.
__device__ inline void tile_of_block(int id, int nbx, int nby, int* bx, int* by) {
  const int total = nbx * nby;
  constexpr int kXcd = 8;
  int t = id;
  if (total % kXcd == 0) {
    const int per = total / kXcd;
    t = (id % kXcd) * per + id / kXcd;
  }
  // walk the tiles in column-major panels of 8 row blocks so neighbours share B
  *by = t % nby;
  *bx = t / nby;
}

// The same with a two-dimensional split: the 8 XCDs form a grid of rg x 8/rg
// and each owns nby/rg row blocks x nbx/(8/rg) column blocks, the shape that
// makes the sum of the A rows and B columns an L2 has to fetch smallest
// (plan_xcd_rows on the host).  rg == 0: plain order.
__device__ inline void tile_of_block_2d(int id, int nbx, int nby, int rg, int* bx, int* by) {
  if (rg == 0) {
    *by = id % nby;
    *bx = id / nby;
    return;
  }
  constexpr int kXcd = 8;
  const int x = id % kXcd, i = id / kXcd;
  const int r = nby / rg, c = nbx / (kXcd / rg);
  *by = (x % rg) * r + i % r;
  *bx = (x / rg) * c + i / r;
}

template <int DT, int BITS, bool GROUPED, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ codes,
    const uint16_t* __restrict__ bias, const uint16_t* __restrict__ scale, void* __restrict__ out,
    int M, int K, int N, int gshift, int out_f32, int nbx, int nby, int act) {
  constexpr int NT = 64 * WM * WN;
  constexpr int BM = WM * TM * 16, BN = WN * TN * 16;
  constexpr int TK = BITS == 8 ? 64 : 128;     // k per 16-byte lane load
  constexpr int kDw = BITS == 8 ? 2 : 1;       // dwords per k step
  constexpr int kRow = TK + 8;                 // padded LDS row, in elements
  constexpr int kChunks = BM * (TK / 8) / NT;  // 16-byte pieces of the A tile per thread
  static_assert(BM * (TK / 8) % NT == 0, "A tile must split evenly over the threads");
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];  // 2 x BM x kRow

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int j = lane & 15, kb = lane >> 4;
  int bx, by;
  tile_of_block(blockIdx.x, nbx, nby, &bx, &by);
  const int m0 = by * BM;
  const int strip0 = bx * (BN / 16) + wn * TN;
  const int nstrips = N / kStripCols;

  // this thread's pieces of the A tile: row r, 8 elements at column 8*cc
  const uint16_t* aptr[kChunks];
  int aoff[kChunks];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int id = tid + c * NT, r = id / (TK / 8), cc = id % (TK / 8);
    int m = m0 + r;
    m = m < M ? m : M - 1;  // rows past M are computed on valid data and never stored
    aptr[c] = x + static_cast<int64_t>(m) * K + cc * 8;
    aoff[c] = r * kRow + cc * 8;
  }
  // this lane's 16 bytes of every strip of the wavefront
  const uint8_t* bptr[TN];
#pragma unroll
  for (int s = 0; s < TN; ++s) {
    const int st = strip0 + s < nstrips ? strip0 + s : nstrips - 1;  // past N: valid data, never stored
    bptr[s] = codes + static_cast<int64_t>(st) * strip_bytes(K, BITS) + lane * 16;
  }

  f32x4 tot[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) tot[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nfull = K / TK;
  const int niter = nfull + ((K % TK) ? 1 : 0);
  u32x4 areg[kChunks];
  u32x4 wcur[TN], wnext[TN];

  auto load_a = [&](int it) {
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      // the int4 half tile at the end of K has only TK/2 columns
      const bool ok = it < nfull || (aoff[c] % kRow) < TK / 2;
      areg[c] = ok ? *reinterpret_cast<const u32x4*>(aptr[c] + it * TK) : u32x4{0u, 0u, 0u, 0u};
    }
  };
  auto store_a = [&](int buf) {
#pragma unroll
    for (int c = 0; c < kChunks; ++c)
      *reinterpret_cast<u32x4*>(&lds[buf * BM * kRow + aoff[c]]) = areg[c];
  };
  auto load_b = [&](u32x4 (&w)[TN], int it) {
#pragma unroll
    for (int s = 0; s < TN; ++s) {
      if (it < nfull) {
        w[s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(bptr[s] + it * 1024));
      } else {  // 8 bytes per lane in the half tile
        const u32x2 q = *reinterpret_cast<const u32x2*>(bptr[s] - lane * 8 + nfull * 1024);
        w[s] = u32x4{q.x, q.y, 0u, 0u};
      }
    }
  };

  load_a(0);
  load_b(wcur, 0);
  store_a(0);
  __syncthreads();

  for (int it = 0; it < niter; ++it) {
    const bool more = it + 1 < niter;
    if (more) {
      load_a(it + 1);
      load_b(wnext, it + 1);
    }
    const uint16_t* As = lds + (it & 1) * BM * kRow;
    const int nsub = (it < nfull ? TK : TK / 2) / 64;
#pragma unroll
    for (int sb = 0; sb < TK / 64; ++sb) {
      if (sb >= nsub) break;
      f32x4 part[GROUPED ? TM : 1][GROUPED ? TN : 1];
      if (GROUPED) {
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
          for (int b = 0; b < TN; ++b) part[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const int step = sb * 2 + st;
        u32x4 bfrag[TN];
#pragma unroll
        for (int s = 0; s < TN; ++s) {
          const uint32_t w[4] = {wcur[s].x, wcur[s].y, wcur[s].z, wcur[s].w};
          bfrag[s] = std::conditional_t<GROUPED, DequantExact<DT, BITS>, DequantExactFma<DT, BITS>>::run(&w[step * kDw]);
        }
#pragma unroll
        for (int a = 0; a < TM; ++a) {
          const int row = (wm * TM + a) * 16 + j;
          const u32x4 af = *reinterpret_cast<const u32x4*>(&As[row * kRow + step * 32 + kb * 8]);
#pragma unroll
          for (int s = 0; s < TN; ++s) {
            if (GROUPED) part[a][s] = mfma16<DT>(af, bfrag[s], part[a][s]);
            else tot[a][s] = mfma16<DT>(af, bfrag[s], tot[a][s]);
          }
        }
      }
      if (GROUPED) {
        const int g = (it * TK + sb * 64) >> gshift;
#pragma unroll
        for (int s = 0; s < TN; ++s) {
          const int st = strip0 + s < nstrips ? strip0 + s : nstrips - 1;
          const float sc = to_f32<DT>(scale[static_cast<int64_t>(g) * N + st * 16 + j]);
#pragma unroll
          for (int a = 0; a < TM; ++a) tot[a][s] += part[a][s] * sc;
        }
      }
    }
    if (more) store_a((it + 1) & 1);
    __syncthreads();
    if (more) {
#pragma unroll
      for (int s = 0; s < TN; ++s) wcur[s] = wnext[s];
    }
  }

  // ---- epilogue: scale, bias, cast; 16-row slabs leave through LDS ----
  float sc[TN], bv[TN];
#pragma unroll
  for (int s = 0; s < TN; ++s) {
    const int st = strip0 + s < nstrips ? strip0 + s : nstrips - 1;
    const int n = st * 16 + j;
    sc[s] = GROUPED ? 1.0f : to_f32<DT>(scale[n]);
    bv[s] = bias != nullptr ? to_f32<DT>(bias[n]) : 0.0f;
  }
  if (out_f32) {
#pragma unroll
    for (int s = 0; s < TN; ++s) {
      if (strip0 + s >= nstrips) continue;
      const int n = (strip0 + s) * 16 + j;
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + (wm * TM + a) * 16 + kb * 4 + r;
          if (m < M) static_cast<float*>(out)[static_cast<int64_t>(m) * N + n] = act_apply(tot[a][s][r] * sc[s] + bv[s], act);
        }
    }
    return;
  }
  constexpr int kSlabRow = TN * 16 + 8;              // padded, in elements
  uint16_t* slab = lds + wave * 16 * kSlabRow;       // private to the wavefront (A buffers are free now)
  static_assert(WM * WN * 16 * kSlabRow <= 2 * BM * kRow, "slabs must fit in the A buffers");
  constexpr int kPieces = 16 * (TN * 16 / 8);        // 16-byte pieces of a slab
#pragma unroll
  for (int a = 0; a < TM; ++a) {
#pragma unroll
    for (int s = 0; s < TN; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        slab[(kb * 4 + r) * kSlabRow + s * 16 + j] = cast_out<DT>(act_apply(tot[a][s][r] * sc[s] + bv[s], act));
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int p = lane; p < kPieces; p += 64) {
      const int r = p / (TN * 2), c = p % (TN * 2);   // row of the slab, 8-column piece
      const int m = m0 + (wm * TM + a) * 16 + r;
      const int n = strip0 * 16 + c * 8;
      const u32x4 v = *reinterpret_cast<const u32x4*>(&slab[r * kSlabRow + c * 8]);
      if (m < M && n < N)
        *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(out) + static_cast<int64_t>(m) * N + n) = v;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// Fast path: K a multiple of the tile depth.
//
// The wavefront tile is built from 32 x 32 blocks of v_mfma_f32_32x32x16: TM x TN
// of them.  (wol_linear_wide.hip's 16x16x32 tiles with 64 rows, three stages deep,
// are level here: 64 rows, K = 8192, N = 28672, int4 g128 fp16 53.3 us against 53.4
// with K in two runs, 51.0 in four; 4096 x 11008 bf16 23.4 against 21.3.)  Both operands travel
// global -> LDS with direct-to-LDS loads (no registers, no LDS store
// instructions), two k tiles deep: while tile `it` is consumed the loads of
// tile it+1 are in flight.  A lands in LDS as unpadded rows whose 16-byte pieces are XOR-swizzled by row so a lane group's fragment reads
// fall into distinct banks.  The raw packed B tiles land exactly as they lie
// in memory (16-column strips in 16x16x32 order); a 32x32x16 B operand is
// assembled by letting lane l = 32*b + 16*sp + j read the 16 bytes that lane
// j + 16*(2h + b) of strip sp owns: MFMA (step, h) then contracts over
// k = 32*step + 16*h + 8*b + i, and the A fragment for it is simply piece
// 4*step + 2*h + b of the row.
//
// G = 0: per-channel scales, applied in the epilogue.  G = 64 or 128:
// group-wise scales; the MFMAs of a group accumulate into `part`, which is
// folded into the running sum with the group's scale (an fp32 FMA per
// accumulator element), so code * scale is never rounded to T.
//
// OFFS selects the offset dequantiser: a fraction of the VALU work, and the
// constant offset of every code is taken out again as -offset * (sum of the
// row's activations), which one more MFMA per A fragment and slice forms against
// a constant B operand (into `canc`, added when the scale is applied) -- the
// right trade when M is small: the matrix pipe idles, the VALU does not.
//
// With nsplit > 1 a workgroup covers only a run of k tiles and leaves its
// fp32 sums (scaled, without bias) in a partial buffer; reduce_partials_kernel
// adds the runs.  That is what fills the CUs when M is small.
//
// (A device function with the parameters by value: as the kernel's own body the
// same loops come out in another order.)
template <int DT, int BITS, int G, bool OFFS, int WM, int WN, int TM, int TN>
__device__ __forceinline__ void dma_tile(const DmaParams p) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stubs
  constexpr int NW = WM * WN;
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
  constexpr int TK = BITS == 8 ? 64 : 128;       // k per tile
  constexpr int kDw = BITS == 8 ? 2 : 1;         // dwords per 8 codes
  constexpr int C = TK / 8;                      // 16-byte pieces per A row
  constexpr int kABytes = BM * TK * 2;           // one A tile
  constexpr int kBBytes = (BN / 16) * 1024;      // one raw B tile (all strips of the workgroup)
  constexpr int kSBytes = G == 0 ? 0 : NW * 256;  // the tile's group scales: 128 values per wavefront
  constexpr int kScaleOff = kABytes + kBBytes;    // the scales' place in a stage
  constexpr int kStage = kScaleOff + kSBytes;
  constexpr int kStages = 2;                     // k tiles resident or in flight
  constexpr int kLds = kStages * kStage;
  constexpr int kALoads = kABytes / 1024 / NW;   // wave-level loads (1 KiB each) per wavefront
  constexpr int kBLoads = BN / 16 / NW;          // wave-level loads of a raw B tile per wavefront
  static_assert(kABytes / 1024 % NW == 0 && kALoads >= 1, "A tile must split evenly over the wavefronts");
  static_assert(BN / 16 % NW == 0 && kBLoads >= 1, "B tile must split evenly over the wavefronts");
  constexpr int Q = TK / 16;  // 16-k slices (one MFMA per 32x32 block each) per tile
  // group-wise scales: a fold every kFold slices, kGT folds (groups or halves of one) per tile
  constexpr int kFoldK = G == 0 ? TK : (G < TK ? G : TK);
  constexpr int kFold = kFoldK / 16;
  constexpr int kGT = TK / kFoldK;
  constexpr int kGShift = G == 128 ? 7 : 6;
  static_assert(kGT * BN <= NW * 128, "the tile's scales must fit the wavefronts' 4-byte loads");
  // direct-to-LDS loads every lane issues per stage.  They are the only vector
  // memory loads of the main loop, and loads complete in issue order, so
  // s_waitcnt vmcnt(n) can tell which stages have landed.
  constexpr int kPerStage = kALoads + kBLoads + (G == 0 ? 0 : 1);
  static_assert(Q >= 2 && (Q - 2) % kFold != 0 && (Q - 2) % kFold != kFold - 1,
                "the slice that holds the barrier neither starts nor ends a group");
  constexpr bool kFmaDequant = BITS == 4 && !OFFS;  // the shorter int4 dequantiser (see DequantExactFma)
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const uint16_t* __restrict__ x = p.x;
  const uint16_t* __restrict__ scale = p.scale;
  const uint16_t* __restrict__ bias = p.bias;
  const uint8_t* __restrict__ codes = p.codes;
  void* outp = p.out;
  int M = p.M;
  const int K = p.K, N = p.N;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int j = lane & 15, sp = (lane >> 4) & 1, b = lane >> 5, r32 = lane & 31;
  int bx, by, expert = -1, row0 = 0, rows = 0;
  const int ntiles = p.nbx * p.nby;
  const int split = blockIdx.x / ntiles;
  tile_of_block_2d(blockIdx.x - split * ntiles, p.nbx, p.nby, p.xcd_rows, &bx, &by);
  int m0 = by * BM;
  if (p.moe_table != nullptr) {
    const MoeTile t = reinterpret_cast<const MoeTile*>(p.moe_table)[by];
    if (t.expert < 0) return;
    expert = t.expert;
    row0 = t.row0;
    rows = t.rows;
  }
  if (expert >= 0) {
    // this tile belongs to one expert: shift every base to that expert and to
    // the tile's first row, and let M be the rows that exist
    x += static_cast<int64_t>(row0) * K;
    if (p.nsplit > 1) outp = static_cast<float*>(outp) + static_cast<int64_t>(row0) * N;  // partial sums
    else outp = static_cast<uint16_t*>(outp) + static_cast<int64_t>(row0) * N;
    codes += static_cast<int64_t>(expert) * p.moe_codes_stride;
    scale += static_cast<int64_t>(expert) * N;
    if (bias != nullptr) bias += static_cast<int64_t>(expert) * N;
    M = rows;
    m0 = 0;
  }
  const int strip_blk = p.strip_lo + bx * (BN / 16);
  const int nstrips = p.strip_hi;
  const int n_hi = p.strip_hi * kStripCols;
  // this workgroup's run of k tiles
  const int t0 = split * p.tiles_per_split;
  const int niter = (K / TK - t0) < p.tiles_per_split ? (K / TK - t0) : p.tiles_per_split;
  auto tile_index = [&](int it) {  // past the end of the run: the last tile again
    return it < niter ? it : niter - 1;
  };

  // global source of this lane for each of its A loads: LDS piece q holds row
  // q / C, piece (q % C) ^ swizzle(row) of the tile
  const uint16_t* asrc[kALoads];
#pragma unroll
  for (int c = 0; c < kALoads; ++c) {
    const int q = (c * NW + wave) * 64 + lane;
    const int row = q / C, slot = q % C;
    const int cc = slot ^ a_swizzle<C>(row);
    int m = m0 + row;
    m = m < M ? m : M - 1;  // rows past M are computed on valid data and never stored
    asrc[c] = x + static_cast<int64_t>(m) * K + static_cast<int64_t>(t0) * TK + cc * 8;
  }
  const uint8_t* bsrc[kBLoads];
#pragma unroll
  for (int c = 0; c < kBLoads; ++c) {
    int st = strip_blk + c * NW + wave;
    st = st < nstrips ? st : nstrips - 1;  // past the last column: valid data, never stored
    bsrc[c] = codes + static_cast<int64_t>(st) * strip_bytes(K, BITS) + static_cast<int64_t>(t0) * 1024 + lane * 16;
  }
  const int swz = a_swizzle<C>(lane & 15);  // fragment rows are 32*t + r32; the swizzle has period 16

  // Group scales travel with the tile: value v = 2 * (64 * wave + lane) of the
  // flattened [kGT][BN] block of the tile's scale rows, two values per lane.
  const int sval = 2 * (wave * 64 + lane) < kGT * BN ? 2 * (wave * 64 + lane) : 0;
  const int sfold = sval / BN;
  int scol = strip_blk * kStripCols + sval % BN;
  scol = scol < n_hi ? scol : n_hi - 2;  // past the last column: valid data, never used
  // The loads of tile `it` into its stage: [scales,] A loads, B loads.  They go out right behind the barrier that frees the
  // stage.
  auto issue = [&](int it) {
    const int t = tile_index(it);  // past the end: reload the last tile into a spare stage
    unsigned char* stage = smem + (it % kStages) * kStage;
    if (G != 0) {
      const int64_t row = (static_cast<int64_t>(t0 + t) * TK + sfold * kFoldK) >> kGShift;
      __builtin_amdgcn_global_load_lds(scale + row * N + scol,
                                       (lds_ptr_t)(stage + kScaleOff + wave * 256), 4, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < kALoads; ++c)
      __builtin_amdgcn_global_load_lds(asrc[c] + t * TK, (lds_ptr_t)(stage + (c * NW + wave) * 1024), 16, 0, 0);
#pragma unroll
    for (int c = 0; c < kBLoads; ++c)
      __builtin_amdgcn_global_load_lds(bsrc[c] + t * 1024,
                                       (lds_ptr_t)(stage + kABytes + (c * NW + wave) * 1024), 16, 0, 0);
  };

  // columns of this lane's accumulators: block c of the wavefront, column r32
  const int col0 = (strip_blk + wn * TN * 2) * 16;
  int ncol[TN];
#pragma unroll
  for (int c = 0; c < TN; ++c) {
    const int n = col0 + c * 32 + r32;
    ncol[c] = n < n_hi ? n : n_hi - 1;
  }
  // this lane's scales of the tile in `stage`, out of LDS
  auto read_scales = [&](const unsigned char* stage, uint16_t (&dst)[kGT > 0 ? kGT : 1][TN]) {
    if (G != 0) {
#pragma unroll
      for (int f = 0; f < kGT; ++f)
#pragma unroll
        for (int c = 0; c < TN; ++c)
          dst[f][c] = *reinterpret_cast<const uint16_t*>(
              stage + kScaleOff + (f * BN + (wn * TN + c) * 32 + r32) * 2);
    }
  };

  f32x16 tot[TM][TN];
  f32x16 part[G != 0 ? TM : 1][G != 0 ? TN : 1];
  f32x16 canc[OFFS ? TM : 1];
#pragma unroll
  for (int a = 0; a < TM; ++a) {
#pragma unroll
    for (int c = 0; c < TN; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) tot[a][c][r] = 0.0f;
    if (OFFS) {
#pragma unroll
      for (int r = 0; r < 16; ++r) canc[a][r] = 0.0f;
    }
  }
  uint32_t magic = Dequant<DT, BITS>::kMagic;
  asm volatile("" : "+v"(magic));  // keep the constant in a VGPR

  // byte offsets inside a stage that do not change from tile to tile
  const int a_row_off = (wm * TM * 32 + r32) * (TK * 2);
  const int b_off = kABytes + (wn * TN * 2 + sp) * 1024 + (j + 16 * b) * 16;
  constexpr int kValuPerMfma = ((BITS == 8 ? 16 : kFmaDequant && DT == WOL_DTYPE_BF16 ? 18 : 12) * TN + TM * TN - 1) / (TM * TN) + 2;
  constexpr int kHalf = (TM * TN + 1) / 2;  // MFMAs of a slice issued before the barrier

  // The wavefront's pipeline registers: raw codes of the current and the next
  // tile, and two sets of operands -- the one the MFMAs of slice q use and the
  // one being prepared for slice q+1 (A fragments read from LDS, B fragments
  // dequantised).
  u32x4 braw[2][TN][2];
  uint16_t sraw[kGT > 0 ? kGT : 1][TN];
  u32x4 af[2][TM];
  u32x4 bf[2][TN];
  auto read_b = [&](const unsigned char* stage, u32x4 (&dst)[TN][2]) {
#pragma unroll
    for (int c = 0; c < TN; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        dst[c][h] = *reinterpret_cast<const u32x4*>(stage + b_off + c * 2048 + h * 512);
  };
  auto read_a = [&](const unsigned char* stage, u32x4 (&dst)[TM], int q) {
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      const int slot = (2 * q + b) ^ swz;
      dst[a] = *reinterpret_cast<const u32x4*>(stage + a_row_off + a * 32 * (TK * 2) + slot * 16);
    }
  };
  auto dequant = [&](u32x4 (&dst)[TN], const u32x4 (&raw)[TN][2], int q) {
    const int step = q / 2, h = q % 2;
#pragma unroll
    for (int c = 0; c < TN; ++c) {
      const uint32_t w4[4] = {raw[c][h].x, raw[c][h].y, raw[c][h].z, raw[c][h].w};
      if (OFFS) dst[c] = Dequant<DT, BITS>::run(&w4[step * kDw], magic);
      else if constexpr (kFmaDequant) dst[c] = DequantExactFma<DT, BITS>::run(&w4[step * kDw]);
      else dst[c] = DequantExact<DT, BITS>::run(&w4[step * kDw]);
    }
  };
  // MFMAs lo .. hi-1 (numbered a * TN + c) of slice q
  auto mfmas = [&](const u32x4 (&a4)[TM], const u32x4 (&b4)[TN], int q, int lo, int hi) {
    const bool first = q % kFold == 0;
    f32x16 zero;
#pragma unroll
    for (int r = 0; r < 16; ++r) zero[r] = 0.0f;
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int c = 0; c < TN; ++c)
        if (a * TN + c >= lo && a * TN + c < hi) {
          if (OFFS && c == 0) {
            const u32x4 cb = {Dequant<DT, BITS>::kCancel, Dequant<DT, BITS>::kCancel,
                              Dequant<DT, BITS>::kCancel, Dequant<DT, BITS>::kCancel};
            canc[a] = mfma32<DT>(a4[a], cb, (G != 0 && first) ? zero : canc[a]);
          }
          if (G == 0) {
            tot[a][c] = mfma32<DT>(a4[a], b4[c], tot[a][c]);
          } else if (first) {
            part[a][c] = mfma32<DT>(a4[a], b4[c], zero);
          } else {
            part[a][c] = mfma32<DT>(a4[a], b4[c], part[a][c]);
          }
        }
  };
  // after the last slice of a group: tot += part * scale
  auto fold = [&](const uint16_t (&sr)[kGT > 0 ? kGT : 1][TN], int q) {
    if (G != 0 && q % kFold == kFold - 1) {
#pragma unroll
      for (int c = 0; c < TN; ++c) {
        const float sc = to_f32<DT>(sr[q / kFold][c]);
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            tot[a][c][r] = fmaf(OFFS ? part[a][c][r] + canc[a][r] : part[a][c][r], sc, tot[a][c][r]);
      }
    }
  };

  issue(0);
  issue(1);
  wait_vmcnt<kPerStage>();  // tile 0 has landed
  __builtin_amdgcn_s_barrier();
  read_b(smem, braw[0]);
  read_a(smem, af[0], 0);
  dequant(bf[0], braw[0], 0);
  // Every slice runs its MFMAs with the preparation of the next slice's
  // operands (A fragments read from LDS, B fragments dequantised) spread
  // between them, so that the VALU work executes in the shadow of the matrix
  // pipe.  The workgroup barrier that hands the stage of tile `it` over to
  // tile it+2 sits in the middle of the last but one slice, once the
  // wavefront has fetched its last operands of the tile; the raw codes of tile
  // it+1 are read right behind it and have a whole slice to arrive.
  auto tile = [&](int it, u32x4 (&raw)[TN][2], u32x4 (&raw_next)[TN][2]) {
    const unsigned char* stage = smem + (it % kStages) * kStage;
    const unsigned char* next = smem + ((it + 1) % kStages) * kStage;
    read_scales(stage, sraw);  // before the stage is handed over
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (q != Q - 2) {
        const bool last = q == Q - 1;
        read_a(last ? next : stage, af[(q + 1) & 1], last ? 0 : q + 1);
        dequant(bf[(q + 1) & 1], last ? raw_next : raw, last ? 0 : q + 1);
        mfmas(af[q & 1], bf[q & 1], q, 0, TM * TN);
#pragma unroll
        for (int i = 0; i < TM * TN; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                   // one MFMA
          if (i < TM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // one LDS read
          __builtin_amdgcn_sched_group_barrier(0x002, kValuPerMfma, 0);        // VALU
        }
        __builtin_amdgcn_sched_barrier(0);
        fold(sraw, q);
      } else {
        read_a(stage, af[(q + 1) & 1], q + 1);
        mfmas(af[q & 1], bf[q & 1], q, 0, kHalf);
#pragma unroll
        for (int i = 0; i < kHalf; ++i) {
          if (2 * i < TM) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // this wavefront needs nothing more from the tile's stage; once every
        // wavefront is there, tile it+1 (landed by now) may be read and the
        // stage refilled with tile it+2
        __builtin_amdgcn_s_waitcnt(0x0070 | (0xF << 0) | (3 << 14));  // lgkmcnt(0)
        wait_vmcnt<0>();
        __builtin_amdgcn_s_barrier();
        issue(it + kStages);
        read_b(next, raw_next);
        dequant(bf[(q + 1) & 1], raw, q + 1);
        mfmas(af[q & 1], bf[q & 1], q, kHalf, TM * TN);
#pragma unroll
        for (int i = 0; i < TM * TN - kHalf + 1; ++i) {
          if (i < TM * TN - kHalf) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (i < 2 * TN) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 2 * kValuPerMfma, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  for (int it = 0; it < niter; it += 2) {
    tile(it, braw[0], braw[1]);
    if (it + 1 < niter) tile(it + 1, braw[1], braw[0]);
  }
  wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();  // the spare loads are done and every wavefront has stopped reading

  // ---- epilogue: scale, bias, cast; 32-row slabs leave through LDS as 16-byte stores ----
  // accumulator element r of lane l is row 8*(r/4) + 4*(l/32) + r%4, column l%32 of its block
  float sc[TN], bv[TN];
#pragma unroll
  for (int c = 0; c < TN; ++c) {
    sc[c] = G == 0 ? to_f32<DT>(scale[ncol[c]]) : 1.0f;
    bv[c] = (bias != nullptr && p.nsplit == 1) ? to_f32<DT>(bias[ncol[c]]) : 0.0f;
  }
  if (OFFS && G == 0) {
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int c = 0; c < TN; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[a][c][r] += canc[a][r];
  }
  if (p.out_f32 || p.nsplit > 1) {
    // fp32 results (verification mode) or partial sums of this run of k tiles: plain stores
    // partial sums are kept compact: row length = the columns of this launch
    const int64_t ld = p.nsplit > 1 ? static_cast<int64_t>(p.strip_hi - p.strip_lo) * kStripCols : N;
    const int ncol0 = p.nsplit > 1 ? p.strip_lo * kStripCols : 0;
    const int64_t run_rows = expert >= 0 ? p.moe_rows : M;  // rows of one run's partial sums
    float* outf = static_cast<float*>(outp) + (p.nsplit > 1 ? static_cast<int64_t>(split) * run_rows * ld : 0);
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int c = 0; c < TN; ++c) {
        const int n = col0 + c * 32 + r32;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + (wm * TM + a) * 32 + 8 * (r / 4) + 4 * b + r % 4;
          if (m < M && n < n_hi) {
            const float v = tot[a][c][r] * sc[c] + bv[c];  // a partial sum when K is cut into runs
            outf[static_cast<int64_t>(m) * ld + (n - ncol0)] = p.nsplit > 1 ? v : act_apply(v, p.act);
          }
        }
      }
    return;
  }
  uint16_t* out = static_cast<uint16_t*>(outp);
  constexpr int kSlabRow = TN * 32 + 8;   // padded, in elements
  static_assert(NW * 32 * kSlabRow * 2 <= kLds, "slabs must fit in the stage buffers");
  uint16_t* slab = reinterpret_cast<uint16_t*>(smem) + wave * 32 * kSlabRow;
  constexpr int kPieces = 32 * (TN * 32 / 8);
#pragma unroll
  for (int a = 0; a < TM; ++a) {
#pragma unroll
    for (int c = 0; c < TN; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        slab[(8 * (r / 4) + 4 * b + r % 4) * kSlabRow + c * 32 + r32] =
            cast_out<DT>(act_apply(tot[a][c][r] * sc[c] + bv[c], p.act));
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = lane; q < kPieces; q += 64) {
      const int r = q / (TN * 4), cc = q % (TN * 4);
      const int m = m0 + (wm * TM + a) * 32 + r;
      const int n = col0 + cc * 8;
      const u32x4 v = *reinterpret_cast<const u32x4*>(&slab[r * kSlabRow + cc * 8]);
      if (m < M && n < n_hi) *reinterpret_cast<u32x4*>(out + static_cast<int64_t>(m) * N + n) = v;
    }
    __builtin_amdgcn_wave_barrier();
  }
#endif
}

template <int DT, int BITS, int G, bool OFFS, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_dma_kernel(const DmaParams p) {
  dma_tile<DT, BITS, G, OFFS, WM, WN, TM, TN>(p);
}

// out[m, col0 + c] = T( sum over the runs of part[run][m][c] + bias[col0 + c] ) for the ncols
// columns from col0 on; four columns per thread; total = M * ncols.  valid_rows (may be null):
// rows from *valid_rows on were never computed and are left alone.
template <int DT>
__global__ __launch_bounds__(256) void reduce_partials_kernel(
    const float* __restrict__ part, int nsplit, const uint16_t* __restrict__ bias,
    void* __restrict__ out, int out_f32, int64_t total, int N, int col0, int ncols, int act,
    const int64_t* __restrict__ valid_rows = nullptr) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  if (valid_rows != nullptr && i / ncols >= *valid_rows) return;
  const int64_t o = i / ncols * N + col0 + i % ncols;  // position in out
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  // W loads in flight at a time (past the last run: the last run again, not
  // added), added in run order: one trip to memory for up to W runs
  auto add_runs = [&](auto width) {
    constexpr int W = decltype(width)::value;
    for (int r0 = 0; r0 < nsplit; r0 += W) {
      f32x4 v[W];
#pragma unroll
      for (int u = 0; u < W; ++u) {
        const int r = r0 + u < nsplit ? r0 + u : nsplit - 1;
        v[u] = *reinterpret_cast<const f32x4*>(part + r * total + i);
      }
#pragma unroll
      for (int u = 0; u < W; ++u)
        if (r0 + u < nsplit) {
#pragma unroll
          for (int e = 0; e < 4; ++e) s[e] += v[u][e];
        }
    }
  };
  if (nsplit <= 4) add_runs(std::integral_constant<int, 4>());
  else add_runs(std::integral_constant<int, 8>());
  if (bias != nullptr) {
    const int n = col0 + static_cast<int>(i % ncols);
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += to_f32<DT>(bias[n + e]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] = act_apply(s[e], act);
  if (out_f32) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(out) + o) = s;
  } else {
    u32x2 v;
    v.x = cast_out<DT>(s[0]) | (static_cast<uint32_t>(cast_out<DT>(s[1])) << 16);
    v.y = cast_out<DT>(s[2]) | (static_cast<uint32_t>(cast_out<DT>(s[3])) << 16);
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(out) + o) = v;
  }
}

// The same for a gate|up projection: out[m, c] = T(silu(g) * u) with g and u the sums (plus bias)
// of columns c and N/2 + c; out is [M, N/2], four columns per thread, total = M * N / 2,
// N % 8 == 0.  The runs are [run][M][N].
template <int DT>
__global__ __launch_bounds__(256) void reduce_partials_swiglu_kernel(
    const float* __restrict__ part, int nsplit, const uint16_t* __restrict__ bias,
    void* __restrict__ out, int out_f32, int64_t total, int N) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  const int half = N / 2;
  const int64_t m = i / half;
  const int c = static_cast<int>(i % half);
  const int64_t run = total * 2;
  f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  for (int r0 = 0; r0 < nsplit; r0 += 4) {
    f32x4 v[4][2];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = r0 + u < nsplit ? r0 + u : nsplit - 1;
#pragma unroll
      for (int h = 0; h < 2; ++h) v[u][h] = *reinterpret_cast<const f32x4*>(part + r * run + m * N + h * half + c);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (r0 + u < nsplit) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) s[h][e] += v[u][h][e];
      }
  }
  if (bias != nullptr) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[h][e] += to_f32<DT>(bias[h * half + c + e]);
  }
  f32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = act_swiglu(s[0][e], s[1][e]);
  if (out_f32) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(out) + i) = o;
  } else {
    u32x2 v;
    v.x = cast_out<DT>(o[0]) | (static_cast<uint32_t>(cast_out<DT>(o[1])) << 16);
    v.y = cast_out<DT>(o[2]) | (static_cast<uint32_t>(cast_out<DT>(o[3])) << 16);
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(out) + i) = v;
  }
}

typedef GemmArgs Args;

template <int DT, int BITS, bool GROUPED, int WM, int WN, int TM, int TN>
void launch_one(const Args& a) {
  constexpr int BM = WM * TM * 16, BN = WN * TN * 16, TK = BITS == 8 ? 64 : 128;
  const int nbx = (a.N + BN - 1) / BN, nby = (a.M + BM - 1) / BM;
  const size_t lds = 2 * static_cast<size_t>(BM) * (TK + 8) * sizeof(uint16_t);
  auto kern = gemm_kernel<DT, BITS, GROUPED, WM, WN, TM, TN>;
  static std::atomic<uint32_t> configured{0};  // per instantiation
  allow_lds(reinterpret_cast<const void*>(kern), lds, configured);
  kern<<<dim3(static_cast<unsigned>(nbx * nby)), dim3(64 * WM * WN), lds, a.stream>>>(
      static_cast<const uint16_t*>(a.x), static_cast<const uint8_t*>(a.codes),
      static_cast<const uint16_t*>(a.bias), static_cast<const uint16_t*>(a.scale), a.out, a.M, a.K,
      a.N, a.gshift, a.out_f32, nbx, nby, a.act);
}

// Row groups rg of the XCD grid for tile_of_block_2d: among the divisors of 8
// that split both tile counts evenly, the one with the least bytes per XCD and
// k step, rows * a_bytes + columns * b_bytes (bytes of one row block / column
// block per k).  0 when the tiles do not divide over the XCDs.
inline int plan_xcd_rows(int nbx, int nby, int a_bytes, int b_bytes) {
  int best = 0;
  int64_t best_cost = INT64_MAX;
  for (int rg = 1; rg <= 8; rg *= 2) {
    const int cg = 8 / rg;
    if (nby % rg != 0 || nbx % cg != 0) continue;
    const int64_t cost = static_cast<int64_t>(nby / rg) * a_bytes + static_cast<int64_t>(nbx / cg) * b_bytes;
    if (cost < best_cost) { best_cost = cost; best = rg; }
  }
  return best;
}

template <int BITS, int G, int WM, int WN, int TM, int TN>
constexpr size_t dma_lds_bytes() {
  return 2 * (static_cast<size_t>(WM * TM * 32) * (BITS == 8 ? 64 : 128) * 2 +
              (WN * TN * 32 / 16) * 1024 + (G == 0 ? 0 : WM * WN * 256));
}

// Launches the fast kernel on the columns of strips [strip_lo, strip_hi), K
// cut into nsplit runs (nsplit > 1 needs a.ws: nsplit x M x columns floats).
template <int DT, int BITS, int G, bool OFFS, int WM, int WN, int TM, int TN>
void launch_dma(const Args& a, int strip_lo, int strip_hi, int nsplit) {
  constexpr int BM = WM * TM * 32, BN = TN * WN * 32;
  constexpr int TK = BITS == 8 ? 64 : 128;
  if (strip_hi <= strip_lo) return;
  constexpr size_t lds = dma_lds_bytes<BITS, G, WM, WN, TM, TN>();
  auto kern = gemm_dma_kernel<DT, BITS, G, OFFS, WM, WN, TM, TN>;
  static std::atomic<uint32_t> configured{0};  // per instantiation
  allow_lds(reinterpret_cast<const void*>(kern), lds, configured);
  const int ncols = (strip_hi - strip_lo) * kStripCols;
  if (nsplit > 1 && (a.ws == nullptr ||
                     a.ws_bytes < static_cast<size_t>(nsplit) * a.M * ncols * sizeof(float)))
    nsplit = 1;  // never write past the scratch buffer
  DmaParams p;
  p.x = static_cast<const uint16_t*>(a.x);
  p.codes = static_cast<const uint8_t*>(a.codes);
  p.bias = static_cast<const uint16_t*>(a.bias);
  p.scale = static_cast<const uint16_t*>(a.scale);
  p.out = nsplit > 1 ? a.ws : a.out;
  p.M = a.M; p.K = a.K; p.N = a.N;
  p.out_f32 = a.out_f32;
  p.strip_lo = strip_lo; p.strip_hi = strip_hi;
  p.nbx = ((strip_hi - strip_lo) * kStripCols + BN - 1) / BN;
  p.nby = (a.M + BM - 1) / BM;
  const int tiles = a.K / TK;
  p.tiles_per_split = (tiles + nsplit - 1) / nsplit;
  p.nsplit = (tiles + p.tiles_per_split - 1) / p.tiles_per_split;
  p.xcd_rows = plan_xcd_rows(p.nbx, p.nby, BM * 2, WN * TN * 32 * BITS / 8);
  p.act = a.act;
  p.moe_table = nullptr;
  p.moe_codes_stride = 0;
  p.moe_rows = 0;
  p.stamps = nullptr;
  kern<<<dim3(static_cast<unsigned>(p.nbx * p.nby * p.nsplit)), dim3(64 * WM * WN), lds, a.stream>>>(p);
  if (nsplit > 1) {
    const int64_t total = static_cast<int64_t>(a.M) * ncols;
    if (a.act == WOL_ACT_SWIGLU) {
      // a gate|up projection whose runs cover all of N (the small-M configurations): the kernel
      // that adds the runs forms silu(gate) * up, out is [M, N / 2]
      reduce_partials_swiglu_kernel<DT><<<dim3(static_cast<unsigned>((total / 8 + 255) / 256)), dim3(256), 0, a.stream>>>(
          static_cast<const float*>(a.ws), p.nsplit, p.bias, a.out, a.out_f32, total / 2, a.N);
      return;
    }
    reduce_partials_kernel<DT><<<dim3(static_cast<unsigned>((total / 4 + 255) / 256)), dim3(256), 0, a.stream>>>(
        static_cast<const float*>(a.ws), p.nsplit, p.bias, a.out, a.out_f32, total, a.N,
        strip_lo * kStripCols, ncols, a.act);
  }
}

// Launches a tile of wol_linear_wide.hip on the columns of strips [strip_lo,
// strip_hi); the rest as launch_dma.
template <int DT>
void launch_wide(const Args& a, int bits, int group, WideTile tile, int swi, int strip_lo, int strip_hi, int nsplit) {
  const int bm = tile == WideTile::kHalf ? 128 : 256, bn = swi ? 128 : 256;
  if (strip_hi <= strip_lo) return;
  if (swi) nsplit = 1;
  const int ncols = (strip_hi - strip_lo) * kStripCols;
  if (nsplit > 1 && (a.ws == nullptr || a.ws_bytes < static_cast<size_t>(nsplit) * a.M * ncols * sizeof(float)))
    nsplit = 1;  // never write past the scratch buffer
  DmaParams p{};
  p.x = static_cast<const uint16_t*>(a.x);
  p.codes = static_cast<const uint8_t*>(a.codes);
  p.bias = static_cast<const uint16_t*>(a.bias);
  p.scale = static_cast<const uint16_t*>(a.scale);
  p.out = nsplit > 1 ? a.ws : a.out;
  p.M = a.M; p.K = a.K; p.N = a.N;
  p.out_f32 = a.out_f32;
  p.strip_lo = strip_lo; p.strip_hi = strip_hi;
  p.nbx = (ncols + bn - 1) / bn;
  p.nby = (a.M + bm - 1) / bm;
  const int tiles = a.K / 64;
  p.tiles_per_split = (tiles + nsplit - 1) / nsplit;
  if (group == 128 || bits == 4) p.tiles_per_split = (p.tiles_per_split + 1) & ~1;  // every run starts on a group (a raw tile) of two tiles
  p.nsplit = (tiles + p.tiles_per_split - 1) / p.tiles_per_split;
  p.act = a.act;
  if (DT == WOL_DTYPE_BF16) launch_wide_bf16(p, bits, group, tile, swi, a.stream);
  else launch_wide_f16(p, bits, group, tile, swi, a.stream);
  if (nsplit > 1) {
    const int64_t total = static_cast<int64_t>(a.M) * ncols;
    reduce_partials_kernel<DT><<<dim3(static_cast<unsigned>((total / 4 + 255) / 256)), dim3(256), 0, a.stream>>>(
        static_cast<const float*>(a.ws), p.nsplit, p.bias, a.out, a.out_f32, total, a.N,
        strip_lo * kStripCols, ncols, a.act);
  }
}

// Number of 256-column tiles given to the 256-row kernel; the remaining
// columns run with half-size tiles.  Cost model: a workgroup owns its CU, so a
// launch takes ceil(tiles / CUs) tile times; a half-size tile costs kSmall of a
// full one (a little more than half; 0.58 for int4 with group-wise scales, where
// full tiles run on gemm_dma_kernel_tall).  int4 with group-wise scales also counts
// a last partial round that plan_tail cuts into K runs as the share of a round that
// a run is plus the partial sums' way through memory (kRuns).  480 problems (65 to
// 8192 rows, K 1024 to 14336, N 1024 to 28672), timed with every number of
// 256-column tiles that fills whole rounds: the choice is slower than the best of
// them by 0.3 % (int4 with groups), 0.2 % (int8 with groups) and 0.3 % (per channel)
// on average; at worst 11 % (1218 x 5120 -> 7104 int4 g64: half-size tiles with K
// runs 128 us, whole ones 115), 17 % (3642 x 2432 -> 17824 int8 g64 374 against 320:
// half-size tiles throughout, 68 of the 70 column tiles whole) and 15 % (3499 x 6528 -> 2592
// int8 137 against 120: half-size tiles with K runs, which only int4 with groups
// counts).  No other pair of constants was better everywhere: 0.62 with groups gains
// 5 to 12 % on seven of the eleven problems it decides otherwise and loses 7 and 2 %
// on two (360 x 13696 -> 25248 int4 g128 276 -> 296).
inline int plan_big_columns(int M, int K, int N, int bits, int group) {
  const int cus = num_cus();
  const bool g4 = bits == 4 && group != 0;
  const double kSmall = g4 ? 0.58 : 0.55;
  constexpr double kRuns = 0.25;
  const int nbx = (N + 255) / 256, nby_big = (M + 255) / 256, nby_small = (M + 127) / 128;
  int best = nbx;
  double best_t = 1e30;
  // the estimate grows with the number of half-size tiles, so for every number of whole rounds only the most
  // columns that fit them matter (walking all columns took 1 to 2 us of a call on a wide weight)
  for (int c = nbx; c >= 0;) {
    const int small = (nbx - c) * nby_small;
    const int rounds = (c * nby_big + cus - 1) / cus;
    double t = static_cast<double>(rounds);
    const int rest = small % cus;
    int runs = g4 && rest > 0 ? cus / rest : 1;
    runs = runs > 4 ? 4 : runs;
    while (runs > 1 && K / 128 / runs < 8) --runs;
    if (runs > 1) t += kSmall * (small / cus) + kSmall / runs + kRuns;
    else t += kSmall * static_cast<double>((small + cus - 1) / cus);
    if (t < best_t - 1e-9) { best_t = t; best = c; }
    const int fewer = rounds > 0 ? static_cast<int>(static_cast<int64_t>(rounds - 1) * cus / nby_big) : -1;
    c = fewer < c ? fewer : c - 1;
  }
  return best;
}

// Rows up to which the small-M configurations (one row block of 32 or 64
// rows, K split across workgroups) are used.  They run two stages deep
// instead of three: the smaller LDS footprint lets a third (32 rows, and
// int8) or second (64 rows, int4) workgroup share the CU, which hides more
// latency than the third stage did.
constexpr int kSkinnyMaxM = 64;

// How a small-M problem is cut up.  A workgroup takes 256 columns, or 512
// (two 32-column blocks per wavefront: half the activation bytes out of L2
// and half the A-fragment reads out of LDS per MFMA, for twice the weight
// bytes per k tile), and K is split into runs: at most 16, of at least 4 k
// tiles, and no more than the scratch buffer holds.  Of all such pairs the one
// with the lowest estimated time is taken.  The estimate, in k-tile times of a
// 256-column workgroup:
//   ceil(workgroups / CUs) x (tiles per run + 8) x (1.3 if 512 columns)
//     + runs x M x N / 300000
// The workgroups of a CU share its load path, so what counts is how many
// the fullest CU gets, not how many are resident; the 8 is a workgroup's
// start (the first tile's latency) and end (writing the partial sums); the
// last term is the traffic of the partial sums, which every run writes and
// the reduction reads.  The three constants are fitted to three sweeps, on
// three machines, over every admissible pair on 160 problems (4096 <= K, N <=
// 28672; 17, 32, 48, 64 rows; int4 and int8, with and without groups),
// scoring a pair by the slowest of its three times: launches with more
// workgroups than CUs but fewer than resident slots vary by up to 30 %
// between machines, launches of at most one workgroup per CU by 3 %.  The
// choice is 1.8 % slower than the best pair on average and 14 % at worst; the
// rule it replaces (width by N and K alone, rounds by resident slots, no
// traffic term) was 9.6 % and 29 % off.  int4 with group size 64 and 64-row
// tiles does not fit the registers at 512 columns.
struct SkinnyPlan {
  bool wide;  // 512 columns per workgroup instead of 256
  int ns;     // K runs
};
inline SkinnyPlan plan_skinny(int M, int K, int N, int bits, int group, size_t ws_bytes) {
  const int tk = bits == 8 ? 64 : 128, tiles = K / tk;
  const int cus = num_cus();
  const size_t per_run = static_cast<size_t>(M) * N * sizeof(float);
  const double traffic = static_cast<double>(M) * N / 300000.0;
  SkinnyPlan best{false, 1};
  double best_cost = 1e300;
  for (int wide = 0; wide < 2; ++wide) {
    if (wide && bits == 4 && group == 64 && M > 32) continue;
    const int cols = wide ? 512 : 256;
    const int64_t nbx = (N + cols - 1) / cols;
    for (int ns = 1; ns <= 16; ++ns) {
      const int tps = (tiles + ns - 1) / ns;
      const int eff = (tiles + tps - 1) / tps;
      if (eff != ns || (ns > 1 && tps < 4)) continue;
      if (ns > 1 && per_run * ns > ws_bytes) continue;
      const int64_t rounds = (nbx * ns + cus - 1) / cus;
      const double cost = static_cast<double>(rounds) * (tps + 8) * (wide ? 1.3 : 1.0) +
                          (ns > 1 ? ns * traffic : 0.0) + 1e-6 * ns;  // the last term prefers fewer runs on ties
      if (cost < best_cost) { best_cost = cost; best = SkinnyPlan{wide != 0, ns}; }
    }
  }
  return best;
}

// First strip of the columns that get 128 x 256 tiles (above 64 rows); those in
// front of it get 256 x 256 tiles.
constexpr int kHalfRows = 128, kHalfCols = 256;
inline int half_tile_strip(int M, int K, int N, int bits, int group) {
  const int c = plan_big_columns(M, K, N, bits, group) * 16, nstrips = N / kStripCols;
  return c < nstrips ? c : nstrips;
}

// How a half-size configuration (one workgroup per CU) covers ncols columns:
// the column tiles of whole rounds of the CUs run as they are; the tiles of
// the last, partial round leave CUs idle for a whole tile time, so K is cut
// into as many runs as fit the idle CUs (2..4, each at least 8 k tiles long,
// and only if the scratch buffer holds ns x M x columns floats).  The extra
// traffic is worth it below half occupancy.  full_tiles = 0 with ns = 1 means
// one plain launch over everything.
struct TailPlan {
  int full_tiles;  // column tiles launched without a K split
  int ns;          // K runs of the remaining column tiles
};
inline TailPlan plan_tail(int M, int K, int ncols, int bm, int bn, int tk, size_t ws_bytes) {
  const int cus = num_cus(), tiles = K / tk;
  const int nbx = (ncols + bn - 1) / bn, nby = (M + bm - 1) / bm;
  const int blocks = nbx * nby;
  if (blocks == 0) return {0, 1};
  const int full = blocks > cus ? (blocks / cus) * cus / nby : 0;
  const int rest = (nbx - full) * nby;
  if (rest == 0) return {0, 1};
  const size_t rest_cols = static_cast<size_t>(ncols) - static_cast<size_t>(full) * bn;
  int ns = cus / rest;
  ns = ns > 4 ? 4 : ns;
  while (ns > 1 && (tiles / ns < 8 || static_cast<size_t>(ns) * M * rest_cols * sizeof(float) > ws_bytes)) --ns;
  if (ns <= 1) return {0, 1};
  return {full, ns};
}

template <int DT, int BITS, int G>
void launch_fast(const Args& a) {
  const int nstrips = a.N / kStripCols;
  if (a.M <= kSkinnyMaxM) {
    const SkinnyPlan sp = plan_skinny(a.M, a.K, a.N, BITS, G, a.ws != nullptr ? a.ws_bytes : 0);
    const bool wide = sp.wide;
    const int ns = sp.ns;
    if constexpr (BITS == 4) {
      if (a.M <= 32) {
        if (wide) launch_dma<DT, BITS, G, true, 1, 8, 1, 2>(a, 0, nstrips, ns);
        else launch_dma<DT, BITS, G, true, 1, 8, 1, 1>(a, 0, nstrips, ns);
        return;
      }
    }
    if constexpr (!(BITS == 4 && G == 64)) {
      if (wide) { launch_dma<DT, BITS, G, false, 1, 8, 2, 2>(a, 0, nstrips, ns); return; }
    }
    launch_dma<DT, BITS, G, false, 1, 8, 2, 1>(a, 0, nstrips, ns);
    return;
  }
  // 256 x 256 tiles for as many column tiles as fill whole rounds of the CUs; the
  // rest, which would leave CUs idle for a whole tile time, goes to 128 x 256
  // tiles.  (256 x 128 ones, four A blocks per dequantised B block in the former
  // kernel, are nowhere faster any more: int8, 512 rows, K = 4096, N = 12288 52.6
  // against 50.6 us; 1237 rows, K = 11008, N = 4096 116 against 112.)
  const int lo = half_tile_strip(a.M, a.K, a.N, BITS, G);
  const TailPlan t = plan_tail(a.M, a.K, (nstrips - lo) * kStripCols, kHalfRows, kHalfCols, BITS == 8 ? 64 : 128,
                               a.ws != nullptr ? a.ws_bytes : 0);
  const int mid = lo + t.full_tiles * (kHalfCols / kStripCols);  // strips [lo, mid) unsplit, [mid, nstrips) in t.ns runs
  launch_wide<DT>(a, BITS, G, WideTile::kWhole, 0, 0, lo, 1);
  launch_wide<DT>(a, BITS, G, WideTile::kHalf, 0, lo, mid, 1);
  launch_wide<DT>(a, BITS, G, WideTile::kHalf, 0, mid, nstrips, t.ns);
}

// How high the row tiles of gemm_experts_kernel may be.  A round of workgroups
// takes the time of its highest tile, and a high tile costs less than its share
// (part of a tile's time is the same for any height), so one limit of 256 rows
// is right where tiles fill many rounds and leaves CUs idle where few tiles
// exist or a last round is nearly empty.  Each product, with column tiles of its
// own number, takes the limit with the shortest estimate:
//   time of such a tile x rounds,
// a round being what the CUs of an XCD take of its share of the tiles.  The
// times of 64-, 128- and 192-row tiles against 256-row ones (0.54, 0.66, 0.84) and
// of a 128-column tile against a 256-column one (0.7) are fitted to 200 problems
// timed under every limit and tile width of either product (4 to 16 experts of 65
// rows each up to 8192 in all, evenly and unequally loaded, hidden 1024 to 4096,
// fc1 width 2816 to 28672, int4 and int8).  The choice is 0.5 % slower than the
// best one on average (int4 0.3, int8 0.7) and 6 % at worst, on these and on 200
// other problems alike; 256-row tiles always 24 %; 0.46, 0.66, 0.85, which came from
// 11 problems, 0.9 and 10 %.  A limit of each product's own against one limit for
// both: 4 experts, hidden 4096, width 11008, 900 rows, int4 173 -> 138 us; 8 experts,
// 2048, 16384, 1500 rows, int4 228 -> 191.
struct MoeHeights {
  int xcd_cus;      // CUs of an XCD
  int min_units;    // lowest limit the launch grid has room for; 4 = 256 rows, the highest
  int nbx;          // column tiles
  float tile[4];    // time of a tile of 1 .. 4 units
};
constexpr int kMaxUnits = 4;

__host__ __device__ inline float moe_cost(const MoeHeights& h, int tiles, int units) {
  constexpr int kXcd = 8;
  const int per = (tiles * h.nbx + kXcd - 1) / kXcd;
  return h.tile[units - 1] * static_cast<float>((per + h.xcd_cus - 1) / h.xcd_cus);
}

// One product's table: where it goes and what its tiles may be.
struct MoePlan {
  MoeTile* table;
  int max_tiles;
  MoeHeights heights;
};

// Row-tile table of a grouped launch.  cum[e] is the number of rows of experts
// 0 .. e (the inclusive running total that the reference's moe_dispatch returns
// as token_nums_per_expert,
// paddle/phi/kernels/fusion/cutlass/moe_dispatch.cu:174-182): expert e owns
// rows cum[e-1] .. cum[e]-1 and ceil(rows / bm) tiles.  One workgroup;
// EXPERTS: one per product.
// EXPERTS false: tiles of bm rows, max_tiles entries, unused ones marked -1.
// EXPERTS true (gemm_experts_kernel): bm is chosen here, where the rows of every
// expert are known (MoeHeights), entry 0 holds the number of tiles, and an
// expert's rows are shared out in 64-row units as evenly as its ceil(rows /
// bm) tiles allow (three tiles of 192 rows rather than two of 256 and one of
// 64: the weight side of a tile costs the same whatever its height).
template <bool EXPERTS>
__global__ __launch_bounds__(256) void moe_plan_kernel(const int64_t* __restrict__ cum, int num_experts, int bm,
                                                       int64_t rows, MoePlan first, MoePlan second) {
  const MoePlan& plan = EXPERTS && blockIdx.x == 1 ? second : first;  // EXPERTS: a workgroup per product
  const MoeHeights& heights = plan.heights;
  const int max_tiles = plan.max_tiles;
  MoeTile* __restrict__ table = plan.table;
  __shared__ int first_tile[1025];  // exclusive running total of tiles, by expert
  __shared__ int row_end[1025];     // end of expert e's rows is row_end[e + 1]; row_end[0] = 0
  if (!EXPERTS)
    for (int i = threadIdx.x; i < max_tiles; i += 256) table[i] = MoeTile{-1, 0, 0, 0, 0, {0, 0, 0}};
  // The running totals come from the device and are not trusted: each is
  // clamped to [previous total, rows], so an expert's count is never negative
  // and no tile reaches past the last row of the input.
  if (!EXPERTS) {
    if (threadIdx.x == 0) {
      int acc = 0;
      int64_t prev = 0;
      row_end[0] = 0;
      for (int e = 0; e < num_experts; ++e) {
        first_tile[e] = acc;
        int64_t end = cum[e];
        end = end < prev ? prev : (end > rows ? rows : end);
        acc += static_cast<int>((end - prev + bm - 1) / bm);
        prev = end;
        row_end[e + 1] = static_cast<int>(end);
      }
      first_tile[num_experts] = acc;
    }
  } else if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int tiles[kMaxUnits] = {0, 0, 0, 0};  // row tiles under a limit of 1 .. 4 units
    int carry = 0;
    if (lane == 0) row_end[0] = 0;
    for (int e0 = 0; e0 < num_experts; e0 += 64) {
      const int e = e0 + lane;
      const int64_t total = e < num_experts ? cum[e] : 0;
      int end = static_cast<int>(total < 0 ? 0 : (total > rows ? rows : total));
      end = end > carry ? end : carry;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(end, d);
        end = lane >= d && o > end ? o : end;
      }
      const int before = __shfl_up(end, 1);
      const int units = (end - (lane == 0 ? carry : before) + 63) / 64;
#pragma unroll
      for (int u = 1; u <= kMaxUnits; ++u) tiles[u - 1] += (units + u - 1) / u;
      if (e < num_experts) row_end[e + 1] = end;
      carry = __shfl(end, 63);
    }
    float best = 0.0f;
#pragma unroll
    for (int u = kMaxUnits; u >= 1; --u) {
      int n = tiles[u - 1];
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) n += __shfl_xor(n, d);
      const float cost = moe_cost(heights, n, u);
      if (u == kMaxUnits || (u >= heights.min_units && n <= max_tiles && cost < best)) {
        best = cost;
        bm = u * 64;
      }
    }
    __builtin_amdgcn_wave_barrier();  // row_end is read back by other lanes
    int acc = 0;
    for (int e0 = 0; e0 < num_experts; e0 += 64) {
      const int e = e0 + lane;
      const int nt = e < num_experts ? (row_end[e + 1] - row_end[e] + bm - 1) / bm : 0;
      int sum = nt;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(sum, d);
        sum += lane >= d ? o : 0;
      }
      if (e < num_experts) first_tile[e] = acc + sum - nt;
      acc += __shfl(sum, 63);
    }
    if (lane == 0) {
      first_tile[num_experts] = acc;
      table[0] = MoeTile{acc < max_tiles ? acc : max_tiles, 0, 0, 0, 0, {0, 0, 0}};
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < num_experts; e += 256) {
    const int r0 = row_end[e], r1 = row_end[e + 1];
    const int t0 = first_tile[e], nt = first_tile[e + 1] - t0;
    const int units = (r1 - r0 + 63) / 64;
    int row = r0;
    for (int t = 0; t < nt && t0 + t < max_tiles; ++t) {
      const int left = r1 - row;
      const int h = EXPERTS ? (units / nt + (t < units % nt ? 1 : 0)) * 64 : bm;
      table[(EXPERTS ? 1 : 0) + t0 + t] = MoeTile{e, row, left < h ? left : h, t0, nt, {0, 0, 0}};
      row += h;
    }
  }
}

// Rows of a grouped launch's tiles, by the average number of rows per expert
// (the host knows the total only; the per-expert counts stay on the device).
// Up to 64 rows each -- a decode step of a mixture of experts -- the small-M
// configurations' 64 x 256 (32 x 256 for int4) tiles: a taller one would do up
// to eight times the MFMA work and hold one workgroup per CU where three fit.
// Above, gemm_experts_kernel with tiles of up to 256 rows (MoeHeights).
constexpr int kExpertsRows = 256;
inline int moe_tile_rows(int64_t rows, int num_experts, int bits) {
  const int64_t avg = rows / (num_experts > 0 ? num_experts : 1);
  if (avg <= 32 && bits == 4) return 32;
  if (avg <= 64) return 64;
  return kExpertsRows;
}

// What a grouped launch needs besides the problem: the row-tile table, and
// for K runs (ns > 1; bias must be null, the runs' sums have no expert) the
// scratch for ns x rows x N floats and the device word that holds the number
// of rows that belong to an expert.
struct MoeLaunch {
  const int* table;
  int max_tiles, bm, ns;
  bool narrow;  // gemm_experts_kernel on 128-column tiles instead of 256
  int64_t rows;
  float* partial;
  const int64_t* valid_rows;
};

// One grouped GEMM: every expert's rows against that expert's weights, tiles
// of WM * TM * 32 rows x 256 columns, per-channel scales, out [rows, N] T.
template <int DT, int BITS, bool OFFS, int WM, int WN, int TM, int TN>
void launch_moe_gemm_cfg(const void* x, const MoeLaunch& ml, const void* codes, const void* bias,
                         const void* scale, int64_t K, int64_t N, void* out, hipStream_t stream) {
  const int* table = ml.table;
  const int max_tiles = ml.max_tiles;
  constexpr int BN = TN * WN * 32;  // output columns of a tile
  constexpr size_t lds = dma_lds_bytes<BITS, 0, WM, WN, TM, TN>();
  auto kern = gemm_dma_kernel<DT, BITS, 0, OFFS, WM, WN, TM, TN>;
  static std::atomic<uint32_t> configured{0};
  allow_lds(reinterpret_cast<const void*>(kern), lds, configured);
  DmaParams p;
  p.x = static_cast<const uint16_t*>(x);
  p.codes = static_cast<const uint8_t*>(codes);
  p.bias = static_cast<const uint16_t*>(bias);
  p.scale = static_cast<const uint16_t*>(scale);
  const int tiles = static_cast<int>(K / (BITS == 8 ? 64 : 128));
  const int ns = bias == nullptr && ml.partial != nullptr ? ml.ns : 1;
  p.M = WM * TM * 32; p.K = static_cast<int>(K); p.N = static_cast<int>(N);
  p.out_f32 = 0;
  p.strip_lo = 0; p.strip_hi = static_cast<int>(N / kStripCols);
  p.nbx = static_cast<int>((N + BN - 1) / BN);
  p.nby = max_tiles;
  p.xcd_rows = 0;
  p.tiles_per_split = (tiles + ns - 1) / ns;
  p.nsplit = (tiles + p.tiles_per_split - 1) / p.tiles_per_split;
  p.out = p.nsplit > 1 ? static_cast<void*>(ml.partial) : out;
  p.act = WOL_ACT_NONE;
  p.moe_table = table;
  p.moe_codes_stride = K * N * BITS / 8;
  p.moe_rows = static_cast<int>(ml.rows);
  p.stamps = nullptr;
  kern<<<dim3(static_cast<unsigned>(p.nbx * p.nby * p.nsplit)), dim3(64 * WM * WN), lds, stream>>>(p);
  if (p.nsplit > 1) {
    const int64_t total = ml.rows * N;
    reduce_partials_kernel<DT><<<dim3(static_cast<unsigned>((total / 4 + 255) / 256)), dim3(256), 0, stream>>>(
        ml.partial, p.nsplit, nullptr, out, 0, total, static_cast<int>(N), 0, static_cast<int>(N), WOL_ACT_NONE,
        ml.valid_rows);
  }
}

// The grouped GEMM on tiles of up to 256 rows x 256 (or 128) columns.  swiglu: of
// the product is formed in the epilogue, out is [rows, N / 2] and a tile has half
// as many output columns.
template <int DT>
void launch_experts(const void* x, const MoeLaunch& ml, const void* codes, const void* bias, const void* scale, int bits,
                    int64_t K, int64_t N, void* out, hipStream_t stream, bool swiglu) {
  const int bn = swiglu || ml.narrow ? 128 : 256;  // output columns of a tile
  DmaParams p{};
  p.x = static_cast<const uint16_t*>(x);
  p.codes = static_cast<const uint8_t*>(codes);
  p.bias = static_cast<const uint16_t*>(bias);
  p.scale = static_cast<const uint16_t*>(scale);
  p.out = out;
  p.M = kExpertsRows; p.K = static_cast<int>(K); p.N = static_cast<int>(N);
  const int64_t out_cols = swiglu ? N / 2 : N;
  p.strip_hi = static_cast<int>(out_cols / kStripCols);
  p.nbx = static_cast<int>((out_cols + bn - 1) / bn);
  p.nby = ml.max_tiles;
  p.nsplit = 1;
  p.tiles_per_split = static_cast<int>(K / 64);
  p.act = WOL_ACT_NONE;
  p.moe_table = ml.table;
  p.moe_codes_stride = K * N * bits / 8;
  p.moe_rows = static_cast<int>(ml.rows);
  const unsigned blocks = static_cast<unsigned>((static_cast<int64_t>(p.nbx) * p.nby + 7) / 8 * 8);  // the XCDs' shares are rounded up
  if (DT == WOL_DTYPE_BF16) launch_experts_bf16(p, bits, ml.narrow && !swiglu, swiglu, blocks, stream);
  else launch_experts_f16(p, bits, ml.narrow && !swiglu, swiglu, blocks, stream);
}

// ml.bm: the tile rows the table was built for (moe_tile_rows).  swiglu: out is
// [rows, N / 2], the swiglu of the product (tiles of 256 rows only).
template <int DT, int BITS>
void launch_moe_gemm(const void* x, const MoeLaunch& ml, const void* codes, const void* bias,
                     const void* scale, int64_t K, int64_t N, void* out, hipStream_t stream, bool swiglu = false) {
  if (ml.bm == kExpertsRows) {
    launch_experts<DT>(x, ml, codes, bias, scale, BITS, K, N, out, stream, swiglu);
    return;
  }
  if constexpr (BITS == 4) {
    if (ml.bm == 32) {
      launch_moe_gemm_cfg<DT, 4, true, 1, 8, 1, 1>(x, ml, codes, bias, scale, K, N, out, stream);
      return;
    }
  }
  launch_moe_gemm_cfg<DT, BITS, false, 1, 8, 2, 1>(x, ml, codes, bias, scale, K, N, out, stream);
}

// K runs of a grouped launch with small tiles: as many as bring the workgroups
// (column tiles x row tiles x runs) to the CU count, at most 4, each of at
// least 8 k tiles.  The large tile is not split.
inline int moe_runs(int64_t K, int64_t N, int bits, int bm, int max_tiles) {
  if (bm == kExpertsRows) return 1;
  const int64_t tiles = K / (bits == 8 ? 64 : 128), wgs = (N + 255) / 256 * max_tiles;
  int ns = static_cast<int>((num_cus() + wgs - 1) / wgs);
  ns = ns > 4 ? 4 : ns;
  while (ns > 1 && tiles / ns < 8) --ns;
  return ns < 1 ? 1 : ns;
}
constexpr int kMoeMaxRuns = 4;

template <int DT, int BITS>
void launch_cfg(const Args& a) {
  constexpr int TK = BITS == 8 ? 64 : 128;
  if (a.K % TK == 0 && a.K / TK >= 2) {
    if (a.gshift < 0) launch_fast<DT, BITS, 0>(a);
    else if (a.gshift == 6) launch_fast<DT, BITS, 64>(a);
    else launch_fast<DT, BITS, 128>(a);
    return;
  }
  if (a.gshift >= 0) {
    launch_one<DT, BITS, true, 2, 4, 8, 2>(a);   // 256 x 128, partial accumulators per group
  } else {
    launch_one<DT, BITS, false, 2, 4, 8, 4>(a);  // 256 x 256
  }
}

// out [M, N / 2] = T(swiglu(x . W + bias)) in one launch
template <int DT, int BITS, int G>
void launch_swiglu_gemm(const Args& a) {
  const int gate_strips = a.N / 2 / kStripCols;
  // whole tiles, or half-size ones where their rounds, at 0.6 of a whole tile's, are done sooner
  const int cus = num_cus(), cols = (a.N + 255) / 256;
  const int big = cols * ((a.M + 255) / 256), half = cols * ((a.M + 127) / 128);
  const WideTile tile = (big + cus - 1) / cus >= 0.6 * ((half + cus - 1) / cus) ? WideTile::kHalf : WideTile::kWhole;
  launch_wide<DT>(a, BITS, G, tile, 1, 0, gate_strips, 1);
}
template <int DT, int BITS>
void launch_swiglu_gemm_g(const Args& a) {
  if (a.gshift < 0) launch_swiglu_gemm<DT, BITS, 0>(a);
  else if (a.gshift == 6) launch_swiglu_gemm<DT, BITS, 64>(a);
  else launch_swiglu_gemm<DT, BITS, 128>(a);
}

}  // namespace

#define WOL_CAT_(a, b) a##b
#define WOL_CAT(a, b) WOL_CAT_(a, b)
#if defined(WOL_GEMM_F16_UNIT)
#define WOL_TYPED(name) WOL_CAT(name, _f16)
#else
#define WOL_TYPED(name) WOL_CAT(name, _bf16)
#endif

void WOL_TYPED(gemm)(const GemmArgs& a, int bits) {
  if (bits == 8) launch_cfg<WOL_GEMM_DTYPE, 8>(a); else launch_cfg<WOL_GEMM_DTYPE, 4>(a);
}

void WOL_TYPED(swiglu_gemm)(const GemmArgs& a, int bits) {
  if (bits == 8) launch_swiglu_gemm_g<WOL_GEMM_DTYPE, 8>(a); else launch_swiglu_gemm_g<WOL_GEMM_DTYPE, 4>(a);
}

void WOL_TYPED(moe_gemm)(const MoeGemmArgs& a, int bits) {
  const MoeLaunch ml{a.table, a.max_tiles, a.bm, a.ns, a.narrow, a.rows, a.partial, a.valid_rows};
  if (bits == 8) launch_moe_gemm<WOL_GEMM_DTYPE, 8>(a.x, ml, a.codes, a.bias, a.scale, a.K, a.N, a.out, a.stream, a.swiglu);
  else launch_moe_gemm<WOL_GEMM_DTYPE, 4>(a.x, ml, a.codes, a.bias, a.scale, a.K, a.N, a.out, a.stream, a.swiglu);
}

#if !defined(WOL_GEMM_F16_UNIT)

int launch_reduce_partials(const float* part, int nsplit, const void* bias, int dtype, void* out,
                           bool out_f32, int64_t M, int64_t N, int act, hipStream_t stream) {
  if (act == WOL_ACT_SWIGLU) {  // out is [M, N/2]
    if (N % 8 != 0) return WOL_ERR_BAD_SHAPE;
    const int64_t total = M * N / 2;
    const dim3 grid(static_cast<unsigned>((total / 4 + 255) / 256)), block(256);
    if (dtype == WOL_DTYPE_BF16)
      reduce_partials_swiglu_kernel<WOL_DTYPE_BF16><<<grid, block, 0, stream>>>(
          part, nsplit, static_cast<const uint16_t*>(bias), out, out_f32 ? 1 : 0, total, static_cast<int>(N));
    else
      reduce_partials_swiglu_kernel<WOL_DTYPE_F16><<<grid, block, 0, stream>>>(
          part, nsplit, static_cast<const uint16_t*>(bias), out, out_f32 ? 1 : 0, total, static_cast<int>(N));
    return check_launch();
  }
  const int64_t total = M * N;
  const dim3 grid(static_cast<unsigned>((total / 4 + 255) / 256)), block(256);
  if (dtype == WOL_DTYPE_BF16)
    reduce_partials_kernel<WOL_DTYPE_BF16><<<grid, block, 0, stream>>>(
        part, nsplit, static_cast<const uint16_t*>(bias), out, out_f32 ? 1 : 0, total, static_cast<int>(N), 0,
        static_cast<int>(N), act);
  else
    reduce_partials_kernel<WOL_DTYPE_F16><<<grid, block, 0, stream>>>(
        part, nsplit, static_cast<const uint16_t*>(bias), out, out_f32 ? 1 : 0, total, static_cast<int>(N), 0,
        static_cast<int>(N), act);
  return check_launch();
}

size_t linear_gemm_workspace(int64_t M, int64_t K, int64_t N, int bits, int group_size) {
  const int tk = bits == 8 ? 64 : 128;
  if (K % tk != 0 || K / tk < 2) return 0;
  if (M > kSkinnyMaxM) {
    const int g = group_size > 0 ? group_size : 0;
    const int lo = half_tile_strip(static_cast<int>(M), static_cast<int>(K), static_cast<int>(N), bits, g);
    const int ncols = static_cast<int>(N) - lo * kStripCols;
    const TailPlan t = plan_tail(static_cast<int>(M), static_cast<int>(K), ncols, kHalfRows, kHalfCols, tk, SIZE_MAX);
    return t.ns > 1 ? static_cast<size_t>(t.ns) * M * (ncols - t.full_tiles * kHalfCols) * sizeof(float) : 0;
  }
  const int ns = plan_skinny(static_cast<int>(M), static_cast<int>(K), static_cast<int>(N), bits,
                             group_size > 0 ? group_size : 0, SIZE_MAX).ns;
  return ns > 1 ? static_cast<size_t>(ns) * M * N * sizeof(float) : 0;
}

void describe_linear_gemm(int64_t M, int64_t K, int64_t N, int bits, int group_size, size_t ws_bytes,
                          char* buf, size_t n) {
  const int tk = bits == 8 ? 64 : 128;
  const int g = group_size > 0 ? group_size : 0;
  if (K % tk != 0 || K / tk < 2) {
    snprintf(buf, n, "wol::gemm_kernel (register-staged v_mfma_f32_16x16x32, 256 x %d tiles)", g ? 128 : 256);
    return;
  }
  if (M <= kSkinnyMaxM) {
    const SkinnyPlan sp = plan_skinny(static_cast<int>(M), static_cast<int>(K), static_cast<int>(N), bits, g, ws_bytes);
    const bool wide = sp.wide;
    const int ns = sp.ns;
    snprintf(buf, n, "wol::gemm_dma_kernel: %d rows x %d columns per workgroup, K in %d run(s)%s",
             bits == 4 && M <= 32 ? 32 : 64, wide ? 512 : 256, ns, ns > 1 ? " + reduce_partials_kernel" : "");
    return;
  }
  const int lo = half_tile_strip(static_cast<int>(M), static_cast<int>(K), static_cast<int>(N), bits, g);
  const int nstrips = static_cast<int>(N / kStripCols);
  const TailPlan t = plan_tail(static_cast<int>(M), static_cast<int>(K), (nstrips - lo) * kStripCols, kHalfRows, kHalfCols, tk, ws_bytes);
  const int mid = lo + t.full_tiles * (kHalfCols / kStripCols);
  int len = 0;
  const bool tall = lo > 0 && g != 0;  // group-wise scales on whole tiles have a kernel of their own
  if (tall)
    len += snprintf(buf + len, n - len, "wol::gemm_dma_kernel_tall (v_mfma_f32_32x32x16): 256x256 tiles on columns [0,%d)%s",
                    lo * kStripCols, nstrips > lo ? "; " : "");
  if ((!tall || nstrips > lo) && len < static_cast<int>(n))
    len += snprintf(buf + len, n - len, "%sgemm_dma_kernel_wide (v_mfma_f32_16x16x32):", tall ? "" : "wol::");
  if (lo > 0 && !tall && len < static_cast<int>(n))
    len += snprintf(buf + len, n - len, " 256x256 tiles on columns [0,%d)", lo * kStripCols);
  if (mid > lo && len < static_cast<int>(n))
    len += snprintf(buf + len, n - len, " 128x256 tiles on [%d,%d)", lo * kStripCols, mid * kStripCols);
  if (nstrips > mid && len < static_cast<int>(n))
    len += snprintf(buf + len, n - len, " 128x256 tiles on [%d,%d)%s", mid * kStripCols, nstrips * kStripCols,
                    t.ns > 1 ? " with K in runs + reduce_partials_kernel" : "");
}

// swiglu of a gate | up projection inside the GEMM's epilogue: the tiles with two
// blocks per wavefront, above the small-M configurations.
// Up to 64 rows: where K is cut into runs, in the kernel that adds them.
bool linear_gemm_fuses_swiglu(int64_t M, int64_t K, int64_t N, int bits, int group_size) {
  const int tk = bits == 8 ? 64 : 128;
  if (K % tk != 0 || K / tk < 2 || N % 32 != 0) return false;
  if (M > kSkinnyMaxM) return true;
  return plan_skinny(static_cast<int>(M), static_cast<int>(K), static_cast<int>(N), bits,
                     group_size > 0 ? group_size : 0, SIZE_MAX).ns > 1;
}

// f.act == WOL_ACT_SWIGLU (only where linear_gemm_fuses_swiglu): out is [M, N / 2] T.
int launch_linear_gemm(const void* x, const void* codes, const void* bias, const void* scale,
                       int dtype, int64_t M, int64_t K, int64_t N, int bits, int group_size,
                       void* out, bool out_f32, void* workspace, size_t workspace_bytes,
                       hipStream_t stream, const Fuse& f) {
  const int gshift = group_size == 64 ? 6 : (group_size == 128 ? 7 : -1);
  const Args a{x, codes, bias, scale, out, static_cast<int>(M), static_cast<int>(K),
               static_cast<int>(N), gshift, out_f32 ? 1 : 0, workspace, workspace_bytes, stream, f.act};
  if (f.act == WOL_ACT_SWIGLU && M <= kSkinnyMaxM) {
    // the runs of K must be the ones the plan was made with: all of the scratch is required
    if (out_f32 || !linear_gemm_fuses_swiglu(M, K, N, bits, group_size)) return WOL_ERR_BAD_SHAPE;
    if (workspace == nullptr || workspace_bytes < linear_gemm_workspace(M, K, N, bits, group_size)) return WOL_ERR_WORKSPACE;
  } else if (f.act == WOL_ACT_SWIGLU) {
    if (out_f32 || !linear_gemm_fuses_swiglu(M, K, N, bits, group_size)) return WOL_ERR_BAD_SHAPE;
    if (dtype == WOL_DTYPE_BF16) swiglu_gemm_bf16(a, bits); else swiglu_gemm_f16(a, bits);
    return check_launch();
  }
  if (dtype == WOL_DTYPE_BF16) gemm_bf16(a, bits); else gemm_f16(a, bits);
  return check_launch();
}

// ---- mixture-of-experts FFN ---------------------------------------------------
static size_t moe_up(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }

// Entries of the row-tile table for tiles of bm rows: every expert may end in
// a partial tile.
static int moe_max_tiles(int64_t rows, int num_experts, int bm) {
  return static_cast<int>((rows + bm - 1) / bm) + num_experts;
}

// What the host settles of a gemm_experts_kernel call: the lowest height limit
// each product's grid is laid out for, and whether the second product takes
// 128-column tiles.  The rows of each expert are not known here: even loads are
// assumed, and for the limit the device looks again (moe_plan_kernel).  Workgroups
// that find no tile cost little but not nothing, so a limit below 256 rows is
// offered only where it asks for at most twelve rounds of them.
static MoeHeights plan_moe_heights(int64_t rows, int64_t cols, int bn, int num_experts, float column_cost) {
  const int cus = num_cus();
  MoeHeights h;
  h.xcd_cus = cus / 8 > 0 ? cus / 8 : 1;
  h.nbx = static_cast<int>((cols + bn - 1) / bn);
  const float times[kMaxUnits] = {0.54f, 0.66f, 0.84f, 1.0f};
  for (int u = 0; u < kMaxUnits; ++u) h.tile[u] = times[u] * column_cost;
  h.min_units = 1;
  while (h.min_units < kMaxUnits &&
         static_cast<int64_t>(moe_max_tiles(rows, num_experts, h.min_units * 64)) * h.nbx > 12 * cus)
    ++h.min_units;
  return h;
}

// The best estimate under any limit, the experts evenly loaded.
static float best_moe_cost(const MoeHeights& h, int64_t rows, int num_experts) {
  const int64_t units = ((rows + num_experts - 1) / num_experts + 63) / 64;
  float best = 0.0f;
  for (int u = kMaxUnits; u >= h.min_units; --u) {
    const float c = moe_cost(h, static_cast<int>((units + u - 1) / u) * num_experts, u);
    best = u == kMaxUnits || c < best ? c : best;
  }
  return best;
}

// Scratch: [row-tile tables of the two products][fc1 output rows x inter T][activation rows x inter/2 T]
// [fp32 sums of the second GEMM's K runs, rows x hidden each, when the tiles are small]
size_t moe_ffn_workspace(int64_t rows, int64_t hidden, int64_t inter, int num_experts) {
  // (the table at its longest: 32-row tiles; the runs' sums whenever either bit width would use small tiles)
  const bool small = moe_tile_rows(rows, num_experts, 4) < 128;
  return 2 * moe_up((static_cast<size_t>(moe_max_tiles(rows, num_experts, 32)) + 1) * sizeof(MoeTile)) +
         moe_up(static_cast<size_t>(rows) * inter * 2) + moe_up(static_cast<size_t>(rows) * (inter / 2) * 2) +
         (small ? moe_up(static_cast<size_t>(kMoeMaxRuns) * rows * hidden * sizeof(float)) : 0);
}

int launch_moe_ffn(const void* x, const int64_t* rows_before_expert, const void* ffn1_codes,
                   const void* ffn1_bias, const void* ffn1_scale, const void* ffn2_codes,
                   const void* ffn2_scale, int dtype, int64_t rows, int64_t hidden, int64_t inter,
                   int num_experts, int bits, void* out, void* workspace, hipStream_t stream) {
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  const int bm = moe_tile_rows(rows, num_experts, bits);
  const bool experts = bm == kExpertsRows;
  const size_t table_bytes = moe_up((static_cast<size_t>(moe_max_tiles(rows, num_experts, 32)) + 1) * sizeof(MoeTile));
  MoePlan plan1{reinterpret_cast<MoeTile*>(ws), moe_max_tiles(rows, num_experts, bm), {}}, plan2 = plan1;
  bool narrow = false;
  if (experts) {
    plan1.heights = plan_moe_heights(rows, inter / 2, 128, num_experts, 1.0f);
    plan2.heights = plan_moe_heights(rows, hidden, 256, num_experts, 1.0f);
    const MoeHeights n = plan_moe_heights(rows, hidden, 128, num_experts, 0.7f);
    narrow = best_moe_cost(n, rows, num_experts) < best_moe_cost(plan2.heights, rows, num_experts);
    if (narrow) plan2.heights = n;
    plan1.max_tiles = moe_max_tiles(rows, num_experts, plan1.heights.min_units * 64);
    plan2.max_tiles = moe_max_tiles(rows, num_experts, plan2.heights.min_units * 64);
    plan2.table = reinterpret_cast<MoeTile*>(ws + table_bytes);
  }
  unsigned char* fc1 = ws + 2 * table_bytes;
  unsigned char* act = fc1 + moe_up(static_cast<size_t>(rows) * inter * 2);
  float* partial = reinterpret_cast<float*>(act + moe_up(static_cast<size_t>(rows) * (inter / 2) * 2));
  (experts ? moe_plan_kernel<true> : moe_plan_kernel<false>)<<<dim3(experts ? 2 : 1), dim3(256), 0, stream>>>(
      rows_before_expert, num_experts, bm, rows, plan1, plan2);
  const auto product = [&](const MoeGemmArgs& a) {
    if (dtype == WOL_DTYPE_BF16) moe_gemm_bf16(a, bits); else moe_gemm_f16(a, bits);
  };
  product(MoeGemmArgs{x, reinterpret_cast<const int*>(plan1.table), plan1.max_tiles, bm, 1, false, rows, nullptr, nullptr, ffn1_codes, ffn1_bias, ffn1_scale,
                      hidden, inter, experts ? act : fc1, stream, experts});
  if (!experts) {
    const int rc = launch_swiglu_t(fc1, dtype, rows, inter, act, stream);
    if (rc != WOL_OK) return rc;
  }
  // the second product has hidden / 256 column tiles only: K (= inter / 2) in runs when the tiles are small
  product(MoeGemmArgs{act, reinterpret_cast<const int*>(plan2.table), plan2.max_tiles, bm,
                      moe_runs(inter / 2, hidden, bits, bm, plan2.max_tiles), narrow, rows,
                      experts ? nullptr : partial, rows_before_expert + (num_experts - 1), ffn2_codes, nullptr, ffn2_scale,
                      inter / 2, hidden, out, stream, false});
  return check_launch();
}

// ---- the prefill kernel's inner loop, one ingredient at a time (wol_mfma_probe) ----
namespace {

// The register tile and instruction mix of a 256 x 256 tile of two by four
// wavefronts (4 x 2 blocks of v_mfma_f32_32x32x16 each, k tiles of four
// slices) with its ingredients switched on one by one, and no global memory
// traffic other than what LOADS adds.  No product kernel has this form any more
// (those of wol_linear_wide.hip put their wavefronts side by side); the ladder
// says what each ingredient costs the matrix pipes of this machine:
//   DQ     B fragments dequantised per slice (int8 -> bf16, exact) out of raw
//          codes read from LDS once per tile (0 or 2)
//   NA     A fragments read from LDS per slice (0 or 4)
//   BAR    one workgroup barrier per tile
//   LOADS  six direct-to-LDS loads (1 KiB each) per wavefront and tile out of
//          a 25 MB region of `ops`, two stages, waited for before the barrier
//   M16    v_mfma_f32_16x16x32 on 8 x 4 blocks instead (the same flops)
template <bool M16, int DQ, int NA, bool BAR, bool LOADS>
__global__ __launch_bounds__(512) void mfma_probe_kernel(const u32x4* __restrict__ ops, int iters,
                                                         float* __restrict__ out) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  for (int i = tid; i < 6144; i += 512) reinterpret_cast<u32x4*>(smem)[i] = ops[i & 511];  // 96 KiB of operand pattern
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned char* base = smem + (wave & 3) * 4096 + lane * 16;
  float total = 0.0f;
  if constexpr (!M16) {
    f32x16 acc[4][2];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][c][r] = 0.0f;
    u32x4 af[2][4], bf[2][2], raw[2][2];
#pragma unroll
    for (int a = 0; a < 4; ++a) af[0][a] = af[1][a] = *reinterpret_cast<const u32x4*>(base + a * 1024);
#pragma unroll
    for (int c = 0; c < 2; ++c) bf[0][c] = bf[1][c] = *reinterpret_cast<const u32x4*>(base + 16384 + c * 1024);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) raw[c][h] = *reinterpret_cast<const u32x4*>(base + 32768 + (c * 2 + h) * 1024);
    for (int it = 0; it < iters; ++it) {
      const unsigned char* tb = base + ((it & 3) << 14);
      if (DQ > 0) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int h = 0; h < 2; ++h) raw[c][h] = *reinterpret_cast<const u32x4*>(tb + (c * 2 + h) * 1024 + 8192);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (NA > 0) {
#pragma unroll
          for (int a = 0; a < NA; ++a)
            af[(q + 1) & 1][a] = *reinterpret_cast<const u32x4*>(tb + ((q * 4 + a) & 7) * 1024);
        }
        if (DQ > 0) {
          const int step = ((q + 1) & 3) / 2, h = (q + 1) % 2;
#pragma unroll
          for (int c = 0; c < DQ; ++c) {
            const uint32_t w4[4] = {raw[c][h].x, raw[c][h].y, raw[c][h].z, raw[c][h].w};
            bf[(q + 1) & 1][c] = DequantExact<WOL_DTYPE_BF16, 8>::run(&w4[step * 2]);
          }
        }
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[a][c] = mfma32<WOL_DTYPE_BF16>(af[q & 1][a], bf[q & 1][c], acc[a][c]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (i < NA) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          if (DQ > 0) __builtin_amdgcn_sched_group_barrier(0x002, (14 * DQ + 7) / 8 + 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (LOADS) {
        wait_vmcnt<6>();
        __builtin_amdgcn_s_barrier();
        unsigned char* stage = smem + 65536 + (it & 1) * 49152;
        const unsigned char* g = reinterpret_cast<const unsigned char*>(ops) +
                                 ((static_cast<int>(blockIdx.x) & 63) * 8 + (it & 7)) * 49152;
#pragma unroll
        for (int c = 0; c < 6; ++c)
          __builtin_amdgcn_global_load_lds(g + (c * 8 + wave) * 1024 + lane * 16,
                                           (lds_ptr_t)(stage + (c * 8 + wave) * 1024), 16, 0, 0);
      } else if (BAR) {
        __builtin_amdgcn_s_barrier();
      }
    }
    if (LOADS) wait_vmcnt<0>();
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) total += acc[a][c][r];
  } else {
    f32x4 acc[8][4];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[a][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 af[2][8], bf[2][4], raw[4];
#pragma unroll
    for (int a = 0; a < 8; ++a) af[0][a] = af[1][a] = *reinterpret_cast<const u32x4*>(base + a * 1024);
#pragma unroll
    for (int c = 0; c < 4; ++c) bf[0][c] = bf[1][c] = *reinterpret_cast<const u32x4*>(base + 16384 + c * 1024);
#pragma unroll
    for (int c = 0; c < 4; ++c) raw[c] = *reinterpret_cast<const u32x4*>(base + 32768 + c * 1024);
    for (int it = 0; it < iters; ++it) {
      const unsigned char* tb = base + ((it & 3) << 14);
      if (DQ > 0) {
#pragma unroll
        for (int c = 0; c < 4; ++c) raw[c] = *reinterpret_cast<const u32x4*>(tb + c * 1024 + 8192);
      }
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        if (NA > 0) {
#pragma unroll
          for (int a = 0; a < 2 * NA; ++a)
            af[(st + 1) & 1][a] = *reinterpret_cast<const u32x4*>(tb + ((st * 8 + a) & 7) * 1024);
        }
        if (DQ > 0) {
#pragma unroll
          for (int c = 0; c < 2 * DQ; ++c) {
            const uint32_t w4[4] = {raw[c].x, raw[c].y, raw[c].z, raw[c].w};
            bf[(st + 1) & 1][c] = DequantExact<WOL_DTYPE_BF16, 8>::run(&w4[((st + 1) & 1) * 2]);
          }
        }
#pragma unroll
        for (int a = 0; a < 8; ++a)
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[a][c] = mfma16<WOL_DTYPE_BF16>(af[st & 1][a], bf[st & 1][c], acc[a][c]);
#pragma unroll
        for (int i = 0; i < 32; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (i < 2 * NA) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          if (DQ > 0) __builtin_amdgcn_sched_group_barrier(0x002, (14 * 2 * DQ + 31) / 32 + 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (BAR) __builtin_amdgcn_s_barrier();
    }
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) total += acc[a][c][r];
  }
  out[static_cast<int64_t>(blockIdx.x) * 512 + tid] = total;
#endif
}

template <bool M16, int DQ, int NA, bool BAR, bool LOADS>
void launch_probe(const void* ops, int wgs, int iters, float* out, hipStream_t s) {
  auto kern = mfma_probe_kernel<M16, DQ, NA, BAR, LOADS>;
  static std::atomic<uint32_t> configured{0};
  const size_t lds = LOADS ? 160 * 1024 : 96 * 1024;  // one workgroup per CU either way
  allow_lds(reinterpret_cast<const void*>(kern), lds, configured);
  kern<<<dim3(static_cast<unsigned>(wgs)), dim3(512), lds, s>>>(static_cast<const u32x4*>(ops), iters, out);
}

}  // namespace

int launch_mfma_probe(int variant, const void* ops, int workgroups, int iters, float* out, hipStream_t stream) {
  switch (variant) {
    case 0: launch_probe<false, 0, 0, false, false>(ops, workgroups, iters, out, stream); break;
    case 1: launch_probe<false, 2, 0, false, false>(ops, workgroups, iters, out, stream); break;
    case 2: launch_probe<false, 0, 4, false, false>(ops, workgroups, iters, out, stream); break;
    case 3: launch_probe<false, 2, 4, false, false>(ops, workgroups, iters, out, stream); break;
    case 4: launch_probe<false, 2, 4, true, false>(ops, workgroups, iters, out, stream); break;
    case 5: launch_probe<false, 2, 4, true, true>(ops, workgroups, iters, out, stream); break;
    case 6: launch_probe<false, 0, 0, true, true>(ops, workgroups, iters, out, stream); break;
    case 7: launch_probe<true, 0, 0, false, false>(ops, workgroups, iters, out, stream); break;
    case 8: launch_probe<true, 2, 4, true, false>(ops, workgroups, iters, out, stream); break;
    default: return WOL_ERR_BAD_SHAPE;
  }
  return check_launch();
}

#endif  // !WOL_GEMM_F16_UNIT

}  // namespace wol
