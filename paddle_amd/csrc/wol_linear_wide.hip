// The tiles of 128 and 256 rows of weight_only_linear's GEMM (more than 64 rows, K made of whole k tiles), for bf16:
// gemm_dma_kernel_wide and, for group-wise scales on 256 x 256 tiles, gemm_dma_kernel_tall.
// wol_linear_wide_f16.hip compiles the same source for fp16.  This file is built with the instruction scheduler in front
// of register allocation switched off (build.sh): the loops below give every instruction its place, and that pass, which
// does not see why, costs up to 40 registers and then spills (int4 per channel: 240 registers without it, 256 and
// spills with it).
//
// gemm_dma_kernel_wide.  A workgroup of eight wavefronts, WM x WN, computes WM*TM*16 rows x WN*TN*16 columns from
// v_mfma_f32_16x16x32 blocks, TM x TN per wavefront.  The k tile is 64 deep; three of them are resident or in flight, all
// through direct-to-LDS buffer loads.
//
// What bounds it.  With random operands the part runs into its power limit, so energy counts as much as cycles: the
// 16x16x32 form touches its accumulators once per 32 k, 32x32x16 does every 16 k (a plain fp16 GEMM on these tiles went
// from 1.12 to 1.26 PFLOP/s by the form alone).  In cycles: two wavefronts share a SIMD, an MFMA takes two of its
// ~4.3-cycle issue slots and every VALU instruction one, so beside a 16-cycle MFMA two VALU instructions are free and
// each further one lengthens the loop.  Hence WM = 1: every wavefront covers all rows of 32 columns, a weight is
// dequantised once per workgroup (0.9 VALU instructions per MFMA for int8, 1.2 for exact int4; with two rows of
// wavefronts twice that) at the price of one A fragment out of LDS per two MFMAs, half of what the LDS delivers.
// int8, bf16: M = 2048, K = 4096, N = 8192 109 -> 98 us (1.40 PFLOP/s) against 32x32x16 tiles of two by four wavefronts,
// 100 with two by four wavefronts here; M = 8192, K = N = 4096 215 -> 191; M = 4096, K = 14336, N = 4096 358 -> 319
// (1.51).  int4 per channel M = 2048, N = 8192 112 -> 99, with the exact dequantiser where the row sums of an offset
// form were needed.
//
// Order of a k tile.  Its two halves (32 k each) run TM slots of TN MFMAs, a slot per A block.  The A fragment a slot has
// just used is read again for the next half right behind it, so A needs one set of registers; B fragments have two
// sets, the next half's being dequantised a few instructions per slot.  The workgroup barrier sits a quarter into the
// second half: by then the last reads of the tile have arrived, so nobody waits for LDS there, and everything the next
// tile's first half needs is read and converted behind it.  Tile t+3's loads go out between the barriers of tiles t
// and t+1, a few per slot.
//
// A fragments: rows of 128 bytes, the 16-byte piece XORed with row % 8; the sixteen lanes that a ds_read_b128 serves
// together ({0-3, 12-15, 20-27}, ...) then cover all 64 banks.  B: lane l of a raw strip tile owns column l % 16 and, per
// 32-k step, the eight k from 8 * (l / 16) on: the operand itself.
//
// int4: a raw tile holds 128 k, so it serves two k tiles.  It has two buffers of its own; an odd tile's loads bring the
// first half (by strips) of the next raw tile and the even one's the second (128-column tiles: all of it with the odd
// one).
//
// G != 0 (group-wise scales): one set of accumulators, kept in units of the current group's scale.  Where a group
// starts the running sums are multiplied by (previous unit / new unit) and the group's MFMAs then accumulate straight
// into them; the epilogue multiplies by the last unit.  code * scale is never rounded to T.  A rescaling is off by at most
// 2^-22 relative (v_rcp_f32 by 2^-23, the ratio's and the sums' rounding by 2^-24 each), K / g - 1 times: 223 for K = 14336 in
// groups of 64, 5.3e-5 if all of them fell the same way, where bf16 results are rounded by 2^-9.  Groups of equal scale
// change nothing.  The unit of a column follows its group scale but never
// falls more than 2^64 below the largest scale the column has had so far (a group that small weighs nothing next to the
// others in fp32), so the sums cannot overflow however the scales of a column differ.
//
// SWI: swiglu in the epilogue.  The weight is a gate | up projection, [K, N] with the gate in columns 0 .. N/2-1; half of a
// wavefront's strips are gate columns and the other half the up columns N/2 further on, so that silu(gate) * up is formed
// lane by lane and only [M, N/2] leaves the kernel.
//
// STAMP (a diagnostic instantiation, never on a product path): every wavefront reads the cycle counter at kernel entry,
// around the two waits of every k tile (for its own tile loads, then for the workgroup) and around the epilogue, and
// leaves the sums in p.stamps.
#include "wol_gemm_common.h"

namespace wol {
namespace {

#ifndef WOL_GEMM_DTYPE
#define WOL_GEMM_DTYPE WOL_DTYPE_BF16
#endif

template <int BITS, int G, int WM, int WN, int TM, int TN>
constexpr size_t wide_lds_bytes() {
  const size_t a = static_cast<size_t>(WM) * TM * 16 * 128, b = static_cast<size_t>(WN) * TN * 1024;
  return 3 * (a + (BITS == 8 ? b : 0) + (G == 0 ? 0 : WM * WN * 256)) + (BITS == 4 ? 2 * b : 0);
}

// The tile and the K run of this workgroup: consecutive workgroup ids go to the 8 XCDs in turn, and XCD x takes the x-th
// eighth of the sequence of (run, tile).
__device__ inline void place_of_block(const DmaParams& p, int* bx, int* by, int* split) {
  constexpr int kXcd = 8;
  const int tiles = p.nbx * p.nby, total = tiles * p.nsplit;
  const int x = blockIdx.x % kXcd, q = total / kXcd, r = total % kXcd;
  const int pos = x * q + (x < r ? x : r) + blockIdx.x / kXcd;
  *split = pos / tiles;
  tile_of_position(pos - *split * tiles, p.nbx, p.nby, bx, by);
}

// The same for launches of short K runs (below kShortRun k tiles): every XCD takes a part of every run.  With a run, or part
// of one, to itself an XCD reads the same less than 4 KiB of every row of x, rows that lie a power of two apart more often
// than not, through the few channels of its L2 (256 bytes each in turn, 16 of them) that hold those.  At least as many row
// tiles as column tiles: plain order; fewer: an eighth of the run's tiles, as above, so that the row tiles of a column stay
// together.  us a call, (run, tile) order / plain / eighths of every run: 1300 x 2048 -> 1024 int8, four runs of 8, 22.5 /
// 19.1 / 19.3; 1500 x 1152 -> 1536 int8 g64, two of 9, 25.7 / 22.2 / 25.1; 700 x 1152 -> 4096 int8, two of 9, 24.2 / 22.7 /
// 21.6; 205 x 3584 -> 7904 int8, four of 14, 26.9 / 29.8 / 27.4; 700 x 11008 -> 4096 int8, two of 86, 73.6 / 77.4 / 76.0.
// (A kernel of its own: the other instantiations lose 1 to 3 % by the code alone.)
constexpr int kShortRun = 32;
__device__ inline void place_in_short_run(const DmaParams& p, int* bx, int* by, int* split) {
  constexpr int kXcd = 8;
  const int tiles = p.nbx * p.nby, q = tiles / kXcd, r = tiles % kXcd;
  *split = blockIdx.x / tiles;
  const int w = blockIdx.x - *split * tiles, x = w % kXcd;
  if (p.nby >= p.nbx) {
    *by = w / p.nbx;
    *bx = w - *by * p.nbx;
  } else {
    tile_of_position(x * q + (x < r ? x : r) + w / kXcd, p.nbx, p.nby, bx, by);
  }
}

template <int DT, int BITS, int G, int WM, int WN, int TM, int TN, int SWI, bool STAMP, bool EXPERTS>
__device__ __forceinline__ void wide_tile(const DmaParams& p, const TilePlace at, int split) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NW = WM * WN;
  static_assert(NW == 8, "eight wavefronts");
  constexpr int BM = WM * TM * 16, BN = WN * TN * 16, kStrips = WN * TN;
  constexpr int kABytes = BM * 128, kBBytes = kStrips * 1024;  // an A tile, a raw B tile
  constexpr int kSBytes = G == 0 ? 0 : NW * 256;
  constexpr int kScaleOff = kABytes + (BITS == 8 ? kBBytes : 0);
  constexpr int kStage = kScaleOff + kSBytes;
  constexpr int kRawOff = 3 * kStage;  // int4: the two raw B tiles
  constexpr int kLds = static_cast<int>(wide_lds_bytes<BITS, G, WM, WN, EXPERTS ? 16 / WM : TM, TN>());  // what the launch asks for
  constexpr int kALoads = kABytes / 1024 / NW, kBSlots = kStrips / NW;
  static_assert(kABytes / 1024 % NW == 0 && kStrips % NW == 0, "the tile must split evenly over the wavefronts");
  constexpr int kDw = BITS == 8 ? 2 : 1;  // raw dwords of a B fragment
  static_assert(SWI == 0 || TN % 2 == 0, "gate and up strips in one wavefront");
  // loads of a tile: [scales,] A, B; the B loads of an odd / even tile
  constexpr int kS = G == 0 ? 0 : 1;
  constexpr int kBOdd = BITS == 8 || kBSlots == 1 ? kBSlots : kBSlots / 2;
  constexpr int kBEven = BITS == 8 ? kBSlots : kBSlots - kBOdd;
  constexpr int kLoadsOdd = kS + kALoads + kBOdd, kLoadsEven = kS + kALoads + kBEven;
  // slots of the second half before the barrier, and loads that go out between the barrier and the end of the tile
  constexpr int B0 = TM / 4, kSpan = 2 * TM;  // kSpan: slots from barrier to barrier
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  unsigned long long st_entry = 0, st_prev = 0, st_work = 0, st_loads = 0, st_bar = 0, st_loop0 = 0;
  if (STAMP) st_entry = __builtin_readcyclecounter();

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int lr = lane & 15, kb = lane >> 4;
  const int K = p.K, N = p.N;
  const int m0 = at.row0, M = EXPERTS ? at.row0 + at.rows : p.M;
  const uint16_t* x = p.x;
  const uint16_t* scale = p.scale;
  const uint8_t* codes = p.codes;
  if (EXPERTS) {  // the rows are those of one expert: its weights and scales
    codes += static_cast<int64_t>(at.expert) * p.moe_codes_stride;
    scale += static_cast<int64_t>(at.expert) * N;
  }
  // SWI: BN / 2 gate columns and the BN / 2 up columns that go with them
  const int strip0 = p.strip_lo + at.bx * (SWI ? kStrips / 2 : kStrips);
  const int up_strips = N / 2 / kStripCols;
  const int t0 = split * p.tiles_per_split;  // this workgroup's run of k tiles
  const int nt = (K / 64 - t0) < p.tiles_per_split ? (K / 64 - t0) : p.tiles_per_split;

  const int rows = M - m0 < BM ? M - m0 : BM;
  const int sbytes = static_cast<int>(strip_bytes(K, BITS));
  const int left = p.strip_hi - strip0, strips = left < (SWI ? kStrips / 2 : kStrips) ? left : (SWI ? kStrips / 2 : kStrips);
  // One descriptor per load: it starts at the load's own eight rows (its strip) and ends with the last row (strip) that
  // exists, so edges arrive as zeros and a lane needs the same offset for every load.
  __amdgpu_buffer_rsrc_t ra[kALoads], rb[kBSlots];
#pragma unroll
  for (int c = 0; c < kALoads; ++c) {
    const int r0 = (c * NW + wave) * 8, nr = rows - r0 > 8 ? 8 : (rows > r0 ? rows - r0 : 0);
    ra[c] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x + static_cast<int64_t>(nr > 0 ? m0 + r0 : m0) * K), 0, nr * K * 2, 0x00020000);
  }
  // SWI: LDS slot L of the B tile serves wavefront column L / TN; the first TN / 2 slots of one are its gate strips
#pragma unroll
  for (int c = 0; c < kBSlots; ++c) {
    const int L = c * NW + wave;
    const int st = SWI ? (L / TN) * (TN / 2) + L % TN % (TN / 2) : L;
    const int64_t first = st < strips ? strip0 + st + (SWI && L % TN >= TN / 2 ? up_strips : 0) : 0;
    rb[c] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(codes + first * sbytes), 0, st < strips ? sbytes : 0, 0x00020000);
  }
  const uint32_t aoff = static_cast<uint32_t>((lane / 8) * K + ((lane ^ (lane >> 3)) & 7) * 8) * 2, boff = lane * 16;
  // columns of this wavefront's strips
  auto strip_col = [&](int c) {
    if (SWI) return (strip0 + wn * (TN / 2) + c % (TN / 2)) * kStripCols + (c >= TN / 2 ? N / 2 : 0);
    return (strip0 + wn * TN + c) * kStripCols;
  };
  // group scales travel with the tile: lane l brings columns 2l and 2l + 1 of its wavefront's TN * 16
  int scol = 0;
  if (G != 0) {
    const int v = 2 * lane < TN * 16 ? 2 * lane : 0;
    scol = strip_col(v / 16) + v % 16;
    const int last = (SWI && v / 16 < TN / 2) ? N / 2 : (SWI ? N : p.strip_hi * kStripCols);
    scol = scol < last ? scol : last - 2;  // past the last column: valid data, never used
  }
  constexpr int kGShift = G == 128 ? 7 : 6;
  // load i of tile t (stage st); odd: parity of t
  auto issue1 = [&](int t, int st, bool odd, int i) {
    const int tt = t0 + (t < nt ? t : nt - 1);  // past the end: the last tile again, into a stage that nobody reads
    unsigned char* s = smem + st * kStage;
    if (G != 0 && i == 0) {
      const int64_t row = static_cast<int64_t>(tt) * 64 >> kGShift;
      __builtin_amdgcn_global_load_lds(scale + row * N + scol, (lds_ptr_t)(s + kScaleOff + wave * 256), 4, 0, 0);
      return;
    }
    const int c = i - kS;
    if (c < kALoads) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra[c], (lds_ptr_t)(s + (c * NW + wave) * 1024), 16, aoff, tt * 128, 0, 0);
    } else if (BITS == 8) {
      const int b = c - kALoads;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb[b], (lds_ptr_t)(s + kABytes + (b * NW + wave) * 1024), 16, boff, tt * 1024, 0, 0);
    } else {
      // tile 2T - 1 brings the first part of raw tile T, tile 2T the second (past the end: the last one again)
      const int b = c - kALoads + (odd ? 0 : kBOdd), T = (t + 1) / 2, src = t0 / 2 + (2 * T < nt ? T : nt / 2 - 1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb[b], (lds_ptr_t)(smem + kRawOff + (T & 1) * kBBytes + (b * NW + wave) * 1024), 16, boff,
                                               src * 1024, 0, 0);
    }
  };

  f32x4 acc[TM][TN];
  float unit[TN], mrun[TN];  // G != 0: what one unit of this lane's sums of strip c is worth; the largest scale so far
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int c = 0; c < TN; ++c) acc[a][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < TN; ++c) unit[c] = mrun[c] = 0.0f;
  u32x4 af[TM], raw[TN], bf[2][TN];
  const int arow = (wm * TM * 16 + lr) * 128;
  const int apos = arow + ((kb ^ (lr & 7)) * 16);  // the second half's piece is four further on: XOR 64
  const int bpos = (BITS == 8 ? kABytes : 0) + wn * TN * 1024 + lane * 16;
  auto read_a = [&](const unsigned char* s, int h, int i) { af[i] = *reinterpret_cast<const u32x4*>(s + (h ? apos ^ 64 : apos) + i * 2048); };
  auto read_b = [&](const unsigned char* s, int c) { raw[c] = *reinterpret_cast<const u32x4*>(s + bpos + c * 1024); };
  // part d (of kDw) of B fragment c into set w: `step` is the 32-k step within the raw tile
  auto dequant = [&](int w, int step, int c, int d) {
    const uint32_t v = raw[c][step * kDw + d];
    if constexpr (BITS == 8) {
      // half a fragment: four codes, two dwords
      const uint32_t w2[2] = {v, v};
      const u32x4 o = DequantExact<DT, 8>::run(w2);
      bf[w][c][d * 2] = o.x;
      bf[w][c][d * 2 + 1] = o.y;
    } else {
      bf[w][c] = DequantExactFma<DT, 4>::run(&v);
    }
  };
  constexpr int kUnits = TN * kDw;
  float rho[TN];
  // A group starts: the new unit of every column and what the sums are multiplied by.  A scale of zero before any other (or
  // one in the denormal range, which the reciprocal does not take) leaves the unit what it is.  What was summed under a unit of
  // zero (groups whose scale is zero may hold any codes) counts for nothing; from a group to one of the same scale nothing
  // changes.
  auto new_units = [&](const unsigned char* s) {
#pragma unroll
    for (int c = 0; c < TN; ++c) {
      const float sv = to_f32<DT>(*reinterpret_cast<const uint16_t*>(s + kScaleOff + wave * 256 + (c * 16 + lr) * 2));
      mrun[c] = fmaxf(mrun[c], sv);
      const float u0 = fmaxf(sv, mrun[c] * 0x1p-64f);
      const float u = u0 < 0x1p-126f ? unit[c] : u0;
      rho[c] = unit[c] == 0.0f ? 0.0f : (u == unit[c] ? 1.0f : unit[c] * __builtin_amdgcn_rcpf(u));
      unit[c] = u;
    }
  };
  // the MFMAs of A block a on operand set w; rescale: a group starts here
  auto mfmas = [&](int w, int a, bool rescale) {
#pragma unroll
    for (int c = 0; c < TN; ++c) {
      if (G != 0 && rescale) {
        f32x4 t = acc[a][c];
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] *= rho[c];
        acc[a][c] = t;
      }
      acc[a][c] = mfma16<DT>(af[a], bf[w][c], acc[a][c]);
    }
  };

  // ---- start: tiles 0 and 1 and the part of tile 2 that the first half below does not bring
  constexpr int kFirst = (kLoadsEven * (kSpan - TM)) / kSpan;  // loads of a tile issued before its predecessor-but-two ends
  if (BITS == 4) {  // the first part of raw tile 0, which no tile before tile 0 brings
#pragma unroll
    for (int i = 0; i < kBOdd; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb[i], (lds_ptr_t)(smem + kRawOff + (i * NW + wave) * 1024), 16, boff, t0 / 2 * 1024, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < kLoadsEven; ++i) issue1(0, 0, false, i);
#pragma unroll
  for (int i = 0; i < kLoadsOdd; ++i) issue1(1, 1, true, i);
#pragma unroll
  for (int i = 0; i < kFirst; ++i) issue1(2, 2, false, i);
  wait_vmcnt<kLoadsOdd + kFirst>();  // tile 0 has landed
  __builtin_amdgcn_s_barrier();
  if (STAMP) st_loop0 = st_prev = __builtin_readcyclecounter();
#pragma unroll
  for (int c = 0; c < TN; ++c) read_b(BITS == 8 ? smem : smem + kRawOff, c);
#pragma unroll
  for (int a = 0; a < TM; ++a) read_a(smem, 0, a);
  if (G != 0) new_units(smem);
#pragma unroll
  for (int u = 0; u < kUnits; ++u) dequant(0, 0, u / kDw, u % kDw);

  int st = 0;
  // One k tile; ODD: its parity where that matters (int4's raw tiles, groups of 128).
  auto tile = [&](auto odd_tile, int t) {
    constexpr bool kOdd = decltype(odd_tile)::value;
    // first step of this tile and of the next one within their raw tiles
    constexpr int q0 = BITS == 4 && kOdd ? 2 : 0, q1 = BITS == 4 && !kOdd ? 2 : 0;
    constexpr bool kNewB = BITS == 8 || kOdd;            // the next tile starts a raw tile
    constexpr bool kGroup = G == 64 || (G == 128 && !kOdd);  // this tile starts a group
    constexpr bool kNextGroup = G == 64 || (G == 128 && kOdd);
    constexpr int kN2 = kOdd ? kLoadsOdd : kLoadsEven;   // loads of tile t + 2 (parity of t) ...
    constexpr int kN3 = kOdd ? kLoadsEven : kLoadsOdd;   // ... and of tile t + 3
    const unsigned char* s = smem + st * kStage;
    const int st_n = st == 2 ? 0 : st + 1, st_p = st == 0 ? 2 : st - 1;
    const unsigned char* n = smem + st_n * kStage;
    // The loads of tile t + 3 are spread over the slots from barrier t to barrier t + 1: positions
    // 0 .. TM - B0 - 1 behind the barrier, the others in the next tile's first half and before its barrier
    auto share = [&](int pos, int loads) { return loads * pos / kSpan; };
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      mfmas(0, i, kGroup);
      read_a(s, 1, i);
#pragma unroll
      for (int u = kUnits * i / TM; u < kUnits * (i + 1) / TM; ++u) dequant(1, q0 + 1, u / kDw, u % kDw);
#pragma unroll
      for (int l = share(TM + i, kN2); l < share(i + 1 == TM ? kSpan : TM + i + 1, kN2); ++l) issue1(t + 2, st_p, kOdd, l);
    }
#pragma unroll
    for (int i = 0; i < B0; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      mfmas(1, i, false);
    }
    __builtin_amdgcn_sched_barrier(0);
    unsigned long long st_a = 0, st_b = 0;
    if (STAMP) {
      __builtin_amdgcn_s_waitcnt(0x0070 | 0xF | (3 << 14));  // lgkmcnt(0)
      st_a = __builtin_readcyclecounter();
      wait_vmcnt<kN2>();
      st_b = __builtin_readcyclecounter();
    } else {
      // lgkmcnt(0): this wavefront needs nothing more of the tile; tile t + 1 has landed
      __builtin_amdgcn_s_waitcnt(0x0070 | (kN2 & 0xF) | ((kN2 >> 4) << 14));
    }
    __builtin_amdgcn_s_barrier();
    if (STAMP) {
      const unsigned long long st_c = __builtin_readcyclecounter();
      st_work += st_a - st_prev;
      st_loads += st_b - st_a;
      st_bar += st_c - st_b;
      st_prev = st_c;
    }
    __builtin_amdgcn_sched_barrier(0);
    const unsigned char* nb = BITS == 8 ? n : smem + kRawOff + (((t + 1) / 2) & 1) * kBBytes;
    if (kNewB) {
#pragma unroll
      for (int c = 0; c < TN; ++c) read_b(nb, c);
    }
    constexpr int S = TM - B0;  // slots behind the barrier; reads and conversions from the second one on
#pragma unroll
    for (int i = 0; i < S; ++i) {
      mfmas(1, B0 + i, false);
      if (kNextGroup && i == (S > 1 ? 1 : 0)) new_units(n);
#pragma unroll
      for (int a = (S > 1 && i > 0 ? TM * (i - 1) / (S - 1) : 0); a < (S > 1 ? TM * i / (S - 1) : TM); ++a) read_a(n, 0, a);
#pragma unroll
      for (int u = (S > 1 && i > 0 ? kUnits * (i - 1) / (S - 1) : 0); u < (S > 1 ? kUnits * i / (S - 1) : kUnits); ++u) dequant(0, q1, u / kDw, u % kDw);
#pragma unroll
      for (int l = share(i * TM / S, kN3); l < share((i + 1) * TM / S, kN3); ++l) issue1(t + 3, st, !kOdd, l);
      __builtin_amdgcn_sched_barrier(0);
    }
    st = st_n;
  };
  if constexpr (BITS == 4 || G == 128) {
    for (int t = 0; t < nt; t += 2) {
      tile(std::false_type(), t);
      if (BITS == 4 || t + 1 < nt) tile(std::true_type(), t + 1);  // int4: K is made of whole raw tiles
    }
  } else {
    for (int t = 0; t < nt; ++t) tile(std::false_type(), t);
  }
  __builtin_amdgcn_s_waitcnt(0x0070);
  __builtin_amdgcn_s_barrier();  // the spare loads are done and every wavefront has stopped reading
  unsigned long long st_loop1 = 0;
  if (STAMP) st_loop1 = __builtin_readcyclecounter();

  // ---- epilogue: scale, bias, cast; 32-row slabs leave through LDS as 16-byte stores ----
  // accumulator element r of lane l is row 4 * (l / 16) + r, column l % 16 of its block
  int etid = threadIdx.x;
  asm volatile("" : "+v"(etid));  // nothing of the epilogue's addresses is kept in registers during the loop
  const int el = etid & 63, ec = el & 15, er = (el >> 4) * 4;
  const uint16_t* bias = p.bias;
  if (EXPERTS && bias != nullptr) bias += static_cast<int64_t>(at.expert) * N;
  const int n_hi = p.strip_hi * kStripCols;
  float sc[TN], bv[TN];
#pragma unroll
  for (int c = 0; c < TN; ++c) {
    int n = strip_col(c) + ec;
    const int last = SWI && c >= TN / 2 ? N : n_hi;
    n = n < last ? n : last - 1;
    sc[c] = G != 0 ? unit[c] : to_f32<DT>(scale[n]);
    bv[c] = bias != nullptr && p.nsplit == 1 ? to_f32<DT>(bias[n]) : 0.0f;
  }
  constexpr int kOut = SWI ? TN / 2 : TN;  // strips a wavefront writes
  const int col0 = (strip0 + wn * kOut) * kStripCols;
  const int row_w = m0 + wm * TM * 16;     // first row of this wavefront
  constexpr int kSlabRows = TM >= 2 ? 32 : 16, kPer = kSlabRows / 16;
  if constexpr (SWI == 0 && !EXPERTS) if (p.out_f32 || p.nsplit > 1) {
    // fp32 results (verification mode) or the sums of this run of k tiles, kept compact: a row is as long as the
    // launch has columns
    const int64_t ld = p.nsplit > 1 ? static_cast<int64_t>(p.strip_hi - p.strip_lo) * kStripCols : N;
    const int nc0 = p.nsplit > 1 ? p.strip_lo * kStripCols : 0;
    float* outf = static_cast<float*>(p.out) + (p.nsplit > 1 ? static_cast<int64_t>(split) * M * ld : 0);
    constexpr int kRow = TN * 16 + 4, kPieces = kSlabRows * TN * 4;
    static_assert(NW * kSlabRows * kRow * 4 <= kLds, "slabs must fit in the stages");
    float* slab = reinterpret_cast<float*>(smem) + wave * kSlabRows * kRow;
#pragma unroll
    for (int a = 0; a < TM; a += kPer) {
#pragma unroll
      for (int h = 0; h < kPer; ++h)
#pragma unroll
        for (int c = 0; c < TN; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = acc[a + h][c][r] * sc[c] + bv[c];
            slab[(h * 16 + er + r) * kRow + c * 16 + ec] = p.nsplit > 1 ? v : act_apply(v, p.act);
          }
      __builtin_amdgcn_wave_barrier();
      for (int q = el; q < kPieces; q += 64) {
        const int r = q / (TN * 4), cc = q % (TN * 4), m = row_w + a * 16 + r, n = col0 + cc * 4;
        const f32x4 v = *reinterpret_cast<const f32x4*>(&slab[r * kRow + cc * 4]);
        if (m < M && n < n_hi) *reinterpret_cast<f32x4*>(outf + static_cast<int64_t>(m) * ld + (n - nc0)) = v;
      }
      __builtin_amdgcn_wave_barrier();
    }
    return;
  }
  uint16_t* out = static_cast<uint16_t*>(p.out);
  constexpr int kRow = kOut * 16 + 8, kPieces = kSlabRows * kOut * 2;
  static_assert(NW * kSlabRows * kRow * 2 <= kLds, "slabs must fit in the stages");
  uint16_t* slab = reinterpret_cast<uint16_t*>(smem) + wave * kSlabRows * kRow;
  const int ld = SWI ? N / 2 : N;
#pragma unroll
  for (int a = 0; a < TM; a += kPer) {
#pragma unroll
    for (int h = 0; h < kPer; ++h)
#pragma unroll
      for (int c = 0; c < kOut; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = acc[a + h][c][r] * sc[c] + bv[c];
          if (SWI) {
            float u = acc[a + h][TN / 2 + c][r] * sc[TN / 2 + c] + bv[TN / 2 + c];
            if (SWI == 2) {  // as if fc1 had been written out in T and read back
              v = to_f32<DT>(cast_out<DT>(v));
              u = to_f32<DT>(cast_out<DT>(u));
            }
            v = act_swiglu(v, u);
          } else {
            v = act_apply(v, p.act);
          }
          slab[(h * 16 + er + r) * kRow + c * 16 + ec] = cast_out<DT>(v);
        }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = el; q < kPieces; q += 64) {
      const int r = q / (kOut * 2), cc = q % (kOut * 2), m = row_w + a * 16 + r, n = col0 + cc * 8;
      const u32x4 v = *reinterpret_cast<const u32x4*>(&slab[r * kRow + cc * 8]);
      if (m < M && n < n_hi) *reinterpret_cast<u32x4*>(out + static_cast<int64_t>(m) * ld + n) = v;
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (STAMP && el == 0 && p.stamps != nullptr) {
    unsigned long long* o = p.stamps + (static_cast<size_t>(blockIdx.x) * NW + wave) * 8;
    const unsigned long long st_end = __builtin_readcyclecounter();
    o[0] = st_loop0 - st_entry;   // entry to the first tile's barrier
    o[1] = st_work;               // between the barriers: MFMAs and everything issued among them
    o[2] = st_loads;              // waiting for this wavefront's own tile loads
    o[3] = st_bar;                // waiting for the other wavefronts
    o[4] = st_loop1 - st_prev;    // the last tile's tail and the closing barrier
    o[5] = st_end - st_loop1;     // epilogue
    o[6] = st_end - st_entry;     // all of it
    o[7] = static_cast<unsigned long long>(nt);
  }
#endif
}

// gemm_dma_kernel_tall: group-wise scales on 256 x 256 tiles.  Eight wavefronts of 256 rows x 32 columns each,
// v_mfma_f32_32x32x16, sums in units of the current group's scale as above.
//
// What bounds it.  Rescaling costs a VALU instruction per accumulator register and group, 4 per 32x32x16 MFMA with
// groups of 64; with the dequantiser's 1.75 (3.5 with two rows of wavefronts) and the MFMA's own two slots that is 33
// cycles of issue per 32-cycle MFMA.  The 16x16x32 form would need 42 for the same work, which is why this kernel keeps
// the larger one although it burns more power per product.
//
// Order.  What matters is that the VALU work is even over the tile.  The B fragments of a k tile (four 16-k slices of one
// 32-column block) stay in registers for the whole tile and A streams past them: blocks in pairs, eight MFMAs a pair,
// and behind every MFMA the A fragment it has used is read again for the next pair, and four accumulators of the next
// pair are rescaled.  The next tile's codes and scales are read at the start of a tile and converted during its second and
// third pair, so they travel one tile ahead of the activations: group g of loads brings the activations of tile g and
// the codes and scales of tile g + 1.  The barrier that frees the tile's stage sits after the second MFMA of the last
// pair, when all of the tile's reads have long arrived.
//
// A rows are XORed with (row % 8) ^ (row / 8 % 2): the phases of ds_read_b128 over the 32 rows of a fragment.
//
// bf16: K = 4096, N = 22016, M = 2048 int8 g64 395 -> 343 us against 32x32x16 tiles of two by four wavefronts; M = 8192,
// N = 4096 int8 g128 (fp16) 244 -> 227, int4 g128 247 -> 224 (1.23 PFLOP/s), int4 g64 278 -> 238; swiglu, M = 1237, N =
// 22016 int8 g64 255 -> 221, int4 g128 241 -> 204.  On gemm_dma_kernel_wide's 256-row tiles: int8 g64 M = 2048, N = 8192
// 128 against 126, swiglu 237 against 220, int4 spills.
template <int BITS>
constexpr size_t tall_lds_bytes() {
  return 3 * (32768 + (BITS == 8 ? 16384 : 0) + 2048) + (BITS == 4 ? 32768 : 0);
}

template <int DT, int BITS, int G, int SWI>
__global__ __launch_bounds__(512) void gemm_dma_kernel_tall(const DmaParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NW = 8, BM = 256, kStrips = 16;
  constexpr int kABytes = 32768, kBBytes = 16384;
  constexpr int kScaleOff = kABytes + (BITS == 8 ? kBBytes : 0);
  constexpr int kStage = kScaleOff + 2048;
  constexpr int kRawOff = 3 * kStage;
  constexpr int kLds = static_cast<int>(tall_lds_bytes<BITS>());
  constexpr int kB = BITS == 8 ? 2 : 1;  // B loads of a group
  constexpr int kLoads = 1 + 4 + kB;
  constexpr int kFirst = 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, sp = (lane >> 4) & 1, b = lane >> 5, r32 = lane & 31;
  int bx, by, split;
  place_of_block(p, &bx, &by, &split);
  const int K = p.K, N = p.N, M = p.M, m0 = by * BM;
  const int strip0 = p.strip_lo + bx * (SWI ? kStrips / 2 : kStrips);
  const int up_strips = N / 2 / kStripCols;
  const int t0 = split * p.tiles_per_split;
  const int nt = (K / 64 - t0) < p.tiles_per_split ? (K / 64 - t0) : p.tiles_per_split;
  const int rows = M - m0 < BM ? M - m0 : BM;
  const int sbytes = static_cast<int>(strip_bytes(K, BITS));
  const int left = p.strip_hi - strip0, own = SWI ? kStrips / 2 : kStrips, strips = left < own ? left : own;
  __amdgpu_buffer_rsrc_t ra[4], rb[2];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int r0 = (c * NW + wave) * 8, nr = rows - r0 > 8 ? 8 : (rows > r0 ? rows - r0 : 0);
    ra[c] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.x + static_cast<int64_t>(nr > 0 ? m0 + r0 : m0) * K), 0, nr * K * 2, 0x00020000);
  }
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int L = c * NW + wave, st = SWI ? L / 2 : L;
    const int64_t first = st < strips ? strip0 + st + (SWI && L % 2 ? up_strips : 0) : 0;
    rb[c] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.codes + first * sbytes), 0, st < strips ? sbytes : 0, 0x00020000);
  }
  const uint32_t aoff = static_cast<uint32_t>((lane / 8) * K + ((lane ^ (lane >> 3) ^ (wave & 1)) & 7) * 8) * 2, boff = lane * 16;
  // column of position v (0 .. 31) of this wavefront
  auto column = [&](int v) {
    return SWI ? (strip0 + wave) * kStripCols + v % 16 + (v >= 16 ? N / 2 : 0) : (strip0 + wave * 2) * kStripCols + v;
  };
  int scol;
  {
    const int v = 2 * lane < 32 ? 2 * lane : 0;
    scol = column(v);
    const int last = SWI ? (v < 16 ? N / 2 : N) : p.strip_hi * kStripCols;
    scol = scol < last ? scol : last - 2;
  }
  constexpr int kGShift = G == 128 ? 7 : 6;
  auto clampt = [&](int t) { return t0 + (t < nt ? t : nt - 1); };
  auto issue_s = [&](int t, int st) {
    const int64_t row = static_cast<int64_t>(clampt(t)) * 64 >> kGShift;
    __builtin_amdgcn_global_load_lds(p.scale + row * N + scol, (lds_ptr_t)(smem + st * kStage + kScaleOff + wave * 256), 4, 0, 0);
  };
  auto issue_b = [&](int t, int st, int c) {  // int8: tile t's codes
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rb[c], (lds_ptr_t)(smem + st * kStage + kABytes + (c * NW + wave) * 1024), 16, boff, clampt(t) * 1024, 0, 0);
  };
  auto issue_raw = [&](int T, int c) {  // int4: half c of raw tile T
    const int src = t0 / 2 + (2 * T < nt ? T : nt / 2 - 1);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rb[c], (lds_ptr_t)(smem + kRawOff + (T & 1) * kBBytes + (c * NW + wave) * 1024), 16, boff, src * 1024, 0, 0);
  };
  // load i of group g: scales and codes of tile g + 1, activations of tile g; st: g % 3, odd: parity of g
  auto issue = [&](int g, int st, bool odd, int i) {
    const int st1 = st == 2 ? 0 : st + 1;
    if (i == 0) issue_s(g + 1, st1);
    else if (i <= 4)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra[i - 1], (lds_ptr_t)(smem + st * kStage + ((i - 1) * NW + wave) * 1024), 16, aoff, clampt(g) * 128, 0, 0);
    else if (BITS == 8) issue_b(g + 1, st1, i - 5);
    else issue_raw(odd ? (g + 1) / 2 : (g + 2) / 2, odd ? 1 : 0);
  };

  f32x16 acc[8];
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[a][r] = 0.0f;
  float unit = 0.0f, mrun = 0.0f, rho = 0.0f;
  uint32_t sraw = 0;
  u32x4 af[8], raw[2], bf[2][4];
  const int apos = r32 * 128 + ((b ^ a_swizzle<8>(lane & 15)) * 16);
  const int bpos = (BITS == 8 ? kABytes : 0) + (wave * 2 + sp) * 1024 + (j + 16 * b) * 16;
  auto read_a = [&](const unsigned char* s, int blk, int i) {  // i = which * 4 + q
    af[i] = *reinterpret_cast<const u32x4*>(s + (apos ^ ((i & 3) * 32)) + blk * 4096);
  };
  auto read_b = [&](const unsigned char* s) {
#pragma unroll
    for (int h = 0; h < 2; ++h) raw[h] = *reinterpret_cast<const u32x4*>(s + bpos + h * 512);
  };
  // piece d of B fragment q of a tile (int8: halves of two) into set w; base: the tile's first 32-k step in its raw tile
  auto dequant = [&](int w, int base, int q, int d) {
    if constexpr (BITS == 8) {
      const uint32_t v = raw[q & 1][(q >> 1) * 2 + d];
      const uint32_t w2[2] = {v, v};
      const u32x4 o = DequantExact<DT, 8>::run(w2);
      bf[w][q][d * 2] = o.x;
      bf[w][q][d * 2 + 1] = o.y;
    } else {
      const uint32_t v = raw[q & 1][base + (q >> 1)];
      bf[w][q] = DequantExactFma<DT, 4>::run(&v);
    }
  };
  auto new_unit = [&]() {
    const float sv = to_f32<DT>(static_cast<uint16_t>(sraw));
    mrun = fmaxf(mrun, sv);
    const float u0 = fmaxf(sv, mrun * 0x1p-64f);
    const float u = u0 < 0x1p-126f ? unit : u0;
    const float ratio = unit * __builtin_amdgcn_rcpf(u);
    rho = unit == 0.0f ? 0.0f : (u == unit ? 1.0f : ratio);
    unit = u;
  };
  auto read_s = [&](int st) { sraw = *reinterpret_cast<const uint16_t*>(smem + st * kStage + kScaleOff + wave * 256 + r32 * 2); };

  // ---- start: codes and scales of tile 0, groups 0 and 1
  issue_s(0, 0);
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    if (BITS == 8) issue_b(0, 0, c);
    else issue_raw(0, c);
  }
#pragma unroll
  for (int i = 0; i < kLoads; ++i) issue(0, 0, false, i);
#pragma unroll
  for (int i = 0; i < kLoads; ++i) issue(1, 1, true, i);
  wait_vmcnt<kLoads>();
  __builtin_amdgcn_s_barrier();
  read_b(BITS == 8 ? smem : smem + kRawOff);
  read_s(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) read_a(smem, i >> 2, i);
  new_unit();
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int d = 0; d < (BITS == 8 ? 2 : 1); ++d) dequant(0, 0, q, d);
  // group 2 brings the scales and codes of tile 3 to where tile 0's lie: they have been read by everybody first
  __builtin_amdgcn_s_waitcnt(0x0070 | 0xF | (3 << 14));  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < kFirst; ++i) issue(2, 2, false, i);
  int st = 0;
  auto tile = [&](auto odd_tile, int t) {
    constexpr bool kOdd = decltype(odd_tile)::value;
    constexpr int w = kOdd ? 1 : 0;
    constexpr bool kGroup = G == 64 || !kOdd, kNextGroup = G == 64 || kOdd;
    constexpr bool kNewB = BITS == 8 || kOdd;
    constexpr int base = BITS == 4 && !kOdd ? 2 : 0;  // of tile t + 1
    const int st_n = st == 2 ? 0 : st + 1, st_p = st == 0 ? 2 : st - 1;
    const unsigned char* s = smem + st * kStage;
    const unsigned char* n = smem + st_n * kStage;
#pragma unroll
    for (int pr = 0; pr < 4; ++pr) {
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const int q = m >> 1, which = m & 1, a = 2 * pr + which;
        acc[a] = mfma32<DT>(af[which * 4 + q], bf[w][q], acc[a]);
        if (pr < 3) read_a(s, 2 * (pr + 1) + which, which * 4 + q);
        if (pr == 0 && m == 0) {
          if (kNextGroup) read_s(st_n);
          if (kNewB) read_b(BITS == 8 ? n : smem + kRawOff + (((t + 1) / 2) & 1) * kBBytes);
        }
        if (pr == 3 && m == 1) {
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_waitcnt(0x0070 | kLoads);  // this tile's reads are done, group t + 1 has landed
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
          read_a(n, 0, 0);
          read_a(n, 1, 4);
        }
        if (pr == 3 && m > 1) read_a(n, which, which * 4 + q);
        // rescale the next pair's sums, four elements per MFMA
        if (pr < 3 ? kGroup : kNextGroup) {
          const int na = 2 * ((pr + 1) & 3) + (m >> 2);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[na][(m & 3) * 4 + e] *= rho;
        }
        if (kNextGroup && pr == 2 && m == 7) new_unit();
        if (pr == 1 || pr == 2) {
          const int k = (pr - 1) * 8 + m;  // 0 .. 15
          if (BITS == 8 && k % 2 == 1) dequant(w ^ 1, base, k / 4, (k / 2) % 2);
          if (BITS == 4 && k % 4 == 1) dequant(w ^ 1, base, k / 4, 0);
        }
        if (pr == 3 && (m == 3 || m == 6)) issue(t + 3, st, !kOdd, m / 3 - 1);
        if (pr < 3 && m % 4 == 3 && kFirst + pr * 2 + m / 4 < kLoads) issue(t + 2, st_p, kOdd, kFirst + pr * 2 + m / 4);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    st = st_n;
  };
  for (int t = 0; t < nt; t += 2) {
    tile(std::false_type(), t);
    if (BITS == 4 || t + 1 < nt) tile(std::true_type(), t + 1);
  }
  __builtin_amdgcn_s_waitcnt(0x0070);
  __builtin_amdgcn_s_barrier();

  // ---- epilogue
  int etid = threadIdx.x;
  asm volatile("" : "+v"(etid));
  const int el = etid & 63, ec = el & 31, eb = el >> 5;
  const int n_hi = p.strip_hi * kStripCols;
  float sc, bv;
  {
    int n = column(ec);
    const int last = SWI ? (ec < 16 ? N / 2 : N) : n_hi;
    n = n < last ? n : last - 1;
    sc = unit;
    bv = p.bias != nullptr && p.nsplit == 1 ? to_f32<DT>(p.bias[n]) : 0.0f;
  }
  if (SWI == 0 && (p.out_f32 || p.nsplit > 1)) {
    const int64_t ld = p.nsplit > 1 ? static_cast<int64_t>(p.strip_hi - p.strip_lo) * kStripCols : N;
    const int nc0 = p.nsplit > 1 ? p.strip_lo * kStripCols : 0;
    float* outf = static_cast<float*>(p.out) + (p.nsplit > 1 ? static_cast<int64_t>(split) * M * ld : 0);
    constexpr int kRow = 256 + 4;
    static_assert(128 * kRow * 4 <= kLds, "half the tile must fit in the stages");
    float* slab = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      __syncthreads();
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float v = acc[hf * 4 + a][r] * sc + bv;
          slab[(a * 32 + 8 * (r / 4) + 4 * eb + r % 4) * kRow + wave * 32 + ec] = p.nsplit > 1 ? v : act_apply(v, p.act);
        }
      __syncthreads();
      for (int q = etid; q < 128 * 64; q += 512) {
        const int r = q / 64, cc = q % 64, m = m0 + hf * 128 + r, n = strip0 * kStripCols + cc * 4;
        const f32x4 v = *reinterpret_cast<const f32x4*>(&slab[r * kRow + cc * 4]);
        if (m < M && n < n_hi) *reinterpret_cast<f32x4*>(outf + static_cast<int64_t>(m) * ld + (n - nc0)) = v;
      }
    }
    return;
  }
  uint16_t* out = static_cast<uint16_t*>(p.out);
  constexpr int kCols = SWI ? 128 : 256, kRow = kCols + 8;
  static_assert(256 * kRow * 2 <= kLds, "the tile must fit in the stages");
  uint16_t* slab = reinterpret_cast<uint16_t*>(smem);
#pragma unroll
  for (int a = 0; a < 8; ++a) {
    if constexpr (SWI != 0) {
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float u0 = acc[a][r] * sc + bv, u1 = acc[a][r + 1] * sc + bv;
        // lanes of a gate strip take row r, those of an up strip row r + 1, gate and up of it side by side
        const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(u0), __float_as_uint(u1), false, false);
        float g = __uint_as_float(sw[0]), u = __uint_as_float(sw[1]);
        slab[(a * 32 + 8 * (r / 4) + 4 * eb + r % 4 + ((el >> 4) & 1)) * kRow + wave * 16 + (el & 15)] = cast_out<DT>(act_swiglu(g, u));
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        slab[(a * 32 + 8 * (r / 4) + 4 * eb + r % 4) * kRow + wave * 32 + ec] = cast_out<DT>(act_apply(acc[a][r] * sc + bv, p.act));
    }
  }
  __syncthreads();
  const int ld = SWI ? N / 2 : N;
  for (int q = etid; q < 256 * kCols / 8; q += 512) {
    const int r = q / (kCols / 8), cc = q % (kCols / 8), m = m0 + r, n = strip0 * kStripCols + cc * 8;
    const u32x4 v = *reinterpret_cast<const u32x4*>(&slab[r * kRow + cc * 8]);
    if (m < M && n < n_hi) *reinterpret_cast<u32x4*>(out + static_cast<int64_t>(m) * ld + n) = v;
  }
#endif
}

template <int DT, int BITS, int G, int WM, int WN, int TM, int TN, int SWI, bool STAMP, bool SHORT_RUNS>
__global__ __launch_bounds__(512) void gemm_dma_kernel_wide(const DmaParams p) {
  int bx, by, split;
  if (SHORT_RUNS) place_in_short_run(p, &bx, &by, &split);
  else place_of_block(p, &bx, &by, &split);
  wide_tile<DT, BITS, G, WM, WN, TM, TN, SWI, STAMP, false>(p, TilePlace{bx, 0, by * WM * TM * 16, 0}, split);
}

// The grouped GEMM over experts with many rows each: row tiles of up to four
// 64-row units (256 rows), as many units as the tile has rows for.  A tile's
// MFMAs, activation loads and operand reads follow its height, so an expert
// whose row count is no multiple of the tile pays for 64-row padding only.
// Workgroups are handed out expert by expert, column tile by column tile, all
// row tiles of the expert next to each other, and that sequence is cut into
// eight equal pieces, one per XCD: an expert's row tiles meet its weights in
// one L2 while they are there, and the XCDs stay evenly loaded however the
// rows are spread over the experts.  WM, TN: wavefronts side by side on 256
// columns (1, 2), or two rows of them on 128 columns (2, 2), where one row would
// read an A fragment per MFMA.
template <int DT, int BITS, int WM, int SWI>
__global__ __launch_bounds__(512) void gemm_experts_kernel(const DmaParams p) {
  const MoeTile* table = reinterpret_cast<const MoeTile*>(p.moe_table);
  const int total = table[0].expert * p.nbx;  // the header holds the number of row tiles
  constexpr int kXcd = 8, WN = 8 / WM;
  const int per = (total + kXcd - 1) / kXcd;
  const int slot = blockIdx.x / kXcd, pos = (blockIdx.x % kXcd) * per + slot;
  if (slot >= per || pos >= total) return;
  // position / column tiles = some row tile of the position's expert
  const MoeTile any = table[1 + pos / p.nbx];
  const int w = pos - any.first * p.nbx;
  const MoeTile t = table[1 + any.first + w % any.count];
  const TilePlace at{w / any.count, t.expert, t.row0, t.rows};
  const int units = (t.rows + 63) / 64;
  if (units >= 4) wide_tile<DT, BITS, 0, WM, WN, 16 / WM, 2, SWI, false, true>(p, at, 0);
  else if (units == 3) wide_tile<DT, BITS, 0, WM, WN, 12 / WM, 2, SWI, false, true>(p, at, 0);
  else if (units == 2) wide_tile<DT, BITS, 0, WM, WN, 8 / WM, 2, SWI, false, true>(p, at, 0);
  else wide_tile<DT, BITS, 0, WM, WN, 4 / WM, 2, SWI, false, true>(p, at, 0);
}

// Eight wavefronts side by side, TM 16-row blocks x 32 columns each.
template <int DT, int BITS, int G, int TM, int SWI, bool STAMP = false, bool SHORT_RUNS = false>
void launch(const DmaParams& p, hipStream_t stream) {
  constexpr size_t lds = wide_lds_bytes<BITS, G, 1, 8, TM, 2>();
  auto kern = gemm_dma_kernel_wide<DT, BITS, G, 1, 8, TM, 2, SWI, STAMP, SHORT_RUNS>;
  static std::atomic<uint32_t> configured{0};  // per instantiation
  allow_lds(reinterpret_cast<const void*>(kern), lds, configured);
  kern<<<dim3(static_cast<unsigned>(p.nbx * p.nby * p.nsplit)), dim3(512), lds, stream>>>(p);
}

template <int DT, int BITS, int G, int SWI>
void launch_tall(const DmaParams& p, hipStream_t stream) {
  constexpr size_t lds = tall_lds_bytes<BITS>();
  auto kern = gemm_dma_kernel_tall<DT, BITS, G, SWI>;
  static std::atomic<uint32_t> configured{0};  // per instantiation
  allow_lds(reinterpret_cast<const void*>(kern), lds, configured);
  kern<<<dim3(static_cast<unsigned>(p.nbx * p.nby * p.nsplit)), dim3(512), lds, stream>>>(p);
}

template <int DT, int BITS, int G>
void launch_tile(const DmaParams& p, WideTile tile, int swi, hipStream_t stream) {
  if (tile == WideTile::kHalf) {
    if (swi) launch<DT, BITS, G, 8, 1>(p, stream);
    else if (p.nsplit > 1 && p.tiles_per_split < kShortRun) launch<DT, BITS, G, 8, 0, false, true>(p, stream);
    else launch<DT, BITS, G, 8, 0>(p, stream);
    return;
  }
  if constexpr (G == 0) {
    if (swi) launch<DT, BITS, G, 16, 1>(p, stream);
    else launch<DT, BITS, G, 16, 0>(p, stream);
  } else {
    if (swi) launch_tall<DT, BITS, G, 1>(p, stream);
    else launch_tall<DT, BITS, G, 0>(p, stream);
  }
}

template <int DT, int BITS, int WM, int SWI>
void launch_experts_on(const DmaParams& p, unsigned blocks, hipStream_t stream) {
  constexpr size_t lds = wide_lds_bytes<BITS, 0, WM, 8 / WM, 16 / WM, 2>();
  auto kern = gemm_experts_kernel<DT, BITS, WM, SWI>;
  static std::atomic<uint32_t> configured{0};  // per instantiation
  allow_lds(reinterpret_cast<const void*>(kern), lds, configured);
  kern<<<dim3(blocks), dim3(512), lds, stream>>>(p);
}

template <int DT, int BITS>
void launch_experts(const DmaParams& p, bool narrow, bool swiglu, unsigned blocks, hipStream_t stream) {
  if (swiglu) launch_experts_on<DT, BITS, 1, 2>(p, blocks, stream);
  else if (narrow) launch_experts_on<DT, BITS, 2, 0>(p, blocks, stream);
  else launch_experts_on<DT, BITS, 1, 0>(p, blocks, stream);
}

template <int DT, int BITS>
void launch_group(const DmaParams& p, int group, WideTile tile, int swi, hipStream_t stream) {
  if (group == 0) launch_tile<DT, BITS, 0>(p, tile, swi, stream);
  else if (group == 64) launch_tile<DT, BITS, 64>(p, tile, swi, stream);
  else launch_tile<DT, BITS, 128>(p, tile, swi, stream);
}

}  // namespace

#if defined(WOL_GEMM_F16_UNIT)
#define WOL_WIDE_LAUNCH launch_wide_f16
#define WOL_EXPERTS_LAUNCH launch_experts_f16
#else
#define WOL_WIDE_LAUNCH launch_wide_bf16
#define WOL_EXPERTS_LAUNCH launch_experts_bf16
#endif
void WOL_WIDE_LAUNCH(const DmaParams& p, int bits, int group, WideTile tile, int swi, hipStream_t stream) {
  if (bits == 8) launch_group<WOL_GEMM_DTYPE, 8>(p, group, tile, swi, stream);
  else launch_group<WOL_GEMM_DTYPE, 4>(p, group, tile, swi, stream);
}
void WOL_EXPERTS_LAUNCH(const DmaParams& p, int bits, bool narrow, bool swiglu, unsigned blocks, hipStream_t stream) {
  if (bits == 8) launch_experts<WOL_GEMM_DTYPE, 8>(p, narrow, swiglu, blocks, stream);
  else launch_experts<WOL_GEMM_DTYPE, 4>(p, narrow, swiglu, blocks, stream);
}

#if !defined(WOL_GEMM_F16_UNIT)

// The prefill GEMM's 256 x 256 int8 per-channel bf16 launch with cycle stamps
// (M and N multiples of 256, K a multiple of 64 and at least 192): out [M, N]
// bf16, stamps [(M / 256) * (N / 256)][8 wavefronts][8] counts.
int launch_prefill_phases(const void* x, const void* codes, const void* scale, int64_t M, int64_t K, int64_t N,
                          void* out, unsigned long long* stamps, hipStream_t stream) {
  DmaParams p{};
  p.x = static_cast<const uint16_t*>(x);
  p.codes = static_cast<const uint8_t*>(codes);
  p.scale = static_cast<const uint16_t*>(scale);
  p.out = out;
  p.M = static_cast<int>(M); p.K = static_cast<int>(K); p.N = static_cast<int>(N);
  p.strip_hi = static_cast<int>(N / kStripCols);
  p.nbx = static_cast<int>(N / 256);
  p.nby = static_cast<int>(M / 256);
  p.tiles_per_split = static_cast<int>(K / 64);
  p.nsplit = 1;
  p.act = WOL_ACT_NONE;
  p.stamps = stamps;
  launch<WOL_DTYPE_BF16, 8, 0, 16, 0, true>(p, stream);
  return check_launch();
}

#endif  // !WOL_GEMM_F16_UNIT

}  // namespace wol
