// Streaming weight-only GEMV for gfx950: the INT4 and INT8 products whose K is
// too long for the K-slice kernels' registers, or whose rows are too few to
// give every compute unit several waves of the pair kernel.
//
// A workgroup owns one tile of up to 16 weight rows; its 8 waves split K into
// contiguous slices, so that even with one tile per compute unit (n = 4096) 8
// waves' loads are in flight there.  A wave walks its slice in steps of 128
// bytes of each weight row (256 K of INT4, 128 K of INT8):
//   * weights: two full-line loads per step with the DPP hand-over of the pair
//     kernel, DW steps ahead in registers;
//   * activations: by load-to-LDS into the wave's own stages, as many steps
//     ahead (vector-memory waits retire in issue order, so the shallower ring
//     would bound the deeper one).  No registers hold loads in flight and no
//     barrier is needed; the 16-byte pieces of a row are XOR-ed with the row on
//     the source side, so the MFMA-layout reads have no bank conflicts;
//   * scales and offsets of the tile: contiguous in memory, staged once by
//     load-to-LDS.  (A per-lane load of one group of 16 rows touches 16 lines
//     and takes as long as four weight loads: 64 against 17 clocks.)
// After one barrier the slices' partials are added in wave order
// (deterministic) and stored.  INT4 products are those of the pair kernel
// (64 + q, fp32 partial sums), INT8 codes exact.
//
// Bound: the weight stream plus a start of about 5 us (launch, first misses),
// and from m = 8 on the activations: every workgroup reads all of x, m * k * 2
// bytes at 64 bytes per clock.  Measured (us; pair kernel -> this one):
// INT4 4096 x 14336, groups of 128: m = 1 25.4 -> 10.9, m = 8 51.1 -> 12.2,
// m = 32 152 -> 23; INT8 3584 x 18944: m = 1 38.7 -> 14.1, m = 32 134 -> 33.
#include <algorithm>
#include <type_traits>

#include "gemv_common.hpp"
#include "gemv_stream.hpp"

namespace rlk {
namespace {

// INT4 with groups of whole 128-K chunks; INT4 with groups of 32 or 64; INT8.
enum StreamKind { kInt4, kInt4Small, kInt8 };

struct StreamArgs {
  W4Args a;
  int mode;
  int nsteps;        // steps of 128 row bytes
  int nchunks;       // 128-K chunks
  uint32_t gmul;     // chunk -> group: (c * gmul) >> 21 (kInt4)
  int gsh;           // kInt4Small: log2(group_size / 32)
  int rows_wg;       // weight rows of a workgroup (at most 16)
  int so_bytes;      // LDS bytes of the staged scales (whole KiB); as many for the offsets
  int so_dma;        // the workgroup's scales and offsets are 16-byte aligned, the arrays whole dwords
  int so_shift, so_mask;  // piece p of row r is staged at p ^ ((r >> so_shift) & so_mask)
  float inv_pieces;  // 1 / 16-byte pieces of a row (1 where nothing is swizzled)
};

#define RLK_LDS __attribute__((address_space(3)))

// R: activation rows staged (m <= R); DW: steps in flight.
template <StreamKind KIND, int R, int DW>
struct StreamGeo {
  static constexpr int kMT = R > 16 ? 2 : 1;
  static constexpr int kCPS = KIND == kInt8 ? 1 : 2;  // x chunks per step
  // a step's x: [chunk][row] of 256 bytes, or (R = 2) [row] of both chunks,
  // brought by load-to-LDS instructions of 1 KiB each
  static constexpr bool kPair = R == 2;
  static_assert(!kPair || KIND != kInt8, "a pair of chunks is an INT4 step");
  static constexpr int kStage = R * kCPS * 256;
  static constexpr int kXI = kStage / 1024;
  // vector-memory instructions issued after a step's x when it is needed, and after the scales
  static constexpr int kAhead = 2 + (DW - 1) * (kXI + 2);
  static constexpr int kPrologue = DW * (kXI + 2);
  static_assert(kPrologue < 64, "vmcnt holds 6 bits");
  // two workgroups per compute unit where the LDS has room
  static constexpr int kWavesPerSimd = R > 16 ? 2 : 4;
  static constexpr int kXBytes = std::max(DW * kStage, kMT * 1024);  // a wave's stages; its partials reuse them
};

template <StreamKind KIND, int R, int DW>
__global__ __launch_bounds__(64 * kMaxWaves, (StreamGeo<KIND, R, DW>::kWavesPerSimd)) void gemv_stream_kernel(StreamArgs s) {
  using G = StreamGeo<KIND, R, DW>;
  constexpr int MT = G::kMT, CPS = G::kCPS;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const W4Args& a = s.a;
  const int nw = blockDim.x / 64, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, qd = lane >> 4;
  const bool low = (lane & 8) == 0;
  const int row0 = blockIdx.x * s.rows_wg;
  const int row_end = min(row0 + s.rows_wg, a.n);
  if (row0 >= row_end) return;  // workgroup-uniform
  const int kb = KIND == kInt8 ? a.k : a.k / 2;  // bytes per weight row
  uint8_t* xst = lds + wave * G::kXBytes;  // this wave's x stages
  uint8_t* so_lds = lds + nw * G::kXBytes;  // scales [16 rows][groups], then (so_bytes on) offsets
  // this wave's steps
  const int s0 = wave * s.nsteps / nw, s1 = (wave + 1) * s.nsteps / nw;
  const int nst = s1 - s0;

  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(a.w), 0, static_cast<int>(static_cast<uint32_t>(a.n) * static_cast<uint32_t>(kb)),
      kBufferFlags);
  const __amdgpu_buffer_rsrc_t none = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.w), 0, 0, kBufferFlags);
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.x), 0, a.m * a.k * 2, kBufferFlags);

  // full-line loads: instruction 0 covers rows 0..7 of the tile, 1 rows 8..15;
  // rows past the workgroup's re-read its last one
  const int pc0 = (low ? qd : 4 + qd) * 16, pc1 = (low ? 4 + qd : qd) * 16;
  const int vo0 = min(row0 + (low ? r16 : r16 - 8), row_end - 1) * kb + pc0;
  const int vo1 = min(row0 + (low ? r16 + 8 : r16), row_end - 1) * kb + pc1;
  u32x4 ring[DW][2];
  auto fetch = [&](int slot, int st) {  // steps past the slice read nothing
    const __amdgpu_buffer_rsrc_t res = st < s1 ? wres : none;
    ring[slot][0] = __builtin_amdgcn_raw_buffer_load_b128(res, vo0, st * 128, kNtLoad);
    ring[slot][1] = __builtin_amdgcn_raw_buffer_load_b128(res, vo1, st * 128, kNtLoad);
  };
  // the x of step st -> stage; 16-byte piece p of a row r lands at piece
  // p ^ r; rows past m read zeros, chunks past K the last chunk (not used)
  auto stage_x = [&](int slot, int st) {
#pragma unroll
    for (int i = 0; i < G::kXI; ++i) {
      RLK_LDS void* dst = (RLK_LDS void*)(xst + slot * G::kStage + i * 1024);
      if constexpr (G::kPair) {
        const int c = min(2 * st + ((lane >> 4) & 1), s.nchunks - 1);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, dst, 16, (lane >> 5) * a.k * 2 + c * 256 + (lane & 15) * 16,
                                                 0, 0, 0);
      } else {
        const int h = 4 * i / R, r4 = 4 * i % R;  // chunk and first row of this instruction
        const int r = lane >> 4, sw = ((lane & 15) ^ r) << 4;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, dst, 16, (r4 + r) * a.k * 2 + (sw ^ ((r4 & 15) << 4)),
                                                 min(st * CPS + h, s.nchunks - 1) * 256, 0, 0);
      }
    }
  };

  // this lane's row's bias and (INT8) scale, ahead of use
  // (raw and without a branch: converting or merging them here would wait for them)
  const int my_row = min(row0 + r16, a.n - 1);
  const uint16_t my_bias = (a.bias != nullptr ? a.bias : a.x)[a.bias != nullptr ? my_row : 0];
  uint16_t my_scale = 0;
  if constexpr (KIND == kInt8) my_scale = a.scales[my_row];
  // scales and offsets of the workgroup's rows, contiguous in memory, by
  // load-to-LDS: read per lane, 16 rows' scales of a group touch 16 lines and
  // cost four weight loads' time
  if constexpr (KIND != kInt8) {
    const uint32_t start = static_cast<uint32_t>(row0) * a.groups * 2;
    if (s.so_dma) {
      const int sbytes = a.n * a.groups * 2;
      const __amdgpu_buffer_rsrc_t sres =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.scales), 0, sbytes, kBufferFlags);
      const __amdgpu_buffer_rsrc_t ores =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.offsets), 0, sbytes, kBufferFlags);
      for (int i = wave * 1024; i < 2 * s.so_bytes; i += nw * 1024) {
        const bool off = i >= s.so_bytes;
        const int at = ((off ? i - s.so_bytes : i) >> 4) + lane;  // 16-byte piece of the rows
        const int r = quot(at, s.inv_pieces);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(off ? ores : sres, (RLK_LDS void*)(so_lds + i), 16,
                                                 start + ((at ^ ((r >> s.so_shift) & s.so_mask)) << 4), 0, 0, 0);
      }
    } else {  // unaligned arrays
      const int total = (row_end - row0) * a.groups;
      for (int i = tid; i < total; i += 64 * nw) {
        reinterpret_cast<uint16_t*>(so_lds)[i] = a.scales[start / 2 + i];
        reinterpret_cast<uint16_t*>(so_lds + s.so_bytes)[i] = a.offsets[start / 2 + i];
      }
    }
  }
  // the order of the steady state: a step's x, then its weights
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int d = 0; d < DW; ++d) {
    stage_x(d, s0 + d);
    __builtin_amdgcn_sched_barrier(0);  // the waits count on this order
    fetch(d, s0 + d);
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (KIND != kInt8) {
    // every wave's scales have landed (a bare barrier: __syncthreads() would
    // drain the ring)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(G::kPrologue) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }

  f32x4 acc[2][MT];  // of the chunk's parity (INT8: of the MFMA step's)
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[h][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t magic = opaque(0x54005400u);  // 64.0 in both halves
  constexpr f16x8 kOnes = {1, 1, 1, 1, 1, 1, 1, 1};

  // A operand of MFMA step j: the 16-byte piece of x that matches the codes
  int xrd[MT];  // row offset and swizzle of this lane's activation rows
  int xsz[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = min(16 * mt + r16, R - 1);
    xrd[mt] = r * (G::kPair ? 512 : 256);
    xsz[mt] = G::kPair ? 0 : (r & 15) << 4;
  }
  constexpr int kChunk = G::kPair ? 256 : R * 256;  // from a step's chunk 0 to its chunk 1
  auto xfrag = [&](const uint8_t* xs, int mt, int j) {
    const int piece = KIND == kInt8 ? 8 * (j >> 1) + 2 * qd + (j & 1) : KIND == kInt4 ? 4 * qd + j : 4 * j + qd;
    const u32x4 v = *reinterpret_cast<const u32x4*>(xs + xrd[mt] + ((piece << 4) ^ xsz[mt]));
    return __builtin_bit_cast(f16x8, v);
  };
  auto f16f = [](uint32_t v) { return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(v))); };

  // LDS byte of group g (uniform) of this lane's row: 16-byte pieces swizzled
  // as staged
  const int so_row = r16 * a.groups * 2, so_swz = ((r16 >> s.so_shift) & s.so_mask) << 4;
  auto so_at = [&](int g) { return so_row + ((g << 1 & ~15) ^ so_swz) + (g << 1 & 15); };
  // one step: NC chunks of x (INT4: 2, or 1 at the end of an odd K) against the
  // codes; the chunks' products are independent chains
  auto compute = [&](int st, const f16x8 (&xv)[CPS][MT][4], const u32x4 (&w)[2], auto nc) {
    constexpr int NC = decltype(nc)::value;
    constexpr f32x4 kZero = {0.f, 0.f, 0.f, 0.f};
    if constexpr (KIND == kInt8) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x4 c = w[j >> 1];
        const f16x8 q = int8x8_to_f16((j & 1) ? u32x2{c.z, c.w} : u32x2{c.x, c.y});
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[j & 1][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[0][mt][j], q, acc[j & 1][mt], 0, 0, 0);
      }
    } else if constexpr (KIND == kInt4) {
      f32x4 d[NC][MT], xsum[NC][MT];
#pragma unroll
      for (int h = 0; h < NC; ++h)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) d[h][mt] = xsum[h][mt] = kZero;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int h = 0; h < NC; ++h) {
          const f16x8 q = codes_f16_natural(w[h][j], magic);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            xsum[h][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[h][mt][j], kOnes, xsum[h][mt], 0, 0, 0);
            d[h][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[h][mt][j], q, d[h][mt], 0, 0, 0);
          }
        }
#pragma unroll
      for (int h = 0; h < NC; ++h) {
        const int at = so_at(static_cast<int>((static_cast<uint32_t>(st * CPS + h) * s.gmul) >> 21));
        const float sc = f16f(*reinterpret_cast<const uint16_t*>(so_lds + at));
        const float of = fmaf(-kCodeBias, sc, f16f(*reinterpret_cast<const uint16_t*>(so_lds + s.so_bytes + at)));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[h][mt][e] = fmaf(of, xsum[h][mt][e], fmaf(sc, d[h][mt][e], acc[h][mt][e]));
      }
    } else {
      // groups of 32 or 64: MFMA step j must stay inside one, so the code
      // words are transposed over the four 16-lane rows (two v_permlane32_swap
      // and two v_permlane16_swap per 4 words): word j of lane (qd, r16) is
      // then K 32 j + 8 qd .. + 7
#pragma unroll
      for (int h = 0; h < NC; ++h) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __builtin_bit_cast(float, static_cast<uint32_t>(w[h][j]));
        swap_rows_pair<true>(v[0], v[2]);
        swap_rows_pair<true>(v[1], v[3]);
        swap_rows_pair<false>(v[0], v[1]);
        swap_rows_pair<false>(v[2], v[3]);
        // the chunk's 4 (groups of 32) or 2 scales and offsets lie in one 16-byte piece
        const int at = so_at((st * CPS + h) * 4 >> s.gsh);
        u32x2 sp, op;
        if (s.gsh == 0) {
          sp = *reinterpret_cast<const u32x2*>(so_lds + at);
          op = *reinterpret_cast<const u32x2*>(so_lds + s.so_bytes + at);
        } else {
          const uint32_t s2 = *reinterpret_cast<const uint32_t*>(so_lds + at);
          const uint32_t o2 = *reinterpret_cast<const uint32_t*>(so_lds + s.so_bytes + at);
          sp = u32x2{(s2 & 0xFFFFu) * 0x10001u, (s2 >> 16) * 0x10001u};
          op = u32x2{(o2 & 0xFFFFu) * 0x10001u, (o2 >> 16) * 0x10001u};
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float sc = f16f(sp[j >> 1] >> (16 * (j & 1)));
          const float of = fmaf(-kCodeBias, sc, f16f(op[j >> 1] >> (16 * (j & 1))));
          const f16x8 q = codes_f16_natural(__builtin_bit_cast(uint32_t, v[j]), magic);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const f32x4 xsum = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[h][mt][j], kOnes, kZero, 0, 0, 0);
            const f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[h][mt][j], q, kZero, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[h][mt][e] = fmaf(of, xsum[e], fmaf(sc, d[e], acc[h][mt][e]));
          }
        }
      }
    }
  };

  for (int i = 0; i < nst; i += DW) {
#pragma unroll
    for (int d = 0; d < DW; ++d) {
      const int st = s0 + i + d;
      if (st < s1) {  // wave-uniform
        // the step's x, requested from LDS in one batch while its weights may
        // still be on their way (read where each product needs it, every
        // product waited for an LDS round trip)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(G::kAhead) : "memory");
        f16x8 xv[CPS][MT][4];
#pragma unroll
        for (int h = 0; h < CPS; ++h)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int j = 0; j < 4; ++j) xv[h][mt][j] = xfrag(xst + d * G::kStage + h * kChunk, mt, j);
        __builtin_amdgcn_sched_barrier(0);
        // the hand-over of the pair kernel: w[0] is chunk 0 (INT8: codes 16 qd
        // of the first 64), w[1] chunk 1 (the second 64) of the lane's own row
        u32x4 w[2];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          w[0][e] = low ? ring[d][0][e] : ring[d][1][e];
          w[1][e] = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(
              static_cast<int>(low ? ring[d][1][e] : ring[d][0][e]), 0x128, 0xF, 0xF, false));  // row_ror:8
        }
        if (CPS == 1 || 2 * st + 1 < s.nchunks) compute(st, xv, w, std::integral_constant<int, CPS>{});
        else compute(st, xv, w, std::integral_constant<int, 1>{});
      }
      __builtin_amdgcn_sched_barrier(0);  // the stage's reads are done: its refill may land
      stage_x(d, st + DW);
      __builtin_amdgcn_sched_barrier(0);  // the waits count on this order
      fetch(d, st + DW);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // partials into the wave's own stages, once every load-to-LDS in flight has landed there
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  f32x4* part = reinterpret_cast<f32x4*>(xst);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) part[mt * kWave + lane] = acc[0][mt] + acc[1][mt];
  __syncthreads();
  if (wave >= MT) return;
  // the slices, added in wave order; wave mt takes activation tile mt
  const f32x4* from = reinterpret_cast<const f32x4*>(lds) + wave * kWave + lane;
  f32x4 v[kMaxWaves];
#pragma unroll
  for (int w = 0; w < kMaxWaves; ++w) v[w] = from[min(w, nw - 1) * (G::kXBytes / 16)];
  f32x4 sum = v[0];
#pragma unroll
  for (int w = 1; w < kMaxWaves; ++w)
    if (w < nw) sum += v[w];
  const float b = a.bias != nullptr ? f16f(my_bias) : 0.f;
  if constexpr (KIND == kInt8) sum *= f16f(my_scale);
  const int row = row0 + r16 < row_end ? row0 + r16 : a.n;  // rows past the workgroup's are not stored
  const int m0 = 16 * wave + 4 * qd;
  if (s.mode == kModeF16) store_tile<kModeF16>(a, sum, b, m0, row, r16);
  else if (s.mode == kModeF32) store_tile<kModeF32>(a, sum, b, m0, row, r16);
  else store_tile<kModeSwiglu>(a, sum, b, m0, row, r16);
}

template <StreamKind KIND, int R, int DW>
int launch(StreamArgs s, hipStream_t stream) {
  using G = StreamGeo<KIND, R, DW>;
  const W4Args& a = s.a;
  // (wave mt stores activation tile mt: at least MT waves)
  const int nw = std::max(G::kMT, std::min(kMaxWaves, s.nsteps));
  // The rows spread evenly over whole rounds of compute units, 16 at most per
  // workgroup and an even number (gate/up pairs): 3584 rows are 256
  // workgroups of 14, not 224 of 16 (k = 18944 INT8, m = 1: 14.1 against 16.0 us).
  const int cus = compute_units();
  const int rounds = (a.n + 16 * cus - 1) / (16 * cus);
  s.rows_wg = (a.n + rounds * cus - 1) / (rounds * cus);
  s.rows_wg += s.rows_wg & 1;
  size_t lds = static_cast<size_t>(nw) * G::kXBytes;
  if (KIND != kInt8) {
    const int row_bytes = a.groups * 2;
    s.so_bytes = (16 * row_bytes + 1023) / 1024 * 1024;
    // load-to-LDS of the scales needs whole 16-byte pieces from the workgroup's first row on
    s.so_dma = s.so_dma && s.rows_wg * row_bytes % 16 == 0;
    s.inv_pieces = 1.0f;
    if (s.so_dma && row_bytes % 16 == 0) {
      // The 16 lanes of a read take one group of 16 rows: rows whose pitch
      // falls on the same 256-byte span (64 banks) get their pieces XOR-ed with
      // different values, inside the power of two that divides a row's pieces
      // (groups of 32 at k = 4096: 16 rows in one bank otherwise).
      const int pieces = row_bytes / 16;
      int span = pieces % 16, w = 1;  // w: rows until the pitch repeats
      while (span * w % 16 != 0) w *= 2;
      s.so_shift = __builtin_ctz(w);
      s.so_mask = std::min(pieces & -pieces, 16) - 1;
      s.inv_pieces = 1.0f / static_cast<float>(pieces);
    }
    lds += 2 * static_cast<size_t>(s.so_bytes);
  }
  if (lds > kLdsBudget) return kNoFit;
  auto kernel = gemv_stream_kernel<KIND, R, DW>;
  if (lds > 64 * 1024) {
    const hipError_t e = grant_dynamic_lds(reinterpret_cast<const void*>(kernel), kLdsBudget);
    if (e != hipSuccess)
      return fail(RLK_EUNSUPPORTED, "weight-only GEMV: %zu bytes of LDS refused (%s)", lds, hipGetErrorString(e));
  }
  kernel<<<(a.n + s.rows_wg - 1) / s.rows_wg, 64 * nw, lds, stream>>>(s);
  return RLK_OK;
}

// Steps in flight: as many as the x stages allow in half the LDS (m > 16: in
// all of it).
template <StreamKind KIND>
int launch_rows(const StreamArgs& s, hipStream_t stream) {
  const int m = s.a.m;
  constexpr bool k8 = KIND == kInt8;
  if constexpr (!k8)
    if (m <= 2) return launch<KIND, 2, 4>(s, stream);
  // Groups of 32 and 64 at one step per wave: 4 steps in flight are 3 too many
  // (groups of 32, m = 4, k = 2048, slab / streaming time at n = 28672 and 65536:
  // 0.97 and 0.94 with 4 rows staged and 4 steps in flight).
  if (m <= 4 && !(KIND == kInt4Small && s.nsteps <= kMaxWaves)) return launch<KIND, 4, 4>(s, stream);
  if (m <= 8) return launch<KIND, 8, k8 ? 4 : 2>(s, stream);
  if (m <= 16) return launch<KIND, 16, 2>(s, stream);
  return launch<KIND, 32, k8 ? 2 : 1>(s, stream);
}

}  // namespace

int launch_gemv_stream(const StreamCall& c, hipStream_t stream) {
  const bool int8 = c.offsets == nullptr;
  const int kb = int8 ? c.k : c.k / 2;
  if (c.k % 128 != 0 || static_cast<uint64_t>(c.n) * kb > kMaxBufferBytes) return kNoFit;
  StreamArgs s{};
  W4Args& a = s.a;
  a.x = c.x;
  a.w = c.w;
  a.scales = c.scales;
  a.offsets = c.offsets;
  a.bias = c.bias;
  a.y = c.y;
  a.m = c.m;
  a.n = c.n;
  a.k = c.k;
  a.group_size = c.group_size;
  a.y_ld = c.y_ld;
  s.mode = c.mode;
  s.nchunks = c.k / 128;
  if (int8) {
    s.nsteps = s.nchunks;
    return launch_rows<kInt8>(s, stream);
  }
  a.groups = c.k / c.group_size;
  // (the buffers' bounds are checked by dwords: an odd number of scales, as
  // odd n and odd groups give, would have the last one half outside)
  s.so_dma = (reinterpret_cast<uintptr_t>(a.scales) | reinterpret_cast<uintptr_t>(a.offsets)) % 16 == 0 &&
             static_cast<int64_t>(a.n) * a.groups % 2 == 0;
  s.nsteps = (s.nchunks + 1) / 2;
  if (c.group_size % 128 == 0) {
    const int gq = c.group_size / 128;
    if (gq > 1024) return kNoFit;  // (c * gmul) >> 21 is exact for chunks < 2^11, gq <= 2^10
    s.gmul = ((1u << 21) + gq - 1) / gq;
    return launch_rows<kInt4>(s, stream);
  }
  if (c.group_size != 32 && c.group_size != 64) return kNoFit;
  s.gsh = c.group_size == 64;
  return launch_rows<kInt4Small>(s, stream);
}

}  // namespace rlk
