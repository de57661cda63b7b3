// Block-scaled MXFP8 GEMM for gfx950, stream form: the kernel of the small and middle sizes
// (see mxfp8_gemm.hip for the operand formats, the instruction and the large-problem kernel).
//
// What bounds it: a workgroup's K steps in sequence. The weight comes from memory once per launch,
// so a step must not wait for its own loads: a ring of kSlots K steps in LDS keeps two or three
// steps (about 100 KB per CU) in flight while one is computed. A step of a 128 x 256 tile is 32
// scaled MFMAs per wave (1024 cycles) and measured 1430 cycles, 0.70 us at the 2.0 GHz clock the
// power limit leaves (0.57 us without its DMAs, 0.50 us also without its scale reads); a first
// form with double-buffered fragments read at the head of each step took 0.82 us.
//   step s:  the first A groups' MFMAs; wait for step s + 1's tiles (the later steps' loads stay in
//            flight) and barrier: every wave holds its fragments of step s in registers, so slot
//            s % kSlots is free; the other MFMAs, with step s + kSlots's DMAs into that slot spread
//            over them and each fragment register read again for step s + 1 after its last use.
// Measured against the kernels it replaced at these sizes (us per launch, weights not in cache; M x
// N x K): 77 x 5120 x 5120 48 -> 31, 512 x 5120 x 5120 49 -> 31, 960 x 5120 x 5120 68 -> 43,
// 960 x 5120 x 13824 159 -> 98, 2048 x 1536 x 6144 67 -> 29; below 3072 rows of the large kernel
// 3330 x 5376 x 14336 296 -> 222.
#include "mxfp8_gemm.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace vdn {
namespace {

// f(integral_constant<int, 0>) .. f(integral_constant<int, n - 1>)
template <int... I, typename F>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for(std::make_integer_sequence<int, N>{}, f);
}

typedef __attribute__((address_space(3))) void lds_void_t;

constexpr int kSM = 128;        // tile rows

// Empty asm statements: the MFMA that produces g (the shift that produces x) is issued before
// whatever follows. Without them the pure MFMA calls sink past the cursor's branches to the end
// of the loop, and their fragments are copied for it.
__device__ __forceinline__ void pinv(uint32_t& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin1(const f32x4& g) { asm volatile("" ::"a"(g) : "memory"); }

// A raw buffer's base and size: loads past its end return zero. (Kept as plain values and made
// a resource where it is used, so that it stays in scalar registers across the K loop.)
struct Span {
  const uint8_t* base;
  int bytes;
};
__device__ __forceinline__ Span make_span(const uint8_t* base, int64_t bytes) {
  return Span{base, static_cast<int>(bytes < 0x7fffffffll ? bytes : 0x7fffffffll)};
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t span_rsrc(const Span& s) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(s.base), 0, s.bytes, 0x00020000);
}

// LDS DMA: lane l's kBytes at soffset + voffset + kOffset land at LDS byte base + kOffset + kBytes l.
// The compiler sets M0 to the wave's LDS base and counts these loads on vmcnt only.
template <int kBytes, int kOffset>
__device__ __forceinline__ void dma_to_lds(const Span& src, uint8_t* base, uint32_t voffset, int soffset) {
#ifdef __HIP_DEVICE_COMPILE__   // a dependent builtin call: the host pass has none to find
  if constexpr (kBytes == 16)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(span_rsrc(src), (lds_void_t*)base, 16, voffset, soffset, kOffset, 0);
  else
    __builtin_amdgcn_raw_ptr_buffer_load_lds(span_rsrc(src), (lds_void_t*)base, 4, voffset, soffset, kOffset, 0);
#endif
}

// Tile t of the launch, rows fastest within bands of 8 tile rows: the tiles an XCD runs
// together (consecutive t) share W panels, and a band's A panels stay in its L2.
__device__ __forceinline__ void stream_tile(int t, int tiles_m, int tiles_n, int& tm, int& tn) {
  constexpr int kBand = 8;
  const int in_band = kBand * tiles_n;
  const int first = (t / in_band) * kBand;
  const int rows = min(tiles_m - first, kBand);
  tm = first + (t % in_band) % rows;
  tn = (t % in_band) / rows;
}

// How a launch's tiles fall on its workgroups: workgroup w runs tiles w, w + grid, .. A tile's K
// steps stay in one workgroup, in one sequence, as in the other GEMM kernels: shared between
// workgroups, their partial sums would round differently, and a row's output would depend on how
// many rows the call has and on the tile it falls in.
struct StreamPlan {
  int bn, tiles_m, tiles_n;
  int grid;    // workgroups
  int rounds;  // tiles of every workgroup; the first `rest` have one more
  int rest;
};

// ---- epilogue of a wave's 16-row group: kTN blocks of 16 columns, lane l holding rows l % 16,
// columns 16 nt + 4 (l / 16) .. + 3 of block nt ----
template <int BN, int kMode>
struct StreamEpilogue {
  static constexpr int kTN = 4;                       // a wave's 64 columns
  static constexpr int kStride = 144;                 // strip row: 64 bf16 + 16 pad bytes
  static constexpr int kWaveStrip = 16 * kStride;
  static constexpr int kStripBytes = 4 * kWaveStrip;  // also the SwiGLU hand-over: 2 x 4 KB

  const Epilogue& ep;
  uint8_t* strips;
  int lane, wave, wn, c_lo, frag_row;
  int64_t out_rows, n, mp;
  bool bad = false;
  u16x2 mag_max = {0, 0};
  int64_t m0 = 0, n0 = 0;
  float b8[8], g8[8];        // modes 0, 1: bias and gate of the lane's 8 columns
  float b4[kTN][4];          // modes 2, 3: bias of the lane's 16 columns
  u32x4 res[2];              // mode 1: the next group's residual

  __device__ __forceinline__ StreamEpilogue(const Epilogue& e, uint8_t* s, int lane_, int wave_, int wn_,
                                            int64_t rows, int64_t n_, int64_t mp_)
      : ep(e), strips(s), lane(lane_), wave(wave_), wn(wn_), c_lo(lane_ >> 4), frag_row(lane_ & 15),
        out_rows(rows), n(n_), mp(mp_) {}

  __device__ __forceinline__ int64_t store_col() const { return n0 + wn * 64 + (lane & 7) * 8; }

  __device__ __forceinline__ void load_residual(int row_in_tile) {
    if constexpr (kMode == 1) {
      const int64_t col = store_col();
#pragma unroll
      for (int pass = 0; pass < 2; ++pass) {
        const int64_t row = m0 + row_in_tile + pass * 8 + (lane >> 3);
        if (col < n && row < out_rows)
          res[pass] = *reinterpret_cast<const u32x4*>(ep.residual + row * ep.ld_res + col);
      }
    }
  }

  __device__ __forceinline__ void begin_tile(int64_t m, int64_t nn) {
    m0 = m;
    n0 = nn;
    if constexpr (kMode < 2) {
      const int64_t col = store_col();   // n is a multiple of 8 here: all 8 columns or none
      // a missing bias is -0 and a missing gate 1: both leave every value as it is
      u32x4 bw = {0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
      u32x4 gw = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
      if (ep.bias != nullptr && col < n) bw = *reinterpret_cast<const u32x4*>(ep.bias + col);
      if (ep.gate != nullptr && col < n) gw = *reinterpret_cast<const u32x4*>(ep.gate + col);
      unpack8(bw, b8);
      unpack8(gw, g8);
    } else {
      // SwiGLU's bias is interleaved like its weight, over the whole padded width
      const int64_t width = kMode == 3 ? 2 * ep.kp_out : n;
#pragma unroll
      for (int nt = 0; nt < kTN; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int64_t col = n0 + wn * 64 + nt * 16 + c_lo * 4 + v;
          b4[nt][v] = ep.bias != nullptr && col < width ? bf16_bits_to_f32(ep.bias[col]) : -0.f;
        }
    }
  }

  // Rows row_in_tile .. + 15. Mode 3 holds workgroup barriers: every wave calls it.
  __device__ __forceinline__ void group(int row_in_tile, const f32x4 (&a)[kTN], int next_row) {
    if constexpr (kMode < 2) {
      uint8_t* strip = strips + wave * kWaveStrip;
      u32x4 cur[2];
      if constexpr (kMode == 1) {
        cur[0] = res[0];
        cur[1] = res[1];
        if (next_row >= 0) load_residual(next_row);
      }
#pragma unroll
      for (int nt = 0; nt < kTN; ++nt) {
        u32x2 packed;
        packed[0] = pack_bf16x2(a[nt][0], a[nt][1]);
        packed[1] = pack_bf16x2(a[nt][2], a[nt][3]);
        *reinterpret_cast<u32x2*>(strip + frag_row * kStride + nt * 32 + c_lo * 8) = packed;
      }
      u32x4 yv[2];
#pragma unroll
      for (int pass = 0; pass < 2; ++pass)
        yv[pass] = *reinterpret_cast<const u32x4*>(strip + (pass * 8 + (lane >> 3)) * kStride + (lane & 7) * 16);
      const int64_t col = store_col();
      if (col < n) {
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
          const int64_t row = m0 + row_in_tile + pass * 8 + (lane >> 3);
          if (row >= out_rows) continue;
          float y[8], r[8];
          unpack8(yv[pass], y);
          if constexpr (kMode == 1) unpack8(cur[pass], r);
          u32x4 packed;
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            float v0 = y[e] + b8[e], v1 = y[e + 1] + b8[e + 1];
            if constexpr (kMode == 1) {
              round_bf16_pair(v0, v1);
              v0 *= g8[e];
              v1 *= g8[e + 1];
              round_bf16_pair(v0, v1);
              v0 += r[e];
              v1 += r[e + 1];
            }
            packed[e / 2] = pack_bf16x2(v0, v1);
          }
          *reinterpret_cast<u32x4*>(ep.out + row * ep.ldc + col) = packed;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            mag_max = __builtin_elementwise_max(mag_max, __builtin_bit_cast(u16x2, packed[i] & 0x7fff7fffu));
        }
      }
    } else {
      const int64_t row = m0 + row_in_tile + frag_row;
      float y[kTN][4];
#pragma unroll
      for (int nt = 0; nt < kTN; ++nt)
#pragma unroll
        for (int v = 0; v < 4; v += 2) {
          float p = a[nt][v], q = a[nt][v + 1];
          round_bf16_pair(p, q);
          p += b4[nt][v];
          q += b4[nt][v + 1];
          round_bf16_pair(p, q);
          y[nt][v] = p;
          y[nt][v + 1] = q;
        }
      // a lane's columns of the output: SwiGLU's a half (wn 0, 1) of 128-column block n0 / 256
      const int64_t ocol = kMode == 3 ? (n0 >> 1) + (wn & 1) * 64 : n0 + wn * 64;
      if constexpr (kMode == 3) {
        // the g waves (wn 2, 3) hand g * sigmoid(g) to the a waves of the same columns
        float* slot = reinterpret_cast<float*>(strips) + ((wn & 1) * 64 + lane) * 16;
        if (wn >= 2) {
#pragma unroll
          for (int nt = 0; nt < kTN; ++nt)
            *reinterpret_cast<f32x4*>(slot + nt * 4) = f32x4{swiglu_gate(y[nt][0]), swiglu_gate(y[nt][1]),
                                                             swiglu_gate(y[nt][2]), swiglu_gate(y[nt][3])};
        }
        __syncthreads();
        if (wn < 2) {
#pragma unroll
          for (int nt = 0; nt < kTN; ++nt) {
            const f32x4 gs = *reinterpret_cast<const f32x4*>(slot + nt * 4);
#pragma unroll
            for (int v = 0; v < 4; v += 2) {
              float p = y[nt][v] * gs[v], q = y[nt][v + 1] * gs[v + 1];
              round_bf16_pair(p, q);
              y[nt][v] = p;
              y[nt][v + 1] = q;
            }
          }
        }
        __syncthreads();   // the slots are free for the next group
        if (wn >= 2) return;
      } else if (ep.act == 1) {
#pragma unroll
        for (int nt = 0; nt < kTN; ++nt)
#pragma unroll
          for (int v = 0; v < 4; v += 2) {
            float p = gelu_tanh(y[nt][v]), q = gelu_tanh(y[nt][v + 1]);
            round_bf16_pair(p, q);
            y[nt][v] = p;
            y[nt][v + 1] = q;
          }
      }
#pragma unroll
      for (int nt = 0; nt < kTN; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const bool in = row < out_rows && ocol + nt * 16 + c_lo * 4 + v < n;
          bad = bad || (in && !(fabsf(y[nt][v]) < INFINITY));
          y[nt][v] = in ? y[nt][v] : 0.f;
        }
      // two 32-column MXFP8 blocks: their codes and two of the chunk's four scale bytes
      const bool store = (ocol >> 7) < (ep.kp_out >> 7) && row < mp;
      uint32_t scales = 0;
      uint32_t cw[kTN];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        float amax = 0.f;
#pragma unroll
        for (int nt = 2 * b; nt < 2 * b + 2; ++nt)
#pragma unroll
          for (int v = 0; v < 4; ++v) amax = fmaxf(amax, fabsf(y[nt][v]));
        amax = max_quad_rows(amax);
        float inv;
        const uint32_t byte = e8m0_from_amax(amax, &inv);
        scales |= byte << (8 * b);
        const float sf = e8m0_scale(byte);
#pragma unroll
        for (int nt = 2 * b; nt < 2 * b + 2; ++nt)
          cw[nt] = e4m3x4_scaled(y[nt][0], y[nt][1], y[nt][2], y[nt][3], sf);
      }
      // 4 x 4 transpose of code words over the row's lanes: lane c_lo gets the 16 contiguous
      // code bytes of columns 16 c_lo ..
      const auto a02 = __builtin_amdgcn_permlane32_swap(cw[0], cw[2], false, false);
      const auto a13 = __builtin_amdgcn_permlane32_swap(cw[1], cw[3], false, false);
      const auto b01 = __builtin_amdgcn_permlane16_swap(a02[0], a13[0], false, false);
      const auto b23 = __builtin_amdgcn_permlane16_swap(a02[1], a13[1], false, false);
      if (store) {
        *reinterpret_cast<u32x4*>(ep.q_out + row * ep.kp_out + ocol + 16 * c_lo) =
            u32x4{b01[0], b01[1], b23[0], b23[1]};
        if (c_lo == 0)
          *reinterpret_cast<uint16_t*>(ep.s_out + swizzled_scale_offset(row, ocol >> 5, ep.kp_out >> 7)) =
              static_cast<uint16_t>(scales);
      }
    }
  }

  __device__ __forceinline__ void finish() {
    const bool b = bad || mag_max[0] >= 0x7f80 || mag_max[1] >= 0x7f80;
    if (ep.nonfinite != nullptr && __ballot(b) != 0 && lane == 0) atomicOr(ep.nonfinite, 1u);
  }
};

template <int BN, int kSlots, int kMode>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
mxfp8_gemm_stream_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ As,
                         const uint8_t* __restrict__ W, const uint8_t* __restrict__ Ws, int64_t mp,
                         int64_t np, int64_t kp, Epilogue ep, int64_t out_rows, int64_t n,
                         StreamPlan plan) {
  constexpr int WGN = BN / 64, WGM = 4 / WGN;       // 4 waves: 1 x 4 (BN 256) or 2 x 2 (BN 128)
  constexpr int WM = kSM / WGM;
  constexpr int TM = WM / 16, TN = 4;
  constexpr int kSegA = kSM / 32, kSegW = BN / 32;  // 1 KB (8-row) DMA segments per wave and step
  constexpr int kRuns = 1 + BN / 128;               // 512-byte scale runs per step
  constexpr int kScaleOff = (kSM + BN) * kBK;
  constexpr int kStep = kScaleOff + kRuns * 512;
  constexpr int kDma = kSegA + kSegW + 2;           // DMAs per wave and step
  constexpr int kHead = TM / 4;                     // A groups before the step's barrier
  using Epi = StreamEpilogue<BN, kMode>;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kSlots * kStep + Epi::kStripBytes];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const int grid = gridDim.x;
  // workgroup ids are dealt to the 8 XCDs round robin: give each XCD a contiguous range
  int w;
  {
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, per = grid >> 3, rem = grid & 7;
    w = xcd < rem ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
  }
  const int nk = static_cast<int>(kp / kBK);
  const int64_t col_tiles = kp >> 7;
  const int tiles = plan.rounds + (w < plan.rest ? 1 : 0);   // of this workgroup

  // ---- DMA side ----
  // A wave loads rows kRowsA wave .. of the A tile and kRowsW wave .. of the W tile, 8 rows (1 KB)
  // per DMA: lane l writes 16 bytes at LDS offset 16 l, physical chunk l % 8 of row l / 8, so it
  // fetches chunk (l % 8) ^ ((row >> 1) & 7). A DMA's immediate offset moves its LDS address and
  // its global address alike, so four DMAs share one LDS base (M0) and their per-lane offsets,
  // constant over the kernel, hold the difference (8 rows are at least 1 KB apart); the K step
  // is the scalar offset. A DMA is then one instruction.
  constexpr int kRowsA = kSegA * 8, kRowsW = kSegW * 8;
  const uint32_t kpu = static_cast<uint32_t>(kp);
  uint32_t voff_a[kSegA], voff_w[kSegW];
  auto lane_offset = [&](int row) __attribute__((always_inline)) {
    const uint32_t r = row + (lane >> 3);
    return r * kpu + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
  };
#pragma unroll
  for (int i = 0; i < kSegA; ++i) voff_a[i] = lane_offset(wave * kRowsA + i * 8) - (i & 3) * 1024;
#pragma unroll
  for (int i = 0; i < kSegW; ++i) voff_w[i] = lane_offset(wave * kRowsW + i * 8) - (i & 3) * 1024;
  const uint32_t voff_s = lane * 4;
  struct Cursor {
    int i;          // tiles taken
    int ks, left;   // current tile: next K step and steps left (0: past the last tile)
  };
  Cursor d{0, 0, 0};
  Span d_a, d_w, d_s;
  // scale run of this wave: 0 the A block, 1 .. W's blocks (waves past the runs load one again)
  const int run = wave % kRuns;
  auto dma_tile = [&]() __attribute__((always_inline)) {
    d.ks = 0;
    if (d.i >= tiles) {   // past the last tile: empty resources, whose loads touch no memory
      d.left = 0;
      d_a = d_w = d_s = make_span(A, 0);
      return;
    }
    int tm, tn;
    stream_tile(w + d.i * grid, plan.tiles_m, plan.tiles_n, tm, tn);
    ++d.i;
    d.left = nk;
    const int64_t dm0 = static_cast<int64_t>(tm) * kSM, dn0 = static_cast<int64_t>(tn) * BN;
    d_a = make_span(A + dm0 * kp, (mp - dm0) * kp);
    d_w = make_span(W + dn0 * kp, (np - dn0) * kp);
    // a W block past the padded end repeats the last one (its codes are zero)
    const int64_t blk = run == 0 ? tm : min<int64_t>(dn0 / 128 + run - 1, np / 128 - 1);
    d_s = make_span((run == 0 ? As : Ws) + blk * col_tiles * 512, col_tiles * 512);
  };
  auto dma_advance = [&]() __attribute__((always_inline)) {
    if (d.left != 0) {
      ++d.ks;
      if (--d.left == 0) dma_tile();
    }
  };
  // DMA i (0 .. kDma - 1) of the cursor's step into slot `slot`
  auto dma_one = [&](int slot, auto i_tag) __attribute__((always_inline)) {
    constexpr int i = decltype(i_tag)::value;
    uint8_t* base = lds + slot * kStep;
    if constexpr (i < kSegA) {
      dma_to_lds<16, (i & 3) * 1024>(d_a, base + (wave * kSegA + (i & ~3)) * 1024, voff_a[i], d.ks * kBK);
    } else if constexpr (i < kSegA + kSegW) {
      constexpr int j = i - kSegA;
      dma_to_lds<16, (j & 3) * 1024>(d_w, base + kSM * kBK + (wave * kSegW + (j & ~3)) * 1024, voff_w[j],
                                     d.ks * kBK);
    } else {   // two 256-byte halves of the wave's run
      dma_to_lds<4, (i - kSegA - kSegW) * 256>(d_s, base + kScaleOff + run * 512, voff_s, d.ks * 512);
    }
  };

  // ---- consumer side ----
  const int frag_row = lane & 15, c_lo = lane >> 4;
  const int block_shift = 8 * c_lo;
  auto frag = [&](const uint8_t* base, int row) __attribute__((always_inline)) {
    const int sw = (row >> 1) & 7;
    const i32x4 lo = *reinterpret_cast<const i32x4*>(base + row * kBK + ((c_lo ^ sw) << 4));
    const i32x4 hi = *reinterpret_cast<const i32x4*>(base + row * kBK + (((c_lo + 4) ^ sw) << 4));
    return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  // Scale words of rows row0 + 16 t + frag_row (t < cnt) of a 128-row run: even t in the 16 bytes
  // at 16 frag_row, odd t in those at 16 (frag_row + 16), from dword row0 / 32 on.
  auto read_scales = [&](const uint8_t* r, int row0, int cnt, uint32_t* s) __attribute__((always_inline)) {
    const uint8_t* p = r + frag_row * 16 + (row0 >> 5) * 4;
    if (cnt == 8) {
      const u32x4 e = *reinterpret_cast<const u32x4*>(p), o = *reinterpret_cast<const u32x4*>(p + 256);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[2 * i] = e[i];
        s[2 * i + 1] = o[i];
      }
    } else {
      const u32x2 e = *reinterpret_cast<const u32x2*>(p), o = *reinterpret_cast<const u32x2*>(p + 256);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        s[2 * i] = e[i];
        s[2 * i + 1] = o[i];
      }
    }
  };
  const int w_row = wn * 64;
  uint32_t sa[TM], sb[TN], sa_n[TM], sb_n[TN];
  auto read_all_scales = [&](const uint8_t* buf) __attribute__((always_inline)) {
    read_scales(buf + kScaleOff, wm * WM, TM, sa_n);
    read_scales(buf + kScaleOff + 512 * (1 + (w_row >> 7)), w_row & 127, TN, sb_n);
  };
  auto a_frag = [&](const uint8_t* buf, int mt) __attribute__((always_inline)) {
    return frag(buf, wm * WM + mt * 16 + frag_row);
  };
  auto b_frag = [&](const uint8_t* buf, int nt) __attribute__((always_inline)) {
    return frag(buf + kSM * kBK, w_row + nt * 16 + frag_row);
  };

  f32x4 acc[TM][TN];
  i32x8 af[TM], bf[TN];
  int slot = 0;   // slot of the step being computed
  auto mfma = [&](int mt, int nt) __attribute__((always_inline)) {
    acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
        bf[nt], af[mt], acc[mt][nt], 0, 0, 0, static_cast<int>(sb[nt]), 0, static_cast<int>(sa[mt]));
  };
  // The DMAs that go out after MFMA k of a step, counted from its barrier: one DMA instruction
  // keeps the CU's address unit busy for 16 cycles, so a step's 4 waves x kDma of them take most
  // of its MFMA time and are spread over all of it.
  auto dmas_after = [&](int slot_, auto k_tag) __attribute__((always_inline)) {
    constexpr int k = decltype(k_tag)::value;
    constexpr int lo = (k * kDma + TM * TN - 1) / (TM * TN), hi = ((k + 1) * kDma + TM * TN - 1) / (TM * TN);
    static_assert(hi - lo <= 1, "DMAs per MFMA");
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (lo < hi) dma_one(slot_, std::integral_constant<int, lo>{});
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int kTail = (TM - kHead) * TN;   // MFMAs after the barrier

  // One K step. Each fragment register is read again, for step s + 1, right after its last MFMA of
  // step s, and the MFMAs are ordered so that every read has several MFMAs to arrive: columns
  // 0, 1 before columns 2, 3, so the B fragments read last are not the ones needed first.
  auto step = [&]() __attribute__((always_inline)) {
    const int nslot = slot + 1 == kSlots ? 0 : slot + 1;
    const int pslot = slot == 0 ? kSlots - 1 : slot - 1;
    const uint8_t* nxt = lds + nslot * kStep;
    constexpr int kTailRows = TM - kHead;
    // A groups 0 .. kHead - 1; the last DMAs of step s + kSlots - 1
    static_for<kHead * TN>([&](auto i_tag) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value, mt = i / TN, nt = i % TN;
      mfma(mt, nt);
      pin1(acc[mt][nt]);
      dmas_after(pslot, std::integral_constant<int, kTail + i>{});
    });
    dma_advance();
    // step s + 1 has landed (steps s + 2 .. s + kSlots - 1 stay in flight), and every wave holds
    // step s's fragments: its slot is free
    constexpr int kFlight = (kSlots - 2) * kDma;
    static_assert(kFlight < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((kFlight & 15) | ((kFlight >> 4) << 14) | (7 << 4) | (0 << 8));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_all_scales(nxt);
#pragma unroll
    for (int mt = 0; mt < kHead; ++mt) af[mt] = a_frag(nxt, mt);
    static_for<2>([&](auto h_tag) __attribute__((always_inline)) {
      constexpr int h = decltype(h_tag)::value;
      static_for<kTailRows * 2>([&](auto i_tag) __attribute__((always_inline)) {
        constexpr int i = decltype(i_tag)::value, mt = kHead + i / 2, nt = 2 * h + i % 2;
        mfma(mt, nt);
        pin1(acc[mt][nt]);
        dmas_after(slot, std::integral_constant<int, h * kTailRows * 2 + i>{});
        if constexpr (mt == TM - 1) {
          bf[nt] = b_frag(nxt, nt);
          sb[nt] = sb_n[nt] >> block_shift;
          pinv(sb[nt]);
        }
        if constexpr (h == 1 && i % 2 == 1) {
          af[mt] = a_frag(nxt, mt);
          sa[mt] = sa_n[mt] >> block_shift;
          pinv(sa[mt]);
          if constexpr (mt - kHead < kHead) {
            sa[mt - kHead] = sa_n[mt - kHead] >> block_shift;
            pinv(sa[mt - kHead]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    slot = nslot;
  };

  // prologue: kSlots - 1 steps in flight, and of the next the DMAs that would have gone out before
  // step 0 (the rest follow among step 0's first MFMAs)
  dma_tile();
#pragma unroll
  for (int s = 0; s + 1 < kSlots; ++s) {
    static_for<kDma>([&](auto i) __attribute__((always_inline)) { dma_one(s, i); });
    dma_advance();
  }
  static_for<(kTail * kDma + TM * TN - 1) / (TM * TN)>(
      [&](auto i) __attribute__((always_inline)) { dma_one(kSlots - 1, i); });

  Epi epi(ep, lds + kSlots * kStep, lane, wave, wn, out_rows, n, mp);
  for (int t = 0; t < tiles; ++t) {
    // the tile's first step has landed for every wave (and so have the last epilogue's stores)
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    {
      const uint8_t* buf = lds + slot * kStep;
      read_all_scales(buf);
#pragma unroll
      for (int nt = 0; nt < TN; ++nt) {
        bf[nt] = b_frag(buf, nt);
        sb[nt] = sb_n[nt] >> block_shift;
      }
#pragma unroll
      for (int mt = 0; mt < TM; ++mt) {
        af[mt] = a_frag(buf, mt);
        sa[mt] = sa_n[mt] >> block_shift;
      }
    }
#pragma unroll
    for (int mt = 0; mt < TM; ++mt)
#pragma unroll
      for (int nt = 0; nt < TN; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int left = nk; left > 0; --left) step();
    int tm, tn;
    stream_tile(w + t * grid, plan.tiles_m, plan.tiles_n, tm, tn);
    epi.begin_tile(static_cast<int64_t>(tm) * kSM, static_cast<int64_t>(tn) * BN);
    epi.load_residual(wm * WM);
    // one copy of the epilogue code: the accumulators are picked by a uniform branch chain
#pragma nounroll
    for (int mt = 0; mt < TM; ++mt) {
      f32x4 row[TN];
#pragma unroll
      for (int m = 0; m < TM; ++m) {
        if (m != mt) continue;
#pragma unroll
        for (int nt = 0; nt < TN; ++nt) {
          row[nt] = acc[m][nt];
          asm volatile("" : "+v"(row[nt]));   // opaque: stays in this branch
        }
      }
      const int r = wm * WM + mt * 16;
      epi.group(r, row, mt + 1 < TM ? r + 16 : -1);
    }
  }
  // DMAs past the last step must land before the workgroup's LDS is released
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  epi.finish();
}

template <int BN, int kSlots, int kMode>
void launch_stream_mode(const GemmArgs& g, const StreamPlan& p, hipStream_t stream) {
  hipLaunchKernelGGL((mxfp8_gemm_stream_kernel<BN, kSlots, kMode>), dim3(p.grid), dim3(256), 0, stream, g.a,
                     g.as, g.w, g.ws, g.mp, g.np, g.kp, g.ep, g.out_rows, g.n, p);
}

template <int BN, int kSlots>
int launch_stream(const GemmArgs& g, const StreamPlan& p, int mode, hipStream_t stream) {
  if (mode == 0)
    launch_stream_mode<BN, kSlots, 0>(g, p, stream);
  else if (mode == 1)
    launch_stream_mode<BN, kSlots, 1>(g, p, stream);
  else if (mode == 2)
    launch_stream_mode<BN, kSlots, 2>(g, p, stream);
  else if constexpr (BN == 256)
    launch_stream_mode<BN, kSlots, 3>(g, p, stream);
  return check_launch("vdn_mxfp8_gemm");
}

// ---- choice of the kernel by estimated time ----
// Microseconds, fitted to launches at M 77 .. 7395, N 1536 .. 21504, K 1536 .. 14336 on 256 CUs
// with weights not in cache (estimates within 20% of launches of 25 us and more; the shorter ones,
// all of the stream kernel, take as little as two thirds of theirs):
//   large kernel    18 + per wave of 256 x 256 tiles 4 + 1.25 (1.32 over several waves) a K step
//   stream, 256     10 + per 128 x 256 tile in sequence 3 + 0.80 (0.88) a K step
//   stream, 128     10 + per 128 x 128 tile in sequence 2 + 0.47 (0.52) a K step
// Every kernel sums an output over K in one sequence, so the choice moves no bit of the result.
// (Tiles left over after whole rounds with their K steps shared between workgroups: 1560 x 5120 x
// 5120 55 us against 65, 77 x 5120 x 5120 18 against 31, but a row's bits then followed the row
// count and the tile it fell in.)
struct GemmPlan {
  int64_t large_rows;   // rows of the large kernel (a multiple of 256, or all); the rest: stream
  StreamPlan stream;
};

double large_cost(int64_t waves, int nk) { return 18 + waves * (4 + nk * (waves > 1 ? 1.32 : 1.25)); }

StreamPlan stream_plan(int64_t mp, int64_t np, int bn, int cus) {
  StreamPlan p;
  p.bn = bn;
  p.tiles_m = static_cast<int>(mp / kSM);
  p.tiles_n = static_cast<int>((np + bn - 1) / bn);
  const int64_t tiles = static_cast<int64_t>(p.tiles_m) * p.tiles_n;
  p.rounds = static_cast<int>(tiles / cus);
  p.rest = static_cast<int>(tiles % cus);
  p.grid = p.rounds > 0 ? cus : p.rest;
  return p;
}

double best_stream(int64_t mp, int64_t np, int nk, int cus, StreamPlan* best) {
  double best_cost = 1e30;
  for (int bn = 256; bn >= 128; bn -= 128) {
    if (bn * static_cast<int64_t>(nk) * kBK >= (1ll << 31)) continue;   // 32-bit offsets in a tile
    const StreamPlan p = stream_plan(mp, np, bn, cus);
    const double tile = bn == 256 ? 3 : 2;
    const double step = bn == 256 ? (p.rounds > 0 ? 0.88 : 0.80) : (p.rounds > 0 ? 0.52 : 0.47);
    const double cost = 10 + (p.rounds + (p.rest > 0 ? 1 : 0)) * (nk * step + tile);
    if (cost < best_cost) {
      best_cost = cost;
      *best = p;
    }
  }
  return best_cost;
}

// The large kernel wins once its tiles fill the CUs for whole waves (its step moves half the
// bytes per FLOP); what is left over, and small problems, run faster in the stream kernel's
// smaller tiles. 5% in the estimate decides for one launch of the large kernel. It is considered from
// 1024 padded rows and columns on, where it was measured; by the estimate it would also win at 641 to
// 896 rows of wide projections (896 x 15360 x 5120: 72 us, the stream kernel 88 measured).
GemmPlan plan_gemm(int64_t mp, int64_t np, int64_t kp, int mode) {
  const int cus = cu_count(), nk = static_cast<int>(kp / kBK);
  GemmPlan plan{0, {}};
  double best = best_stream(mp, np, nk, cus, &plan.stream);
  if (mp >= 1024 && np >= 1024) {
    const int64_t tiles_m = (mp + 255) / 256, tiles_n = (np + 255) / 256, tiles = tiles_m * tiles_n;
    const int64_t waves = tiles / cus, rows = waves * cus / tiles_n;
    if (waves > 0 && rows > 0 && rows < tiles_m) {
      StreamPlan rest;
      const double both = large_cost((rows * tiles_n + cus - 1) / cus, nk) +
                          best_stream(mp - rows * 256, np, nk, cus, &rest);
      if (both < best) {
        best = both;
        plan.large_rows = rows * 256;
        plan.stream = rest;
      }
    }
    if (best >= 0.95 * large_cost((tiles + cus - 1) / cus, nk)) plan.large_rows = mp;
  }
  // SwiGLU's halves meet in a 256-column tile
  if (mode == 3 && plan.stream.bn == 128) plan.stream = stream_plan(mp - plan.large_rows, np, 256, cus);
  return plan;
}

}  // namespace

void gemm_choice(int64_t mp, int64_t np, int64_t kp, int mode, int64_t* large_rows, int* tile_cols) {
  const GemmPlan plan = plan_gemm(mp, np, kp, mode);
  *large_rows = plan.large_rows;
  *tile_cols = plan.large_rows < mp ? plan.stream.bn : 0;
}

int launch_gemm_planned(const GemmArgs& g, int mode, hipStream_t stream) {
  const GemmPlan plan = plan_gemm(g.mp, g.np, g.kp, mode);
  if (plan.large_rows > 0) {
    GemmArgs top = g;
    if (plan.large_rows < g.mp) {
      top.mp = plan.large_rows;
      top.out_rows = std::min(g.out_rows, plan.large_rows);
    }
    const int status = launch_persistent(top, stream);
    if (status != kOk || plan.large_rows >= g.mp) return status;
  }
  // the rows below: row blocks of 128 are contiguous in the codes and in the scales
  GemmArgs low = g;
  const int64_t r = plan.large_rows;
  low.a += r * g.kp;
  low.as += r / 128 * (g.kp / 128) * 512;
  low.mp -= r;
  low.out_rows = std::max<int64_t>(0, g.out_rows - r);
  if (g.ep.q_out == nullptr) {
    if (low.out_rows == 0) return kOk;
    low.ep.out += r * g.ep.ldc;
    if (g.ep.residual != nullptr) low.ep.residual += r * g.ep.ld_res;
  } else {
    low.ep.q_out += r * g.ep.kp_out;
    low.ep.s_out += r / 128 * (g.ep.kp_out / 128) * 512;
  }
  return plan.stream.bn == 256 ? launch_stream<256, 3>(low, plan.stream, mode, stream)
                               : launch_stream<128, 4>(low, plan.stream, mode, stream);
}

}  // namespace vdn
