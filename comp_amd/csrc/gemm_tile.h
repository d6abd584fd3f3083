// Tiled matrix-core GEMM for many activation columns (prompts, large batches): the result definition, arguments and
// optional S of gemm.hip's kernel, with the activations staged once per workgroup in LDS, in the form the matrix
// instruction takes, instead of read and rearranged by every wave.
//
// Bound.  Each block's exact integer dot is scaled in f32 by its own d_w * d_x, so the VALU runs a fixed number of
// instructions per output and block beside the matrix cores, and a matrix instruction of 16 cycles takes about two VALU
// issues from them (measured: 8 of them 65 ns, 32 v_fma_f32 61, both 92).  The batched kernel in gemm.hip spends per
// 16x16 tile and 32-value block 12 VALU instructions on the scaling (convert, multiply, fused multiply-add of 4 outputs a lane) and about as
// many on rearranging operands, re-read per 64 columns.  Here:
//   32-value blocks (Q4_0, IQ4_NL, Q8_0) and Q4_K go through v_mfma_f32_16x16x32_f16 with both operands as integers in
//     f16.  Every product and partial sum is an integer below 2^24 (Q8_0: 32 * 128 * 128 = 2^19; Q4_K: the 6-bit
//     sub-block scale times the nibble, at most 945, over half a block: 945 * 128 * 128 = 15.5 M; the two halves are
//     added in f32, which rounds where the integer sum's conversion would), so the f32 result is the exact block dot,
//     whatever order the matrix core adds in, and needs no conversion: 8 instructions instead of 12.  The products
//     d_w * d_x of four tiles are one v_mfma_f32_16x16x1_4b_f32 (16 multiplications take 30 ns of the VALU, it 15, and the
//     scales reach it as a dword a lane instead of four and one), which leaves 4 instructions: Q4_0 14336 x 4096 at 512
//     columns 117 -> 105 us (with 256-row tiles), Q4_K 4096 x 14336 at 1001 columns 192 -> 188 a call.  One f16
//     instruction covers a 32-value block in the time the int8 one does (its int8 form of K 32 has no higher rate).
//   TQ2_0's 256-value blocks stay on v_mfma_i32_16x16x64_i8 (twice the f16 rate; the scaling is 1/8 as often).
//
//   With one column tile (up to 16 columns) the 32-value blocks go through v_mfma_i32_16x16x32_i8: there the way of the
//     weights and activations to f16 costs more than the converted results.
//
// Tile.  A workgroup of WK x RW waves owns 16*WN*RW weight rows x 16*CN columns.  The waves of a K group split its rows
// (each unpacks its own weights, no wave twice) and share its staged activations; the WK groups take contiguous K ranges
// and add their partial sums at the end in group order.  A K step is 64 bytes of each weight row (Q8_0: 128): 128 values
// (TQ2_0: 256).  Two LDS buffers: during step i every thread unpacks its share of step i+1's activations (loaded a step
// earlier) into the other buffer, so one barrier a step suffices and every global load has a whole step to arrive.  A K
// group of one wave (RW 1) reads back its own staging only and has no barrier at all.
//
// Loads.  Four consecutive lanes read 64 consecutive bytes, and the wave's own LDS turns the weights into operand order.
// Loaded in operand order (16 rows apart lane by lane) a load held the address unit 49 cycles instead of 16, half of
// the kernel's time at 16 columns: Q4_0 28672 x 4096 24.0 -> 20.1 us, Q8_0 4096 x 14336 16.6 -> 13.3.
//
// LDS.  Operand unit (piece, group g) of a column is 16 bytes; units lie [piece][g][column ^ g], so a fragment read
// covers 256 contiguous, aligned bytes per 16 lanes (a permutation of 4 columns within it).  The staging writes several
// pieces (TQ2_0: and groups) of one column at a time: a pad of 64 bytes after each piece and the column's low bits
// crossed with g put those on different banks.  (Padding every unit row by 16 bytes instead left the reads with 42% of
// their LDS cycles in conflicts.)
//
// What it reaches: Q4_0 14336 x 4096 at 512 columns 105 us, of which VALU issue (4 clocks an instruction, 8 a matrix
// instruction, 28 an outer product) is 77 on the CUs that have a workgroup (224 of 256); Q4_K 4096 x 14336 at 1001 columns
// 188 a call, issue 116 and LDS half the time; TQ2_0 6912 x 2560 at 2048 columns 64.
#pragma once

#include <hip/hip_ext.h>

#include <type_traits>

#include "komp_device.h"
#include "komp_internal.h"

namespace komp {
namespace gemm_tile {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kRsrcWord3 = 0x00020000;  // buffer descriptor word 3 on gfx9: 32-bit data, no swizzle
constexpr unsigned kOob = 0x7FFFFFF0u;  // an offset past every descriptor's range: the load returns zeros

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, int64_t bytes) {
  const int n = static_cast<int>(bytes <= 0 ? 0 : (bytes < 0x7FFFFFF0 ? bytes : 0x7FFFFFF0));
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, n, kRsrcWord3);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc32(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), kRsrcWord3);
}

__device__ __forceinline__ f16x2 as_h2(unsigned v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ unsigned as_u(f16x2 v) { return __builtin_bit_cast(unsigned, v); }
__device__ __forceinline__ f16x2 h2(float a) { return f16x2{static_cast<_Float16>(a), static_cast<_Float16>(a)}; }

// The four signed bytes of q as f16 integers: bytes 0 and 2 in e, bytes 1 and 3 in o (the order the nibble forms give).
__device__ __forceinline__ void bytes_to_f16(unsigned q, unsigned& e, unsigned& o) {
  const unsigned u = q ^ 0x80808080u;  // byte + 128
  e = as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04020400u)) - h2(1152.f));
  o = as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030401u)) - h2(1152.f));
}

__device__ __forceinline__ f16x8 frag(unsigned a, unsigned b, unsigned c, unsigned d) {
  return __builtin_bit_cast(f16x8, u32x4{a, b, c, d});
}

// Four 16 x 16 outer products in C layout: block b (dwords 4b..4b+3) holds a of lanes 16b.. times b of lanes 16b..,
// rounded to f32 once, as the multiplication would.
__device__ __forceinline__ f32x16 outer4(float a, float b) {
  return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, f32x16{}, 0, 0, 0);
}

// LDS bytes of one K group's part: two activation buffers, two d_x buffers and (Q4_K) two buffers of 16-value sums; and
// of one wave's scales.
constexpr bool blk32(int fmt) { return fmt == FMT_Q4_0 || fmt == FMT_IQ4_NL || fmt == FMT_Q8_0; }

template <int FMT, int CN>
struct Lds {
  static constexpr int kUnit = blk32(FMT) && CN == 1 ? 8 : 16;  // int8 operands, or f16 ones (TQ2_0: 16 int8)
  static constexpr int kRow = 16 * CN * kUnit;             // a unit row: a unit a column
  static constexpr int kPiece = 4 * kRow + 64;             // the four groups' rows of a piece, and the pad
  static constexpr int kBuf = 4 * kPiece;
  static constexpr int kDxRow = 16 * CN + 16;  // 32-value blocks: d_x lies [block][column], 16 banks apart block by block
  static constexpr int kDx = FMT == FMT_TQ2_0 || FMT == FMT_Q4_K ? 16 * CN * 4 : 4 * kDxRow * 4;
  static constexpr int kSums = FMT == FMT_Q4_K ? 2 * kRow : 0;
  static constexpr int kGroup = 2 * (kBuf + kDx + kSums);
  // one wave's part: 64 weight bytes of each row, f32 scales (4 blocks of 16 rows a tile; TQ2_0 one; Q4_K d and dmin)
  // and (Q4_K) the rows' 16 scale-plane bytes
  static constexpr int weights(int wn) { return wn * 1024; }
  static constexpr int scales(int wn) {
    return wn * 16 * (FMT == FMT_TQ2_0 ? 1 : FMT == FMT_Q4_K ? 2 : 4) * 4 + (FMT == FMT_Q4_K ? wn * 256 : 0);
  }
  static constexpr int wave(int wn) { return weights(wn) + scales(wn); }
};

template <int FMT, int RW, int WN, int CN, int WK>
constexpr size_t lds_bytes() {
  const size_t stage = static_cast<size_t>(WK) * Lds<FMT, CN>::kGroup + WK * RW * Lds<FMT, CN>::wave(WN);
  const size_t red = static_cast<size_t>(WK - 1) * RW * WN * CN * 4 * 64 * 4;
  return stage > red ? stage : red;
}

template <int FMT, int RW, int WN, int CN, int WK, bool STORE_S>
__global__ void __launch_bounds__(64 * RW * WK, RW * WK == 4 ? 2 : 1)
tile_gemm_kernel(int N, int M, int K, int nblk, int64_t SW, const uint8_t* __restrict__ WQ,
                 const int16_t* __restrict__ WS, const int8_t* __restrict__ XQ, const float* __restrict__ XD,
                 float* __restrict__ Y, int32_t* __restrict__ S) {
  constexpr bool NIB4 = FMT == FMT_Q4_0 || FMT == FMT_IQ4_NL;
  constexpr bool Q8 = FMT == FMT_Q8_0;
  constexpr bool BLK32 = NIB4 || Q8;
  constexpr bool TQ2 = FMT == FMT_TQ2_0;
  constexpr bool QK = FMT == FMT_Q4_K;
  constexpr bool I8 = BLK32 && CN == 1;
  using L = Lds<FMT, CN>;
  constexpr int T = 64 * RW;          // threads of a K group
  constexpr int COLS = 16 * CN;
  constexpr int WGR = 16 * WN * RW;   // rows of the workgroup
  constexpr int WV = Q8 ? 2 : 1;      // 16-byte weight loads per row tile and step
  constexpr int XB = TQ2 ? 256 : 128;  // activation bytes per column and step
  constexpr bool F16 = !TQ2 && !I8;    // activations staged as f16
  constexpr int XV = F16 ? 2 : 1;      // 16-byte loads an item
  constexpr int PC = XB / 16 / XV;     // staging items of a column and step: 16 bytes (F16: a block's 32)
  constexpr int BI = COLS * PC / T;    // staging items a thread
  static_assert(BI * T == COLS * PC, "the threads split the staged columns evenly");
  extern __shared__ __align__(16) unsigned char lds[];
  // the bias (1024 in both f16) in a VGPR, so that masking a nibble pair and putting it on is one v_and_or_b32 (which
  // takes one literal)
  unsigned bias;
  asm("v_mov_b32 %0, 0x64006400" : "=v"(bias));
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave / RW;   // K group
  const int wr = wave % RW;   // row group
  const int tid = threadIdx.x - wk * T;
  const int r16 = lane & 15;
  const int g = lane >> 4;
  const int n0 = blockIdx.x * WGR;
  if (n0 >= N) return;  // a padding workgroup: the whole workgroup leaves before any barrier
  const int nw = n0 + 16 * WN * wr;
  const int m0 = blockIdx.y * COLS;
  const int rows = max(0, min(16 * WN, N - nw));
  const int cols = min(COLS, M - m0);
  const int nsteps = QK ? 2 * nblk : (TQ2 ? nblk : (nblk + 3) / 4);
  const int per = QK ? 2 * ((nblk + WK - 1) / WK) : (nsteps + WK - 1) / WK;  // steps a K group (the same for all)
  const int s0 = wk * per;
  const int s1 = min(nsteps, s0 + per);

  unsigned char* const gl = lds + wk * L::kGroup;
  unsigned char* const dxl = gl + 2 * L::kBuf;
  unsigned char* const suml = dxl + 2 * L::kDx;
  unsigned char* const wl = lds + WK * L::kGroup + wave * L::wave(WN);
  float* const scl = reinterpret_cast<float*>(wl + L::weights(WN));

  // The range of 32-value blocks, whose last K step may be partial, ends with the last row's blocks, not its stride: the
  // plane may be a view of some of a larger one's columns.  (In 32 bits, which the plan's limits allow: computed in 64, as
  // the others are, Q4_0 28672 x 1280 at 32 columns took 15.8 us against 15.4, and with the others in 32 as well Q8_0
  // 6912 x 8192 at 49 columns took 34.0 against 32.2.)
  const unsigned last = static_cast<unsigned>(nblk) * (Q8 ? 32 : 16);  // the last row's bytes
  const auto wq = BLK32 ? rsrc32(WQ + nw * SW, rows > 0 ? (rows - 1) * static_cast<unsigned>(SW) + last : 0)
                        : rsrc(WQ + nw * SW, rows * SW);
  const auto ws = rsrc(WS + static_cast<int64_t>(nw) * nblk * (QK ? 8 : 1),
                       static_cast<int64_t>(rows) * nblk * (QK ? 16 : 2));
  const auto xq = rsrc(XQ + static_cast<int64_t>(m0) * K, static_cast<int64_t>(cols) * K);
  const auto xd = rsrc(XD + static_cast<int64_t>(m0) * nblk, static_cast<int64_t>(cols) * nblk * 4);

  // ---- global loads, a step's worth each ----
  // Four consecutive lanes read consecutive addresses in every load (a row's 64 weight bytes, its 4 scales, 4 pieces of
  // a column): the address unit takes such a quad at once, and lanes that jump from row to row one by one (Q4_0
  // 28672 x 4096 at 16 columns, loads in the operands' lane order: 49 cycles a load, half of the kernel's time).
  const int lr = lane >> 2, lp = lane & 3;  // the lane's row and piece of a tile's load
  unsigned va[WN], vs[WN];
#pragma unroll
  for (int t = 0; t < WN; ++t) {
    va[t] = static_cast<unsigned>((16 * t + lr) * SW + 16 * lp);
    vs[t] = TQ2 ? static_cast<unsigned>((16 * t + r16) * nblk * 2) : static_cast<unsigned>((16 * t + lr) * nblk * (QK ? 16 : 2));
  }
  unsigned vx[BI], lx[BI];  // an item's source offset and its LDS offset
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    const int idx = i * T + tid;
    const int p = idx % PC, c = idx / PC;
    vx[i] = static_cast<unsigned>(c * K + 16 * XV * p);
    if constexpr (TQ2) {  // half p/8, crumb (p%8)/2, 16-byte half p%2 of the 32
      const int j = (p & 7) >> 1, gq = (p >> 3) * 2 + (p & 1);
      lx[i] = static_cast<unsigned>(j * L::kPiece + gq * L::kRow + 16 * (c ^ gq));
    } else if constexpr (F16) {  // block p: its unit of every group
      lx[i] = static_cast<unsigned>(p * L::kPiece + L::kUnit * c);
    } else {  // half p%2 of block p/2: half of the block's unit of every group
      lx[i] = static_cast<unsigned>((p >> 1) * L::kPiece + L::kUnit * c + (p & 1) * (L::kUnit / 2));
    }
  }
  // A tile's weights in the wave's LDS: row lr at 64 lr, its 16-byte pieces in the order p ^ f, f = -(row / 4) mod 4, so
  // that a dword of each row, or a piece of each row, is read from all banks
  const unsigned lw = static_cast<unsigned>(64 * lr + 16 * (lp ^ (-(lr >> 2) & 3)));
  const unsigned fr = static_cast<unsigned>(-(r16 >> 2) & 3);
  struct Weights {  // one step's weights and scales of the wave's rows
    u32x4 a[WN][WV];
    unsigned e[QK ? WN : 1];     // Q4_K: dword lp of the block's 16 scale-plane bytes
    unsigned short h[QK ? 1 : WN];
  };
  Weights wraw;
  auto load_w = [&](Weights& w, int s) {
    const unsigned off = s < s1 ? 64u * WV * s : kOob;
#pragma unroll
    for (int t = 0; t < WN; ++t) {
#pragma unroll
      for (int v = 0; v < WV; ++v)
        w.a[t][v] = __builtin_amdgcn_raw_buffer_load_b128(wq, va[t] + off + 64 * v, 0, 0);
      if constexpr (QK)
        w.e[t] = __builtin_amdgcn_raw_buffer_load_b32(ws, vs[t] + (s < s1 ? 16u * (s >> 1) + 4u * lp : kOob), 0, 0);
      else if constexpr (TQ2)
        w.h[t] = __builtin_amdgcn_raw_buffer_load_b16(ws, vs[t] + (s < s1 && g == 0 ? 2u * s : kOob), 0, 0);
      else  // a block past K has scale zero
        w.h[t] = __builtin_amdgcn_raw_buffer_load_b16(ws, vs[t] + (s < s1 && 4 * s + lp < nblk ? 8u * s + 2u * lp : kOob),
                                                       0, 0);
    }
  };
  constexpr int DN = BLK32 ? COLS * 4 : COLS;  // d_x of a step: [column][block]
  constexpr int DI = (DN + T - 1) / T;
  struct Acts {  // one step's activations, this thread's share
    u32x4 x[BI][XV];
    float d[DI];
  };
  Acts xraw;
  auto load_x = [&](Acts& a, int s) {
    const unsigned off = s < s1 ? static_cast<unsigned>(XB) * s : kOob;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int v = 0; v < XV; ++v) a.x[i][v] = __builtin_amdgcn_raw_buffer_load_b128(xq, vx[i] + off + 16 * v, 0, 0);
#pragma unroll
    for (int i = 0; i < DI; ++i) {
      const int idx = i * T + tid;
      unsigned o;
      if constexpr (BLK32)
        o = s < s1 && idx < DN && 4 * s + (idx & 3) < nblk
                ? static_cast<unsigned>((idx >> 2) * nblk + 4 * s + (idx & 3)) * 4u : kOob;  // fmt: skip
      else
        o = s < s1 && idx < DN ? static_cast<unsigned>(idx * nblk + (QK ? s >> 1 : s)) * 4u : kOob;
      a.d[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xd, o, 0, 0));
    }
  };
  // step s's activations from the registers into LDS buffer s & 1
  auto stage = [&](const Acts& a, int s) {
    unsigned char* const b = gl + ((s - s0) & 1) * L::kBuf;
    float* const dxb = reinterpret_cast<float*>(dxl + ((s - s0) & 1) * L::kDx);
#pragma unroll
    for (int i = 0; i < BI; ++i) {
      if constexpr (TQ2) {
        *reinterpret_cast<u32x4*>(b + lx[i]) = a.x[i][0];
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if constexpr (F16) {  // group q: values 4q..4q+3 and 16+4q..16+4q+3
            u32x4 u;
            unsigned e, o;
            bytes_to_f16(a.x[i][0][q], e, o);
            u[0] = e;
            u[1] = o;
            bytes_to_f16(a.x[i][1][q], e, o);
            u[2] = e;
            u[3] = o;
            *reinterpret_cast<u32x4*>(b + (lx[i] ^ (16 * q)) + q * L::kRow) = u;
          } else {  // dword q of the piece: group q's half of the block's unit
            *reinterpret_cast<unsigned*>(b + lx[i] + q * L::kRow) = a.x[i][0][q];
          }
        }
        if constexpr (QK) {  // the block's two 16-value sums (at most 16 * 128: exact in f16)
          const int idx = i * T + tid;
          int lo = 0, hi = 0;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            lo = __builtin_amdgcn_sdot4(static_cast<int>(a.x[i][0][q]), 0x01010101, lo, false);
            hi = __builtin_amdgcn_sdot4(static_cast<int>(a.x[i][1][q]), 0x01010101, hi, false);
          }
          const f16x2 p = {static_cast<_Float16>(static_cast<float>(lo)), static_cast<_Float16>(static_cast<float>(hi))};
          *reinterpret_cast<unsigned*>(suml + (((s - s0) >> 1) & 1) * L::kSums + (s & 1) * L::kRow + 16 * (idx / PC) +
                                       4 * (idx % PC)) = as_u(p);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < DI; ++i) {
      const int idx = i * T + tid;
      if (DI * T == DN || idx < DN) dxb[BLK32 ? (idx & 3) * L::kDxRow + (idx >> 2) : idx] = a.d[i];
    }
  };

  f32x4 acc[WN][CN];
#pragma unroll
  for (int t = 0; t < WN; ++t)
#pragma unroll
    for (int u = 0; u < CN; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};

  f32x4 half[QK ? WN : 1][QK ? CN : 1];  // Q4_K: the dots of a block's first half

  auto store_s = [&](const f32x4& v, int t, int u, int b, int stride, int at, bool add) {
    const int col = m0 + 16 * u + r16;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = nw + 16 * t + 4 * g + r;
      if (col < M && row < N) {
        int32_t* p = S + ((static_cast<int64_t>(col) * N + row) * nblk + b) * stride + at;
        const int x = static_cast<int>(v[r]);
        *p = add ? *p + x : x;
      }
    }
  };

  // The step's products run as a pipeline over (piece, column tile): the operand fragments are read from LDS two tiles
  // ahead, and a tile's result is scaled while the next tile's matrix instruction runs.  The scheduling barriers keep
  // that order (left alone, the compiler scales each result right behind its matrix instruction and waits for it), and
  // the empty asm statements pin each sum's update to its place (otherwise it may be moved down to the sum's next use, a
  // step later, with every result of the step kept live: 1000 bytes a lane of spills).
  // wf[t][v]: a tile's weights in operand order.  TQ2_0: the lane's 16 bytes (row r16, piece g); else dword g of the
  // row's four 16-byte pieces (nibble formats: of 4 blocks, Q8_0: of 4 half blocks)
  auto compute = [&](const u32x4 (&wf)[WN][WV], int s, auto odd) {
    const unsigned char* const b = gl + ((s - s0) & 1) * L::kBuf + (I8 ? r16 * 8 : (r16 ^ g) * 16) + g * L::kRow;
    const unsigned char* const dxp = dxl + ((s - s0) & 1) * L::kDx;
    if constexpr (I8) {
      // one column tile: the nibbles' way to f16 would cost more than the converted results save (Q4_0 9 instructions a
      // tile and block against 3 and 4 conversions), and so would the activations'
      long x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)  // (vector types may alias the staged dwords; long may not)
        x[j] = __builtin_bit_cast(long, *reinterpret_cast<const u32x2*>(b + j * L::kPiece));
      i32x4 corr[4], cc[2][WN];
      f32x16 pr[WN];  // d_w * d_x: instruction block j is the step's block j
      const float dx = reinterpret_cast<const float*>(dxp)[g * L::kDxRow + r16];
#pragma unroll
      for (int t = 0; t < WN; ++t) pr[t] = outer4(scl[t * 64 + lane], dx);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        corr[j] = i32x4{0, 0, 0, 0};
        if constexpr (FMT == FMT_Q4_0)  // the nibbles go in unsigned: start at -8 times the block's activation sum
          corr[j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(static_cast<long>(0xF8F8F8F8F8F8F8F8ull), x[j], corr[j], 0, 0, 0);
      }
      auto scale = [&](int j) {
#pragma unroll
        for (int t = 0; t < WN; ++t) {
          f32x4 cf;
#pragma unroll
          for (int r = 0; r < 4; ++r) cf[r] = static_cast<float>(cc[j & 1][t][r]);
          if (STORE_S && 4 * s + j < nblk && s < s1) store_s(cf, t, 0, 4 * s + j, 1, 0, false);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[t][0][r] = __builtin_fmaf(cf[r], pr[t][4 * j + r], acc[t][0][r]);
          asm volatile("" : "+v"(acc[t][0]));
        }
      };
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int t = 0; t < WN; ++t) {
          unsigned lo, hi;
          if constexpr (FMT == FMT_Q4_0) {
            lo = wf[t][0][j] & 0x0F0F0F0Fu;
            hi = (wf[t][0][j] >> 4) & 0x0F0F0F0Fu;
          } else if constexpr (FMT == FMT_IQ4_NL) {
            iq4_nl_lut(wf[t][0][j], lo, hi);
          } else {
            lo = wf[t][j >> 1][2 * (j & 1)];
            hi = wf[t][j >> 1][2 * (j & 1) + 1];
          }
          cc[j & 1][t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, u32x2{lo, hi}), x[j], corr[j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (j > 0) scale(j - 1);
      }
      scale(3);
    } else if constexpr (BLK32) {
      constexpr int NI = 4 * CN;  // i = j * CN + u: block j of the step, column tile u
      static_assert(CN == 2 || CN % 4 == 0, "four consecutive i share one product instruction");
      f16x8 a[2][WN], x[4];
      f32x4 cc[2][WN];
      f32x16 pr[WN];  // d_w * d_x of tiles i & ~3 .. i | 3
      float pa[WN], pb;
      auto fetch_scales = [&](int i) {  // of the product instruction's block g: tile i + g
        const int j = CN == 2 ? i / CN + (g >> 1) : i / CN;
        const int c = CN == 2 ? 16 * (g & 1) : 16 * (i % CN + g);
#pragma unroll
        for (int t = 0; t < WN; ++t) pa[t] = scl[(t * 4 + j) * 16 + r16];
        pb = reinterpret_cast<const float*>(dxp)[j * L::kDxRow + c + r16];
      };
      auto fetch = [&](int i) {
        x[i & 3] = *reinterpret_cast<const f16x8*>(b + (i / CN) * L::kPiece + 256 * (i % CN));
      };
      auto unpack = [&](int j) {
#pragma unroll
        for (int t = 0; t < WN; ++t) {
          if constexpr (FMT == FMT_Q4_0) {
            const unsigned p = wf[t][0][j], q = p >> 8;
            a[j & 1][t] =
                frag(as_u(as_h2((p & 0x000F000Fu) | bias) - h2(1032.f)), as_u(as_h2((q & 0x000F000Fu) | bias) - h2(1032.f)),
                     as_u(__builtin_elementwise_fma(as_h2((p & 0x00F000F0u) | bias), h2(0.0625f), h2(-72.f))),
                     as_u(__builtin_elementwise_fma(as_h2((q & 0x00F000F0u) | bias), h2(0.0625f), h2(-72.f))));
          } else {
            unsigned lo, hi, e0, o0, e1, o1;
            if constexpr (FMT == FMT_IQ4_NL) {
              iq4_nl_lut(wf[t][0][j], lo, hi);
            } else {
              lo = wf[t][j >> 1][2 * (j & 1)];
              hi = wf[t][j >> 1][2 * (j & 1) + 1];
            }
            bytes_to_f16(lo, e0, o0);
            bytes_to_f16(hi, e1, o1);
            a[j & 1][t] = frag(e0, o0, e1, o1);
          }
        }
      };
      auto scale = [&](int i) {
        const int j = i / CN, u = i % CN;
#pragma unroll
        for (int t = 0; t < WN; ++t) {
          if (STORE_S && 4 * s + j < nblk && s < s1) store_s(cc[i & 1][t], t, u, 4 * s + j, 1, 0, false);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[t][u][r] = __builtin_fmaf(cc[i & 1][t][r], pr[t][4 * (i & 3) + r], acc[t][u][r]);
          asm volatile("" : "+v"(acc[t][u]));
        }
      };
      fetch(0);
      fetch(1);
      fetch_scales(0);
      unpack(0);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int j = i / CN;
        __builtin_amdgcn_sched_barrier(0);
        if (i + 2 < NI) fetch(i + 2);
#pragma unroll
        for (int t = 0; t < WN; ++t)
          cc[i & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j & 1][t], x[i & 3], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (i > 0) scale(i - 1);
        if (i % 4 == 0) {
#pragma unroll
          for (int t = 0; t < WN; ++t) pr[t] = outer4(pa[t], pb);
          if (i + 4 < NI) fetch_scales(i + 4);
        }
        if (i % CN == CN - 1 && j < 3) unpack(j + 1);
      }
      scale(NI - 1);
    } else if constexpr (TQ2) {
      constexpr bool OUT4 = CN % 4 == 0;  // d_w * d_x of tiles u & ~3 .. u | 3 from one matrix instruction
      i32x4 a[WN][4], x[2][4], cc[2][WN];
      f32x4 dw[WN];
      float dx[CN], pa[WN], pb;
      f32x16 pr[WN];
      auto fetch = [&](int u) {
#pragma unroll
        for (int v = 0; v < 4; ++v) x[u & 1][v] = *reinterpret_cast<const i32x4*>(b + v * L::kPiece + 256 * u);
      };
      auto scale = [&](int u) {
#pragma unroll
        for (int t = 0; t < WN; ++t) {
          f32x4 cf;
#pragma unroll
          for (int r = 0; r < 4; ++r) cf[r] = static_cast<float>(cc[u & 1][t][r]);
          if (STORE_S && s < s1) store_s(cf, t, u, s, 1, 0, false);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[t][u][r] = __builtin_fmaf(OUT4 ? pr[t][4 * (u & 3) + r] : dx[u] * dw[t][r], cf[r], acc[t][u][r]);
          asm volatile("" : "+v"(acc[t][u]));
        }
      };
      fetch(0);
      if constexpr (OUT4) {
        pb = reinterpret_cast<const float*>(dxp)[lane];
      } else {
#pragma unroll
        for (int u = 0; u < CN; ++u) dx[u] = *reinterpret_cast<const float*>(dxp + (16 * u + r16) * 4);
      }
#pragma unroll
      for (int t = 0; t < WN; ++t) {
        if constexpr (OUT4)
          pa[t] = scl[t * 16 + r16];
        else
          dw[t] = *reinterpret_cast<const f32x4*>(scl + t * 16 + 4 * g);
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int d = 0; d < 4; ++d)  // crumbs 0..3 -> -1, 0, 1, 2 (a byte table lookup)
            a[t][v][d] = static_cast<int>(__builtin_amdgcn_perm(0, 0x020100FFu, (wf[t][0][d] >> (2 * v)) & 0x03030303u));
      }
#pragma unroll
      for (int u = 0; u < CN; ++u) {
        __builtin_amdgcn_sched_barrier(0);
        if (u + 1 < CN) fetch(u + 1);
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int t = 0; t < WN; ++t)
            cc[u & 1][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[t][v], x[u & 1][v],
                                                                 v == 0 ? i32x4{0, 0, 0, 0} : cc[u & 1][t], 0, 0, 0);
        if (u > 0) scale(u - 1);
        if constexpr (OUT4) {
          if (u % 4 == 0) {
#pragma unroll
            for (int t = 0; t < WN; ++t) pr[t] = outer4(pa[t], pb);
            if (u + 4 < CN) pb = reinterpret_cast<const float*>(dxp)[16 * (u + 4) + lane];
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      scale(CN - 1);
    } else {
      // Q4_K: half s % 2 of block s / 2, sub-blocks i = 0..3 of the half: the low (even i) or high nibbles of pieces
      // 2(i/2), 2(i/2) + 1.  The operand is scale * nibble (at most 945), so the half's four sub-blocks run one chain;
      // the block's mins term takes one more instruction over its 16 sums of 16 activations, at the odd half.
      constexpr bool hb = decltype(odd)::value;
      constexpr int NF = hb ? 5 : 4;  // operand fragments a column tile: four sub-blocks and (odd half) the sums
      constexpr int NI = NF * CN;
      f16x8 a[WN][4], x[4];
      f32x4 dw[WN], dm[WN], cc[2][WN], cm[hb ? 2 : 1][WN];
      f16x8 am[WN];
      constexpr bool OUT4 = CN % 4 == 0 && hb;  // d * d_x and dmin * d_x of tiles u & ~3 .. u | 3, each one instruction
      float dx[CN], pa[WN], qa[WN], pb;
      f32x16 pr[WN], qr[WN];
      const unsigned char* const sp = suml + (((s - s0) >> 1) & 1) * L::kSums + (g & 1) * L::kRow + r16 * 16;
      auto fetch = [&](int i) {
        const int u = i / NF, f = i % NF;
        x[i & 3] = *reinterpret_cast<const f16x8*>(f < 4 ? b + f * L::kPiece + 256 * u : sp + 256 * u);
      };
      auto scale = [&](int u) {
#pragma unroll
        for (int t = 0; t < WN; ++t) {
          if constexpr (!hb) {
            half[t][u] = cc[u & 1][t];
            asm volatile("" : "+v"(half[t][u]));
          } else {
            // the block's sd: a sum of two exact integers, rounded once as the integer's conversion would be
            if constexpr (STORE_S) {
              if (s < s1) {
                store_s(half[t][u], t, u, s >> 1, 2, 0, false);
                store_s(cc[u & 1][t], t, u, s >> 1, 2, 0, true);
                store_s(cm[u & 1][t], t, u, s >> 1, 2, 1, false);
              }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float sd = half[t][u][r] + cc[u & 1][t][r];
              acc[t][u][r] += OUT4 ? __builtin_fmaf(sd, pr[t][4 * (u & 3) + r], -cm[u & 1][t][r] * qr[t][4 * (u & 3) + r])
                                   : __builtin_fmaf(sd, dw[t][r] * dx[u], -cm[u & 1][t][r] * (dm[t][r] * dx[u]));
            }
            asm volatile("" : "+v"(acc[t][u]));  // as above
          }
        }
      };
      fetch(0);
      fetch(1);
      if constexpr (OUT4) {
        pb = reinterpret_cast<const float*>(dxp)[lane];
      } else if constexpr (hb) {
#pragma unroll
        for (int u = 0; u < CN; ++u) dx[u] = *reinterpret_cast<const float*>(dxp + (16 * u + r16) * 4);
      }
#pragma unroll
      for (int t = 0; t < WN; ++t) {
        if constexpr (OUT4) {
          pa[t] = scl[t * 32 + r16];
          qa[t] = scl[t * 32 + 16 + r16];
        } else if constexpr (hb) {
          dw[t] = *reinterpret_cast<const f32x4*>(scl + t * 32 + 4 * g);
          dm[t] = *reinterpret_cast<const f32x4*>(scl + t * 32 + 16 + 4 * g);
        }
        const u32x4 e = *reinterpret_cast<const u32x4*>(scl + WN * 32 + t * 64 + r16 * 4);
        const unsigned sc = hb ? (e[3] & 0x0F0F0F0Fu) | ((e[1] >> 2) & 0x30303030u) : e[1] & 0x3F3F3F3Fu;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          constexpr unsigned kSel[4] = {0x04000400u, 0x04010401u, 0x04020402u, 0x04030403u};
          // (1024 + s) - 1024: the scale in both halves; then 1024 + q times it, less 1024 times it (odd i: 16 q)
          const f16x2 f = as_h2(__builtin_amdgcn_perm(0x64646464u, sc, kSel[i])) - h2(1024.f);
          const f16x2 m = (i & 1) ? f * h2(0.0625f) : f;
          const f16x2 k = f * h2((i & 1) ? -64.f : -1024.f);
          const unsigned mask = (i & 1) ? 0x00F000F0u : 0x000F000Fu;
          const unsigned p0 = wf[t][0][2 * (i >> 1)], p1 = wf[t][0][2 * (i >> 1) + 1];
          a[t][i] = frag(as_u(__builtin_elementwise_fma(as_h2((p0 & mask) | bias), m, k)),
                         as_u(__builtin_elementwise_fma(as_h2(((p0 >> 8) & mask) | bias), m, k)),
                         as_u(__builtin_elementwise_fma(as_h2((p1 & mask) | bias), m, k)),
                         as_u(__builtin_elementwise_fma(as_h2(((p1 >> 8) & mask) | bias), m, k)));
        }
        // slot e of groups 0 and 1: the min of sub-block 4g + e/2; groups 2 and 3 hold zeros
        const unsigned mw = g >= 2 ? 0u
                            : g == 0 ? e[2] & 0x3F3F3F3Fu
                                     : ((e[3] >> 4) & 0x0F0F0F0Fu) | ((e[2] >> 2) & 0x30303030u);
        am[t] = frag(as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, mw, 0x04000400u)) - h2(1024.f)),
                     as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, mw, 0x04010401u)) - h2(1024.f)),
                     as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, mw, 0x04020402u)) - h2(1024.f)),
                     as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, mw, 0x04030403u)) - h2(1024.f)));
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int u = i / NF, f = i % NF;
        __builtin_amdgcn_sched_barrier(0);
        if (i + 2 < NI) fetch(i + 2);
#pragma unroll
        for (int t = 0; t < WN; ++t) {
          if (f < 4)
            cc[u & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                a[t][f], x[i & 3], f == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : cc[u & 1][t], 0, 0, 0);
          else
            cm[hb ? u & 1 : 0][t] =
                __builtin_amdgcn_mfma_f32_16x16x32_f16(am[t], x[i & 3], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (f == 1 && u > 0) scale(u - 1);
        if constexpr (OUT4) {
          if (f == 1 && u % 4 == 0) {
#pragma unroll
            for (int t = 0; t < WN; ++t) {
              pr[t] = outer4(pa[t], pb);
              qr[t] = outer4(qa[t], pb);
            }
            if (u + 4 < CN) pb = reinterpret_cast<const float*>(dxp)[16 * (u + 4) + lane];
          }
        }
      }
      scale(CN - 1);
    }
  };
  // this step's weights and f32 scales through the wave's own LDS, from where its lanes read them back in operand and C
  // layout (rows 4g + r); the wave's own LDS accesses stay in order, and the compiler fences keep them so
  auto take_w = [&](const Weights& w, u32x4 (&wf)[WN][WV]) {
#pragma unroll
    for (int t = 0; t < WN; ++t) {
      if constexpr (BLK32) {
        scl[(t * 4 + lp) * 16 + lr] = f16_bits_to_f32(static_cast<int16_t>(w.h[t]));
      } else if constexpr (TQ2) {
        if (g == 0) scl[t * 16 + r16] = f16_bits_to_f32(static_cast<int16_t>(w.h[t]));
      } else {  // d from the even pieces' lanes, dmin from the odd ones': both in dword 0
        reinterpret_cast<unsigned*>(scl)[WN * 32 + t * 64 + lane] = w.e[t];
        const unsigned d0 = static_cast<unsigned>(dpp_i<0x00>(static_cast<int>(w.e[t])));  // quad_perm [0, 0, 0, 0]
        scl[t * 32 + (lp & 1) * 16 + lr] = f16_bits_to_f32(static_cast<int16_t>(d0 >> (16 * (lp & 1))));
      }
    }
#pragma unroll
    for (int v = 0; v < WV; ++v) {
#pragma unroll
      for (int t = 0; t < WN; ++t) *reinterpret_cast<u32x4*>(wl + t * 1024 + lw) = w.a[t][v];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int t = 0; t < WN; ++t) {
        if constexpr (TQ2) {
          wf[t][v] = *reinterpret_cast<const u32x4*>(wl + t * 1024 + 64 * r16 + 16 * (g ^ fr));
        } else {
#pragma unroll
          for (unsigned j = 0; j < 4; ++j)
            wf[t][v][j] = *reinterpret_cast<const unsigned*>(wl + t * 1024 + 64 * r16 + 4 * g + 16 * (j ^ fr));
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  };
  auto barrier = [&] {  // the staged buffer is published; global loads stay in flight
    if constexpr (RW == 1) {  // a wave reads back its own staging only: its LDS accesses stay in order
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    } else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
  };

  // Step i: its weights and step i + 1's activations from the registers into LDS, then the loads of the next ones into the
  // same registers.  (Deeper rings of loads measured no faster: a longer loop round costs more in cold instructions than
  // it hides in latency.)
  auto step = [&](int i, auto odd) {
    const int s = s0 + i;
    u32x4 wf[WN][WV];
    take_w(wraw, wf);
    load_w(wraw, s + 1);
    stage(xraw, s + 1);  // past the group's last step: zeros into the idle buffer
    load_x(xraw, s + 2);
    compute(wf, s, odd);
    barrier();
  };
  load_x(xraw, s0);
  load_w(wraw, s0);
  stage(xraw, s0);
  load_x(xraw, s0 + 1);
  barrier();
  if constexpr (QK) {  // per is even: s0 + i is the first half of a block
    for (int i = 0; i < per; i += 2) {
      step(i, std::false_type{});
      step(i + 1, std::true_type{});
    }
  } else {
    for (int i = 0; i < per; ++i) step(i, std::false_type{});
  }

  if constexpr (WK > 1) {  // partial sums of the other K groups, added in group order
    float* red = reinterpret_cast<float*>(lds);
    if constexpr (RW == 1) __syncthreads();  // every wave is done with its staging
    if (wk > 0) {
#pragma unroll
      for (int t = 0; t < WN; ++t)
#pragma unroll
        for (int u = 0; u < CN; ++u)
          *reinterpret_cast<f32x4*>(red + ((((wk - 1) * RW + wr) * WN + t) * CN + u) * 256 + lane * 4) = acc[t][u];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int q = 0; q < WK - 1; ++q)
#pragma unroll
      for (int t = 0; t < WN; ++t)
#pragma unroll
        for (int u = 0; u < CN; ++u)
          acc[t][u] += *reinterpret_cast<const f32x4*>(red + (((q * RW + wr) * WN + t) * CN + u) * 256 + lane * 4);
  }
  const bool wide = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0;  // whole 16-byte groups of rows
#pragma unroll
  for (int t = 0; t < WN; ++t)
#pragma unroll
    for (int u = 0; u < CN; ++u) {
      const int row = nw + 16 * t + 4 * g;
      const int col = m0 + 16 * u + r16;
      if (col >= M) continue;
      float* y = Y + static_cast<int64_t>(col) * N + row;
      if (wide) {
        if (row < N) *reinterpret_cast<f32x4*>(y) = acc[t][u];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (row + r < N) y[r] = acc[t][u][r];
      }
    }
}

template <int FMT, int RW, int WN, int CN, int WK, bool STORE_S>
hipError_t launch_plan(const GemmCall& c, hipStream_t stream) {
  // as gemm.hip: with several column groups the row groups are padded to a multiple of 8, so that the column groups of a
  // row group run on one XCD and share its L2
  const unsigned gx = (c.n + 16 * WN * RW - 1) / (16 * WN * RW), gy = (c.m + 16 * CN - 1) / (16 * CN);
  const dim3 grid(gy > 1 ? (gx + 7) / 8 * 8 : gx, gy);
  constexpr size_t lds = lds_bytes<FMT, RW, WN, CN, WK>();
  static_assert(lds <= 160 * 1024, "LDS of a workgroup");
  auto kern = tile_gemm_kernel<FMT, RW, WN, CN, WK, STORE_S>;
  static std::atomic<unsigned> lds_limit[kMaxDevices];  // this instantiation's allowed dynamic LDS, per device
  const hipError_t le = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds, lds_limit);
  if (le != hipSuccess) return le;
  const Timing tm = timing_slot(gemv_kind(FMT));
  hipExtLaunchKernelGGL(kern, grid, dim3(64 * RW * WK), lds, stream, tm.start, tm.stop, 0, c.n, c.m, c.k,
                        c.k / fmt_info(FMT).block, c.sw, c.wq, c.ws, c.xq, c.xd, c.y, c.s);
  return hipGetLastError();
}

// The instantiated plans (gemm_tile_plan in abi.hip picks one; with S, tile_plan_with_s of it).
template <int FMT>
hipError_t launch_fmt(const GemmCall& c, const TilePlan& p, hipStream_t stream) {
  if (c.s != nullptr) {
    const TilePlan q = tile_plan_with_s(p);
#define KOMP_TILE_PLAN_S(RW, WN, CN, WK) \
  if (q.rw == RW && q.wn == WN && q.cn == CN && q.wk == WK) return launch_plan<FMT, RW, WN, CN, WK, true>(c, stream);
    KOMP_TILE_PLAN_S(2, 1, 2, 1)
    KOMP_TILE_PLAN_S(2, 1, 2, 2)
    KOMP_TILE_PLAN_S(1, 1, 1, 4)
    KOMP_TILE_PLAN_S(1, 1, 1, 8)
#undef KOMP_TILE_PLAN_S
    return hipErrorInvalidConfiguration;
  }
#define KOMP_TILE_PLAN(ON, RW, WN, CN, WK)                                  \
  if constexpr (ON)                                                         \
    if (p.rw == RW && p.wn == WN && p.cn == CN && p.wk == WK) return launch_plan<FMT, RW, WN, CN, WK, false>(c, stream);
  constexpr bool q4 = FMT == FMT_Q4_0 || FMT == FMT_IQ4_NL, tq2 = FMT == FMT_TQ2_0, q8 = FMT == FMT_Q8_0, qk = FMT == FMT_Q4_K;
  KOMP_TILE_PLAN(true, 1, 1, 1, 8)
  KOMP_TILE_PLAN(true, 1, 2, 1, 8)
  KOMP_TILE_PLAN(true, 1, 2, 1, 4)
  KOMP_TILE_PLAN(q4 || tq2, 1, 1, 1, 4)
  KOMP_TILE_PLAN(tq2, 2, 1, 1, 4)
  KOMP_TILE_PLAN(q4 || tq2, 2, 2, 1, 4)
  KOMP_TILE_PLAN(!q8, 2, 1, 2, 4)
  KOMP_TILE_PLAN(true, 2, 2, 2, 4)
  KOMP_TILE_PLAN(qk, 2, 1, 4, 4)
  KOMP_TILE_PLAN(true, 4, 1, 4, 2)
  KOMP_TILE_PLAN(q4 || tq2, 4, 2, 4, 2)
  KOMP_TILE_PLAN(q4 || q8, 4, 2, 4, 1)
  KOMP_TILE_PLAN(qk, 4, 1, 8, 2)
  KOMP_TILE_PLAN(q4 || tq2, 4, 2, 8, 1)
  KOMP_TILE_PLAN(q4 || q8, 4, 2, 8, 2)
  KOMP_TILE_PLAN(!q4, 8, 1, 8, 1)
  KOMP_TILE_PLAN(!qk, 8, 2, 8, 1)  // (Q4_K's waves also hold a block's first half of every output: too many registers)
#undef KOMP_TILE_PLAN
  return hipErrorInvalidConfiguration;
}

}  // namespace gemm_tile
}  // namespace komp
