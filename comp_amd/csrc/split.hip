// Weight ingestion on the device: ggml block bytes -> KURN's split planes, the device counterpart of the reference's
// host.split (src/komp/host.py:16-22).
//
// W holds N rows of K/blk ggml blocks, each `nbytes` long (Q4_0 and IQ4_NL: f16 d then 16 quant bytes, 18 bytes;
// Q8_0: f16 d then 32 int8, 34 bytes; TQ2_0: 64 quant bytes then f16 d, 66 bytes; Q4_K: f16 d, f16 dmin, 12 scale
// bytes, 128 quant bytes, 144 bytes).  Outputs: WQ u8 [N][SW] (the quant bytes of row r at WQ + r*SW, blocks in
// order) and WS i16 [N][K/blk] (the f16 bit patterns; Q4_K: [N][8 K/256], each block's first 16 bytes).  Pure byte
// movement, so the planes equal host.split's bit for bit.
//
// A workgroup moves 256 16-byte chunks of WQ, one a thread (Q4_0, IQ4_NL: a block each, Q8_0: half a block, TQ2_0: a
// quarter, Q4_K: an eighth).  Their ggml bytes (16.5 to 18 a chunk) are a whole number of 16-byte pieces at a 16-byte
// offset: they are read in such pieces and go through LDS, where a chunk's bytes start 0 or 2 bytes into a dword (block
// sizes and offsets are even): five dwords funnel-shifted into place (v_alignbyte_b32).  The thread of a block's chunk 0
// also moves its scale-plane bytes (2, or Q4_K's 16 in one store).
//
// HBM-bound: it reads each ggml byte once and writes each plane byte once.  No cache line is needed twice and the planes
// of a whole model are past every cache by the first token, so loads and stores are non-temporal.  Q4_0, buffers that
// rotate past the caches, us at 128256 x 4096 (591 MB in and out) / 14336 x 4096 / 4096 x 4096: a thread reading its own 18
// bytes in dwords 105.5 / 14.8 / 5.0; through LDS 97.9 / 13.3 / 4.6; non-temporal as well 89.6 (6.6 TB/s; a plain copy of
// 16 bytes a lane 5.6) / 12.0 / 4.4; four tiles a workgroup 94.2 / 12.1 / 4.3.
#include <hip/hip_ext.h>

#include "komp_device.h"
#include "komp_internal.h"

namespace komp {
namespace split_impl {

constexpr int kRsrcWord3 = 0x00020000;  // buffer descriptor word 3 on gfx9: 32-bit data, no swizzle
constexpr int kThreads = 256;
constexpr int kNt = 2;                  // buffer load cache policy: non-temporal
constexpr unsigned kOob = 0x7FFFFFF0u;  // an offset past every descriptor's range: the load returns zeros

// chunks: WQ chunks in this launch (blocks * chunks per block); nblk: blocks per row; cpb_log2: log2(chunks per
// block); nbytes, qoff, soff: the ggml block's size, quant offset and scale offset; wbytes: the launch's ggml bytes.
// W, WQ and WS point at the launch's first row.
__global__ void __launch_bounds__(kThreads)
split_kernel(int chunks, int nblk, int cpb_log2, int nbytes, int qoff, int soff, int sbytes, int wbytes, int64_t SW,
             const uint8_t* __restrict__ W, uint8_t* __restrict__ WQ, int16_t* __restrict__ WS) {
  constexpr int kPieces = 2;  // 16-byte pieces a thread: the workgroup's at most 18 bytes a chunk are at most 288
  __shared__ __align__(16) unsigned char lds[kPieces * kThreads * 16];
  const auto w = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(W), 0, wbytes, kRsrcWord3);
  const int tid = threadIdx.x;
  const int blocks = kThreads >> cpb_log2;  // of the workgroup
  const int b0 = blockIdx.x * blocks;
  const unsigned first = static_cast<unsigned>(b0) * nbytes;
  const int bytes = min(blocks * nbytes, wbytes - static_cast<int>(first));
  u32x4 v[kPieces];
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int o = 16 * (i * kThreads + tid);
    v[i] = __builtin_amdgcn_raw_buffer_load_b128(w, o + 16 <= bytes ? first + o : kOob, 0, kNt);
  }
#pragma unroll
  for (int i = 0; i < kPieces; ++i) *reinterpret_cast<u32x4*>(lds + 16 * (i * kThreads + tid)) = v[i];
  __syncthreads();
  const int tail = bytes & 15;  // the launch's last bytes, short of a piece: 2 bytes a thread
  if (tail != 0) {              // the same for the whole workgroup
    if (2 * tid < tail)
      *reinterpret_cast<uint16_t*>(lds + bytes - tail + 2 * tid) =
          __builtin_amdgcn_raw_buffer_load_b16(w, first + bytes - tail + 2 * tid, 0, 0);
    __syncthreads();
  }
  if (blockIdx.x * kThreads + tid >= static_cast<unsigned>(chunks)) return;
  const int lb = tid >> cpb_log2;             // block within the workgroup
  const int c = tid & ((1 << cpb_log2) - 1);  // chunk within the block
  const int b = b0 + lb;
  const int row = b / nblk;
  const int col = b - row * nblk;
  const unsigned src = static_cast<unsigned>(lb * nbytes + qoff + 16 * c);
  const unsigned* const d = reinterpret_cast<const unsigned*>(lds + (src & ~3u));
  u32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = __builtin_amdgcn_alignbyte(d[j + 1], d[j], src & 3u);
  uint8_t* const wq = WQ + row * SW + (static_cast<int64_t>(col) << (cpb_log2 + 4)) + 16 * c;
  __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(wq));
  if (c == 0) {
    const unsigned char* const so = lds + lb * nbytes + soff;
    if (sbytes == 16)  // Q4_K: 144-byte blocks, so the 16 bytes start 16-byte aligned
      __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(so),
                                  reinterpret_cast<u32x4*>(WS + 8 * static_cast<int64_t>(b)));
    else
      __builtin_nontemporal_store(*reinterpret_cast<const int16_t*>(so), WS + b);
  }
}

}  // namespace split_impl

// Rows are launched in batches whose ggml bytes stay below 2^31 (32-bit buffer offsets).
hipError_t launch_split(int fmt, const uint8_t* w, uint8_t* wq, int16_t* ws, int64_t n, int64_t k, int64_t sw,
                        hipStream_t stream) {
  const FmtInfo f = fmt_info(fmt);
  const int blk = f.block;
  const int nbytes = f.nbytes;
  const int qoff = f.qoff;
  const int soff = f.soff;
  const int cpb_log2 = f.qbytes == 16 ? 0 : f.qbytes == 32 ? 1 : f.qbytes == 64 ? 2 : 3;  // 16-byte chunks per block
  const int64_t nblk = k / blk;
  const int64_t row_bytes = nblk * nbytes;
  int64_t rows_per = row_bytes > 0 ? (int64_t{1} << 30) / row_bytes : n;
  if (rows_per < 1) rows_per = 1;
  if (rows_per >= 8) rows_per &= ~int64_t{7};  // each batch starts 16-byte aligned to the first
  for (int64_t r0 = 0; r0 < n; r0 += rows_per) {
    const int64_t rows = n - r0 < rows_per ? n - r0 : rows_per;
    const int64_t chunks = rows * nblk << cpb_log2;
    if (chunks == 0) continue;
    const dim3 grid(static_cast<unsigned>((chunks + split_impl::kThreads - 1) / split_impl::kThreads));
    const Timing tm = timing_slot(KIND_PROBE);
    hipExtLaunchKernelGGL(split_impl::split_kernel, grid, dim3(split_impl::kThreads), 0, stream, tm.start, tm.stop, 0,
                          static_cast<int>(chunks), static_cast<int>(nblk), cpb_log2, nbytes, qoff, soff, f.sbytes,
                          static_cast<int>(rows * row_bytes), sw, w + r0 * row_bytes, wq + r0 * sw,
                          ws + r0 * nblk * (f.sbytes / 2));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace komp
