// Exact-order batched projection of the prompt on the fp32 matrix instructions (gfx950).
//
// Every output is the decode step's sum for its row, bit for bit: lane class c
// (0..63) of a wave adds the products of k = 512 j + 8 c + e sequentially (j,
// then e ascending, one fused multiply-add each) and the 64 class sums are
// added in wave64_sum's tree, a balanced binary tree over c.
// v_mfma_f32_16x16x1_4b_f32 can do that: it has K = 1, so one instruction is
// ONE fused multiply-add per accumulator, rounded once to nearest even
// (compared bit for bit with fmaf chains of 128 steps over the whole fp16
// range, subnormals included).  Its four blocks are four classes: block b
// adds A_b[i] * B_b[j] to its own 16 x 16 sums, so a wave's instruction
// advances 4 classes x 256 outputs, and the tree runs lane by lane on the
// accumulators.  An fp16 value and the product of two are exact in fp32, and
// every partial sum is a multiple of 2^-48, so no subnormal ever occurs.
// (The fp16 matrix instructions do not round to nearest: fed one product at a
// time, 1 sum in 50 differed.)
//
// What bounds it: these instructions run on the vector FP32 units (66-68 T
// FMA/s with two waves per SIMD), and every other vector instruction takes its
// time from them: ~4 cycles each with two waves per SIMD, ~7.5 with one,
// against an MFMA's 32.  So there is none in the loop: operands are converted
// to fp32 by the memory path (buffer_load_format_xyzw: four fp16 in, four fp32
// out; equal to the conversion for all finite halves), wait in LDS as fp32,
// and all offsets are fixed per lane, the position in K in a scalar register.
// What remains beside the products, by leaving each out at 1000 tokens and K =
// 5504 (222 us with all): the loads 13 us, the LDS stores 22 us; and the class
// tree's 63 adds per output (6% at K = 2048).
//
// 2048-row products of a 127-token prompt: K = 2048 12.9 us, K = 5504 28.8 us
// (50 T FMA/s); 6144 x 2048 35.6 us.  The FMA-pipe kernels before it, which
// spent an LDS read and a wave reduction per pair of tokens, took 25-27, 66-72
// and 64-70 us (1000 tokens: 174 -> 90, 532 -> 218, 472 -> 268 us).
#include "qd_device.h"
#include "qd_internal.h"

namespace qd {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int kXcds = 8;   // MI355X: workgroups are dealt to 8 XCDs in turn

// Y^T = W X^T in workgroup tiles of 16 WB rows of W by 16 TB tokens.  Wave g of
// eight holds the whole tile, WB x TB blocks of 16 x 16 outputs, over classes
// 8 g .. 8 g + 7: its elements are k = 512 j + 64 g .. + 64 for every j, 128
// bytes of a row (one line) each.  Step q (0, 1) of such a chunk multiplies
// classes 4 q .. 4 q + 3: lane l holds class 4 q + l / 16 of row l % 16 of each
// block, four elements (a quarter of the chunk) at a time.  The waves share
// nothing until the end, where their sums meet in LDS in the upper three levels
// of the tree: no barrier in the loop, and two waves on every SIMD from a
// single workgroup per CU.  (Tiles of 64 x 64 outputs staged by the whole
// workgroup behind a barrier per chunk ran 6-13% faster at 1000 tokens and
// 15-45% slower at 127; four-wave workgroups of two groups per wave, two per
// CU, and persistent workgroups that load the next tile's first chunk before
// the sums meet gained nothing.)
//
// A wave's chunk comes in whole 128-byte lines into registers while the chunk
// before it is multiplied, then goes to the wave's own 256-byte LDS rows (piece
// p of four elements of row r at p ^ (r % 8): no bank conflicts on either side)
// to be read in the products' layout.  (Loading that layout directly touches 16
// lines per load: 75 cycles of the L1 each against 17, 50.5 us against 35.6.)
//
// Where K is not a multiple of 512 the last j misses some classes: the groups
// past it have one chunk less, and the elements past K of a partly filled chunk
// are zeros, which leave a sum as it is (no sum is ever -0).  Rows past n or
// t read as zeros too and feed only outputs that are not stored.
template <int WB, int TB, int kEpi>
__global__ __launch_bounds__(512, 2) void gemm_exact_mfma_kernel(BatchedGemvParams p) {
  constexpr int kN = 16 * WB, kT = 16 * TB;
  constexpr int kRows = kN + kT;
  constexpr int kOps = kRows / 4;                      // loads per chunk: 4 rows each
  constexpr int kItems = WB * TB * 64;                 // f32x4 sums of the tile
  __shared__ __align__(128) char lds[8][kRows * 256];  // a wave's chunk each; at the end its sums
  static_assert(kItems * 16 <= kRows * 256, "a wave's sums fit its part of LDS");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int g = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ttiles = (p.t + kT - 1) / kT;
  // XCD x takes a contiguous run of (W tile, token tile) pairs, token tile
  // fastest, so the tokens' workgroups of a W tile share its rows in one L2.
  const int nwg = gridDim.x, xcd = blockIdx.x % kXcds;
  const int tile = xcd * (nwg / kXcds) + min(xcd, nwg % kXcds) + blockIdx.x / kXcds;
  const int n0 = (tile / ttiles) * kN, t0 = (tile % ttiles) * kT;

  const int K = p.k;
  const int nj = (K + 511) / 512;
  const int rem = K - 512 * (nj - 1);                  // elements of the last j (1..512)
  const int cnt = 64 * g < rem ? nj : nj - 1;          // this wave's chunks

  // Load i of a chunk: rows 4 i .. + 4 of the tile (W's, then X's), lane l row
  // l / 16's piece l % 16 (four elements), stored at piece (l % 16) ^ (row % 8).
  const i32x4 rw = buffer_rsrc_f16x4(p.w + (long long)n0 * K, (unsigned)min(p.n - n0, kN) * (unsigned)K * 2u);
  const i32x4 rx = buffer_rsrc_f16x4(p.x + (long long)t0 * p.ldx,
                                     (unsigned)(((long long)(min(p.t - t0, kT) - 1) * p.ldx + K) * 2));
  unsigned voff[kOps];
#pragma unroll
  for (int i = 0; i < kOps; ++i) {
    const unsigned row = 4 * (i < kN / 4 ? i : i - kN / 4) + (lane >> 4);
    voff[i] = row * (i < kN / 4 ? (unsigned)K : (unsigned)p.ldx) * 2u + 8u * (lane & 15);
  }
  f32x4 stage[kOps];
  auto load = [&](int j) {                             // chunk j, nothing past the last
    if (j >= cnt) return;
    const int so = (512 * j + 64 * g) * 2;
#pragma unroll
    for (int i = 0; i < kOps; ++i)
      stage[i] = raw_buffer_load_format4(i < kN / 4 ? rw : rx, (int)voff[i], so, 0);
  };
  char* const mine = lds[g];
  const int woff0 = (lane >> 4) * 256 + 16 * ((lane & 15) ^ (lane >> 4));        // even i: rows 0..3 of 8
  const int woff1 = (lane >> 4) * 256 + 16 * ((lane & 15) ^ (4 + (lane >> 4)));  // odd i: rows 4..7
  auto store = [&](int j) {
    // the last chunk's elements past K (the loads read what follows the row)
    if (j == nj - 1 && 64 * g + 4 * (lane & 15) >= rem) {
#pragma unroll
      for (int i = 0; i < kOps; ++i) stage[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int i = 0; i < kOps; ++i)
      *reinterpret_cast<f32x4*>(mine + ((i & 1) ? woff1 : woff0) + i * 1024) = stage[i];
  };

  const int fr = lane & 15, fg = lane >> 4;
  // row fr of block i, class 4 q + fg, half h: the block adds 4096 bytes, q 128
  const int roff0 = fr * 256 + 16 * ((2 * fg) ^ (fr & 7)), roff1 = fr * 256 + 16 * ((2 * fg + 1) ^ (fr & 7));
  typedef f32x4 Frags[WB + TB];
  auto read = [&](int s, Frags& f) {                   // quarter s = 2 q + h
#pragma unroll
    for (int i = 0; i < WB + TB; ++i)
      f[i] = *reinterpret_cast<const f32x4*>(mine + ((s & 1) ? roff1 : roff0) + i * 4096 + 128 * (s >> 1));
  };
  f32x16 acc[2][WB][TB];
  auto multiply = [&](const Frags& f, f32x16 (&c)[WB][TB], bool first) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < WB; ++i)
#pragma unroll
        for (int j = 0; j < TB; ++j)
          c[i][j] = __builtin_amdgcn_mfma_f32_16x16x1f32(f[i][e], f[WB + j][e],
                                                         first && e == 0 ? f32x16{} : c[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  Frags f0, f1;
  // Multiplies chunk j, in LDS and (quarter 0) f0, with chunk j + 1 on its way
  // to the registers; stores that over it once its last quarter is read (a
  // wave's LDS operations are served in order) and loads chunk j + 2.
  auto chunk = [&](int j, bool first) {
    read(1, f1);
    multiply(f0, acc[0], first);
    read(2, f0);
    multiply(f1, acc[0], false);
    read(3, f1);
    multiply(f0, acc[1], first);
    if (j + 1 < cnt) {
      store(j + 1);
      load(j + 2);
      read(0, f0);
    }
    multiply(f1, acc[1], false);
  };
  if (cnt > 0) {
    load(0);
    store(0);
    load(1);
    read(0, f0);
    chunk(0, true);
#pragma unroll 1
    for (int j = 1; j < cnt; ++j) chunk(j, false);
  }
  // blocks b of acc[q] are classes 8 g + 4 q + b: the tree's three lower levels
#pragma unroll
  for (int i = 0; i < WB; ++i)
#pragma unroll
    for (int j = 0; j < TB; ++j) {
      f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
      if (cnt > 0) {
        const f32x16 a = acc[0][i][j], b = acc[1][i][j];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          s[r] = ((a[r] + a[4 + r]) + (a[8 + r] + a[12 + r])) + ((b[r] + b[4 + r]) + (b[8 + r] + b[12 + r]));
      }
      *reinterpret_cast<f32x4*>(mine + ((i * TB + j) * 64 + lane) * 16) = s;
    }
  __syncthreads();

  // item (block, lane): rows n .. n + 3 of W for token t, four adjacent outputs
  const bool vec = ((reinterpret_cast<uintptr_t>(p.y) | reinterpret_cast<uintptr_t>(p.res)) & 7u) == 0 && p.ldy % 4 == 0;
  for (int it = tid; it < kItems; it += 512) {
    const int i = it / (64 * TB), j = it / 64 % TB;
    const int t = t0 + 16 * j + fr, n = n0 + 16 * i + 4 * fg;
    if (t >= p.t || n >= p.n) continue;
    f32x4 s[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) s[w] = *reinterpret_cast<const f32x4*>(lds[w] + it * 16);
    f16x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      v[r] = to_f16(((s[0][r] + s[1][r]) + (s[2][r] + s[3][r])) + ((s[4][r] + s[5][r]) + (s[6][r] + s[7][r])));
    _Float16* dst = reinterpret_cast<_Float16*>(p.y) + (long long)t * p.ldy + n;
    const _Float16* res = reinterpret_cast<const _Float16*>(p.res) + (long long)t * p.ldy + n;
    if (vec && n + 4 <= p.n) {
      if constexpr (kEpi == 1) {
        const f16x4 rv = *reinterpret_cast<const f16x4*>(res);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (_Float16)((float)rv[r] + (float)v[r]);
      }
      *reinterpret_cast<f16x4*>(dst) = v;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < p.n) dst[r] = kEpi == 1 ? (_Float16)((float)res[r] + (float)v[r]) : v[r];
    }
  }
}

template <int WB, int TB>
long long tiles_of(const BatchedGemvParams& p) {
  return (long long)((p.n + 16 * WB - 1) / (16 * WB)) * ((p.t + 16 * TB - 1) / (16 * TB));
}

template <int WB, int TB>
hipError_t launch(const BatchedGemvParams& p, int epi, hipStream_t stream) {
  const dim3 grid((unsigned)tiles_of<WB, TB>(p)), block(512);
  if (epi == 0)
    hipLaunchKernelGGL((gemm_exact_mfma_kernel<WB, TB, 0>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((gemm_exact_mfma_kernel<WB, TB, 1>), grid, block, 0, stream, p);
  return hipGetLastError();
}

}  // namespace

// The tile.  32 x 32 outputs have half the operand bytes per product of 16 x
// 16, but one workgroup per CU (250 VGPRs); 16 x 16 tiles run two per CU and
// leave fewer idle in the last round.  A round of 32 x 32 tiles takes as long
// as ~3.7 16 x 16 tiles per CU, whatever K (n = 6144, K = 2048: 11 us against
// 2.9 us per 256 tiles; 127 tokens 35.6 against 37.1 us, 100 tokens 35.1 and
// 33.9, 64 tokens 24.0 and 19.6; n = 2048, 127 tokens 12.9 and 14.2 us).
hipError_t launch_gemm_exact_mfma(const BatchedGemvParams& p, int epi, int cus, hipStream_t stream) {
  const long long rounds = (tiles_of<2, 2>(p) + cus - 1) / cus;
  if (27 * tiles_of<1, 1>(p) < 100 * rounds * cus) return launch<1, 1>(p, epi, stream);
  return launch<2, 2>(p, epi, stream);
}

}  // namespace qd
