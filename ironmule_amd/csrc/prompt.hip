// MI355X (gfx950) kernels for more than 32 activation rows (prompts, expert batches) and
// their C ABI (include/ironmule_prompt.h): activations packed into MFMA operand order, and a
// matrix product that reads the 4-bit weights as they are stored.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <string>

#include "../../include/ironmule_prompt.h"
#include "common.h"
#include "runtime.h"

namespace {

using namespace imq_dev;

using imq_rt::aligned;
using imq_rt::current_device;
using imq_rt::DeviceInfo;
using imq_rt::fail;
using imq_rt::ok;

typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;

// ------------------------------------------------------------ packed activations
//
// Rows are packed in blocks of 32, columns in chunks of four groups (256 columns).  A
// (block, chunk) is kChunkBytes: four groups of 4 KB, then 2 KB of group sums.
//   group    piece c (columns 8c .. 8c+7 of the group) of row m at c * 512 + m * 16, its eight
//            bf16 in the pair order of the unpacked nibbles (x0 x4 x1 x5 x2 x6 x3 x7): lane
//            (m, h) of an MFMA reads piece 4 h + j as its A operand of k-step j.
//   sums     X = the row's sum over the group, as three bf16 terms (hi + mid + lo = X to 24
//            bits): half (t, h) at (2 t + h) * 512, row m at m * 16, eight bf16
//            (X of groups 0..3, then -16 X of groups 0..3), of hi for (0, 0), mid for (0, 1),
//            lo for (1, 0) and zero for (1, 1): the A operands of two k-steps against
//            (biases of the four groups, scales of the four groups).
// A group holding a value that could overflow fp32 sums (|x| >= 2^96, infinities, NaN) has NaN
// for its sums: the product finds the row's outputs NaN and computes them value by value.
constexpr int kGroupBytes = 4096;
constexpr int kSumBytes = 2048;
constexpr int kChunkBytes = 4 * kGroupBytes + kSumBytes;
constexpr uint32_t kHuge = 0x6f80u;  // bf16 exponent field of 2^96

__device__ __forceinline__ uint32_t exponent_max(uint32_t u, uint32_t m) {
  const uint32_t lo = u & 0x7f80u, hi = (u >> 16) & 0x7f80u;
  m = m > lo ? m : lo;
  return m > hi ? m : hi;
}

// One row's group g (0..3 of its chunk) from eight lanes into the (block, chunk) at `to`: lane c
// (0..7) holds columns 8 c .. of the group in d.
__device__ __forceinline__ void emit_group(uint4 d, int c, int g, int row, char* to) {
  *reinterpret_cast<uint4*>(to + g * kGroupBytes + c * 512 + row * 16) = pair_order(d);
  uint32_t e = exponent_max(d.x, 0u);
  e = exponent_max(d.y, e);
  e = exponent_max(d.z, e);
  e = exponent_max(d.w, e);
  float s = e >= kHuge ? __uint_as_float(0x7fc00000u) : sum8(d);
  s += dpp<0xB1>(s);   // lanes ^ 1
  s += dpp<0x4E>(s);   // lanes ^ 2
  s += dpp<0x141>(s);  // the other four of the eight
  // lane t of the eight writes term t (hi, mid, lo, zero)
  const uint32_t hi = f32_to_bf16_bits(s);
  const float s1 = s - bf16_bits_to_f32(hi);
  const uint32_t mid = f32_to_bf16_bits(s1);
  const uint32_t lo = f32_to_bf16_bits(s1 - bf16_bits_to_f32(mid));
  const uint32_t term = c == 0 ? hi : c == 1 ? mid : c == 2 ? lo : 0u;
  if (c < 4) {
    uint16_t* const at = reinterpret_cast<uint16_t*>(to + 4 * kGroupBytes + c * 512 + row * 16) + g;
    at[0] = (uint16_t)term;
    at[4] = (uint16_t)(__float_as_uint(-16.0f * bf16_bits_to_f32(term)) >> 16);
  }
}

// One workgroup per (eight rows, chunk).  `src` (may be null): the x row of each packed row, -1
// for a row of zeros, and `expert` the expert of each tile of `tm` blocks, -1 for tiles not in
// use; without them packed row r is x row r, zeros past M.
__global__ __launch_bounds__(kThreads) void pack_rows_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                             const int32_t* __restrict__ src,
                                                             const int32_t* __restrict__ expert, int tm, int M, int K,
                                                             char* __restrict__ packed) {
  const int chunk = blockIdx.y, chunks = gridDim.y, block = blockIdx.x >> 2;
  const int l = threadIdx.x & 31, in = 8 * (blockIdx.x & 3) + (threadIdx.x >> 5);  // row of the block
  if (expert && expert[block / tm] < 0) return;
  const int col = 256 * chunk + 8 * l, r = 32 * block + in;
  const int64_t row = src ? src[r] : (r < M ? r : -1);
  uint4 d = make_uint4(0u, 0u, 0u, 0u);
  if (row >= 0 && col < K) d = *reinterpret_cast<const uint4*>(x + row * ldx + col);
  emit_group(d, l & 7, l >> 3, in, packed + ((int64_t)block * chunks + chunk) * kChunkBytes);
}

// ------------------------------------------------------------ the product
//
// y[m][n] = sum_g s[n][g] sum_k (16 + q) x + (b[n][g] - 16 s[n][g]) sum_k x over the groups g.
//
// A workgroup of four wavefronts computes 32 TM rows x 128 columns over a K-range of whole
// chunks; a wavefront all of the rows for 32 columns, on v_mfma_f32_32x32x16_bf16.
//   * The packed rows go memory -> LDS by the buffer loads' LDS path, group by group, into a
//     ring of four arrays, three groups ahead; the four wavefronts share them.
//   * Each wavefront's weights go straight to registers a chunk ahead: lane (n, h) loads 16
//     bytes per group, words 4h .. 4h+3 of its row, word 4h+j being its B operand of k-step j
//     as the exact bf16 values 16 + q.
//   * Per group each 32 x 32 tile takes four MFMAs from zero and 16 FMAs by the column's
//     scale; per chunk two more MFMAs of the rows' group sums against the four biases and
//     scales.  The products are exact and every sum is fp32.
// One barrier per group.  Within a wavefront the scaling of one tile, the LDS reads of the
// next and the unpacking of the next group's weights are issued between a tile's MFMAs.
//
// What bounds it: issue.  By the counters of a 512-token prompt's layer the MFMAs are busy 38% of
// gate/up's CU cycles (TM = 2, 1216 workgroups, 79 us) and 34% of down's (TM = 4, three K-ranges,
// 45.5 us), with no LDS bank conflicts; the 16 FMAs and 8 unpackings per four MFMAs overlap them only
// in part, and waves spend a quarter to half of their cycles waiting to issue.  Taking out the
// counted waits, the barriers or the distance to memory (every load from one line) changed a group
// by 3% or less.  Small launches add a start and an end: q/k/v (TM = 1) 39 us, o (160 workgroups) 36.
// 2048 x 4096 x 2560 60 us, 712 TFLOP/s; 8192 x 15360 x 3840 1338 us, 722.  Not faster: 64 x 64 per
// wavefront (half the LDS reads, twice the unpacking), eight wavefronts over 256 columns, one wait for
// a unit's four operands in place of one each (large launches 4% faster, 1024 x 9728 2% slower).
// Against imq_dequant and a library product (two conversions of the activations besides): 1024 x 9728
// x 2560 90 -> 80 us in fp16, 77 x 2560 x 9728 70.9 -> 26 us in fp32; from about 2048 rows over weights
// of 2500 rows and more that way is the faster one (4096 x 15360 x 3840 524 us, 613 here), at fp16's
// range and rounding.
struct ProductProblem {
  const uint32_t* w;
  const uint16_t* s;
  const uint16_t* b;
  void* y;
  int64_t ldy;    // with planes: the problem's first column in a plane
  int32_t N;
  int32_t tile0;  // first column tile of the launch
};

struct ProductArgs {
  ProductProblem p[IMQ_PROMPT_MAX_PROBLEMS];
  const char* packed;
  float* planes;          // fp32 partials (split, row, column of the launch), or null
  const int32_t* expert;  // per row tile: the expert of its rows, -1 none; null: one weight
  const int32_t* dest;    // per packed row: the output row, -1 none (with expert)
  int64_t plane_stride;   // elements between splits
  int64_t plane_ld;       // elements between rows of a plane
  int32_t count, M, G, chunks, blocks;
  int32_t row_tiles, col_tiles, splits, range;  // range: chunks per split
  int32_t y_f32;
  char* act;              // PAIR: the packed rows of silu(gate) * up
};

// A value every lane holds, in a scalar register.
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// s_waitcnt immediate that waits for vmcnt <= n and nothing else (gfx9 encoding)
constexpr int vmcnt_imm(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8); }

// Nibbles p and p + 4 of word u as the bf16 pair (16 + q_p, 16 + q_{p+4}), exact: q in
// mantissa bits 3..6 of 16.0.
__device__ __forceinline__ bf16x8_t nibbles16(uint32_t u, uint32_t magic) {
  const u32x4_t t = {((u << 3) & 0x00780078u) | magic, ((u >> 1) & 0x00780078u) | magic,
                     ((u >> 5) & 0x00780078u) | magic, ((u >> 9) & 0x00780078u) | magic};
  return __builtin_bit_cast(bf16x8_t, t);
}

constexpr int kColumns = 128;  // of a workgroup

// AL: G % 4 == 0 and 8-byte aligned scales and biases.  PAIR: the launch's two weights are gate
// and up; a workgroup takes the same 64 columns of both and writes bf16(silu(bf16(gate)) *
// bf16(up)) as packed rows, the operand of the down projection, in place of two outputs that
// another launch would read (512 x 2 x 9728: 20 MB written and read, and 12 us of that launch).
template <int TM, bool AL, bool PAIR>
__global__ __launch_bounds__(kThreads, 2) void product_kernel(ProductArgs a) {
  constexpr int kXB = TM;                      // row loads per wavefront and group
  constexpr int kSB = TM > 1 ? TM / 2 : 1;     // sum loads per wavefront and chunk
  constexpr int kSN = 2;                       // scale and bias loads per chunk, at least
  __shared__ __attribute__((aligned(16))) uint4 x0[TM * 256];
  __shared__ __attribute__((aligned(16))) uint4 x1[TM * 256];
  __shared__ __attribute__((aligned(16))) uint4 x2[TM * 256];
  __shared__ __attribute__((aligned(16))) uint4 x3[TM * 256];
  __shared__ __attribute__((aligned(16))) uint4 xsum[4 * kSB * 64];

  // Consecutive workgroups go to the XCDs in turn; each XCD takes a run of tiles in which
  // the row tiles of a column tile are neighbours, so that its weights stay in one L2.
  const int total = a.row_tiles * a.col_tiles * a.splits;
  const int per = (total + 7) >> 3;
  const int t = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (t >= total) return;
  // (divisions leave a uniform value in a vector register: taken back to scalars)
  const int cs = __builtin_amdgcn_readfirstlane(t / a.row_tiles), rt = t - cs * a.row_tiles;
  const int ct = __builtin_amdgcn_readfirstlane(cs / a.splits), split = cs - ct * a.splits;
  int expert = 0;
  if (a.expert) {
    expert = __builtin_amdgcn_readfirstlane(a.expert[rt]);
    if (expert < 0) return;
  }
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int pi = PAIR ? wave >> 1 : 0;
  if (!PAIR)
#pragma unroll
    for (int i = 1; i < IMQ_PROMPT_MAX_PROBLEMS; ++i)
      if (i < a.count && ct >= a.p[i].tile0) pi = i;
  const ProductProblem P = pi == 0 ? a.p[0] : pi == 1 ? a.p[1] : a.p[2];
  const int G = a.G, chunks = a.chunks, N = P.N;
  const int q0 = split * a.range, q1 = min(chunks, q0 + a.range);

  // this wavefront's columns: the problem's rows col0 .. of W.  Every load stays inside its
  // tensor: lanes past the last row read the last one, groups and blocks past the end the last.
  const int col0 = PAIR ? ct * (kColumns / 2) + (wave & 1) * 32 : (ct - P.tile0) * kColumns + wave * 32;
  const int rows = min(32, max(1, N - col0));
  const int64_t wrow = (int64_t)expert * N + min(col0, N - 1);
  const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(P.w + wrow * (8 * G), (uint32_t)rows * (uint32_t)(32 * G));
  const __amdgpu_buffer_rsrc_t sr = buffer_rsrc(P.s + wrow * G, (uint32_t)rows * (uint32_t)(2 * G));
  const __amdgpu_buffer_rsrc_t br = buffer_rsrc(P.b + wrow * G, (uint32_t)rows * (uint32_t)(2 * G));
  const uint32_t block_bytes = (uint32_t)chunks * kChunkBytes;
  const int nblocks = min(TM, a.blocks - rt * TM);
  const __amdgpu_buffer_rsrc_t xr =
      buffer_rsrc(a.packed + (int64_t)rt * TM * block_bytes, (uint32_t)nblocks * block_bytes);
  const uint32_t xoff = 16u * lane;
  uint32_t piece[kXB], sums[kSB];  // this wavefront's 1 KB pieces of a group, and of a chunk's sums
#pragma unroll
  for (int e = 0; e < kXB; ++e) {
    const int p = wave * kXB + e;
    piece[e] = __builtin_amdgcn_readfirstlane((uint32_t)min(p >> 2, nblocks - 1) * block_bytes + (uint32_t)(p & 3) * 1024u);
  }
#pragma unroll
  for (int e = 0; e < kSB; ++e) {
    const int p = wave * kSB + e;  // with one block two wavefronts fill a spare part
    sums[e] = __builtin_amdgcn_readfirstlane((uint32_t)min(p >> 1, nblocks - 1) * block_bytes +
                                             (uint32_t)(p & 1) * 1024u + 4 * kGroupBytes);
  }
  const uint32_t r0 = (uint32_t)min(n, rows - 1);
  const uint32_t woff = r0 * (uint32_t)(32 * G) + 16u * h, soff = r0 * (uint32_t)(2 * G);

  f32x16_t acc[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) acc[i] = f32x16_t{};
  uint4 wq[4], nwq[4];        // this and the next chunk's weights
  u32x2_t sc, bi, nsc, nbi;   // scales and biases
  const uint32_t magic = in_vgpr(0x41804180u);

  // a chunk's weights: the four loads of a lane share a cache line
  auto load_w = [&](int q, int i) {
    const uint32_t at = uniform(32u * (uint32_t)min(4 * q + i, G - 1));
    const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(wr, woff, at, 0);
    nwq[i] = make_uint4(v.x, v.y, v.z, v.w);
  };
  auto load_scales = [&](int q) {
    const int c = min(q, chunks - 1);
    if (AL) {
      nsc = __builtin_amdgcn_raw_buffer_load_b64(sr, soff, 8 * c, 0);
      nbi = __builtin_amdgcn_raw_buffer_load_b64(br, soff, 8 * c, 0);
    } else {  // rows of any alignment; groups past the row's end read zero
      uint32_t s4[4], b4[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t o = 4 * c + e < G ? soff + 2u * (uint32_t)(4 * c + e) : kPastBuffer;
        s4[e] = __builtin_amdgcn_raw_buffer_load_b16(sr, o, 0, 0);
        b4[e] = __builtin_amdgcn_raw_buffer_load_b16(br, o, 0, 0);
      }
      nsc = u32x2_t{s4[0] | (s4[1] << 16), s4[2] | (s4[3] << 16)};
      nbi = u32x2_t{b4[0] | (b4[1] << 16), b4[2] | (b4[3] << 16)};
    }
  };
  auto load_x = [&](int q, int i, int e, uint4* dst) {
    const uint32_t at =
        uniform(piece[e] + (uint32_t)min(q, q1 - 1) * kChunkBytes + (uint32_t)i * kGroupBytes);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        xr, (__attribute__((address_space(3))) void*)(dst + (wave * kXB + e) * 64), 16, xoff, at, 0, 0);
  };
  auto load_sums = [&](int q) {
#pragma unroll
    for (int e = 0; e < kSB; ++e) {
      const uint32_t at = uniform(sums[e] + (uint32_t)q * kChunkBytes);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          xr, (__attribute__((address_space(3))) void*)(xsum + (wave * kSB + e) * 64), 16, xoff, at, 0, 0);
    }
  };
  // The pipeline over units, a unit being one row tile of one group: its four MFMAs run while
  // the unit before it is scaled into its accumulator, the unit after it is read from LDS and
  // the next group's weights are unpacked.  Unit u of group i uses buffers (i TM + u) & 1.
  bf16x8_t xa[2][4], wb[2][4];
  f32x16_t p[2];
  float s[2];
  auto read_unit = [&](const uint4* xs, int m, bf16x8_t* dst) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[k] = __builtin_bit_cast(bf16x8_t, xs[m * 256 + (4 * h + k) * 32 + n]);
  };
  auto unpack = [&](const uint4& src, int k, bf16x8_t* dst) __attribute__((always_inline)) {
    dst[k] = nibbles16(k == 0 ? src.x : k == 1 ? src.y : k == 2 ? src.z : src.w, magic);
  };
  auto scale_unit = [&](float by, const f32x16_t& from, int m) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[m][e] = fmaf(by, from[e], acc[m][e]);
  };
  // group i (0..3, a constant at every call) of chunk q, its rows in xs, the next group's in
  // xnext; xfree is the array the group three ahead goes to
  auto group = [&](int i, const uint4* xs, const uint4* xnext, uint4* xfree, int q) __attribute__((always_inline)) {
    // this wavefront's part of the next group has landed (all that the last group did not
    // issue); past the barrier every wavefront's has, and nobody reads xfree
    __builtin_amdgcn_sched_barrier(0);
    if (i == 0 || i == 3)
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(kXB));
    else if (i == 1)
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(kXB + kSB + 4));
    else
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(kXB + kSN));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (i == 0) load_sums(q);
    if (i == 1) load_scales(q + 1);
    const uint32_t two = i < 2 ? sc.x : sc.y;
    s[i & 1] = __uint_as_float((i & 1) ? (two & 0xffff0000u) : (two << 16));
#pragma unroll
    for (int u = 0; u < TM; ++u) {
      const int at = (i * TM + u) & 1;
      // this unit's share of the loads, between the units' MFMAs: issued all at once they
      // held the wavefronts at the start of the group
      __builtin_amdgcn_sched_barrier(0);
      load_x(q + (i + 3) / 4, (i + 3) % 4, u, xfree);
      if (i == 0)
#pragma unroll
        for (int k = u * 4 / TM; k < (u + 1) * 4 / TM; ++k) load_w(q + 1, k);
      __builtin_amdgcn_sched_barrier(0);
      if (u + 1 < TM)
        read_unit(xs, u + 1, xa[at ^ 1]);
      else
        read_unit(xnext, 0, xa[at ^ 1]);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        p[at] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[at][k], wb[i & 1][k], k ? p[at] : f32x16_t{}, 0, 0, 0);
      if (u == 0)
        scale_unit(s[(i & 1) ^ 1], p[at ^ 1], TM - 1);
      else
        scale_unit(s[i & 1], p[at ^ 1], u - 1);
#pragma unroll
      for (int k = u * 4 / TM; k < (u + 1) * 4 / TM; ++k) unpack(i < 3 ? wq[(i + 1) & 3] : nwq[0], k, wb[(i & 1) ^ 1]);
      if (i == 3) {
        // the chunk's group sums against its biases and scales, between the tile's third and
        // fourth groups: one order for every row, so its bits do not depend on its place
        const bf16x8_t u0 = __builtin_bit_cast(bf16x8_t, xsum[u * 128 + h * 32 + n]);
        const bf16x8_t u1 = __builtin_bit_cast(bf16x8_t, xsum[u * 128 + 64 + h * 32 + n]);
        const bf16x8_t c = __builtin_bit_cast(bf16x8_t, u32x4_t{bi.x, bi.y, sc.x, sc.y});
        acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(u0, c, acc[u], 0, 0, 0);
        acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(u1, c, acc[u], 0, 0, 0);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA,
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one operand read,
        __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);  // six scalings and unpackings
      }
    }
    if (i == 3) {
      sc = nsc;
      bi = nbi;
#pragma unroll
      for (int k = 0; k < 4; ++k) wq[k] = nwq[k];
    }
  };

  load_scales(q0);
#pragma unroll
  for (int k = 0; k < 4; ++k) load_w(q0, k);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < kXB; ++e) load_x(q0, 0, e, x0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < kXB; ++e) load_x(q0, 1, e, x1);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < kXB; ++e) load_x(q0, 2, e, x2);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(kXB));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  read_unit(x0, 0, xa[0]);
  sc = nsc;
  bi = nbi;
  s[1] = 0.0f;
  p[1] = f32x16_t{};
#pragma unroll
  for (int k = 0; k < 4; ++k) wq[k] = nwq[k];
#pragma unroll
  for (int k = 0; k < 4; ++k) unpack(wq[0], k, wb[0]);
  for (int qv = q0; qv < q1; ++qv) {
    const int q = __builtin_amdgcn_readfirstlane(qv);
    group(0, x0, x1, x3, q);
    group(1, x1, x2, x0, q);
    group(2, x2, x3, x1, q);
    group(3, x3, x0, x2, q);
  }
  scale_unit(s[1], p[1], TM - 1);  // the range's last unit (4 TM is even)
  wait_vmem();  // the loads past the range's end, before the LDS is given up

  // Rows with values too large for the sums came out NaN: every output of the range by itself.
  const int col = col0 + n;
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    bool nan = false;
#pragma unroll
    for (int e = 0; e < 16; ++e) nan = nan || acc[m][e] != acc[m][e];
    if (__ballot(nan) == 0) continue;
    if (rt * TM + m >= a.blocks) continue;
#pragma unroll 1
    for (int r = 0; r < 32; ++r) {
      bool mine = false;
#pragma unroll
      for (int e = 0; e < 16; ++e)
        mine = mine || (8 * (e >> 2) + 4 * h + (e & 3) == r && acc[m][e] != acc[m][e]);
      if (__ballot(mine) == 0) continue;
      const char* const xrow = a.packed + (int64_t)(rt * TM + m) * block_bytes + r * 16;
      float v = 0.0f;
      if (col < N) {
        const int64_t row = wrow + n;
        for (int g = 4 * q0; g < min(4 * q1, G); ++g) {
          const float sg = bf16_bits_to_f32(P.s[row * G + g]), bg = bf16_bits_to_f32(P.b[row * G + g]);
          const char* const xg = xrow + (int64_t)(g >> 2) * kChunkBytes + (g & 3) * kGroupBytes;
          for (int k = 0; k < 4; ++k) {
            const uint32_t u = P.w[(row * G + g) * 8 + 4 * h + k];
            const uint4 d = *reinterpret_cast<const uint4*>(xg + (4 * h + k) * 512);
            const uint32_t pair[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              v = fmaf(fmaf(sg, (float)((u >> (4 * e)) & 15u), bg), bf16_bits_to_f32(pair[e] & 0xffffu), v);
              v = fmaf(fmaf(sg, (float)((u >> (4 * e + 16)) & 15u), bg), bf16_bits_to_f32(pair[e] >> 16), v);
            }
          }
        }
      }
      v = add_xor32(v);
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (8 * (e >> 2) + 4 * h + (e & 3) == r) acc[m][e] = v;
    }
  }

  if (PAIR) {
    // The gate's and the up's wavefront of the same columns exchange half their values through
    // x0 or x1, so that both apply the activation; the products as rows of 64 columns in x2, then
    // eight columns a lane into the packed rows.
    __syncthreads();
    float* const shared = reinterpret_cast<float*>((wave & 1) ? x1 : x0);
    const int keep = wave < 2 ? 0 : 8;  // the half of each tile's 16 values this wavefront computes
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        shared[((m * 2 + (wave < 2 ? 1 : 0)) * 8 + e) * 64 + lane] = wave < 2 ? acc[m][8 + e] : acc[m][e];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float mine = bf16_bits_to_f32(f32_to_bf16_bits(wave < 2 ? acc[m][e] : acc[m][8 + e]));
        const float other =
            bf16_bits_to_f32(f32_to_bf16_bits(shared[((m * 2 + (wave < 2 ? 0 : 1)) * 8 + e) * 64 + lane]));
        const float gate = wave < 2 ? mine : other, up = wave < 2 ? other : mine;
        const int at = keep + e, r = m * 32 + 8 * (at >> 2) + 4 * h + (at & 3);
        reinterpret_cast<uint16_t*>(x2)[r * 64 + (wave & 1) * 32 + n] =
            col < N ? f32_to_bf16_bits(gate / (1.0f + expf(-gate)) * up) : (uint16_t)0;
      }
    __syncthreads();
    const int act_chunks = (N + 255) >> 8;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int block = rt * TM + i, r = tid >> 3, c = tid & 7;
      if (block >= a.blocks) break;
      emit_group(x2[(i * 32 + r) * 8 + c], c, ct & 3, r, a.act + ((int64_t)block * act_chunks + (ct >> 2)) * kChunkBytes);
    }
    return;
  }

  // lane (n, h) holds column n of rows 8 (e / 4) + 4 h + e % 4
  if (col >= N) return;
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int r = (rt * TM + m) * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
      int64_t row = r < a.M ? r : -1;
      if (a.dest) row = r < a.blocks * 32 ? a.dest[r] : -1;
      if (row < 0) continue;
      if (a.planes)
        a.planes[split * a.plane_stride + row * a.plane_ld + P.ldy + col] = acc[m][e];
      else if (a.y_f32)
        static_cast<float*>(P.y)[row * P.ldy + col] = acc[m][e];
      else
        static_cast<uint16_t*>(P.y)[row * P.ldy + col] = f32_to_bf16_bits(acc[m][e]);
    }
}

// y = the splits' planes added in split order, for the launch's problems; four columns a
// thread.
struct SumArgs {
  ProductProblem p[IMQ_PROMPT_MAX_PROBLEMS];  // ldy: the output's; tile0: the plane's column
  const float* planes;
  int64_t plane_stride, plane_ld;
  int32_t count, M, splits, y_f32;
};

__global__ __launch_bounds__(kThreads) void sum_planes_kernel(SumArgs a) {
  const int64_t at = 4 * ((int64_t)blockIdx.x * kThreads + threadIdx.x);
  if (at >= a.plane_ld * a.M) return;
  const float* src = a.planes + at;
  float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int s = 0; s < a.splits; ++s) {
    const float4 u = *reinterpret_cast<const float4*>(src + s * a.plane_stride);
    v.x += u.x;
    v.y += u.y;
    v.z += u.z;
    v.w += u.w;
  }
  const int row = (int)(at / a.plane_ld), col = (int)(at - row * a.plane_ld);
  const float out[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < IMQ_PROMPT_MAX_PROBLEMS; ++i) {
    if (i >= a.count) break;
    const ProductProblem& P = a.p[i];
    const int c = col - P.tile0;  // planes' columns of a problem start at a multiple of four
    if (c < 0 || c >= P.N) continue;
    const int64_t o = row * P.ldy + c;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < P.N) {
        if (a.y_f32)
          static_cast<float*>(P.y)[o + e] = out[e];
        else
          static_cast<uint16_t*>(P.y)[o + e] = f32_to_bf16_bits(out[e]);
      }
  }
}

// ------------------------------------------------------------ rows sorted by expert

// One workgroup: counts the pairs of each expert, gives every expert whole tiles of `tile`
// packed rows, and writes each packed row's source row (pair / rows_per_x) and output row
// (the pair), -1 for the rows that fill up a tile, and each tile's expert, -1 past the last.
// An index below zero counts from the last expert; a pair whose index is outside the stack
// becomes a row of zeros.  The order of an expert's pairs within its tiles is not fixed, and no
// output depends on it: a row's sums involve no other row.  Bound by its own round trips (one
// CU, two passes over the indices).  With it 1024 pairs of 32 experts of 2560 x 768 take 41 us in
// place of 14.2 ms (every pair's expert dequantised to fp32 and one batched product).
constexpr int kSortThreads = 1024;
__global__ __launch_bounds__(kSortThreads) void sort_pairs_kernel(const int32_t* __restrict__ idx, int pairs,
                                                                  int experts, int rows_per_x, int tile, int tiles,
                                                                  int32_t* __restrict__ src,
                                                                  int32_t* __restrict__ dest,
                                                                  int32_t* __restrict__ tile_expert) {
  __shared__ int32_t count[IMQ_PROMPT_MAX_EXPERTS];
  __shared__ int32_t first[IMQ_PROMPT_MAX_EXPERTS];
  __shared__ int32_t scan[kSortThreads];
  const int tid = threadIdx.x;
  count[tid] = 0;
  __syncthreads();
  for (int p = tid; p < pairs; p += kSortThreads) {
    int e = idx[p];
    if (e < 0) e += experts;
    atomicAdd(&count[e >= 0 && e < experts ? e : 0], 1);
  }
  __syncthreads();
  const int mine = count[tid], need = (mine + tile - 1) / tile;
  scan[tid] = need;
  __syncthreads();
  for (int d = 1; d < kSortThreads; d <<= 1) {
    const int add = tid >= d ? scan[tid - d] : 0;
    __syncthreads();
    scan[tid] += add;
    __syncthreads();
  }
  const int tile0 = scan[tid] - need;
  first[tid] = tile0 * tile;
  for (int i = 0; i < need; ++i) tile_expert[tile0 + i] = tid;
  for (int r = mine; r < need * tile; ++r) {
    src[tile0 * tile + r] = -1;
    dest[tile0 * tile + r] = -1;
  }
  const int used = scan[kSortThreads - 1];
  for (int i = used + tid; i < tiles; i += kSortThreads) tile_expert[i] = -1;
  __syncthreads();
  for (int p = tid; p < pairs; p += kSortThreads) {
    int e = idx[p];
    if (e < 0) e += experts;
    const bool in = e >= 0 && e < experts;
    const int at = atomicAdd(&first[in ? e : 0], 1);
    src[at] = in ? p / rows_per_x : -1;
    dest[at] = p;
  }
}

// ------------------------------------------------------------ a prompt through a layer

constexpr int kD = 128;  // head dimension

// h[row] += bf16(the planes' sum) (planes may be null); with `weight`, x = bf16(rms_norm(h) *
// weight) packed.  A workgroup per packed row, thread t holding the 8-column pieces t, t + 256, ..
// (at most NP); rows past M are packed as zeros.  Consecutive workgroups go to the XCDs in turn:
// eight consecutive rows, which share the packed lines, go to one.  A wavefront per row and
// eight rows per workgroup took 14.5 us at 512 x 2560 with three planes, on 64 CUs.
template <int NP>
__global__ __launch_bounds__(kThreads) void norm_pack_kernel(float* __restrict__ h, const float* __restrict__ planes,
                                                             int splits, int64_t plane_stride,
                                                             const uint16_t* __restrict__ weight, int M, int dim,
                                                             float eps, int chunks, char* __restrict__ packed) {
  __shared__ float part[kThreads / 64];
  const int tid = threadIdx.x, b = blockIdx.x & 63;
  const int row = ((int)blockIdx.x & ~63) + (b & 7) * 8 + (b >> 3);
  if (row >= (M + 31) / 32 * 32) return;
  const bool live = row < M;
  float* const hr = h + (int64_t)row * dim;
  float v[NP][8];
  uint4 wv[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int col = 8 * (tid + kThreads * i);
    float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f), c = a;
    wv[i] = make_uint4(0u, 0u, 0u, 0u);
    if (col < dim && live) {
      a = *reinterpret_cast<const float4*>(hr + col);
      c = *reinterpret_cast<const float4*>(hr + col + 4);
      if (weight) wv[i] = *reinterpret_cast<const uint4*>(weight + col);
    }
    v[i][0] = a.x, v[i][1] = a.y, v[i][2] = a.z, v[i][3] = a.w;
    v[i][4] = c.x, v[i][5] = c.y, v[i][6] = c.z, v[i][7] = c.w;
  }
  if (planes && live) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int col = 8 * (tid + kThreads * i);
      if (col >= dim) continue;
      const float* const pr = planes + (int64_t)row * dim + col;
      float d[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
      for (int s0 = 0; s0 < splits; s0 += 4) {
        float4 p[4][2];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          p[s][0] = p[s][1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          if (s0 + s < splits) {
            p[s][0] = *reinterpret_cast<const float4*>(pr + (s0 + s) * plane_stride);
            p[s][1] = *reinterpret_cast<const float4*>(pr + (s0 + s) * plane_stride + 4);
          }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          d[0] += p[s][0].x, d[1] += p[s][0].y, d[2] += p[s][0].z, d[3] += p[s][0].w;
          d[4] += p[s][1].x, d[5] += p[s][1].y, d[6] += p[s][1].z, d[7] += p[s][1].w;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] += bf16_bits_to_f32(f32_to_bf16_bits(d[e]));
      *reinterpret_cast<float4*>(hr + col) = make_float4(v[i][0], v[i][1], v[i][2], v[i][3]);
      *reinterpret_cast<float4*>(hr + col + 4) = make_float4(v[i][4], v[i][5], v[i][6], v[i][7]);
    }
  }
  if (!weight) return;
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < NP; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(v[i][e], v[i][e], ss);
  ss = wave_sum(ss);
  if ((tid & 63) == 0) part[tid >> 6] = ss;
  __syncthreads();
  const float inv = 1.0f / sqrtf(((part[0] + part[1]) + (part[2] + part[3])) / (float)dim + eps);
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int piece = tid + kThreads * i;
    if (piece >= 32 * chunks) break;  // (whole groups of eight lanes)
    const uint32_t w[4] = {wv[i].x, wv[i].y, wv[i].z, wv[i].w};
    uint32_t out[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t lo = f32_to_bf16_bits(v[i][2 * e] * inv * bf16_bits_to_f32(w[e] & 0xffffu));
      const uint32_t hi = f32_to_bf16_bits(v[i][2 * e + 1] * inv * bf16_bits_to_f32(w[e] >> 16));
      out[e] = lo | (hi << 16);
    }
    uint4 d = make_uint4(out[0], out[1], out[2], out[3]);
    if (!live || 8 * piece >= dim) d = make_uint4(0u, 0u, 0u, 0u);
    emit_group(d, piece & 7, (piece >> 3) & 3, row & 31,
               packed + ((int64_t)(row >> 5) * chunks + (piece >> 5)) * kChunkBytes);
  }
}

// Per token and head: q and k heads get the per-head RMSNorm (rounded to bf16) and the
// non-interleaved rotary embedding at the token's position, angles in double; q in place, k and
// v into the slot's pools.  A workgroup per token, a wavefront per head at a time; lane i holds
// dimensions i and i + 64, the pair that turns together.  Four wavefronts, each with its own
// angles, took 10.9 us at 512 tokens of 48 heads.
constexpr int kRopeThreads = 1024;
__global__ __launch_bounds__(kRopeThreads) void prompt_rope_kernel(uint16_t* __restrict__ q,
                                                                   const uint16_t* __restrict__ k,
                                                                   const uint16_t* __restrict__ v,
                                                                   const uint16_t* __restrict__ q_norm,
                                                                   const uint16_t* __restrict__ k_norm,
                                                                   uint16_t* __restrict__ k_pool,
                                                                   uint16_t* __restrict__ v_pool, int Hq, int Hkv,
                                                                   int capacity, double log2_theta, float eps) {
  __shared__ float turn[2][64];
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave == 0) {
    double sn, cs;
    sincos((double)t * exp2(-(double)lane * (log2_theta / 64.0)), &sn, &cs);
    turn[0][lane] = (float)sn;
    turn[1][lane] = (float)cs;
  }
  const float qw[2] = {bf16_bits_to_f32(q_norm[lane]), bf16_bits_to_f32(q_norm[lane + 64])};
  const float kw[2] = {bf16_bits_to_f32(k_norm[lane]), bf16_bits_to_f32(k_norm[lane + 64])};
  __syncthreads();
  const float s = turn[0][lane], c = turn[1][lane];
  for (int hh = wave; hh < Hq + 2 * Hkv; hh += kRopeThreads / 64) {
    const bool is_q = hh < Hq, is_v = hh >= Hq + Hkv;
    const int head = is_q ? hh : is_v ? hh - Hq - Hkv : hh - Hq;
    const uint16_t* const src = is_q ? q + ((int64_t)t * Hq + head) * kD : (is_v ? v : k) + ((int64_t)t * Hkv + head) * kD;
    uint16_t* const dst = is_q ? q + ((int64_t)t * Hq + head) * kD
                               : (is_v ? v_pool : k_pool) + ((int64_t)head * capacity + t) * kD;
    if (is_v) {
      reinterpret_cast<uint32_t*>(dst)[lane] = reinterpret_cast<const uint32_t*>(src)[lane];
      continue;
    }
    float a = bf16_bits_to_f32(src[lane]), b = bf16_bits_to_f32(src[lane + 64]);
    const float inv = 1.0f / sqrtf(wave_sum(fmaf(a, a, b * b)) / (float)kD + eps);
    a = bf16_bits_to_f32(f32_to_bf16_bits(a * inv * (is_q ? qw[0] : kw[0])));
    b = bf16_bits_to_f32(f32_to_bf16_bits(b * inv * (is_q ? qw[1] : kw[1])));
    dst[lane] = f32_to_bf16_bits(a * c - b * s);
    dst[lane + 64] = f32_to_bf16_bits(a * s + b * c);
  }
}

// Causal attention of a prompt: out[t][head] = softmax(q . K / sqrt(128)) V over positions
// 0 .. t of one slot.
//
// A workgroup takes 64 queries of one head, a wavefront 16 of them; four wavefronts walk the even
// blocks of 64 keys and four the odd ones, each with the next block's K and V in flight in
// registers, and the two halves are merged at the end.  Scores are K Q^T on
// v_mfma_f32_16x16x32_bf16, so that a lane holds keys of one query: P^T is then the B operand
// of V^T P^T without leaving its lane (key order 4 g .. of two 16-key tiles per 32-key step).  P
// goes in as three bf16 terms that add up to its 24 bits, so P V keeps fp32's accuracy.  K lies
// in LDS in rows of swizzled 16-byte pieces, V transposed with padded rows; both twice.  Heavy
// query blocks, the last ones, start first.  The output goes out as packed rows, the operand of
// the o projection, zeros past T (and past an odd last head).
//
// Bound by the chain of key blocks at a few hundred tokens: 512 tokens of 32 heads are 256
// workgroups of at most eight blocks (21.7 us; 25.8 with four wavefronts on all of them and the
// next block's loads waited for in every turn, and 5.3 us of packing behind it).
constexpr int kQ = 64, kKeys = 64, kVRow = 2 * kKeys + 8;  // V^T row bytes: 16 mod 128 banks apart

__global__ __launch_bounds__(2 * kThreads) void prompt_attention_kernel(const uint16_t* __restrict__ q,
                                                                        const uint16_t* __restrict__ k_pool,
                                                                        const uint16_t* __restrict__ v_pool,
                                                                        char* __restrict__ packed, int T, int Hq,
                                                                        int Hkv, int capacity) {
  __shared__ __attribute__((aligned(16))) char kl[2][2][kKeys * 256];
  __shared__ __attribute__((aligned(16))) char vl[2][2][kD * kVRow];
  const int qblocks = gridDim.x / Hq;
  const int head = blockIdx.x % Hq, qb = qblocks - 1 - (int)blockIdx.x / Hq;
  const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tid = threadIdx.x & (kThreads - 1);
  const int lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4;
  const int64_t kv = (int64_t)(head / (Hq / Hkv)) * capacity * kD;
  const int query = qb * kQ + 16 * wave + n;
  const int last = T - 1;

  u32x4_t kr[4], va[2], vb[2];
  auto load = [&](int block) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = tid + kThreads * i;
      kr[i] = *reinterpret_cast<const u32x4_t*>(k_pool + kv + (int64_t)min(block * kKeys + (p >> 4), last) * kD + 8 * (p & 15));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int p = tid + kThreads * i, key = block * kKeys + 2 * (p >> 4);
      va[i] = *reinterpret_cast<const u32x4_t*>(v_pool + kv + (int64_t)min(key, last) * kD + 8 * (p & 15));
      vb[i] = *reinterpret_cast<const u32x4_t*>(v_pool + kv + (int64_t)min(key + 1, last) * kD + 8 * (p & 15));
    }
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = tid + kThreads * i, row = p >> 4;
      *reinterpret_cast<u32x4_t*>(kl[half][b] + row * 256 + (((p & 15) ^ (row & 15)) << 4)) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int p = tid + kThreads * i;
      char* const to = vl[half][b] + 8 * (p & 15) * kVRow + 4 * (p >> 4);
      const u32x4_t a = va[i], c = vb[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        *reinterpret_cast<uint32_t*>(to + (2 * e) * kVRow) = __builtin_amdgcn_perm(c[e], a[e], 0x05040100u);
        *reinterpret_cast<uint32_t*>(to + (2 * e + 1) * kVRow) = __builtin_amdgcn_perm(c[e], a[e], 0x07060302u);
      }
    }
  };

  constexpr float kLog2e = 1.44269504088896340736f, kScale = 0.08838834764831845f;  // 128^-1/2
  f32x4_t o[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) o[d] = f32x4_t{};
  float top = -INFINITY, sum = 0.0f;
  u32x4_t qr[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
    qr[t] = *reinterpret_cast<const u32x4_t*>(q + ((int64_t)min(query, last) * Hq + head) * kD + 32 * t + 8 * g);
  load(half);
  stage(0);
  bf16x8_t qf[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    // the queries are waited for here: a wait at their first use inside the loop would cover
    // the next block's loads, in every turn
    asm volatile("" : "+v"(qr[t]));
    qf[t] = __builtin_bit_cast(bf16x8_t, qr[t]);
  }
  __syncthreads();
  // Every turn loads and stages a block, past the last one rows that nothing uses: without
  // branches around them the loads stay in flight over the turn.
  for (int at = 0; 2 * at <= qb; ++at) {
    const int block = 2 * at + half;
    load(block + 2);
    if (block <= qb) {
      const char* const kb = kl[half][at & 1];
      const char* const vt = vl[half][at & 1];
      // four independent chains over the dimensions, and the first half of V on its way
      f32x4_t s[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) s[b] = f32x4_t{};
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(kb + (16 * b + n) * 256 + (((4 * t + g) ^ n) << 4));
          s[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf), qf[t], s[b], 0, 0, 0);
        }
      bf16x8_t vf[8];
      auto read_v = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < 8; ++d) {
          const char* const from = vt + (16 * d + n) * kVRow + 64 * j + 8 * g;
          const u32x2_t lo = *reinterpret_cast<const u32x2_t*>(from), hi = *reinterpret_cast<const u32x2_t*>(from + 32);
          vf[d] = __builtin_bit_cast(bf16x8_t, u32x4_t{lo.x, lo.y, hi.x, hi.y});
        }
      };
      read_v(0);
      float most = -INFINITY;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[b][e] *= kScale;
          if (block == qb && block * kKeys + 16 * b + 4 * g + e > query) s[b][e] = -INFINITY;
          most = fmaxf(most, s[b][e]);  // (a NaN score comes back through its exponential)
        }
      most = fmaxf(most, top);
      most = max_xor32(max_xor16(most));
      const float base = most == -INFINITY ? 0.0f : most;
      const float keep = exp2f((top - base) * kLog2e);
      top = most;
      sum *= keep;
      uint32_t p0[4][2], p1[4][2], p2[4][2];  // the three terms, two keys a word
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          uint32_t w[2][3];
#pragma unroll
          for (int z = 0; z < 2; ++z) {
            const float v = exp2f((s[b][e + z] - base) * kLog2e);
            sum += v;
            w[z][0] = __float_as_uint(v);
            const float r = v - __uint_as_float(w[z][0] & 0xffff0000u);
            w[z][1] = __float_as_uint(r);
            w[z][2] = __float_as_uint(r - __uint_as_float(w[z][1] & 0xffff0000u));
          }
          p0[b][e >> 1] = __builtin_amdgcn_perm(w[1][0], w[0][0], 0x07060302u);
          p1[b][e >> 1] = __builtin_amdgcn_perm(w[1][1], w[0][1], 0x07060302u);
          p2[b][e >> 1] = __builtin_amdgcn_perm(w[1][2], w[0][2], 0x07060302u);
        }
#pragma unroll
      for (int d = 0; d < 8; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[d][e] *= keep;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (j) read_v(1);
        const u32x4_t term[3] = {{p0[2 * j][0], p0[2 * j][1], p0[2 * j + 1][0], p0[2 * j + 1][1]},
                                 {p1[2 * j][0], p1[2 * j][1], p1[2 * j + 1][0], p1[2 * j + 1][1]},
                                 {p2[2 * j][0], p2[2 * j][1], p2[2 * j + 1][0], p2[2 * j + 1][1]}};
#pragma unroll
        for (int t = 0; t < 3; ++t)  // eight independent chains over the terms
#pragma unroll
          for (int d = 0; d < 8; ++d)
            o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[d], __builtin_bit_cast(bf16x8_t, term[t]), o[d], 0, 0, 0);
      }
    }
    stage((at + 1) & 1);
    __syncthreads();
  }
  sum = add_xor32(add_xor16(sum));

  // the odd half's state to the even half's lanes
  float* const state = reinterpret_cast<float*>(vl[0][0]);  // 34 floats a lane, 34 KB of the 68
  if (half) {
    state[tid] = top;
    state[kThreads + tid] = sum;
#pragma unroll
    for (int d = 0; d < 8; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e) state[(2 + 4 * d + e) * kThreads + tid] = o[d][e];
  }
  __syncthreads();
  uint16_t* const rows = reinterpret_cast<uint16_t*>(kl[0][0]);  // 64 x 128
  if (!half) {
    const float other = state[tid], most = fmaxf(top, other), base = most == -INFINITY ? 0.0f : most;
    const float mine = exp2f((top - base) * kLog2e), theirs = exp2f((other - base) * kLog2e);
    const float total = sum * mine + state[kThreads + tid] * theirs;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        w[e] = f32_to_bf16_bits((o[d][e] * mine + state[(2 + 4 * d + e) * kThreads + tid] * theirs) / total);
      const u32x2_t four = {w[0] | (w[1] << 16), w[2] | (w[3] << 16)};
      *reinterpret_cast<u32x2_t*>(rows + (16 * wave + n) * kD + 16 * d + 4 * g) = query <= last ? four : u32x2_t{};
    }
  }
  __syncthreads();
  const int chunks = (Hq + 1) >> 1, blocks = (T + 31) >> 5;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = threadIdx.x + 2 * kThreads * i, r = p >> 4, c = p & 15, row = qb * kQ + r;
    if (row >= 32 * blocks) continue;  // (whole groups of eight lanes)
    char* const to = packed + ((int64_t)(row >> 5) * chunks + (head >> 1)) * kChunkBytes;
    const uint4 d = *reinterpret_cast<const uint4*>(rows + r * kD + 8 * c);
    emit_group(d, c & 7, 2 * (head & 1) + (c >> 3), row & 31, to);
    if (head == Hq - 1 && !(head & 1)) emit_group(make_uint4(0u, 0u, 0u, 0u), c & 7, 2 + (c >> 3), row & 31, to);
  }
}

// ------------------------------------------------------------ host side

int ceil_div(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }
size_t round_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

struct Plan {
  int tm, splits, range;  // 32-row blocks of a tile, K-ranges, chunks per range
  int row_tiles, col_tiles;
};

int column_tiles(const int32_t* N, int count) {
  int tiles = 0;
  for (int i = 0; i < count; ++i) tiles += ceil_div(N[i], kColumns);
  return tiles;
}

// The tile height and the K-ranges with the least expected time.  Measured at K = 2560 (40
// groups) over 32 to 2048 workgroups, a launch takes about 14 / 11 / 9 us, and per group and
// workgroup of the busiest CU 0.56 / 0.31 / 0.20 us, with tiles of 128 / 64 / 32 rows: tall
// tiles reuse the weights, short ones fill the CUs.  K-ranges add the planes' traffic (about
// 4 TB/s each way) and the launch that adds them; a layer's o and down are charged both too, though
// norm_pack_kernel adds their planes.  Predicted / traced for 512 tokens of 2560 hidden: q/k/v 33 /
// 39 us, o 31 / 36, gate/up 73 / 79, down in three ranges 56 / 45.
Plan plan_product(const int32_t* N, int count, int M, int K, int cus, int max_splits = 8) {
  const int chunks = ceil_div(K, 256), col_tiles = column_tiles(N, count);
  double columns = 0.0, best = 0.0;
  for (int i = 0; i < count; ++i) columns += N[i];
  Plan plan;
  plan.tm = 0;
  for (int tm = 4; tm >= 1; tm >>= 1) {
    const double start = tm == 4 ? 14.0 : tm == 2 ? 11.0 : 9.0, group = tm == 4 ? 0.56 : tm == 2 ? 0.31 : 0.20;
    const int row_tiles = ceil_div(M, 32 * tm);
    for (int splits = 1; splits <= max_splits && splits <= chunks; ++splits) {
      const int range = ceil_div(chunks, splits);
      if (ceil_div(chunks, range) != splits) continue;
      double us = start + group * 4.0 * range * ceil_div((int64_t)row_tiles * col_tiles * splits, cus);
      if (splits > 1) us += 5.0 + splits * (double)M * columns * 8.0 / 4e6;
      if (plan.tm && us >= best) continue;
      best = us;
      plan = Plan{tm, splits, range, row_tiles, col_tiles};
    }
  }
  return plan;
}

// Tiles for rows sorted by expert: at most pairs / (32 tm) full ones and a part-full one per
// expert.  Tiles of 32 rows while the experts used get up to 28 pairs on average, mostly one tile
// each, or while the tiles to expect (half of one part-full per expert) make at most three
// workgroups per CU; 64 beyond, where the weights read twice count for more than the rows of zeros.
// 32 / 64 / 128 rows, us, at pairs per expert: 32 experts of 2560 x 768 at 20 27.4 / 35.2 / 67.8, at 32
// 39.9 / 36.6 / 65.9, at 256 127 / 115 / 146; 8 of 2048 x 2048 at 64 33.5 / 36.1 / 46.0, at 256 69.9 /
// 59.3 / 68.4, at 4000 664 / 531 / 544; 64 of 512 x 1024 at 32 30.9 / 39.0 / 59.7, at 96 53.1 / 55.2 /
// 64.4.  Over 117 such points of ten stacks the choice is at most 13% above the best of the
// three, 0.7% on average; 128 rows are the best of none.
struct ExpertPlan {
  int tm, tiles, blocks;
};

ExpertPlan expert_tiles(int experts, int pairs, int tm) {
  const int tiles = pairs / (32 * tm) + std::min(experts, pairs);
  return ExpertPlan{tm, tiles, tiles * tm};
}

ExpertPlan plan_experts(int experts, int pairs, int N, int cus) {
  const int64_t used = std::min(experts, pairs), columns = ceil_div(N, kColumns);
  const bool small = pairs <= 28 * used || (pairs / 32 + used / 2) * columns <= 3 * (int64_t)cus;
  return expert_tiles(experts, pairs, small ? 1 : 2);
}

size_t packed_bytes(int64_t blocks, int K) { return (size_t)blocks * ceil_div(K, 256) * kChunkBytes; }

void pack_rows(const uint16_t* x, int64_t ldx, const int32_t* src, const int32_t* expert, int tm, int M,
               int64_t blocks, int K, void* packed, hipStream_t stream) {
  hipLaunchKernelGGL(pack_rows_kernel, dim3((uint32_t)blocks * 4, ceil_div(K, 256)), dim3(kThreads), 0, stream, x, ldx,
                     src, expert, tm, M, K, static_cast<char*>(packed));
}

template <int TM>
void launch_product(const ProductArgs& a, bool al, uint32_t grid, hipStream_t stream) {
  if (a.act && al)
    hipLaunchKernelGGL((product_kernel<TM, true, true>), dim3(grid), dim3(kThreads), 0, stream, a);
  else if (a.act)
    hipLaunchKernelGGL((product_kernel<TM, false, true>), dim3(grid), dim3(kThreads), 0, stream, a);
  else if (al)
    hipLaunchKernelGGL((product_kernel<TM, true, false>), dim3(grid), dim3(kThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((product_kernel<TM, false, false>), dim3(grid), dim3(kThreads), 0, stream, a);
}

// Fills the shape fields and launches; p[], planes and the expert tables are the caller's.
int32_t run_product(ProductArgs& a, const Plan& p, const void* packed, int64_t blocks, int M, int K,
                    hipStream_t stream) {
  const int chunks = ceil_div(K, 256);
  a.packed = static_cast<const char*>(packed);
  a.M = M;
  a.G = K / 64;
  a.chunks = chunks;
  a.blocks = (int32_t)blocks;
  a.row_tiles = p.row_tiles;
  a.col_tiles = p.col_tiles;
  a.splits = p.splits;
  a.range = p.range;
  bool al = a.G % 4 == 0;
  for (int i = 0; i < a.count; ++i) al = al && aligned(a.p[i].s, 8) && aligned(a.p[i].b, 8);
  const uint32_t grid = 8u * (uint32_t)ceil_div((int64_t)p.row_tiles * p.col_tiles * p.splits, 8);
  if (p.tm == 4)
    launch_product<4>(a, al, grid, stream);
  else if (p.tm == 2)
    launch_product<2>(a, al, grid, stream);
  else
    launch_product<1>(a, al, grid, stream);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(IMQ_ELAUNCH, std::string("product launch failed: ") + hipGetErrorString(e));
  return ok();
}

int32_t check_weight(const uint32_t* w, const uint16_t* s, const uint16_t* b, int32_t N, int32_t K,
                     int32_t group_size, int32_t bits) {
  if (bits != 4) return fail(IMQ_EUNSUPPORTED, "only 4-bit weights are supported");
  if (group_size != 64) return fail(IMQ_EUNSUPPORTED, "only group size 64 is supported");
  if (N < 1) return fail(IMQ_EINVAL, "N must be >= 1");
  if (K < 64 || K % 64 != 0) return fail(IMQ_EINVAL, "K must be a positive multiple of 64");
  if (K > IMQ_PROMPT_MAX_K) return fail(IMQ_EUNSUPPORTED, "K too large");
  if (!w || !s || !b) return fail(IMQ_EINVAL, "w, scales and biases must be non-null");
  if (!aligned(w, 16)) return fail(IMQ_EINVAL, "w must be 16-byte aligned");
  if (!aligned(s, 2) || !aligned(b, 2)) return fail(IMQ_EINVAL, "scales/biases must be 2-byte aligned");
  return IMQ_OK;
}

// Columns of the launch's planes: each problem's, from a multiple of four.
int64_t plane_columns(const int32_t* N, int count) {
  int64_t cols = 0;
  for (int i = 0; i < count; ++i) cols += round_up(N[i], 4);
  return cols;
}

int32_t check_product(const imq_problem* p, int32_t count, int32_t M, int32_t group_size, int32_t bits,
                      int32_t y_dtype, const void* packed, int32_t* N, int32_t* K) {
  if (!p || count < 1) return fail(IMQ_EINVAL, "at least one problem");
  if (count > IMQ_PROMPT_MAX_PROBLEMS) return fail(IMQ_EUNSUPPORTED, "too many problems");
  if (M < 1 || M > IMQ_PROMPT_MAX_ROWS) return fail(IMQ_EINVAL, "M out of range");
  if (y_dtype != IMQ_BF16 && y_dtype != IMQ_F32) return fail(IMQ_EINVAL, "y_dtype must be bf16 or fp32");
  if (!packed || !aligned(packed, 16)) return fail(IMQ_EINVAL, "packed rows must be non-null and 16-byte aligned");
  for (int i = 0; i < count; ++i) {
    const int32_t code = check_weight(p[i].w, p[i].scales, p[i].biases, p[i].N, p[i].K, group_size, bits);
    if (code != IMQ_OK) return code;
    if (p[i].K != p[0].K) return fail(IMQ_EINVAL, "the problems of one call share K");
    if (!p[i].y || !aligned(p[i].y, y_dtype == IMQ_F32 ? 4 : 2)) return fail(IMQ_EINVAL, "y is null or misaligned");
    if (p[i].ldy < p[i].N) return fail(IMQ_EINVAL, "ldy must be >= N");
    N[i] = p[i].N;
  }
  *K = p[0].K;
  return IMQ_OK;
}

// y = x W^T as the plan's fp32 planes (one where it does not split): the residual add takes them.
int32_t product_planes(const imq_qweight& w, const void* packed, int M, int N, int K, float* planes, int cus,
                       int* splits, hipStream_t stream) {
  const int32_t n = N;
  const Plan plan = plan_product(&n, 1, M, K, cus);
  ProductArgs a;
  memset(&a, 0, sizeof(a));
  a.p[0] = ProductProblem{w.w, w.scales, w.biases, nullptr, 0, N, 0};
  a.count = 1;
  a.planes = planes;
  a.plane_ld = N;
  a.plane_stride = (int64_t)M * N;
  *splits = plan.splits;
  return run_product(a, plan, packed, ceil_div(M, 32), M, K, stream);
}

void norm_pack(float* h, const float* planes, int splits, int64_t stride, const uint16_t* weight, int M, int dim,
               float eps, void* packed, hipStream_t stream) {
  const int chunks = ceil_div(dim, 256);
  char* const to = static_cast<char*>(packed);
  const dim3 grid(64 * ceil_div(M, 64)), threads(kThreads);
  const int pieces = ceil_div(32 * chunks, kThreads);
  if (pieces <= 1)
    hipLaunchKernelGGL(norm_pack_kernel<1>, grid, threads, 0, stream, h, planes, splits, stride, weight, M, dim, eps, chunks, to);
  else if (pieces <= 2)
    hipLaunchKernelGGL(norm_pack_kernel<2>, grid, threads, 0, stream, h, planes, splits, stride, weight, M, dim, eps, chunks, to);
  else
    hipLaunchKernelGGL(norm_pack_kernel<4>, grid, threads, 0, stream, h, planes, splits, stride, weight, M, dim, eps, chunks, to);
}

// The parts of a prompt's workspace, each 256-byte aligned.
struct LayerSpace {
  size_t x, attn, act, q, k, v, planes, bytes;
};

int32_t check_shape(const imq_prompt_shape* s) {
  if (!s) return fail(IMQ_EINVAL, "the shape is null");
  if (s->tokens < 1 || s->tokens > IMQ_PROMPT_MAX_ROWS) return fail(IMQ_EINVAL, "tokens out of range");
  if (s->heads < 1 || s->kv_heads < 1 || s->heads % s->kv_heads) return fail(IMQ_EINVAL, "need kv_heads >= 1 dividing heads");
  if (s->heads > 1024) return fail(IMQ_EUNSUPPORTED, "too many heads");
  if (s->hidden < 64 || s->hidden % 64 || s->intermediate < 64 || s->intermediate % 64)
    return fail(IMQ_EINVAL, "hidden and intermediate must be positive multiples of 64");
  if (s->hidden > 8192 || s->intermediate > IMQ_PROMPT_MAX_K) return fail(IMQ_EUNSUPPORTED, "hidden or intermediate too large");
  if (s->capacity < s->tokens) return fail(IMQ_EINVAL, "the prompt does not fit the capacity");
  if (s->slot < 0 || s->slot >= s->num_slots) return fail(IMQ_EINVAL, "slot out of range");
  if (!(s->eps >= 0.0f) || !(s->theta > 1.0)) return fail(IMQ_EINVAL, "eps must be >= 0 and theta > 1");
  return IMQ_OK;
}

LayerSpace layer_space(const imq_prompt_shape& s, int cus) {
  const int T = s.tokens, blocks = ceil_div(T, 32), qd = s.heads * kD, kd = s.kv_heads * kD;
  const int32_t n = s.hidden;
  const int so = plan_product(&n, 1, T, qd, cus).splits, sd = plan_product(&n, 1, T, s.intermediate, cus).splits;
  LayerSpace l;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t here = at;
    at += round_up(bytes, 256);
    return here;
  };
  l.planes = take((size_t)(so > sd ? so : sd) * T * s.hidden * 4);
  l.x = take(packed_bytes(blocks, s.hidden));
  l.attn = take(packed_bytes(blocks, qd));
  l.act = take(packed_bytes(blocks, s.intermediate));
  l.q = take((size_t)T * qd * 2);
  l.k = take((size_t)T * kd * 2);
  l.v = take((size_t)T * kd * 2);
  l.bytes = at;
  return l;
}

int32_t launched(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(IMQ_ELAUNCH, std::string(what) + " launch failed: " + hipGetErrorString(e));
  return ok();
}

}  // namespace

extern "C" {

size_t imq_prompt_layer_workspace(const imq_prompt_shape* shape) {
  int32_t code;
  if (check_shape(shape) != IMQ_OK) return 0;
  const DeviceInfo* dev = current_device(&code);
  return dev ? layer_space(*shape, dev->cu_count).bytes : 0;
}

int32_t imq_prompt_layer(const imq_step_layer* layer, const imq_prompt_shape* shape, float* h, int32_t first,
                         void* workspace, size_t workspace_bytes, void* stream) {
  int32_t code = check_shape(shape);
  if (code != IMQ_OK) return code;
  if (!layer || !h || !workspace) return fail(IMQ_EINVAL, "layer, h and workspace must be non-null");
  if (!aligned(h, 16) || !aligned(workspace, 256)) return fail(IMQ_EINVAL, "h must be 16-byte aligned, the workspace 256-byte");
  const imq_prompt_shape& s = *shape;
  const int T = s.tokens, blocks = ceil_div(T, 32), qd = s.heads * kD, kd = s.kv_heads * kD;
  const imq_qweight* const ws[7] = {&layer->q, &layer->k, &layer->v, &layer->o, &layer->gate, &layer->up, &layer->down};
  const int32_t ns[7] = {qd, kd, kd, s.hidden, s.intermediate, s.intermediate, s.hidden};
  const int32_t ks[7] = {s.hidden, s.hidden, s.hidden, qd, s.hidden, s.hidden, s.intermediate};
  for (int i = 0; i < 7; ++i)
    if ((code = check_weight(ws[i]->w, ws[i]->scales, ws[i]->biases, ns[i], ks[i], 64, 4)) != IMQ_OK) return code;
  if (!layer->input_norm || !layer->post_norm || !layer->q_norm || !layer->k_norm || !layer->k_pool || !layer->v_pool)
    return fail(IMQ_EINVAL, "null norm weight or pool");
  if (!aligned(layer->input_norm, 16) || !aligned(layer->post_norm, 16) || !aligned(layer->k_pool, 16) ||
      !aligned(layer->v_pool, 16))
    return fail(IMQ_EINVAL, "norm weights and pools must be 16-byte aligned");
  const DeviceInfo* dev = current_device(&code);
  if (!dev) return code;
  const LayerSpace l = layer_space(s, dev->cu_count);
  if (workspace_bytes < l.bytes) return fail(IMQ_EINVAL, "the workspace is too small");
  char* const at = static_cast<char*>(workspace);
  float* const planes = reinterpret_cast<float*>(at + l.planes);
  uint16_t *const q = reinterpret_cast<uint16_t*>(at + l.q), *const k = reinterpret_cast<uint16_t*>(at + l.k);
  uint16_t* const v = reinterpret_cast<uint16_t*>(at + l.v);
  const int64_t pool = (int64_t)s.slot * s.kv_heads * s.capacity * kD;
  hipStream_t st = static_cast<hipStream_t>(stream);

  const int32_t n = s.hidden;
  int splits = plan_product(&n, 1, T, s.intermediate, dev->cu_count).splits;  // of the layer before
  norm_pack(h, first ? nullptr : planes, splits, (int64_t)T * s.hidden, layer->input_norm, T, s.hidden, s.eps, at + l.x, st);
  ProductArgs a;
  memset(&a, 0, sizeof(a));
  uint16_t* const qkv[3] = {q, k, v};
  int tile0 = 0;
  for (int i = 0; i < 3; ++i) {
    a.p[i] = ProductProblem{ws[i]->w, ws[i]->scales, ws[i]->biases, qkv[i], ns[i], ns[i], tile0};
    tile0 += ceil_div(ns[i], kColumns);
  }
  a.count = 3;
  const Plan three = plan_product(ns, 3, T, s.hidden, dev->cu_count, 1);
  if ((code = run_product(a, three, at + l.x, blocks, T, s.hidden, st)) != IMQ_OK) return code;
  hipLaunchKernelGGL(prompt_rope_kernel, dim3(T), dim3(kRopeThreads), 0, st, q, k, v, layer->q_norm, layer->k_norm,
                     layer->k_pool + pool, layer->v_pool + pool, s.heads, s.kv_heads, s.capacity,
                     log2(s.theta), s.eps);
  hipLaunchKernelGGL(prompt_attention_kernel, dim3(ceil_div(T, kQ) * s.heads), dim3(2 * kThreads), 0, st, q,
                     layer->k_pool + pool, layer->v_pool + pool, at + l.attn, T, s.heads, s.kv_heads, s.capacity);
  if ((code = product_planes(layer->o, at + l.attn, T, s.hidden, qd, planes, dev->cu_count, &splits, st)) != IMQ_OK)
    return code;
  norm_pack(h, planes, splits, (int64_t)T * s.hidden, layer->post_norm, T, s.hidden, s.eps, at + l.x, st);
  memset(&a, 0, sizeof(a));
  for (int i = 0; i < 2; ++i)
    a.p[i] = ProductProblem{ws[4 + i]->w, ws[4 + i]->scales, ws[4 + i]->biases, nullptr, 0, s.intermediate, 0};
  a.count = 2;
  a.act = at + l.act;
  // a column tile per group of act, up to whole chunks (the last ones, past N, are zeros)
  Plan two = plan_product(ns + 4, 2, T, s.hidden, dev->cu_count, 1);
  two.col_tiles = 4 * ceil_div(s.intermediate, 256);
  if ((code = run_product(a, two, at + l.x, blocks, T, s.hidden, st)) != IMQ_OK) return code;
  if ((code = product_planes(layer->down, at + l.act, T, s.hidden, s.intermediate, planes, dev->cu_count, &splits, st)) != IMQ_OK)
    return code;
  return launched("prompt layer");
}

int32_t imq_prompt_finish(const imq_prompt_shape* shape, float* h, int32_t rows, void* workspace,
                          size_t workspace_bytes, void* stream) {
  int32_t code = check_shape(shape);
  if (code != IMQ_OK) return code;
  if (!h || !workspace || !aligned(h, 16) || !aligned(workspace, 256)) return fail(IMQ_EINVAL, "h or workspace null or misaligned");
  if (rows < 1 || rows > shape->tokens) return fail(IMQ_EINVAL, "rows must be 1 .. tokens");
  const DeviceInfo* dev = current_device(&code);
  if (!dev) return code;
  const LayerSpace l = layer_space(*shape, dev->cu_count);
  if (workspace_bytes < l.bytes) return fail(IMQ_EINVAL, "the workspace is too small");
  const int32_t n = shape->hidden;
  const int64_t stride = (int64_t)shape->tokens * n, skip = (int64_t)(shape->tokens - rows) * n;
  const int splits = plan_product(&n, 1, shape->tokens, shape->intermediate, dev->cu_count).splits;
  const float* const planes = reinterpret_cast<const float*>(static_cast<char*>(workspace) + l.planes);
  norm_pack(h + skip, planes + skip, splits, stride, nullptr, rows, n, 0.0f, workspace, static_cast<hipStream_t>(stream));
  return launched("prompt finish");
}

size_t imq_prompt_packed_bytes(int32_t M, int32_t K) {
  if (M < 1 || M > IMQ_PROMPT_MAX_ROWS || K < 64 || K % 64 || K > IMQ_PROMPT_MAX_K) return 0;
  return packed_bytes(ceil_div(M, 32), K);
}

int32_t imq_prompt_pack(const uint16_t* x, int64_t ldx, int32_t M, int32_t K, void* packed, void* stream) {
  if (!x || !packed) return fail(IMQ_EINVAL, "x and packed must be non-null");
  if (M < 1 || M > IMQ_PROMPT_MAX_ROWS) return fail(IMQ_EINVAL, "M out of range");
  if (K < 64 || K % 64 || K > IMQ_PROMPT_MAX_K) return fail(IMQ_EINVAL, "K must be a multiple of 64 in range");
  if (ldx < K || ldx % 8) return fail(IMQ_EINVAL, "ldx must be >= K and a multiple of 8");
  if (!aligned(x, 16) || !aligned(packed, 16)) return fail(IMQ_EINVAL, "x and packed must be 16-byte aligned");
  int32_t code;
  if (!current_device(&code)) return code;
  pack_rows(x, ldx, nullptr, nullptr, 1, M, ceil_div(M, 32), K, packed, static_cast<hipStream_t>(stream));
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(IMQ_ELAUNCH, std::string("pack launch failed: ") + hipGetErrorString(e));
  return ok();
}

size_t imq_prompt_product_workspace(const imq_problem* p, int32_t count, int32_t M) {
  if (!p || count < 1 || count > IMQ_PROMPT_MAX_PROBLEMS || M < 1) return 0;
  int32_t code, N[IMQ_PROMPT_MAX_PROBLEMS];
  const DeviceInfo* dev = current_device(&code);
  if (!dev) return 0;
  for (int i = 0; i < count; ++i) N[i] = p[i].N;
  const Plan plan = plan_product(N, count, M, p[0].K, dev->cu_count);
  return plan.splits > 1 ? (size_t)plan.splits * M * plane_columns(N, count) * 4 : 0;
}

int32_t imq_prompt_product(const imq_problem* p, int32_t count, const void* packed, int32_t M, int32_t group_size,
                           int32_t bits, int32_t y_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  int32_t N[IMQ_PROMPT_MAX_PROBLEMS], K = 0;
  int32_t code = check_product(p, count, M, group_size, bits, y_dtype, packed, N, &K);
  if (code != IMQ_OK) return code;
  const DeviceInfo* dev = current_device(&code);
  if (!dev) return code;
  const Plan plan = plan_product(N, count, M, K, dev->cu_count);
  const int64_t cols = plane_columns(N, count);
  const bool split = plan.splits > 1;
  if (split && (!workspace || !aligned(workspace, 16) || workspace_bytes < (size_t)plan.splits * M * cols * 4))
    return fail(IMQ_EINVAL, "the workspace is null, misaligned or too small");
  ProductArgs a;
  SumArgs sum;
  memset(&a, 0, sizeof(a));
  memset(&sum, 0, sizeof(sum));
  a.count = sum.count = count;
  int tile0 = 0, col0 = 0;
  for (int i = 0; i < count; ++i) {
    a.p[i] = ProductProblem{p[i].w, p[i].scales, p[i].biases, p[i].y, split ? col0 : p[i].ldy, N[i], tile0};
    sum.p[i] = ProductProblem{nullptr, nullptr, nullptr, p[i].y, p[i].ldy, N[i], col0};
    tile0 += ceil_div(N[i], kColumns);
    col0 += (int)round_up(N[i], 4);
  }
  a.y_f32 = sum.y_f32 = y_dtype == IMQ_F32;
  if (split) a.planes = static_cast<float*>(workspace);
  a.plane_ld = cols;
  a.plane_stride = cols * M;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if ((code = run_product(a, plan, packed, ceil_div(M, 32), M, K, st)) != IMQ_OK || !split) return code;
  sum.planes = a.planes;
  sum.plane_ld = cols;
  sum.plane_stride = a.plane_stride;
  sum.M = M;
  sum.splits = plan.splits;
  hipLaunchKernelGGL(sum_planes_kernel, dim3(ceil_div(cols * M, 4 * kThreads)), dim3(kThreads), 0, st, sum);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(IMQ_ELAUNCH, std::string("sum launch failed: ") + hipGetErrorString(e));
  return ok();
}

int32_t imq_prompt_plan(const int32_t* N, int32_t count, int32_t M, int32_t K, int32_t max_splits, int32_t cus,
                        int32_t* tile_rows, int32_t* splits) {
  if (!N || !tile_rows || !splits || count < 1 || count > IMQ_PROMPT_MAX_PROBLEMS || M < 1 ||
      M > IMQ_PROMPT_MAX_ROWS || K < 64 || K % 64 || K > IMQ_PROMPT_MAX_K || max_splits < 1 || cus < 1)
    return fail(IMQ_EINVAL, "null pointer or a size out of range");
  for (int i = 0; i < count; ++i)
    if (N[i] < 1) return fail(IMQ_EINVAL, "N must be >= 1");
  const Plan plan = plan_product(N, count, M, K, cus, max_splits);
  *tile_rows = 32 * plan.tm;
  *splits = plan.splits;
  return ok();
}

size_t imq_prompt_matmul_workspace(int32_t M, int32_t N, int32_t K) {
  const size_t packed = imq_prompt_packed_bytes(M, K);
  if (!packed || N < 1) return 0;
  imq_problem p;
  memset(&p, 0, sizeof(p));
  p.N = N;
  p.K = K;
  return round_up(packed, 256) + imq_prompt_product_workspace(&p, 1, M);
}

int32_t imq_prompt_matmul(const uint32_t* w, const uint16_t* scales, const uint16_t* biases, const uint16_t* x,
                          int64_t ldx, void* y, int64_t ldy, int32_t M, int32_t N, int32_t K, int32_t group_size,
                          int32_t bits, int32_t y_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const imq_problem p = {w, scales, biases, nullptr, 0, y, ldy, N, K};
  int32_t n, k, code = check_product(&p, 1, M, group_size, bits, y_dtype, workspace, &n, &k);
  if (code != IMQ_OK) return code;
  const size_t packed = round_up(imq_prompt_packed_bytes(M, K), 256);
  if (workspace_bytes < packed) return fail(IMQ_EINVAL, "the workspace is too small");
  if ((code = imq_prompt_pack(x, ldx, M, K, workspace, stream)) != IMQ_OK) return code;
  return imq_prompt_product(&p, 1, workspace, M, group_size, bits, y_dtype, static_cast<char*>(workspace) + packed,
                            workspace_bytes - packed, stream);
}

size_t imq_prompt_experts_workspace(int32_t experts, int32_t pairs, int32_t K) {
  if (experts < 1 || experts > IMQ_PROMPT_MAX_EXPERTS || pairs < 1 || pairs > IMQ_PROMPT_MAX_ROWS || K < 64 ||
      K % 64 || K > IMQ_PROMPT_MAX_K)
    return 0;
  // for any N: the short tiles are the more, the tall ones the more blocks
  const int tiles = expert_tiles(experts, pairs, 1).tiles, blocks = expert_tiles(experts, pairs, 2).blocks;
  return round_up((size_t)tiles * 4, 256) + 2 * round_up((size_t)blocks * 32 * 4, 256) + packed_bytes(blocks, K);
}

int32_t imq_prompt_experts_plan(int32_t experts, int32_t pairs, int32_t N, int32_t cus, int32_t* tile_rows) {
  if (!tile_rows || experts < 1 || experts > IMQ_PROMPT_MAX_EXPERTS || pairs < 1 || pairs > IMQ_PROMPT_MAX_ROWS ||
      N < 1 || cus < 1)
    return fail(IMQ_EINVAL, "null pointer or a size out of range");
  *tile_rows = 32 * plan_experts(experts, pairs, N, cus).tm;
  return ok();
}

int32_t imq_prompt_experts(const uint32_t* w, const uint16_t* scales, const uint16_t* biases, int32_t experts,
                           const uint16_t* x, int64_t ldx, int32_t rows_per_x, const int32_t* idx, int32_t pairs,
                           void* y, int64_t ldy, int32_t N, int32_t K, int32_t group_size, int32_t bits,
                           int32_t y_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const imq_problem one = {w, scales, biases, nullptr, 0, y, ldy, N, K};
  int32_t n, k, code = check_product(&one, 1, pairs, group_size, bits, y_dtype, workspace, &n, &k);
  if (code != IMQ_OK) return code;
  if (experts < 1) return fail(IMQ_EINVAL, "experts must be >= 1");
  if (experts > IMQ_PROMPT_MAX_EXPERTS) return fail(IMQ_EUNSUPPORTED, "too many experts");
  if (!x || !idx || !aligned(x, 16) || !aligned(idx, 4)) return fail(IMQ_EINVAL, "x or idx is null or misaligned");
  if (ldx < K || ldx % 8) return fail(IMQ_EINVAL, "ldx must be >= K and a multiple of 8");
  if (rows_per_x < 1) return fail(IMQ_EINVAL, "rows_per_x must be >= 1");
  if (workspace_bytes < imq_prompt_experts_workspace(experts, pairs, K))
    return fail(IMQ_EINVAL, "the workspace is too small");
  const DeviceInfo* dev = current_device(&code);
  if (!dev) return code;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const ExpertPlan e = plan_experts(experts, pairs, N, dev->cu_count);
  char* at = static_cast<char*>(workspace);
  int32_t* const tile_expert = reinterpret_cast<int32_t*>(at);
  at += round_up((size_t)e.tiles * 4, 256);
  int32_t* const src = reinterpret_cast<int32_t*>(at);
  at += round_up((size_t)e.blocks * 32 * 4, 256);
  int32_t* const dest = reinterpret_cast<int32_t*>(at);
  at += round_up((size_t)e.blocks * 32 * 4, 256);
  hipLaunchKernelGGL(sort_pairs_kernel, dim3(1), dim3(kSortThreads), 0, st, idx, pairs, experts, rows_per_x,
                     32 * e.tm, e.tiles, src, dest, tile_expert);
  pack_rows(x, ldx, src, tile_expert, e.tm, 0, e.blocks, K, at, st);
  ProductArgs a;
  memset(&a, 0, sizeof(a));
  a.p[0] = ProductProblem{w, scales, biases, y, ldy, N, 0};
  a.count = 1;
  a.y_f32 = y_dtype == IMQ_F32;
  a.expert = tile_expert;
  a.dest = dest;
  const Plan p = {e.tm, 1, ceil_div(K, 256), e.tiles, ceil_div(N, kColumns)};
  return run_product(a, p, at, e.blocks, pairs, K, st);
}

}  // extern "C"
