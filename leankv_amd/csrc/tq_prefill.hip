// Causal prefill attention that reads the TurboQuant packed KV cache.
//
// Reference semantics: during a prefill (or any update of S > 1 tokens)
// TurboQuantCache.update returns cat(dequantize(cold).fp16, hot)
// (leankv/turboquant/cache.py:119-125, 169-189) and HF SDPA runs causal GQA
// attention of the S new queries over it (transformers/integrations/
// sdpa_attention.py:79-105): query i, at position kv_len - S + i, sees keys
// 0 .. kv_len - S + i, where keys below kv_len - hot_cap are the dequantized
// cold tokens and the rest the fp16 hot window.  As in the decode kernels no
// dequantized K/V is formed: with K_hat_t = n_t c[idx_t] PiK,
//   q . K_hat_t = n_t (q PiK^T) . c[idx_t],   sum_t p_t V_hat_t = (sum_t p_t n_t c[idx_t]) PiV,
// and hot tokens enter the same rotated domain as k PiK^T / v PiV^T (exact in
// real arithmetic, rounded to fp16 here), so one accumulator serves all keys
// and one un-rotation by PiV finishes each output row.
//
// Launches of lkv_tq_prefill_attn (two, on the caller's stream):
//   1. rotate16_kernel (fp16 MFMA, PiK / PiV split into fp16 hi + lo parts, 22
//      bits and more): the hot rings k @ PiK^T and v @ PiV^T (fp16);
//   2. tq_prefill_attn_kernel: grid (query tiles, kv heads, batch), 8 waves.
//      A block owns 256 (query, head) columns: 256 / G consecutive queries x
//      the G heads of one kv head, 32 columns per wave.  Its prologue rotates
//      the block's queries, q_rot = (q @ PiK^T) * scale * log2(e) in fp16 (the
//      score operand), with PiK split as in 1 and staged in the tile buffers.
//      It walks the keys in tiles of 64, decoded once per block into LDS as
//      fp16 centroid values [key][dim] (key codes by waves 0-3, value codes by
//      waves 4-7), and every wave runs, on v_mfma_f32_32x32x16_f16,
//      * scores transposed, A = 32 keys x 16 dims from LDS, B = its rotated
//        queries (registers), so a lane holds 32 keys of one column (the
//        other half of a tile's keys in lane ^ 32);
//      * the online softmax per lane (key norms, causal mask, exp2 domain).
//        The offset keeps a headroom above the max, so most tiles need neither
//        a max over the column's lanes nor a rescale of the accumulators: they
//        only check that no score passes the offset;
//      * values transposed, A = 32 dims x 16 keys gathered from the [key][dim]
//        rows by transposed LDS reads, B = p * n_t from the lane's own softmax
//        registers.
//      In its epilogue the block un-rotates its normalised rows, out = rows @
//      PiV on the same MFMA (PiV staged in the free tile buffers, both operands
//      split into hi + lo), and writes them as fp16.
//
// What bounds it: two waves per SIMD (256 registers each), so LDS latency,
// vector work (~200 instructions per wave and tile) and the matrix products
// (1024 cycles) overlap in part only.  16x16x32 products cost an issue slot of
// the vector port each (16 of them beside 48 vector instructions take 367
// cycles, alone 271): the 32x32 form halves that.  Measured, one block's cost
// per 64-key tile 2.47 -> 1.83 us, and per call (4096 tokens, 32/8 heads) 225 ->
// 201 us on one box, 512 queries over 2048 keys 102 -> 82 us: one column per
// lane, no cross-lane max on most tiles (2.47 -> 2.1), code loads through
// scalar descriptors and a decode without per-lane branches (2.02 -> 1.83).
// One wave per SIMD with 64 columns was slower (384 us: the compiler moves the
// accumulators between register files); four tile buffers instead of two, more
// reads in flight and interleaved products and softmax changed little.
#include "kernels.h"
#include "tq_attn_common.h"
#include "tq_common.h"

namespace lkv {
namespace {

constexpr int kD = 128;
constexpr int kThreads = 256;   // rotate16_kernel
constexpr int kKT = 64;         // keys per tile
// Waves of an attention block, 32 (query, head) columns each; waves 0-3 decode
// the key codes of a tile, waves 4-7 the value codes.
constexpr int kPWaves = 8;
constexpr int kPThreads = 64 * kPWaves;
constexpr int kCols = 32 * kPWaves;  // (query, head) columns per block
constexpr int kKRow = kD + 8;   // fp16 row of the decoded key tile (padded)
// Value rows [key][column] as decoded, 72 dwords: the MFMA's V^T operand is
// gathered by ds_read_b64_tr_b16, whose 8-byte chunks (rows 4 g + i, 4 chunks
// each) then fall in distinct banks.
constexpr int kVRow = kD + 16;
constexpr int kKBuf = kKT * kKRow, kVBuf = kKT * kVRow;  // fp16 per tile buffer
constexpr int kBufs = 4;                                 // two pairs of tiles
static_assert(kKT == 64, "the decode / compute lane maps assume 64-key tiles");
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kXcds = 8;  // MI355X: 8 accelerator complex dies, one L2 each

struct PrefillParams {
  const uint16_t* q16;     // [B, Hq, S, 128] fp16
  const float* PiK;        // [128, 128]
  float scale_log2;        // scale * log2(e)
  const float* PiV;        // [128, 128]: the output rows are un-rotated in the epilogue
  uint16_t* out;           // [B, Hq, S, 128] fp16
  const uint8_t* k_codes;  // [B, Hkv, cap, 64]
  const float* k_norms;    // [B, Hkv, cap]
  const uint8_t* v_codes;
  const float* v_norms;
  const uint16_t* hk;      // [B, Hkv, hot_cap, 128] fp16: hot keys @ PiK^T (ring slots)
  const uint16_t* hv;      // hot values @ PiV^T
  const float* centroids;  // [2^bits]
  int S, Hq, Hkv, G, cap, hot_cap, kv_len, cold_len, ncent;
};

// y = x @ Pi^T for fp16 rows of 128, on fp16 MFMA: Pi split into fp16 parts hi +
// lo / 2048 (22 bits and more of the 24), fp32 accumulate.  Wave w computes output
// dims 32 w .. 32 w + 31 with its Pi operands in registers; a block takes 64-row
// tiles, staged through LDS both ways so every row is read once and written
// with 16-byte stores.  The two hot rings are rotated by one launch, blockIdx.y
// picking the ring.
constexpr int kRotRows = 64;
struct RotSeg {
  const uint16_t* x;
  const float* Pi;
  uint16_t* y;
};
struct RotSegs {
  RotSeg s[2];
  int64_t M;  // rows of each
};
__global__ __launch_bounds__(kThreads) void rotate16_kernel(RotSegs segs) {
  const RotSeg& sg = segs.s[blockIdx.y];
  const uint16_t* __restrict__ x = sg.x;
  const float* __restrict__ Pi = sg.Pi;
  uint16_t* __restrict__ y = sg.y;
  const int64_t M = segs.M;
  constexpr int kRow = kD + 8;  // padded LDS row
  __shared__ __align__(16) uint16_t s_in[kRotRows * kRow];
  __shared__ __align__(16) uint16_t s_out[kRotRows * kRow];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  // B operands: column d = 32 wave + 16 dt + c16, k = input dim e = 32 kb + 8 g + i: B[e][d] = Pi[d][e]
  u32x4 bh[2][4], bl[2][4];
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const int d = 32 * wave + 16 * dt + c16, e0 = 32 * kb + 8 * g;
      const float4 u0 = *reinterpret_cast<const float4*>(Pi + d * kD + e0);
      const float4 u1 = *reinterpret_cast<const float4*>(Pi + d * kD + e0 + 4);
      const float p[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint16_t h0 = f2h(p[2 * j]), h1 = f2h(p[2 * j + 1]);
        bh[dt][kb][j] = static_cast<uint32_t>(h0) | (static_cast<uint32_t>(h1) << 16);
        bl[dt][kb][j] = pack2h((p[2 * j] - h2f(h0)) * 2048.f, (p[2 * j + 1] - h2f(h1)) * 2048.f);
      }
    }
  constexpr int kPerRow = kD / 8;                            // 16-byte chunks of a row
  constexpr int kChunks = kRotRows * kPerRow / kThreads;     // per thread, in and out
  const int64_t ntiles = (M + kRotRows - 1) / kRotRows;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t row0 = tile * kRotRows;
    // ---- rows in (rows past M read row M - 1, never stored)
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const int f = c * kThreads + tid, r = f / kPerRow, q = f % kPerRow;
      const int64_t gr = min(row0 + r, M - 1);
      *reinterpret_cast<uint4*>(s_in + r * kRow + 8 * q) = *reinterpret_cast<const uint4*>(x + gr * kD + 8 * q);
    }
    __syncthreads();
#pragma unroll
    for (int rg = 0; rg < kRotRows / 16; ++rg) {
      u32x4 a[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        a[kb] = *reinterpret_cast<const u32x4*>(s_in + (16 * rg + c16) * kRow + 32 * kb + 8 * g);
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) {
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f}, accl = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          acc = mfma16x16x32(a[kb], bh[dt][kb], acc);
          accl = mfma16x16x32(a[kb], bl[dt][kb], accl);
        }
        // D: column d = 32 wave + 16 dt + c16, rows 16 rg + 4 g + i
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = acc[i] + accl[i] * (1.f / 2048.f);
          __asm__ volatile("" : "+v"(v));  // rounded to fp32 before fp16, as a scaled product is
          s_out[(16 * rg + 4 * g + i) * kRow + 32 * wave + 16 * dt + c16] = f2h(v);
        }
      }
    }
    __syncthreads();
    // ---- rows out
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const int f = c * kThreads + tid, r = f / kPerRow, q = f % kPerRow;
      if (row0 + r < M)
        *reinterpret_cast<uint4*>(y + (row0 + r) * kD + 8 * q) = *reinterpret_cast<const uint4*>(s_out + r * kRow + 8 * q);
    }
    __syncthreads();  // s_in and s_out are rewritten by the next tile
  }
}

// fp16 positions 0..7 of a natural-order group reordered to kPermDim.
__device__ __forceinline__ uint4 perm_group(uint4 a) {
  return uint4{__builtin_amdgcn_perm(a.y, a.x, 0x05040100u), __builtin_amdgcn_perm(a.w, a.z, 0x05040100u),
               __builtin_amdgcn_perm(a.y, a.x, 0x07060302u), __builtin_amdgcn_perm(a.w, a.z, 0x07060302u)};
}

// Largest of a lane's 32 scores.
__device__ __forceinline__ float max32(const float (&s)[32]) {
  float a = vmax3(s[0], s[1], s[2]), b = vmax3(s[3], s[4], s[5]);
#pragma unroll
  for (int j = 6; j < 30; j += 4) {
    a = vmax3(a, s[j], s[j + 1]);
    b = vmax3(b, s[j + 2], s[j + 3]);
  }
  return fmaxf(vmax3(a, s[30], s[31]), b);
}
// Max / sum over the two lanes l, l ^ 32 that share a column.
__device__ __forceinline__ float xhalf_max(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float xhalf_sum(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
__device__ __forceinline__ void split_hl(float x, uint16_t& hi, uint16_t& lo) {
  hi = f2h(x);
  lo = f2h((x - h2f(hi)) * 2048.f);
}
__device__ __forceinline__ uint32_t pair16(uint16_t lo, uint16_t hi) { return lo | (static_cast<uint32_t>(hi) << 16); }

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
// D (lane l: column l % 32, rows 8 (i / 4) + 4 (l / 32) + i % 4, i = 0..15) += A (row l % 32) x B (column l % 32),
// both with k slots 8 (l / 32) + j, j = 0..7
__device__ __forceinline__ f32x16 mfma32x32x16(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <bool PERM, int CB>
__global__ __launch_bounds__(kPThreads, 1) void tq_prefill_attn_kernel(PrefillParams P) {
  static_assert(CB == 4 || PERM, "narrow code rows use the v_perm decode");
  constexpr int RB = kD * CB / 8;  // code bytes per token
  __shared__ __align__(16) uint16_t sK[kBufs * kKBuf];   // decoded keys
  __shared__ __align__(16) uint16_t sVt[kBufs * kVBuf];  // decoded values
  __shared__ __align__(16) float sN[kBufs][2][kKT];    // [buffer][key, value] norms (1 hot, 0 past the end)
  __shared__ uint32_t s_lut[256];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c32 = lane & 31, hf = lane >> 5;
  const int G = P.G, QT = kCols / G;
  // The latest queries see the most keys: their tiles are dispatched first.
  // Workgroups go to the 8 XCDs round-robin by linear id and every query tile
  // of a (batch, kv head) reads the same cold store, so the tiles are placed
  // XCD by XCD: with I = B * Hkv items, XCD x serves items x, x + 8, .. (I a
  // multiple of 8) or every (8 / I)-th tile of item x % I (I = 1, 2, 4), its
  // own tiles heaviest first; other shapes keep the plain order.
  int qtile, kvh, b;
  {
    const int nx = static_cast<int>(gridDim.x), I = static_cast<int>(gridDim.y * gridDim.z);
    const int p = static_cast<int>(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
    const int x = p % kXcds, s = p / kXcds;
    int item, t;
    if (I % kXcds == 0) {
      const int per = I / kXcds;  // items per XCD
      item = x + kXcds * (s % per);
      t = s / per;
    } else if (kXcds % I == 0 && nx % (kXcds / I) == 0) {
      const int k = kXcds / I;  // XCDs per item
      item = x % I;
      t = s * k + x / I;
    } else {
      item = p / nx;
      t = p % nx;
    }
    // (divisions leave them in vector registers: made scalar again)
    qtile = __builtin_amdgcn_readfirstlane(nx - 1 - t);
    kvh = __builtin_amdgcn_readfirstlane(item % static_cast<int>(gridDim.y));
    b = __builtin_amdgcn_readfirstlane(item / static_cast<int>(gridDim.y));
  }
  const int q0 = qtile * QT;
  const int qpos0 = P.kv_len - P.S;  // position of query 0
  const size_t bh = static_cast<size_t>(b) * P.Hkv + kvh;
  const int cold_len = P.cold_len, kv_len = P.kv_len;

  // ---- per-thread code registers of a key tile (as nibbles), loaded an
  // iteration before their decode:
  //   waves 0-3: key codes of key tid / 4, dims 32 (tid % 4) .. +32
  //   waves 4-7: value codes of keys 4 kp + e, dims 8 j4 .. +8 (the 16 lanes of a row group take the 16 column
  //              chunks of one row: conflict-free 16-byte stores, coalesced code loads)
  // and key (wave 0) and value norms (wave 4) of key lane
  const uint8_t* kcod = P.k_codes + bh * static_cast<size_t>(P.cap) * RB;
  const uint8_t* vcod = P.v_codes + bh * static_cast<size_t>(P.cap) * RB;
  const bool key_thr = wave < 4;  // wave-uniform
  const float* norms = (key_thr ? P.k_norms : P.v_norms) + bh * static_cast<size_t>(P.cap);
  const bool nrm_thr = wave == 0 || wave == 4;
  const int kk = (tid & 255) >> 2, part = tid & 3;
  const int kp = (tid & 255) >> 4, j4 = tid & 15;
  const uint8_t* const cod = key_thr ? kcod : vcod;
  const int voff = key_thr ? kk * RB + 4 * CB * part : 4 * kp * RB + CB * j4;
  uint32_t tw[2][4];
  float tn[2] = {0.f, 0.f};
  // through buffer descriptors over the tile's cold rows (rows past them read 0, their values come from
  // elsewhere): constant lane offsets, the tile's position in the scalar base
  auto load_tile = [&](int t0, int u) {
    const int n = __builtin_amdgcn_readfirstlane(max(0, min(kKT, cold_len - t0)));  // (the clamp compiles to vector code)
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(cod + static_cast<size_t>(t0) * RB, n * RB);
    if (key_thr) {
      const u32x4 w = load_raw32<CB>(rc, voff);
#pragma unroll
      for (int e = 0; e < 4; ++e) tw[u][e] = widen32<CB>(w, e);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) tw[u][e] = widen8<CB>(load_raw8<CB>(rc, voff + e * RB));
    }
    if (nrm_thr)
      tn[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(make_rsrc(norms + t0, n * 4), 4 * lane, 0, 0));
  };

  // ---- prologue loads, all in flight together: the first tile's codes, the
  // block's queries, the rotation matrices
  load_tile(0, 0);
  load_tile(kKT, 1);
  // the wave's (query, head) column c = 32 wave + lane % 32: query q0 + c / G, head c % G
  const int qq = q0 + (32 * wave + c32) / G, qh = (32 * wave + c32) % G;
  const size_t qrow = ((static_cast<size_t>(b) * P.Hq + kvh * G + qh) * P.S + min(qq, P.S - 1)) * kD;
  u32x4 bq[8];  // B: the column's q row, dims 16 kb + 8 hf .. +7
#pragma unroll
  for (int kb = 0; kb < 8; ++kb) {
    const uint4 u = *reinterpret_cast<const uint4*>(P.q16 + qrow + 16 * kb + 8 * hf);
    bq[kb] = u32x4{u.x, u.y, u.z, u.w};
  }
  constexpr int kPiRows = kPThreads / 32, kPiLd = kD / kPiRows;  // thread: input dims 4 (tid % 32) .. of 8 rows
  float4 pk[kPiLd];
  // PiK row for staged row R = 32 t + r: the column of the key tile that output element (lane, i) of row tile
  // t belongs to (r = 8 (i / 4) + 4 hf + i % 4), C = 16 (2 t + i / 8) + 8 hf + i % 8, so that the product's
  // output is the score operand, k step 2 t + i / 8, slot i % 8; the dim of C in the decode's order
#pragma unroll
  for (int j = 0; j < kPiLd; ++j) {
    const int R = tid / 32 + kPiRows * j, r = R & 31;
    const int C = (R & ~31) + 16 * (r >> 4) + 8 * ((r >> 2) & 1) + 4 * ((r >> 3) & 1) + (r & 3);
    const int dim = PERM ? (C & ~7) + ((C & 3) << 1) + ((C >> 2) & 1) : C;
    pk[j] = *reinterpret_cast<const float4*>(P.PiK + dim * kD + 4 * (tid & 31));
  }
  // ---- centroid tables
  uint32_t tab[4] = {0u, 0u, 0u, 0u};
  if constexpr (PERM) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // fewer than 8 centroids (1, 2 bits): zero entries, never selected
      const float cj = P.centroids[min(j, P.ncent - 1)];
      const uint32_t c16 = f2h(j < P.ncent ? cj : 0.f);
      tab[j >> 2] |= (c16 & 0xffu) << (8 * (j & 3));
      tab[2 + (j >> 2)] |= (c16 >> 8) << (8 * (j & 3));
    }
  } else {
    const int cmax = P.ncent - 1;
    if (tid < 256) s_lut[tid] = pack2h(P.centroids[min(tid & 15, cmax)], P.centroids[min(tid >> 4, cmax)]);
  }

  // ---- q_rot = (q @ PiK^T) * scale * log2(e) in fp16 (the score operand):
  // A = 32 rows of PiK (split into fp16 hi + lo / 2048, in the tile buffers,
  // free until the first decode), B = the wave's 32 query rows
#pragma unroll
  for (int j = 0; j < kPiLd; ++j) {
    const int R = tid / 32 + kPiRows * j, e4 = tid & 31;
    const float x[4] = {pk[j].x, pk[j].y, pk[j].z, pk[j].w};
    uint16_t hi[4], lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) split_hl(x[i], hi[i], lo[i]);
    *reinterpret_cast<uint2*>(sK + R * kKRow + 4 * e4) = uint2{pair16(hi[0], hi[1]), pair16(hi[2], hi[3])};
    *reinterpret_cast<uint2*>(sVt + R * kKRow + 4 * e4) = uint2{pair16(lo[0], lo[1]), pair16(lo[2], lo[3])};
  }
  static_assert(kD * kKRow <= kBufs * kKBuf && kD * kKRow <= kBufs * kVBuf, "PiK staging fits the tile buffers");
  __syncthreads();  // PiK staged
  const bool ok = qq < P.S;
  const int lim = ok ? qpos0 + qq + 1 : 0;  // keys [0, lim) visible to the lane's column (0: no such query)
  u32x4 qa[8];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f32x16 acc = {}, accl = {};
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) {
      const u32x4 ah = *reinterpret_cast<const u32x4*>(sK + (32 * t + c32) * kKRow + 16 * kb + 8 * hf);
      const u32x4 al = *reinterpret_cast<const u32x4*>(sVt + (32 * t + c32) * kKRow + 16 * kb + 8 * hf);
      acc = mfma32x32x16(ah, bq[kb], acc);
      accl = mfma32x32x16(al, bq[kb], accl);
    }
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      const float v0 = (acc[i] + accl[i] * (1.f / 2048.f)) * P.scale_log2;
      const float v1 = (acc[i + 1] + accl[i + 1] * (1.f / 2048.f)) * P.scale_log2;
      qa[2 * t + (i >> 3)][(i & 7) >> 1] = ok ? pack2h(v0, v1) : 0u;
    }
  }
  // the fewest keys a column of the wave sees: its first column's (queries ascend); none past the last query
  const int wq = q0 + 32 * wave / G;
  const int wmin = wq < P.S ? qpos0 + wq + 1 : 0x7fffffff;
  __syncthreads();  // every wave is past its PiK reads: the tile buffers are free

  // keys [0, kend) are visible to some column of the block
  const int kend = qpos0 + min(q0 + QT, P.S);
  const int ntile = (kend + kKT - 1) / kKT;

  // decode the loaded tile into LDS buffer `buf`: keys and values [key][dim], dims in kPermDim order within
  // 8-dim groups with PERM; in a tile that reaches past the cold store the rows from cold_len on are then written
  // again (by the thread that wrote them)
  uint16_t* const kdst = sK + kk * kKRow + 32 * part;
  uint16_t* const vdst = sVt + 4 * kp * kVRow + 8 * j4;
  auto decode_tile = [&](int t0, int buf, int u) {
    uint16_t* dst = key_thr ? kdst + buf * kKBuf : vdst + buf * kVBuf;
    const int step = key_thr ? 8 : kVRow;  // keys: the row's four chunks; values: four rows' chunk
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t d[4];
      decode_dw<PERM>(tw[u][e], tab, s_lut, d);
      *reinterpret_cast<uint4*>(dst + e * step) = uint4{d[0], d[1], d[2], d[3]};
    }
    if (nrm_thr) {
      const int tk = t0 + lane;
      sN[buf][key_thr ? 0 : 1][lane] = tk < cold_len ? tn[u] : (tk < kv_len ? 1.f : 0.f);
    }
    if (t0 + kKT > cold_len) {  // uniform
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int tk = key_thr ? t0 + kk : t0 + 4 * kp + e;
        if (tk < cold_len) continue;
        uint4 v = uint4{0u, 0u, 0u, 0u};
        if (tk < kv_len) {
          v = *reinterpret_cast<const uint4*>((key_thr ? P.hk : P.hv) +
                                              (bh * P.hot_cap + static_cast<size_t>(tk % P.hot_cap)) * kD +
                                              (key_thr ? 32 * part + 8 * e : 8 * j4));
          if constexpr (PERM) v = perm_group(v);
        }
        *reinterpret_cast<uint4*>(dst + e * step) = v;
      }
    }
  };

  // columns past the last query keep offset 0 over their zero scores: they never ask for the general path
  float m = ok ? -INFINITY : 0.f, l = 0.f;
  f32x16 o[4];  // element i: column's output dim (in the key tile's order) 32 db + 8 (i / 4) + 4 hf + i % 4
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = f32x16{};

  // one key tile from LDS buffer `buf`: element i of key block kt is key t0 + 32 kt + 8 (i / 4) + 4 hf + i % 4
  auto compute_tile = [&](int t0, int buf) {
    const uint16_t* sKb = sK + buf * kKBuf;
    const uint16_t* sVb = sVt + buf * kVBuf;
    const float* sNb = &sN[buf][0][0];
    f32x16 sc[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      sc[kt] = f32x16{};
#pragma unroll
      for (int kb = 0; kb < 8; ++kb)
        sc[kt] = mfma32x32x16(
            *reinterpret_cast<const u32x4*>(sKb + (32 * kt + c32) * kKRow + 16 * kb + 8 * hf), qa[kb], sc[kt]);
    }
    // log2 weights relative to the running offset: score * key norm - m.  Most
    // tiles hold no masked key and no score above the offset (which keeps a
    // headroom above the max): they need no max over the column's two lanes and
    // no rescale.  The others, and the first (m = -inf), go through the general
    // path.
    float s[32];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const f32x4 kn = *reinterpret_cast<const f32x4*>(sNb + 8 * q + 4 * hf);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[4 * q + i] = fmaf(sc[q >> 2][4 * (q & 3) + i], kn[i], -m);
    }
    // wave-uniform; a NaN score passes as it would below
    if (t0 + kKT > wmin || wave_ballot(max32(s) > 0.f) != 0) {
      const int left = lim - t0 - 4 * hf;  // key 8 q + i of the lane is visible below this
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const f32x4 kn = *reinterpret_cast<const f32x4*>(sNb + 8 * q + 4 * hf);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = sc[q >> 2][4 * (q & 3) + i] * kn[i];
          s[4 * q + i] = 8 * q + i < left ? v : -INFINITY;
        }
      }
      const float mx = xhalf_max(max32(s));
      const float mn = mx > m ? mx + kHeadroom : m;  // -inf stays -inf
      const float mu = mn == -INFINITY ? 0.f : mn;
      const float alpha = fast_exp2(m - mu);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db) o[db] = o[db] * alpha;
#pragma unroll
      for (int j = 0; j < 32; ++j) s[j] -= mu;
    }
    // weights, and p * value norm in fp16: the value MFMA's operand (slots = the lane's 8 keys of a 16-key step)
    u32x4 pb[4];
    float ps[2] = {0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const f32x4 vn = *reinterpret_cast<const f32x4*>(sNb + kKT + 8 * q + 4 * hf);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[4 * q + i] = fast_exp2(s[4 * q + i]);
        ps[i & 1] += s[4 * q + i];
      }
      pb[q >> 1][2 * (q & 1)] = mul2h(s[4 * q], vn[0], s[4 * q + 1], vn[1]);
      pb[q >> 1][2 * (q & 1) + 1] = mul2h(s[4 * q + 2], vn[2], s[4 * q + 3], vn[3]);
    }
    l += ps[0] + ps[1];
    // values: O^T (32 dims x 32 columns) += V^T (the lane's keys 16 ks + 4 hf + .., and 8 further on) x P^T.
    // ds_read_b64_tr_b16: in each 16-lane group, lane l receives element l % 4 of the 8 bytes that
    // lanes 4 i + l / 4 (i = 0..3) address: a lane addresses key l / 4 of the group's four, columns 4 (l % 4) ..
    // +3 of the group's 16, and receives its own column of those four keys.
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const uint16_t* src = sVb + (16 * ks + 4 * hf + ((lane & 15) >> 2)) * kVRow + 32 * db + 16 * ((lane >> 4) & 1) +
                              4 * (lane & 3);
        typedef short v4s __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) v4s lds_v4s;
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(src));
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(src + 8 * kVRow));
        const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
        o[db] = mfma32x32x16(u32x4{l2.x, l2.y, h2.x, h2.y}, pb[ks], o[db]);
      }
  };

  // Two tiles per barrier and two pairs of LDS buffers in turn: while pair it is
  // computed, pair it + 1 is decoded into the other buffers (last read by the
  // compute of pair it - 1, before the last barrier) from registers loaded an
  // iteration earlier.  Waves 4-7 decode before they compute, waves 0-3 after,
  // so the two waves of a SIMD are out of step: the matrix products and LDS
  // reads of one run under the softmax arithmetic of the other.
  const int npair = (ntile + 1) / 2;
  auto next_pair = [&](int it) {
#pragma unroll
    for (int u = 0; u < 2; ++u) decode_tile((2 * it + u) * kKT, (2 * it + u) % kBufs, u);
    if (it + 1 < npair) {
#pragma unroll
      for (int u = 0; u < 2; ++u) load_tile((2 * it + 2 + u) * kKT, u);
    }
  };
  next_pair(0);
  __syncthreads();
#pragma unroll 1
  for (int it = 0; it < npair; ++it) {
    if (!key_thr && it + 1 < npair) next_pair(it + 1);
#pragma unroll 1
    for (int u = 2 * it; u < min(2 * it + 2, ntile); ++u) compute_tile(u * kKT, u % kBufs);
    if (key_thr && it + 1 < npair) next_pair(it + 1);
    __syncthreads();
  }

  // ---- PiV^T in LDS, [e][c], hi in sK, lo in sVt (the tile buffers are free): thread's blocks of 4 output dims e
  // = 4 (tid % 32) .. x 4 columns c of the key tile's order (one 8-byte store per dim and part)
  {
    const int e0 = 4 * (tid & 31);
    constexpr int kStep = 4 * kPThreads / 32;  // columns per round
    float4 pv[kD / kStep][4];
#pragma unroll
    for (int r = 0; r < kD / kStep; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = kStep * r + 4 * (tid >> 5) + i;
        pv[r][i] = *reinterpret_cast<const float4*>(
            P.PiV + (PERM ? (c & ~7) + ((c & 3) << 1) + ((c >> 2) & 1) : c) * kD + e0);
      }
#pragma unroll
    for (int r = 0; r < kD / kStep; ++r)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uint16_t hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          split_hl(k == 0 ? pv[r][i].x : k == 1 ? pv[r][i].y : k == 2 ? pv[r][i].z : pv[r][i].w, hi[i], lo[i]);
        const int at = (e0 + k) * kKRow + kStep * r + 4 * (tid >> 5);
        *reinterpret_cast<uint2*>(sK + at) = uint2{pair16(hi[0], hi[1]), pair16(hi[2], hi[3])};
        *reinterpret_cast<uint2*>(sVt + at) = uint2{pair16(lo[0], lo[1]), pair16(lo[2], lo[3])};
      }
  }
  // ---- normalise, un-rotate (out = o_rot @ PiV) and write fp16 rows: A = 32
  // output dims of PiV^T, B = the lane's own normalised sums (k slots of step
  // (db, u): its dims 32 db + 16 u + 4 hf + .., and 8 further on), both split
  // into fp16 hi + lo / 2048 (hi.hi + hi.lo + lo.hi, the lo.lo term
  // dropped: ~2^-22 relative).
  const float L = xhalf_sum(l);
  const float inv = L > 0.f ? 1.f / L : 0.f;
  u32x4 obh[8], obl[8];
#pragma unroll
  for (int st = 0; st < 8; ++st)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint16_t h0, l0, h1, l1;
      split_hl(o[st >> 1][8 * (st & 1) + 2 * j] * inv, h0, l0);
      split_hl(o[st >> 1][8 * (st & 1) + 2 * j + 1] * inv, h1, l1);
      obh[st][j] = pair16(h0, h1);
      obl[st][j] = pair16(l0, l1);
    }
  __syncthreads();  // PiV staged
#pragma unroll 1
  for (int et = 0; et < 4; ++et) {
    f32x16 acc = {}, accl = {}, accm = {};
    const int er = (32 * et + c32) * kKRow + 4 * hf;
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const uint2 h0 = *reinterpret_cast<const uint2*>(sK + er + 16 * st);
      const uint2 h1 = *reinterpret_cast<const uint2*>(sK + er + 16 * st + 8);
      const uint2 l0 = *reinterpret_cast<const uint2*>(sVt + er + 16 * st);
      const uint2 l1 = *reinterpret_cast<const uint2*>(sVt + er + 16 * st + 8);
      const u32x4 ah = u32x4{h0.x, h0.y, h1.x, h1.y}, al = u32x4{l0.x, l0.y, l1.x, l1.y};
      acc = mfma32x32x16(ah, obh[st], acc);
      accl = mfma32x32x16(ah, obl[st], accl);
      accm = mfma32x32x16(al, obh[st], accm);
    }
    if (ok) {
      uint16_t* dst = P.out + qrow + 32 * et + 4 * hf;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = acc[4 * q + i] + (accl[4 * q + i] + accm[4 * q + i]) * (1.f / 2048.f);
        *reinterpret_cast<uint2*>(dst + 8 * q) = uint2{pack2h(r[0], r[1]), pack2h(r[2], r[3])};
      }
    }
  }
}

}  // namespace
}  // namespace lkv

using namespace lkv;

extern "C" size_t lkv_tq_prefill_attn_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t S,
                                                      int64_t hot_cap) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || S <= 0 || hot_cap <= 0) return 0;
  auto al = [](size_t v) { return (v + 255) / 256 * 256; };
  const size_t hot = static_cast<size_t>(B * Hkv * hot_cap) * kD * 2;
  return 2 * al(hot);  // the rotated hot rings (queries and outputs are rotated in the kernel)
}

extern "C" int lkv_tq_prefill_attn(const void* q, const uint8_t* k_codes, const float* k_norms,
                                   const uint8_t* v_codes, const float* v_norms, const void* k_hot,
                                   const void* v_hot, const float* PiK, const float* PiV, const float* centroids,
                                   int bits, int64_t kv_len, int64_t B, int64_t Hq, int64_t Hkv, int64_t S,
                                   int64_t cap, int64_t hot_cap, float scale, void* out, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  LKV_REQUIRE(bits >= 1 && bits <= 4, "tq_prefill_attn: bits=%d unsupported (1..4 are bit-packed)", bits);
  LKV_REQUIRE(B >= 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0, "tq_prefill_attn: need Hq %% Hkv == 0 (Hq=%lld Hkv=%lld)",
              (long long)Hq, (long long)Hkv);
  const int64_t G = Hq / Hkv;
  LKV_REQUIRE(G <= 16 && (16 % G) == 0, "tq_prefill_attn: Hq/Hkv=%lld must be 1, 2, 4, 8 or 16", (long long)G);
  LKV_REQUIRE(hot_cap >= 1 && hot_cap <= (1 << 20), "tq_prefill_attn: hot_cap=%lld out of range", (long long)hot_cap);
  LKV_REQUIRE(S >= 0 && S <= kv_len, "tq_prefill_attn: need 0 <= S <= kv_len (S=%lld kv_len=%lld)", (long long)S,
              (long long)kv_len);
  LKV_REQUIRE(kv_len - hot_cap <= cap, "tq_prefill_attn: kv_len - hot_cap = %lld cold tokens exceed cap=%lld",
              (long long)(kv_len - hot_cap), (long long)cap);
  LKV_REQUIRE(kv_len < (1ll << 30) && cap < (1ll << 30) && B * Hq * S < (1ll << 31),
              "tq_prefill_attn: problem too large");
  if (B == 0 || S == 0) return LKV_OK;
  LKV_REQUIRE(q && k_codes && k_norms && v_codes && v_norms && k_hot && v_hot && PiK && PiV && centroids && out &&
                  workspace,
              "tq_prefill_attn: null pointer");
  LKV_REQUIRE(aligned16(q) && aligned16(k_codes) && aligned16(v_codes) && aligned16(k_hot) && aligned16(v_hot) &&
                  aligned16(PiK) && aligned16(PiV) && aligned16(out) && aligned16(workspace),
              "tq_prefill_attn: q, codes, hot, Pi, out and workspace must be 16-byte aligned");
  const size_t need = lkv_tq_prefill_attn_workspace_bytes(B, Hq, Hkv, S, hot_cap);
  LKV_REQUIRE(workspace_bytes >= need, "tq_prefill_attn: workspace of %zu bytes required, got %zu", need,
              workspace_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto al = [](size_t v) { return (v + 255) / 256 * 256; };
  uint16_t* hk = static_cast<uint16_t*>(workspace);
  uint16_t* hv = reinterpret_cast<uint16_t*>(static_cast<char*>(workspace) +
                                             al(static_cast<size_t>(B * Hkv * hot_cap) * kD * 2));
  const int64_t cold_len = kv_len > hot_cap ? kv_len - hot_cap : 0;

  // the hot rings in the rotated domains (one launch; every hot slot is rotated, only the current tokens' are read)
  {
    const RotSegs segs{{{static_cast<const uint16_t*>(k_hot), PiK, hk}, {static_cast<const uint16_t*>(v_hot), PiV, hv}},
                       B * Hkv * hot_cap};
    const int64_t tiles = (segs.M + kRotRows - 1) / kRotRows, most = 2 * static_cast<int64_t>(device_cu_count());
    hipLaunchKernelGGL(rotate16_kernel, dim3(static_cast<unsigned>(tiles < most ? tiles : most), 2), dim3(kThreads), 0, st,
                       segs);
    LKV_LAUNCH_CHECK("tq_prefill_attn rotation");
  }
  PrefillParams P;
  P.q16 = static_cast<const uint16_t*>(q);
  P.PiK = PiK;
  P.scale_log2 = scale * kLog2e;
  P.PiV = PiV;
  P.out = static_cast<uint16_t*>(out);
  P.k_codes = k_codes;
  P.k_norms = k_norms;
  P.v_codes = v_codes;
  P.v_norms = v_norms;
  P.hk = hk;
  P.hv = hv;
  P.centroids = centroids;
  P.S = static_cast<int>(S);
  P.Hq = static_cast<int>(Hq);
  P.Hkv = static_cast<int>(Hkv);
  P.G = static_cast<int>(G);
  P.cap = static_cast<int>(cap);
  P.hot_cap = static_cast<int>(hot_cap);
  P.kv_len = static_cast<int>(kv_len);
  P.cold_len = static_cast<int>(cold_len);
  P.ncent = 1 << bits;
  const int64_t QT = kCols / G;
  const dim3 grid(static_cast<unsigned>((S + QT - 1) / QT), static_cast<unsigned>(Hkv), static_cast<unsigned>(B));
  switch (bits) {
    case 1: hipLaunchKernelGGL((tq_prefill_attn_kernel<true, 1>), grid, dim3(kPThreads), 0, st, P); break;
    case 2: hipLaunchKernelGGL((tq_prefill_attn_kernel<true, 2>), grid, dim3(kPThreads), 0, st, P); break;
    case 3: hipLaunchKernelGGL((tq_prefill_attn_kernel<true, 4>), grid, dim3(kPThreads), 0, st, P); break;
    default: hipLaunchKernelGGL((tq_prefill_attn_kernel<false, 4>), grid, dim3(kPThreads), 0, st, P);
  }
  LKV_LAUNCH_CHECK("tq_prefill_attn");
  return LKV_OK;
}
