// Read-back of a whole cache layer: K and V in position order as fp16.
//
// Semantics: TurboQuantCache._get_full_cache (leankv/turboquant/cache.py:169-189:
// the cold tokens dequantized, quantizer.py:131-137, (c[codes] @ Pi) * norm in
// fp32 rounded to fp16, then the fp16 hot window).
//
// The rotation of 128-dim centroid rows runs on v_mfma_f32_16x16x32_f16 with
// both operands split into fp16 parts, v = hi + lo / 2048 (v itself but for the
// last bit of a quarter of the fp32 values, 2^-23 relative), all four products of
// the parts kept in fp32 accumulators: 64 MFMA cycles per 32 input dims where
// the fp32 MFMA chain takes 256.  Its results are the closer ones: of 4.2 M
// values, 2341-2678 are not the 64-bit result rounded to fp16 (1 to 4 bits), of
// the fp32 chain's 4197-4267.
//
// One block of 4 waves walks tiles of 16 tokens; wave w owns output dims 32 w
// .. 32 w + 31, its parts of Pi in registers.  Transposed products: A = 16
// output dims x 32 input dims of Pi, B = 16 tokens' centroids, decoded in
// registers (v_perm lookups; a byte table in LDS at 4 bits), so that a lane
// ends with 8 consecutive dims of one token and stores them as 16 bytes.  Input
// dims are taken in the order that a lane's 16 code bytes hold them.
//
// Bound by the chain of a wave's tiles (codes, lookup, products, 16-byte stores;
// 8 tiles each at one sequence), not by bytes: 21 MB, 4.4 us at the copy rate of
// 4.9 TB/s.  One launch for both sides, read where the cache holds them and written
// in place: 15 us per 4096-token layer (8 kv heads, 3 bits, back to back, on the
// card and on the host alike), against 88 us for four copies of the strided store,
// two fp32-MFMA dequantize launches, two ring gathers and two concatenations.
#include <algorithm>

#include "kernels.h"
#include "tq_attn_common.h"
#include "tq_common.h"

namespace lkv {
namespace {

constexpr int kD = 128;
constexpr int kThreads = 256;
constexpr int kRows = 16;  // tokens per tile

struct ReadSide {
  const uint8_t* codes;  // [R][cap][row bytes]
  const float* norms;    // [R][cap]
  const float* Pi;
  const uint16_t* hot;   // [R][hot_cap][128] fp16 ring
  uint16_t* out;         // [R][n][128] fp16
};
struct ReadArgs {
  ReadSide side[2];
  const float* centroids;
  int ncent;
  int64_t cap;
  uint32_t R, n, cold, hot_cap;  // tokens cold .. n - 1 come from the ring, slot t % hot_cap
};

__device__ __forceinline__ void split_hl(float x, uint16_t& hi, uint16_t& lo) {
  hi = f2h(x);
  lo = f2h((x - h2f(hi)) * 2048.f);
}

template <int CB, bool PERM>
__global__ __launch_bounds__(kThreads, 2) void read_kernel(ReadArgs P) {
  static_assert(CB == 4 || PERM, "narrow code rows (1, 2 bits) decode through v_perm");
  constexpr int RB = kD * CB / 8;
  __shared__ uint32_t s_hi[PERM ? 1 : 256], s_lo[PERM ? 1 : 256];
  const ReadSide& W = P.side[blockIdx.y];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  const uint32_t n = P.n, cold = P.cold;

  // ---- the hot window, 16 bytes per thread
  {
    const uint32_t nh = n - cold, total = P.R * nh;
    const uint32_t c = tid & 15;
    for (uint32_t i = blockIdx.x * (kThreads / 16) + (tid >> 4); i < total; i += gridDim.x * (kThreads / 16)) {
      const uint32_t row = i / nh, t = cold + i % nh;
      *reinterpret_cast<uint4*>(W.out + (static_cast<size_t>(row) * n + t) * kD + 8 * c) =
          *reinterpret_cast<const uint4*>(W.hot + (static_cast<size_t>(row) * P.hot_cap + t % P.hot_cap) * kD + 8 * c);
    }
  }
  const uint32_t M = P.R * cold;
  const uint32_t ntiles = (M + kRows - 1) / kRows;
  uint32_t tile = blockIdx.x;
  if (tile >= ntiles) return;  // uniform over the block

  // ---- centroid tables: hi and lo parts
  uint32_t th[4] = {0u, 0u, 0u, 0u}, tl[4] = {0u, 0u, 0u, 0u};
  if constexpr (PERM) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // fewer than 8 centroids (1, 2 bits): zero entries, never selected
      uint16_t hi, lo;
      split_hl(j < P.ncent ? P.centroids[min(j, P.ncent - 1)] : 0.f, hi, lo);
      const int q = j >> 2, s = 8 * (j & 3);
      th[q] |= (hi & 0xffu) << s;
      th[2 + q] |= static_cast<uint32_t>(hi >> 8) << s;
      tl[q] |= (lo & 0xffu) << s;
      tl[2 + q] |= static_cast<uint32_t>(lo >> 8) << s;
    }
  } else {
    const int cmax = P.ncent - 1;
    uint16_t h0, l0, h1, l1;
    split_hl(P.centroids[min(tid & 15, cmax)], h0, l0);
    split_hl(P.centroids[min(tid >> 4, cmax)], h1, l1);
    s_hi[tid] = h0 | (static_cast<uint32_t>(h1) << 16);
    s_lo[tid] = l0 | (static_cast<uint32_t>(l1) << 16);
  }

  // ---- a tile's codes and norms: vector r = 16 tile + lane % 16, dims 32 g .. 32 g + 31
  uint4 cw;
  float nrm;
  auto locate = [&](uint32_t r) { return static_cast<size_t>(r / cold) * P.cap + r % cold; };
  auto load_tile = [&](uint32_t tl_) {
    const size_t at = locate(min(tl_ * kRows + c16, M - 1));
    cw = codes32<CB>(W.codes + at * RB + 4 * CB * g);
    nrm = W.norms[at];
  };
  load_tile(tile);

  // ---- A operands: row m of column tile t is output dim 32 wave + 8 (m / 4) + 4 t + m % 4, k slot (kb, g, j)
  // input dim 32 g + 8 kb + j in the decode's order
  u32x4 ah[2][4], al[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const float* src = W.Pi + (32 * g + 8 * kb) * kD + 32 * wave + 8 * (c16 >> 2) + 4 * t + (c16 & 3);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint16_t h0, l0, h1, l1;
        split_hl(src[(PERM ? kPermDim[2 * j] : 2 * j) * kD], h0, l0);
        split_hl(src[(PERM ? kPermDim[2 * j + 1] : 2 * j + 1) * kD], h1, l1);
        ah[t][kb][j] = h0 | (static_cast<uint32_t>(h1) << 16);
        al[t][kb][j] = l0 | (static_cast<uint32_t>(l1) << 16);
      }
    }
  if constexpr (!PERM) __syncthreads();  // byte tables

  for (; tile < ntiles; tile += gridDim.x) {
    const uint32_t r = tile * kRows + c16;
    const uint32_t w[4] = {cw.x, cw.y, cw.z, cw.w};
    const float sc = nrm;
    if (tile + gridDim.x < ntiles) load_tile(tile + gridDim.x);  // in flight during the products
    f32x4 hh[2], hl[2], ll[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) hh[t] = hl[t] = ll[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      uint32_t dh[4], dl[4];
      decode_dw<PERM>(w[kb], th, s_hi, dh);
      decode_dw<PERM>(w[kb], tl, s_lo, dl);
      const u32x4 bh = u32x4{dh[0], dh[1], dh[2], dh[3]}, bl = u32x4{dl[0], dl[1], dl[2], dl[3]};
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        hh[t] = mfma16x16x32(ah[t][kb], bh, hh[t]);
        hl[t] = mfma16x16x32(ah[t][kb], bl, hl[t]);
        hl[t] = mfma16x16x32(al[t][kb], bh, hl[t]);
        ll[t] = mfma16x16x32(al[t][kb], bl, ll[t]);
      }
    }
    if (r < M) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int t = e >> 2, i = e & 3;
        v[e] = fmaf(fmaf(ll[t][i], 1.f / 2048.f, hl[t][i]), 1.f / 2048.f, hh[t][i]) * sc;
      }
      const size_t o = (static_cast<size_t>(r / cold) * n + r % cold) * kD + 32 * wave + 8 * g;
      *reinterpret_cast<uint4*>(W.out + o) =
          uint4{pack2h(v[0], v[1]), pack2h(v[2], v[3]), pack2h(v[4], v[5]), pack2h(v[6], v[7])};
    }
  }
}

}  // namespace
}  // namespace lkv

using namespace lkv;

extern "C" int lkv_tq_cache_read(const uint8_t* k_codes, const float* k_norms, const uint8_t* v_codes,
                                 const float* v_norms, const void* k_hot, const void* v_hot, const float* PiK,
                                 const float* PiV, const float* centroids, int bits, int64_t R, int64_t n,
                                 int64_t cap, int64_t hot_cap, void* k_out, void* v_out, void* stream) {
  const char* who = "tq_cache_read";
  LKV_REQUIRE(bits >= 1 && bits <= 4, "%s: bits=%d unsupported (1..4 are bit-packed)", who, bits);
  LKV_REQUIRE(R >= 0 && n >= 0 && cap >= 0 && hot_cap >= 1, "%s: bad sizes R=%lld n=%lld cap=%lld hot_cap=%lld", who,
              (long long)R, (long long)n, (long long)cap, (long long)hot_cap);
  const int64_t cold = std::max<int64_t>(0, n - hot_cap);
  LKV_REQUIRE(cold <= cap, "%s: %lld cold tokens exceed cap=%lld", who, (long long)cold, (long long)cap);
  if (R == 0 || n == 0) return LKV_OK;
  LKV_REQUIRE(hot_cap < (1ll << 31) && R < (1ll << 31) && n < (1ll << 31) && R * n < (1ll << 31),
              "%s: problem too large", who);
  LKV_REQUIRE(k_codes && k_norms && v_codes && v_norms && k_hot && v_hot && PiK && PiV && centroids && k_out && v_out,
              "%s: null pointer", who);
  LKV_REQUIRE(aligned16(k_codes) && aligned16(v_codes) && aligned16(k_hot) && aligned16(v_hot) && aligned16(PiK) &&
                  aligned16(PiV) && aligned16(k_out) && aligned16(v_out),
              "%s: codes, rings, Pi and outputs must be 16-byte aligned", who);
  ReadArgs P{};
  P.side[0] = ReadSide{k_codes, k_norms, PiK, static_cast<const uint16_t*>(k_hot), static_cast<uint16_t*>(k_out)};
  P.side[1] = ReadSide{v_codes, v_norms, PiV, static_cast<const uint16_t*>(v_hot), static_cast<uint16_t*>(v_out)};
  P.centroids = centroids;
  P.ncent = 1 << bits;
  P.cap = cap;
  P.R = static_cast<uint32_t>(R);
  P.n = static_cast<uint32_t>(n);
  P.cold = static_cast<uint32_t>(cold);
  P.hot_cap = static_cast<uint32_t>(hot_cap);
  // one block per CU and side (each reads a whole Pi), fewer where there are fewer tiles and window rows
  const int64_t ntiles = (R * cold + kRows - 1) / kRows, hot = R * (n - cold);
  const int64_t want = std::max<int64_t>({ntiles, (hot + 15) / 16, int64_t(1)});
  const dim3 grid(static_cast<unsigned>(std::min<int64_t>(want, device_cu_count())), 2);
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (bits) {
    case 1: hipLaunchKernelGGL((read_kernel<1, true>), grid, dim3(kThreads), 0, st, P); break;
    case 2: hipLaunchKernelGGL((read_kernel<2, true>), grid, dim3(kThreads), 0, st, P); break;
    case 3: hipLaunchKernelGGL((read_kernel<4, true>), grid, dim3(kThreads), 0, st, P); break;
    default: hipLaunchKernelGGL((read_kernel<4, false>), grid, dim3(kThreads), 0, st, P); break;
  }
  LKV_LAUNCH_CHECK(who);
  return LKV_OK;
}
