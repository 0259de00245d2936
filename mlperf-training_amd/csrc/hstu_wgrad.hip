// Weight gradients over the token axis of the HSTU layer's projections,
//   C[n1][n2] = sa * sb * sum_t A[t][n1] * B[t][n2],
// from row-major operands that hold one token per row: x^T dz of the UVQK
// projection (A = LN(x) [T, 512], B = d(uvqk) [T, 2048]) and y^T dout of the
// output projection (A = y [T, 1536], B = dout [T, 512]), for MI355X (gfx950).
// Reference behaviour followed (paths relative to
// recommendation_v4/hstu/generative_recommenders/):
//   bf16 wgrad dw = x^T dz         ops/triton/triton_addmm.py:1737-1750
//   output-projection wgrad        ops/triton/triton_hstu_linear.py (torch.mm(y.t(), dout))
//   split-K over tokens, fixed-    ops/triton/fp8_wgrad.py:27-160 (fp8_wgrad: fp32
//   order second pass                partials [SPLIT, N1, N2], reduce, then the scales)
//
// Design: the output is small (0.75-1 M elements) and the contraction long
// (T ~ 162 K tokens), so the tokens are split over workgroups: tiles x split
// ~ one workgroup per CU.  A workgroup owns a 256 (n1) x 256 (n2) tile of one
// token range; 8 waves as 4 (n1) x 2 (n2) of 64 x 128.  Token rows lie in LDS
// as in memory, and the MFMA operands come out with the transposed reads
// (ds_read_b64_tr_b16, _b8), which turn a token-major tile into
// k(token)-contiguous fragments with the same token order in both operands.
// The MFMA (v_mfma_f32_16x16x32_bf16, 16x16x128_f8f6f4) runs with B as its A
// operand, so a lane's result is 4 consecutive n2 of one n1 row.
// What bounds it: the transposed reads and the MFMAs, close to equal (for fp8
// 1 900 LDS cycles against 2 050 MFMA cycles a step), so the two must
// overlap although the eight waves meet at a barrier every step: the
// fragments roll.  A fragment's registers are refilled with the next step's as
// soon as its last MFMA is issued, so the LDS reads of step k + 1 run under the
// MFMAs of step k, and step k's LDS buffer is already free while its MFMAs run:
// LDS DMA (inline assembly, explicit waits, spread between the MFMAs) fills it
// with the step that comes a whole ring later.  One barrier per step.
// Rows are unpadded; 16-byte chunk c of row r sits at c ^ swz(r), which spreads
// the transposed reads over all banks.
// Measured, product + second pass, against operands loaded through registers and
// read from padded LDS all at once behind the barrier, in us:
//                                       512 x 2048      1536 x 512
//   bf16 T = 162 251                   327 -> 296      256 -> 232  (1.15 / 1.10 PFLOP/s)
//   bf16 T = 162 251, column sums too  346 -> 327      265 -> 249
//   bf16 T =  37 429                  95.2 -> 87.7    76.8 -> 70.9
//   fp8  T = 162 251                   183 -> 176      140 -> 137
//   fp8  T =  37 429                  57.9 -> 55.5    48.9 -> 47.4
// Matrix cores busy 61 % (bf16) and 46 % (fp8) of the time, the LDS at 0.55 and
// 0.43 of its read rate: the two overlap, but not wholly across the barrier.
// Workgroups are numbered so that the tiles of one token range run on one XCD
// and share its L2.  With split > 1 every workgroup writes an fp32 partial
// tile; a second kernel sums the splits in a fixed order, applies sa * sb and
// writes bf16 or fp32 (bitwise reproducible, no atomics).  Optionally (bf16)
// the workgroups of the first n1 tile also sum B's columns from LDS (the
// projection's bias gradient), so the layer needs no separate pass over
// d(uvqk) for it.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "hstu_common.h"
#include "hstu_mi355x.h"

namespace {
using namespace hstu;

constexpr int kWThreads = 512;  // 8 waves
constexpr int kBN1 = 256, kBN2 = 256;  // output tile
constexpr int kCus = 256;

// Per operand format: bf16 steps of 32 tokens (512-byte tile rows) in a ring of
// four, fp8 steps of 128 tokens (256-byte rows) in a ring of two: 128 KiB.
template <bool F8>
struct WCfg {
  static constexpr int KT = F8 ? 128 : 32;  // tokens per k-step
  static constexpr int RING = F8 ? 2 : 4;
  static constexpr int ES = F8 ? 1 : 2;     // bytes per element
  static constexpr int ROW = kBN1 * ES;     // tile row bytes
  static constexpr int TILE = KT * ROW;
  static constexpr int STAGE = 2 * TILE;    // A tile then B tile
  static constexpr int LDS = RING * STAGE;
  static constexpr int CPR = ROW / 16;      // 16-byte chunks per tile row
  static constexpr int NDMA = TILE / 1024 / 8;  // loads per wave and operand
  // bf16: a pass of a transposed read takes 8 rows x 2 chunks; fp8: 16 rows x 1
  __host__ __device__ static constexpr int swz(int r) { return F8 ? r & 15 : 2 * (r & 7); }
};
constexpr int kWLds = WCfg<false>::LDS;
static_assert(WCfg<true>::LDS == kWLds, "one LDS size");


struct WgradParams {
  const uint8_t* A;
  const uint8_t* B;
  int64_t lda, ldb;  // bytes
  int64_t T;
  int64_t tps;  // tokens per split, a multiple of kKT
  int N1, N2;
  int split, tiles_n2, tiles;
  float* ws;     // [split][N1][N2] fp32 partials when split > 1
  float* cs_ws;  // [split][N2] column-sum partials when split > 1
  float* colsum; // fp32 [N2]: sum over the tokens of B, or null (bf16 only)
  void* out;
  int64_t ldo;  // elements
  int out_f32;
  const float* sa;
  const float* sb;
};

// F8: A and B fp8 with MFMA formats FA / FB (0 e4m3, 1 e5m2); else bf16.
template <bool F8, int FA, int FB>
__global__ void __launch_bounds__(kWThreads, 1) wgrad_kernel(WgradParams p) {
  using C = WCfg<F8>;
  constexpr int kKT = C::KT;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  // XCD-contiguous numbering: workgroup b runs on XCD b % 8; consecutive idx
  // (one token range, all its tiles) land on one XCD.
  const int total = p.tiles * p.split;
  const int per_xcd = (total + 7) / 8;
  const int idx = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (idx >= total) return;
  const int s = idx / p.tiles, tile = idx - s * p.tiles;
  const int t1 = tile / p.tiles_n2, t2 = tile - t1 * p.tiles_n2;
  const int n10 = t1 * kBN1, n20 = t2 * kBN2;
  const int64_t tb = (int64_t)s * p.tps;
  const int64_t te = min(tb + p.tps, p.T);
  const int nk = (int)((te - tb + kKT - 1) / kKT);

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15,
            g = lane >> 4;
  const int w1 = (wave >> 1) * 64, w2 = (wave & 1) * 128;

  // Token rows tb .. te-1 of the tile's column band; rows past te (the next
  // split's, or past T) read as zero.
  const uint32_t lda = (uint32_t)p.lda, ldb = (uint32_t)p.ldb;
  const uint32_t a_bytes = (uint32_t)((te - tb - 1) * p.lda + C::ROW), b_bytes = (uint32_t)((te - tb - 1) * p.ldb + C::ROW);
  const i32x4 ar = rsrc_sgprs(p.A + tb * p.lda + n10 * C::ES, a_bytes);
  const i32x4 br = rsrc_sgprs(p.B + tb * p.ldb + n20 * C::ES, b_bytes);
  // LDS slot q = 64 i + lane of a tile is row q / CPR, position q % CPR
  uint32_t va[C::NDMA], vb[C::NDMA];
#pragma unroll
  for (int j = 0; j < C::NDMA; ++j) {
    const int q = 64 * (C::NDMA * wave + j) + lane, row = q / C::CPR, ch = (q % C::CPR) ^ C::swz(row);
    va[j] = row * lda + ch * 16;
    vb[j] = row * ldb + ch * 16;
  }
  const uint32_t lds0 =
      __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t*)smem);
  // load i (0 .. 2 NDMA - 1) of step kk < nk; rows past the range read zeros
  auto issue = [&](int kk, auto i_c) {
    constexpr int i = decltype(i_c)::value, j = i % C::NDMA;
    const uint32_t dst = lds0 + (uint32_t)((kk % C::RING) * C::STAGE) + 1024u * (uint32_t)(C::NDMA * wave + j);
    if constexpr (i < C::NDMA) dma_to_lds(dst, va[j], ar, (uint32_t)kk * kKT * lda);
    else dma_to_lds(dst + C::TILE, vb[j], br, (uint32_t)kk * kKT * ldb);
  };
  // all but this wave's last `later` (< RING) steps of loads have landed, then every wave's
  auto wait_steps = [&](int later) {
    constexpr int S = 2 * C::NDMA;
    if (later >= 3) dma_barrier<3 * S>();
    else if (later == 2) dma_barrier<2 * S>();
    else if (later == 1) dma_barrier<S>();
    else dma_barrier<0>();
  };

  // column sums of B (the bias gradient of the layer's projection) by the
  // workgroups of the first n1 tile: thread tid sums chunk tid % 32 of rows
  // tid / 32 + 16 q of every step
  const bool do_cs = !F8 && p.colsum != nullptr && t1 == 0;
  float cs[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto add_cols = [&](const uint8_t* bt) {
#pragma unroll
    for (int q = 0; q < kKT / 16; ++q) {
      const int row = (tid >> 5) + 16 * q;
      const u32x4 v = lds_ld128(bt + row * C::ROW + (((tid & 31) ^ C::swz(row)) * 16));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = v[e];
        cs[2 * e] += __builtin_bit_cast(float, w << 16);
        cs[2 * e + 1] += __builtin_bit_cast(float, w & 0xffff0000u);
      }
    }
  };

  f32x4 acc[8][4];  // [n2 block][n1 block], lane: n1 = 16i + li, n2 = 16j + 4g .. +3
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[j][i] = zero4();

  // Transposed reads of column block c0 (16 columns).  bf16: lane (li, g) of
  // the two reads addresses token rows 4g + li/4 (+16), columns 4 (li % 4); fp8:
  // rows 8g + li/2 (+32 per read, four reads), columns 8 (li % 2); a lane then
  // holds the same tokens of its column in both operands.
  const int r0 = F8 ? 8 * g + (li >> 1) : 4 * g + (li >> 2);
  const int in0 = (li & 1) * 8, ch0 = F8 ? 0 : (li >> 1) & 1;
  const int rd0 = r0 * C::ROW + in0, sw0 = (ch0 ^ C::swz(r0)) * 16;
  using Frag = std::conditional_t<F8, i32x8, u32x4>;
  auto frag = [&](const uint8_t* t, int c0) {  // c0 * ES is a multiple of 16 (fp8) or 32 (bf16) bytes
    const uint8_t* q = t + rd0 + ((c0 * C::ES) ^ sw0);
    if constexpr (F8) {
      const u32x2 x0 = lds_tr8(q), x1 = lds_tr8(q + 32 * C::ROW);
      const u32x2 x2 = lds_tr8(q + 64 * C::ROW), x3 = lds_tr8(q + 96 * C::ROW);
      i32x8 f;
      f[0] = (int)x0[0]; f[1] = (int)x0[1]; f[2] = (int)x1[0]; f[3] = (int)x1[1];
      f[4] = (int)x2[0]; f[5] = (int)x2[1]; f[6] = (int)x3[0]; f[7] = (int)x3[1];
      return f;
    } else {
      return cat_tr(lds_tr16(q), lds_tr16(q + 16 * C::ROW));
    }
  };
  Frag af[4], bfr[8];
  if (nk > 0) {
    static_for<C::RING>([&](auto k_c) {
      if (decltype(k_c)::value < nk)
        static_for<2 * C::NDMA>([&](auto i_c) { issue(decltype(k_c)::value, i_c); });
    });
    wait_steps(min(C::RING, nk) - 1);  // step 0 has landed
#pragma unroll
    for (int i = 0; i < 4; ++i) af[i] = frag(smem, w1 + 16 * i);
#pragma unroll
    for (int j = 0; j < 8; ++j) bfr[j] = frag(smem + C::TILE, w2 + 16 * j);
    if (do_cs) add_cols(smem + C::TILE);
  }
  // step kk, at whose start step kk + 1 has landed and every wave has read step
  // kk: its buffer takes step kk + RING (MORE); NEXT: there is a step kk + 1
  auto step = [&](int kk, auto more_c, auto next_c) {
    constexpr bool MORE = decltype(more_c)::value, NEXT = decltype(next_c)::value;
    const uint8_t* nb = smem + ((kk + 1) % C::RING) * C::STAGE;
    static_for<8>([&](auto j_c) {
      constexpr int j = decltype(j_c)::value;
      static_for<4>([&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        if constexpr (F8)
          acc[j][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bfr[j], af[i], acc[j][i], FB, FA, 0, 0, 0, 0);
        else
          acc[j][i] = mfma_bf16(bfr[j], af[i], acc[j][i]);
        if constexpr (NEXT && j == 7) af[i] = frag(nb, w1 + 16 * i);
      });
      if constexpr (NEXT) bfr[j] = frag(nb + C::TILE, w2 + 16 * j);
      if constexpr (MORE && j < 2 * C::NDMA) issue(kk + C::RING, j_c);
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (NEXT) {
      if (do_cs) add_cols(nb + C::TILE);
    }
  };
  // the last RING steps issue nothing: loads of zeros past the range kept one
  // wait count for all steps, but cost the shortest calls 0.5 us of LDS writes
  // (T = 33 12.5 -> 11.7 us, T = 300 20.3 -> 19.7; 512 x 2048, bf16)
  int kk = 0;
  for (; kk + C::RING < nk; ++kk) {
    dma_barrier<(C::RING - 2) * 2 * C::NDMA>();
    step(kk, std::true_type{}, std::true_type{});
  }
  for (; kk + 1 < nk; ++kk) {
    wait_steps(min(C::RING - 2, nk - 2 - kk));
    step(kk, std::false_type{}, std::true_type{});
  }
  if (nk > 0) step(kk, std::false_type{}, std::false_type{});
  if (do_cs) __syncthreads();  // every wave has read the last steps' buffers, which the sums below overwrite

  if (do_cs) {
    // fold the 16 row slots (tid / 32) of each column in LDS, in a fixed order
    float* red = (float*)smem;
#pragma unroll
    for (int e = 0; e < 8; ++e) red[(tid >> 5) * 256 + (tid & 31) * 8 + e] = cs[e];
    __syncthreads();
    if (tid < 256) {
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < 16; ++k) t += red[k * 256 + tid];
      if (p.split > 1) p.cs_ws[(int64_t)s * p.N2 + n20 + tid] = t;
      else p.colsum[n20 + tid] = t;
    }
  }
  if (p.split > 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n1 = n10 + w1 + 16 * i + li;
      float* row = p.ws + ((int64_t)s * p.N1 + n1) * p.N2 + n20 + w2 + 4 * g;
#pragma unroll
      for (int j = 0; j < 8; ++j) *(f32x4*)(row + 16 * j) = acc[j][i];
    }
    return;
  }
  const float sc = (p.sa ? p.sa[0] : 1.f) * (p.sb ? p.sb[0] : 1.f);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n1 = n10 + w1 + 16 * i + li;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int n2 = n20 + w2 + 16 * j + 4 * g;
      const f32x4 v = acc[j][i] * sc;
      if (p.out_f32) *(f32x4*)((float*)p.out + (int64_t)n1 * p.ldo + n2) = v;
      else *(u32x2*)((uint16_t*)p.out + (int64_t)n1 * p.ldo + n2) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    }
  }
}

// out[n1][n2] = sa * sb * sum_{s < split} ws[s][n1][n2], summed in split order;
// 4 consecutive n2 per thread; the threads past N1 * N2 / 4 do the same for
// the column sums (colsum[n2] = sum_s cs_ws[s][n2], unscaled).  split == 0
// writes zeros (no tokens).
__global__ void __launch_bounds__(256) wgrad_reduce_kernel(const float* __restrict__ ws, int split, int N1, int N2,
                                                           const float* __restrict__ sa,
                                                           const float* __restrict__ sb, void* __restrict__ out,
                                                           int64_t ldo, int out_f32, const float* __restrict__ cs_ws,
                                                           float* __restrict__ colsum) {
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t numel = (int64_t)N1 * N2;
  if (e >= numel) {
    const int64_t c = e - numel;
    if (colsum == nullptr || c >= N2) return;
    f32x4 t = zero4();
    for (int s = 0; s < split; ++s) t += *(const f32x4*)(cs_ws + (int64_t)s * N2 + c);
    *(f32x4*)(colsum + c) = t;
    return;
  }
  f32x4 acc = zero4();
  for (int s = 0; s < split; ++s) acc += *(const f32x4*)(ws + s * numel + e);
  acc *= (sa ? sa[0] : 1.f) * (sb ? sb[0] : 1.f);
  const int64_t n1 = e / N2, n2 = e - n1 * N2;
  if (out_f32) *(f32x4*)((float*)out + n1 * ldo + n2) = acc;
  else *(u32x2*)((uint16_t*)out + n1 * ldo + n2) = u32x2{pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3])};
}

hipError_t set_wgrad_lds(const void* fn) {
  static std::mutex mu;
  static std::vector<const void*> done;
  std::lock_guard<std::mutex> lock(mu);
  for (const void* d : done)
    if (d == fn) return hipSuccess;
  hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kWLds);
  if (e == hipSuccess) done.push_back(fn);
  return e;
}

// tokens per split for a requested split (<= 0: about one workgroup per CU,
// at least 4 k-steps per split), and the split that results
constexpr int kPlanKT = 128;  // token ranges are multiples of both formats' k-steps
void plan(int64_t T, int N1, int N2, int split, int64_t* tps, int* eff) {
  const int tiles = (N1 / kBN1) * (N2 / kBN2);
  if (split <= 0) split = (int)std::max<int64_t>(1, std::min<int64_t>(kCus / std::max(tiles, 1), (T + 127) / 128));
  if (T <= 0) {
    *tps = kPlanKT;
    *eff = 0;
    return;
  }
  const int64_t per = (T + split - 1) / split;
  *tps = (per + kPlanKT - 1) / kPlanKT * kPlanKT;
  *eff = (int)((T + *tps - 1) / *tps);
}

}  // namespace

extern "C" int hstu_wgrad_split(int64_t T, int N1, int N2, int split) {
  if (T < 0 || N1 <= 0 || N2 <= 0 || N1 % kBN1 || N2 % kBN2) return -1;
  int64_t tps;
  int eff;
  plan(T, N1, N2, split, &tps, &eff);
  return eff;
}

extern "C" int64_t hstu_wgrad_workspace_bytes(int64_t T, int N1, int N2, int split) {
  const int eff = hstu_wgrad_split(T, N1, N2, split);
  if (eff < 0) return -1;
  return eff > 1 ? (int64_t)eff * (N1 + 1) * N2 * 4 : 0;  // product and column-sum partials
}

extern "C" int hstu_wgrad(int a_dtype, const void* A, int64_t lda, int b_dtype, const void* B, int64_t ldb, int64_t T,
                          int N1, int N2, const float* scale_a, const float* scale_b, void* out, int64_t ldo,
                          int out_dtype, float* colsum_b, int split, void* workspace, int64_t workspace_bytes,
                          hipStream_t stream) {
  if (T < 0 || N1 <= 0 || N2 <= 0 || !out || (T > 0 && (!A || !B)) || lda < N1 || ldb < N2 || ldo < N2 ||
      (out_dtype != HSTU_DTYPE_BF16 && out_dtype != HSTU_DTYPE_FP32))
    return HSTU_E_BAD_ARG;
  const bool bf16 = a_dtype == HSTU_DTYPE_BF16 && b_dtype == HSTU_DTYPE_BF16;
  const bool f8 = a_dtype == HSTU_DTYPE_FP8_E4M3 && (b_dtype == HSTU_DTYPE_FP8_E4M3 || b_dtype == HSTU_DTYPE_FP8_E5M2);
  if (!bf16 && !f8) return HSTU_E_UNSUPPORTED;
  const int es = bf16 ? 2 : 1;
  if (colsum_b && (!bf16 || (uintptr_t)colsum_b % 16)) return HSTU_E_UNSUPPORTED;
  if (N1 % kBN1 || N2 % kBN2 || (lda * es) % 16 || (ldb * es) % 16 || ((uintptr_t)A | (uintptr_t)B) % 16 ||
      (uintptr_t)out % (out_dtype == HSTU_DTYPE_FP32 ? 16 : 8) || ldo % 4)
    return HSTU_E_UNSUPPORTED;
  int64_t tps;
  int eff;
  plan(T, N1, N2, split, &tps, &eff);
  const int64_t need = eff > 1 ? (int64_t)eff * (N1 + 1) * N2 * 4 : 0;
  if (workspace_bytes < need || (need > 0 && !workspace)) return HSTU_E_BAD_ARG;
  // one split's rows must stay within 32-bit buffer offsets
  if ((tps + kPlanKT) * std::max(lda, ldb) * es >= ((int64_t)1 << 32)) return HSTU_E_UNSUPPORTED;
  const int tiles = (N1 / kBN1) * (N2 / kBN2);
  const int out_f32 = out_dtype == HSTU_DTYPE_FP32;
  if (eff > 0) {
    WgradParams p{};
    p.A = (const uint8_t*)A;
    p.B = (const uint8_t*)B;
    p.lda = lda * es;
    p.ldb = ldb * es;
    p.T = T;
    p.tps = tps;
    p.N1 = N1;
    p.N2 = N2;
    p.split = eff;
    p.tiles_n2 = N2 / kBN2;
    p.tiles = tiles;
    p.ws = (float*)workspace;
    p.cs_ws = eff > 1 ? (float*)workspace + (int64_t)eff * N1 * N2 : nullptr;
    p.colsum = colsum_b;
    p.out = out;
    p.ldo = ldo;
    p.out_f32 = out_f32;
    p.sa = scale_a;
    p.sb = scale_b;
    const int64_t total = (int64_t)tiles * eff;
    if (total >= ((int64_t)1 << 31)) return HSTU_E_UNSUPPORTED;
    const int grid = (int)((total + 7) / 8 * 8);
    const void* kern = bf16 ? (const void*)wgrad_kernel<false, 0, 0>
                       : b_dtype == HSTU_DTYPE_FP8_E5M2 ? (const void*)wgrad_kernel<true, 0, 1>
                                                         : (const void*)wgrad_kernel<true, 0, 0>;
    hipError_t e = set_wgrad_lds(kern);
    if (e != hipSuccess) return (int)e;
    void* args[] = {&p};
    e = hipLaunchKernel(kern, dim3(grid), dim3(kWThreads), args, (size_t)kWLds, stream);
    if (e != hipSuccess) return (int)e;
  }
  if (eff != 1) {
    const int64_t threads = (int64_t)N1 * N2 / 4 + (colsum_b ? N2 / 4 : 0);
    const float* cs_ws = eff > 1 ? (const float*)workspace + (int64_t)eff * N1 * N2 : nullptr;
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream,
                       (const float*)workspace, eff, N1, N2, scale_a, scale_b, out, ldo, out_f32, cs_ws, colsum_b);
  }
  return (int)hipGetLastError();
}
