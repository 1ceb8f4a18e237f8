// Prompt prefill for gfx950: the decoder layers over S prompt rows with fp32
// arithmetic carried on the fp16 matrix cores, the K/V rows written to the
// static cache, and the last row's greedy token.
//
// fp32 on fp16 MFMA.  The weights are fp16, so only the activations need more
// than one fp16 value: an activation row x is scaled by a power of two that
// puts its largest value in [2^13, 2^14) and split into hi = fp16(x) and
// lo = fp16(x - hi), 22 bits in all (values down to 2^-15 of the largest keep
// them; below that the split's absolute error is 2^-39 of the largest).
// W.x = W.hi + W.lo then takes two MFMAs per tile with exact products and
// fp32 accumulation.  Measured against 64 bits on N(0, 1) rows, K = 2048: 4.1e-7
// relative, where an fp32 GEMM has 8.1e-7.  gfx950 has no faster fp32-input
// MFMA (157 TFLOP/s, against 2 x 16 bits of 2500).
//
// One layer is nine launches:
//   rows      h += the previous GEMM's partials; RMSNorm; split image + scale
//   gemm      qkv partials
//   qkv_prep  q/k head RMSNorm + M-RoPE, K/V cache rows, split images of q, k
//             and of V transposed (the attention's operand orders)
//   attention causal flash attention on the split images, split image out
//   gemm      o_proj partials
//   rows      h += partials; RMSNorm; split image
//   gemm      gate_up partials
//   silu      silu(gate) * up, split image + scale
//   gemm      down partials
// A GEMM may split K over z workgroups per tile (few rows, where a tile grid
// leaves CUs idle); its z partial planes are summed in order by the next
// launch, which reads them anyway.
//
// Replaces the prefill of the reference's greedy engine
// (evaluation_wrapper.py:218-228, a full HF forward).

#include <math.h>

#include <type_traits>

#include "qd_common.h"
#include "qd_kernels.h"

namespace qd {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kHD = 128;        // head dim
constexpr int kKvTile = 64;     // K/V rows per attention tile
constexpr int kMaxExp = 110;

// ---------------------------------------------------------------- fp16 splits

// Exponent e with amax * 2^-e in [2^13, 2^14), clamped so that 2^e and 2^-e
// are normal fp32 numbers (0 and non-finite maxima give a clamped one).
__device__ __forceinline__ int split_exp(float amax) {
  const int e = (int)((__builtin_bit_cast(unsigned, amax) >> 23) & 0xffu) - 127 - 13;
  return min(max(e, -kMaxExp), kMaxExp);
}
__device__ __forceinline__ float pow2f(int e) {   // -126 <= e <= 127
  return __builtin_bit_cast(float, (unsigned)(e + 127) << 23);
}
// x is made opaque first: where it is a product, the compiler may otherwise
// round the stored hi straight from the exact product (v_fma_mixlo_f16) and the
// hi inside lo from the fp32 product, which differ by an fp16 step now and then.
__device__ __forceinline__ void split2(float x, _Float16& hi, _Float16& lo) {
  asm("" : "+v"(x));
  hi = (_Float16)x;
  lo = (_Float16)(x - (float)hi);
}

// 8 consecutive values (already scaled) to the two planes.
__device__ __forceinline__ void store_split8(uint16_t* hi, uint16_t* lo, const float* u) {
  h8 a, b;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    _Float16 x, y;
    split2(u[i], x, y);
    a[i] = x;
    b[i] = y;
  }
  *reinterpret_cast<h8*>(hi) = a;
  *reinterpret_cast<h8*>(lo) = b;
}

__device__ __forceinline__ float block_max(float v, float* s_red, int nw) {
  v = wave_max(v);
  if (lane_id() == 0) s_red[threadIdx.x / kWave] = v;
  __syncthreads();
  v = s_red[0];
  for (int i = 1; i < nw; ++i) v = fmaxf(v, s_red[i]);
  __syncthreads();
  return v;
}
__device__ __forceinline__ float block_sum(float v, float* s_red, int nw) {
  v = wave_sum(v);
  if (lane_id() == 0) s_red[threadIdx.x / kWave] = v;
  __syncthreads();
  v = s_red[0];
  for (int i = 1; i < nw; ++i) v += s_red[i];
  __syncthreads();
  return v;
}

// ---------------------------------------------------------------- asynchronous LDS tiles

// A word at a wave-uniform address, written by an earlier launch, as a scalar
// load: a vector load would make its reader wait for the tile loads in flight.
__device__ __forceinline__ int ld_scalar(const int* p) {
  return *(const __attribute__((address_space(4))) int*)p;
}

// 16 bytes per lane from global memory straight to LDS (lane i lands at
// l + 16 i; l is wave-uniform).
__device__ __forceinline__ void load_lds16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                   (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

// This wave's LDS reads are done and at most N of its loads are in flight,
// then the workgroup barrier.  The loads that a tile's readers need are older
// than the N allowed ones, and a tile is refilled only after the barrier that
// follows its last read.
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0070);   // vmcnt(N) lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

// Stage I of a kernel's tile ring.  Separate variables, not slices of one: the
// compiler then knows that reading one stage does not depend on the loads in
// flight to another and puts no wait of its own between them.
template <int I, int N>
__device__ __forceinline__ char* lds_stage() {
  __shared__ __align__(16) char buf[N];
  return buf;
}

}  // namespace

// ---------------------------------------------------------------- split GEMM

// y[z][m][n] = scale[m] * sum over the z-th K range (K / BK blocks, divided as
// evenly as they go) of W[n][k] (hi + lo)[m][k].
//
// Tile BM x BN, BK of K per stage (hi, lo and W rows), NS stages filled by
// asynchronous global-to-LDS loads NS - 1 steps ahead.  16-byte chunk c of row
// r sits at c ^ (r % 8) (rows of 128 or 256 bytes; c ^ (r / 2 % 4) for 64), so that
// the 16 rows a fragment read touches spread over all banks; the permutation is
// applied to the source address, since the load's LDS side is contiguous.  W is
// the MFMA A operand, so a lane holds four consecutive outputs of one row.
// Consecutive tiles of one XCD share their W rows (the m tiles of one n band),
// which then come out of its L2.
template <int BM, int BN, int BK, int WM, int WN, int NS>
__global__ __launch_bounds__(kWave * WM * WN) void split_gemm_kernel(const SplitGemmArgs a) {
  constexpr int NW = WM * WN;
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int CH = BK / 8;
  constexpr int RPI = kWave / CH;                       // rows per load
  constexpr int GA = BM / RPI, GW = BN / RPI;           // loads per stage: of one plane, of W
  constexpr int LA = (GA + NW - 1) / NW, LW = (GW + NW - 1) / NW;   // and wave
  constexpr int LOADS = 2 * LA + LW;
  constexpr int PA = 2 * BM * BK, STAGE = 2 * PA + 2 * BN * BK;   // bytes
  static_assert(BM % RPI == 0 && BN % RPI == 0 && TM % 16 == 0 && TN % 16 == 0 && (CH == 16 || CH == 8 || CH == 4) &&
                    LOADS * (NS - 1) < 64 && NS == 3, "tile shape");
  const int lane = lane_id();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int tiles_m = (a.M + BM - 1) / BM;
  const int q = (int)gridDim.x >> 3, r = (int)gridDim.x & 7, xcd = (int)blockIdx.x & 7, loc = (int)blockIdx.x >> 3;
  const int t = xcd * q + min(xcd, r) + loc;
  const int m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;
  const int kblocks = a.K / BK, kfirst = kblocks * (int)blockIdx.y / (int)gridDim.y;
  const int nk = kblocks * ((int)blockIdx.y + 1) / (int)gridDim.y - kfirst;
  const long kbase = (long)kfirst * BK;
  const int lr = lane / CH, lc = lane % CH;
  // where the waves do not divide the loads, the last load is issued more than
  // once (same data, same place), so that every wave counts the same number
  unsigned offA[LA], offW[LW];
  int dstA[LA], dstW[LW];
  auto swz = [](int r) { return CH == 4 ? ((r >> 1) & 3) : (r & 7); };
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int g = min(i * NW + w, GA - 1), r = g * RPI + lr;
    dstA[i] = g * 1024;
    offA[i] = ((unsigned)min(m0 + r, a.M - 1) * (unsigned)a.K + (lc ^ swz(r)) * 8) * 2u;
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int g = min(i * NW + w, GW - 1), r = g * RPI + lr;
    dstW[i] = 2 * PA + g * 1024;
    offW[i] = ((unsigned)min(n0 + r, a.N - 1) * (unsigned)a.K + (lc ^ swz(r)) * 8) * 2u;
  }
  const char* Ah = reinterpret_cast<const char*>(a.hi + kbase);
  const char* Al = reinterpret_cast<const char*>(a.lo + kbase);
  const char* Wp = reinterpret_cast<const char*>(a.W + kbase);
  auto issue = [&](auto S, int k) {
    char* st = lds_stage<decltype(S)::value, STAGE>();
    const long ko = (long)k * BK * 2;
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      load_lds16(Ah + ko + offA[i], st + dstA[i]);
      load_lds16(Al + ko + offA[i], st + PA + dstA[i]);
    }
#pragma unroll
    for (int i = 0; i < LW; ++i) load_lds16(Wp + ko + offW[i], st + dstW[i]);
  };
  f32x4 acc[TM / 16][TN / 16];
#pragma unroll
  for (int i = 0; i < TM / 16; ++i)
#pragma unroll
    for (int j = 0; j < TN / 16; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = w / WN, wn = w % WN;
  const int fr = lane & 15, fg = lane >> 4;
  const int fs = swz(fr);
  // byte offsets of this lane's fragments, opaque so that every fragment
  // address stays one base plus a constant
  unsigned bA[BK / 32], bW[BK / 32];
#pragma unroll
  for (int ks = 0; ks < BK / 32; ++ks) {
    const unsigned co = ((4 * ks + fg) ^ fs) * 16;
    bA[ks] = (wm * TM + fr) * BK * 2 + co;
    bW[ks] = 2 * PA + (wn * TN + fr) * BK * 2 + co;
    asm("" : "+v"(bA[ks]));
    asm("" : "+v"(bW[ks]));
  }
  auto compute = [&](auto S) {
    const char* st = lds_stage<decltype(S)::value, STAGE>();
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      h8 fw[TN / 16];
#pragma unroll
      for (int j = 0; j < TN / 16; ++j) fw[j] = *reinterpret_cast<const h8*>(st + bW[ks] + 32 * j * BK);
#pragma unroll
      for (int i = 0; i < TM / 16; ++i) {
        const h8 fh = *reinterpret_cast<const h8*>(st + bA[ks] + 32 * i * BK);
        const h8 fl = *reinterpret_cast<const h8*>(st + bA[ks] + PA + 32 * i * BK);
#pragma unroll
        for (int j = 0; j < TN / 16; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[j], fh, acc[i][j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < TN / 16; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[j], fl, acc[i][j], 0, 0, 0);
      }
    }
  };
  auto full = [&](auto S, int k) {   // steady state: stage k + 2 is refilled while k is used
    wait_barrier<LOADS>();
    issue(std::integral_constant<int, (decltype(S)::value + 2) % 3>{}, k + 2);
    compute(S);
  };
  auto tail = [&](auto S, int k) {
    if (k >= nk) return;
    if (k + 1 < nk)
      wait_barrier<LOADS>();
    else
      wait_barrier<0>();
    if (k + 2 < nk) issue(std::integral_constant<int, (decltype(S)::value + 2) % 3>{}, k + 2);
    compute(S);
  };
  const std::integral_constant<int, 0> s0;
  const std::integral_constant<int, 1> s1;
  const std::integral_constant<int, 2> s2;
  issue(s0, 0);
  if (nk > 1) issue(s1, 1);
  int k = 0;
#pragma unroll 1
  for (; k + 4 < nk; k += 3) {
    full(s0, k);
    full(s1, k + 1);
    full(s2, k + 2);
  }
#pragma unroll 1
  for (; k < nk; k += 3) {
    tail(s0, k);
    tail(s1, k + 1);
    tail(s2, k + 2);
  }
  float scale[TM / 16];
#pragma unroll
  for (int i = 0; i < TM / 16; ++i)
    scale[i] = a.scale[min(m0 + wm * TM + 16 * i + fr, a.M - 1)];
  float* y = a.y + (long)blockIdx.y * a.M * a.N;
#pragma unroll
  for (int i = 0; i < TM / 16; ++i) {
    const int m = m0 + wm * TM + 16 * i + fr;
    if (m < a.M) {
#pragma unroll
      for (int j = 0; j < TN / 16; ++j) {
        const int n = n0 + wn * TN + 16 * j + 4 * fg;
        if (n < a.N) *reinterpret_cast<f32x4*>(y + (long)m * a.N + n) = acc[i][j] * scale[i];
      }
    }
  }
}

namespace {

// Tile shapes (8 waves; wide wave tiles read the LDS least, since a wave reads its
// W rows once for both planes) and their cost: `ramp` us per workgroup and `us`
// per 1024 of K with every CU busy, `idle` of that on an almost idle chip, and
// the TB/s its loads and stores reach.  Fitted to every shape and K split at
// 1 .. 4001 rows of the four 2B products (W cold, one workgroup per CU; 4 to 8 %
// rms, the chosen pair 2.8 % behind the best measured one on average); other products
// and more rows run on what that extrapolates, which nothing measured.  The widths
// of 192 and the rows below 64 are there for the rounds: 1024 x 12288 x 2048 takes
// 192 workgroups of 256 x 256 (98 us) or 256 of 256 x 192 (88), 512 rows 58 or 53
// us; 1300 x 12288 x 2048 148 us on 128 x 128, 134 on 192 x 192.  16 rows of 12288
// x 2048 take 14.1 us on 64-row tiles, 11.6 on 32 x 128 with 128 of K per stage.
struct GemmTile {
  int bm, bn, bk;
  float ramp, us, idle, tbs;
};
constexpr GemmTile kGemmTiles[] = {
    {256, 256, 32, 12.0f, 46.6f, 0.71f, 3.75f}, {256, 192, 32, 9.2f, 37.8f, 0.76f, 3.69f},
    {192, 192, 32, 7.3f, 31.6f, 0.80f, 3.71f},  {128, 256, 32, 7.5f, 26.2f, 0.75f, 3.45f},
    {128, 128, 64, 4.2f, 14.4f, 0.77f, 3.59f},  {64, 256, 64, 4.3f, 15.9f, 0.77f, 4.71f},
    {64, 192, 64, 3.5f, 12.6f, 0.82f, 5.02f},   {64, 128, 64, 2.4f, 9.7f, 0.86f, 4.48f},
    {64, 64, 128, 2.1f, 6.1f, 0.95f, 4.15f},    {32, 128, 128, 2.4f, 7.3f, 0.82f, 5.36f},
    {32, 64, 128, 2.0f, 4.7f, 0.92f, 5.20f},    {16, 128, 128, 2.0f, 5.5f, 0.99f, 5.27f},
};

template <int BM, int BN, int BK, int WM, int WN>
int launch_gemm(const SplitGemmArgs& a, int z, hipStream_t s) {
  const unsigned t = (unsigned)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN));
  hipLaunchKernelGGL((split_gemm_kernel<BM, BN, BK, WM, WN, 3>), dim3(t, (unsigned)z), dim3(kWave * WM * WN), 0, s, a);
  return qd_host::launch_status("split_gemm_kernel");
}

}  // namespace

// The tile shape and K split with the least estimated time: rounds of workgroups
// over the CUs or the bytes they move, whichever is longer (summed in the fourth
// power, as the two overlap), plus the partial planes read again (~4 TB/s).
GemmPlan split_gemm_plan(long M, long N, long K) {
  GemmPlan best{-1, 1};
  float best_us = 0.f;
  const int cus = qd_host::cu_count();
  for (int c = 0; c < (int)(sizeof(kGemmTiles) / sizeof(kGemmTiles[0])); ++c) {
    const GemmTile& g = kGemmTiles[c];
    if (K % g.bk != 0) continue;
    for (int z : {1, 2, 3, 4, 6, 8, 12, kPrefillMaxSplit}) {
      if (K / g.bk < z) break;
      const long wgs = ((M + g.bm - 1) / g.bm) * ((N + g.bn - 1) / g.bn) * z;
      const long rounds = (wgs + cus - 1) / cus;
      const float fill = (float)wgs / (float)(rounds * cus);
      const float compute =
          (float)rounds * (g.ramp + (g.idle + (1.f - g.idle) * fill * fill) * g.us * (float)K / (float)z / 1024.f);
      const float planes = 4.f * (float)z * (float)M * (float)N;
      const float memory = 2.f + (2.f * (float)N * (float)K + 4.f * (float)M * (float)K + planes) / (g.tbs * 1e6f);
      const float c2 = compute * compute, m2 = memory * memory;
      const float us = sqrtf(sqrtf(c2 * c2 + m2 * m2)) + planes / 4e6f;
      if (best.tile < 0 || us < best_us) {
        best = GemmPlan{c, z};
        best_us = us;
      }
    }
  }
  return best;
}

int split_gemm_launch(const SplitGemmArgs& a, const GemmPlan& p, hipStream_t s) {
  constexpr int kTiles = sizeof(kGemmTiles) / sizeof(kGemmTiles[0]);
  if (a.M < 1 || a.N < 4 || a.N % 4 != 0 || p.tile < 0 || p.tile >= kTiles || p.z < 1 || p.z > kPrefillMaxSplit || a.K % kGemmTiles[p.tile].bk != 0 ||
      a.K / kGemmTiles[p.tile].bk < p.z)
    return QD_ERR_SHAPE;
  // 32-bit byte offsets into the operands
  if ((size_t)a.M * a.K * 2 >> 32 || (size_t)a.N * a.K * 2 >> 32) return QD_ERR_SHAPE;
  switch (p.tile) {
    case 0: return launch_gemm<256, 256, 32, 4, 2>(a, p.z, s);
    case 1: return launch_gemm<256, 192, 32, 4, 2>(a, p.z, s);
    case 2: return launch_gemm<192, 192, 32, 4, 2>(a, p.z, s);
    case 3: return launch_gemm<128, 256, 32, 4, 2>(a, p.z, s);
    case 4: return launch_gemm<128, 128, 64, 4, 2>(a, p.z, s);
    case 5: return launch_gemm<64, 256, 64, 4, 2>(a, p.z, s);
    case 6: return launch_gemm<64, 192, 64, 4, 2>(a, p.z, s);
    case 7: return launch_gemm<64, 128, 64, 4, 2>(a, p.z, s);
    case 8: return launch_gemm<64, 64, 128, 4, 2>(a, p.z, s);
    case 9: return launch_gemm<32, 128, 128, 2, 4>(a, p.z, s);
    case 10: return launch_gemm<32, 64, 128, 2, 4>(a, p.z, s);
    default: return launch_gemm<16, 128, 128, 1, 8>(a, p.z, s);
  }
}

namespace {

// ---------------------------------------------------------------- elementwise launches

// cos / sin of every (row, rotary pair), fp32 angles as the decode step's, and
// the argmax counter's zeros.
__global__ __launch_bounds__(256) void prefill_init_kernel(const PrefillArgs a) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < 64) a.argmax_count[i] = 0u;
  if (i >= (long)a.S * (kHD / 2)) return;
  const int row = (int)(i / (kHD / 2)), j = (int)(i % (kHD / 2));
  int st = 0;
  if (j % 3 == 1 && j < 3 * a.sec_h) st = 1;
  if (j % 3 == 2 && j < 3 * a.sec_w) st = 2;
  float s, c;
  sincosf((float)a.position_ids[(long)st * a.S + row] * a.inv_freq[j], &s, &c);
  a.cs[i] = make_float2(c, s);
}

constexpr int kRowChunks = 4;   // 8-value chunks per thread of a row: H up to 8192

// One row per workgroup, rows row0 .. row0 + grid: h[row] (+ the GEMM's z
// partial rows, or the prompt's embedding instead, layer 0), RMSNorm, split
// image and its scale (the partials, image and scales hold the grid's rows only).
// HBM / L2 bound: reads (z + 1) and writes 2 x 4 bytes per value.
template <bool EMBED>
__global__ __launch_bounds__(256) void prefill_rows_kernel(const PrefillArgs a, const float* part, int z,
                                                           const uint16_t* gamma, int row0) {
  __shared__ float s_red[4];
  const int row = row0 + (int)blockIdx.x;
  const long out = blockIdx.x, n = gridDim.x;
  const long H = a.H;
  float* hr = a.h + row * H;
  float u[kRowChunks][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < kRowChunks; ++c) {
    const long k = (long)c * 2048 + threadIdx.x * 8;
    if (k >= H) continue;
    if constexpr (EMBED) {
      if (row < a.n_vision) {
        if (a.vision_f32)
          load_act8<float>(reinterpret_cast<const float*>(a.vision) + row * H, k, u[c]);
        else
          load_act8<uint16_t>(reinterpret_cast<const uint16_t*>(a.vision) + row * H, k, u[c]);
      } else {
        load_act8<uint16_t>(a.embed + a.text_ids[row - a.n_vision] * H, k, u[c]);
      }
    } else {
      load_act8<float>(hr, k, u[c]);
      float p[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      const float* src = part + out * H + k;
#pragma unroll 8
      for (int i = 0; i < z; ++i) {
        float v[8];
        load_act8<float>(src, i * n * H, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] += v[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) u[c][e] += p[e];
    }
    store_act8<float>(hr, k, u[c]);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(u[c][e], u[c][e], ss);
  }
  if (gamma == nullptr) return;   // after the last layer only h is wanted
  const float rstd = rsqrtf(block_sum(ss, s_red, 4) / (float)H + a.eps);
  float mx = 0.f;
#pragma unroll
  for (int c = 0; c < kRowChunks; ++c) {
    const long k = (long)c * 2048 + threadIdx.x * 8;
    if (k >= H) continue;
    float g[8];
    unpack8(ld16(gamma + k), g);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      u[c][e] = (u[c][e] * rstd) * g[e];
      mx = fmaxf(mx, fabsf(u[c][e]));
    }
  }
  const int e2 = split_exp(block_max(mx, s_red, 4));
  const float sc = pow2f(-e2);
#pragma unroll
  for (int c = 0; c < kRowChunks; ++c) {
    const long k = (long)c * 2048 + threadIdx.x * 8;
    if (k >= H) continue;
#pragma unroll
    for (int e = 0; e < 8; ++e) u[c][e] *= sc;
    store_split8(a.img + out * H + k, a.img + (n + out) * H + k, u[c]);
  }
  if (threadIdx.x == 0) a.scale[out] = pow2f(e2);
}

constexpr int kMaxI = 16384;

// One row per workgroup: hidden = silu(gate) * up from the gate_up partials,
// split image and scale.  A few rows are bound by the chain of plane loads of a
// thread's chunks, so up to one row per CU takes 1024 threads and, at I = 6144, one
// chunk per thread; beyond, workgroups of 256 hide it and end more evenly.
// Measured, 256 / 1024 threads, us: 17 rows 5.8 / 4.5, 37 6.8 / 5.1, 128 6.6 / 5.6,
// 256 6.8 / 6.1, 300 7.3 / 8.1, 700 10.4 / 12.2, 4001 48.6 (6.1 TB/s) / 59.4.
template <int NT>
__global__ __launch_bounds__(NT) void prefill_silu_kernel(const PrefillArgs a, int z) {
  constexpr int kChunks = kMaxI / (8 * NT), kPlanes = NT > 256 ? 4 : 2;
  __shared__ float s_red[NT / kWave];
  const long row = blockIdx.x, n = gridDim.x;
  const long I = a.I;
  float u[kChunks][8];
  float mx = 0.f;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const long k = (long)c * 8 * NT + threadIdx.x * 8;
    if (k >= I) continue;
    float g[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, p[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll kPlanes
    for (int i = 0; i < z; ++i) {
      const float* src = a.part + (i * n + row) * 2 * I;
      float v[8], w[8];
      load_act8<float>(src, k, v);
      load_act8<float>(src + I, k, w);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        g[e] += v[e];
        p[e] += w[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      u[c][e] = (g[e] / (1.0f + expf(-g[e]))) * p[e];
      mx = fmaxf(mx, fabsf(u[c][e]));
    }
  }
  const int e2 = split_exp(block_max(mx, s_red, NT / kWave));
  const float sc = pow2f(-e2);
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const long k = (long)c * 8 * NT + threadIdx.x * 8;
    if (k >= I) continue;
#pragma unroll
    for (int e = 0; e < 8; ++e) u[c][e] *= sc;
    store_split8(a.img + row * I + k, a.img + (n + row) * I + k, u[c]);
  }
  if (threadIdx.x == 0) a.scale[row] = pow2f(e2);
}

// Exponent of a head-normalised and rotated vector's image: |x| <= sqrt(2 D) max |w|.
constexpr float kHeadBound = 16.f;
__device__ __forceinline__ int head_exp(const uint16_t* w) {
  const int j = lane_id();
  return split_exp(wave_max(fmaxf(fabsf(h2f(w[j])), fabsf(h2f(w[j + kHD / 2])))) * kHeadBound);
}

constexpr int kPrepThreads = 1024;

// Workgroups [0, q/k groups): 16 lanes per (row, q or k head), 4 rotary pairs
// each: head RMSNorm, rotation, split image; k also to the cache.  The others: one (kv head, 64
// rows) tile of V each: cache rows, and the split image of the tile transposed,
// [128 dims][64 rows] with the rows of each half in the order the PV product's
// operand holds its probabilities in: position 8 g + e is row
// 16 (e / 4) + 4 g + e % 4.  A thread owns one 16-byte chunk of that image, so 8
// rows of one dim; all its loads are issued before its first store (32 rows a
// thread, each stored before the next was loaded: 66 us instead of ~9 for 37
// rows and 8 planes).  The tile's exponent goes to vexp.
__global__ __launch_bounds__(kPrepThreads) void prefill_qkv_prep_kernel(const PrefillArgs a, const PrefillLayer L,
                                                                        int z, int qk_groups) {
  __shared__ float s_red[kPrepThreads / kWave];
  const long NQ = (long)(a.Hq + 2 * a.Hkv) * kHD;
  if ((int)blockIdx.x < qk_groups) {
    const long item = (long)blockIdx.x * (kPrepThreads / 16) + threadIdx.x / 16;
    const int heads = a.Hq + a.Hkv;
    const bool live = item < (long)a.S * heads;
    const int row = live ? (int)(item / heads) : a.S - 1, head = (int)(item % heads);
    const int j = (lane_id() & 15) * 4;   // dims [j, j + 4) and [64 + j, 64 + j + 4)
    const bool is_q = head < a.Hq;
    const uint16_t* nw = is_q ? L.q_norm : L.k_norm;
    const f32x4* csp = reinterpret_cast<const f32x4*>(a.cs + (long)row * (kHD / 2) + j);
    const f32x4 cs[2] = {csp[0], csp[1]};
    float f[2][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[0][e] = h2f(nw[j + e]);
      f[1][e] = h2f(nw[j + kHD / 2 + e]);
    }
    const float* src = a.part + (long)row * NQ + (long)head * kHD + j;
    f32x4 x[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll 4
    for (int i = 0; i < z; ++i) {
      x[0] += *reinterpret_cast<const f32x4*>(src + (long)i * a.S * NQ);
      x[1] += *reinterpret_cast<const f32x4*>(src + (long)i * a.S * NQ + kHD / 2);
    }
    float ss = 0.f, mx = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ss = __builtin_fmaf(x[h][e], x[h][e], ss);
        mx = fmaxf(mx, fabsf(f[h][e]));
      }
    const float rstd = rsqrtf(row16_sum(ss) / (float)kHD + a.eps);
    const float sc = pow2f(-split_exp(row16_max(mx) * kHeadBound));
    if (!live) return;
    h4 hi[2], lo[2], kc[2];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float c = cs[e / 2][2 * (e & 1)], s = cs[e / 2][2 * (e & 1) + 1];
      const float n0 = (x[0][e] * rstd) * f[0][e], n1 = (x[1][e] * rstd) * f[1][e];
      const float o[2] = {n0 * c - n1 * s, n1 * c + n0 * s};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        _Float16 a0, b0;
        split2(o[h] * sc, a0, b0);
        hi[h][e] = a0;
        lo[h][e] = b0;
        kc[h][e] = (_Float16)o[h];
      }
    }
    const int hh = is_q ? head : head - a.Hq;
    const long plane = (long)(is_q ? a.Hq : a.Hkv) * a.S * kHD;
    uint16_t* dst = (is_q ? a.q_img : a.k_img) + ((long)hh * a.S + row) * kHD + j;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      *reinterpret_cast<h4*>(dst + h * (kHD / 2)) = hi[h];
      *reinterpret_cast<h4*>(dst + plane + h * (kHD / 2)) = lo[h];
      if (!is_q) *reinterpret_cast<h4*>(L.k_cache + ((long)hh * a.T + row) * kHD + j + h * (kHD / 2)) = kc[h];
    }
    return;
  }
  const int tiles = (a.S + kKvTile - 1) / kKvTile;
  const int it = (int)blockIdx.x - qk_groups;
  const int kvh = it / tiles, tile = it % tiles;
  const int d = threadIdx.x & (kHD - 1), chunk = threadIdx.x / kHD;   // chunk = 4 half + g
  const int r0 = tile * kKvTile + (chunk / 4) * 32 + 4 * (chunk % 4);
  const float* src = a.part + (long)(a.Hq + a.Hkv + kvh) * kHD + d;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int p = 0; p < z; ++p) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      x[e] = src[((long)p * a.S + min(r0 + 16 * (e / 4) + e % 4, a.S - 1)) * NQ];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += x[e];
  }
  float mx = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int r = r0 + 16 * (e / 4) + e % 4;
    if (r < a.S) {
      L.v_cache[((long)kvh * a.T + r) * kHD + d] = f2h(v[e]);
      mx = fmaxf(mx, fabsf(v[e]));
    } else {
      v[e] = 0.f;
    }
  }
  const int ex = split_exp(block_max(mx, s_red, kPrepThreads / kWave));
  const float sc = pow2f(-ex);
  const long plane = (long)a.Hkv * tiles * kHD * kKvTile;
  uint16_t* dst = a.vt_img + ((long)it * kHD + d) * kKvTile + 8 * chunk;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] *= sc;
  store_split8(dst, dst + plane, v);
  if (threadIdx.x == 0) a.vexp[(long)tile * a.Hkv + kvh] = ex;
}

// ---------------------------------------------------------------- causal attention

constexpr int kProbExp = 9;       // probabilities relative to the running maximum, times 2^9
constexpr float kMaxLag = 6.f;
constexpr int kUnitSlack = 6;     // a V tile this far below the accumulators' unit keeps it
constexpr int kUnitDrop = 72;     // the unit falls at most so far below the largest one passed

// One workgroup: one q head, 4 waves of 16 QT rows each, the K/V tiles of 64
// rows up to the diagonal.  S^T = K.Q^T and O^T = V^T.P^T, so that a lane's
// probabilities (one q row, 4 + 4 kv rows per 32) already are the operand of
// the second product, and the softmax's row factors are one value per lane.  Each
// product of split operands is three MFMAs (hi.hi + lo.hi + hi.lo; the dropped
// lo.lo is 2^-22 of a term).
//
// Exponents.  Probabilities are scaled by 2^9, the accumulators hold the output
// in units of 2^(unit - 9), and a V tile's exponent against `unit` goes into its
// probabilities.  Their fp16 pair ends at 2^-25, so `unit` follows a tile that is
// larger, or smaller by more than 2^6 (which leaves them 2^-28 of a row's largest
// probability; fp32 has 2^-24 of each), the accumulators rescaled by the exact power
// of two.  Tiles of one magnitude hardly ever do; one factor for the whole layer would
// leave the probabilities of a tile 2^-r below the layer's largest 34 - r bits.  Below
// a tile 2^72 larger the unit stays, or what that tile left in the accumulators
// could overflow.  The output rows' scale is the largest |v| of any kv head up to
// the end of their 64-row tile, which bounds |o|: rows to come have no part in it.
//
// Iteration t multiplies K tile t + 1, takes tile t through the softmax and
// multiplies V tile t; the tiles of the next iteration are loaded meanwhile into
// the other of two buffers each, at one barrier per tile.  One workgroup per CU
// (128 KB of tiles); the grid's heavy (late) tiles start first and the light ones
// fill in.  Per layer, with one exponent for the whole layer / as it is, us: 4001
// rows 222 / 226, 1024 rows 35.4 / 36.6, 37 rows 6.8 / 7.3 (cards differ by 15 %).
// (A lone workgroup's tile takes 2.55 us, one under load 3.15, of which its MFMAs
// take 1.3 at the nominal clock.)  Measured slower: single-buffered tiles with two
// workgroups per CU (258 / 43 us at 4001 / 1024 rows), two q heads of 64 rows on 8
// waves, which reads the LDS twice as much (213 / 48), one MFMA to three VALU
// instructions enforced (255 / 44).
template <int QT>
__global__ __launch_bounds__(256, 1) void prefill_attention_kernel(const PrefillArgs a, const PrefillLayer L,
                                                                   int q_tiles) {
  constexpr int kPlane = kKvTile * kHD * 2;   // bytes of one K or V plane of a tile
  const int lane = lane_id();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int c = lane & 15, g = lane >> 4;
  // one kv head's workgroups share an XCD's L2 when Hkv = 8
  const int kvh = (int)blockIdx.x % a.Hkv, rest = (int)blockIdx.x / a.Hkv;
  const int group = a.Hq / a.Hkv;
  const int head = kvh * group + rest % group;
  const int qt = q_tiles - 1 - rest / group;
  const int q0 = qt * 64 * QT + w * 16 * QT;    // this wave's first row
  const int tiles = (a.S + kKvTile - 1) / kKvTile;
  const int nt = min((qt + 1) * QT, tiles);
  const long kplane = (long)a.Hkv * a.S * kHD, vplane = (long)a.Hkv * tiles * kHD * kKvTile;
  const uint16_t* ki = a.k_img + (long)kvh * a.S * kHD;
  const uint16_t* vi = a.vt_img + (long)kvh * tiles * kHD * kKvTile;

  // K tile: 64 rows of 16 chunks, 4 rows per load, chunk c of row r at
  // c ^ (r % 8); V tile: 128 rows (dims) of 8 chunks, 8 rows per load.  Wave w
  // loads rows [16 w, 16 w + 16) of both K planes and dims [32 w, 32 w + 32) of V.
  auto issue_k = [&](auto B, int t) {
    char* st = lds_stage<decltype(B)::value, 2 * kPlane>();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * w + 4 * i + (lane >> 4);
      const int ch = (lane & 15) ^ (r & 7);
      const uint16_t* src = ki + (long)min(t * kKvTile + r, a.S - 1) * kHD + ch * 8;
      load_lds16(src, st + (16 * w + 4 * i) * 256);
      load_lds16(src + kplane, st + kPlane + (16 * w + 4 * i) * 256);
    }
  };
  auto issue_v = [&](auto B, int t) {
    char* st = lds_stage<2 + decltype(B)::value, 2 * kPlane>();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 32 * w + 8 * i + (lane >> 3);
      const int ch = (lane & 7) ^ (r & 7);
      const uint16_t* src = vi + ((long)t * kHD + r) * kKvTile + ch * 8;
      load_lds16(src, st + (32 * w + 8 * i) * 128);
      load_lds16(src + vplane, st + kPlane + (32 * w + 8 * i) * 128);
    }
  };
  const std::integral_constant<int, 0> b0;
  const std::integral_constant<int, 1> b1;
  // This wave's rows lie in one 64-row tile, the last whose V rows they see.  The
  // exponents that bound its output are loaded ahead of everything else and
  // used at the end (a loop over them here waits for its loads: 1.3 us a workgroup).
  const int last = min(q0 / kKvTile, tiles - 1), n_exp = (last + 1) * a.Hkv;
  i32x4 ex[QT];
#pragma unroll
  for (int i = 0; i < QT; ++i)
    ex[i] = *reinterpret_cast<const i32x4*>(a.vexp + min(4 * (kWave * i + lane), (n_exp - 1) & ~3));
  // Q operand: column c = row q0 + 16 i + c, k 8 g .. 8 g + 7 of each 32 dims
  h8 qh[QT][4], ql[QT][4];
  const long qplane = (long)a.Hq * a.S * kHD;
#pragma unroll
  for (int i = 0; i < QT; ++i) {
    const uint16_t* src = a.q_img + ((long)head * a.S + min(q0 + 16 * i + c, a.S - 1)) * kHD + 8 * g;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      qh[i][ks] = *reinterpret_cast<const h8*>(src + 32 * ks);
      ql[i][ks] = *reinterpret_cast<const h8*>(src + qplane + 32 * ks);
    }
  }
  // log2 units: scale * log2(e) * 2^(q exponent + k exponent).  Both head norms
  // all zero would underflow it to 0 (their scores are 0) and the masked -inf
  // scores times that to NaN; other fp16 weights keep it above 2^-76.
  const float fac = fmaxf(
      a.attn_scale * 1.44269504088896340736f * pow2f(head_exp(L.q_norm)) * pow2f(head_exp(L.k_norm)), 0x1p-120f);
  issue_k(b0, 0);
  issue_v(b0, 0);
  if (nt > 1) issue_k(b1, 1);
  const int* vexp = a.vexp + kvh;
  int unit = ld_scalar(vexp), top = unit;

  f32x4 o[QT][8];
  float m[QT], l[QT];
#pragma unroll
  for (int i = 0; i < QT; ++i) {
    m[i] = -INFINITY;
    l[i] = 0.f;
#pragma unroll
    for (int d = 0; d < 8; ++d) o[i][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  unsigned bk[4], bv[2];   // this lane's fragment bases (opaque, see split_gemm_kernel)
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    bk[ks] = c * 256 + (((4 * ks + g) ^ (c & 7)) << 4);
    asm("" : "+v"(bk[ks]));
  }
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    bv[ks] = c * 128 + (((4 * ks + g) ^ (c & 7)) << 4);
    asm("" : "+v"(bv[ks]));
  }
  // (MFMAs of one product over all accumulators before the next product: three
  // in a row on one accumulator would wait for each other's result)
  auto scores = [&](auto B, f32x4 (&s)[QT][4]) {
    const char* sk = lds_stage<decltype(B)::value, 2 * kPlane>();
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int i = 0; i < QT; ++i) s[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      h8 kh[4], kl[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        kh[n] = *reinterpret_cast<const h8*>(sk + bk[ks] + n * 16 * 256);
        kl[n] = *reinterpret_cast<const h8*>(sk + bk[ks] + kPlane + n * 16 * 256);
      }
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int i = 0; i < QT; ++i) s[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh[n], qh[i][ks], s[i][n], 0, 0, 0);
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int i = 0; i < QT; ++i) s[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl[n], qh[i][ks], s[i][n], 0, 0, 0);
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int i = 0; i < QT; ++i) s[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh[n], ql[i][ks], s[i][n], 0, 0, 0);
    }
  };
  f32x4 sc[2][QT][4];   // scores of tiles t and t + 1, alternating
  wait_barrier<0>();
  scores(b0, sc[0]);

  // iteration t (t % 2 = B): softmax of sc[B], V tile t in V buffer B; MORE: scores of
  // tile t + 1 from K buffer 1 - B
  auto body = [&](auto B, auto MORE, int t) {
    constexpr int b = decltype(B)::value;
    const std::integral_constant<int, 1 - b> nb;
    const int ev = ld_scalar(vexp + min(t, last) * a.Hkv);   // (past `last` no row sees the tile)
    wait_barrier<0>();   // this iteration's tiles; every wave is done with the buffers refilled below
    if constexpr (decltype(MORE)::value) {
      if (t + 2 < nt) issue_k(B, t + 2);
      issue_v(nb, t + 1);
      scores(nb, sc[1 - b]);
    }
    f32x4 (&s)[QT][4] = sc[b];
    if (t * kKvTile + kKvTile - 1 > q0) {   // the diagonal: kv 16 n + 4 g + j is visible up to lim
#pragma unroll
      for (int i = 0; i < QT; ++i) {
        const int lim = q0 + 16 * i + c - t * kKvTile - 4 * g;
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (16 * n + j > lim) s[i][n][j] = -INFINITY;
      }
    }
    // The running maximum follows only when a row's has grown by more than
    // kMaxLag (log2): until then probabilities stay below 2^(kProbExp + kMaxLag),
    // within fp16, and the accumulators need no rescaling.
    float mx[QT];
    bool grow = false;
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      float v = s[i][0][0];
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int j = 0; j < 4; ++j) v = fmaxf(v, s[i][n][j]);
      v = fmaxf(v, __shfl_xor(v, 16));
      mx[i] = fmaxf(v, __shfl_xor(v, 32)) * fac;
      grow = grow || mx[i] > m[i] + kMaxLag;
    }
    const int to = ev > unit || ev < unit - kUnitSlack ? max(ev, top - kUnitDrop) : unit;
    if (to != unit || __any(grow)) {
      const float f = ldexpf(1.f, unit - to);
#pragma unroll
      for (int i = 0; i < QT; ++i) {
        const float mn = fmaxf(m[i], mx[i]);
        const float al = __builtin_amdgcn_exp2f(m[i] - mn);
        m[i] = mn;
        l[i] *= al;
#pragma unroll
        for (int d = 0; d < 8; ++d) o[i][d] *= al * f;
      }
      unit = to;
      top = max(top, to);
    }
    // probabilities leave exp2 already times 2^ve (2^-60 has them vanish)
    const int ve = max(ev - unit + kProbExp, -60);
    h8 ph[QT][2], pl[QT][2];
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      const float sub = (float)ve - m[i];
      float ps = 0.f;
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
          f32x2 p;
          p.x = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i][n][j], fac, sub));
          p.y = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i][n][j + 1], fac, sub));
          ps += p.x;
          ps += p.y;
          const h2 hi = __builtin_convertvector(p, h2);
          const h2 lo = __builtin_convertvector(p - __builtin_convertvector(hi, f32x2), h2);
          ph[i][n / 2][4 * (n & 1) + j] = hi.x;
          ph[i][n / 2][4 * (n & 1) + j + 1] = hi.y;
          pl[i][n / 2][4 * (n & 1) + j] = lo.x;
          pl[i][n / 2][4 * (n & 1) + j + 1] = lo.y;
        }
      l[i] = __builtin_fmaf(ps, pow2f(-ve), l[i]);
    }
    const char* sv = lds_stage<2 + b, 2 * kPlane>();
#pragma unroll
    for (int d0 = 0; d0 < 8; d0 += 4)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        h8 vh[4], vl[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          vh[d] = *reinterpret_cast<const h8*>(sv + bv[ks] + (d0 + d) * 16 * 128);
          vl[d] = *reinterpret_cast<const h8*>(sv + bv[ks] + kPlane + (d0 + d) * 16 * 128);
        }
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int i = 0; i < QT; ++i)
            o[i][d0 + d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh[d], ph[i][ks], o[i][d0 + d], 0, 0, 0);
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int i = 0; i < QT; ++i)
            o[i][d0 + d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl[d], ph[i][ks], o[i][d0 + d], 0, 0, 0);
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int i = 0; i < QT; ++i)
            o[i][d0 + d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh[d], pl[i][ks], o[i][d0 + d], 0, 0, 0);
      }
  };
  const std::integral_constant<bool, true> more;
  const std::integral_constant<bool, false> end;
  int t = 0;
#pragma unroll 1
  for (; t + 2 < nt; t += 2) {
    body(b0, more, t);
    body(b1, more, t + 1);
  }
  if (t + 1 < nt) {
    body(b0, more, t);
    body(b1, end, t + 1);
  } else {
    body(b0, end, t);
  }
  const long HD = (long)a.Hq * kHD;
  int bound = -kMaxExp;
  auto fold = [&](const i32x4& x, int first) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (first + j < n_exp) bound = max(bound, x[j]);
  };
#pragma unroll
  for (int i = 0; i < QT; ++i) fold(ex[i], min(4 * (kWave * i + lane), (n_exp - 1) & ~3));
  for (int i = 4 * (kWave * QT + lane); i < n_exp; i += 4 * kWave)
    fold(*reinterpret_cast<const i32x4*>(a.vexp + i), i);
  const int o_exp = (int)wave_max((float)bound);
#pragma unroll
  for (int i = 0; i < QT; ++i) {
    l[i] += __shfl_xor(l[i], 16);
    l[i] += __shfl_xor(l[i], 32);
    const int row = q0 + 16 * i + c;
    const float inv = ldexpf(1.f / ((float)(1 << kProbExp) * l[i]), unit - o_exp);
    if (row < a.S) {
      if (head == 0 && g == 0) a.scale[row] = pow2f(o_exp);
      uint16_t* dst = a.img + (long)row * HD + (long)head * kHD + 4 * g;
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        h4 hi, lo;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          _Float16 x, y;
          split2(o[i][d][j] * inv, x, y);
          hi[j] = x;
          lo[j] = y;
        }
        *reinterpret_cast<h4*>(dst + 16 * d) = hi;
        *reinterpret_cast<h4*>(dst + (long)a.S * HD + 16 * d) = lo;
      }
    }
  }
}

}  // namespace

// ---------------------------------------------------------------- host

PrefillPlan prefill_plan(long S, int H, int Hq, int Hkv, int I) {
  PrefillPlan p;
  const long qn = (long)(Hq + 2 * Hkv) * kHD, qs = (long)Hq * kHD;
  p.qkv = split_gemm_plan(S, qn, H);
  p.part_floats = p.qkv.z * qn * S;
  for (int l = 0; l < 2; ++l) {
    const long M = l ? 1 : S;
    p.o_proj[l] = split_gemm_plan(M, H, qs);
    p.gate_up[l] = split_gemm_plan(M, 2L * I, H);
    p.down[l] = split_gemm_plan(M, H, I);
    for (long x : {(long)p.o_proj[l].z * H, p.gate_up[l].z * 2L * I, (long)p.down[l].z * H})
      if (x * M > p.part_floats) p.part_floats = x * M;
  }
  return p;
}

int prefill_launch(const PrefillArgs& a, const PrefillLayer* layers, int first, int n, const PrefillPlan& p,
                   hipStream_t s) {
  const int tiles = (a.S + kKvTile - 1) / kKvTile;
  const int qs = a.Hq * kHD, qn = (a.Hq + 2 * a.Hkv) * kHD;
  int st;
  if (first == 0) {
    const long init = (long)a.S * (kHD / 2);
    hipLaunchKernelGGL(prefill_init_kernel, dim3((unsigned)((init + 255) / 256)), dim3(256), 0, s, a);
    if ((st = qd_host::launch_status("prefill_init_kernel"))) return st;
  }
  // M rows of the image, whose planes lie `plane` values apart
  auto gemm = [&](const uint16_t* img, long plane, const uint16_t* W, const float* scale, int M, int N, int K,
                  const GemmPlan& g) {
    SplitGemmArgs x;
    x.hi = img; x.lo = img + plane; x.scale = scale; x.W = W; x.y = a.part;
    x.M = M; x.N = N; x.K = K;
    return split_gemm_launch(x, g, s);
  };
  auto rows = [&](int M, int z, const uint16_t* gamma) {   // the last M rows
    hipLaunchKernelGGL((prefill_rows_kernel<false>), dim3((unsigned)M), dim3(256), 0, s, a, a.part, z, gamma, a.S - M);
    return qd_host::launch_status("prefill_rows_kernel");
  };
  constexpr int kPrepItems = kPrepThreads / 16;
  const int qk_groups = (int)(((long)a.S * (a.Hq + a.Hkv) + kPrepItems - 1) / kPrepItems);
  // 128 q rows per workgroup read the LDS half as often, 64 give twice the
  // workgroups; they meet at 1.25 workgroups of 128 rows per CU (28 layers of 2B, 64 /
  // 128 rows: 1800 rows 13.6 / 14.1 ms, 2432 17.98 / 18.10, 2560 18.60 / 18.60, 3000
  // 22.9 / 22.4, 3800 28.2 / 27.0)
  const int q_rows = (long)((a.S + 127) / 128) * a.Hq * 4 >= 5L * qd_host::cu_count() ? 128 : 64;
  const int q_tiles = (a.S + q_rows - 1) / q_rows;
  for (int li = first; li < first + n; ++li) {
    const PrefillLayer& L = layers[li - first];
    if (li == 0) {
      hipLaunchKernelGGL((prefill_rows_kernel<true>), dim3((unsigned)a.S), dim3(256), 0, s, a, nullptr, 0, L.input_norm, 0);
      if ((st = qd_host::launch_status("prefill_rows_kernel"))) return st;
    } else if ((st = rows(a.S, p.down[0].z, L.input_norm))) {
      return st;
    }
    if ((st = gemm(a.img, (long)a.S * a.H, L.qkv, a.scale, a.S, qn, a.H, p.qkv))) return st;
    hipLaunchKernelGGL(prefill_qkv_prep_kernel, dim3((unsigned)(qk_groups + a.Hkv * tiles)), dim3(kPrepThreads), 0, s, a,
                       L, p.qkv.z, qk_groups);
    if ((st = qd_host::launch_status("prefill_qkv_prep_kernel"))) return st;
    // the last layer's K/V rows are written: past them only the last row is used
    const int last = li + 1 == a.layers_n, M = last ? 1 : a.S;
    const unsigned groups = (unsigned)a.Hq * (last ? 1u : (unsigned)q_tiles);   // last: its final tile
    if (q_rows == 128)
      hipLaunchKernelGGL((prefill_attention_kernel<2>), dim3(groups), dim3(256), 0, s, a, L, q_tiles);
    else
      hipLaunchKernelGGL((prefill_attention_kernel<1>), dim3(groups), dim3(256), 0, s, a, L, q_tiles);
    if ((st = qd_host::launch_status("prefill_attention_kernel"))) return st;
    if ((st = gemm(a.img + (long)(a.S - M) * qs, (long)a.S * qs, L.o_proj, a.scale + (a.S - M), M, a.H, qs,
                   p.o_proj[last])))
      return st;
    if ((st = rows(M, p.o_proj[last].z, L.post_norm))) return st;
    if ((st = gemm(a.img, (long)M * a.H, L.gate_up, a.scale, M, 2 * a.I, a.H, p.gate_up[last]))) return st;
    if (M <= qd_host::cu_count())
      hipLaunchKernelGGL(prefill_silu_kernel<1024>, dim3((unsigned)M), dim3(1024), 0, s, a, p.gate_up[last].z);
    else
      hipLaunchKernelGGL(prefill_silu_kernel<256>, dim3((unsigned)M), dim3(256), 0, s, a, p.gate_up[last].z);
    if ((st = qd_host::launch_status("prefill_silu_kernel"))) return st;
    if ((st = gemm(a.img, (long)M * a.I, L.down, a.scale, M, a.H, a.I, p.down[last]))) return st;
  }
  return first + n == a.layers_n ? rows(1, p.down[1].z, nullptr) : QD_OK;
}

}  // namespace qd
