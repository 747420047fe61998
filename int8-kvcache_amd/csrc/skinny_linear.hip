// Matrix products of the decode step: x [M, K] times W [N, K]^T for M <= 32 activation rows, bf16
// operands, fp32 accumulation, for gfx950.
//
// Bound: HBM, the weights (every byte used once per step; 0.47 GB per Qwen2.5-7B layer).
// Layout: the product is cut along K into slots of at most kMaxBlocks blocks of 64, one slot per
// wave.  A wave keeps its slot of x in registers for the whole kernel (32 x 448 bf16 values at
// K = 3584: 112 VGPRs) and streams 16 rows of W at a time (one MFMA row block) through its
// remaining registers, so x is read once per workgroup.  The eight waves of a workgroup hold
// adjacent slots of the same 16 rows; their partial sums meet in LDS (2 KB per wave and row block,
// against 14 KB of weights).  Each register of W is requested again for the next row block as
// soon as it is consumed: 14 KB per wave, 112 KB per compute unit in flight throughout.  Where K
// exceeds eight slots (the 18944-wide down projection), groups of eight slots leave fp32
// partial sums that the residual add + RMSNorm kernel behind it (or a reduce kernel) adds.
// Loads: eight adjacent lanes read one whole 128-byte line, and the registers are turned into
// MFMA operands (16 rows x 16 bytes across lanes) through 2 KB of LDS per wave.  Loaded in operand
// order instead (16 half lines per instruction) the same bytes stream at 5.3 TB/s (5.8 without
// the non-temporal hint) instead of 6.5.
// Measured (HIP-graph replays on cold weights, 32 rows, against the library GEMM torch picks, us):
// qkv 11.3 vs 13.2, o_proj 8.6 vs 12.8, gate_up with SwiGLU 49 vs 58 + 5, down with the norm 28.2
// vs 110 + 5, LM head (1.09 GB) 185 vs 258; one row: 9.7 / 7.3 / 47.7 / 25.5 / 169 us (6.4 TB/s).

#include <hip/hip_runtime.h>

#include <cstdint>

#include "silu.h"
#include "skinny_linear.h"

namespace int8kv_loop {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kWaves = 8;      // waves (K slots) per workgroup
constexpr int kMaxBlocks = 8;  // 64-wide blocks of K per slot
constexpr int kMaxRows = 32;
constexpr int kBiasBlocks = kWaves * 64 / 16;  // row blocks whose bias is staged: one value per thread

struct LinearArgs {
  const uint16_t* x;
  int64_t xs;
  const uint16_t* w;
  int64_t ws;
  const uint16_t* bias;
  uint16_t* out;
  int64_t os;
  float* part;     // [groups][M][n] partial sums (EPI_PART)
  int32_t m;       // activation rows
  int32_t n;       // output columns
  int32_t blocks;  // K / 64
  int32_t groups;  // groups of kWaves slots along K
  int32_t nb;      // workgroups per group
  int32_t tiles;   // row blocks
  int32_t tiles_q, tiles_r;  // tiles = nb tiles_q + tiles_r: the first tiles_r workgroups take one more
};

enum Epilogue { kEpiStore = 0, kEpiPart = 1, kEpiSilu = 2 };

__device__ __forceinline__ float round_bf16(float f) {
  return static_cast<float>(static_cast<__bf16>(f));
}
__device__ __forceinline__ float bf16_value(uint16_t h) {
  return __uint_as_float(static_cast<uint32_t>(h) << 16);
}
__device__ __forceinline__ uint16_t bf16_bits(float f) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}

// Barrier for data exchanged through LDS: waits for this wave's LDS accesses only, so that the
// weight loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Non-temporal at every size: seven model shapes of hidden 512 to 4096, the smallest with all its
// weights within the Infinity Cache, run 1.2 to 2.3 times the step rate of library products.
__device__ __forceinline__ u32x4 load_w(const uint16_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}

// 16 rows x 64 columns of bf16 (2 KB) between load order and operand order.  In load order lane l
// of load j holds columns 8 (l % 8) .. + 7 of row 8 j + l / 8; as an MFMA operand lane (i, g)
// holds columns 32 ks + 8 g .. + 7 of row i.  Piece c (8 columns) of row r lies at 128 r +
// 16 (c ^ (r / 2 % 8)): both accesses then cover every bank evenly.  The buffer is the wave's
// own and a wave's LDS accesses run in order, so no barrier is needed.
__device__ __forceinline__ void stage_store(char* buf, int lane, const u32x4 (&v)[2]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * j + (lane >> 3);
    *reinterpret_cast<u32x4*>(buf + 128 * r + 16 * ((lane & 7) ^ ((r >> 1) & 7))) = v[j];
  }
}
__device__ __forceinline__ void stage_read(const char* buf, int lane, bf16x8 (&op)[2]) {
  const int i = lane & 15;
  const int g = lane >> 4;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    op[ks] = __builtin_bit_cast(
        bf16x8, *reinterpret_cast<const u32x4*>(buf + 128 * i + 16 * ((4 * ks + g) ^ ((i >> 1) & 7))));
}

// One workgroup: K group blockIdx.x / nb, a contiguous run of the row blocks.  MT: 16-row column
// tiles of x.  KB: 64-wide blocks of the longest slot; every slot has KB or KB - 1 (host).
template <int MT, int KB, int EPI>
__global__ __launch_bounds__(kWaves * 64) void skinny_kernel(LinearArgs a) {
  __shared__ float s_part[2][kWaves][MT][256];
  __shared__ __align__(16) char s_stage[kWaves][2][2048];
  __shared__ float s_bias[EPI == kEpiStore ? 16 * kBiasBlocks : 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t kg = blockIdx.x / (uint32_t)a.nb;
  const uint32_t wg = blockIdx.x - kg * a.nb;
  const uint32_t more = a.tiles_r;  // the first `more` workgroups take one row block more
  int tile = (int)(wg * a.tiles_q + (wg < more ? wg : more));
  const int tile_end = tile + a.tiles_q + (wg < more ? 1 : 0);
  const uint32_t slots = a.groups * kWaves;
  const uint32_t slot = kg * kWaves + wave;
  const int b0 = (int)(slot * a.blocks / slots);
  const int b1 = (int)((slot + 1) * a.blocks / slots);
  const bool last = b1 - b0 == KB;  // wave-uniform
  // The bias of this workgroup's first kBiasBlocks row blocks goes through LDS: loaded where it is
  // added, its wait would be a wait for every weight load in flight.
  float bias0 = 0.f;
  if constexpr (EPI == kEpiStore) {
    const int64_t col = 16 * (int64_t)tile + threadIdx.x;
    if (a.bias && col < a.n) bias0 = bf16_value(a.bias[col]);
  }

  // x before W.  Columns past the last row of x repeat it (their results are never stored); the
  // block a short slot lacks is read inside the row and not used.
  u32x4 xv[MT][KB][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int m = 16 * mt + 8 * j + (lane >> 3);
      const uint16_t* xp = a.x + (int64_t)(m < a.m ? m : a.m - 1) * a.xs + 8 * (lane & 7);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int b = kb < KB - 1 ? b0 + kb : min(b0 + kb, a.blocks - 1);
        xv[mt][kb][j] = *reinterpret_cast<const u32x4*>(xp + 64 * (int64_t)b);
      }
    }
  // Weight rows of a row block: 16 consecutive ones, or (kEpiSilu) 8 gate rows (load 0) and the 8
  // up rows of the same columns (load 1).
  constexpr int kRowsPerTile = EPI == kEpiSilu ? 8 : 16;
  const uint16_t* wp = a.w + ((int64_t)kRowsPerTile * tile + (lane >> 3)) * a.ws + 64 * (int64_t)b0 +
                       8 * (lane & 7);
  const int64_t second = (EPI == kEpiSilu ? (int64_t)a.n : 8) * a.ws;  // load 1's rows
  const int64_t step = kRowsPerTile * a.ws;
  u32x4 wr[KB][2];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
    if (kb < KB - 1 || last) {
      wr[kb][0] = load_w(wp + 64 * kb);
      wr[kb][1] = load_w(wp + second + 64 * kb);
    }
  bf16x8 xr[MT][KB][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      char* buf = s_stage[wave][kb & 1];
      stage_store(buf, lane, xv[mt][kb]);
      stage_read(buf, lane, xr[mt][kb]);
    }
  if constexpr (EPI == kEpiStore) s_bias[threadIdx.x] = bias0;

  int buf = 0;
  int done = 0;  // row blocks this workgroup has finished
  auto row_block = [&](bool refill, const uint16_t* next) {
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      if (kb < KB - 1 || last) {
        char* stage = s_stage[wave][kb & 1];
        stage_store(stage, lane, wr[kb]);
        bf16x8 op[2];
        stage_read(stage, lane, op);
        if (refill) {
          wr[kb][0] = load_w(next + 64 * kb);
          wr[kb][1] = load_w(next + second + 64 * kb);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op[ks], xr[mt][kb][ks], acc[mt], 0, 0, 0);
      }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      *reinterpret_cast<f32x4*>(&s_part[buf][wave][mt][4 * lane]) = acc[mt];
    lds_barrier();
    // One wave, in turn, adds the eight partial blocks and stores: lane (m, h) columns 8 h .. + 7
    // of row m (accumulator element (row 4 q + r, column m % 16) of tile m / 16 is register r of
    // lane 16 q + m % 16).  The other waves go on.
    const int m = lane & 31;
    const int h = lane >> 5;
    if (wave == (done & (kWaves - 1)) && m < a.m && (MT == 2 || m < 16) &&
        (EPI != kEpiSilu || h == 0)) {
      auto column_sum = [&](int q) {
        f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < kWaves; ++v)
          y += *reinterpret_cast<const f32x4*>(&s_part[buf][v][m >> 4][4 * (16 * q + (m & 15))]);
        return y;
      };
      const f32x4 lo = column_sum(2 * h);
      const f32x4 hi = column_sum(2 * h + 1);
      float y[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if constexpr (EPI == kEpiSilu) {
        const f32x4 ulo = column_sum(2);
        const f32x4 uhi = column_sum(3);
        const float u[8] = {ulo[0], ulo[1], ulo[2], ulo[3], uhi[0], uhi[1], uhi[2], uhi[3]};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float g = round_bf16(y[j]);
          const float mid = silu_middle(g);
          const float end = silu_ends(g);  // (no branch: its values would need registers x and W hold)
          y[j] = round_bf16(fabsf(g) < kSiluMiddle ? mid : end) * round_bf16(u[j]);
        }
      }
      const int64_t col = kRowsPerTile * (int64_t)tile + 8 * h;
      if constexpr (EPI == kEpiPart) {
        float* p = a.part + ((int64_t)kg * a.m + m) * a.n + col;
        *reinterpret_cast<f32x4*>(p) = f32x4{y[0], y[1], y[2], y[3]};
        *reinterpret_cast<f32x4*>(p + 4) = f32x4{y[4], y[5], y[6], y[7]};
      } else {
        if (EPI == kEpiStore && a.bias) {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            y[j] += done < kBiasBlocks ? s_bias[16 * done + 8 * h + j] : bf16_value(a.bias[col + j]);
        }
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[j] = bf16_bits(y[2 * j]) | ((uint32_t)bf16_bits(y[2 * j + 1]) << 16);
        *reinterpret_cast<u32x4*>(a.out + (int64_t)m * a.os + col) = o;
      }
    }
    // The next row block writes the other buffer; this one is written again only after the
    // barrier in between, which every wave passes with its reads of it done.
    buf ^= 1;
    ++done;
  };
  for (; tile + 1 < tile_end; ++tile) {
    wp += step;
    row_block(true, wp);
  }
  row_block(false, wp);
}

// out = bf16(sum of the groups' partial sums + bias), one thread per 4 columns.
__global__ __launch_bounds__(256) void reduce_parts_kernel(LinearArgs a) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t per_row = a.n / 4;
  if (t >= per_row * a.m) return;
  const int64_t m = t / per_row;
  const int64_t c = 4 * (t - m * per_row);
  f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < a.groups; ++s)
    y += *reinterpret_cast<const f32x4*>(a.part + ((int64_t)s * a.m + m) * a.n + c);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    a.out[m * a.os + c + j] = bf16_bits(a.bias ? y[j] + bf16_value(a.bias[c + j]) : y[j]);
}

// Residual add + RMSNorm behind a product: the delta row is the sum of `groups` fp32 partial rows
// (rounded to bf16, as the product's own output would be).  One workgroup per row, four columns
// per thread, all of a thread's partial rows requested together: with 32 rows the call is one
// memory latency plus the block reduction.
constexpr int kNormThreads = 1024;
constexpr int kNormVec = 2;  // 2 x 1024 x 4 = 8192 columns at most

template <int G>
__global__ __launch_bounds__(kNormThreads) void parts_add_rms_norm_kernel(
    uint16_t* residual, int64_t rs, const float* part, int m, int n, const uint16_t* weight,
    uint16_t* out, int64_t os, float eps) {
  const int64_t row = blockIdx.x;
  float x[kNormVec][4];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < kNormVec; ++j) {
    const int c = 4 * ((int)threadIdx.x + j * kNormThreads);
    if (c < n) {
      uint2* rp = reinterpret_cast<uint2*>(residual + row * rs + c);
      const uint2 r = *rp;
      f32x4 p[G];
#pragma unroll
      for (int s = 0; s < G; ++s)
        p[s] = *reinterpret_cast<const f32x4*>(part + ((int64_t)s * m + row) * n + c);
      f32x4 d = p[0];
#pragma unroll
      for (int s = 1; s < G; ++s) d += p[s];
      const float r4[4] = {bf16_value((uint16_t)r.x), bf16_value((uint16_t)(r.x >> 16)),
                           bf16_value((uint16_t)r.y), bf16_value((uint16_t)(r.y >> 16))};
      uint32_t b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[j][i] = round_bf16(r4[i] + round_bf16(d[i]));
        b[i] = bf16_bits(x[j][i]);
        ss += x[j][i] * x[j][i];
      }
      *rp = uint2{b[0] | (b[1] << 16), b[2] | (b[3] << 16)};
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off, 64);
  __shared__ float s_sum[kNormThreads / 64];
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int v = 0; v < kNormThreads / 64; ++v) tot += s_sum[v];
  const float inv = rsqrtf(tot / static_cast<float>(n) + eps);
#pragma unroll
  for (int j = 0; j < kNormVec; ++j) {
    const int c = 4 * ((int)threadIdx.x + j * kNormThreads);
    if (c < n) {
      const uint2 w = *reinterpret_cast<const uint2*>(weight + c);
      const float w4[4] = {bf16_value((uint16_t)w.x), bf16_value((uint16_t)(w.x >> 16)),
                           bf16_value((uint16_t)w.y), bf16_value((uint16_t)(w.y >> 16))};
      uint32_t b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = bf16_bits(w4[i] * round_bf16(x[j][i] * inv));
      *reinterpret_cast<uint2*>(out + row * os + c) = uint2{b[0] | (b[1] << 16), b[2] | (b[3] << 16)};
    }
  }
}

constexpr int kMaxGroups = 8;  // K up to 8 x 8 x 8 x 64 = 32768

int cu_count() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    return 256;
  return n;
}

// Fewest groups of kWaves slots that hold K.
int min_groups(int64_t k) {
  const int64_t per = (int64_t)kWaves * kMaxBlocks * 64;
  return (int)((k + per - 1) / per);
}

// Groups along K of a product with `tiles` row blocks: one where K fits it (the result then needs
// no partial sums: qkv and o_proj of Qwen2.5-7B, 32 rows, 11.3 and 8.6 us against 11.9-16 and
// 10.6-13.8 us with 2-8 groups); otherwise the count whose busiest workgroup reads least, its
// row blocks times their 1 / groups of a row.  18944 x 3584 on 256 compute units: 8 groups give
// every workgroup 7 row blocks (28.2 us with the norm), 5 groups 4 or 5 longer ones (30.5 us).
int groups_of(int64_t k, int64_t tiles, int cus) {
  const int least = min_groups(k);
  if (least == 1) return 1;
  int best = least;
  double cost = 0.0;
  for (int g = least; g <= kMaxGroups; ++g) {
    const int64_t per = cus / g > 0 ? cus / g : 1;
    const double c = (double)((tiles + per - 1) / per) / g;
    if (g == least || c < cost) {
      best = g;
      cost = c;
    }
  }
  return best;
}

bool rows16(const void* p, int64_t stride) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0 && stride % 8 == 0;
}

template <int MT, int EPI>
void launch_blocks(int kb, dim3 grid, hipStream_t s, const LinearArgs& a) {
  const dim3 block(kWaves * 64);
  switch (kb) {
#define INT8KV_SKINNY(K)                                                        \
  case K:                                                                       \
    hipLaunchKernelGGL((skinny_kernel<MT, K, EPI>), grid, block, 0, s, a);      \
    break;
    INT8KV_SKINNY(1) INT8KV_SKINNY(2) INT8KV_SKINNY(3) INT8KV_SKINNY(4)
    INT8KV_SKINNY(5) INT8KV_SKINNY(6) INT8KV_SKINNY(7) INT8KV_SKINNY(8)
#undef INT8KV_SKINNY
    default: break;
  }
}

// Launches the product: at most one workgroup per compute unit, each K group's workgroups
// striding over its row blocks.
template <int EPI>
int launch_linear(LinearArgs& a, hipStream_t s) {
  const int cus = cu_count();
  a.groups = groups_of((int64_t)a.blocks * 64, a.tiles, cus);
  const int slots = a.groups * kWaves;
  const int kb = (a.blocks + slots - 1) / slots;
  const int per_group = cus / a.groups;
  a.nb = per_group < 1 ? 1 : (per_group > a.tiles ? a.tiles : per_group);
  a.tiles_q = a.tiles / a.nb;
  a.tiles_r = a.tiles - a.nb * a.tiles_q;
  const dim3 grid((unsigned)(a.nb * a.groups));
  if (a.m <= 16)
    launch_blocks<1, EPI>(kb, grid, s, a);
  else
    launch_blocks<2, EPI>(kb, grid, s, a);
  return (int)hipGetLastError();
}

int check_linear(LinearArgs& a, const void* x, int64_t rows, int64_t k, int64_t xs, const void* w,
                 int64_t n, int64_t ws) {
  if (!x || !w) return INT8KV_E_NULL;
  if (!int8kv_skinny_linear_ok(rows, k, n)) return INT8KV_E_SHAPE;
  if (!rows16(x, xs) || !rows16(w, ws) || xs < k || ws < k) return INT8KV_E_STRIDE;
  a = LinearArgs{};
  a.x = static_cast<const uint16_t*>(x);
  a.xs = xs;
  a.w = static_cast<const uint16_t*>(w);
  a.ws = ws;
  a.m = (int32_t)rows;
  a.n = (int32_t)n;
  a.blocks = (int32_t)(k / 64);
  a.tiles = (int32_t)(n / 16);
  return INT8KV_OK;
}

template <int G>
void launch_norm(const LinearArgs& a, uint16_t* residual, int64_t rs, const uint16_t* weight,
                 uint16_t* out, int64_t os, float eps, hipStream_t s) {
  hipLaunchKernelGGL((parts_add_rms_norm_kernel<G>), dim3((unsigned)a.m), dim3(kNormThreads), 0, s,
                     residual, rs, a.part, a.m, a.n, weight, out, os, eps);
}

}  // namespace
}  // namespace int8kv_loop

using namespace int8kv_loop;

extern "C" int32_t int8kv_skinny_linear_ok(int64_t rows, int64_t k, int64_t n) {
  return rows >= 1 && rows <= kMaxRows && k >= 64 && k % 64 == 0 &&
         k <= (int64_t)kMaxGroups * kWaves * kMaxBlocks * 64 && n >= 16 && n % 16 == 0 &&
         n <= 0x7fffffff;
}

extern "C" int64_t int8kv_skinny_linear_workspace_bytes(int64_t rows, int64_t k, int64_t n) {
  if (!int8kv_skinny_linear_ok(rows, k, n)) return 0;
  return (int64_t)(min_groups(k) == 1 ? 1 : kMaxGroups) * rows * n * 4;
}

extern "C" int int8kv_skinny_linear(const void* x, int64_t rows, int64_t k, int64_t x_row_stride,
                                    const void* w, int64_t n, int64_t w_row_stride,
                                    const void* bias, void* out, int64_t out_row_stride,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  LinearArgs a;
  const int st = check_linear(a, x, rows, k, x_row_stride, w, n, w_row_stride);
  if (st != INT8KV_OK) return st;
  if (!out) return INT8KV_E_NULL;
  if (!rows16(out, out_row_stride) || out_row_stride < n) return INT8KV_E_STRIDE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  a.bias = static_cast<const uint16_t*>(bias);
  a.out = static_cast<uint16_t*>(out);
  a.os = out_row_stride;
  if (min_groups(k) == 1) return launch_linear<kEpiStore>(a, s);
  if (!workspace || workspace_bytes < int8kv_skinny_linear_workspace_bytes(rows, k, n) ||
      reinterpret_cast<uintptr_t>(workspace) % 16)
    return INT8KV_E_WORKSPACE;
  a.part = static_cast<float*>(workspace);
  const int e = launch_linear<kEpiPart>(a, s);
  if (e != 0) return e;
  const int64_t threads = rows * (n / 4);
  hipLaunchKernelGGL(reduce_parts_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}

extern "C" int int8kv_skinny_linear_silu_mul(const void* x, int64_t rows, int64_t k,
                                             int64_t x_row_stride, const void* w, int64_t ffn,
                                             int64_t w_row_stride, void* out,
                                             int64_t out_row_stride, void* stream) {
  LinearArgs a;
  if (ffn <= 0 || ffn % 8 || ffn > 0x3fffffff || k > (int64_t)kWaves * kMaxBlocks * 64)
    return INT8KV_E_SHAPE;
  const int st = check_linear(a, x, rows, k, x_row_stride, w, 2 * ffn, w_row_stride);
  if (st != INT8KV_OK) return st;
  if (!out) return INT8KV_E_NULL;
  if (!rows16(out, out_row_stride) || out_row_stride < ffn) return INT8KV_E_STRIDE;
  a.n = (int32_t)ffn;
  a.tiles = (int32_t)(ffn / 8);
  a.out = static_cast<uint16_t*>(out);
  a.os = out_row_stride;
  return launch_linear<kEpiSilu>(a, static_cast<hipStream_t>(stream));
}

extern "C" int int8kv_skinny_linear_add_rms_norm(
    const void* x, int64_t rows, int64_t k, int64_t x_row_stride, const void* w, int64_t n,
    int64_t w_row_stride, void* residual, int64_t residual_row_stride, const void* norm_weight,
    void* out, int64_t out_row_stride, float eps, void* workspace, int64_t workspace_bytes,
    void* stream) {
  LinearArgs a;
  const int st = check_linear(a, x, rows, k, x_row_stride, w, n, w_row_stride);
  if (st != INT8KV_OK) return st;
  if (!residual || !norm_weight || !out) return INT8KV_E_NULL;
  if (n > (int64_t)kNormVec * kNormThreads * 4) return INT8KV_E_SHAPE;
  if (!rows16(residual, residual_row_stride) || !rows16(out, out_row_stride) ||
      !rows16(norm_weight, 0) || residual_row_stride < n || out_row_stride < n)
    return INT8KV_E_STRIDE;
  if (!workspace || workspace_bytes < int8kv_skinny_linear_workspace_bytes(rows, k, n) ||
      reinterpret_cast<uintptr_t>(workspace) % 16)
    return INT8KV_E_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  a.part = static_cast<float*>(workspace);
  const int e = launch_linear<kEpiPart>(a, s);
  if (e != 0) return e;
  auto* r = static_cast<uint16_t*>(residual);
  auto* nw = static_cast<const uint16_t*>(norm_weight);
  auto* o = static_cast<uint16_t*>(out);
  switch (a.groups) {
#define INT8KV_NORM(G)                                                        \
  case G:                                                                     \
    launch_norm<G>(a, r, residual_row_stride, nw, o, out_row_stride, eps, s); \
    break;
    INT8KV_NORM(1) INT8KV_NORM(2) INT8KV_NORM(3) INT8KV_NORM(4)
    INT8KV_NORM(5) INT8KV_NORM(6) INT8KV_NORM(7) INT8KV_NORM(8)
#undef INT8KV_NORM
    default: return INT8KV_E_SHAPE;
  }
  return (int)hipGetLastError();
}
