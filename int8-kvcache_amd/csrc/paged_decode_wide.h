// Range kernel of the paged decode for GQA groups above 16 query heads (multi-query attention):
// one wave holds CT column tiles of 16 query heads of one kv head, so each K/V byte is read and
// dequantised once for up to 16 CT heads.  Compiled per cache type (paged_decode_wide_*.hip).
//
// Bound: with one wave per column tile (decode_kernel's layout) every tile of 16 heads read,
// dequantised and multiplied its kv head's K/V again, and 71 heads on one kv head took 5 waves'
// time for one wave's bytes (head_dim 64, INT8, B = 40 x 4096, 21.7 MB: 40.4 us per call, 0.54
// TB/s).  Here the tile's K and V operands are built once and serve all CT tiles; what is left
// per extra tile is its MFMAs and its softmax (per 32 tokens and wave 0.43 + 0.29 CT us, against
// 1.04 us per wave and tile): 27.3 us per call, bound by that arithmetic and by ~12 us from the
// launch to a range's first tile and from its last tile to its records.  How many tiles a wave
// takes, and which calls keep one wave per tile: wide_column_tiles (paged_decode.hip).
// Split: a range of the token stream (the plan of decode_kernel) belongs to a workgroup of four
// waves, one per SIMD, which share each of its sequences' tiles and combine their softmax states
// in LDS.  One wave per range instead would leave four times the partial records, and a record
// of 71 heads (19 KB) is as large as the K/V of 150 tokens.

#ifndef INT8KV_PAGED_DECODE_WIDE_H
#define INT8KV_PAGED_DECODE_WIDE_H

#include "paged_decode_kernels.h"

namespace int8kv {

constexpr int kWideWaves = 4;

// Column tile c of grid head y (kv head y / cg, column tiles CT (y % cg) ..): g <= 0 where the
// group has no such tile.
template <int CT>
__device__ __forceinline__ HeadMap wide_map(const DecodeArgs& a, int y, int c) {
  const int kv = y / a.col_tiles;
  const int t = (y - kv * a.col_tiles) * CT + c;
  const int rest = a.group - 16 * t;
  return {kv, kv * a.group + 16 * t, rest < 16 ? rest : 16};
}

// tile_scores for CT column tiles: each K operand is built once and multiplied by every tile's
// query operand; the softmax update runs per tile.
template <int CACHE, int HD, int CT, bool QSPLIT>
__device__ __forceinline__ void wide_scores(const KTile<CACHE, 2, HD>& r,
                                            const typename MfmaOp<CACHE>::T (&qop)[CT][HD / 32],
                                            const typename MfmaOp<CACHE>::T (&qlo)[CT][HD / 32],
                                            f32x4 (&acc)[CT][HD / 16], float (&m_run)[CT],
                                            float (&l_part)[CT], int valid, int lg,
                                            const float (&s_scale)[CT],
                                            typename MfmaOp<CACHE>::T (&pop)[CT][2]) {
  typedef typename MfmaOp<CACHE>::T OpT;
  typedef typename MfmaOp<CACHE>::E E;
  f32x4 S[CT][2];
#pragma unroll
  for (int c = 0; c < CT; ++c) S[c][0] = S[c][1] = (f32x4)(0.0f);
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int ks = 0; ks < HD / 32; ++ks) {
      OpT kop;
      if constexpr (CACHE == kI8) {
        const uint32_t d0 = r.k[s][ks >> 1][(ks & 1) * 2] ^ kSignFlip;
        const uint32_t d1 = r.k[s][ks >> 1][(ks & 1) * 2 + 1] ^ kSignFlip;
        kop = i8x8_to_f16(d0, d1);
      } else {
        kop = __builtin_bit_cast(OpT, r.k[s][ks]);
      }
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        S[c][s] = mfma(kop, qop[c][ks], S[c][s]);
        if constexpr (QSPLIT) S[c][s] = mfma(kop, qlo[c][ks], S[c][s]);
      }
    }
  // Every tile's scores and maxima first, then one branch for all of them: with a branch per tile
  // the tiles' exchanges and exponentials ran one after another, each at its own latency (one
  // wave per SIMD: nothing else hides it).
  float mx[CT];
  bool need = false;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
#pragma unroll
    for (int s = 0; s < 2; ++s) S[c][s] *= s_scale[c];
  }
  if (valid < 2 * kRows) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)
        if (16 * s + 4 * lg + rr >= valid) {
#pragma unroll
          for (int c = 0; c < CT; ++c) S[c][s][rr] = -INFINITY;
        }
  }
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    float m = S[c][0][0];
#pragma unroll
    for (int e = 1; e < 8; ++e) m = fmaxf(m, S[c][e >> 2][e & 3]);
    mx[c] = m;
  }
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    mx[c] = rows_max(mx[c]);
    need |= mx[c] > m_run[c] + kLazyRescale;
  }
  if (__any(need)) {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const float m_new = mx[c] > m_run[c] + kLazyRescale ? mx[c] : m_run[c];
      // (m_run = m_new = -inf before a tile's first finite score: exp2(NaN) would spoil the zeros)
      const float alpha = m_new == m_run[c] ? 1.0f : exp2_fast(m_run[c] - m_new);
      m_run[c] = m_new;
      l_part[c] *= alpha;
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt) acc[c][dt] *= alpha;
    }
  }
#pragma unroll
  for (int c = 0; c < CT; ++c) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float pe = exp2_fast(S[c][e >> 2][e & 3] - m_run[c]);
      l_part[c] += pe;
      const E hi = (E)pe;
      pop[c][0][e] = hi;
      pop[c][1][e] = (E)(pe - (float)hi);
    }
  }
}

// tile_pv for CT column tiles: each V operand is built once.
template <int CACHE, int HD, int CT>
__device__ __forceinline__ void wide_pv(VTile<CACHE, 2, HD>& r,
                                        const typename MfmaOp<CACHE>::T (&pop)[CT][2],
                                        f32x4 (&acc)[CT][HD / 16], int valid, int lg) {
  typedef typename MfmaOp<CACHE>::T OpT;
  constexpr int DW = v_dwords<CACHE, HD>();
  if constexpr (CACHE != kI8) {
    // 16-bit rows past the sequence end may hold non-finite garbage; 0 * NaN would leak.
    if (valid < 2 * kRows) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          if (16 * s + 4 * lg + rr >= valid) {
#pragma unroll
            for (int k = 0; k < DW; ++k) r.v[s][rr][k] = 0u;
          }
    }
  }
  uint32_t pk[2][2][DW][2];  // INT8: [row group][token pair][row dword][byte pair 01/23]
  if constexpr (CACHE == kI8) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int rp = 0; rp < 2; ++rp)
#pragma unroll
        for (int h = 0; h < DW; ++h) {
          const uint32_t a0 = r.v[s][2 * rp][h] ^ kSignFlip;
          const uint32_t b0 = r.v[s][2 * rp + 1][h] ^ kSignFlip;
          pk[s][rp][h][0] = perm(a0, b0, 0x01050004u);
          pk[s][rp][h][1] = perm(a0, b0, 0x03070206u);
        }
  }
#pragma unroll
  for (int dt = 0; dt < HD / 16; ++dt) {
    u32x4 w;
    OpT vop;
    if constexpr (CACHE == kI8) {
      const int h = dt >> 2, bp = (dt >> 1) & 1;
      const uint32_t sel = (dt & 1) ? kSelHi : kSelLo;
      w[0] = perm(kMagic, pk[0][0][h][bp], sel);
      w[1] = perm(kMagic, pk[0][1][h][bp], sel);
      w[2] = perm(kMagic, pk[1][0][h][bp], sel);
      w[3] = perm(kMagic, pk[1][1][h][bp], sel);
      vop = __builtin_bit_cast(f16x8, w) - (f16x8)(_Float16)1152.0f;
    } else {
      const int wd = dt >> 1;
      const uint32_t sel = (dt & 1) ? 0x07060302u : 0x05040100u;
      w[0] = perm(r.v[0][1][wd], r.v[0][0][wd], sel);
      w[1] = perm(r.v[0][3][wd], r.v[0][2][wd], sel);
      w[2] = perm(r.v[1][1][wd], r.v[1][0][wd], sel);
      w[3] = perm(r.v[1][3][wd], r.v[1][2][wd], sel);
      vop = __builtin_bit_cast(OpT, w);
    }
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      acc[c][dt] = mfma(vop, pop[c][0], acc[c][dt]);
      acc[c][dt] = mfma(vop, pop[c][1], acc[c][dt]);
    }
  }
}

// Barrier for data exchanged through LDS: waits for this wave's LDS accesses only, so that the tile
// loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The query operands of a segment's column tiles, built once per workgroup (wave w builds tiles w,
// w + 4) and read by every wave: [hi / lo][k-step][lane], and the score factor per lane.
template <int CT, int HD, bool QSPLIT>
struct WideQuery {
  u32x4 op[CT][(QSPLIT ? 2 : 1) * (HD / 32)][kWave];
  float scale[CT][kWave];
};

// Tiles [ta, tb) of sequence b (length L) for the column tiles of grid head y, one wave (an empty
// share too: every wave of the workgroup comes here); leaves the softmax states in the wave's LDS
// slots: g_acc [CT][HD/4][64], g_m / g_l [CT][16].  Two tiles of K/V loads in flight, block ids
// staged in LDS, as run_segment.  The tile body is instantiated twice only (even and odd tiles;
// refills past the share's end request its last tile again, at most two of them): a short call
// spends its time on instruction fetches otherwise (five copies, 71 KB of code, took 16 us for
// two tiles per wave).
template <int CACHE, int QT, bool NT, int HD, int CT, bool PAD>
__device__ __forceinline__ void wide_segment(const DecodeArgs& a, int32_t* ids, int64_t b, int64_t L,
                                             int y, int64_t ta, int64_t tb, int lane, int wave,
                                             WideQuery<CT, HD, QT == kF32>& sq, float* g_acc,
                                             float* g_m, float* g_l) {
  typedef typename MfmaOp<CACHE>::T OpT;
  constexpr bool kSpread = CACHE != kI8;
  constexpr bool QSPLIT = QT == kF32;
  constexpr int kTileTokens = 2 * kRows;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int kvh = y / a.col_tiles;
  const char* kb = a.kc + (int64_t)kvh * a.kc_sh;
  const char* vb = a.vc + (int64_t)kvh * a.vc_sh;
  const int64_t nblk = (L + (1 << a.block_shift) - 1) >> a.block_shift;
  const int gmask = (1 << (a.block_shift - 4)) - 1;

  f32x4 acc[CT][HD / 16];
  float m_run[CT], l_part[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    m_run[c] = -INFINITY;
    l_part[c] = 0.0f;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) acc[c][dt] = (f32x4)(0.0f);
  }

  int64_t c0 = ta;
  int64_t c1 = (tb - c0 > kChunkTiles) ? c0 + kChunkTiles : tb;
  KTile<CACHE, 2, HD> kt[2];
  VTile<CACHE, 2, HD> vt[2];
  TileRows<2> ph[2];
  OpT pop[CT][2];
  auto blocks_of = [&](int64_t t, TileRows<2>& p) {
    t = t < c1 ? t : c1 - 1;
    const int j = 2 * (int)(t - c0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      p.id[s] = __builtin_amdgcn_readfirstlane(ids[j + s]);
      p.row[s] = (((int)t * 2 + s) & gmask) * kRows;
    }
  };
  auto request = [&](int64_t t, int d) {
    blocks_of(t, ph[d]);
    issue_k<CACHE, 2, NT, HD, PAD, kSpread>(kt[d], kb, ph[d], a, li, lg);
    issue_v<CACHE, 2, NT, HD, PAD>(vt[d], vb, ph[d], a, li, lg);
  };

  // The first chunk's block ids and tiles are requested before the query operands are built.
  const bool any = ta < tb;  // wave-uniform
  if (any) {
    stage_block_ids<2>(a, ids, b, c0, c1, nblk, lane);
    request(c0, 0);
    request(c0 + 1, 1);
  }
  constexpr int kMine = (CT + kWideWaves - 1) / kWideWaves;
  const float ksc[2] = {CACHE == kI8 ? a.k_scale[kvh] : 1.0f, 1.0f};
  QueryRaw<QT, HD> raw[kMine];
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    const int c = wave + kWideWaves * j;
    if (c < CT) issue_query<QT, HD, false, PAD, kSpread>(a, b, wide_map<CT>(a, y, c), li, lg, raw[j]);
  }
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    const int c = wave + kWideWaves * j;
    if (c >= CT) break;
    OpT hi[HD / 32];
    OpT lo[HD / 32];  // (a quantised fp32 query is exact in the hi operand alone)
    i32x4 unused[HD / 64];
#pragma unroll
    for (int ks = 0; ks < HD / 32; ++ks) lo[ks] = (OpT)(0.0f);
    sq.scale[c][lane] = finish_query<CACHE, QT, false, HD, false, true>(a, raw[j], ksc, hi, lo, unused);
#pragma unroll
    for (int ks = 0; ks < HD / 32; ++ks) {
      sq.op[c][ks][lane] = __builtin_bit_cast(u32x4, hi[ks]);
      if constexpr (QSPLIT) sq.op[c][HD / 32 + ks][lane] = __builtin_bit_cast(u32x4, lo[ks]);
    }
  }
  lds_barrier();
  OpT qop[CT][HD / 32];
  OpT qlo[CT][HD / 32];  // unused (and removed by the compiler) unless QSPLIT
  float s_scale[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    s_scale[c] = sq.scale[c][lane];
#pragma unroll
    for (int ks = 0; ks < HD / 32; ++ks) {
      qop[c][ks] = __builtin_bit_cast(OpT, sq.op[c][ks][lane]);
      if constexpr (QSPLIT) qlo[c][ks] = __builtin_bit_cast(OpT, sq.op[c][HD / 32 + ks][lane]);
    }
  }

  auto tile = [&](int64_t t, int d) {
    const int64_t left = L - t * kTileTokens;
    const int valid = left >= kTileTokens ? kTileTokens : (int)left;
    wide_scores<CACHE, HD, CT, QSPLIT>(kt[d], qop, qlo, acc, m_run, l_part, valid, lg, s_scale, pop);
    blocks_of(t + 2, ph[d]);
    issue_k<CACHE, 2, NT, HD, PAD, kSpread>(kt[d], kb, ph[d], a, li, lg);
    __builtin_amdgcn_sched_barrier(0);
    wide_pv<CACHE, HD, CT>(vt[d], pop, acc, valid, lg);
    issue_v<CACHE, 2, NT, HD, PAD>(vt[d], vb, ph[d], a, li, lg);
    __builtin_amdgcn_sched_barrier(0);
  };
  while (any) {
    for (int64_t t = c0; t < c1; t += 2) {
      tile(t, 0);
      if (t + 1 < c1) tile(t + 1, 1);
    }
    if (c1 >= tb) break;
    c0 = c1;
    c1 = (tb - c0 > kChunkTiles) ? c0 + kChunkTiles : tb;
    stage_block_ids<2>(a, ids, b, c0, c1, nblk, lane);
    request(c0, 0);
    request(c0 + 1, 1);
  }

#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const float l = rows_sum(l_part[c]);
#pragma unroll
    for (int rr = 0; rr < 4; ++rr)
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt)
        g_acc[((c * 4 + rr) * (HD / 16) + dt) * kWave + lane] = acc[c][dt][rr];
    if (lg == 0) {
      g_m[16 * c + li] = m_run[c];
      g_l[16 * c + li] = l;
    }
  }
}

// grid (max_ranges, kv heads x col_tiles), four waves.  The plan, the walk and the records are
// decode_kernel's (one range per workgroup); the workgroup's waves share each segment.
template <int CACHE, int QT, bool NT, int HD, int CT, bool PAD>
__global__ __launch_bounds__(kWideWaves * 64) __attribute__((amdgpu_waves_per_eu(1))) void wide_kernel(DecodeArgs a) {
  __shared__ int32_t s_ids[kWideWaves][kChunkTiles * 2];
  __shared__ float s_acc[kWideWaves][CT * (HD / 4) * kWave];
  __shared__ float s_m[kWideWaves][CT * 16];
  __shared__ float s_l[kWideWaves][CT * 16];
  __shared__ WideQuery<CT, HD, QT == kF32> s_q;
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int y = blockIdx.y;

  const int64_t L0 = seq_len_of(a, lane);
  const Plan plan = make_plan(a, lane, L0);
  const int64_t r = blockIdx.x;
  const bool cut_writer = a.cut_desc && y == 0 && threadIdx.x == 0;
  if (cut_writer) {
    a.ws_cut[4 * r] = -1;
    a.ws_cut[4 * r + 2] = plan.U;
    a.ws_cut[4 * r + 3] = pack_plan(plan);
  }
  if (r >= plan.P) return;  // uniform over the workgroup
  const int64_t u0 = range_start(plan, r);
  const int64_t u1 = range_start(plan, r + 1);
  const bool last_range = r == plan.P - 1;

  // One segment: tiles [ta, te) of sequence b, every wave an equal share.
  auto segment = [&](int64_t b, int64_t L, int64_t ta, int64_t te, bool full, int64_t rec) {
    const int64_t n = te - ta;
    wide_segment<CACHE, QT, NT, HD, CT, PAD>(a, s_ids[wave], b, L, y, ta + wave * n / kWideWaves,
                                             ta + (wave + 1) * n / kWideWaves, lane, wave, s_q,
                                             s_acc[wave], s_m[wave], s_l[wave]);
    __syncthreads();
    // Online-softmax merge of the four states, one accumulator row group per wave (group_kernel).
    const int kv = y / a.col_tiles;
    const float vscale = (CACHE == kI8 && full) ? fmaxf(a.v_scale[kv], 1e-6f) : 1.0f;
    const int rr = wave;
    float Mc[CT], Lc[CT], Oc[CT][HD / 16];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      float m[kWideWaves], l[kWideWaves];
#pragma unroll
      for (int w = 0; w < kWideWaves; ++w) {
        m[w] = s_m[w][16 * c + li];
        l[w] = s_l[w][16 * c + li];
      }
      Mc[c] = fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3]));
      Lc[c] = 0.0f;
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt) Oc[c][dt] = 0.0f;
#pragma unroll
      for (int w = 0; w < kWideWaves; ++w) {
        // (nothing finite anywhere: added unscaled, so a NaN still reaches the output)
        const float f = Mc[c] == -INFINITY ? 1.0f : exp2_fast(m[w] - Mc[c]);
        Lc[c] += l[w] * f;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt)
          Oc[c][dt] += s_acc[w][((c * 4 + rr) * (HD / 16) + dt) * kWave + lane] * f;
      }
    }
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const HeadMap hm = wide_map<CT>(a, y, c);
      if (li >= hm.g) continue;
      float (&O)[HD / 16] = Oc[c];
      const float M = Mc[c], Ls = Lc[c];
      const int h = hm.q0 + li;
      const int e = HD / 4 * lg + HD / 16 * rr;  // first head_dim element
      if (full) {
        const float inv = Ls > 0.0f ? vscale / Ls : 0.0f;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) O[dt] *= inv;
        if (!PAD || e < a.head_dim)
          store_n<QT, HD / 16>(a.out + (b * a.o_sb + (int64_t)h * a.o_sh + e) * esize<QT>(), O);
      } else {
        const int64_t row = rec * a.num_q_heads + h;
        store_n<kF32, HD / 16>(reinterpret_cast<char*>(a.ws_acc + row * HD + e), O);
        if (rr == 0 && lg == 0) {
          a.ws_m[row] = M;
          a.ws_l[row] = Ls;
        }
      }
    }
    __syncthreads();  // before the next segment's states overwrite these
  };

  int64_t cum = 0;  // units of the sequences before this 64-sequence chunk
  int64_t L = L0;
  for (int64_t base = 0; base < a.batch; base += kWave) {
    if (base > 0) L = seq_len_of(a, base + lane);
    const int64_t n = tiles_of(a, L);
    const int64_t u = units_of(a, n);
    const int64_t incl = units_scan(a, u, lane) + cum;
    const int64_t excl = incl - u;
    const int64_t chunk_end = readlane64(incl, kWave - 1);
    if (chunk_end >= u0) {
      // Empty sequences occupy no units: the range holding their position writes their zeros.
      uint64_t zmask = __ballot(base + lane < a.batch && n == 0 && excl >= u0 &&
                                (excl < u1 || (last_range && excl == plan.U)));
      while (zmask) {
        const int j = __builtin_ctzll(zmask);
        zmask &= zmask - 1;
        for (int c = wave; c < CT; c += kWideWaves) {
          const HeadMap hm = wide_map<CT>(a, y, c);
          if (hm.g > 0) write_zero_rows<QT, HD, PAD>(a, base + j, hm, lane);
        }
      }
      uint64_t mask = __ballot(n > 0 && incl > u0 && excl + a.seq_cost < u1);
      while (mask) {
        const int j = __builtin_ctzll(mask);
        mask &= mask - 1;
        const int64_t first = readlane64(excl, j) + a.seq_cost;  // unit of tile 0
        const int64_t nb = readlane64(n, j);
        const int64_t Lb = readlane64(L, j);
        const int64_t ta = (u0 > first ? u0 : first) - first;
        const int64_t te = (u1 < first + nb ? u1 : first + nb) - first;
        if (ta >= te) continue;
        if (cut_writer && ta == 0 && te < nb) {  // b starts here and runs past this range
          a.ws_cut[4 * r] = base + j;
          a.ws_cut[4 * r + 1] = first + nb - 1;
        }
        segment(base + j, Lb, ta, te, ta == 0 && te == nb, 2 * r + cut_slot(ta));
      }
    }
    if (chunk_end >= u1 && !last_range) break;
    cum = chunk_end;
  }
}

// ------------------------------------------------------------------------ launchers
template <int CACHE, int QT, int HD, int CT, bool PAD>
inline void launch_wide_nt(const DecodeArgs& a, bool nt, dim3 grid, hipStream_t s) {
  const dim3 block(kWideWaves * kWave);
  if constexpr (!PAD && (CACHE == kI8 || HD == 128)) {  // where plan_call asks for it
    if (nt) {
      hipLaunchKernelGGL((wide_kernel<CACHE, QT, true, HD, CT, PAD>), grid, block, 0, s, a);
      return;
    }
  }
  hipLaunchKernelGGL((wide_kernel<CACHE, QT, false, HD, CT, PAD>), grid, block, 0, s, a);
}

template <int CACHE, int QT, int HD, bool PAD>
inline int launch_wide_ct(const DecodeArgs& a, const HostPlan& hp, hipStream_t s) {
  const dim3 grid((unsigned)a.max_ranges, (unsigned)a.num_kv_heads);
  constexpr int kMost = wide_most_tiles(HD);
  switch (hp.ct) {
    case 2:
      if constexpr (kMost >= 2) launch_wide_nt<CACHE, QT, HD, 2, PAD>(a, hp.nt, grid, s);
      break;
    case 3:
      if constexpr (kMost >= 3) launch_wide_nt<CACHE, QT, HD, 3, PAD>(a, hp.nt, grid, s);
      break;
    case 4:
      if constexpr (kMost >= 4) launch_wide_nt<CACHE, QT, HD, 4, PAD>(a, hp.nt, grid, s);
      break;
    case 5:
      if constexpr (kMost >= 5) launch_wide_nt<CACHE, QT, HD, 5, PAD>(a, hp.nt, grid, s);
      break;
    default:
      return INT8KV_E_SHAPE;
  }
  return (int)hipGetLastError();
}

template <int CACHE, bool PAD, int QT>
int launch_wide_hd(const DecodeArgs& a, const HostPlan& hp, hipStream_t s) {
  return hp.hd == 64 ? launch_wide_ct<CACHE, QT, 64, PAD>(a, hp, s)
                     : launch_wide_ct<CACHE, QT, 128, PAD>(a, hp, s);
}

template <int CACHE, bool PAD>
int launch_wide_q(const DecodeArgs& a, const HostPlan& hp, int query_dtype, hipStream_t s) {
  switch (query_dtype) {
    case INT8KV_F32: return launch_wide_hd<CACHE, PAD, kF32>(a, hp, s);
    case INT8KV_F16: return launch_wide_hd<CACHE, PAD, kF16>(a, hp, s);
    default: return launch_wide_hd<CACHE, PAD, kBF16>(a, hp, s);
  }
}

}  // namespace int8kv

#endif  // INT8KV_PAGED_DECODE_WIDE_H
