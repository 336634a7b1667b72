// Attention forward of a decode step for gfx950, bf16/f16, head dim 64 or 128: at most 16 query rows share a kv head
// (rows of the sequence times the heads of the group), every key is theirs up to the batch's count.
//
// HBM-bound: every K / V byte is read once and used for all the rows.  One workgroup = four wavefronts that share out
// the 32-key steps of one part of one (batch, kv head); a wavefront streams K and V straight from memory into registers,
// two steps (32 KB at head dim 128) on their way, and the four results meet in LDS.  About 512 workgroups, two per
// compute unit, keep 64 MB requested.  Where the sequences are fewer, their keys are split into parts that
// fwd_split_merge_kernel adds up.
//
// The products run on the 16x16x32 matrix op, transposed: S^T = K Q^T with 16 keys a block, O^T = V^T P^T.  Lane (n, g),
// n = lane % 16, g = lane / 16, holds of a step
//   K  two rows' quarter: row m = n of block blk is key 16 blk + 4 (m % 4) + m / 4, elements 32 ks + 8 g .. +7 of it
//   V  eight rows' sixteenth: keys 4 s + g, s = 0 .. 7, elements PV n .. +PV-1 (one load instruction covers whole rows)
// Register i of block blk of the score tile is then key 4 (4 blk + i) + g of row n: slot s = 4 blk + i of the lane's own V
// pieces, so the probabilities, packed in pairs, are the second product's operand.  V's elements are paired
// across keys with one byte permutation per register and pair: matrix op e takes element e of every key, output row PV n + e.
// (On the 32x32x16 op through LDS, a wavefront per head with one of its 32 rows live, fwd_mfma_w32.hip spends as long on the
// matrix ops as on the bytes, reads K and V once per head where the group's heads do not divide its wavefronts, and
// walks one tile per trip at the start.)
#include <algorithm>

#include "fwd_mfma.h"
#include "split_merge.h"

namespace mi355 {
namespace {

constexpr int kStep = 32;  // keys of a step
constexpr int kWaves = 4;  // wavefronts that share a part

template <typename T>
struct Mma16;
template <>
struct Mma16<bf16_t> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
};
template <>
struct Mma16<f16_t> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
};

template <typename T, int D>
__global__ __launch_bounds__(64 * kWaves, 2) void fwd_few_rows_kernel(FwdM p) {
  constexpr int KS = D / 32;  // contraction steps of S^T
  constexpr int PV = D / 16;  // elements of a lane's V piece = matrix ops of O^T
  constexpr int VW = PV / 2;  // ... in dwords
  typedef __attribute__((ext_vector_type(VW))) uint32_t vpiece_t;
  struct Step {
    u32x4 k[2][KS];
    vpiece_t v[8];
  };
  __shared__ __attribute__((aligned(16))) float o_lds[kWaves][16][D + 4];  // (+4: rows of different lanes in different banks)
  __shared__ float m_lds[kWaves][16], l_lds[kWaves][16];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int rep = p.Hq / p.Hkv, R = rep * p.L;
  const int split = blockIdx.x % p.n_split, bhk = blockIdx.x / p.n_split;
  const int b = bhk / p.Hkv, hk = bhk % p.Hkv;
  int S = p.S;
  if (p.kv_lens) S = min(S, max(p.kv_lens[b], 0));
  // the steps of this part (with key counts: an equal share of the batch's own)
  const int steps = (S + kStep - 1) / kStep;
  const int per = p.split_tiles && !p.kv_lens ? p.split_tiles : (steps + p.n_split - 1) / p.n_split;
  const int first = split * per, end = min(steps, first + per);

  const int row = min(n, R - 1);  // row r of the workgroup: head r % rep of the group, sequence row r / rep
  u32x4 qf[KS];
  {
    const T* q = (const T*)p.q + b * p.q_sb + (int64_t)(hk * rep + row % rep) * p.q_sh + (int64_t)(row / rep) * p.q_sl + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const u32x4*)(q + 32 * ks);
  }
  const char* const kb = (const char*)((const T*)p.k + b * p.k_sb + hk * p.k_sh) + 16 * g;
  const char* const vb = (const char*)((const T*)p.v + b * p.v_sb + hk * p.v_sh) + 2 * PV * n;
  const uint32_t ksl = (uint32_t)p.k_sl * 2, vsl = (uint32_t)p.v_sl * 2;  // (host checked: a (batch, head) slab spans < 2^31 bytes)
  const int last = S - 1;
  // (rows of a step past the last key clamp to it; non-temporal: the cache is read once)
  auto load = [&](Step& w, int step) {
    const int base = step * kStep;
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
      const char* kr = kb + (uint32_t)min(base + 16 * blk + 4 * (n & 3) + (n >> 2), last) * ksl;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) w.k[blk][ks] = __builtin_nontemporal_load((const u32x4*)(kr + 64 * ks));
    }
#pragma unroll
    for (int s = 0; s < 8; ++s)
      w.v[s] = __builtin_nontemporal_load((const vpiece_t*)(vb + (uint32_t)min(base + 4 * s + g, last) * vsl));
  };

  f32x4 oacc[PV];
#pragma unroll
  for (int e = 0; e < PV; ++e) oacc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;  // m_run: the row's largest raw score so far; l_run: this lane's share of its sum
  const float c = p.scale * kLog2eF;
  auto compute = [&](Step& w, int step) {
    if (step * kStep + kStep > S) {  // (keys past the last one: zeros, so that an infinite last row is not multiplied by 0)
#pragma unroll
      for (int s = 0; s < 8; ++s)
        if (step * kStep + 4 * s + g > last) w.v[s] = vpiece_t{};
    }
    f32x4 s[2];
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
      s[blk] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s[blk] = Mma16<T>::run(w.k[blk][ks], qf[ks], s[blk]);
    }
    float t[8], tm = -INFINITY;
    const int key0 = step * kStep + g;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      t[i] = key0 + 4 * i <= last ? s[i >> 2][i & 3] : -INFINITY;
      tm = fmaxf(tm, t[i]);
    }
    tm = fmaxf(tm, __shfl_xor(tm, 16, 64));
    tm = fmaxf(tm, __shfl_xor(tm, 32, 64));
    const float m_new = fmaxf(m_run, tm);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;  // (scores that are all -inf: probabilities 0)
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * c), mc = m_use * c;
    m_run = m_new;
    float pr[8], ps = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      pr[i] = __builtin_amdgcn_exp2f(fmaf(t[i], c, -mc));
      ps += pr[i];
    }
    l_run = fmaf(l_run, alpha, ps);
    const u32x4 pf = {Mma<T>::pack(pr[0], pr[1]), Mma<T>::pack(pr[2], pr[3]), Mma<T>::pack(pr[4], pr[5]), Mma<T>::pack(pr[6], pr[7])};
#pragma unroll
    for (int d = 0; d < VW; ++d) {
      u32x4 lo, hi;  // elements 2 d and 2 d + 1 of the eight keys
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t a = w.v[2 * j][d], a1 = w.v[2 * j + 1][d];
        lo[j] = __builtin_amdgcn_perm(a1, a, 0x05040100);
        hi[j] = __builtin_amdgcn_perm(a1, a, 0x07060302);
      }
      oacc[2 * d] = Mma16<T>::run(lo, pf, oacc[2 * d] * alpha);
      oacc[2 * d + 1] = Mma16<T>::run(hi, pf, oacc[2 * d + 1] * alpha);
    }
  };

  // Step i of this wavefront is step t + i kWaves of the sequence; two are on their way.  (Nothing is requested past the
  // last one: such loads, of a row that is in the cache, held up the barrier below by a whole trip.  Branches around the
  // loads would cost as much, every wait behind one being for all loads: the last one or two steps are code of their own.)
  const int t = first + wave, mine = (end - t + kWaves - 1) / kWaves;
  if (t < end) {
    Step wa, wb;
    int i = 0;
    load(wa, t);
    for (; i + 2 < mine; i += 2) {
      load(wb, t + (i + 1) * kWaves);
      __builtin_amdgcn_sched_barrier(0);  // (a step's loads stay ahead of the work they overlap)
      compute(wa, t + i * kWaves);
      __builtin_amdgcn_sched_barrier(0);
      load(wa, t + (i + 2) * kWaves);
      __builtin_amdgcn_sched_barrier(0);
      compute(wb, t + (i + 1) * kWaves);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (i + 1 < mine) {
      load(wb, t + (i + 1) * kWaves);
      __builtin_amdgcn_sched_barrier(0);
      compute(wa, t + i * kWaves);
      __builtin_amdgcn_sched_barrier(0);
      compute(wb, t + (i + 1) * kWaves);
    } else {
      compute(wa, t + i * kWaves);
    }
  }
  // ---- the four wavefronts' rows ------------------------------------------------------------------------
  float l_tot = l_run + __shfl_xor(l_run, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  if (n < R) {
    // (register a of matrix op e is row PV (4 g + a) + e of O^T)
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int e = 0; e < PV; e += 4)
        *(f32x4*)(&o_lds[wave][n][PV * (4 * g + a) + e]) = f32x4{oacc[e][a], oacc[e + 1][a], oacc[e + 2][a], oacc[e + 3][a]};
    if (g == 0) m_lds[wave][n] = m_run, l_lds[wave][n] = l_tot;
  }
  __syncthreads();
  for (int i = tid; i < R * (D / 4); i += 64 * kWaves) {
    const int r = i / (D / 4), d = (i % (D / 4)) * 4;
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) M = fmaxf(M, m_lds[w][r]);
    const float ref = M == -INFINITY ? 0.f : M;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float f = __builtin_amdgcn_exp2f((m_lds[w][r] - ref) * c);
      L = fmaf(l_lds[w][r], f, L);
      o += *(const f32x4*)(&o_lds[w][r][d]) * f;
    }
    const float inv = L == 0.f ? 0.f : 1.f / L;
    const float lse = L > 0.f ? ref * p.scale + __builtin_logf(L) : -INFINITY;
    const int h = hk * rep + r % rep, l = r / rep;
    if (p.n_split > 1) {
      const int64_t prow = (((int64_t)b * p.Hq + h) * p.n_split + split) * p.L + l;
      *(f32x4*)(p.part_o + prow * D + d) = o * inv;
      if (d == 0) p.part_lse[prow] = part_lse_of(L, lse);
    } else {
      *(u32x2*)((T*)p.out + b * p.o_sb + h * p.o_sh + l * p.o_sl + d) = u32x2{Mma<T>::pack(o[0] * inv, o[1] * inv), Mma<T>::pack(o[2] * inv, o[3] * inv)};
      if (d == 0 && p.lse) p.lse[((int64_t)b * p.Hq + h) * p.L + l] = lse;
    }
  }
}

}  // namespace

bool few_rows_supported(const FwdM& g, int head_dim) {
  return head_dim <= 128 && g.d_real == head_dim && g.dv_real == head_dim && (g.Hq / g.Hkv) * (int64_t)g.L <= 16 && !g.causal &&
         g.bias_kind == 0 && g.keep_scale == 0.f && g.window == 0 && !g.sink_logit && !g.sm.any;
}

// Parts per (batch, kv head).  One workgroup per compute unit, or two, each with the same share: what is asked for beyond
// that only queues at the memory (B=8, 32/8 heads, 2049 keys: 256 workgroups 17.0 us, 384 19.0, 512 18.3, 1024 19.7), and a
// turn that fills the chip in part leaves bandwidth unused (2048 keys: B=20 in 160 workgroups 41.5, 480 34.4; B=40 in 320 71,
// 640 64, 960 59.6).  At least four steps, one per wavefront, and twelve in all, for less the second launch weighs more
// (32/8 heads, 1000 keys: 8 parts 8.7, 4 parts 10.0, 2 parts 13.3; 512 keys, B=4: 4 parts 8.9, one 9.9).
//   No parts at all where what they save, at 6.3 TB/s or 1.75 us a step of a workgroup (head dim 128), is less than the merge
// costs: 3 us, and 2.5 more per thousand rows (1.75 at head dim 64), a workgroup each, whose parts go to memory and back in
// float32.  Keys from memory, as planned above / one part, us, D=128: 96 kv heads in all of 16 rows, S=383 12.7 / 11.7, S=2049
// 26.4 / 38.1;  192 of 16, S=1000 29.9 / 22.7, of one row 24.0 / 22.1;  288 of one row, S=1000 32.2 / 37.8, S=383 18.7 / 18.0;
// 768 of 16, S=383 48.3 / 29.3, S=1000 88.3 / 65.3, of one row 65.2 / 63.0.  D=64: 288 of 16, S=1000 25.3 / 21.6, S=2049
// 37.5 / 38.7.  (Beyond 512 workgroups the turns overlap: an unfilled one costs half its idle part.)
void few_rows_plan(FwdM& g) {
  const int64_t groups = (int64_t)g.B * g.Hkv;
  const int steps = (g.S + kStep - 1) / kStep;
  g.split_tiles = 0, g.n_split = 1;
  if (steps < 12) return;
  auto filled = [&](int n) {  // share of the chip's turns that `n` parts fill
    const int64_t wgs = groups * n, slots = wgs <= 256 ? 256 : 512;
    return (double)wgs / (double)(slots * ((wgs + slots - 1) / slots));
  };
  int best = 1;
  double best_use = 0.;
  for (int n = 1; n <= std::min(steps / 4, 256) && (n - 1) * groups <= 1024; ++n) {
    const double use = filled(n) - 0.02 * (n * groups > 256) * (n - 1);
    if (use > best_use) best_use = use, best = n;
  }
  const double width = g.d_real / 128.;
  auto us = [&](int n) {  // estimated, without the merge
    const double f = filled(n), use = groups * n <= 512 ? f : 0.5 + 0.5 * f;
    const int per = (steps + n - 1) / n;
    return std::max((double)groups * g.S * g.d_real * 4 / 6.3e6 / use, 2.5 + 1.75 * width * ((per + kWaves - 1) / kWaves));
  };
  if (best >= 2 && us(1) - us(best) > 3. + (1e-3 + 1.5e-3 * width) * (double)g.B * g.Hq * g.L) {
    g.split_tiles = (steps + best - 1) / best;
    g.n_split = (steps + g.split_tiles - 1) / g.split_tiles;
  }
}

int launch_fwd_few_rows(const FwdM& g, int dtype, int head_dim, hipStream_t s) {
  const int64_t blocks = (int64_t)g.B * g.Hkv * g.n_split;
  if (blocks > 0x7fffffff) {
    set_error("SDPA: too many sequences (%lld)", (long long)blocks);
    return MI355_SDPA_ERR_UNSUPPORTED;
  }
  const dim3 grid((unsigned)blocks), block(64 * kWaves);
  if (dtype == MI355_SDPA_BF16) {
    if (head_dim == 128) hipLaunchKernelGGL((fwd_few_rows_kernel<bf16_t, 128>), grid, block, 0, s, g);
    else hipLaunchKernelGGL((fwd_few_rows_kernel<bf16_t, 64>), grid, block, 0, s, g);
  } else {
    if (head_dim == 128) hipLaunchKernelGGL((fwd_few_rows_kernel<f16_t, 128>), grid, block, 0, s, g);
    else hipLaunchKernelGGL((fwd_few_rows_kernel<f16_t, 64>), grid, block, 0, s, g);
  }
  return check_launch("fwd_few_rows_kernel");
}

}  // namespace mi355
