// dK / dV for head dims above 128 at the full width (256 / 256, narrower rows zero padded), bf16/f16, without a bias
// or dropout: two wavefronts per 32 keys.
//
// The dK and dV accumulators of 32 keys take 256 registers at this width and the K and V fragments 128
// more: one wavefront that holds all of them has a SIMD to itself, and nobody covers its
// S -> P -> dP -> dS -> dV -> dK chain (31 % of the cycles on the matrix pipe).  Here the chain is cut where the fewest
// values cross: wavefront A of a pair holds K and dV, wavefront B holds V and dK,
//   A   S = Q K^T,  P = exp2(c S - lse),   dV^T += dO^T P
//   B   dP = dO V^T,  dS = P (dP - delta),  dK^T += Q^T dS
// and the probabilities, as packed for the second product (times the derivative of a score functor), go from
// A to B through 2 KB of LDS, lane by lane in accumulator order.  Each half is 32 matrix ops per 32 query rows, 64
// registers of fragments and 128 of accumulators: two wavefronts per SIMD, an A and a B.  B works one item (32 query
// rows of one head) behind A, so there is one barrier per item and neither waits for the other inside it.
//
// One workgroup = 128 keys, 8 wavefronts: wavefronts 0-3 are A, 4-7 are B of the same four blocks of 32 keys.
// Q and dO tiles sit in four slots each, requested two items ahead of A (item n in slot n % 4: when item n + 2 is
// requested, B is done with item n - 2).  Products, packing and sums are those of bwd_wide_dkdv_kernel.
//
// B=2, 16 heads, S=4096, D=256, dK/dV before (one wavefront per SIMD, spilling up to 184 B/lane) and now: window 1024 with
// a soft cap 577 -> 350 us, window alone 500 -> 323, soft cap 1033 -> 598, causal alone 706 -> 564 (975 TFLOP/s).
// What bounds it: every matrix op reads one 1 KB operand from LDS (a wavefront has registers for 32 keys, so none
// is used twice), and the two wavefronts of a SIMD reach their products at the same time.  Without the tile loads window and cap took 305 us
// instead of 345, without the softmax as well 300; more operands requested ahead change nothing.
#include "bwd_wide.h"

namespace mi355 {
namespace {

constexpr int SLOTS = 4;
constexpr int TILE_BYTES = TILE_ELEMS * 2;
constexpr int PAIR_Q = 0, PAIR_DO = SLOTS * TILE_BYTES;
constexpr int PAIR_P = 2 * SLOTS * TILE_BYTES;        // [4 blocks of keys][2][2 KB]
constexpr int PAIR_STATS = PAIR_P + 4 * 2 * 2048;     // [SLOTS][lse, delta][64 floats, 32 used]
constexpr int PAIR_LDS = PAIR_STATS + SLOTS * 512;

template <typename V>
__device__ __forceinline__ V lds_read(uint32_t addr) {
  return *(const V __attribute__((address_space(3)))*)(addr);
}
__device__ __forceinline__ u32x2 lds_tr_read(uint32_t addr) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(addr)));
}

// MODE 0: no score functor; 1: a soft cap alone; 2: any functor or document ids.  Key counts, the causal mask and a
// window with sink keys in all of them.
template <typename T, int MODE>
__global__ __launch_bounds__(512, 2) void bwd_wide_pair_kernel(BwdM p) {
  constexpr int KS = DW / 16, DB = DW / 32, NOPS = KS + 2 * DB;
  // operands requested ahead of the matrix op in hand: in the first product, across the vector work, in the second product (where
  // the score tile's registers are free)
  constexpr int AHEAD1 = 4, AHEAD_MID = MODE == 0 ? 3 : 2, AHEAD2 = 5;
  extern __shared__ __attribute__((aligned(1024))) unsigned char pair_lds[];
  typedef __attribute__((address_space(3))) unsigned char* lds_bytes;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_bytes)pair_lds;  // (a multiple of 1024)
  const int streams = p.B * p.Hkv;
  // (split query tiles: part by part, so that a (batch, kv head) keeps its place modulo 8 in the launch order)
  const int part = p.parts > 1 ? (int)blockIdx.x / (streams * p.n_kt) : 0;
  const int blk = blockIdx.x - part * (streams * p.n_kt);
  const int kt = blk / streams;  // low key tiles see the most queries under a causal mask: first
  const int st = blk % streams, b = st / p.Hkv, hk = st % p.Hkv, rep = p.Hq / p.Hkv;
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31;
  // (what depends on the lane is worked out where it is used, a few instructions per item: kept in registers across
  // items it is a dozen of them, and the compiler spills)
  auto lane_now = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave_id & 3;
  const bool is_b = wave_id >= 4;
  const int k0 = kt * 128, kw0 = k0 + wave * 32, key = kw0 + col;

  int S = p.S;  // keys of this batch that take part
  if (p.kv_lens) S = min(S, max(p.kv_lens[b], 0));
  u32x4 f[KS];  // A: this lane's key row of K, B: of V
  {
    // (through a buffer whose bounds turn the columns past a narrow row's end into zeros: with a test around each load
    // the sixteen trips to memory are made one after the other)
    const int kc = max(min(key, S - 1), 0), width = is_b ? p.dv_real : p.d_real;  // (a live row: rows past the batch's keys may hold anything)
    const int64_t sl = is_b ? p.v_sl : p.k_sl;
    const uint16_t* const rows = is_b ? (const uint16_t*)p.v + b * p.v_sb + hk * p.v_sh : (const uint16_t*)p.k + b * p.k_sb + hk * p.k_sh;
    const int row0 = max(min(kw0, S - 1), 0);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr((char*)(rows + row0 * sl)), 0,
                                                                       __builtin_amdgcn_readfirstlane((int)((31 * sl + width) * 2)), 0x00020000);
    const uint32_t at = (uint32_t)((kc - row0) * (int)sl * 2) + (lane >> 5) * 16;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      f[ks] = __builtin_amdgcn_raw_buffer_load_b128(rs, (lane >> 5) * 8 + ks * 16 < width ? at + ks * 32 : 0xfffffff0u, 0, 0);
  }
  f32x16 acc[DB];  // A: dV^T, B: dK^T
#pragma unroll
  for (int i = 0; i < DB; ++i) zero(acc[i]);

  // Items: query tile by query tile from the last one down, heads inside: the workgroups of a kv head,
  // which share an XCD, then want the same Q / dO tile at about the same time and find it in its L2.
  // (window: rows past the window of the block's last key see none of its keys, unless it holds sink keys)
  const int nqs = (p.L + BT - 1) / BT, qs_begin = p.causal ? min(k0 / BT, nqs) : 0;
  int qs_top = nqs;
  if (p.window > 0 && k0 >= p.sink_keys) qs_top = max(min(nqs, (k0 + 128 + p.window - 2) / BT + 1), qs_begin);
  int qs_hi = qs_top, qs_lo = qs_begin;
  if (p.parts > 1) {
    const int chunk = (qs_top - qs_begin + p.parts - 1) / p.parts;
    qs_hi = qs_top - part * chunk, qs_lo = max(qs_hi - chunk, qs_begin);
  }
  const int n_items = k0 >= S ? 0 : max(qs_hi - qs_lo, 0) * rep;  // (no live key in this block: zeros)
  auto advance = [&](int& qs, int& hg) {
    if (++hg == rep) hg = 0, --qs;
  };

  // The next item into its slot: 4 tile loads per wavefront, after one load of the row statistics by wavefronts 0
  // (lse) and 1 (delta): a wait for all but the youngest four then covers both.  Rows past L come as zeros, in the
  // statistics as well: with dO and delta zero such rows add nothing whatever finite P they get.  The three addresses move
  // along with the items (worked out from the item each time they are 155 scalar instructions per item and wavefront).
  int rq = qs_hi - 1, rh = 0;
  const uint16_t* q_at = (const uint16_t*)p.q + b * p.q_sb + hk * rep * p.q_sh + (int64_t)rq * BT * p.q_sl;
  const uint16_t* go_at = (const uint16_t*)p.go + b * p.go_sb + hk * rep * p.go_sh + (int64_t)rq * BT * p.go_sl;
  const float* st_at = (wave_id == 1 ? p.delta : p.lse2) + ((int64_t)b * p.Hq + hk * rep) * p.L + rq * BT;
  auto request = [&](int slot) {
    const int rows = min(p.L - rq * BT, BT);  // >= 1
    const int lane = lane_now();
    if (wave_id < 2) {
      const u32x4 s_rsrc = wide_descriptor(st_at, rows * 4);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                   :: "s"(__builtin_amdgcn_readfirstlane((int)(lds0 + PAIR_STATS + slot * 512 + wave_id * 256))), "v"(lane * 4), "s"(s_rsrc) : "memory", "m0");
    }
    const u32x4 q_rsrc = wide_descriptor(q_at, ((rows - 1) * (int)p.q_sl + p.d_real) * 2);
    const u32x4 go_rsrc = wide_descriptor(go_at, ((rows - 1) * (int)p.go_sl + p.dv_real) * 2);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int ld = wave_id + 8 * n;
      const uint32_t at = lds0 + slot * TILE_BYTES + ld * 1024;
      wide_tile_load(q_rsrc, wide_chunk_off(ld, lane, (int)p.q_sl, p.d_real), at + PAIR_Q);
      wide_tile_load(go_rsrc, wide_chunk_off(ld, lane, (int)p.go_sl, p.dv_real), at + PAIR_DO);
    }
    if (++rh < rep) {
      q_at += p.q_sh, go_at += p.go_sh, st_at += p.L;
    } else {
      rh = 0, --rq;
      q_at -= (rep - 1) * p.q_sh + BT * p.q_sl, go_at -= (rep - 1) * p.go_sh + BT * p.go_sl, st_at -= (int64_t)(rep - 1) * p.L + BT;
    }
  };

  const float c = p.scale * kLog2eF;
  // soft cap: see fwd_mfma_w32.hip; with r = 1 / (1 + 2^(2 log2(e) s / cap)) tanh is 1 - 2 r (exact but for r)
  const float cap_k = MODE == 1 ? 2.f * c / p.sm.softcap : 0.f, cap_l = MODE == 1 ? p.sm.softcap * kLog2eF : 0.f;

  auto compute = [&](int slot, int parity, int qs, int hg, int next_slot) {
    const int q0 = qs * BT;
    const uint32_t q_tile = lds0 + PAIR_Q + slot * TILE_BYTES, do_tile = lds0 + PAIR_DO + slot * TILE_BYTES;
    // Addresses inside a tile, for this lane: row col at contraction step j (16 bytes at 16 j + 8 half), and the
    // transposing read of d block db.  Steps and blocks within a 256-byte window differ by an XOR of the address (the
    // swizzle is one), the second window and the second 16 rows by an immediate offset.
    const int lane = lane_now(), col = lane & 31, half = lane >> 5;
    const int tr_row = half * 4 + ((lane & 15) >> 2);
    const uint32_t xr = (is_b ? do_tile : q_tile) + (uint32_t)(col * (DW * 2) + ((half ^ tile_swz<DW>(col)) << 4));
    const uint32_t yt = (is_b ? q_tile : do_tile) +
                        (uint32_t)(tr_row * (DW * 2) + (((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ tile_swz<DW>(tr_row)) << 4) + (lane & 1) * 8);
    // operand k: row fragments of the first product, then the transposed fragments of the second
    auto operand = [&](auto kc) {
      constexpr int k = decltype(kc)::value;
      if constexpr (k < KS) {
        return lds_read<u32x4>((xr ^ ((k % 8) << 5)) + (k / 8) * 256);
      } else {
        constexpr int db = (k - KS) % DB, off = (db / 4) * 256 + ((k - KS) / DB) * 16 * DW * 2;
        const u32x2 lo = lds_tr_read((yt ^ ((db % 4) << 6)) + off);
        const u32x2 hi = lds_tr_read((yt ^ ((db % 4) << 6) ^ 32) + off + 8 * DW * 2);  // (eight rows on: the swizzle's other half)
        return u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
    };
#pragma unroll
    for (int i = 0; i < DB; ++i) asm volatile("" : "+a"(acc[i]));
    u32x4 ring[8];
    static_for<AHEAD1>([&](auto kc) { ring[decltype(kc)::value] = operand(kc); });
    f32x16 s;
    static_for<KS>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      if constexpr (k + AHEAD1 < KS + AHEAD_MID) ring[(k + AHEAD1) & 7] = operand(std::integral_constant<int, k + AHEAD1>{});
      if constexpr (k == 0) MmaV<T>::first(s, ring[0], f[0]);
      else MmaV<T>::next(s, ring[k & 7], f[k]);
      __builtin_amdgcn_sched_barrier(0);
    });
    uint32_t pk[8];
    const int ln = lane_now(), half_m = ln >> 5, key_m = kw0 + (ln & 31);
    const uint32_t stats = lds0 + PAIR_STATS + slot * 512 + (is_b ? 256 : 0) + half_m * 16;  // (this lane's rows: A lse, B delta)
    const f32x4 row_stats = lds_read<f32x4>(stats);
    mfma_to_valu_gap(s);
    const uint32_t p_at = lds0 + PAIR_P + wave * 4096 + parity * 2048 + ln * 16;  // the pair's 2 x 2 KB
    if (!is_b) {
      uint32_t pf[MODE == 0 ? 1 : 8];  // the probabilities times the functors' derivative
      float f_w = 1.f;
      if constexpr (MODE == 2) {
        // every score through the functors: s = mod(scale * s) / scale (one loop per functor behind one test each)
        const int hq = hk * rep + hg, kc = max(min(key_m, p.S - 1), 0);
        float f_kb = 0.f;
        if (p.sm.key_weight) f_w = p.sm.key_weight[(int64_t)hq * p.S + kc];
        if (p.sm.key_bias) f_kb = p.sm.key_bias[(int64_t)hq * p.S + kc];
        const float sw = p.scale * f_w;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = fmaf(s[r], sw, f_kb);
        if (p.sm.alibi) {
          const float slope = p.sm.alibi[hq], base = (float)(key_m - q0 - half_m * 4);
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] = fmaf(slope, base - (float)((r >> 2) * 8 + (r & 3)), s[r]);
        }
        if (p.sm.softcap > 0.f) {
          const float cap = p.sm.softcap, inv_cap = 1.f / p.sm.softcap;
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] = cap * tanh_fast(s[r] * inv_cap);
        }
        if (p.sm.doc_q && p.sm.doc_k) {
          const int32_t mine = p.sm.doc_k[(int64_t)b * p.S + kc];
          const int32_t* dq = p.sm.doc_q + (int64_t)b * p.L;
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] = dq[min(q0 + (r >> 2) * 8 + half_m * 4 + (r & 3), p.L - 1)] != mine ? -INFINITY : s[r];
        }
        const float inv_scale = 1.f / p.scale;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] *= inv_scale;
      }
      // (rows of this item and keys of this wavefront that all take part, as in most items, cost no test per score)
      auto probabilities = [&](auto edge_c) {
        constexpr bool EDGE = decltype(edge_c)::value;
        // the first row of the item that sees this lane's key, and the first one that does not any more
        const int lo = p.causal ? key_m - q0 - half_m * 4 : 0;
        const int hi = (p.window > 0 && key_m >= p.sink_keys ? min(key_m + p.window, p.L) : p.L) - q0 - half_m * 4;
        f32x4 l_next = row_stats;
        const float icap = (MODE == 2 && p.sm.softcap > 0.f) ? p.scale / p.sm.softcap : 0.f;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const f32x4 l4 = l_next;  // (requested a group ahead: the groups are fenced off from each other)
          if (r4 < 3) l_next = lds_read<f32x4>(stats + r4 * 32 + 32);
          float pr[4], pd[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = r4 * 4 + e, row = r4 * 8 + e;
            float x, d = 1.f;
            if constexpr (MODE == 1) {
              const float rc = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[r] * cap_k));
              const float th = fmaf(rc, -2.f, 1.f);
              x = fmaf(th, cap_l, -l4[e]);
              d = fmaf(-th, th, 1.f);
              if (EDGE) d = fminf(d, 1.f);  // (a dropped score may be anything, a NaN too: finite again)
            } else {
              x = fmaf(s[r], c, -l4[e]);
              if constexpr (MODE == 2) {
                const float th = s[r] * icap;
                d = fmaf(-th, th, 1.f) * f_w;
              }
            }
            // (masked before the exponential: a select around it is compiled into a branch per element)
            if constexpr (EDGE) x = ((row < lo) | (row >= hi)) ? -INFINITY : x;
            pr[e] = __builtin_amdgcn_exp2f(x);
            if constexpr (MODE == 2) pd[e] = pr[e] == 0.f ? 0.f : pr[e] * d;
            else pd[e] = pr[e] * d;
          }
          pk[r4 * 2] = Mma<T>::pack(pr[0], pr[1]), pk[r4 * 2 + 1] = Mma<T>::pack(pr[2], pr[3]);
          if constexpr (MODE != 0) pf[r4 * 2] = Mma<T>::pack(pd[0], pd[1]), pf[r4 * 2 + 1] = Mma<T>::pack(pd[2], pd[3]);
          if (r4 & 1) {
            typedef u32x4 __attribute__((address_space(3)))* lds_u32x4;
            const int g = r4 * 2 - 2;
            if constexpr (MODE == 0) *(lds_u32x4)(p_at + (r4 >> 1) * 1024) = u32x4{pk[g], pk[g + 1], pk[g + 2], pk[g + 3]};
            else *(lds_u32x4)(p_at + (r4 >> 1) * 1024) = u32x4{pf[g], pf[g + 1], pf[g + 2], pf[g + 3]};
          }
          __builtin_amdgcn_sched_barrier(0);  // (group by group: all at once they need more registers than there are)
        }
      };
      const bool edge = MODE == 2 || (p.causal && q0 < kw0 + 31) || (p.window > 0 && q0 + 31 - kw0 >= p.window) || q0 + BT > p.L;
      if (edge) probabilities(std::true_type{});
      else probabilities(std::false_type{});
    } else {
      const u32x4 w0 = lds_read<u32x4>(p_at), w1 = lds_read<u32x4>(p_at + 1024);
      f32x4 d_next = row_stats;
      const uint32_t w[8] = {w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const f32x4 d4 = d_next;
        if (r4 < 3) d_next = lds_read<f32x4>(stats + r4 * 32 + 32);
        float ds[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) ds[e] = Mma<T>::unpack(w[r4 * 2 + (e >> 1)], e & 1) * (s[r4 * 4 + e] - d4[e]);
        pk[r4 * 2] = Mma<T>::pack(ds[0], ds[1]), pk[r4 * 2 + 1] = Mma<T>::pack(ds[2], ds[3]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    static_for<AHEAD2 - AHEAD_MID>([&](auto kc) {
      constexpr int k = KS + AHEAD_MID + decltype(kc)::value;
      ring[k & 7] = operand(std::integral_constant<int, k>{});
    });
    static_for<2 * DB>([&](auto ic) {
      constexpr int i = decltype(ic)::value, k = KS + i, r0 = (i / DB) * 4;
      if constexpr (k + AHEAD2 < NOPS) ring[(k + AHEAD2) & 7] = operand(std::integral_constant<int, k + AHEAD2>{});
      if constexpr (i == 4) {
        if (next_slot >= 0) request(next_slot);
      }
      acc[i % DB] = Mma<T>::run(ring[k & 7], u32x4{pk[r0], pk[r0 + 1], pk[r0 + 2], pk[r0 + 3]}, acc[i % DB]);
      __builtin_amdgcn_sched_barrier(0);
    });
#pragma unroll
    for (int i = 0; i < DB; ++i) asm volatile("" : "+a"(acc[i]));
  };

  int cq = qs_hi - 1, ch = 0;  // this wavefront's next item
  // (A goes first where both want to issue: its softmax then runs under B's products; causal, no cap: 688 -> 655 us)
  if (!is_b) __builtin_amdgcn_s_setprio(1);
  if (n_items > 0) {
    request(0);
    if (n_items > 1) {
      request(1);
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    // (the fragments are awaited here: left pending, their first use inside the loop would be a wait for every
    // outstanding load there, the tiles in flight included)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(f[ks]));
    __syncthreads();
    for (int i = 0; i <= n_items; ++i) {
      // (requested between the matrix ops of the second product where there is one)
      int next_slot = i + 2 < n_items ? (i + 2) & (SLOTS - 1) : -1;
      const int it = is_b ? i - 1 : i;
      if (it >= 0 && it < n_items) {
        const int q0 = cq * BT;
        // (uniform for the pair: rows above the diagonal, no live key, every row past the window of every key of the pair)
        const bool past_window = p.window > 0 && q0 - (kw0 + 31) >= p.window && kw0 >= p.sink_keys;
        if (!((p.causal && q0 + BT - 1 < kw0) || kw0 >= S || past_window)) compute(it & (SLOTS - 1), it & 1, cq, ch, next_slot), next_slot = -1;
        advance(cq, ch);
      }
      if (next_slot >= 0) request(next_slot);
      if (i < n_items) {  // item i + 1 and A's probabilities of item i are everybody's from here on
        if (i + 2 < n_items) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
      }
    }
  }
  // Results leave through buffer stores whose offset is pushed past the buffer's end where a lane has nothing to
  // write (a key past S, columns past the real width): the hardware drops such a store.  (Every column of an
  // accumulator is one key's own: a key past the batch's count, whose column holds whatever its stand-in row gave, is zeroed here.)
  constexpr uint32_t kDrop = 0xfffffff0u;
  const int half = lane >> 5;
  const bool in = key < p.S, live = key < S;
  const int width = is_b ? p.d_real : p.dv_real;
  if (p.parts > 1) {  // float32 rows for bwd_dkdv_merge_kernel, which also multiplies dK by the scale
    const int64_t row0 = (((int64_t)part * p.B + b) * p.Hkv + hk) * p.S;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr((char*)((is_b ? p.part_dk : p.part_dv) + row0 * width)), 0,
                                                                       __builtin_amdgcn_readfirstlane((int)((int64_t)p.S * width * 4)), 0x00020000);
    const uint32_t o = (uint32_t)((key * width + half * 4) * 4);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = db * 32 + g * 8;
        f32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = live ? acc[db][g * 4 + e] : 0.f;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, w), rs, (in && d + half * 4 < width) ? o + d * 4 : kDrop, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);  // (block by block: left alone, every accumulator is read out before the first store)
    }
  } else {
    const int64_t sl = is_b ? p.gk_sl : p.gv_sl;
    uint16_t* const base = is_b ? (uint16_t*)p.gk + b * p.gk_sb + hk * p.gk_sh : (uint16_t*)p.gv + b * p.gv_sb + hk * p.gv_sh;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        uniform_ptr((char*)base), 0, __builtin_amdgcn_readfirstlane((int)(((int64_t)(p.S - 1) * sl + width) * 2)), 0x00020000);
    const uint32_t o = (uint32_t)(((int64_t)key * sl + half * 4) * 2);
    const float scale = is_b ? p.scale : 1.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = db * 32 + g * 8;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = live ? acc[db][g * 4 + e] * scale : 0.f;
        const u32x2 w = {Mma<T>::pack(v[0], v[1]), Mma<T>::pack(v[2], v[3])};
        __builtin_amdgcn_raw_buffer_store_b64(w, rs, (in && d + half * 4 < width) ? o + d * 2 : kDrop, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <typename T, int MODE>
int launch_mode(const BwdM& g, hipStream_t s) {
  static LdsOnce once;
  const hipError_t attr = reserve_lds(once, (const void*)bwd_wide_pair_kernel<T, MODE>, PAIR_LDS);
  if (attr != hipSuccess) {
    set_error("SDPA: cannot reserve %d bytes of LDS for bwd_wide_pair_kernel: %s", PAIR_LDS, hipGetErrorString(attr));
    return MI355_SDPA_ERR_LAUNCH;
  }
  const int64_t blocks = (int64_t)g.B * g.Hkv * g.n_kt * g.parts;
  hipLaunchKernelGGL((bwd_wide_pair_kernel<T, MODE>), dim3((unsigned)blocks), dim3(512), PAIR_LDS, s, g);
  return check_launch("bwd_wide_pair_kernel");
}
template <typename T>
int launch_t(const BwdM& g, hipStream_t s) {
  if (!g.sm.any) return launch_mode<T, 0>(g, s);
  const bool cap_only = g.sm.softcap > 0.f && !g.sm.alibi && !g.sm.key_bias && !g.sm.key_weight && !g.sm.doc_q;
  return cap_only ? launch_mode<T, 1>(g, s) : launch_mode<T, 2>(g, s);
}

}  // namespace

int launch_bwd_wide_pair(const BwdM& g, int dtype, hipStream_t s) {
  return dtype == MI355_SDPA_BF16 ? launch_t<bf16_t>(g, s) : launch_t<f16_t>(g, s);
}

}  // namespace mi355
