// Flash-attention backward for gfx950 at head dims up to 64, bf16/f16: plain and causal calls, per-batch
// key counts, dropout.  (Calls with a bias, a window or a score functor: bwd_dq_w32.hip, bwd_dkdv_w32.hip, and
// dK/dV of causal calls of grouped heads with too few workgroups here: bwd_dkdv_w32.hip, see w32_dkdv.)
//
//   bwd_d64_dq_kernel     128 query rows per workgroup (4 wavefronts x 32), 64-key tiles:
//                           S^T = K Q^T, dP^T = V dO^T, dS^T = P^T (dP^T - delta), dQ^T += K^T dS^T
//                         it also forms delta = rowsum(dO * O) and leaves it, with the log2-domain
//                         log-sum-exp, in the workspace for the second kernel
//                         (with few workgroups both run in one launch, behind one that forms these: see together)
//   bwd_d64_dkdv_kernel   128 keys per workgroup (4 wavefronts x 32 keys), 64-row query tiles of every head
//                         of the group (the GQA sum of decompositions.py:2595-2598 happens in registers):
//                           S = Q K^T, dP = dO V^T, dV^T += dO^T P, dK^T += Q^T dS
//
// At this width a 32 x 32 score block is 16 (dK/dV) or 12 (dQ) matrix ops of 32 cycles against about a
// hundred vector instructions, and the calls are short (heads of 64 go with sequences of a few hundred
// to two thousand): what bounds them is neither pipe but the chain score - probability - dS - product of
// one wavefront, the instructions it issues one after the other and the waits around them.  The dQ kernel keeps its
// registers to a third of the file (168), and the chain of one wavefront runs under the other two's of its SIMD; nothing
// in it is pipelined by hand (in the two phases of the dK/dV kernel it measured the same, 986 / 1004 us for the backward of
// B=4, 32 heads, S=4096 causal, within 1 % elsewhere, with dropout 2 % slower).  The dK/dV kernel, which holds
// 128 registers of operands and accumulators, works on two blocks at a time instead (see dkdv_body), but for calls of
// just over two workgroups per compute unit and few items, which take it block by block in three (see three_per_cu).
// A wavefront keeps all four products of its keys (at head dim 128 they do not fit and are split over two
// wavefronts that exchange P through LDS).
//
// Tiles go from global memory straight into LDS (row-major, XOR swizzled, see tile_swz), three buffers,
// two tiles ahead, one barrier per tile; transposed operands come out of the transposing LDS read.
//
// Dropout: the keep-mask is bytes.  The dQ kernel reads them (16 of a row per lane, the halves of a wavefront
// exchange what the other one needs) and leaves one BIT per score behind for the dK/dV kernel, whose lanes
// are keys: read as bytes there the mask is a load per score.  32 keys per word, four words per query row and
// block of 128 keys, laid out [batch][kv head][block][head of the group][row]: a dK/dV workgroup reads one run of
// them, at 32-bit offsets however many there are in all.  (Rows of bits over all keys: a load's 64 lanes touch as
// many lines, backward of B=4, 16 heads, S=2048 causal 217 us against 189, of B=2, 16/4 heads, S=4096 688 / 636.)
//
// Math follows torch_neuronx/_sdpa_math.py:98-176: float32 accumulation, rows with lse = -inf give zero
// gradients, scale multiplies dQ and dK once at the end.
#include <algorithm>
#include <type_traits>

#include "bwd_mfma.h"

namespace mi355 {
namespace {

constexpr int D = 64, KS = D / 16, DB = D / 32, CH = D / 8;
constexpr int BQ = 64;            // rows of a staged tile (query rows or keys)
constexpr int TILE = BQ * D;      // its elements
constexpr int TILE_BYTES = TILE * 2;
constexpr int NCH = BQ * CH / 256;  // 16-byte chunks of a tile per thread

typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 tr_read(const uint16_t* ptr) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(ptr));
  return __builtin_bit_cast(u32x2, v);
}

// element offsets of the LDS reads inside a swizzled tile (see bwd_dkdv_w32.hip for the lane layouts)
struct TileReads {
  int tr_off[2][DB], row_off[KS];
  __device__ __forceinline__ void init(int lane) {
    const int col = lane & 31, half = lane >> 5, jj = lane & 15, g = lane >> 4;
#pragma unroll
    for (int sec = 0; sec < 2; ++sec)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const int row = 8 * sec + (g >> 1) * 4 + (jj >> 2), d = db * 32 + 16 * (g & 1) + 4 * (jj & 3);
        tr_off[sec][db] = row * D + (((d >> 3) ^ tile_swz<D>(row)) << 3) + (d & 7);
      }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) row_off[ks] = col * D + (((2 * ks + half) ^ tile_swz<D>(col)) << 3);
  }
  // rows of 32-row block mb, contraction step ks
  __device__ __forceinline__ u32x4 rows(const uint16_t* tile, int mb, int ks) const { return *(const u32x4*)(tile + row_off[ks] + mb * 32 * D); }
  // columns of d block db over the 16 rows of step st (of the 64 rows)
  __device__ __forceinline__ u32x4 cols(const uint16_t* tile, int st, int db) const {
    const u32x2 lo = tr_read(tile + tr_off[0][db] + st * 16 * D), hi = tr_read(tile + tr_off[1][db] + st * 16 * D);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  }
};

// raw buffer resource, in scalar registers
__device__ __forceinline__ u32x4 descriptor(const void* base, int64_t bytes) {
  const uint64_t a = (uint64_t)base;
  return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}
// global memory straight into LDS, 16 / 4 bytes per lane at consecutive LDS addresses from lds_addr (inline
// assembly: the compiler's own form makes every later LDS read wait for all outstanding loads; m0 holds
// the LDS address, one wait state after it is written)
__device__ __forceinline__ void lds_load16(const u32x4& rsrc, uint32_t voffset, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(voffset), "s"(rsrc) : "memory", "m0");
}
__device__ __forceinline__ void lds_load4(const u32x4& rsrc, uint32_t voffset, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(voffset), "s"(rsrc) : "memory", "m0");
}
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
typedef __attribute__((address_space(3))) unsigned char* lds_bytes;
__device__ __forceinline__ uint32_t lds_address(const void* p) { return (uint32_t)(uintptr_t)(lds_bytes)p; }

// byte offsets of this thread's chunks of a tile whose first row is at offset 0 (a chunk past a narrow
// row's end asks for an offset beyond the buffer and reads as zeros)
__device__ __forceinline__ void chunk_offsets(uint32_t (&off)[NCH], int tid, int64_t row_stride, int width) {
  const int row = tid / CH, ch = (tid % CH) ^ tile_swz<D>(row);  // (row + 32 has the swizzle of row)
#pragma unroll
  for (int n = 0; n < NCH; ++n) off[n] = ch * 8 < width ? (uint32_t)(((row + (256 / CH) * n) * row_stride + ch * 8) * 2) : 0x7ffffff0u;
}

// words of keep bits of one block of 128 keys of one (batch, kv head): four per query row of the group's heads
__host__ __device__ __forceinline__ int64_t block_words(const BwdM& p) { return (int64_t)(p.Hq / p.Hkv) * p.L * 4; }

// this lane's 16 elements of an accumulator packed to the input dtype, in B-operand order
template <typename T>
__device__ __forceinline__ u32x4 pack8(const float* x) {
  return u32x4{Mma<T>::pack(x[0], x[1]), Mma<T>::pack(x[2], x[3]), Mma<T>::pack(x[4], x[5]), Mma<T>::pack(x[6], x[7])};
}

// The 32 rows of a wavefront, a lane holding 4-element pieces of its own row in accumulator layout, leave
// through the wavefront's own 4 KB of LDS as whole rows, 16 bytes per lane (as 8-byte pieces of 32 rows
// per instruction the dK/dV kernel wrote 94 MB to memory for 50 MB of gradients)
template <typename T>
__device__ __forceinline__ void store_rows(const f32x16 (&acc)[DB], float scale, uint16_t* lds, int lane, uint16_t* out, int64_t row_stride, int row0, int n_rows, int dr) {
  const int col = lane & 31, half = lane >> 5;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const u32x2 w = {Mma<T>::pack(acc[db][g * 4] * scale, acc[db][g * 4 + 1] * scale), Mma<T>::pack(acc[db][g * 4 + 2] * scale, acc[db][g * 4 + 3] * scale)};
      *(u32x2*)(lds + col * D + (((db * 4 + g) ^ (col & 7)) << 3) + half * 4) = w;
    }
  const int r = lane >> 3, ch = lane & 7;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const u32x4 w = *(const u32x4*)(lds + (i * 8 + r) * D + ((ch ^ r) << 3));
    if (row0 + i * 8 + r < n_rows && ch * 8 < dr) *(u32x4*)(out + (int64_t)(row0 + i * 8 + r) * row_stride + ch * 8) = w;
  }
}

// (TERMS: leaves delta and the log2-domain log-sum-exp behind)
template <typename T, bool DROP, bool TERMS>
__device__ __forceinline__ void dq_body(const BwdM& p, uint32_t* keep_bits, int bid, int chunk, uint16_t (*k_t)[TILE], uint16_t (*v_t)[TILE]) {
  const int rep = p.Hq / p.Hkv;
  const BlockMap bm = block_map(bid, p.B * p.Hkv, p.n_qt, rep, chunk);
  if (bm.stream >= p.B * p.Hkv) return;  // (their number is no multiple of eight)
  const int qt = p.n_qt - 1 - bm.tile, b = bm.stream / p.Hkv, hk = bm.stream % p.Hkv, h = hk * rep + bm.unit;  // heavy query tiles first
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int q0 = qt * 128, qw0 = q0 + wave * 32, qrow = qw0 + col, qc = min(qrow, p.L - 1);
  const int dr = p.d_real;
  const int S = p.kv_lens ? min(p.S, max(p.kv_lens[b], 0)) : p.S;  // keys of this batch that take part
  int nt = (S + BQ - 1) / BQ;
  if (p.causal) nt = min(nt, (min(q0 + 128, p.L) - 1) / BQ + 1);
  const int lim = p.causal ? min(qrow, S - 1) : S - 1;

  // staging of K and V: the buffers end with the last key row, rows beyond it read as zeros
  const u32x4 k_rsrc = descriptor((const uint16_t*)p.k + b * p.k_sb + hk * p.k_sh, S > 0 ? ((int64_t)(S - 1) * p.k_sl + dr) * 2 : 0);
  const u32x4 v_rsrc = descriptor((const uint16_t*)p.v + b * p.v_sb + hk * p.v_sh, S > 0 ? ((int64_t)(S - 1) * p.v_sl + dr) * 2 : 0);
  uint32_t k_off[NCH], v_off[NCH];
  chunk_offsets(k_off, tid, p.k_sl, dr);
  chunk_offsets(v_off, tid, p.v_sl, dr);
  const uint32_t lds_k = lds_address(k_t) + wave * 1024, lds_v = lds_address(v_t) + wave * 1024;
  auto load_tile = [&](int t, int buf) {
    const uint32_t kb = (uint32_t)(t * BQ * p.k_sl * 2), vb = (uint32_t)(t * BQ * p.v_sl * 2);
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      lds_load16(k_rsrc, k_off[n] >= 0x7ffffff0u ? k_off[n] : k_off[n] + kb, lds_k + (uint32_t)(buf * TILE_BYTES + n * 4096));
      lds_load16(v_rsrc, v_off[n] >= 0x7ffffff0u ? v_off[n] : v_off[n] + vb, lds_v + (uint32_t)(buf * TILE_BYTES + n * 4096));
    }
  };
  // (dropout) keep bytes of this lane's row: keys 16 half .. +15 of each 32-key block of tile t, through a
  // buffer of this wavefront's rows (rows past L: the last one again)
  const int keep_rows = min(32, p.L - qw0), qw0c = min(qw0, p.L - 1);
  const __amdgpu_buffer_rsrc_t keep_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr((const char*)p.keep + (DROP ? (((int64_t)b * p.Hq + h) * p.L + qw0c) * p.keep_ld : 0)), 0,
      __builtin_amdgcn_readfirstlane(DROP ? (int)((int64_t)max(keep_rows, 1) * p.keep_ld) : 0), 0x00020000);
  const uint32_t keep_off = DROP ? (uint32_t)((int64_t)(qc - qw0c) * p.keep_ld + half * 16) : 0u;
  u32x4 kraw[DROP ? 2 : 1];
  auto load_keep = [&](int t) {
    if constexpr (DROP) {
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) kraw[mb] = __builtin_amdgcn_raw_buffer_load_b128(keep_rsrc, keep_off + (uint32_t)(t * BQ + mb * 32), 0, 0);
    }
  };
  auto await_keep = [&]() {  // (awaited here, with the tiles: left to its first use, the wait would cover the next tile's loads)
    if constexpr (DROP) asm volatile("" : "+v"(kraw[0]), "+v"(kraw[1]));
  };

  if (nt > 0) load_tile(0, 0);
  load_keep(0);
  u32x4 qf[KS], dof[KS];
  float lse2, dl;
  {
    const uint16_t* qr = (const uint16_t*)p.q + b * p.q_sb + h * p.q_sh + (int64_t)qc * p.q_sl + half * 8;
    const uint16_t* gr = (const uint16_t*)p.go + b * p.go_sb + h * p.go_sh + (int64_t)qc * p.go_sl + half * 8;
    const uint16_t* orow = (const uint16_t*)p.out + b * p.o_sb + h * p.o_sh + (int64_t)qc * p.o_sl + half * 8;
    const int64_t idx = ((int64_t)b * p.Hq + h) * p.L + qc;
    const float l = p.lse[idx];
    float dsum = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qf[ks] = dof[ks] = u32x4{0u, 0u, 0u, 0u};
      if (half * 8 + ks * 16 < dr) {
        qf[ks] = *(const u32x4*)(qr + ks * 16), dof[ks] = *(const u32x4*)(gr + ks * 16);
        dsum += dot8<T>(dof[ks], *(const u32x4*)(orow + ks * 16));
      }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]), "+v"(dof[ks]));
    dl = dsum + __shfl_xor(dsum, 32, 64);
    // +inf turns exp2(x - lse) into 0 for rows past L and for rows without a live key
    lse2 = (qrow < p.L && l != -INFINITY) ? l * kLog2eF : INFINITY;
    if (TERMS && qrow < p.L && half == 0) p.delta[idx] = dl, p.lse2[idx] = lse2;
  }
  TileReads rd;
  rd.init(lane);
  f32x16 acc[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) zero(acc[i]);
  const float c = p.scale * kLog2eF;
  uint32_t* const bit_row = DROP ? keep_bits + (int64_t)bm.stream * p.n_kt * block_words(p) + ((int64_t)bm.unit * p.L + qc) * 4 : nullptr;

  wait_loads();
  await_keep();
  __syncthreads();
  if (nt > 1) load_tile(1, 1);
  // (the buffer of a tile is a compile-time constant, three copies of the step: with a run-time index every
  // LDS read carries an addition)
  auto step = [&](int t, auto buf_c) {
    constexpr int buf = decltype(buf_c)::value;
    u32x4 kcur[DROP ? 2 : 1];
    if constexpr (DROP) {
      kcur[0] = kraw[0], kcur[1] = kraw[1];
      if (t + 1 < nt) load_keep(t + 1);
    }
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
      const int kv0 = t * BQ + mb * 32;
      // (uniform per wavefront; rows past the last one: backward of B=64, 12 heads, S=197 71.3 -> 69.8 us)
      if (kv0 >= S || qw0 >= p.L || (p.causal && kv0 > qw0 + 31)) continue;
      f32x16 s, dp;
      zero(s), zero(dp);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = Mma<T>::run(rd.rows(k_t[buf], mb, ks), qf[ks], s);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) dp = Mma<T>::run(rd.rows(v_t[buf], mb, ks), dof[ks], dp);
      if (__builtin_expect(kv0 + 31 >= S || (p.causal && kv0 + 31 > qw0), 0)) {
        asm volatile("" : "+v"(s));  // (a block of its own: as selects every block would pay for them)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = kv0 + (r >> 2) * 8 + half * 4 + (r & 3) > lim ? -INFINITY : s[r];
      }
      if constexpr (DROP) {
        // the lane's bytes are keys 16 half .. +15; accumulator group g wants keys 8 g + 4 half .. +3:
        // the halves swap dwords 1 <-> 0 and 3 <-> 2
        uint32_t w[4] = {kcur[mb][0], kcur[mb][1], kcur[mb][2], kcur[mb][3]};
        const auto s0 = __builtin_amdgcn_permlane32_swap(w[0], w[1], false, false), s1 = __builtin_amdgcn_permlane32_swap(w[2], w[3], false, false);
        w[0] = s0[0], w[2] = s0[1], w[1] = s1[0], w[3] = s1[1];
        uint32_t bits = 0u;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
          for (int e = 0; e < 4; ++e) dp[4 * g + e] *= (float)((w[g] >> (8 * e)) & 0xffu);
          bits |= __builtin_amdgcn_udot4(w[g], 0x08040201u, 0u, false) << (8 * g);
        }
        bits <<= 4 * half;
        bits |= __shfl_xor(bits, 32, 64);
        if (qrow < p.L && half == 0) bit_row[(t >> 1) * block_words(p) + (t & 1) * 2 + mb] = bits;
      }
      float ds[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pr = __builtin_amdgcn_exp2f(fmaf(s[r], c, -lse2));
        ds[r] = pr * (DROP ? fmaf(dp[r], p.keep_scale, -dl) : dp[r] - dl);
      }
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const u32x4 bS = pack8<T>(ds + 8 * st);
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] = Mma<T>::run(rd.cols(k_t[buf], 2 * mb + st, db), bS, acc[db]);
      }
    }
    wait_loads();
    await_keep();
    __syncthreads();
    // (the buffer of tile t - 1: its last readers passed the barrier above)
    if (t + 2 < nt) load_tile(t + 2, (buf + 2) % 3);
  };
  for (int t = 0;;) {
    if (t >= nt) break;
    step(t, std::integral_constant<int, 0>{});
    if (++t >= nt) break;
    step(t, std::integral_constant<int, 1>{});
    if (++t >= nt) break;
    step(t, std::integral_constant<int, 2>{});
    ++t;
  }
  store_rows<T>(acc, p.scale, &k_t[0][0] + wave * 32 * D, lane, (uint16_t*)p.gq + b * p.gq_sb + h * p.gq_sh, p.gq_sl, qw0, p.L, dr);
}

template <typename T, bool DROP>
__global__ __launch_bounds__(256, 3) void bwd_d64_dq_kernel(BwdM p, uint32_t* keep_bits, int chunk) {
  __shared__ __attribute__((aligned(16))) uint16_t k_t[3][TILE];
  __shared__ __attribute__((aligned(16))) uint16_t v_t[3][TILE];
  dq_body<T, DROP, true>(p, keep_bits, blockIdx.x, chunk, k_t, v_t);
}

template <bool DROP>
using KeepTile = uint32_t[DROP ? 4 : 1][BQ];  // [wavefront's 32 keys][row]
// AHEAD: the items whose blocks are all live for a wavefront in two phases, one block ahead; without it every item block by block
template <typename T, bool DROP, bool AHEAD>
__device__ __forceinline__ void dkdv_body(const BwdM& p, const uint32_t* keep_bits, int bid, int chunk, uint16_t (*q_t)[TILE], uint16_t (*do_t)[TILE],
                                          float (*lse_s)[BQ], float (*dl_s)[BQ], KeepTile<DROP>* bit_s) {
  const int streams = p.B * p.Hkv;
  // (the launch order and the split of a key block's items over workgroups: see bwd_dkdv_w32.hip)
  int kt, st, ph = 0, pq = 0;
  if (p.parts > 1) {
    const int vstreams = streams * p.parts_h;
    const int v = bid % vstreams, rest = bid / vstreams;
    kt = rest % p.n_kt, pq = rest / p.n_kt;
    st = v / p.parts_h, ph = v % p.parts_h;
  } else {
    const BlockMap bm = block_map(bid, streams, p.n_kt, 1, chunk);
    kt = bm.tile, st = bm.stream;  // low key tiles see the most queries under a causal mask: first
    if (st >= streams) return;
  }
  const int b = st / p.Hkv, hk = st % p.Hkv;
  const int rep_all = p.Hq / p.Hkv, rep = p.parts > 1 ? rep_all / p.parts_h : rep_all, h0 = hk * rep_all + ph * rep;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int k0 = kt * 128, kw0 = k0 + wave * 32, key = kw0 + col;
  const int dr = p.d_real;
  const int S = p.kv_lens ? min(p.S, max(p.kv_lens[b], 0)) : p.S;
  const int nqs = (p.L + BQ - 1) / BQ, qs_begin = p.causal ? min(k0 / BQ, nqs) : 0;
  int n_items = k0 >= S ? 0 : rep * (nqs - qs_begin);  // no live key in this block: zeros
  int it0 = 0;
  if (p.parts > 1) {
    it0 = pq * p.chunk_items;
    n_items = max(min(n_items - it0, p.chunk_items), 0);
    if (n_items == 0 && pq > 0) return;  // (bwd_dkdv_merge_kernel counts the filled shares in the same way)
  }
  // items: query tile by query tile from the last one down, the group's heads inside.  Where the next item to fetch lies:
  // byte offsets that follow from item to item by one addition each (worked out from an item's number they are a hundred
  // scalar instructions per item, which the wavefronts issue one after the other like any others)
  const int t0 = nqs - 1 - it0 / rep, hl0 = it0 % rep;
  struct {
    int hl;
    uint32_t q, go, bit;
    int64_t stat;
    uint32_t q_bytes, go_bytes, rows4;  // (the buffers end with the head's last row)
  } at;
  const uint32_t q_head = (uint32_t)(p.q_sh * 2), go_head = (uint32_t)(p.go_sh * 2), bit_head = (uint32_t)p.L * 16;
  const int64_t st_head = (int64_t)p.L * 4;
  const uint32_t q_tile = (uint32_t)(p.q_sl * BQ * 2), go_tile = (uint32_t)(p.go_sl * BQ * 2);
  {
    const int rows = min(p.L - t0 * BQ, BQ);
    at.hl = hl0;
    at.q = hl0 * q_head + t0 * q_tile, at.go = hl0 * go_head + t0 * go_tile;
    at.stat = hl0 * st_head + t0 * (BQ * 4), at.bit = (ph * rep + hl0) * bit_head + t0 * (BQ * 16);
    at.q_bytes = (uint32_t)((rows - 1) * p.q_sl + dr) * 2, at.go_bytes = (uint32_t)((rows - 1) * p.go_sl + dr) * 2, at.rows4 = rows * 4;
  }
  const u32x4 bit_rsrc = descriptor(DROP ? keep_bits + ((int64_t)st * p.n_kt + kt) * block_words(p) : nullptr, DROP ? block_words(p) * 4 : 0);
  uint32_t q_off[NCH], go_off[NCH];
  chunk_offsets(q_off, tid, p.q_sl, dr);
  chunk_offsets(go_off, tid, p.go_sl, dr);
  const uint32_t lds_q = lds_address(q_t) + wave * 1024, lds_do = lds_address(do_t) + wave * 1024;
  const char* const q_base = (const char*)((const uint16_t*)p.q + b * p.q_sb + h0 * p.q_sh);
  const char* const go_base = (const char*)((const uint16_t*)p.go + b * p.go_sb + h0 * p.go_sh);
  const char* const stat_base = (const char*)((wave == 0 ? p.lse2 : p.delta) + ((int64_t)b * p.Hq + h0) * p.L);  // (wavefronts 0 and 1)
  const uint32_t lds_stat = wave == 0 ? lds_address(lse_s) : lds_address(dl_s);
  // (the buffers of an item are its tile's own and end with the head's last row: a row past L must not be another
  // head's, whose NaN would survive the zero probabilities)
  auto load_item = [&](int buf) {
    const u32x4 q_rsrc = descriptor(q_base + at.q, at.q_bytes), go_rsrc = descriptor(go_base + at.go, at.go_bytes);
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      lds_load16(q_rsrc, q_off[n], lds_q + (uint32_t)(buf * TILE_BYTES + n * 4096));
      lds_load16(go_rsrc, go_off[n], lds_do + (uint32_t)(buf * TILE_BYTES + n * 4096));
    }
    if (wave < 2) lds_load4(descriptor(stat_base + at.stat, at.rows4), lane * 4, lds_stat + buf * (BQ * 4));  // log-sum-exps, deltas
    if constexpr (DROP) lds_load4(bit_rsrc, at.bit + lane * 16 + wave * 4, lds_address(bit_s) + (uint32_t)((buf * 4 + wave) * (BQ * 4)));
    const bool wrap = ++at.hl == rep;
    at.q += q_head, at.go += go_head, at.stat += st_head, at.bit += bit_head;
    if (wrap) {
      at.hl = 0;
      at.q -= rep * q_head + q_tile, at.go -= rep * go_head + go_tile, at.stat -= rep * st_head + BQ * 4, at.bit -= rep * bit_head + BQ * 16;
      at.q_bytes = (uint32_t)((BQ - 1) * p.q_sl + dr) * 2, at.go_bytes = (uint32_t)((BQ - 1) * p.go_sl + dr) * 2, at.rows4 = BQ * 4;
    }
  };
  // rows past L: no probability whatever stands there (wavefront 0, which loaded the values it writes over and has
  // waited for them)
  auto finish_item = [&](int q0, int buf) {
    if (q0 + BQ > p.L && tid < BQ && q0 + tid >= p.L) lse_s[buf][tid] = INFINITY;
  };
  if (n_items > 0) load_item(0);
  u32x4 kf[KS], vf[KS];  // this lane's key as B operand
  {
    const int kc = max(min(key, S - 1), 0);  // (a live row: rows past the batch's keys may hold anything)
    const uint16_t* kr = (const uint16_t*)p.k + b * p.k_sb + hk * p.k_sh + (int64_t)kc * p.k_sl + half * 8;
    const uint16_t* vr = (const uint16_t*)p.v + b * p.v_sb + hk * p.v_sh + (int64_t)kc * p.v_sl + half * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kf[ks] = vf[ks] = u32x4{0u, 0u, 0u, 0u};
      if (half * 8 + ks * 16 < dr) kf[ks] = *(const u32x4*)(kr + ks * 16), vf[ks] = *(const u32x4*)(vr + ks * 16);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(kf[ks]), "+v"(vf[ks]));
  }
  TileReads rd;
  rd.init(lane);
  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) zero(dk[i]), zero(dv[i]);
  const float c = p.scale * kLog2eF;
  int q0 = t0 * BQ, hl = hl0, buf = 0, before = 0, next = 1;  // the item that is computed, and the buffers of it and its neighbours
  // item `it + 1` is there for everyone, and the buffer of item it - 1, which everyone is done with, is filled again
  auto publish = [&](int it) {
    wait_loads();
    if (it + 1 < n_items) finish_item(hl + 1 == rep ? q0 - BQ : q0, next);
    __syncthreads();
    if (it + 2 < n_items) load_item(next == 2 ? 0 : next + 1);
  };
  auto advance = [&]() {
    if (++hl == rep) hl = 0, q0 -= BQ;
    before = buf, buf = next, next = next == 2 ? 0 : next + 1;
  };
  auto mask = [&](f32x16& s, int qb) {  // scores of a block of 32 rows that not every key of the wavefront takes part in
    if (__builtin_expect((p.causal && qb < kw0 + 31) || kw0 + 31 >= S, 0)) {
      // this lane's key takes no part in the block's first `dead` rows (one register, not one per row kept across the loop)
      int dead = (key >= S ? 32 : p.causal ? key - qb : 0) - half * 4;
      asm volatile("" : "+v"(s), "+v"(dead));
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = (r >> 2) * 8 + (r & 3) < dead ? -INFINITY : s[r];
    }
  };
  // items with both blocks of 32 rows live for this wavefront (under a causal mask the others come last)
  int n_main = AHEAD && kw0 < S ? n_items : 0;
  if (p.causal) n_main = max(min(n_main, rep * (nqs - (kw0 + 32) / BQ) - it0), 0);
  if (n_items > 0) {
    wait_loads();
    finish_item(q0, 0);
    __syncthreads();
    if (n_items > 1) load_item(1);
  }

  // A block of 32 query rows in two phases of eight slots, a matrix op and the vector work on two scores each: P, under the
  // products dP of this block and dK of the block before; then dS, under the scores of the next block and dV of this one.
  // So every product has vector work of its own wavefront to run under, and one register tile each of scores and dP is
  // enough.  Operands are requested four ops ahead of their use, statistics of four rows four slots ahead, across the phases.
  int it = 0;
  if (AHEAD && n_main > 0) {
    f32x16 s, dp;
    uint32_t pk[8], bs[8];  // P and dS in pairs
    u32x4 ring[4];
    f32x4 rs[2];
    u32x4 wd[DROP ? 2 : 1];
    const lds_bytes q_l = (lds_bytes)&q_t[0][0], do_l = (lds_bytes)&do_t[0][0], lse_l = (lds_bytes)&lse_s[0][0] + half * 16, dl_l = (lds_bytes)&dl_s[0][0] + half * 16;
    const lds_bytes bit_l = DROP ? (lds_bytes)&bit_s[0][0][0] + wave * (BQ * 4) + half * 16 : nullptr;
    uint32_t row_a[KS], col_a[2][DB];  // byte offsets in a tile
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) row_a[ks] = rd.row_off[ks] * 2;
#pragma unroll
    for (int i = 0; i < 2 * DB; ++i) col_a[i >> 1][i & 1] = rd.tr_off[i >> 1][i & 1] * 2;
    auto rows = [&](lds_bytes tiles, int b, int mb, int ks) { return *(const __attribute__((address_space(3))) u32x4*)(tiles + (row_a[ks] + b * TILE_BYTES) + mb * 32 * D * 2); };
    auto cols = [&](lds_bytes tiles, int b, int mb, int i) {
      typedef s16x4 __attribute__((address_space(3)))* ptr;
      const int st = 2 * mb + (i >> 1), db = i & 1;
      const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(tiles + (col_a[0][db] + b * TILE_BYTES) + st * 16 * D * 2)));
      const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(tiles + (col_a[1][db] + b * TILE_BYTES) + st * 16 * D * 2)));
      return u32x4{lo[0], lo[1], hi[0], hi[1]};
    };
    auto stat_of = [&](lds_bytes rows_l, int b, int mb, int g) { return *(const __attribute__((address_space(3))) f32x4*)(rows_l + b * (BQ * 4) + (mb * 32 + g * 8) * 4); };
    auto words_of = [&](int b, int mb, int g) { return *(const __attribute__((address_space(3))) u32x4*)(bit_l + b * (BQ * 16) + (mb * 32 + g * 8) * 4); };
    auto add_rows = [&](f32x16 (&acc)[DB], const uint32_t (&w)[8], const u32x4& a, int i) {  // i = 2 * 16-row step + column block
      const int sg = i >> 1;
      acc[i & 1] = Mma<T>::run(a, u32x4{w[4 * sg], w[4 * sg + 1], w[4 * sg + 2], w[4 * sg + 3]}, acc[i & 1]);
    };
    auto phase_p = [&](int mb, int b_before, int b_next) {
      zero(dp);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const u32x4 a = ring[i % 4];
        if (i < KS) dp = Mma<T>::run(a, vf[i], dp);
        else add_rows(dk, bs, a, i - KS);
        ring[i % 4] = i < KS ? cols(q_l, b_before, mb ^ 1, i) : rows(q_l, b_next, mb ^ 1, i - KS);
        const int e = (2 * i) & 3, g = i >> 1;
        const f32x4& l4 = rs[g & 1];
        pk[i] = Mma<T>::pack(__builtin_amdgcn_exp2f(fmaf(s[2 * i], c, -l4[e])), __builtin_amdgcn_exp2f(fmaf(s[2 * i + 1], c, -l4[e + 1])));
        asm volatile("" : "+v"(pk[i]));  // (here: the compiler would move it behind the next branch)
        if (i & 1) rs[g & 1] = g < 2 ? stat_of(lse_l, buf, mb, g + 2) : stat_of(dl_l, buf, mb, g - 2);
        if constexpr (DROP) {
          if (i >= 6) wd[i & 1] = words_of(buf, mb, i - 6);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // dS is formed from P as the matrix pipe gets it, rounded to the input dtype (as in the kernels that
    // exchange P through LDS: a mask given as a tensor runs there, and the same mask as a flag here)
    auto phase_ds = [&](int mb, int b_next) {
      uint32_t pm[DROP ? 8 : 1];
      zero(s);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const u32x4 a = ring[i % 4];
        if (i < KS) s = Mma<T>::run(a, kf[i], s);
        else if constexpr (DROP) add_rows(dv, pm, a, i - KS);
        else add_rows(dv, pk, a, i - KS);
        ring[i % 4] = i < KS ? cols(do_l, buf, mb, i) : rows(do_l, b_next, mb ^ 1, i - KS);
        if constexpr (DROP) {
          // the first four slots: this key's bit of each row's word, as a mask of all ones or zeros, on dP and on the P that dV gets
          if (i < 4) {
            const u32x4 w4 = wd[i & 1];
#pragma unroll
            for (int j = 2 * i; j < 2 * i + 2; ++j) {
              const int e = (2 * j) & 3;
              const uint32_t m0 = (uint32_t)__builtin_amdgcn_sbfe((int)w4[e], (uint32_t)col, 1u), m1 = (uint32_t)__builtin_amdgcn_sbfe((int)w4[e + 1], (uint32_t)col, 1u);
              const float dp0 = dp[2 * j], dp1 = dp[2 * j + 1];  // (copied out: a bit cast of a vector element reads element 0)
              dp[2 * j] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, dp0) & m0);
              dp[2 * j + 1] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, dp1) & m1);
              pm[j] = pk[j] & __builtin_amdgcn_perm(m1, m0, 0x05040100u);
            }
            if (i < 2) wd[i & 1] = words_of(buf, mb, i + 2);
          } else {
            const int g = i - 4;
            const f32x4 d4 = rs[g & 1];
#pragma unroll
            for (int j = 2 * g; j < 2 * g + 2; ++j) {
              const int e = (2 * j) & 3;
              bs[j] = Mma<T>::pack(Mma<T>::unpack(pk[j], 0) * fmaf(dp[2 * j], p.keep_scale, -d4[e]), Mma<T>::unpack(pk[j], 1) * fmaf(dp[2 * j + 1], p.keep_scale, -d4[e + 1]));
              asm volatile("" : "+v"(bs[j]));
            }
            rs[g & 1] = g < 2 ? stat_of(dl_l, buf, mb, g + 2) : stat_of(lse_l, b_next, mb ^ 1, g - 2);
          }
        } else {
          const int e = (2 * i) & 3, g = i >> 1;
          const f32x4& d4 = rs[g & 1];
          bs[i] = Mma<T>::pack(Mma<T>::unpack(pk[i], 0) * (dp[2 * i] - d4[e]), Mma<T>::unpack(pk[i], 1) * (dp[2 * i + 1] - d4[e + 1]));
          asm volatile("" : "+v"(bs[i]));
          if (i & 1) rs[g & 1] = g < 2 ? stat_of(dl_l, buf, mb, g + 2) : stat_of(lse_l, b_next, mb ^ 1, g - 2);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // (no block in front of the first one: the dK that its first phase adds is of zero dS, with the other rows of the same
    // tile, which every key of the wavefront sees anyway)
#pragma unroll
    for (int i = 0; i < 8; ++i) bs[i] = 0u;
    zero(s);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = Mma<T>::run(rows(q_l, 0, 0, ks), kf[ks], s);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ring[ks] = rows(do_l, 0, 0, ks);
    rs[0] = stat_of(lse_l, 0, 0, 0), rs[1] = stat_of(lse_l, 0, 0, 1);
#pragma nounroll
    do {
      mask(s, q0);
      phase_p(0, before, buf);
      phase_ds(0, buf);
      publish(it);
      mask(s, q0 + 32);
      phase_p(1, buf, next);
      phase_ds(1, next);  // (behind the last item the scores of a tile that nobody asked for, and nobody uses)
      advance();
    } while (++it < n_main);
#pragma unroll
    for (int i = 0; i < 4; ++i) add_rows(dk, bs, cols(q_l, before, 1, i), i);
  }
  // the rest, block by block: nothing of a block that no key of the wavefront sees is computed, whatever its rows hold
#pragma nounroll
  for (; it < n_items; ++it) {
    publish(it);
    for (int mb = 0; mb < 2; ++mb) {
      const int qb = q0 + mb * 32;
      if (kw0 >= S || (p.causal && qb + 31 < kw0)) continue;  // (uniform per wavefront)
      const uint16_t *const qt = q_t[buf] + mb * 32 * D, *const dot = do_t[buf] + mb * 32 * D;
      f32x16 s, dp;
      zero(s), zero(dp);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = Mma<T>::run(rd.rows(qt, 0, ks), kf[ks], s);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) dp = Mma<T>::run(rd.rows(dot, 0, ks), vf[ks], dp);
      mask(s, qb);
      uint32_t pm[8], ds[8];
      f32x4 l4, d4;  // (with dropout four rows' at a time; without, in the kernel of 168 registers, that sends some to scratch)
      u32x4 w4;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int e = (2 * i) & 3, r0 = mb * 32 + (i >> 1) * 8 + half * 4 + e;  // the rows of scores 2 i and 2 i + 1
        if constexpr (DROP) {
          if (e == 0) l4 = *(const f32x4*)&lse_s[buf][r0], d4 = *(const f32x4*)&dl_s[buf][r0], w4 = *(const u32x4*)&bit_s[buf][wave][r0];
        }
        const float l0 = DROP ? l4[e] : lse_s[buf][r0], l1 = DROP ? l4[e + 1] : lse_s[buf][r0 + 1];
        const float d0 = DROP ? d4[e] : dl_s[buf][r0], d1 = DROP ? d4[e + 1] : dl_s[buf][r0 + 1];
        const uint32_t pk = Mma<T>::pack(__builtin_amdgcn_exp2f(fmaf(s[2 * i], c, -l0)), __builtin_amdgcn_exp2f(fmaf(s[2 * i + 1], c, -l1)));
        float g0 = dp[2 * i], g1 = dp[2 * i + 1];
        pm[i] = pk;
        if constexpr (DROP) {
          const uint32_t m0 = (uint32_t)__builtin_amdgcn_sbfe((int)w4[e], (uint32_t)col, 1u), m1 = (uint32_t)__builtin_amdgcn_sbfe((int)w4[e + 1], (uint32_t)col, 1u);
          pm[i] &= __builtin_amdgcn_perm(m1, m0, 0x05040100u);
          g0 = fmaf(m0 ? g0 : 0.f, p.keep_scale, -d0), g1 = fmaf(m1 ? g1 : 0.f, p.keep_scale, -d1);
        } else {
          g0 -= d0, g1 -= d1;
        }
        ds[i] = Mma<T>::pack(Mma<T>::unpack(pk, 0) * g0, Mma<T>::unpack(pk, 1) * g1);
      }
#pragma unroll
      for (int sg = 0; sg < 2; ++sg)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          dv[db] = Mma<T>::run(rd.cols(dot, sg, db), u32x4{pm[4 * sg], pm[4 * sg + 1], pm[4 * sg + 2], pm[4 * sg + 3]}, dv[db]);
          dk[db] = Mma<T>::run(rd.cols(qt, sg, db), u32x4{ds[4 * sg], ds[4 * sg + 1], ds[4 * sg + 2], ds[4 * sg + 3]}, dk[db]);
        }
    }
    advance();
  }
  if (p.parts == 1 && n_items > 0) __syncthreads();  // (the rows leave through the tiles, which others may still read)
  if (p.parts > 1) {
    if (key >= p.S) return;  // float32 rows for bwd_dkdv_merge_kernel, which also applies the factors
    const int64_t row = ((((int64_t)(pq * p.parts_h + ph)) * p.B + b) * p.Hkv + hk) * p.S + key;
    float *gk = p.part_dk + row * dr + half * 4, *gv = p.part_dv + row * dr + half * 4;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if (db * 32 + g * 8 + half * 4 < dr) {
          *(f32x4*)(gk + db * 32 + g * 8) = f32x4{dk[db][g * 4], dk[db][g * 4 + 1], dk[db][g * 4 + 2], dk[db][g * 4 + 3]};
          *(f32x4*)(gv + db * 32 + g * 8) = f32x4{dv[db][g * 4], dv[db][g * 4 + 1], dv[db][g * 4 + 2], dv[db][g * 4 + 3]};
        }
    return;
  }
  store_rows<T>(dk, p.scale, &q_t[0][0] + wave * 32 * D, lane, (uint16_t*)p.gk + b * p.gk_sb + hk * p.gk_sh, p.gk_sl, kw0, p.S, dr);
  store_rows<T>(dv, DROP ? p.keep_scale : 1.f, &do_t[0][0] + wave * 32 * D, lane, (uint16_t*)p.gv + b * p.gv_sb + hk * p.gv_sh, p.gv_sl, kw0, p.S, dr);
}

// One block ahead: two workgroups per compute unit, the two phases of a block hold 211 to 240 registers.  (Against the four
// products one after the other in 168 registers, three workgroups: B=4, 12 heads, S=512, not causal, the whole backward 32.2 -> 27.5 us,
// B=1, S=1024 causal 39.1 -> 30.1, B=64, S=197 79.6 -> 77.7, B=4, 32 heads, S=4096 causal 1027 -> 1004; with dropout B=32, S=512
// 148 -> 139, with key counts as well 158 -> 148.  Where those are still taken: three_per_cu.  Neither goes to scratch;
// 16 to 24 scalar registers are kept in vector lanes.)
template <typename T, bool DROP, bool AHEAD>
__global__ __launch_bounds__(256, AHEAD ? 2 : 3) void bwd_d64_dkdv_kernel(BwdM p, const uint32_t* keep_bits, int chunk) {
  __shared__ __attribute__((aligned(16))) uint16_t q_t[3][TILE];
  __shared__ __attribute__((aligned(16))) uint16_t do_t[3][TILE];
  __shared__ __attribute__((aligned(16))) float lse_s[3][BQ], dl_s[3][BQ];
  __shared__ __attribute__((aligned(16))) KeepTile<DROP> bit_s[DROP ? 3 : 1];
  dkdv_body<T, DROP, AHEAD>(p, keep_bits, blockIdx.x, chunk, q_t, do_t, lse_s, dl_s, bit_s);
}

// The launch's parameters, read anew.  A workgroup of both kernels is one or the other; parameters that the compiler reads at
// the top for either want 83 to 108 scalar registers more than there are, and come back lane by lane in the loops.  Read where
// each body begins they all fit: causal, 4 heads, in us: B=7, S=2000 77.5 / 75.8, B=8, S=1700 67.2 / 63.1, B=10, S=1536 68.4 / 65.8;
// 12 heads: B=4, S=1024 45.6 / 43.0, B=1, S=128 12.8 / 11.6, B=4, S=512, not causal 26.3 / 24.8.
// (The kernels of their own hold 0 to 24 in vector lanes, outside their loops, and measure the same either way.)
__device__ __forceinline__ const BwdM& own_args() {
  auto args = (const __attribute__((address_space(4))) BwdM*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  return *(const BwdM*)args;
}

// Both in one launch, behind bwd_d64_terms_kernel: a dK/dV and a dQ workgroup by turns, eight of each (the XCDs), the
// heaviest of both first.  (See together for where.)
template <typename T, bool AHEAD>
__global__ __launch_bounds__(256, AHEAD ? 2 : 3) void bwd_d64_both_kernel(BwdM /* first: see own_args */, int dq_blocks, int dkdv_blocks, int dq_chunk, int dkdv_chunk) {
  __shared__ __attribute__((aligned(16))) uint16_t a_t[3][TILE];
  __shared__ __attribute__((aligned(16))) uint16_t b_t[3][TILE];
  __shared__ __attribute__((aligned(16))) float lse_s[3][BQ], dl_s[3][BQ];
  const int eight = blockIdx.x >> 3, in = blockIdx.x & 7, turns = min(dq_blocks + 7, dkdv_blocks + 7) >> 3;
  const bool dq = eight < 2 * turns ? (eight & 1) != 0 : dq_blocks > dkdv_blocks;
  const int bid = (eight < 2 * turns ? eight >> 1 : eight - turns) * 8 + in;
  if (bid >= (dq ? dq_blocks : dkdv_blocks)) return;
  if (dq) dq_body<T, false, false>(own_args(), nullptr, bid, dq_chunk, a_t, b_t);
  else dkdv_body<T, false, AHEAD>(own_args(), nullptr, bid, dkdv_chunk, a_t, b_t, lse_s, dl_s, nullptr);
}

// delta and the log2-domain log-sum-exp of 32 rows per wavefront, the sums in dq_body's order
template <typename T>
__global__ __launch_bounds__(256) void bwd_d64_terms_kernel(BwdM p, int blocks32) {
  const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), bh = w / blocks32;
  const int row = (int)(w % blocks32) * 32 + col;
  if (bh >= (int64_t)p.B * p.Hq || row >= p.L) return;  // (both halves of a row, which the shuffle pairs)
  const int b = (int)(bh / p.Hq), h = (int)(bh % p.Hq);
  const uint16_t* gr = (const uint16_t*)p.go + b * p.go_sb + h * p.go_sh + (int64_t)row * p.go_sl + half * 8;
  const uint16_t* orow = (const uint16_t*)p.out + b * p.o_sb + h * p.o_sh + (int64_t)row * p.o_sl + half * 8;
  float dsum = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    if (half * 8 + ks * 16 < p.d_real) dsum += dot8<T>(*(const u32x4*)(gr + ks * 16), *(const u32x4*)(orow + ks * 16));
  const float dl = dsum + __shfl_xor(dsum, 32, 64);
  const int64_t idx = bh * p.L + row;
  const float l = p.lse[idx];
  if (half == 0) p.delta[idx] = dl, p.lse2[idx] = l != -INFINITY ? l * kLog2eF : INFINITY;
}

// Streams of an XCD that it takes at a time, their two tensors having `rows` rows and `units` workgroups each, in equal chunks.
// Without the causal mask all of them where its 4 MB of L2 hold them, otherwise as many as fill a quarter of it (a keep-mask and
// the rows that are written pass through the same L2).  All / in chunks, backward in us, 8 heads: 3.1 MB: B=24, S=512 70 / 69;  4.0: B=20, S=785 127 / 131;
// 4.2: B=64, S=256 61 / 58, with dropout 72 / 67, B=32, S=512 87 / 84;  4.7: B=48, S=384 83 / 81;  6.3: B=48, S=512 122 / 118
// Under the mask the first workgroups of a chunk are the long ones, and the last chunk's should not start late:
//   up to four workgroups a stream, where they differ little, from 3.25 MB (three and four workgroups: 4) on in chunks of 32 to 48 workgroups.  All / so: B=64, S=256 55 / 54, B=48, S=320 56 / 52, S=384
//     69 / 62, S=448 81 / 80, S=512 95 / 89;  B=64, S=512 114 / 115, with dropout B=40, S=512 96 / 91;  less: B=32, S=256 with dropout 34 / 37, S=448 56 / 61, B=64, S=197 46 / 47.5, B=24, S=512 59 / 61
//     three, more than 32 streams of 288 keys and more: sixteens.  All / so: 33: S=300 43.9 / 41.3, S=384 51.8 / 51.2;  36: S=300 47.0 / 42.7, S=330 50.8 / 47.5;  40: S=300 48.5 / 45.9, S=330 54.7 / 50.9;
//       44: S=300 51.3 / 51.0, S=360 62.3 / 58.7;  48: S=330 61.5 / 57.0;  less: 32: S=300 37.9 / 37.4, S=384 46.7 / 45.3, 44: S=270 47.6 / 52.7, 56: S=260 56.2 / 61.9, S=286 58.3 / 60.7
//     four, 25 to 42 streams: two chunks, beyond 32 three.  All / eights / two / three: 25: S=390 47.9 / 51.9 / 45.0, S=512 58.1 / 65.3 / 57.9;  28: S=420 55.3 / 56.2 / 52.6, S=480 61.8 / 60.9 / 58.2, S=512 66.9 / 64.2 / 62.8,
//       with dropout 76.0 / 76.6 / 73.6;  31: S=390 55.1 / 57.9 / 55.7, S=512 69.4 / 68.7 / 65.4;  32: S=420 54.0 / 59.4 / 57.2, S=480 63.2 / 65.2 / 63.0, S=512 67.9 / 69.2 / 66.4;  33: S=420 59.9 / 67.4 / 60.7 / -,
//       S=480 69.0 / 70.7 / 67.0 / 66.0;  36: S=512 80.3 / 78.6 / 77.2 / 75.8;  38: S=512 with dropout 94.1 / 94.2 / 93.1 / 91.0;  40: S=512 with key counts 80.6 / 78.7 / 81.7 / 77.2
//   otherwise none up to 24 MB, six times the L2: B=11, 12 heads, S=1948 235, in two chunks of eight and a last one of a single stream 284; B=8, 8 heads, S=2500 199, two
//     of 4 MB 253, three of 2 MB 228; B=24, S=1024 120, 134, 127; B=8, 32/8, S=4096 (dK/dV: 33 MB) 1834, 1944, -.  Beyond it as many as the L2 holds, but 128 workgroups at
//     least: B=64, S=2048 1133 / 1061, B=96, S=1500 1053 / 991, B=32, 32/8, S=2048 2120 / 1990;  with dropout beyond 15 MB: 22 MB: B=116, S=747 522 / 498;  16.4: B=64, S=1000 442 / 428;  15.4: B=100, S=600 315 / 315;  11: B=60, S=747 256 / 260
// (A number of streams that does not divide over the XCDs: see pinned_streams, mfma_common.h)
int stream_chunk(const BwdM& g, int64_t rows, int64_t units) {
  const int64_t streams = (int64_t)g.B * g.Hkv, bytes = std::max<int64_t>(1, rows * D * 4), all = (streams + 7) / 8;
  if (!pinned_streams(streams, units)) return 0;
  int64_t chunk = all;
  if (!g.causal)
    chunk = all * bytes < (4 << 20) ? all : (1 << 20) / bytes;
  else if (units == 4 && g.Hq == g.Hkv && all > 24 && all <= 42 && all * bytes >= (all < 32 ? 9 << 18 : 4000000))
    chunk = all <= 32 ? 16 : 14;
  else if (units == 3 && g.Hq == g.Hkv && all > 32 && bytes >= 9 << 13)
    chunk = 16;
  else if (units <= 4)
    chunk = all * bytes < (units == 4 || (units == 3 && g.Hq == g.Hkv) ? 4 << 20 : 13 << 18) ? all : units == 4 ? 8 : 16;
  else if (all * bytes > (g.keep_scale != 0.f ? 15 << 20 : 24 << 20))
    chunk = std::max<int64_t>((4 << 20) / bytes, 128 / units);
  if (chunk < 1) chunk = 1;
  if (chunk >= all) return (int)std::max<int64_t>(1, all);
  const int64_t n = (all + chunk - 1) / chunk;
  return (int)((all + n - 1) / n);
}
// the two grids: a chunk (0: streams are not pinned) and the workgroups
struct Grid {
  int chunk;
  int64_t blocks;
};
Grid dq_grid(const BwdM& g) {
  const int64_t units = (int64_t)(g.Hq / g.Hkv) * g.n_qt, streams = (int64_t)g.B * g.Hkv;
  const int chunk = stream_chunk(g, g.S, units);
  return {chunk, mapped_blocks(streams, units, chunk)};
}
Grid dkdv_grid(const BwdM& g) {
  const int64_t streams = (int64_t)g.B * g.Hkv;
  const int chunk = g.parts > 1 ? 0 : stream_chunk(g, (int64_t)g.L * (g.Hq / g.Hkv), g.n_kt);
  return {chunk, mapped_blocks(streams, (int64_t)g.n_kt * g.parts, chunk)};
}

// Causal calls whose dK/dV workgroups are too few to hide the longest of them, which is long: a key block of the first keys sees
// every query row of several heads, the last one a few, all of them are on the chip at once, and at the end the long ones'
// chains run with nobody beside them.  The kernel of 8 wavefronts per workgroup (bwd_dkdv_w32.hip) has the shorter chain.  Below 384
// key blocks the items are split (bwd_dkdv_w32_plan), above two workgroups of this file's per compute unit the rest of the grid
// hides it.  Backward, us, dK/dV here / there (D=64):
//   four heads a kv head, 384 blocks: B=12, 32/8, S=512 99 / 91, B=6, 64/8, S=1024 307 / 264, B=3, 32/8, S=2048 294 / 254;  512: B=16, S=512 115 / 113, B=8, S=1024 181 / 168,
//     B=2, S=4096 630 / 563;  640: B=10, S=1024 204 / 218;  768: B=6, S=2048 422 / 459;  1024: B=8, S=2048 544 / 589;  short, 384: B=24, S=256 74 / 81
//   three: 384: B=6, 24/8, S=1024 111 / 111;  512: B=8, S=1024 139 / 131, B=4, S=2048 254 / 230;  seven: 512: B=16, 28/4, S=1024 308 / 287;  640: 345 / 371
//   two: 384: B=3, 16/8, S=2048 135 / 135;  512: B=4, S=2048 157 / 162, B=16, S=512 63 / 70
// (dQ's kernel there, two wavefronts a SIMD, and its dK/dV lose to both here with one head per kv head: B=6, 12 heads, S=1024 63 / 73, B=5, S=1500
// 90 / 107, B=4, S=2048 116 / 135, B=2, S=4096 203 / 245.)
bool w32_dkdv(const BwdM& g) {
  const int64_t blocks = (int64_t)g.B * g.Hkv * g.n_kt;
  return g.causal && g.keep_scale == 0.f && g.Hq >= 3 * g.Hkv && g.L > 5 * BQ && blocks >= 384 && blocks <= 512;
}

// Calls whose two kernels leave the chip half empty, each for as long as its longest chain of tiles: one launch of both,
// behind the one that forms the row terms (4 us).  The line is the number of workgroups in all (two of them share a compute
// unit), by the length of a chain, which is what the second launch would wait for.  Two launches / one, us, 12 heads and
// D=64 where not said:
//   not causal, 192: B=2, S=512 26.4 / 20.4;  384: B=8, S=197 20.3 / 20.2, B=4, S=512 29.9 / 27.5;  448: B=2, 16 heads, S=785 41.1 / 38.9;  3072: B=64, S=197 78 / 92
//     beyond 512 by the number of tiles, 640, 8 heads: B=40, S=64 16.0 / 17.6, S=128 22.5 / 23.3, B=20, S=256 27.8 / 28.6;  720: B=15, S=320 29.3 / 30.2, S=384 34.0 / 33.3,
//       B=9, S=640 45.6 / 43.8;  768: B=3, 16, S=1000 71.7 / 68.9;  816: B=17, S=384 34.7 / 39.2
//     two heads a kv head, 576: 16/8, B=24, S=128 21.8 / 24.6, B=6, S=512 43.6 / 41.9;  768: 16/8, B=32, S=128 23.2 / 26.9, B=8, S=512 44.4 / 48.0, split items B=6, 8/4, S=934 84.8 / 81.2, B=2, S=1498 79 / 70
//     three and more, 640: 32/8, B=16, S=100 27.8 / 25.1, S=128 27.2 / 25.7;  672: B=3, S=400 51.2 / 50.3;  704: 12/4, B=22, S=200 38.9 / 37.2;  768: B=16, S=330 51.2 / 49.5
//   causal, up to six 64-row tiles, 192: B=16, 6 heads, S=128 14.9 / 12.8;  384: B=16, 6, S=200 20.0 / 17.2, S=256 21.2 / 17.8
//     432: B=6, 12/6 heads, S=400 35.5 / 30.2;  576: B=6, S=400 27.8 / 23.7, B=12, S=256 24.3 / 27.7;  768: B=8, S=400 29.8 / 31.4
//     three heads a kv head and more: B=2, 12/4, S=400 39.2 / 34.1, 16/4, S=200 31.7 / 28.4, 28/4, S=150 36.8 / 34.8, B=8, 28/4, S=100 29.6 / 27.2
//   seven tiles and more, 480: B=4, S=600 33.2 / 25.8;  648: B=6, 12/6, S=700 51.3 / 43.4;  720: B=6, S=600 36.5 / 35.7
//     768: B=4, S=1024 51.1 / 47.7;  864: B=6, S=700 39.4 / 40.9;  1120: B=5, 16, S=777 50.6 / 54.4
//     grouped beyond 768: B=4, 32/8, S=700 77.5 / 80.2
//   fifteen and more, 1024: B=4, 16, S=1024 65.2 / 57.5, B=2, 16, S=2048 90.5 / 88.7;  2048: B=4, 16, S=2048 154 / 157
bool together(const BwdM& g) {
  if (g.keep_scale != 0.f || w32_dkdv(g)) return false;
  const int64_t all = (int64_t)g.B * g.Hq * g.n_qt + (int64_t)g.B * g.Hkv * g.n_kt * g.parts;
  if (!g.causal) return all <= (g.Hq >= 3 * g.Hkv ? 768 : g.L <= 5 * BQ ? 512 : g.Hq == g.Hkv || g.parts > 1 ? 768 : 704);
  return all <= (g.L < 7 * BQ ? 512 : g.Hq > g.Hkv || g.L <= 14 * BQ ? 768 : 1024);
}
// ... and which of them with dK/dV block by block, in three workgroups a compute unit: calls under the causal mask of more
// than two and a half each and short chains, which then are one turn.  Two launches / one, a block ahead / one, block by block, us:
//   576: S=448 29.8 / 23.5 / 26.5, S=512 33.7 / 27.5 / 29.9;  672: S=448 30.4 / 29.3 / 28.8, S=512 34.7 / 32.3 / 31.9;  768: S=448 31.3 / 31.1 / 29.2, S=512 35.3 / 33.2 / 32.0
//   longer: 680: S=576 35.9 / 31.2 / 32.7, S=640 39.8 / 35.3 / 35.6;  768: S=700 40.5 / 35.3 / 37.9, S=1024 53.2 / 45.7 / 48.0;  960: S=1536 77.3 / 68.3 / 66.3, S=2048 91.5 / 83.3 / 83.7
//   grouped, 768: 16/8, S=512 41.7 / 37.3 / 43.6
bool together_three_per_cu(const BwdM& g) {
  const int64_t all = (int64_t)g.B * g.Hq * g.n_qt + (int64_t)g.B * g.Hkv * g.n_kt * g.parts;
  return g.causal && g.Hq == g.Hkv && g.L <= 8 * BQ && all > 640 && all <= 768;
}

// Calls whose dK/dV runs block by block, three workgroups per compute unit: more key blocks than two per compute unit, but
// not than three, which then take one turn instead of two, and so few items each that the second turn is longer than what
// the two phases save.  A block ahead / block by block, the whole backward in us, D=64:
//   one item, 576 blocks: B=72, 8 heads, S=32 18.7 / 16.4, S=64 21.4 / 19.8;  768: S=32 18.9 / 17.0, S=64 22.9 / 21.8, causal 23.8 / 22.2, 32/8 heads, S=32 40.4 / 36.7
//     512: S=32 13.8 / 14.5, S=64 16.8 / 17.5;  832: S=32 22.8 / 22.8, S=64 28.0 / 28.5
//   two: 640, S=128 35.0 / 34.0, causal 35.9 / 34.2;  832: 44.5 / 44.1, causal 45.2 / 45.7;  three: S=160 31.0 / 30.7, S=192 35.2 / 34.5
//   causal, up to eight: 576, S=160 27.5 / 27.8, S=320 30.6 / 32.1;  704: S=256 41.0 / 38.0, S=320 36.7 / 34.0, S=384 42.7 / 38.5, S=512 56.1 / 54.2
//     768: S=256 42.6 / 39.8, S=384 45.6 / 41.1, S=512 53.6 / 51.0;  ten: S=640 54.4 / 53.9
// (With dropout, whose kernel takes more registers, a block ahead everywhere: B=64, 12 heads, S=64 25.0 / 26.7, S=100 39.2 / 42.0.)
bool three_per_cu(const BwdM& g) {
  const int64_t blocks = (int64_t)g.B * g.Hkv * (g.causal ? std::min(g.n_kt, (g.L + 127) / 128) : g.n_kt);  // (key blocks past the last row have no item)
  const int tiles = (g.L + BQ - 1) / BQ, items = g.Hq / g.Hkv * tiles;
  return blocks > 512 && blocks <= 768 && (tiles <= 1 || items <= 2 || (g.causal && items <= 8 && blocks > 640));
}

template <typename T>
int launch_together(const BwdM& g, hipStream_t s) {
  const int blocks32 = (g.L + 31) / 32;
  hipLaunchKernelGGL((bwd_d64_terms_kernel<T>), dim3((unsigned)(((int64_t)g.B * g.Hq * blocks32 + 3) / 4)), dim3(256), 0, s, g, blocks32);
  if (int rc = check_launch("bwd_d64_terms_kernel")) return rc;
  const Grid dq = dq_grid(g), dkdv = dkdv_grid(g);
  const int grid = (int)((dq.blocks + 7) / 8 + (dkdv.blocks + 7) / 8) * 8;
  if (together_three_per_cu(g)) hipLaunchKernelGGL((bwd_d64_both_kernel<T, false>), dim3(grid), dim3(256), 0, s, g, (int)dq.blocks, (int)dkdv.blocks, dq.chunk, dkdv.chunk);
  else hipLaunchKernelGGL((bwd_d64_both_kernel<T, true>), dim3(grid), dim3(256), 0, s, g, (int)dq.blocks, (int)dkdv.blocks, dq.chunk, dkdv.chunk);
  return check_launch("bwd_d64_both_kernel");
}

template <typename T, bool DROP>
int launch_t(const BwdM& g, uint32_t* bits, hipStream_t s) {
  if (!DROP && together(g)) {
    const int rc = launch_together<T>(g, s);
    if (rc || g.parts == 1) return rc;
    return launch_bwd_dkdv_merge(g, std::is_same<T, bf16_t>::value ? MI355_SDPA_BF16 : MI355_SDPA_F16, s);
  }
  const Grid dq = dq_grid(g), dkdv = dkdv_grid(g);
  hipLaunchKernelGGL((bwd_d64_dq_kernel<T, DROP>), dim3((unsigned)dq.blocks), dim3(256), 0, s, g, bits, dq.chunk);
  int rc = check_launch("bwd_d64_dq_kernel");
  if (rc) return rc;
  if (!DROP && w32_dkdv(g)) return launch_bwd_dkdv_w32(g, std::is_same<T, bf16_t>::value ? MI355_SDPA_BF16 : MI355_SDPA_F16, 64, s);
  if (!DROP && three_per_cu(g)) hipLaunchKernelGGL((bwd_d64_dkdv_kernel<T, false, false>), dim3((unsigned)dkdv.blocks), dim3(256), 0, s, g, nullptr, dkdv.chunk);
  else hipLaunchKernelGGL((bwd_d64_dkdv_kernel<T, DROP, true>), dim3((unsigned)dkdv.blocks), dim3(256), 0, s, g, (const uint32_t*)bits, dkdv.chunk);
  rc = check_launch("bwd_d64_dkdv_kernel");
  if (rc || g.parts == 1) return rc;
  return launch_bwd_dkdv_merge(g, std::is_same<T, bf16_t>::value ? MI355_SDPA_BF16 : MI355_SDPA_F16, s);
}

}  // namespace

bool bwd_d64_takes(const BwdM& g) {
  if (g.Hkv < 1) return false;  // (asked for the size of a workspace before anything is checked)
  if (g.d_real > 64 || g.dv_real != g.d_real || g.bias_kind || g.gbias || g.window > 0 || g.sm.any || g.dq_split_tiles) return false;
  // (32-bit byte offsets from the start of a batch, and of a key block's keep bits; the latter are the smaller ones
  // but for heads expanded from one)
  return bwd_dkdv_w32_fits(g, 64) && bwd_dq_w32_fits(g, 64) && (g.keep_scale == 0.f || block_words(g) * 4 < (1ll << 32));
}

size_t bwd_d64_bits_bytes(const BwdM& g) {
  if (g.keep_scale == 0.f || !bwd_d64_takes(g)) return 0;
  return ((size_t)g.B * g.Hkv * g.n_kt * block_words(g) * sizeof(uint32_t) + 255) & ~(size_t)255;
}

int launch_bwd_d64(const BwdM& g0, int dtype, uint32_t* keep_bits, hipStream_t s) {
  BwdM g = g0;
  if (!bwd_dkdv_plan_parts(g)) return MI355_SDPA_ERR_INVALID;
  if (g.keep_scale != 0.f && (!g.keep || !keep_bits)) {
    set_error("SDPA: dropout in the backward at head dim 64 needs a keep-mask and room for its bits in the workspace");
    return MI355_SDPA_ERR_INVALID;
  }
  const bool bf = dtype == MI355_SDPA_BF16;
  if (g.keep_scale != 0.f) return bf ? launch_t<bf16_t, true>(g, keep_bits, s) : launch_t<f16_t, true>(g, keep_bits, s);
  return bf ? launch_t<bf16_t, false>(g, nullptr, s) : launch_t<f16_t, false>(g, nullptr, s);
}

}  // namespace mi355
