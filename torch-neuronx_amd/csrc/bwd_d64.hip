// Flash-attention backward for gfx950 at head dims up to 64, bf16/f16: plain and causal calls, per-batch
// key counts, dropout.  (Calls with a bias, a window or a score functor, and causal ones with too few workgroups
// here, see w32_dkdv: bwd_dq_w32.hip, bwd_dkdv_w32.hip.)
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
// one wavefront and the waits around it.  So nothing here is pipelined by hand; the registers are kept
// to a third of the file (168) instead, three workgroups share a compute unit, and the chain of one
// wavefront runs under the other two's (dK/dV with dropout or of at most 512 workgroups: two, see OCC).
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

// blockIdx -> (tile, stream = (batch, kv head), unit within the stream's group of heads).  Workgroups of a
// stream read the same K / V (dQ) or Q / dO (dK/dV) and should meet in one L2: the streams are dealt to the
// XCDs (block i runs on XCD i % 8), and an XCD takes them in chunks whose tensors fill half of its 4 MB,
// all tiles of a chunk before the next one, heaviest tiles first within it.  (All streams of the XCD tile
// by tile, 48 of them of 128 KB: B=32, 12 heads, S=512, every tile pass fetches K and V from memory
// again, 274 MB for 126 MB of tensors, and the dQ kernel takes 142 thousand cycles instead of 130.)
struct BlockMap {
  int tile, stream, unit;
};
__device__ __forceinline__ BlockMap block_map(int bid, int streams, int n_tiles, int units, int chunk) {
  BlockMap m;
  if (chunk == 0) {  // (streams do not divide over the XCDs)
    m.tile = bid / (streams * units);
    const int r = bid % (streams * units);
    m.stream = r / units, m.unit = r % units;
    return m;
  }
  const int per_xcd = streams / 8, xcd = bid & 7;
  int r = bid >> 3;
  const int c = r / (chunk * n_tiles * units), in_chunk = min(chunk, per_xcd - c * chunk);
  r -= c * chunk * n_tiles * units;
  m.unit = r % units;
  r /= units;
  m.stream = (c * chunk + r % in_chunk) * 8 + xcd;
  m.tile = r / in_chunk;
  return m;
}

// (TERMS: leaves delta and the log2-domain log-sum-exp behind)
template <typename T, bool DROP, bool TERMS>
__device__ __forceinline__ void dq_body(const BwdM& p, uint32_t* keep_bits, int bid, int chunk, uint16_t (*k_t)[TILE], uint16_t (*v_t)[TILE]) {
  const int rep = p.Hq / p.Hkv;
  const BlockMap bm = block_map(bid, p.B * p.Hkv, p.n_qt, rep, chunk);
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
      if (kv0 >= S || (p.causal && kv0 > qw0 + 31)) continue;  // (uniform per wavefront)
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
template <typename T, bool DROP>
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
  }
  const int b = st / p.Hkv, hk = st % p.Hkv;
  const int rep_all = p.Hq / p.Hkv, rep = p.parts > 1 ? rep_all / p.parts_h : rep_all, h0 = hk * rep_all + ph * rep;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int k0 = kt * 128, kw0 = k0 + wave * 32, key = kw0 + col;
  const int dr = p.d_real;
  const int S = p.kv_lens ? min(p.S, max(p.kv_lens[b], 0)) : p.S;
  const int first_q = key >= S ? INT_MAX : p.causal ? key : INT_MIN;  // the first query row that sees this lane's key
  const int nqs = (p.L + BQ - 1) / BQ, qs_begin = p.causal ? min(k0 / BQ, nqs) : 0;
  int n_items = k0 >= S ? 0 : rep * (nqs - qs_begin);  // no live key in this block: zeros
  int it0 = 0;
  if (p.parts > 1) {
    it0 = pq * p.chunk_items;
    n_items = max(min(n_items - it0, p.chunk_items), 0);
    if (n_items == 0 && pq > 0) return;  // (bwd_dkdv_merge_kernel counts the filled shares in the same way)
  }
  // items: query tile by query tile from the last one down, the group's heads inside
  const uint32_t rep_inv = (uint32_t)((0x100000000ull + (uint32_t)rep - 1) / (uint32_t)rep);
  auto item_tile = [&](int it) { return rep == 1 ? it + it0 : (int)__umulhi((uint32_t)(it + it0), rep_inv); };
  auto item_head = [&](int it) { return h0 + (it + it0 - item_tile(it) * rep); };
  auto item_q0 = [&](int it) { return (nqs - 1 - item_tile(it)) * BQ; };

  const u32x4 bit_rsrc = descriptor(DROP ? keep_bits + ((int64_t)st * p.n_kt + kt) * block_words(p) : nullptr, DROP ? block_words(p) * 4 : 0);
  uint32_t q_off[NCH], go_off[NCH];
  chunk_offsets(q_off, tid, p.q_sl, dr);
  chunk_offsets(go_off, tid, p.go_sl, dr);
  const uint32_t lds_q = lds_address(q_t) + wave * 1024, lds_do = lds_address(do_t) + wave * 1024;
  // (the buffers of an item are its tile's own and end with the head's last row: a row past L must not be another
  // head's, whose NaN would survive the zero probabilities)
  auto load_item = [&](int it, int buf) {
    const int h = item_head(it), q0 = item_q0(it), rows = min(p.L - q0, BQ);
    const u32x4 q_rsrc = descriptor((const uint16_t*)p.q + b * p.q_sb + h * p.q_sh + (int64_t)q0 * p.q_sl, ((int64_t)(rows - 1) * p.q_sl + dr) * 2);
    const u32x4 go_rsrc = descriptor((const uint16_t*)p.go + b * p.go_sb + h * p.go_sh + (int64_t)q0 * p.go_sl, ((int64_t)(rows - 1) * p.go_sl + dr) * 2);
#pragma unroll
    for (int n = 0; n < NCH; ++n) {
      lds_load16(q_rsrc, q_off[n], lds_q + (uint32_t)(buf * TILE_BYTES + n * 4096));
      lds_load16(go_rsrc, go_off[n], lds_do + (uint32_t)(buf * TILE_BYTES + n * 4096));
    }
    if (wave < 2) {  // the rows' statistics: wavefront 0 log-sum-exps, wavefront 1 deltas
      const u32x4 st_rsrc = descriptor((wave == 0 ? p.lse2 : p.delta) + ((int64_t)b * p.Hq + h) * p.L + q0, rows * 4);
      lds_load4(st_rsrc, lane * 4, wave == 0 ? lds_address(lse_s[buf]) : lds_address(dl_s[buf]));
    }
    if constexpr (DROP) lds_load4(bit_rsrc, (uint32_t)((h - hk * rep_all) * p.L + q0 + lane) * 16 + wave * 4, lds_address(bit_s[buf][wave]));
  };
  // rows past L: no probability whatever stands there (wavefront 0, which loaded the values it writes over and has
  // waited for them)
  auto finish_item = [&](int it, int buf) {
    const int q0 = item_q0(it);
    if (q0 + BQ > p.L && tid < BQ && q0 + tid >= p.L) lse_s[buf][tid] = INFINITY;
  };
  if (n_items > 0) load_item(0, 0);
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
  if (n_items > 0) {
    wait_loads();
    finish_item(0, 0);
    __syncthreads();
    if (n_items > 1) load_item(1, 1);
  }
  auto step = [&](int it, auto buf_c) {
    constexpr int buf = decltype(buf_c)::value;
    const int q0 = item_q0(it);
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
      const int qb = q0 + mb * 32;
      if ((p.causal && qb + 31 < kw0) || kw0 >= S) continue;  // (uniform per wavefront)
      f32x16 s, dp;
      zero(s), zero(dp);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = Mma<T>::run(rd.rows(q_t[buf], mb, ks), kf[ks], s);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) dp = Mma<T>::run(rd.rows(do_t[buf], mb, ks), vf[ks], dp);
      if (__builtin_expect((p.causal && qb < kw0 + 31) || kw0 + 31 >= S, 0)) {
        asm volatile("" : "+v"(s));
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = qb + (r >> 2) * 8 + half * 4 + (r & 3) < first_q ? -INFINITY : s[r];
      }
      // dS is formed from P as the matrix pipe gets it, rounded to the input dtype (as in the kernels that
      // exchange P through LDS: a mask given as a tensor runs there, and the same mask as a flag here)
      uint32_t pk[8], pm[DROP ? 8 : 1];  // P in pairs; (dropout) the kept ones, for dV
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 l4 = *(const f32x4*)(&lse_s[buf][mb * 32 + g * 8 + half * 4]), d4 = *(const f32x4*)(&dl_s[buf][mb * 32 + g * 8 + half * 4]);
        u32x4 w4 = {0u, 0u, 0u, 0u};
        if constexpr (DROP) w4 = *(const u32x4*)(&bit_s[buf][wave][mb * 32 + g * 8 + half * 4]);
        const uint32_t words_e[4] = {w4[0], w4[1], w4[2], w4[3]};
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = __builtin_amdgcn_exp2f(fmaf(s[4 * g + e], c, -l4[e]));
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          pk[2 * g + j] = Mma<T>::pack(x[2 * j], x[2 * j + 1]);
          if constexpr (DROP) pm[2 * g + j] = 0u;
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int r = 4 * g + 2 * j + e;
            const float pr = Mma<T>::unpack(pk[2 * g + j], e);
            if constexpr (DROP) {
              // this key's bit of the row's word, as a mask of all ones or zeros
              const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)words_e[2 * j + e], (uint32_t)col, 1u);
              const float dpr = dp[r];  // (copied out: a bit cast of a vector element reads element 0)
              const float dpk = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, dpr) & m);
              dp[r] = pr * fmaf(dpk, p.keep_scale, -d4[2 * j + e]);
              pm[2 * g + j] |= m & (e ? 0xffff0000u : 0xffffu);
            } else {
              dp[r] = pr * (dp[r] - d4[2 * j + e]);
            }
          }
          if constexpr (DROP) pm[2 * g + j] &= pk[2 * g + j];
        }
      }
#pragma unroll
      for (int sg = 0; sg < 2; ++sg) {
        u32x4 bP;
        if constexpr (DROP) bP = u32x4{pm[4 * sg], pm[4 * sg + 1], pm[4 * sg + 2], pm[4 * sg + 3]};
        else bP = u32x4{pk[4 * sg], pk[4 * sg + 1], pk[4 * sg + 2], pk[4 * sg + 3]};
        float ds[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) ds[r] = dp[8 * sg + r];
        const u32x4 bS = pack8<T>(ds);
#pragma unroll
        for (int db = 0; db < DB; ++db) dv[db] = Mma<T>::run(rd.cols(do_t[buf], 2 * mb + sg, db), bP, dv[db]);
#pragma unroll
        for (int db = 0; db < DB; ++db) dk[db] = Mma<T>::run(rd.cols(q_t[buf], 2 * mb + sg, db), bS, dk[db]);
      }
    }
    constexpr int nb = (buf + 1) % 3;
    wait_loads();
    if (it + 1 < n_items) finish_item(it + 1, nb);
    __syncthreads();
    // (the buffer of item it - 1: its last readers passed the barrier above)
    if (it + 2 < n_items) load_item(it + 2, (buf + 2) % 3);
  };
  for (int it = 0;;) {
    if (it >= n_items) break;
    step(it, std::integral_constant<int, 0>{});
    if (++it >= n_items) break;
    step(it, std::integral_constant<int, 1>{});
    if (++it >= n_items) break;
    step(it, std::integral_constant<int, 2>{});
    ++it;
  }
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

// OCC: workgroups per compute unit that the registers are kept to.  Three is better where there are that many
// (B=32, 12 heads, S=512: 123 us for the whole backward against 127 with two, B=4, 32 heads, S=4096 causal 997
// / 1033), two where there are not (B=4, 12 heads, S=1024 causal, 384 workgroups: 54 / 58; at three a few
// values go to scratch) and with dropout (193 registers; B=32, 12 heads, S=512 155 / 161, B=4, 16, S=2048 causal 198 / 229).
template <typename T, bool DROP, int OCC>
__global__ __launch_bounds__(256, OCC) void bwd_d64_dkdv_kernel(BwdM p, const uint32_t* keep_bits, int chunk) {
  __shared__ __attribute__((aligned(16))) uint16_t q_t[3][TILE];
  __shared__ __attribute__((aligned(16))) uint16_t do_t[3][TILE];
  __shared__ __attribute__((aligned(16))) float lse_s[3][BQ], dl_s[3][BQ];
  __shared__ __attribute__((aligned(16))) KeepTile<DROP> bit_s[DROP ? 3 : 1];
  dkdv_body<T, DROP>(p, keep_bits, blockIdx.x, chunk, q_t, do_t, lse_s, dl_s, bit_s);
}

// Both in one launch, behind bwd_d64_terms_kernel: a dK/dV and a dQ workgroup by turns, eight of each (the XCDs), the
// heaviest of both first.  (See together for where.)
template <typename T>
__global__ __launch_bounds__(256, 3) void bwd_d64_both_kernel(BwdM p, int dq_blocks, int dkdv_blocks, int dq_chunk, int dkdv_chunk) {
  __shared__ __attribute__((aligned(16))) uint16_t a_t[3][TILE];
  __shared__ __attribute__((aligned(16))) uint16_t b_t[3][TILE];
  __shared__ __attribute__((aligned(16))) float lse_s[3][BQ], dl_s[3][BQ];
  const int eight = blockIdx.x >> 3, in = blockIdx.x & 7, turns = min(dq_blocks + 7, dkdv_blocks + 7) >> 3;
  const bool dq = eight < 2 * turns ? (eight & 1) != 0 : dq_blocks > dkdv_blocks;
  const int bid = (eight < 2 * turns ? eight >> 1 : eight - turns) * 8 + in;
  if (bid >= (dq ? dq_blocks : dkdv_blocks)) return;
  if (dq) dq_body<T, false, false>(p, nullptr, bid, dq_chunk, a_t, b_t);
  else dkdv_body<T, false>(p, nullptr, bid, dkdv_chunk, a_t, b_t, lse_s, dl_s, nullptr);
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

// streams of an XCD whose two tensors of `rows` rows fill half of its 4 MB of L2
int stream_chunk(const BwdM& g, int64_t rows) {
  const int streams = g.B * g.Hkv;
  if (streams % 8 != 0) return 0;
  return (int)std::max<int64_t>(1, std::min<int64_t>(streams / 8, (2 << 20) / (rows * D * 4)));
}

// Causal calls whose workgroups (tiles times streams) are too few to hide the longest of them: a key block of the first
// keys sees every query row, the last one a few, all of them are on the chip at once, and at the end the long ones' chains
// run with nobody beside them.  The kernels of 8 wavefronts per workgroup (bwd_dq_w32.hip, bwd_dkdv_w32.hip) have the shorter
// chain.  Below 384 key blocks their items are split (bwd_dkdv_w32_plan), above 1024 the rest of the grid hides it.
// Backward, us, both kernels here / dQ here and dK/dV there / both there (D=64):
//   grouped heads, 384 blocks: B=3, 32/8 heads, S=2048 337 / 253 / 263;  B=6, 64/8, S=1024 344 / 263 / 291
//     512: B=2, 32/8, S=4096 700 / 554 / 569;  B=8, 32/8, S=1024 200 / 170 / 194;  1024: B=8, 32/8, S=2048 626 / 580 / 639
//   dQ's own grid (B * Hq query tiles), 576: B=6, 12 heads, S=1024 83 / 78 / 72;  768: B=2, 12, S=4096 277 / 261 / 243
//     512: B=2, 8, S=4096 176 / 165 / 184;  768, S=512 (8 tiles): B=16, 12 53 / 57 / 56.  With key counts or narrow rows
//     the other dQ kernel is its masked variant: B=3, 12, S=2048 with key counts 109 here / 122 there, D=48 103 / 115
bool w32_dkdv(const BwdM& g) {
  const int64_t blocks = (int64_t)g.B * g.Hkv * g.n_kt;
  return g.causal && g.keep_scale == 0.f && g.Hq > g.Hkv && blocks >= 384 && blocks <= 1024;
}
bool w32_both(const BwdM& g) {
  const int64_t tiles = (int64_t)g.B * g.Hq * g.n_qt;
  return g.causal && g.keep_scale == 0.f && !g.kv_lens && g.d_real == D && (int64_t)g.B * g.Hkv * g.n_kt >= 384 && tiles > 512 && tiles <= 768 && g.L > 14 * BQ;
}

// Calls whose two kernels leave the chip half empty, each for as long as its longest chain of tiles: one launch of both.
// Up to one workgroup per compute unit in all, nobody shares anything; beyond it a causal call's long workgroups run
// beside short ones, up to three per compute unit, where the chains are long enough to pay for the third kernel in front
// (4 us) and for the registers (168, some in scratch).  Workgroups in all and us, two launches / one (12 heads, D=64):
//   up to 256: S=64, 6 heads 11.0 / 10.4;  B=4, S=197 not causal 19.8 / 17.9;  B=2, S=512 not causal 28.7 / 24.0;  B=1, S=1024 46.8 / 38.8
//     336: B=2, S=785 not causal 43.2 / 42.8;  384: B=8, S=197 not causal 20.5 / 21.9
//   causal, 384: B=16, 6 heads, S=200 19.3 / 18.3;  B=16, S=128 16.2 / 16.7;  grouped, 384: 16/4 heads, S=1021 47.6 / 41.1
//     512: B=4, 16/4, S=500 42.8 / 38.6;  1536: B=2, 32/8, S=1000 77.2 / 78.3;  768: B=16, S=256 25.6 / 26.9;  B=8, S=512 34.9 / 32.7;  B=4, S=1024 55.1 / 49.6
//     1024: B=8, 16 heads, S=512 39.0 / 44.8;  B=4, 16, S=1024 58.3 / 55.5;  B=2, 16, S=2048 96.2 / 85.5;  1152: B=12, S=512 56.0 / 57.9
// Three heads per kv head and more, whole chains in dK/dV (three query tiles, or items that are not split): dK/dV walks as
// many times dQ's tiles, dQ under it saves little, and its chain is the slower one in these registers.  Causal, two launches /
// one: B=2, 12/4 heads, S=400 46.3 / 47.6;  16/4, S=200 36.9 / 39.7, split, S=400 43.2 / 41.7;  28/4, S=100 33.6 / 36.8, S=150 43.8 / 49.5,
// split, S=200 34.5 / 33.8;  16/2, S=64 22.8 / 24.9, split, S=150 34.1 / 35.7, S=200 29.9 / 29.1.  (Two heads: 12/6, S=64 13.4 / 12.9, S=400 36.2 / 35.2.)
bool together(const BwdM& g) {
  if (g.keep_scale != 0.f || w32_dkdv(g)) return false;
  if (g.Hq >= 3 * g.Hkv && (g.parts == 1 || g.L <= 3 * BQ)) return false;
  const int64_t all = (int64_t)g.B * g.Hq * g.n_qt + (int64_t)g.B * g.Hkv * g.n_kt * g.parts;
  return all <= (!g.causal || g.L < 3 * BQ ? 256 : g.L < 7 * BQ ? 384 : g.Hq > g.Hkv ? 512 : g.L <= 14 * BQ ? 768 : 1024);
}

template <typename T>
int launch_together(const BwdM& g, hipStream_t s) {
  const int blocks32 = (g.L + 31) / 32;
  hipLaunchKernelGGL((bwd_d64_terms_kernel<T>), dim3((unsigned)(((int64_t)g.B * g.Hq * blocks32 + 3) / 4)), dim3(256), 0, s, g, blocks32);
  if (int rc = check_launch("bwd_d64_terms_kernel")) return rc;
  const int dq = g.B * g.Hq * g.n_qt, dkdv = g.B * g.Hkv * g.n_kt * g.parts;
  const int grid = ((dq + 7) / 8 + (dkdv + 7) / 8) * 8;
  hipLaunchKernelGGL((bwd_d64_both_kernel<T>), dim3(grid), dim3(256), 0, s, g, dq, dkdv, stream_chunk(g, g.S), stream_chunk(g, (int64_t)g.L * (g.Hq / g.Hkv)));
  return check_launch("bwd_d64_both_kernel");
}

template <typename T, bool DROP>
int launch_t(const BwdM& g, uint32_t* bits, hipStream_t s) {
  if (!DROP && together(g)) {
    const int rc = launch_together<T>(g, s);
    if (rc || g.parts == 1) return rc;
    return launch_bwd_dkdv_merge(g, std::is_same<T, bf16_t>::value ? MI355_SDPA_BF16 : MI355_SDPA_F16, s);
  }
  hipLaunchKernelGGL((bwd_d64_dq_kernel<T, DROP>), dim3((unsigned)((int64_t)g.B * g.Hq * g.n_qt)), dim3(256), 0, s, g, bits, stream_chunk(g, g.S));
  int rc = check_launch("bwd_d64_dq_kernel");
  if (rc) return rc;
  if (!DROP && w32_dkdv(g)) return launch_bwd_dkdv_w32(g, std::is_same<T, bf16_t>::value ? MI355_SDPA_BF16 : MI355_SDPA_F16, 64, s);
  const int64_t blocks = (int64_t)g.B * g.Hkv * g.n_kt * g.parts;
  const int chunk = stream_chunk(g, (int64_t)g.L * (g.Hq / g.Hkv));
#define DKDV(OCC) hipLaunchKernelGGL((bwd_d64_dkdv_kernel<T, DROP, OCC>), dim3((unsigned)blocks), dim3(256), 0, s, g, (const uint32_t*)bits, chunk)
  if (DROP || blocks <= 512) DKDV(2);
  else if constexpr (!DROP) DKDV(3);
#undef DKDV
  rc = check_launch("bwd_d64_dkdv_kernel");
  if (rc || g.parts == 1) return rc;
  return launch_bwd_dkdv_merge(g, std::is_same<T, bf16_t>::value ? MI355_SDPA_BF16 : MI355_SDPA_F16, s);
}

}  // namespace

bool bwd_d64_takes(const BwdM& g) {
  if (g.Hkv < 1) return false;  // (asked for the size of a workspace before anything is checked)
  if (g.d_real > 64 || g.dv_real != g.d_real || g.bias_kind || g.gbias || g.window > 0 || g.sm.any || g.dq_split_tiles || w32_both(g)) return false;
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
