// Causal GQA block-sparse flash-attention prefill for gfx950.
//
// Semantics follow the reference Triton kernel (tasft/kernels/block_sparse_fa.py:108-269)
// and its host preparation (:493-514):
//   * one query block of BS rows attends to the key blocks whose mask byte is non-zero;
//     with causal=1 the mask is AND-ed with the block lower triangle and, inside the
//     diagonal block, key > query is excluded;
//   * scores are fp32 (bf16 or fp16 MFMA, fp32 accumulate) times `scale`; online softmax in
//     fp32; P is rounded to the input type before the PV product (:252); l stays fp32;
//   * rows with no active key output 0 (:257-258); rows >= S are never stored (:268-269).
//
// GQA is native: query head h reads key/value head h / (Hq / Hkv) in place, so K/V are
// never expanded (the reference callers repeat_interleave them first,
// tasft/modules/tasft_attention.py:725-729).
//
// Mapping onto CDNA4. A wave owns 32 query rows (block 32: the workgroup is one such wave;
// blocks 64 and 128: two waves per 64 rows). Each key tile is computed as
// S^T = K . Q^T with v_mfma_f32_32x32x16_bf16 (_f16 for fp16 inputs), so a lane owns one query column of S^T:
// its running max and sum live in that lane (plus the lane 32 away), and the P^T
// accumulator registers feed the PV product O^T = V^T . P^T directly as the B operand
// with no shuffle. K and V tiles reach LDS by DMA, row major under an XOR swizzle; V^T
// operands are read transposed from there.
#include <algorithm>
#include <type_traits>

#include "common.h"


#include "../../include/tasft_amd.h"

namespace tasft {

struct PrefillParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  const uint8_t* mask;
  int64_t sq[3], sk[3], sv[3], so[3];  // element strides of dims (b, h, s); d stride is 1
  int64_t sm[4];                       // byte strides of the mask dims (b, h, qb, kb)
  int B, Hq, Hkv, G, S, NB;
  float scale_log2;  // softmax scale * log2(e)
  int causal;
  int small_spans;   // S * row bytes of K and V below 2^31: 32-bit DMA address math
  int small_q;       // the same of Q (block 32, head dim 64)
  // Packed variable-length batch: sequence b holds tokens cu_seqlens[b] .. cu_seqlens[b+1]-1
  // of dimension s (the b strides are 0), S is the longest length and NB its block count.
  // Null for a dense [B, H, S, D] launch.
  const int* cu_seqlens;
  // Mask index shift: 64-token query block qb and key block kb read mask entry
  // (qb >> mshift, kb >> mshift). 1 runs a block-128 mask on the block-64 kernels (a
  // 128-token block is active iff each of its 64-token quarters is); 0 otherwise.
  int mshift;
};

// Static order of the (batch, query head, query block) work items. gfx950 dispatches
// workgroup i to XCD i % 8; each XCD walks the KV groups congruent to it modulo 8 one at
// a time (all query heads and query blocks of the group, longest causal rows first) so
// the group's K/V stays in that XCD's L2. With a number of KV groups that is not a
// multiple of 8 the order is group-major.
struct PrefillItem {
  int b, kvh, h, qb;
};

__device__ __forceinline__ PrefillItem prefill_item(const PrefillParams& p, int64_t idx64) {
  // 32-bit arithmetic: the host rejects B * Hq * NB >= 2^31.
  const uint32_t idx = (uint32_t)idx64;
  const uint32_t groups = (uint32_t)(p.B * p.Hkv);
  const uint32_t per_group = (uint32_t)(p.G * p.NB);
  uint32_t grp, r;
  if ((groups & 7) == 0) {
    const uint32_t j = idx >> 3;
    grp = (idx & 7) + 8 * (j / per_group);
    r = j % per_group;
  } else {
    grp = idx / per_group;
    r = idx % per_group;
  }
  const int qslot = (int)(r / (uint32_t)p.G);
  PrefillItem it;
  it.qb = p.causal ? (p.NB - 1 - qslot) : qslot;
  it.b = (int)(grp / (uint32_t)p.Hkv);
  it.kvh = (int)(grp % (uint32_t)p.Hkv);
  it.h = it.kvh * p.G + (int)(r % (uint32_t)p.G);
  return it;
}

// Token span of batch entry b: the whole sequence dimension (dense launch), or sequence b
// of a packed batch (its first token and length, clamped to [0, S]).
struct SeqSpan {
  int S, NB;
  int64_t tok0;
};

template <int BS>
__device__ __forceinline__ SeqSpan seq_span(const PrefillParams& p, int b) {
  if (!p.cu_seqlens) return {p.S, p.NB, 0};
  const int t0 = p.cu_seqlens[b];
  int len = p.cu_seqlens[b + 1] - t0;
  len = len < 0 ? 0 : (len > p.S ? p.S : len);
  return {len, (len + BS - 1) / BS, (int64_t)t0};
}

// The softmax rescale is lazy where it pays: the running maximum used for exp2 is only moved
// when a new score exceeds it by more than this (so P stays <= 2^8); numerator and denominator
// share the same reference, so the normalised output is unchanged.
constexpr float kRescaleLog2 = 8.f;
// Head dim 64: moving it earlier keeps the largest probabilities of a row near a power of two,
// with less rounding error (8: 1% more error against 64 bits than one reference per 32 keys,
// 2: less, at 1-2% of the time).
constexpr float kRescale64Log2 = 2.f;

// 16-byte chunk position of chunk `cc` of K row `r` in LDS.
template <int D>
__device__ __forceinline__ int swz_k(int r, int cc) {
  return cc ^ (D == 128 ? (r & 15) : ((r >> 1) & 7));
}
// Same for V rows. ds_read_b64_tr_b16 serves 32 lanes (256 bytes) per LDS cycle: 4 rows
// x 4 chunks, which this swizzle spreads over all 64 banks.
template <int D>
__device__ __forceinline__ int swz_v(int r, int cc) {
  return cc ^ (D == 128 ? ((r & 3) << 2) : (((r >> 1) & 1) << 2));
}

// Next active key block of a mask row, scanning 64 mask bytes per ballot. Returns -1 at
// the end. All lanes of all waves see the same sequence.
__device__ __forceinline__ int next_active_block(const uint8_t* mrow, int64_t stride, int kb_end,
                                                 int lane, int& chunk, uint64_t& bits,
                                                 int mshift) {
  while (bits == 0) {
    chunk += kWave;
    if (chunk >= kb_end) return -1;
    const int kbl = chunk + lane;
    bits = __ballot(kbl < kb_end && mrow[(int64_t)(kbl >> mshift) * stride] != 0);
  }
  const int kb = chunk + __builtin_ctzll(bits);
  bits &= bits - 1;
  return kb;
}

// Raw buffer resource (stride 0) over `bytes` bytes starting at `base`.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const void* base, int64_t bytes) {
  const int n = bytes > 0x7fffffff ? 0x7fffffff : (bytes < 0 ? 0 : (int)bytes);
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, n, 0x00020000);
}

// One DMA instruction: 16 bytes per lane from r[voff] to 1 KB of LDS at `dst`.
template <int AUX>
__device__ __forceinline__ void dma16_lds(__amdgpu_buffer_rsrc_t r, uint8_t* dst, int voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (TASFT_LDS void*)dst, 16, voff, 0, 0, AUX);
}

// ---------------------------------------------------------------------------------------
// Block size 64 (and 128, through the mask index shift): two waves per query block.
//
// Wave w owns query rows 32*w..+31 and all 64 keys of every active key block: 16 S MFMAs
// (two 32-key tiles) and 16 PV MFMAs per block, so a row needs no merge of partial
// results. Four such workgroups (32 KB of LDS each: one K tile and one V tile) share a CU,
// two waves per SIMD. Per block: the V DMA starts once every wave has read the previous
// V tile, and the next block's K DMA once every wave has read this K tile; PV waits for V
// only. The barriers carry no memory fence (a __syncthreads() fence would also wait for
// the DMA still in flight): each is preceded by the explicit wait it needs. Each DMA
// instruction moves 1 KB; one LDS base (M0) serves four of them
// through the instruction offset, which the hardware adds to both the global and the LDS
// address (the field holds 12 bits, so units four apart need their own base).
// Q and O pass through the V tile, which is free before the row's first V DMA and after
// its last PV: Q arrives by DMA in the K layout (whole 256-byte rows per request) and is
// read into the MFMA operand registers like K; O is written there per wave and stored as
// whole rows, four per instruction. Loading Q and storing O directly in the MFMA layouts
// touched 32 rows, 32 bytes each, per instruction (1 KB of data in 32 cache lines).
//
// Head dim 64 takes 16 KB of LDS and three waves per SIMD (129 registers; four, with 122,
// measured 4% faster at B=4, S=8192 and 4% slower on dense masks). Against four waves per query
// block with two LDS stages and a merge of key halves, 32/8 heads, a fifth of the blocks: B=2,
// S=4096 55.7 us (68.6), with blocks of 128 55.3 us (68.4), nine tenths of the blocks 160 us
// (167); B=4, S=8192 298 us (330).
// ---------------------------------------------------------------------------------------
// Workgroup barrier without a memory fence. The caller waits (s_waitcnt) for what the
// barrier publishes; the memory clobber keeps the compiler from moving memory accesses
// across it.
__device__ __forceinline__ void block_barrier() { asm volatile("s_barrier" ::: "memory"); }

// AUX: the DMA's cache policy bits (0: default; 2: non-temporal, for Q, which a row reads
// once, so that it does not push its KV group's K and V out of L2).
template <int D, int AUX = 0>
__device__ __forceinline__ void dma_tile_2w(uint8_t* tile, __amdgpu_buffer_rsrc_t rsrc,
                                            const int* voff, int wave) {
  if constexpr (D == 128) {
    TASFT_LDS void* b0 = (TASFT_LDS void*)(tile + wave * 8192);
    TASFT_LDS void* b1 = (TASFT_LDS void*)(tile + wave * 8192 + 4096);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, b0, 16, voff[0], 0, 0, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, b0, 16, voff[1], 0, 1024, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, b0, 16, voff[2], 0, 2048, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, b0, 16, voff[3], 0, 3072, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, b1, 16, voff[4], 0, 0, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, b1, 16, voff[5], 0, 1024, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, b1, 16, voff[6], 0, 2048, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, b1, 16, voff[7], 0, 3072, AUX);
  } else {
    // Four units per wave, each with its own LDS base: row strides below 128 bytes stay legal.
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16_lds<AUX>(rsrc, tile + wave * 4096 + i * 1024, voff[i]);
  }
}

// PAIRS = 2 (few rows): such a launch is as long as its longest row, a chain of steps of one
// pair of waves. A second pair takes every other active block, with tiles of its own, and the
// pairs' (max, sum, output) meet in LDS after the row. Both pairs meet the same barriers; on
// an odd last block the second pair runs an empty one (zero K and V, all keys masked). One
// pair against two, D=128, 32/8 heads, a fifth of the blocks: S=1024 13.5 to 12.6 us; 8/2
// heads, S=4096 31.4 to 23.7 us, half of the blocks 63.7 to 42.8 us; D=64, 32/8 heads, S=1024
// 12.2 to 9.9 us.
template <int D, int DT, int PAIRS>
__global__ void __launch_bounds__(128 * PAIRS) __attribute__((amdgpu_waves_per_eu(D == 64 ? 3 : 2, D == 64 ? 3 : 2)))
bsfa_prefill_bs64_2w_kernel(const PrefillParams p) {
  constexpr int BS = 64;
  constexpr int KSTEPS = D / 16;
  constexpr int DTILES = D / 32;
  constexpr int ROWB = D * 2;
  constexpr int TILE = BS * ROWB;
  constexpr int UPW = (TILE / 1024) / 2;  // DMA units per wave and tile
  constexpr int kWaitTile = 0x0f70 | UPW;  // vmcnt: all but the last tile's units have landed
  constexpr float kMove = D == 128 ? kRescaleLog2 : kRescale64Log2;
  constexpr int LOW = D == 128 ? 1024 : 0;  // what dma_tile_2w's instruction offsets add per unit

  __shared__ __attribute__((aligned(1024))) uint8_t k_lds[PAIRS * TILE];
  __shared__ __attribute__((aligned(1024))) uint8_t v_lds[PAIRS * TILE];

  const int lane = threadIdx.x & 63;
  const int wave4 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar DMA addresses
  const int wave = PAIRS == 1 ? wave4 : wave4 & 1;  // row half
  const int pair = PAIRS == 1 ? 0 : wave4 >> 1;
  uint8_t* const kS = k_lds + pair * TILE;
  uint8_t* const vS = v_lds + pair * TILE;
  const int col = lane & 31;
  const int half = lane >> 5;

  // Per-lane source offsets of this wave's DMA units (the lane loads the
  // chunk that the self-inverse swizzle maps to its 16 bytes), less the instruction
  // offset that dma_tile_2w adds. Unit u starts at tile row 4u >= 4 (u & 3), so the
  // difference stays non-negative.
  int kvoff[UPW], vvoff[UPW];
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    const int byte = (wave * UPW + i) * 1024 + lane * 16;
    const int row = byte / ROWB, pos = (byte % ROWB) / 16;
    kvoff[i] = (row * (int)p.sk[2] + swz_k<D>(row, pos) * 8) * 2 - (i & 3) * LOW;
    vvoff[i] = (row * (int)p.sv[2] + swz_v<D>(row, pos) * 8) * 2 - (i & 3) * LOW;
  }
  const int grp16 = lane >> 4, t16 = lane & 15;  // ds_read_tr group and lane in group
  const int tr_row = t16 >> 2;                   // source row offset within a 4-row run
  const int tr_cb = t16 & 3;                     // source 8-byte column block
  const uint32_t krb = (uint32_t)p.sk[2] * 2u, vrb = (uint32_t)p.sv[2] * 2u;

  const PrefillItem item = prefill_item(p, (int64_t)blockIdx.x);
  const int qb = item.qb, b = item.b, kvh = item.kvh, h = item.h;
  // Varlen launch: items past the last query block of a shorter sequence have no work.
  const SeqSpan span = seq_span<BS>(p, b);
  if (qb >= span.NB) return;
  const int S = span.S, NB = span.NB;

  const uint16_t* qbase = p.q + b * p.sq[0] + span.tok0 * p.sq[2] + h * p.sq[1];
  const uint16_t* kbase = p.k + b * p.sk[0] + span.tok0 * p.sk[2] + kvh * p.sk[1];
  const uint16_t* vbase = p.v + b * p.sv[0] + span.tok0 * p.sv[2] + kvh * p.sv[1];
  uint16_t* obase = p.o + b * p.so[0] + span.tok0 * p.so[2] + h * p.so[1];
  const uint8_t* mrow = p.mask + b * p.sm[0] + h * p.sm[1] + (int64_t)(qb >> p.mshift) * p.sm[2];

  const int qrow = qb * BS + wave * 32 + col;
  const int kb_end = p.causal ? qb + 1 : NB;
  // Blocks from here on need element masks (causal diagonal or partial last block).
  const int mask_from = p.causal ? qb : ((S % BS) != 0 ? NB - 1 : NB);
  // Loads in the order their results are needed: mask bytes, Q, then the first K DMA.
  uint8_t mb = 0;
  if (lane < kb_end) mb = mrow[(int64_t)(lane >> p.mshift) * p.sm[3]];
  // The query block's rows go HBM->LDS by DMA into the V tile (unused until the first V
  // DMA), in the K tile's swizzled layout: each 1 KB unit is 4 whole rows, so every
  // request covers full cache lines. Rows past the end arrive as zeros (never stored).
  {
    int qvoff[UPW];
#pragma unroll
    for (int i = 0; i < UPW; ++i) {
      const int byte = (wave * UPW + i) * 1024 + lane * 16;
      const int row = byte / ROWB, pos = (byte % ROWB) / 16;
      qvoff[i] = (row * (int)p.sq[2] + swz_k<D>(row, pos) * 8) * 2 - (i & 3) * LOW;
    }
    dma_tile_2w<D, 2>(vS, tile_rsrc(qbase + (int64_t)qb * BS * p.sq[2],
                                    (int64_t)(S - qb * BS) * p.sq[2] * 2 + (D == 64 ? ROWB - p.sq[2] * 2 : 0)),
                      qvoff, wave);
  }
  // Buffer resource of key block kb of K or V (rows >= S are out of range: zeros). At D=64 it
  // ends exactly with row S-1, also when rows overlap (token strides below D).
  auto block_rsrc = [&](const uint16_t* base, uint32_t rb, int64_t stride, int kb) {
    if (PAIRS > 1 && kb < 0)  // the empty block: no rows, all zeros
      return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, 0, 0x00020000);
    if (p.small_spans) {
      const uint32_t key0 = (uint32_t)kb * BS, left = (uint32_t)S - key0;
      return __builtin_amdgcn_make_buffer_rsrc((void*)((const uint8_t*)base + key0 * rb), (short)0,
                                               (int)(left * rb + (D == 64 ? ROWB - rb : 0u)), 0x00020000);
    }
    const int key0 = kb * BS;
    return tile_rsrc(base + (int64_t)key0 * stride,
                     (int64_t)(S - key0) * stride * 2 + (D == 64 ? ROWB - stride * 2 : 0));
  };

  f32x16_t oacc[DTILES];
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) oacc[dt] = (f32x16_t){};
  float m_ref = -INFINITY;  // exp2 reference of this lane's query row (log2 domain)
  float l_run = 0.f;

  int chunk = 0;
  uint64_t bits = __ballot(mb != 0);
  // The next active block, or with two pairs the next two: the first in `lead`, this pair's
  // (-1: none) returned.
  int lead = 0;
  auto next_block = [&]() {
    const int first = next_active_block(mrow, p.sm[3], kb_end, lane, chunk, bits, p.mshift);
    lead = first;
    if constexpr (PAIRS == 1) return first;
    const int second =
        first >= 0 ? next_active_block(mrow, p.sm[3], kb_end, lane, chunk, bits, p.mshift) : -1;
    return pair == 0 ? first : second;
  };
  int kb = next_block();
  u32x4_t qf[KSTEPS];
  if (lead >= 0) {
    dma_tile_2w<D>(kS, block_rsrc(kbase, krb, p.sk[2], kb), kvoff, wave);
    __builtin_amdgcn_s_waitcnt(kWaitTile);  // own share of Q landed, K in flight
  } else {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  }
  block_barrier();  // Q visible; the loop's first barrier orders these reads before V's DMA
  {
    const int r = wave * 32 + col;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks)
      qf[ks] = *(const u32x4_t*)(vS + r * ROWB + swz_k<D>(r, ks * 2 + half) * 16);
  }
  if (D == 64 && !p.small_q) {
    // Token strides the DMA's 32-bit offsets do not cover: the rows again, from memory.
    const uint16_t* qr = qbase + (int64_t)min(qrow, S - 1) * p.sq[2] + half * 8;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) qf[ks] = *(const u32x4_t*)(qr + ks * 16);
  }

  while (lead >= 0) {
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): own share of K(kb) landed
    block_barrier();                      // K(kb) visible; every wave is done with the V tile
    dma_tile_2w<D>(vS, block_rsrc(vbase, vrb, p.sv[2], kb), vvoff, wave);
    u32x4_t kf[2][KSTEPS];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        const int r = kt * 32 + col;
        kf[kt][ks] = *(const u32x4_t*)(kS + r * ROWB + swz_k<D>(r, ks * 2 + half) * 16);
      }
    f32x16_t s0 = (f32x16_t){}, s1 = (f32x16_t){};
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      s0 = mfma16<DT>(kf[0][ks], qf[ks], s0);
      s1 = mfma16<DT>(kf[1][ks], qf[ks], s1);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's K reads returned
    block_barrier();                      // every wave has read K(kb): the K tile is free
    const int kb_next = next_block();
    // Always one K tile's DMA units after V(kb) (the last block of a row loads its own K tile
    // again), so the V wait below is one fixed count.
    dma_tile_2w<D>(kS, block_rsrc(kbase, krb, p.sk[2], lead >= 0 ? kb_next : kb), kvoff, wave);
    const bool empty = PAIRS > 1 && kb < 0;
    if (empty || kb >= mask_from) {
      // Register rr of tile t holds key kb*BS + 32t + 4*half + off(rr), off = 8*(rr/4) +
      // rr%4; a key is admissible iff it is <= min(qrow, S-1) (causal) or S-1, i.e. iff
      // 32t + off <= lim below: one compare per score.
      const int last = p.causal ? min(qrow, S - 1) : S - 1;
      const int lim = empty ? -1 : last - kb * BS - 4 * half;
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) {
        const int off = 8 * (rr >> 2) + (rr & 3);
        s0[rr] = off > lim ? -INFINITY : s0[rr];
        s1[rr] = off + 32 > lim ? -INFINITY : s1[rr];
      }
    }
    // Scores stay unscaled: scale > 0 commutes with max, and exp2 takes one FMA. Two
    // chains of three-input maxima.
    float ma = fmaxf(fmaxf(s0[0], s0[1]), s0[2]), mb = fmaxf(fmaxf(s1[0], s1[1]), s1[2]);
#pragma unroll
    for (int rr = 3; rr < 15; rr += 2) {
      ma = fmaxf(fmaxf(ma, s0[rr]), s0[rr + 1]);
      mb = fmaxf(fmaxf(mb, s1[rr]), s1[rr + 1]);
    }
    const float mraw = fmaxf(fmaxf(ma, s0[15]), fmaxf(mb, s1[15]));
    const float mloc = pair_max32(mraw) * p.scale_log2;
    const bool move = mloc > m_ref + kMove;
    if (__ballot(move)) {
      // exp2(-inf) = 0 clears the (empty) accumulators on a row's first finite score.
      const float alpha = move ? __builtin_amdgcn_exp2f(m_ref - mloc) : 1.f;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DTILES; ++dt) oacc[dt] *= alpha;
      m_ref = move ? mloc : m_ref;
    }
    const float m_use = (m_ref == -INFINITY) ? 0.f : m_ref;
    float lsum0 = 0.f, lsum1 = 0.f;
#pragma unroll
    for (int rr = 0; rr < 16; ++rr) {
      const float e0 = __builtin_amdgcn_exp2f(fmaf(s0[rr], p.scale_log2, -m_use));
      const float e1 = __builtin_amdgcn_exp2f(fmaf(s1[rr], p.scale_log2, -m_use));
      s0[rr] = e0;
      s1[rr] = e1;
      lsum0 += e0;
      lsum1 += e1;
    }
    l_run += lsum0 + lsum1;
    // P^T as the B operand of four 16-key k-steps: keys 16pp + 8*(j>>2) + 4*half + (j&3)
    // for element j, the same key order the V^T reads below use.
    u32x4_t pb[4];
#pragma unroll
    for (int pp = 0; pp < 4; ++pp) {
      const f32x16_t& sv = (pp < 2) ? s0 : s1;
      const int o = 8 * (pp & 1);
      const u32x4_t w = {pack16x2<DT>(sv[o + 0], sv[o + 1]), pack16x2<DT>(sv[o + 2], sv[o + 3]),
                         pack16x2<DT>(sv[o + 4], sv[o + 5]), pack16x2<DT>(sv[o + 6], sv[o + 7])};
      pb[pp] = w;
    }
    __builtin_amdgcn_s_waitcnt(kWaitTile);  // own share of V(kb) landed, next K in flight
    block_barrier();                      // V(kb) visible
    u32x2_t vlo[4][DTILES], vhi[4][DTILES];
#pragma unroll
    for (int pp = 0; pp < 4; ++pp) {
      const int kk = 16 * pp + 4 * (grp16 >> 1);  // first key of run 1
#pragma unroll
      for (int dt = 0; dt < DTILES; ++dt) {
        const int d0 = dt * 32 + 16 * (grp16 & 1) + 4 * tr_cb;  // source column of this lane
        const int cc = d0 >> 3, sub = (d0 & 7) * 2;
        const int r1 = kk + tr_row, r2 = r1 + 8;
        vlo[pp][dt] = ds_read_tr16_b64((const void*)(vS + r1 * ROWB + swz_v<D>(r1, cc) * 16 + sub));
        vhi[pp][dt] = ds_read_tr16_b64((const void*)(vS + r2 * ROWB + swz_v<D>(r2, cc) * 16 + sub));
      }
    }
#pragma unroll
    for (int pp = 0; pp < 4; ++pp)
#pragma unroll
      for (int dt = 0; dt < DTILES; ++dt) {
        const u32x4_t a = {vlo[pp][dt][0], vlo[pp][dt][1], vhi[pp][dt][0], vhi[pp][dt][1]};
        oacc[dt] = mfma16<DT>(a, pb[pp], oacc[dt]);
      }
    kb = kb_next;
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // no DMA into this workgroup's LDS outlives it

  float l_tot = pair_sum32(l_run);
  if constexpr (PAIRS > 1) {
    // The second pair's sums through its own K and V tiles (16 DTILES x 64 floats per wave).
    static_assert(DTILES * 16 * kWave * 4 == TILE, "merge buffers");
    __shared__ float x_m[2][kWave], x_l[2][kWave];
    float* xo = (float*)(wave == 0 ? k_lds + TILE : v_lds + TILE);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's V reads returned
    block_barrier();                      // every wave is done with the tiles
    if (pair == 1) {
#pragma unroll
      for (int dt = 0; dt < DTILES; ++dt)
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) xo[(dt * 16 + rr) * kWave + lane] = oacc[dt][rr];
      x_m[wave][lane] = m_ref;
      x_l[wave][lane] = l_tot;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the stores above are in LDS
    block_barrier();
    if (pair == 1) return;
    const float m1 = x_m[wave][lane], l1 = x_l[wave][lane];
    const float m = fmaxf(m_ref, m1);
    const float mu = (m == -INFINITY) ? 0.f : m;
    const float f0 = __builtin_amdgcn_exp2f(m_ref - mu), f1 = __builtin_amdgcn_exp2f(m1 - mu);
    l_tot = l_tot * f0 + l1 * f1;
#pragma unroll
    for (int dt = 0; dt < DTILES; ++dt)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr)
        oacc[dt][rr] = oacc[dt][rr] * f0 + xo[(dt * 16 + rr) * kWave + lane] * f1;
  }
  const float inv = 1.f / (l_tot > 0.f ? l_tot : 1.f);  // empty rows: O = 0; NaN rows stay NaN
  // The output through LDS: each wave writes its 32 rows into its own 8 KB of the V tile
  // (16-byte chunk c of row r at position c ^ (r & 15)), then stores whole 256-byte rows,
  // four rows per instruction.
  if constexpr (PAIRS == 1) {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's V reads returned
    block_barrier();                      // every wave is done with the V tile
  }
  uint8_t* ost = vS + wave * (32 * ROWB);
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      const int d0 = dt * 32 + 8 * gq + 4 * half;
      const u32x2_t w = {pack16x2<DT>(oacc[dt][4 * gq + 0] * inv, oacc[dt][4 * gq + 1] * inv),
                         pack16x2<DT>(oacc[dt][4 * gq + 2] * inv, oacc[dt][4 * gq + 3] * inv)};
      *(u32x2_t*)(ost + col * ROWB + (((d0 >> 3) ^ (col & (ROWB / 16 - 1))) << 4) + (d0 & 7) * 2) = w;
    }
  constexpr int CPR = ROWB / 16;  // 16-byte chunks per row
  const int row0 = qb * BS + wave * 32;
#pragma unroll
  for (int j = 0; j < 32 * CPR / kWave; ++j) {
    const int r = j * (kWave / CPR) + lane / CPR, c = lane % CPR;
    const u32x4_t v = *(const u32x4_t*)(ost + r * ROWB + ((c ^ (r & (CPR - 1))) << 4));
    // Non-temporal: the output is not read again here, and K/V stay in L2.
    if (row0 + r < S) __builtin_nontemporal_store(v, (u32x4_t*)(obase + (int64_t)(row0 + r) * p.so[2] + c * 8));
  }
}

// ---------------------------------------------------------------------------------------
// Block size 32: one wave per (batch, query head, query block of 32 rows).
//
// Neighbouring 32-row query blocks and query heads have their own masks, so a tile that
// several waves share would be mostly masked work; every wave walks its own blocks with its
// own LDS tiles instead, and needs no barrier at all. A step takes NT active key blocks
// (any two: the tile is gathered), 8 KB of K and 8 KB of V at the most: head dim 128 one
// block, head dim 64 two. K and V arrive by buffer_load_dwordx4 ... lds in the layouts of the
// block-64 kernels; V's DMA runs under the S MFMAs and the softmax, the next K's under the
// softmax and PV. Unlike in the block-64 kernels the exp2 reference follows every new
// maximum, tile by tile: the largest probability of a tile is then exactly 1 and carries no
// rounding error (the lazy rescale measured 9% faster and its fp16 output 8% further from
// 64 bits).
//
// Bound by the latency of a step (DMA, S, softmax and PV of one wave in turn), hidden by the
// waves beside it: LDS allows ten per CU, three per SIMD at D=64 need 168 registers at most
// (two, with 185, measured 5% slower). Against staging through registers with a transpose
// of V by VALU: B=2, 16 heads, S=4000, D=64, a quarter of the blocks, fp16 48 us (106 us);
// B=2, 32/8 heads, S=4096, D=128, a fifth, bf16 98 us (261 us). One block per step at D=64
// took 51.7 us in the first case (and 6% less than two with twice the rows).
// ---------------------------------------------------------------------------------------
// SMALL: every row of Q, K and V lies within 2 GB of its head's first (32-bit offsets).
template <int D, int NT, int DT, bool SMALL>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(D == 64 ? 3 : 2)))
bsfa_prefill_bs32_kernel(const PrefillParams p) {
  constexpr int BS = 32;
  constexpr int KSTEPS = D / 16;
  constexpr int DTILES = D / 32;
  constexpr int ROWB = D * 2;
  constexpr int UPB = BS * ROWB / 1024;  // 1 KB DMA units per block
  constexpr int RPU = 1024 / ROWB;       // rows per unit
  constexpr int WAITN = NT * UPB;        // DMA units of one K or V tile
  static_assert(WAITN == 4 || WAITN == 8, "vmcnt of one tile");

  __shared__ __attribute__((aligned(1024))) uint8_t kS[NT * BS * ROWB];
  __shared__ __attribute__((aligned(1024))) uint8_t vS[NT * BS * ROWB];

  const int lane = threadIdx.x;
  const int col = lane & 31;
  const int half = lane >> 5;

  const PrefillItem item = prefill_item(p, (int64_t)blockIdx.x);
  const int qb = item.qb, b = item.b, kvh = item.kvh, h = item.h;
  // Varlen launch: items past the last query block of a shorter sequence have no work.
  const SeqSpan span = seq_span<BS>(p, b);
  if (qb >= span.NB) return;
  const int S = span.S, NB = span.NB;

  const uint16_t* qbase = p.q + b * p.sq[0] + span.tok0 * p.sq[2] + h * p.sq[1];
  const uint16_t* kbase = p.k + b * p.sk[0] + span.tok0 * p.sk[2] + kvh * p.sk[1];
  const uint16_t* vbase = p.v + b * p.sv[0] + span.tok0 * p.sv[2] + kvh * p.sv[1];
  uint16_t* obase = p.o + b * p.so[0] + span.tok0 * p.so[2] + h * p.so[1];
  const uint8_t* mrow = p.mask + b * p.sm[0] + h * p.sm[1] + (int64_t)qb * p.sm[2];

  const int qrow = qb * BS + col;
  const int kb_end = p.causal ? qb + 1 : NB;
  // Blocks from here on need element masks (causal diagonal or partial last block).
  const int mask_from = p.causal ? qb : ((S % BS) != 0 ? NB - 1 : NB);
  uint8_t mb = 0;
  if (lane < kb_end) mb = mrow[(int64_t)lane * p.sm[3]];

  // One 32-row block to `tile`, unit by unit: the lane loads the global chunk that the
  // (self-inverse) swizzle maps to its 16 bytes. The buffer ends with row S-1, so rows past
  // it (and every row of a block at or past S) arrive as zeros. `voff` is 32-bit: without
  // SMALL each unit gets its own base, and offsets count from there.
  auto dma_block = [&](uint8_t* tile, const uint16_t* base, int64_t stride, int row0,
                       const uint32_t* voff, auto aux) {
    constexpr int AUX = decltype(aux)::value;
    const uint32_t rb = (uint32_t)stride * 2u;
    if constexpr (SMALL) {
      const int left = S - row0;
      const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
          (void*)((const uint8_t*)base + (uint32_t)row0 * rb), (short)0,
          left > 0 ? (int)((uint32_t)(left - 1) * rb + ROWB) : 0, 0x00020000);
#pragma unroll
      for (int u = 0; u < UPB; ++u) dma16_lds<AUX>(r, tile + u * 1024, (int)voff[u]);
    } else {
#pragma unroll
      for (int u = 0; u < UPB; ++u) {
        const int64_t left = (int64_t)S - row0 - u * RPU;
        dma16_lds<AUX>(tile_rsrc((const uint8_t*)base + (int64_t)(row0 + u * RPU) * stride * 2,
                                 left > 0 ? (left - 1) * stride * 2 + ROWB : 0),
                       tile + u * 1024, (int)(voff[u] - (uint32_t)(u * RPU) * rb));
      }
    }
  };
  uint32_t kvoff[UPB], vvoff[UPB];
#pragma unroll
  for (int u = 0; u < UPB; ++u) {
    const int row = u * RPU + lane / (ROWB / 16), pos = lane % (ROWB / 16);
    kvoff[u] = ((uint32_t)row * (uint32_t)p.sk[2] + swz_k<D>(row, pos) * 8) * 2u;
    vvoff[u] = ((uint32_t)row * (uint32_t)p.sv[2] + swz_v<D>(row, pos) * 8) * 2u;
  }
  using Default = std::integral_constant<int, 0>;
  using Streamed = std::integral_constant<int, 2>;  // non-temporal: Q is read once
  {
    // Q through the V tile, unused until the first V DMA, in K's layout.
    uint32_t qvoff[UPB];
#pragma unroll
    for (int u = 0; u < UPB; ++u) {
      const int row = u * RPU + lane / (ROWB / 16), pos = lane % (ROWB / 16);
      qvoff[u] = ((uint32_t)row * (uint32_t)p.sq[2] + swz_k<D>(row, pos) * 8) * 2u;
    }
    dma_block(vS, qbase, p.sq[2], qb * BS, qvoff, Streamed{});
  }

  // The next NT active blocks; -1 where the row has no more (their keys are masked off).
  int chunk = 0;
  uint64_t bits = __ballot(mb != 0);
  auto next_step = [&](int (&kb)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
      kb[t] = (t > 0 && kb[t - 1] < 0)
                  ? -1
                  : next_active_block(mrow, p.sm[3], kb_end, lane, chunk, bits, 0);
  };
  // A missing second block is loaded from row S on, which is all zeros.
  auto dma_k = [&](const int (&kb)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
      dma_block(kS + t * BS * ROWB, kbase, p.sk[2], kb[t] < 0 ? S : kb[t] * BS, kvoff, Default{});
  };
  auto dma_v = [&](const int (&kb)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
      dma_block(vS + t * BS * ROWB, vbase, p.sv[2], kb[t] < 0 ? S : kb[t] * BS, vvoff, Default{});
  };
  // vmcnt of one tile's units: everything older than the last tile has landed.
  auto wait_all_but_one_tile = [&]() {
    if constexpr (WAITN == 8)
      __builtin_amdgcn_s_waitcnt(0x0f78);
    else
      __builtin_amdgcn_s_waitcnt(0x0f74);
    asm volatile("" ::: "memory");
  };

  int kb[NT];
  next_step(kb);
  u32x4_t qf[KSTEPS];
  if (kb[0] >= 0) {
    dma_k(kb);
    wait_all_but_one_tile();  // Q landed, K in flight
  } else {
    __builtin_amdgcn_s_waitcnt(0x0f70);
    asm volatile("" ::: "memory");
  }
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks)
    qf[ks] = *(const u32x4_t*)(vS + col * ROWB + swz_k<D>(col, ks * 2 + half) * 16);

  f32x16_t oacc[DTILES];
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) oacc[dt] = (f32x16_t){};
  float m_ref = -INFINITY;  // exp2 reference of this lane's query row (log2 domain)
  float l_run = 0.f;
  const int grp16 = lane >> 4, t16 = lane & 15;  // ds_read_tr group and lane in group
  const int tr_row = t16 >> 2;                   // source row offset within a 4-row run
  const int tr_cb = t16 & 3;                     // source 8-byte column block

  while (kb[0] >= 0) {
    // vmcnt(0) lgkmcnt(0): K landed, and the reads of the V tile (Q, the last PV) returned.
    __builtin_amdgcn_s_waitcnt(0x0070);
    asm volatile("" ::: "memory");
    dma_v(kb);
    u32x4_t kf[NT][KSTEPS];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        const int r = t * 32 + col;
        kf[t][ks] = *(const u32x4_t*)(kS + r * ROWB + swz_k<D>(r, ks * 2 + half) * 16);
      }
    f32x16_t s[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) s[t] = (f32x16_t){};
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
      for (int t = 0; t < NT; ++t) s[t] = mfma16<DT>(kf[t][ks], qf[ks], s[t]);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the K reads returned, the tile is free
    asm volatile("" ::: "memory");
    int kb_next[NT];
    next_step(kb_next);
    // Always one K tile after V (a row's last step loads its own again), so that the V wait
    // below is one fixed count.
    int kb_load[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) kb_load[t] = kb_next[0] >= 0 ? kb_next[t] : kb[t];
    dma_k(kb_load);
    const bool ragged = kb[NT - 1] < 0;
    if (ragged || kb[NT - 1] >= mask_from) {
      // Register rr of tile t holds key kb[t]*32 + 4*half + off(rr), off = 8*(rr/4) + rr%4,
      // admissible iff off <= lim.
      const int last = p.causal ? min(qrow, S - 1) : S - 1;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int lim = kb[t] < 0 ? -1 : last - kb[t] * BS - 4 * half;
#pragma unroll
        for (int rr = 0; rr < 16; ++rr)
          s[t][rr] = 8 * (rr >> 2) + (rr & 3) > lim ? -INFINITY : s[t][rr];
      }
    }
    // Scores stay unscaled: scale > 0 commutes with max, and exp2 takes one FMA. Each
    // 32-key tile has its own reference (the running maximum after it).
    float ref[NT], alpha[NT];
    bool moved[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float m = fmaxf(fmaxf(s[t][0], s[t][1]), s[t][2]);
#pragma unroll
      for (int rr = 3; rr < 15; rr += 2) m = fmaxf(fmaxf(m, s[t][rr]), s[t][rr + 1]);
      const float mloc = pair_max32(fmaxf(m, s[t][15])) * p.scale_log2;
      const bool move = mloc > m_ref;
      moved[t] = __ballot(move) != 0;
      // exp2(-inf) = 0 clears the (empty) accumulators on a row's first finite score.
      alpha[t] = move ? __builtin_amdgcn_exp2f(m_ref - mloc) : 1.f;
      m_ref = move ? mloc : m_ref;
      ref[t] = (m_ref == -INFINITY) ? 0.f : m_ref;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float lsum = 0.f;
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) {
        const float e = __builtin_amdgcn_exp2f(fmaf(s[t][rr], p.scale_log2, -ref[t]));
        s[t][rr] = e;
        lsum += e;
      }
      l_run = l_run * alpha[t] + lsum;
    }
    // P^T as the B operand of 16-key k-steps: keys 16pp + 8*(j>>2) + 4*half + (j&3) of a
    // tile for element j, the same key order the V^T reads below use.
    u32x4_t pb[2 * NT];
#pragma unroll
    for (int pp = 0; pp < 2 * NT; ++pp) {
      const f32x16_t& sv = s[pp >> 1];
      const int o = 8 * (pp & 1);
      const u32x4_t w = {pack16x2<DT>(sv[o + 0], sv[o + 1]), pack16x2<DT>(sv[o + 2], sv[o + 3]),
                         pack16x2<DT>(sv[o + 4], sv[o + 5]), pack16x2<DT>(sv[o + 6], sv[o + 7])};
      pb[pp] = w;
    }
    wait_all_but_one_tile();  // V landed, the next K in flight
    u32x2_t vlo[2 * NT][DTILES], vhi[2 * NT][DTILES];
#pragma unroll
    for (int pp = 0; pp < 2 * NT; ++pp) {
      const int kk = 16 * pp + 4 * (grp16 >> 1);  // first key of run 1
#pragma unroll
      for (int dt = 0; dt < DTILES; ++dt) {
        const int d0 = dt * 32 + 16 * (grp16 & 1) + 4 * tr_cb;  // source column of this lane
        const int cc = d0 >> 3, sub = (d0 & 7) * 2;
        const int r1 = kk + tr_row, r2 = r1 + 8;
        vlo[pp][dt] = ds_read_tr16_b64((const void*)(vS + r1 * ROWB + swz_v<D>(r1, cc) * 16 + sub));
        vhi[pp][dt] = ds_read_tr16_b64((const void*)(vS + r2 * ROWB + swz_v<D>(r2, cc) * 16 + sub));
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (moved[t]) {
#pragma unroll
        for (int dt = 0; dt < DTILES; ++dt) oacc[dt] *= alpha[t];
      }
#pragma unroll
      for (int pp = 2 * t; pp < 2 * t + 2; ++pp)
#pragma unroll
        for (int dt = 0; dt < DTILES; ++dt) {
          const u32x4_t a = {vlo[pp][dt][0], vlo[pp][dt][1], vhi[pp][dt][0], vhi[pp][dt][1]};
          oacc[dt] = mfma16<DT>(a, pb[pp], oacc[dt]);
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) kb[t] = kb_next[t];
  }
  // No DMA into this workgroup's LDS outlives it, and the reads of the V tile are done.
  __builtin_amdgcn_s_waitcnt(0x0070);
  asm volatile("" ::: "memory");

  const float l_tot = pair_sum32(l_run);
  const float inv = 1.f / (l_tot > 0.f ? l_tot : 1.f);  // empty rows: O = 0; NaN rows stay NaN
  // The output through the V tile, so that whole rows leave: 16-byte chunk c of row r at
  // position c ^ (r mod chunks). One wave's LDS accesses execute in order.
  constexpr int CPR = ROWB / 16;
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      const int d0 = dt * 32 + 8 * gq + 4 * half;
      const u32x2_t w = {pack16x2<DT>(oacc[dt][4 * gq + 0] * inv, oacc[dt][4 * gq + 1] * inv),
                         pack16x2<DT>(oacc[dt][4 * gq + 2] * inv, oacc[dt][4 * gq + 3] * inv)};
      *(u32x2_t*)(vS + col * ROWB + (((d0 >> 3) ^ (col & (CPR - 1))) << 4) + (d0 & 7) * 2) = w;
    }
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < BS * CPR / kWave; ++j) {
    const int r = j * (kWave / CPR) + lane / CPR, c = lane % CPR;
    const u32x4_t v = *(const u32x4_t*)(vS + r * ROWB + ((c ^ (r & (CPR - 1))) << 4));
    // Non-temporal: the output is not read again here, and K/V stay in L2.
    if (qb * BS + r < S)
      __builtin_nontemporal_store(v, (u32x4_t*)(obase + (int64_t)(qb * BS + r) * p.so[2] + c * 8));
  }
}

template <int D, int NT, int DT>
static hipError_t launch_prefill_bs32(const PrefillParams& p, hipStream_t stream) {
  const int64_t grid = (int64_t)p.NB * p.B * p.Hq;
  if (p.small_spans && p.small_q)
    hipLaunchKernelGGL((bsfa_prefill_bs32_kernel<D, NT, DT, true>), dim3((unsigned)grid), dim3(kWave), 0, stream, p);
  else
    hipLaunchKernelGGL((bsfa_prefill_bs32_kernel<D, NT, DT, false>), dim3((unsigned)grid), dim3(kWave), 0, stream, p);
  return hipGetLastError();
}

template <int D, int DT>
static hipError_t launch_prefill_bs64(const PrefillParams& p, hipStream_t stream) {
  const int64_t grid = (int64_t)p.NB * p.B * p.Hq;
  // Two pairs of waves per row fill the card with two workgroups per CU at head dim 128, 512
  // rows; with more, rows wait for a second fill (640 rows of S=1280 16.8 us against 15.6,
  // 1024 of S=2048 24.1 against 22.7; rows of 80 blocks and more still gain, up to 1024 of
  // them and not with few active blocks). At head dim 64 three fit, and up to 1024 rows it is
  // no slower (S=2048 16.4 us both, S=4096 23.2 against 27.5; 1536 rows of S=6144 with few
  // active blocks 22.5 against 21.6). Rows of fewer than 8 blocks have nothing to share out
  // (D=128, S=256 8.8 us against 8.4, S=512 10.7 against 11.6).
  if (grid <= (D == 128 ? 512 : 1024) && p.NB >= 8)
    hipLaunchKernelGGL((bsfa_prefill_bs64_2w_kernel<D, DT, 2>), dim3((unsigned)grid), dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((bsfa_prefill_bs64_2w_kernel<D, DT, 1>), dim3((unsigned)grid), dim3(128), 0, stream, p);
  return hipGetLastError();
}

static bool aligned16(const void* ptr) { return ((uintptr_t)ptr & 15u) == 0; }

// At head dim 128 the kernels of blocks 64 and 128 end a tensor's buffer `rows left` token
// strides after a tile's first row, and their per-lane offsets count on whole rows before
// each unit: rows closer than the head dim (0: one row repeated) would arrive as zeros.
static bool rows_overlap(int64_t head_dim, int64_t block_size, int64_t q_token, int64_t k_token,
                         int64_t v_token) {
  return head_dim == 128 && block_size != 32 && std::min({q_token, k_token, v_token}) < head_dim;
}

template <int DT>
static hipError_t launch_prefill_any(const PrefillParams& p, int64_t head_dim,
                                     int64_t block_size, hipStream_t s) {
  if (block_size == 128 && (head_dim == 128 || head_dim == 64)) {
    // A block-128 mask on the block-64 kernels: each 128-token block is its four 64-token
    // quarters, read through the mask index shift. The same tokens attend to the same
    // keys; the online softmax merely visits them in 64-key steps (2.7x faster than
    // the generic block-128 kernel at config-2 geometry).
    PrefillParams q = p;
    q.mshift = 1;
    q.NB = (p.S + 63) / 64;
    return head_dim == 128 ? launch_prefill_bs64<128, DT>(q, s)
                           : launch_prefill_bs64<64, DT>(q, s);
  }
  if (block_size == 64 && head_dim == 128) return launch_prefill_bs64<128, DT>(p, s);
  if (block_size == 64 && head_dim == 64) return launch_prefill_bs64<64, DT>(p, s);
  if (head_dim == 128) return launch_prefill_bs32<128, 1, DT>(p, s);  // block 32
  return launch_prefill_bs32<64, 2, DT>(p, s);
}

}  // namespace tasft

using namespace tasft;

static int dispatch_prefill(const PrefillParams& p, int64_t head_dim,
                            int64_t block_size, int dtype, hipStream_t s, const char* what) {
  const hipError_t err = dtype == kF16 ? launch_prefill_any<kF16>(p, head_dim, block_size, s)
                                       : launch_prefill_any<kBf16>(p, head_dim, block_size, s);
  if (err != hipSuccess)
    return set_error(kErrLaunch, "%s: launch failed: %s", what, hipGetErrorString(err));
  return kOk;
}

extern "C" size_t tasft_bsfa_prefill_workspace_bytes(int64_t batch, int64_t num_q_heads,
                                                     int64_t seq_len, int64_t block_size) {
  if (batch <= 0 || num_q_heads <= 0 || seq_len <= 0 || block_size <= 0) return 0;
  return 256;  // kept for callers that pass one; no kernel uses it
}

extern "C" int tasft_bsfa_prefill_fwd(const void* q, const void* k, const void* v, void* out,
                                      const uint8_t* block_mask, void* workspace,
                                      size_t workspace_bytes, int64_t batch,
                                      int64_t num_q_heads, int64_t num_kv_heads, int64_t seq_len,
                                      int64_t head_dim, int64_t block_size,
                                      const int64_t* q_strides, const int64_t* k_strides,
                                      const int64_t* v_strides, const int64_t* o_strides,
                                      const int64_t* mask_strides, float scale, int causal,
                                      int dtype, void* stream) {
  if (!q || !k || !v || !out || !block_mask || !q_strides || !k_strides || !v_strides ||
      !o_strides || !mask_strides)
    return set_error(kErrInvalidArgument, "prefill: null pointer argument");
  if (dtype != kBf16 && dtype != kF16)
    return set_error(kErrUnsupported, "prefill: dtype must be bf16 (0) or fp16 (1), got %d", dtype);
  if (batch <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || seq_len <= 0)
    return set_error(kErrInvalidArgument, "prefill: batch, heads and seq_len must be positive");
  if (num_q_heads % num_kv_heads != 0)
    return set_error(kErrInvalidArgument,
                     "prefill: num_q_heads (%lld) must be a multiple of num_kv_heads (%lld)",
                     (long long)num_q_heads, (long long)num_kv_heads);
  if (head_dim != 64 && head_dim != 128)
    return set_error(kErrUnsupported, "prefill: head_dim must be 64 or 128, got %lld",
                     (long long)head_dim);
  if (block_size != 32 && block_size != 64 && block_size != 128)
    return set_error(kErrUnsupported, "prefill: block_size must be 32, 64 or 128, got %lld",
                     (long long)block_size);
  const int64_t* st[4] = {q_strides, k_strides, v_strides, o_strides};
  if (!strides_nonneg(q_strides, 4) || !strides_nonneg(k_strides, 4) ||
      !strides_nonneg(v_strides, 4) || !strides_nonneg(o_strides, 4) ||
      !strides_nonneg(mask_strides, 4))
    return set_error(kErrInvalidArgument, "prefill: strides must be non-negative");
  for (int i = 0; i < 4; ++i) {
    if (st[i][3] != 1)
      return set_error(kErrInvalidArgument, "prefill: head_dim must be the contiguous dimension");
    for (int j = 0; j < 3; ++j)
      if (st[i][j] % 8 != 0)
        return set_error(kErrInvalidArgument,
                         "prefill: strides must be multiples of 8 elements (16-byte rows)");
  }
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out))
    return set_error(kErrInvalidArgument, "prefill: tensors must be 16-byte aligned");
  const int64_t nb = (seq_len + block_size - 1) / block_size;
  // Block 128 runs on the block-64 kernels (launch_prefill_any): twice the query blocks.
  if (nb * (block_size == 128 ? 2 : 1) * batch * num_q_heads > 0x7fffffffLL ||
      seq_len > 0x3fffffffLL)
    return set_error(kErrUnsupported, "prefill: problem too large for one launch");
  const size_t ws_need = tasft_bsfa_prefill_workspace_bytes(batch, num_q_heads, seq_len, block_size);
  if (workspace) {
    if (workspace_bytes < ws_need)
      return set_error(kErrWorkspace, "prefill: workspace too small: need %zu bytes, got %zu",
                       ws_need, workspace_bytes);
    if (((uintptr_t)workspace) & 15u)
      return set_error(kErrInvalidArgument, "prefill: workspace must be 16-byte aligned");
  }
  if (rows_overlap(head_dim, block_size, q_strides[2], k_strides[2], v_strides[2]))
    return set_error(kErrInvalidArgument,
                     "prefill: at head_dim 128 and block_size 64 or 128 the token strides of q, k "
                     "and v must be at least head_dim");

  PrefillParams p;
  p.q = (const uint16_t*)q;
  p.k = (const uint16_t*)k;
  p.v = (const uint16_t*)v;
  p.o = (uint16_t*)out;
  p.mask = block_mask;
  for (int j = 0; j < 3; ++j) {
    p.sq[j] = q_strides[j];
    p.sk[j] = k_strides[j];
    p.sv[j] = v_strides[j];
    p.so[j] = o_strides[j];
  }
  for (int j = 0; j < 4; ++j) p.sm[j] = mask_strides[j];
  p.B = (int)batch;
  p.Hq = (int)num_q_heads;
  p.Hkv = (int)num_kv_heads;
  p.G = (int)(num_q_heads / num_kv_heads);
  p.S = (int)seq_len;
  p.NB = (int)nb;
  p.scale_log2 = scale * kLog2e;
  p.causal = causal ? 1 : 0;
  p.small_spans = (seq_len * k_strides[2] * 2 < 0x7fffffffLL &&
                   seq_len * v_strides[2] * 2 < 0x7fffffffLL) ? 1 : 0;
  p.small_q = seq_len * q_strides[2] * 2 < 0x7fffffffLL ? 1 : 0;
  p.cu_seqlens = nullptr;
  p.mshift = 0;
  return dispatch_prefill(p, head_dim, block_size, dtype, (hipStream_t)stream,
                          "prefill");
}

namespace tasft {

// Zeroes the output rows of the tokens at or after cu_seqlens[num_seqs] of a packed
// [T, H, D] batch (rows no sequence covers), reading that offset on the device: with no
// such row (the usual case) every thread makes one check and exits. Each thread writes
// 16 bytes per step; the grid strides over the tail.
__global__ void __launch_bounds__(256)
varlen_zero_tail_kernel(uint16_t* out, const int32_t* end_ptr, int64_t T, int H, int D,
                        int64_t st_t, int64_t st_h) {
  const int64_t end = *end_ptr;
  const int64_t first = end < 0 ? 0 : (end > T ? T : end);
  const int chunks = D / 8;
  const int64_t per_row = (int64_t)H * chunks;
  const int64_t n = (T - first) * per_row;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = first + i / per_row;
    const int64_t rem = i % per_row;
    const int64_t h = rem / chunks, c = rem % chunks;
    *(u32x4_t*)(out + row * st_t + h * st_h + c * 8) = (u32x4_t){0u, 0u, 0u, 0u};
  }
}

}  // namespace tasft

extern "C" int tasft_bsfa_varlen_zero_tail(void* out, const int32_t* cu_seqlens, int64_t num_seqs,
                                           int64_t tokens, int64_t num_heads, int64_t head_dim,
                                           const int64_t* o_strides, void* stream) {
  if (!out || !cu_seqlens || !o_strides)
    return set_error(kErrInvalidArgument, "varlen_zero_tail: null pointer argument");
  if (num_seqs <= 0 || tokens < 0 || num_heads <= 0 || head_dim <= 0 || head_dim % 8 != 0)
    return set_error(kErrInvalidArgument,
                     "varlen_zero_tail: num_seqs, num_heads positive, tokens >= 0, head_dim a positive multiple of 8");
  if (!strides_nonneg(o_strides, 3) || o_strides[2] != 1 || o_strides[0] % 8 != 0 ||
      o_strides[1] % 8 != 0 || !aligned16(out))
    return set_error(kErrInvalidArgument,
                     "varlen_zero_tail: out must be 16-byte aligned with a contiguous head_dim and "
                     "token and head strides multiples of 8 elements");
  if (tokens == 0) return kOk;
  hipLaunchKernelGGL(varlen_zero_tail_kernel, dim3(256), dim3(256), 0, (hipStream_t)stream,
                     (uint16_t*)out, cu_seqlens + num_seqs, tokens, (int)num_heads, (int)head_dim,
                     o_strides[0], o_strides[1]);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess)
    return set_error(kErrLaunch, "varlen_zero_tail: launch failed: %s", hipGetErrorString(err));
  return kOk;
}

extern "C" int tasft_bsfa_prefill_varlen_fwd(const void* q, const void* k, const void* v,
                                             void* out, const uint8_t* block_mask,
                                             const int32_t* cu_seqlens, int64_t num_seqs,
                                             int64_t num_q_heads, int64_t num_kv_heads,
                                             int64_t max_seqlen, int64_t head_dim,
                                             int64_t block_size, const int64_t* q_strides,
                                             const int64_t* k_strides, const int64_t* v_strides,
                                             const int64_t* o_strides,
                                             const int64_t* mask_strides, float scale, int causal,
                                             int dtype, void* stream) {
  if (!q || !k || !v || !out || !block_mask || !cu_seqlens || !q_strides || !k_strides ||
      !v_strides || !o_strides || !mask_strides)
    return set_error(kErrInvalidArgument, "prefill_varlen: null pointer argument");
  if (dtype != kBf16 && dtype != kF16)
    return set_error(kErrUnsupported, "prefill_varlen: dtype must be bf16 (0) or fp16 (1), got %d",
                     dtype);
  if (num_seqs <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || max_seqlen <= 0)
    return set_error(kErrInvalidArgument,
                     "prefill_varlen: num_seqs, heads and max_seqlen must be positive");
  if (num_q_heads % num_kv_heads != 0)
    return set_error(kErrInvalidArgument,
                     "prefill_varlen: num_q_heads (%lld) must be a multiple of num_kv_heads (%lld)",
                     (long long)num_q_heads, (long long)num_kv_heads);
  if (head_dim != 64 && head_dim != 128)
    return set_error(kErrUnsupported, "prefill_varlen: head_dim must be 64 or 128, got %lld",
                     (long long)head_dim);
  if (block_size != 32 && block_size != 64 && block_size != 128)
    return set_error(kErrUnsupported, "prefill_varlen: block_size must be 32, 64 or 128, got %lld",
                     (long long)block_size);
  const int64_t* st[4] = {q_strides, k_strides, v_strides, o_strides};
  if (!strides_nonneg(q_strides, 3) || !strides_nonneg(k_strides, 3) ||
      !strides_nonneg(v_strides, 3) || !strides_nonneg(o_strides, 3) ||
      !strides_nonneg(mask_strides, 4))
    return set_error(kErrInvalidArgument, "prefill_varlen: strides must be non-negative");
  for (int i = 0; i < 4; ++i) {
    if (st[i][2] != 1)
      return set_error(kErrInvalidArgument,
                       "prefill_varlen: head_dim must be the contiguous dimension");
    for (int j = 0; j < 2; ++j)
      if (st[i][j] % 8 != 0)
        return set_error(kErrInvalidArgument,
                         "prefill_varlen: strides must be multiples of 8 elements (16-byte rows)");
  }
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out))
    return set_error(kErrInvalidArgument, "prefill_varlen: tensors must be 16-byte aligned");
  const int64_t nb = (max_seqlen + block_size - 1) / block_size;
  if (nb * (block_size == 128 ? 2 : 1) * num_seqs * num_q_heads > 0x7fffffffLL ||
      max_seqlen > 0x3fffffffLL)
    return set_error(kErrUnsupported, "prefill_varlen: problem too large for one launch");
  if (rows_overlap(head_dim, block_size, q_strides[0], k_strides[0], v_strides[0]))
    return set_error(kErrInvalidArgument,
                     "prefill_varlen: at head_dim 128 and block_size 64 or 128 the token strides of "
                     "q, k and v must be at least head_dim");

  PrefillParams p;
  p.q = (const uint16_t*)q;
  p.k = (const uint16_t*)k;
  p.v = (const uint16_t*)v;
  p.o = (uint16_t*)out;
  p.mask = block_mask;
  // Packed [tokens, heads, D]: no batch stride; the kernels add cu_seqlens[b] tokens.
  const int64_t* src[4] = {q_strides, k_strides, v_strides, o_strides};
  int64_t* dst[4] = {p.sq, p.sk, p.sv, p.so};
  for (int i = 0; i < 4; ++i) {
    dst[i][0] = 0;
    dst[i][1] = src[i][1];
    dst[i][2] = src[i][0];
  }
  for (int j = 0; j < 4; ++j) p.sm[j] = mask_strides[j];
  p.B = (int)num_seqs;
  p.Hq = (int)num_q_heads;
  p.Hkv = (int)num_kv_heads;
  p.G = (int)(num_q_heads / num_kv_heads);
  p.S = (int)max_seqlen;
  p.NB = (int)nb;
  p.scale_log2 = scale * kLog2e;
  p.causal = causal ? 1 : 0;
  p.small_spans = (max_seqlen * k_strides[0] * 2 < 0x7fffffffLL &&
                   max_seqlen * v_strides[0] * 2 < 0x7fffffffLL) ? 1 : 0;
  p.small_q = max_seqlen * q_strides[0] * 2 < 0x7fffffffLL ? 1 : 0;
  p.cu_seqlens = cu_seqlens;
  p.mshift = 0;
  return dispatch_prefill(p, head_dim, block_size, dtype, (hipStream_t)stream,
                          "prefill_varlen");
}
