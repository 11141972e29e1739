// Gradients of the gate's parameters for gfx950: the whole backward of a gate training step
// behind dL/dsoft.
//
// With u_i = W_q qbar_i + b_in, v_j = W_k kbar_j, pre_ijc = u_ic + v_jc,
// soft_ij = sigmoid(w . relu(pre_ij)) (0 above the block diagonal when causal) and
// g_ij = dL/dsoft_ij soft_ij (1 - soft_ij) (0 where soft was zeroed), the gradient the
// reference gets from autograd (tasft/modules/attn_gate.py:248-273) is
//   dL/dw_c  = sum_ij g_ij relu(pre_ijc)
//   du_ic    = w_c sum_j g_ij [pre_ijc > 0],   dv_jc = w_c sum_i g_ij [pre_ijc > 0]
//   dL/db    = sum_i du_i,   dL/dW_q = sum_i du_i qbar_i^T,   dL/dW_k = sum_j dv_j kbar_j^T
// over every batch entry and head (dv summed over the query heads of a KV head).
//
// Three launches, every sum in a fixed order (no atomics):
//   1. gate_grads_pair_kernel: du, dv per query head and row chunk, dL/dw per workgroup;
//   2. gate_grads_weight_kernel: du^T qbar and dv^T kbar over runs of rows on the fp32 MFMA,
//      with dv's head sum in its operand load;
//   3. gate_grads_reduce_kernel: the sums over the row chunks.
#include <algorithm>

#include "common.h"

#include "../../include/tasft_amd.h"

namespace tasft {

constexpr int kGradUnits = 64;  // hidden units per workgroup: one per lane
constexpr int kGradKeys = 16;   // key blocks per round
constexpr int kGradMaxI = 64;   // query blocks per workgroup, at most
constexpr int kGradDims = 64;   // head dims of one partial weight product
constexpr int kGradBatch = 8;   // k-steps (4 rows) loaded ahead

struct GateGradParams {
  const float* uq;         // [B, Hq, NB, hidden]
  const float* uk;         // [B, Hkv, NB, hidden]
  const float* soft;       // [B, Hq, NB, NB]
  const float* grad_soft;  // [B, Hq, NB, NB]
  const float* qmeans;     // [B, Hq, NB, D]
  const float* kmeans;     // [B, Hkv, NB, D]
  const float* w_out;      // [hidden]
  float* du;               // [B, Hq, NB, hidden]
  float* dv;               // [B, Hkv, NB, hidden]
  float* dvh;              // [ichunks, B, Hq, NB, hidden]
  float* dwo_part;         // [B * Hq * ichunks, hidden]
  float* db_part;          // [qparts, hidden]
  float* dw_part;          // [qparts + kparts, hidden, D]
  float* dw_in;            // [hidden, 2 D]
  float* db_in;            // [hidden]
  float* dw_out;           // [hidden]
  int B, Hq, Hkv, G, NB, D, hidden, causal, ic, ichunks, utiles, dtiles, qparts, kparts, qspan, kspan;
};

// Pairwise sums. A workgroup takes `ic` query blocks of one (b, head) and 64 hidden units; a
// lane is a unit, so u, v and the sums stay in its registers and g_ij is a broadcast. Rows are
// dealt to the four waves in turn (equal causal work); 16 key blocks a round sit in
// registers with their dv sums, which the waves add up through LDS after the round. Seven
// VALU operations per pair and unit bound it (about 35 us of issue at B=4, 32 heads, 128
// blocks, hidden 128): it takes 55 us there, where gate_pairwise_bwd_kernel's 32 x 32 tiles
// (separate passes for rows and columns, ten operations, partial sums per tile in memory)
// take 94 us.
__global__ void __launch_bounds__(256)
gate_grads_pair_kernel(const GateGradParams p) {
  __shared__ float u_s[kGradMaxI][kGradUnits];
  __shared__ float su_s[kGradMaxI][kGradUnits];
  __shared__ __attribute__((aligned(16))) float g_s[2][kGradMaxI][kGradKeys];
  __shared__ float sv_s[2][4][kGradKeys][kGradUnits];
  __shared__ double sw_s[4][kGradUnits];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  // Row chunks from the last (the longest rows under causal) to the first.
  const int64_t nbh = (int64_t)p.B * p.Hq;
  const int64_t per = nbh * p.utiles;
  const int chunk = p.ichunks - 1 - (int)(blockIdx.x / per);
  const int64_t bh = (blockIdx.x % per) / p.utiles;
  const int c = (int)(blockIdx.x % p.utiles) * kGradUnits + lane;
  const bool cok = c < p.hidden;
  const int b = (int)(bh / p.Hq), kvh = (int)(bh % p.Hq) / p.G;
  const int i0 = chunk * p.ic;
  const int rows = min(p.ic, p.NB - i0);
  const int hid = p.hidden;
  const float* uq = p.uq + (bh * p.NB + i0) * (int64_t)hid;
  const float* uk = p.uk + ((int64_t)b * p.Hkv + kvh) * (int64_t)p.NB * hid;
  const int64_t sbase = (bh * p.NB + i0) * (int64_t)p.NB;
  const float w = cok ? p.w_out[c] : 0.f;

  for (int r = wave; r < rows; r += 4) {
    u_s[r][lane] = cok ? uq[(int64_t)r * hid + c] : 0.f;
    su_s[r][lane] = 0.f;
  }
  double sw = 0.0;  // this wave's share of dL/dw_c
  const int jend = p.causal ? min(p.NB, i0 + rows) : p.NB;
  float* dvh = p.dvh + ((int64_t)chunk * nbh + bh) * p.NB * (int64_t)hid;
  // This thread's share of a round's g (rows tid / 16 + 16 q, key tid % 16) and the key units.
  constexpr int kGPT = kGradMaxI * kGradKeys / 256;
  const int gr = tid / kGradKeys, gj = tid % kGradKeys;
  float g[kGPT], v[kGradKeys], vn[kGradKeys];
  auto load_g = [&](int j0) {
    const int j = j0 + gj;
#pragma unroll
    for (int q = 0; q < kGPT; ++q) {
      const int r = gr + 16 * q;
      g[q] = 0.f;
      if (r < rows && j < p.NB && !(p.causal && j > i0 + r)) {
        const int64_t o = sbase + (int64_t)r * p.NB + j;
        const float s = p.soft[o];
        g[q] = p.grad_soft[o] * s * (1.f - s);
      }
    }
  };
  auto load_v = [&](int j0) {
#pragma unroll
    for (int jj = 0; jj < kGradKeys; ++jj)
      vn[jj] = uk[(int64_t)min(j0 + jj, p.NB - 1) * hid + (cok ? c : 0)];
  };
  auto store_g = [&](int buf) {
#pragma unroll
    for (int q = 0; q < kGPT; ++q) g_s[buf][gr + 16 * q][gj] = g[q];
  };
  // One barrier a round: the next round's g and this round's dv sums go to the other halves
  // of their buffers, whose last readers passed the barrier before.
  load_g(0);
  load_v(0);
  store_g(0);
  __syncthreads();
  int buf = 0;
  for (int j0 = 0; j0 < jend; j0 += kGradKeys, buf ^= 1) {
    float sv[kGradKeys];
#pragma unroll
    for (int jj = 0; jj < kGradKeys; ++jj) {
      v[jj] = vn[jj];  // g = 0 for the keys past the end
      sv[jj] = 0.f;
    }
    const bool more = j0 + kGradKeys < jend;
    if (more) {
      load_g(j0 + kGradKeys);
      load_v(j0 + kGradKeys);
    }
    // Rows above every key of the round have g = 0 throughout.
    const int r0 = p.causal ? max(0, j0 - i0) : 0;
    for (int r = wave + ((r0 - wave + 3) & ~3); r < rows; r += 4) {
      const float u = u_s[r][lane];
      float su = 0.f, sl = 0.f;
#pragma unroll
      for (int q4 = 0; q4 < kGradKeys; q4 += 4) {
        const f32x4_t g4 = *(const f32x4_t*)&g_s[buf][r][q4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float act = fmaxf(u + v[q4 + e], 0.f);
          const float t = act > 0.f ? g4[e] : 0.f;
          sl = fmaf(g4[e], act, sl);
          su += t;
          sv[q4 + e] += t;
        }
      }
      su_s[r][lane] += su;
      sw += (double)sl;
    }
#pragma unroll
    for (int jj = 0; jj < kGradKeys; ++jj) sv_s[buf][wave][jj][lane] = sv[jj];
    if (more) store_g(buf ^ 1);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kGradKeys / 4; ++q) {
      const int jj = 4 * q + wave;
      if (cok && j0 + jj < p.NB)
        dvh[(int64_t)(j0 + jj) * hid + c] = w * ((sv_s[buf][0][jj][lane] + sv_s[buf][1][jj][lane]) +
                                                 (sv_s[buf][2][jj][lane] + sv_s[buf][3][jj][lane]));
    }
  }
  // Key blocks no row of this chunk reaches.
  for (int j = ((jend + kGradKeys - 1) / kGradKeys) * kGradKeys + wave; j < p.NB; j += 4)
    if (cok) dvh[(int64_t)j * hid + c] = 0.f;
  float* du = p.du + (bh * p.NB + i0) * (int64_t)hid;
  for (int r = wave; r < rows; r += 4)
    if (cok) du[(int64_t)r * hid + c] = w * su_s[r][lane];
  sw_s[wave][lane] = sw;
  __syncthreads();
  if (wave == 0 && cok)
    p.dwo_part[(bh * p.ichunks + chunk) * (int64_t)hid + c] =
        (float)((sw_s[0][lane] + sw_s[1][lane]) + (sw_s[2][lane] + sw_s[3][lane]));
}

// One partial weight product: 64 hidden units x 64 head dims over a run of rows of du (or dv)
// and of the block means. v_mfma_f32_16x16x4_f32 with M = units (16 per wave), N = dims,
// K = rows: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and receives
// D[4 (l / 16) + r][l % 16]. The rows past the end, the units past `hidden` and the dims past
// D are zeros. Loads of kGradBatch k-steps are in flight together: the operands come from L2
// in 64-byte pieces, whose latency bounds the kernel. B=4, 32/8 heads, 128 blocks, hidden 128,
// D=128: 24 us, and 6 us for the reduction below (32-dim tiles, which read du and dv twice as
// often, 30 us; torch's sums over the tiles and batched products before this took about 130 us
// in some fifteen launches).
__global__ void __launch_bounds__(256)
gate_grads_weight_kernel(const GateGradParams p) {
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const int lr = lane % 16, lq = lane / 16;
  const int tiles = p.utiles * p.dtiles;
  const int part = (int)(blockIdx.x / tiles), tile = (int)(blockIdx.x % tiles);
  const int c = (tile / p.dtiles) * kGradUnits + wave * 16 + lr;  // A's unit of this lane
  const int d0 = (tile % p.dtiles) * kGradDims;
  const bool is_q = part < p.qparts;
  const int hid = p.hidden, D = p.D;
  const bool cok = c < hid;
  const int rows = p.B * (is_q ? p.Hq : p.Hkv) * p.NB;
  const int span = is_q ? p.qspan : p.kspan;
  const int r_begin = (is_q ? part : part - p.qparts) * span;
  const int r_end = min(r_begin + span, rows);
  const float* m = is_q ? p.qmeans : p.kmeans;
  const int64_t plane = (int64_t)p.B * p.Hq * p.NB * hid;
  constexpr int NT = kGradDims / 16;  // 16-dim tiles
  bool dok[NT];
  f32x4_t acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    dok[n] = d0 + 16 * n + lr < D;
    acc[n] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  }
  float bsum = 0.f;
  for (int r0 = r_begin; r0 < r_end; r0 += 4 * kGradBatch) {
    float a[kGradBatch], bm[kGradBatch][NT];
#pragma unroll
    for (int s = 0; s < kGradBatch; ++s) {
      const int r = r0 + 4 * s + lq;
      const bool rok = r < r_end;
#pragma unroll
      for (int n = 0; n < NT; ++n)
        bm[s][n] = (rok && dok[n]) ? m[(int64_t)r * D + d0 + 16 * n + lr] : 0.f;
      a[s] = (is_q && rok && cok) ? p.du[(int64_t)r * hid + c] : 0.f;
    }
    if (!is_q) {
      // dv of a KV head: its query heads' sums over the row chunks, in order.
      const float* src[kGradBatch];
#pragma unroll
      for (int s = 0; s < kGradBatch; ++s) {
        const int r = min(r0 + 4 * s + lq, r_end - 1);
        const int bkv = r / p.NB, j = r % p.NB;
        const int bh = (bkv / p.Hkv) * p.Hq + (bkv % p.Hkv) * p.G;
        src[s] = p.dvh + ((int64_t)bh * p.NB + j) * hid + (cok ? c : 0);
      }
      // Four addends per row at a time, all loaded before the first is added.
      const int n = p.G * p.ichunks;
      int64_t off = 0;  // of addend (head g, chunk ch)
      int ch = 0;
      for (int e0 = 0; e0 < n; e0 += 4) {
        float t[4][kGradBatch];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int s = 0; s < kGradBatch; ++s) t[e][s] = src[s][off];
          if (e0 + e + 1 < n) {  // the last addend is loaded again past the end
            ++ch;
            off += plane;
            if (ch == p.ichunks) {
              ch = 0;
              off += (int64_t)p.NB * hid - p.ichunks * plane;
            }
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int s = 0; s < kGradBatch; ++s) a[s] += e0 + e < n ? t[e][s] : 0.f;
      }
#pragma unroll
      for (int s = 0; s < kGradBatch; ++s) {
        const int r = r0 + 4 * s + lq;
        const bool ok = cok && r < r_end;
        a[s] = ok ? a[s] : 0.f;
        if (ok && d0 == 0) p.dv[(int64_t)r * hid + c] = a[s];
      }
    }
#pragma unroll
    for (int s = 0; s < kGradBatch; ++s) {
      bsum += a[s];
#pragma unroll
      for (int n = 0; n < NT; ++n)
        acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], bm[s][n], acc[n], 0, 0, 0);
    }
  }
  float* out = p.dw_part + (int64_t)part * hid * D;
  const int c_out = (tile / p.dtiles) * kGradUnits + wave * 16 + 4 * lq;
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (dok[n] && c_out + e < hid) out[(int64_t)(c_out + e) * D + d0 + 16 * n + lr] = acc[n][e];
  if (is_q && d0 == 0) {
    bsum += __shfl_xor(bsum, 16, kWave);
    bsum += __shfl_xor(bsum, 32, kWave);
    if (lq == 0 && cok) p.db_part[(int64_t)part * hid + c] = bsum;
  }
}

// The sums over the partials: 64 outputs per workgroup, each by four threads (64-bit sums, a
// quarter of the partials each). Outputs: dW_in [hidden][2 D], then db_in and dw_out.
__global__ void __launch_bounds__(256)
gate_grads_reduce_kernel(const GateGradParams p) {
  __shared__ double red[4][64];
  const int o = threadIdx.x % 64, sl = threadIdx.x / 64;
  const int D = p.D, hid = p.hidden;
  const int64_t n_w = (int64_t)hid * 2 * D;
  const int64_t idx = (int64_t)blockIdx.x * 64 + o;
  const float* src = nullptr;
  float* dst = nullptr;
  int64_t stride = hid;
  int count = 0;
  if (idx < n_w) {
    const int c = (int)(idx / (2 * D)), d = (int)(idx % (2 * D));
    const bool is_q = d < D;
    stride = (int64_t)hid * D;
    src = p.dw_part + (is_q ? 0 : p.qparts * stride) + (int64_t)c * D + (is_q ? d : d - D);
    count = is_q ? p.qparts : p.kparts;
    dst = p.dw_in + idx;
  } else if (idx < n_w + hid) {
    src = p.db_part + (idx - n_w);
    count = p.qparts;
    dst = p.db_in + (idx - n_w);
  } else if (idx < n_w + 2 * hid) {
    src = p.dwo_part + (idx - n_w - hid);
    count = p.B * p.Hq * p.ichunks;
    dst = p.dw_out + (idx - n_w - hid);
  }
  double acc = 0.0;
#pragma unroll 8
  for (int i = sl; i < count; i += 4) acc += (double)src[i * stride];
  red[sl][o] = acc;
  __syncthreads();
  if (sl == 0 && dst) *dst = (float)((red[0][o] + red[1][o]) + (red[2][o] + red[3][o]));
}

// Workgroups of the weight products of du (and as many of dv), at least: two per CU.
constexpr int64_t kGradGroups = 512;
// Rows of a partial product, at most: a run is one serial fp32 sum, and its length sets the
// rounding error whatever the batch (the partial products are added up in 64 bits).
constexpr int64_t kGradRun = 128;

// Sizes of a call: row chunks of 64 query blocks, fewer rows (down to 16) while the launch
// would leave CUs without a workgroup.
struct GateGradPlan {
  int64_t nb, ic, ichunks, utiles, dtiles, qparts, kparts, qspan, kspan;
  int64_t n_du, n_dv, n_dvh, n_dwo, n_db, n_dw;  // floats
};

static GateGradPlan gate_grad_plan(int64_t B, int64_t Hq, int64_t Hkv, int64_t S, int64_t D,
                                   int64_t bs, int64_t hidden) {
  GateGradPlan g;
  g.nb = (S + bs - 1) / bs;
  g.utiles = (hidden + kGradUnits - 1) / kGradUnits;
  g.dtiles = (D + kGradDims - 1) / kGradDims;
  g.ic = kGradMaxI;
  while (g.ic > 16 && B * Hq * g.utiles * ((g.nb + g.ic - 1) / g.ic) < 256) g.ic /= 2;
  g.ichunks = (g.nb + g.ic - 1) / g.ic;
  const int64_t tiles = g.utiles * g.dtiles;
  auto split = [&](int64_t rows, int64_t* parts, int64_t* span) {
    const int64_t want = std::max<int64_t>(1, kGradGroups / tiles);
    const int64_t batch = 4 * kGradBatch;
    *span = std::min(((rows + want - 1) / want + batch - 1) / batch * batch, kGradRun);
    *parts = (rows + *span - 1) / *span;
  };
  split(B * Hq * g.nb, &g.qparts, &g.qspan);
  split(B * Hkv * g.nb, &g.kparts, &g.kspan);
  g.n_du = B * Hq * g.nb * hidden;
  g.n_dv = B * Hkv * g.nb * hidden;
  g.n_dvh = g.ichunks * g.n_du;
  g.n_dwo = B * Hq * g.ichunks * hidden;
  g.n_db = g.qparts * hidden;
  g.n_dw = (g.qparts + g.kparts) * hidden * D;
  return g;
}

}  // namespace tasft

using namespace tasft;

extern "C" size_t tasft_gate_grads_workspace_bytes(int64_t batch, int64_t num_q_heads,
                                                   int64_t num_kv_heads, int64_t seq_len,
                                                   int64_t head_dim, int64_t block_size,
                                                   int64_t hidden) {
  if (batch <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || seq_len <= 0 || head_dim <= 0 ||
      block_size <= 0 || hidden <= 0)
    return 0;
  const GateGradPlan g = gate_grad_plan(batch, num_q_heads, num_kv_heads, seq_len, head_dim,
                                        block_size, hidden);
  return (size_t)(g.n_dvh + g.n_dwo + g.n_db + g.n_dw) * sizeof(float);
}

extern "C" int tasft_gate_grads(const float* soft_scores, const float* grad_soft,
                                const void* fwd_workspace, size_t fwd_workspace_bytes,
                                const float* q_means, const float* k_means, const float* w_out,
                                float* du, float* dv, float* dw_in, float* db_in, float* dw_out,
                                void* workspace, size_t workspace_bytes, int64_t batch,
                                int64_t num_q_heads, int64_t num_kv_heads, int64_t seq_len,
                                int64_t head_dim, int64_t block_size, int64_t hidden, int flags,
                                void* stream) {
  if (!soft_scores || !grad_soft || !fwd_workspace || !q_means || !k_means || !w_out || !du ||
      !dv || !dw_in || !db_in || !dw_out || !workspace)
    return set_error(kErrInvalidArgument, "gate_grads: null pointer argument");
  if (batch <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || seq_len <= 0 || head_dim <= 0 ||
      block_size <= 0 || hidden <= 0)
    return set_error(kErrInvalidArgument, "gate_grads: sizes must be positive");
  if (num_q_heads % num_kv_heads != 0)
    return set_error(kErrInvalidArgument, "gate_grads: num_q_heads must be a multiple of num_kv_heads");
  if (head_dim > 256)
    return set_error(kErrUnsupported, "gate_grads: head_dim must be at most 256, got %lld",
                     (long long)head_dim);
  const size_t fwd_need = tasft_gate_workspace_bytes(batch, num_q_heads, num_kv_heads, seq_len,
                                                     head_dim, block_size, hidden);
  if (fwd_workspace_bytes < fwd_need)
    return set_error(kErrWorkspace, "gate_grads: forward workspace too small: need %zu bytes, got %zu",
                     fwd_need, fwd_workspace_bytes);
  const size_t need = tasft_gate_grads_workspace_bytes(batch, num_q_heads, num_kv_heads, seq_len,
                                                       head_dim, block_size, hidden);
  if (workspace_bytes < need)
    return set_error(kErrWorkspace, "gate_grads: workspace too small: need %zu bytes, got %zu", need,
                     workspace_bytes);
  const GateGradPlan g = gate_grad_plan(batch, num_q_heads, num_kv_heads, seq_len, head_dim,
                                        block_size, hidden);
  const int64_t grid1 = batch * num_q_heads * g.utiles * g.ichunks;
  const int64_t grid2 = (g.qparts + g.kparts) * g.utiles * g.dtiles;
  const int64_t grid3 = (hidden * 2 * head_dim + 2 * hidden + 63) / 64;
  if (batch * num_q_heads * g.nb > 0x7fffffffLL || grid1 > 0x7fffffffLL || grid2 > 0x7fffffffLL || grid3 > 0x7fffffffLL)
    return set_error(kErrUnsupported, "gate_grads: problem too large for one launch");

  GateGradParams p;
  p.uq = (const float*)fwd_workspace;
  p.uk = p.uq + g.n_du;
  p.soft = soft_scores;
  p.grad_soft = grad_soft;
  p.qmeans = q_means;
  p.kmeans = k_means;
  p.w_out = w_out;
  p.du = du;
  p.dv = dv;
  p.dvh = (float*)workspace;
  p.dwo_part = p.dvh + g.n_dvh;
  p.db_part = p.dwo_part + g.n_dwo;
  p.dw_part = p.db_part + g.n_db;
  p.dw_in = dw_in;
  p.db_in = db_in;
  p.dw_out = dw_out;
  p.B = (int)batch;
  p.Hq = (int)num_q_heads;
  p.Hkv = (int)num_kv_heads;
  p.G = (int)(num_q_heads / num_kv_heads);
  p.NB = (int)g.nb;
  p.D = (int)head_dim;
  p.hidden = (int)hidden;
  p.causal = (flags & TASFT_GATE_CAUSAL) ? 1 : 0;
  p.ic = (int)g.ic;
  p.ichunks = (int)g.ichunks;
  p.utiles = (int)g.utiles;
  p.dtiles = (int)g.dtiles;
  p.qparts = (int)g.qparts;
  p.kparts = (int)g.kparts;
  p.qspan = (int)g.qspan;
  p.kspan = (int)g.kspan;

  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(gate_grads_pair_kernel, dim3((unsigned)grid1), dim3(256), 0, s, p);
  hipError_t err = hipGetLastError();
  if (err == hipSuccess) {
    hipLaunchKernelGGL(gate_grads_weight_kernel, dim3((unsigned)grid2), dim3(256), 0, s, p);
    err = hipGetLastError();
  }
  if (err == hipSuccess) {
    hipLaunchKernelGGL(gate_grads_reduce_kernel, dim3((unsigned)grid3), dim3(256), 0, s, p);
    err = hipGetLastError();
  }
  if (err != hipSuccess)
    return set_error(kErrLaunch, "gate_grads: launch failed: %s", hipGetErrorString(err));
  return kOk;
}
