// The thinker's attention mixers for decode and short prefills on gfx950:
//
//   kda_prep_kernel / kda_recurrent_kernel
//                          Kimi delta attention, the recurrent form fla's fused_recurrent_kda computes (called at
//                          engine.py:258 and inside the model's KDA layers): per head a [K, V] fp32 state, per token
//                          q, k l2-normalised (q scaled), a per-key-channel decay exp(g) from the gate, the delta
//                          rule update and the readout. The per-token inputs are prepared for all tokens at once
//                          into a workspace; then a wave holds 4 value columns of one head's state in registers
//                          for all T tokens (the columns are independent), the sums over k go through lanes in a
//                          fixed order and the inputs through LDS 16 tokens at a time.
//   kda_short_kernel       the same recurrence for up to 2 tokens (a decode step) in one launch: a workgroup holds
//                          16 value columns, the sums over k go through lanes, then LDS.
//   short_conv_kernel      the depthwise causal convolution of ShortConvolution's step form (a cache of the last W
//                          inputs per channel), SiLU, T tokens in parallel.
//   rms_norm_gated_kernel  FusedRMSNormGated with a sigmoid gate: bf16(x * rsqrt(mean(x^2) + eps) * w * sigmoid(g)).
//   kda_token_kernel       one decode token of a KDA layer's core (the three above plus the gate's LoRA
//                          up-projections) in one launch, one workgroup per head.
//   mla_split_kernel / mla_merge_kernel
//                          single-token attention of an MLA layer over its static cache (engine.py:523-548: k, v
//                          [heads, max_len, d], rows written at the position with index_copy_): the new k, v rows
//                          are stored at pos, then softmax(scale q . K[0..pos]^T) . V[0..pos] in two passes
//                          (32-position chunks, then a merge of the chunks' softmax states), all in fp32.
#include "mm_common.h"

namespace {

using namespace mmd;

__device__ __forceinline__ float bf_lo(uint32_t x) { return __uint_as_float(x << 16); }
// v, or zero when !ok (a select per dword, no branch)
__device__ __forceinline__ uint4 and_mask16(const uint4& v, bool ok) {
  const uint32_t m = ok ? ~0u : 0u;
  return make_uint4(v.x & m, v.y & m, v.z & m, v.w & m);
}
__device__ __forceinline__ float bf_hi(uint32_t x) { return __uint_as_float(x & 0xffff0000u); }

// Orders a wave's LDS stores before its later loads (and loads before later stores) without a workgroup barrier:
// a wave's LDS instructions execute in program order, so only the compiler's reordering has to be fenced.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The LDS address of a pointer into shared memory, as LDS instructions take it.
__device__ __forceinline__ uint32_t lds_place(const char* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)p));
}

// Every LDS read of the wave has returned (and none moves past): its source may be overwritten.
__device__ __forceinline__ void wait_lgkm0() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (0x7 << 4) | (0 << 8));
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------------------------------------------------- KDA

struct KdaArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const void* g;
  const void* beta;
  int g_dtype, beta_dtype;
  int64_t q_ts, k_ts, v_ts, g_ts, b_ts;  // token strides (elements); head h at h * K (q, k, g), h * V (v), h (beta)
  const float* A_log;                      // [H]
  const float* dt_bias;                    // [H * K]
  float lower_bound;                       // NaN: the softplus gate
  int use_l2norm, use_gate, beta_logits;
  float scale;
  float* state;                            // [H, K, V] fp32, updated in place
  uint16_t* o;                             // [T, H, V] bf16
  int64_t o_ts;
  int T, H, V;
  const int64_t* n_valid;                  // device scalar or null: tokens from n_valid on are padding
};

// The prompt's real tokens: the first n_valid (clamped to [0, T]) when given, else all T. A padding token leaves the
// state exactly as it is: its decay is 1 and its write strength 0 (engine.py:252-253, the padded prefill).
__device__ __forceinline__ int kda_valid(const KdaArgs& a) {
  if (!a.n_valid) return a.T;
  const int64_t n = *a.n_valid;
  return static_cast<int>(n < 0 ? 0 : n > a.T ? a.T : n);
}

__device__ __forceinline__ float ld_any(const void* p, int dt, int64_t i) {
  return dt == MM_BF16 ? bf16_to_f32(static_cast<const uint16_t*>(p)[i]) : static_cast<const float*>(p)[i];
}

// softplus with the usual threshold: x above 20 returns x
__device__ __forceinline__ float softplus20(float x) { return x > 20.f ? x : log1pf(__expf(x)); }

constexpr int kKdaCols = 16;   // value columns per workgroup of kda_short_kernel and kda_token_kernel
constexpr int kKdaChunk = 16;  // tokens kda_recurrent_kernel stages in LDS at a time
constexpr int kKdaShortT = 2;  // prompts up to this long take kda_short_kernel (one launch, no workspace)
// kda_recurrent_kernel's shape: 4 state rows per lane, 4 waves per workgroup. At 16 heads of 128 x 128 that is 256
// workgroups of 4 waves, one per CU and one wave per SIMD (graph-timed over 21 states, 512 / 128 / 16 tokens:
// 114 / 36 / 11 us per call, against 146 / 44 / 13 with 8 rows per lane and one wave per workgroup, 125-133 / 38-41
// with 8 rows and 2 or 4 waves or 4 rows and 2 waves).
constexpr int kKdaRpl = 4, kKdaNwb = 4;

// Prompts of up to kKdaShortT tokens (a decode step) in one launch, without the workspace: grid (V / 16, H) x 256
// threads; each value column of the recurrence is independent (u and o of column v read
// only column v of S), so a head's columns spread over V / 16 workgroups. Wave w, lane (rg = lane / 16,
// c = lane % 16) holds state rows r = 16 i + 4 w + rg (i < K / 16) of column 16 * blockIdx.x + c: one load of a
// wave reads 4 rows x 64 bytes. Per token the first K threads (whole waves) put each key channel's q, k and decay
// into LDS, once for the workgroup, with the sums of q^2 and k^2. Sums over rows: lane-internal, then over the
// 4 row groups of a wave (xor 16, then 32), then over the 4 waves through LDS, in a fixed order.
template <int K>
__global__ __launch_bounds__(256) void kda_short_kernel(KdaArgs a) {
  constexpr int CB = kKdaCols, RPT = K / 16;
  static_assert(K % kWave == 0 && K <= 256, "kda key dim");
  __shared__ float s_q[K], s_k[K], s_dec[K];
  __shared__ float s_red[K / kWave][2];
  __shared__ float part_u[4][CB], part_o[4][CB];
  const int h = blockIdx.y;
  const int tid = threadIdx.x, w = tid / kWave, lane = lane_id();
  const int c = lane % CB, rg = lane / CB;
  const int64_t V = a.V;
  const int64_t col = static_cast<int64_t>(blockIdx.x) * CB + c;
  float* st = a.state + static_cast<int64_t>(h) * K * V + col;
  float S[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) S[i] = st[static_cast<int64_t>(16 * i + 4 * w + rg) * V];
  const bool chan = tid < K;  // whole waves
  float nA = 0.f, dtb = 0.f;
  if (a.use_gate) {
    nA = __expf(a.A_log[h]);
    if (chan) dtb = a.dt_bias[static_cast<int64_t>(h) * K + tid];
  }
  const int nv = kda_valid(a);
  for (int t = 0; t < a.T; ++t) {
    if (chan) {
      const int64_t i = static_cast<int64_t>(h) * K + tid;
      const float qv = bf16_to_f32(a.q[t * a.q_ts + i]);
      const float kv = bf16_to_f32(a.k[t * a.k_ts + i]);
      float gl = ld_any(a.g, a.g_dtype, t * a.g_ts + i);
      if (a.use_gate) {
        const float x = gl + dtb;
        gl = isnan(a.lower_bound) ? -nA * softplus20(x) : a.lower_bound / (1.f + __expf(-nA * x));
      }
      s_q[tid] = qv;
      s_k[tid] = kv;
      s_dec[tid] = t < nv ? __expf(gl) : 1.f;
      if (a.use_l2norm) {
        const float sq = wave_sum(qv * qv), sk = wave_sum(kv * kv);
        if (lane == 0) {
          s_red[w][0] = sq;
          s_red[w][1] = sk;
        }
      }
    }
    const float vc = bf16_to_f32(a.v[t * a.v_ts + static_cast<int64_t>(h) * V + col]);
    float beta = ld_any(a.beta, a.beta_dtype, t * a.b_ts + h);
    if (a.beta_logits) beta = 1.f / (1.f + __expf(-beta));
    if (t >= nv) beta = 0.f;
    __syncthreads();
    float qs = a.scale, ks = 1.f;
    if (a.use_l2norm) {
      float sq = s_red[0][0], sk = s_red[0][1];
#pragma unroll
      for (int j = 1; j < K / kWave; ++j) {
        sq += s_red[j][0];
        sk += s_red[j][1];
      }
      qs = a.scale / sqrtf(sq + 1e-6f);
      ks = 1.f / sqrtf(sk + 1e-6f);
    }
    // decay, then the part of v the state already predicts from k
    float pu = 0.f;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = 16 * i + 4 * w + rg;
      S[i] *= s_dec[r];
      pu = fmaf(s_k[r] * ks, S[i], pu);
    }
    pu += __shfl_xor(pu, 16, kWave);
    pu += __shfl_xor(pu, 32, kWave);
    if (rg == 0) part_u[w][c] = pu;
    __syncthreads();
    const float u = (vc - (((part_u[0][c] + part_u[1][c]) + part_u[2][c]) + part_u[3][c])) * beta;
    float po = 0.f;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = 16 * i + 4 * w + rg;
      S[i] = fmaf(s_k[r] * ks, u, S[i]);
      po = fmaf(s_q[r] * qs, S[i], po);
    }
    po += __shfl_xor(po, 16, kWave);
    po += __shfl_xor(po, 32, kWave);
    if (rg == 0) part_o[w][c] = po;
    // the next token rewrites s_* after this barrier, when every thread has read them; part_u / part_o are
    // rewritten after the next token's first and second barriers, when wave 0 has read them
    __syncthreads();
    if (w == 0 && rg == 0) {
      const float o = ((part_o[0][c] + part_o[1][c]) + part_o[2][c]) + part_o[3][c];
      a.o[t * a.o_ts + static_cast<int64_t>(h) * V + col] = f32_to_bf16(o);
    }
  }
#pragma unroll
  for (int i = 0; i < RPT; ++i) st[static_cast<int64_t>(16 * i + 4 * w + rg) * V] = S[i];
}

// The per-token inputs of the recurrence, prepared for all T tokens in parallel (kda_prep_kernel) into a
// workspace row per (token, head) of 3 K + 4 floats: q l2-normalised times the scale, k l2-normalised, the
// per-channel decay exp(gate(g)), then beta (the sigmoid applied when it comes as logits), q . k of the
// normalised vectors, and 2 zeros.
template <int K>
constexpr int kda_ws_row() { return 3 * K + 4; }

// The prepared inputs of token t, head h for the lane's channels lane + 64 j (one wave): q l2-normalised times the
// scale, k l2-normalised, the decay exp(gate(g)) (1 for a padding token), and, the same in every lane, beta (the
// sigmoid applied when it comes as logits; 0 for padding) and q . k of the normalised vectors.
template <int K>
__device__ __forceinline__ void kda_prep_token(const KdaArgs& a, int64_t t, int h, bool pad, float (&qn)[K / kWave],
                                               float (&kn)[K / kWave], float (&dv)[K / kWave], float& beta,
                                               float& qk) {
  constexpr int NJ = K / kWave;
  const int lane = lane_id();
  const int64_t hk = static_cast<int64_t>(h) * K;
  float qv[NJ], kv[NJ], gv[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int64_t ch = hk + lane + kWave * j;
    qv[j] = bf16_to_f32(a.q[t * a.q_ts + ch]);
    kv[j] = bf16_to_f32(a.k[t * a.k_ts + ch]);
    gv[j] = ld_any(a.g, a.g_dtype, t * a.g_ts + ch);
  }
  float b = ld_any(a.beta, a.beta_dtype, t * a.b_ts + h);
  float qs = a.scale, ks = 1.f;
  if (a.use_l2norm) {
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      sq = fmaf(qv[j], qv[j], sq);
      sk = fmaf(kv[j], kv[j], sk);
    }
    qs = a.scale / sqrtf(wave_sum(sq) + 1e-6f);
    ks = 1.f / sqrtf(wave_sum(sk) + 1e-6f);
  }
  const float nA = a.use_gate ? __expf(a.A_log[h]) : 0.f;
  float d = 0.f;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    float gl = gv[j];
    if (a.use_gate) {
      const float x = gl + a.dt_bias[hk + lane + kWave * j];
      gl = isnan(a.lower_bound) ? -nA * softplus20(x) : a.lower_bound / (1.f + __expf(-nA * x));
    }
    qn[j] = qv[j] * qs;
    kn[j] = kv[j] * ks;
    dv[j] = pad ? 1.f : __expf(gl);
    d = fmaf(qn[j], kn[j], d);
  }
  qk = wave_sum(d);
  if (a.beta_logits) b = 1.f / (1.f + __expf(-b));
  beta = pad ? 0.f : b;
}

// Grid (T H / 4) x 4 waves: wave w prepares row (t, h) = divmod(4 blockIdx.x + w, H), lane i channels i + 64 j.
template <int K>
__global__ __launch_bounds__(256) void kda_prep_kernel(KdaArgs a, float* __restrict__ ws) {
  constexpr int NJ = K / kWave, ROW = kda_ws_row<K>();
  const int lane = lane_id();
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 4 + threadIdx.x / kWave;
  if (idx >= static_cast<int64_t>(a.T) * a.H) return;  // whole waves
  const int64_t t = idx / a.H;
  const int h = static_cast<int>(idx % a.H);
  float qn[NJ], kn[NJ], dv[NJ], beta, qk;
  kda_prep_token<K>(a, t, h, t >= kda_valid(a), qn, kn, dv, beta, qk);
  float* row = ws + idx * ROW;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int c = lane + kWave * j;
    row[c] = qn[j];
    row[K + c] = kn[j];
    row[2 * K + c] = dv[j];
  }
  if (lane < 4) row[3 * K + lane] = lane == 0 ? beta : lane == 1 ? qk : 0.f;
}

// NWB waves per (NWB CPW value columns, head): grid (V / (NWB CPW), H) x 64 NWB threads, CPW = 64 / RG with
// RG = K / RPL row groups. Each value column of the recurrence is independent (u and o of column v read only column
// v of S), so lane (c = lane / RG, rg = lane % RG) holds the RPL state rows rg RPL .. rg RPL + RPL - 1 of one
// column in registers for the whole prompt, and the sums over k are lane-internal, then over the RG lanes of a
// column (DPP steps, and one swizzle across rows of 16 lanes when RG = 32). The prepared rows of the head come into
// LDS 16 tokens at a time by global_load_lds, shared by the workgroup's waves and two chunk buffers deep (the
// next chunk loads while the recurrence runs on this one; one barrier per chunk), and each token's inputs of a lane
// are read from LDS within the chunk's unrolled token steps.
// Per token the two sums over k, k . S and q . S of the decayed state, are independent (pairwise within the
// lane, then their cross-lane steps interleaved), since o = S'^T q with S' = S + k u^T is q . S + u (q . k), q . k
// from the workspace: the token's latency is one chain of sums, not two.
template <int K, int RPL, int NWB>
__global__ __launch_bounds__(64 * NWB) void kda_recurrent_kernel(KdaArgs a, const float* __restrict__ ws) {
  constexpr int RG = K / RPL, CPW = kWave / RG, COLS = NWB * CPW, ROW = kda_ws_row<K>();
  constexpr int NT = NWB * kWave;
  constexpr int CHUNK_UNITS = kKdaChunk * ROW / 4;  // 16-byte pieces of a chunk
  constexpr int NU = (CHUNK_UNITS + NT - 1) / NT;
  constexpr int ROW_UNITS = ROW / 4;
  constexpr int VPT = (kKdaChunk * COLS + NT - 1) / NT;  // v values per thread per chunk
  static_assert(K == 64 || K == 128, "kda key dim");
  static_assert(RPL % 4 == 0 && RG <= kWave && (RG & (RG - 1)) == 0, "rows per lane");
  static_assert(ROW % 4 == 0, "16-byte workspace rows");
  // two chunk buffers (and v buffers: a wave writes the next chunk's values while the workgroup's other waves may
  // still read this chunk's), as separate arrays so that the compiler can tell a chunk's LDS reads from the next
  // chunk's loads in flight into the other buffer, and need not wait for those loads before the reads
  __shared__ __align__(16) float s_in0[kKdaChunk * ROW], s_in1[kKdaChunk * ROW];
  __shared__ float s_v0[kKdaChunk][COLS], s_v1[kKdaChunk][COLS];
  const int h = blockIdx.y, tid = threadIdx.x, wave = tid / kWave, lane = lane_id();
  const int c = lane / RG, rg = lane % RG;
  const int64_t V = a.V;
  const int64_t col0 = static_cast<int64_t>(blockIdx.x) * COLS;
  const int cw = wave * CPW + c;  // the lane's column within the workgroup
  float* st = a.state + static_cast<int64_t>(h) * K * V + col0 + cw;
  float S[RPL];
#pragma unroll
  for (int i = 0; i < RPL; ++i) S[i] = st[static_cast<int64_t>(RPL * rg + i) * V];
  const float* wsh = ws + static_cast<int64_t>(h) * ROW;
  const int64_t ts = static_cast<int64_t>(a.H) * ROW;  // workspace token stride
  uint16_t rv[VPT];  // raw bf16: converted once the chunk's loads are waited for, so the load needs no wait here
  auto issue = [&](int c0, float* dst) {
#pragma unroll
    for (int j = 0; j < NU; ++j) {
      const int u = tid + NT * j, tt = u / ROW_UNITS;
      if (u < CHUNK_UNITS && c0 + tt < a.T)
        load_lds16(wsh + (c0 + tt) * ts + (u % ROW_UNITS) * 4,
                   reinterpret_cast<char*>(dst) + (wave * kWave + NT * j) * 16);
    }
#pragma unroll
    for (int j = 0; j < VPT; ++j) {  // no branch: rows past the prompt (never read) load its last token's row
      const int i = tid + NT * j, tt = min(c0 + i / COLS, a.T - 1);
      rv[j] = a.v[tt * a.v_ts + static_cast<int64_t>(h) * V + col0 + i % COLS];
    }
  };
  // one chunk from buffers (in, vb) while the next one loads into (in_next); called with the arrays themselves
  auto chunk = [&](int c0, const float* in, float (*vb)[COLS], float* in_next) {
    wait_vmcnt<0>();  // this wave's loads of the chunk (and the stores before them)
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int i = tid + NT * j;
      if (i < kKdaChunk * COLS) vb[i / COLS][i % COLS] = bf16_to_f32(rv[j]);
    }
    // every wave's loads of this chunk are in LDS, and every wave is done with the other buffer
    if constexpr (NWB == 1) wave_lds_fence(); else __syncthreads();
    if (c0 + kKdaChunk < a.T) issue(c0 + kKdaChunk, in_next);  // in flight during the recurrence below
    const int n = min(kKdaChunk, a.T - c0);
    const float* base = in + RPL * rg;
    // lane (c, rg) keeps the output of tokens rg, rg + RG, ... of the chunk (every lane of a column holds each
    // token's sum) and stores them after the chunk: the token steps have no branch
    constexpr int OPL = (kKdaChunk + RG - 1) / RG;
    float keep[OPL];
#pragma unroll
    for (int j = 0; j < OPL; ++j) keep[j] = 0.f;
    auto step = [&](int t) {
      const float* r = base + t * ROW;
      float qq[RPL], kk[RPL], dd[RPL];
#pragma unroll
      for (int i = 0; i < RPL; i += 4) {
        const float4 q4 = *reinterpret_cast<const float4*>(r + i);
        const float4 k4 = *reinterpret_cast<const float4*>(r + K + i);
        const float4 d4 = *reinterpret_cast<const float4*>(r + 2 * K + i);
        qq[i] = q4.x, qq[i + 1] = q4.y, qq[i + 2] = q4.z, qq[i + 3] = q4.w;
        kk[i] = k4.x, kk[i + 1] = k4.y, kk[i + 2] = k4.z, kk[i + 3] = k4.w;
        dd[i] = d4.x, dd[i + 1] = d4.y, dd[i + 2] = d4.z, dd[i + 3] = d4.w;
      }
      const float2 bq = *reinterpret_cast<const float2*>(in + t * ROW + 3 * K);  // beta, q . k
      const float vc = vb[t][cw];
      // decay; the part of v the state already predicts from k, and q . S of the decayed state
      float pk[RPL], pq[RPL];
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        S[i] *= dd[i];
        pk[i] = kk[i] * S[i];
        pq[i] = qq[i] * S[i];
      }
#pragma unroll
      for (int w = 1; w < RPL; w *= 2)  // pairwise: (0 + 1) + (2 + 3), ...
#pragma unroll
        for (int i = 0; i < RPL; i += 2 * w) {
          pk[i] += pk[i + w];
          pq[i] += pq[i + w];
        }
      const float pu = group_sum<RG>(pk[0]);
      const float qs = group_sum<RG>(pq[0]);
      const float u = (vc - pu) * bq.x;
      const float po = fmaf(u, bq.y, qs);
#pragma unroll
      for (int i = 0; i < RPL; ++i) S[i] = fmaf(kk[i], u, S[i]);
#pragma unroll
      for (int j = 0; j < OPL; ++j)
        if (t % RG == rg && t / RG == j) keep[j] = po;  // a select, no branch
    };
    if (n == kKdaChunk) {
#pragma unroll
      for (int t = 0; t < kKdaChunk; ++t) step(t);
    } else {
      for (int t = 0; t < n; ++t) step(t);
    }
#pragma unroll
    for (int j = 0; j < OPL; ++j) {
      const int t = rg + RG * j;
      if (t < n) a.o[(c0 + t) * a.o_ts + static_cast<int64_t>(h) * V + col0 + cw] = f32_to_bf16(keep[j]);
    }
    if constexpr (NWB == 1) wave_lds_fence();  // the chunk's reads before the loads two chunks on
  };
  issue(0, s_in0);
  for (int c0 = 0; c0 < a.T; c0 += 2 * kKdaChunk) {
    chunk(c0, s_in0, s_v0, s_in1);
    if (c0 + kKdaChunk < a.T) chunk(c0 + kKdaChunk, s_in1, s_v1, s_in0);
  }
#pragma unroll
  for (int i = 0; i < RPL; ++i) st[static_cast<int64_t>(RPL * rg + i) * V] = S[i];
}

// -------------------------------------------------------------------------------------- KDA, chunked form
//
// The same recurrence over a chunk of C = 16 tokens in closed form (the chunked form of fla's chunk_kda, which the
// engine selects past 192 tokens: engine.py:946-949, 964-967). With chunk-local tokens t = 0 .. C-1, S0 the state
// at the chunk start, d_t the per-channel decay of token t, P_t = d_0 ... d_t and D(j, t) = d_{j+1} ... d_t
// (per-channel products taken directly, never as ratios, so a strong decay underflows to zero instead of 0 / 0):
//   k_t . (the decayed state before token t's write) = a_t + sum_{j<t} A[t][j] u_j,
//       a_t = (k_t P_t) . S0,  A[t][j] = sum_c k_tc k_jc D(j, t)_c
//   u_t = beta_t (v_t - a_t - sum_{j<t} A[t][j] u_j), that is u = M (v - a) with the lower triangular
//       M = (I + diag(beta) A)^-1 diag(beta), found row by row by forward substitution
//   o_t = q_t . S_t = b_t + sum_{j<=t} B[t][j] u_j,
//       b_t = (q_t P_t) . S0,  B[t][j] = sum_c q_tc k_jc D(j, t)_c (j < t),  B[t][t] = q_t . k_t
//   S_end = P_{C-1} S0 + sum_j (k_j D(j, C-1)) u_j^T
// Everything but S0 and v depends on the head alone, not on the value columns: kda_chunk_prep_kernel computes it
// for every (chunk, head) at once into a block of the workspace; kda_chunk_kernel then carries its value columns'
// state from chunk to chunk. All products run on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32: lane l gives
// row l % 16 and k l / 16 of A, column l % 16 and k l / 16 of B, and gets rows 4 (l / 16) + v of column l % 16), with
// the k order of each step chosen so that every result is the next product's operand as it stands: k step s takes
// k = 4 (l / 16) + s. Padding tokens (past n_valid, or past T in the last chunk) have decay 1, beta 0 and v - a taken
// as 0, so their u is 0 and the state passes them unchanged.
//
// us per call at 16 heads of 128 x 128, 32 / 64 / 192 / 512 / 700 / 2048 tokens: 12.2 / 14.3 / 21.9 / 43.7 / 57.8 / 146
// (0.85 a chunk, of which the 28 matrix instructions on the longest path are 0.4, and 10 .. 40 the preparation); 16.9 /
// 21.8 / 39.5 / 85.7 / 116 / 315 with the pair sums and the sums over k on the vector units and the substitution across
// lanes. The state's error against 64 bits over those lengths is 9 .. 14 % smaller than either other form's, its 16
// terms a chunk being summed on their own.

// A (chunk, head) block of the workspace, in floats, each operand in the order of its lanes (one 16-byte piece a lane):
// k P, q P [K / 16][lane][4] (token lane % 16, channels 16 tile + 4 (lane / 16) ..), W = (k D(., C-1))^T [K / 16][lane][4]
// (channel 16 tile + lane % 16, tokens 4 (lane / 16) ..), P_{C-1} [K], M [C][C], B [C][C] (zero above the diagonal).
template <int K>
struct KdaBlk {
  static constexpr int C = kKdaChunk;
  static constexpr int KP = 0, QP = C * K, W = 2 * C * K, PC = 3 * C * K, M = PC + K, B = M + C * C;
  static constexpr int SIZE = B + C * C;
  static_assert(SIZE % 4 == 0, "blocks stay 16-byte aligned");
};

__device__ __forceinline__ floatx4 mfma4(float x, float y, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0);
}

// The sum over the 4 lanes that share lane % 16.
__device__ __forceinline__ float quarter_sum(float v) { return half_pair_sum(row_pair_sum(v)); }

// 8 consecutive bf16 or fp32 values; VEC: their address is 16-byte aligned.
template <bool VEC, bool F32>
__device__ __forceinline__ void ld8(const void* base, int64_t i, float (&x)[8]) {
  if constexpr (F32) {
    const float* p = static_cast<const float*>(base) + i;
    if constexpr (VEC) {
      const float4 lo = *reinterpret_cast<const float4*>(p), hi = *reinterpret_cast<const float4*>(p + 4);
      x[0] = lo.x, x[1] = lo.y, x[2] = lo.z, x[3] = lo.w, x[4] = hi.x, x[5] = hi.y, x[6] = hi.z, x[7] = hi.w;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = p[e];
    }
  } else {
    const uint16_t* p = static_cast<const uint16_t*>(base) + i;
    if constexpr (VEC) {
      const uint4 r = *reinterpret_cast<const uint4*>(p);
      const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) x[2 * e] = bf_lo(w[e]), x[2 * e + 1] = bf_hi(w[e]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = bf16_to_f32(p[e]);
    }
  }
}

// x[0..3] of the 4 lanes of a quad, transposed: lane i of the quad gets value i of lanes 0 .. 3.
__device__ __forceinline__ float4 quad_transpose(const float* x) {
  const int lane = lane_id();
  const bool b0 = lane & 1, b1 = lane & 2;
  const float s0 = dpp_f32<kDppXor1>(b0 ? x[0] : x[1]), s1 = dpp_f32<kDppXor1>(b0 ? x[2] : x[3]);
  const float y0 = b0 ? s0 : x[0], y1 = b0 ? x[1] : s0, y2 = b0 ? s1 : x[2], y3 = b0 ? x[3] : s1;
  const float t0 = dpp_f32<kDppXor2>(b1 ? y0 : y2), t1 = dpp_f32<kDppXor2>(b1 ? y1 : y3);
  return make_float4(b1 ? t0 : y0, b1 ? t1 : y1, b1 ? y2 : t0, b1 ? y3 : t1);
}

// Grid (chunks H, heads within a chunk) x K / 32 waves. Wave p holds channels 32 p .. + 31 of the chunk: lane l token l % 16, channels
// 32 p + 8 (l / 16) .. + 7. The decay products between pairs of tokens split by the highest bit in which the pair
// differs: for t in the upper and j in the lower half of a block of 2^(L+1) tokens, D(j, t) is the product over the rest
// of j's half times that over t's half up to t, so with F_L = that part for each token, level L's pairs are
// (k F_L) (k F_L)^T and (q F_L) (k F_L)^T on the matrix units; the halves' products double from level to level by lane
// exchanges, and after the last they are P and D(., C-1). The waves' parts meet in LDS, wave L (and L + 2 when there are
// two) summing level L. VEC: q, k, g, dt_bias by 16-byte loads; GF32: g is fp32.
template <int K, bool VEC, bool GF32>
__global__ __launch_bounds__(2 * K, 3) void kda_chunk_prep_kernel(KdaArgs a, float* __restrict__ blk) {
  using L = KdaBlk<K>;
  constexpr int C = L::C, NW = K / 32, AR = C + 4;
  __shared__ __align__(16) float s_A[C * AR];
  __shared__ __align__(16) float s_beta[C];
  __shared__ float s_qk[NW][C], s_nq[NW][C], s_nk[NW][C];
  __shared__ floatx4 s_acc[4][2][NW][kWave];
  const int p = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id();
  const int ci = blockIdx.x / a.H, h = blockIdx.x % a.H;
  const int t = lane & 15, g = lane >> 4;
  const int64_t row = min(ci * C + t, a.T - 1), ch = static_cast<int64_t>(h) * K + 32 * p + 8 * g;
  const bool in = ci * C + t < a.T, pad = ci * C + t >= kda_valid(a);
  float q[8], k[8], d[8], dt[8];
  ld8<VEC, false>(a.q, row * a.q_ts + ch, q);
  ld8<VEC, false>(a.k, row * a.k_ts + ch, k);
  ld8<VEC, GF32>(a.g, row * a.g_ts + ch, d);
  if (a.use_gate) ld8<VEC, true>(a.dt_bias, ch, dt);
  float beta = ld_any(a.beta, a.beta_dtype, row * a.b_ts + h);
  const float nA = a.use_gate ? __expf(a.A_log[h]) : 0.f;
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    sq = fmaf(q[e], q[e], sq);
    sk = fmaf(k[e], k[e], sk);
  }
  sq = quarter_sum(sq);
  sk = quarter_sum(sk);
  if (g == 0) s_nq[p][t] = sq, s_nk[p][t] = sk;
  // one branch on the gate's form for all 8, none within
  if (a.use_gate && isnan(a.lower_bound)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x = d[e] + dt[e], y = log1pf(__expf(x));
      d[e] = -nA * (x > 20.f ? x : y);  // an x that is NaN gives y, NaN
    }
  } else if (a.use_gate) {
#pragma unroll
    for (int e = 0; e < 8; ++e) d[e] = a.lower_bound / (1.f + __expf(-nA * (d[e] + dt[e])));
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) d[e] = in && !pad ? __expf(d[e]) : 1.f;
  __syncthreads();
  float qs = a.scale, ks = 1.f;
  if (a.use_l2norm) {
    sq = s_nq[0][t] + s_nq[1][t];
    sk = s_nk[0][t] + s_nk[1][t];
#pragma unroll
    for (int w = 2; w < NW; ++w) sq += s_nq[w][t], sk += s_nk[w][t];
    qs = a.scale / sqrtf(sq + 1e-6f);
    ks = 1.f / sqrtf(sk + 1e-6f);
  }
  float qk = 0.f;
  float pre[8], suf[8], tot[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    q[e] = in ? q[e] * qs : 0.f;
    k[e] = in ? k[e] * ks : 0.f;
    qk = fmaf(q[e], k[e], qk);
    pre[e] = tot[e] = d[e];
    suf[e] = 1.f;
  }
  qk = quarter_sum(qk);
  if (g == 0) s_qk[p][t] = qk;
#pragma unroll
  for (int lv = 0; lv < 4; ++lv) {
    const bool up = (t >> lv) & 1;
    floatx4 accA = floatx4{0.f, 0.f, 0.f, 0.f}, accB = accA;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = up ? pre[e] : suf[e];
      const float x = k[e] * f, y = q[e] * f;
      accA = mfma4(x, x, accA);
      accB = mfma4(y, x, accB);
      // the other half's product (the same in all its lanes)
      const float o = lv == 0 ? dpp_f32<kDppXor1>(tot[e]) : lv == 1 ? dpp_f32<kDppXor2>(tot[e])
                    : lv == 2 ? dpp_f32<kDppHalfMirror>(tot[e]) : dpp_f32<kDppMirror>(tot[e]);
      pre[e] = up ? pre[e] * o : pre[e];
      suf[e] = up ? suf[e] : suf[e] * o;
      tot[e] *= o;
    }
    s_acc[lv][0][p][lane] = accA;
    s_acc[lv][1][p][lane] = accB;
  }
  float* out = blk + (static_cast<int64_t>(ci) * a.H + h) * L::SIZE;
  const int tile = 2 * p + g / 2;
#pragma unroll
  for (int e = 0; e < 8; e += 4) {  // channels 8 (g % 2) + e .. of the tile
    const int at = (tile * kWave + 16 * (2 * (g % 2) + e / 4) + t) * 4;
    *reinterpret_cast<float4*>(out + L::KP + at) =
        make_float4(k[e] * pre[e], k[e + 1] * pre[e + 1], k[e + 2] * pre[e + 2], k[e + 3] * pre[e + 3]);
    *reinterpret_cast<float4*>(out + L::QP + at) =
        make_float4(q[e] * pre[e], q[e + 1] * pre[e + 1], q[e + 2] * pre[e + 2], q[e + 3] * pre[e + 3]);
    const float w[4] = {k[e] * suf[e], k[e + 1] * suf[e + 1], k[e + 2] * suf[e + 2], k[e + 3] * suf[e + 3]};
    *reinterpret_cast<float4*>(out + L::W + (tile * kWave + 16 * (t / 4) + 8 * (g % 2) + e + t % 4) * 4) = quad_transpose(w);
    if (t == 0)
      *reinterpret_cast<float4*>(out + L::PC + 32 * p + 8 * g + e) = make_float4(tot[e], tot[e + 1], tot[e + 2], tot[e + 3]);
  }
  if (p == 0 && g == 0) {
    if (a.beta_logits) beta = 1.f / (1.f + __expf(-beta));
    s_beta[t] = in && !pad ? beta : 0.f;
  }
  __syncthreads();
  // rows 4 g + v, column t of A and B: the level of the pair's highest differing bit
  for (int lv = p; lv < 4; lv += NW) {
    floatx4 x = s_acc[lv][0][0][lane] + s_acc[lv][0][1][lane], y = s_acc[lv][1][0][lane] + s_acc[lv][1][1][lane];
#pragma unroll
    for (int w = 2; w < NW; ++w) x += s_acc[lv][0][w][lane], y += s_acc[lv][1][w][lane];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = 4 * g + v;
      if ((r ^ t) >> lv == 1) {
        s_A[r * AR + t] = x[v];
        out[L::B + r * C + t] = r > t ? y[v] : 0.f;
      } else if (lv == 0 && r == t) {
        float z = s_qk[0][t] + s_qk[1][t];
#pragma unroll
        for (int w = 2; w < NW; ++w) z += s_qk[w][t];
        out[L::B + r * C + t] = z;
      }
    }
  }
  __syncthreads();
  if (p > 0) return;
  // column t of M, row after row (every lane group the same), every row of A read before the first is used
  float m[C];
  float4 ar[C][C / 4];
#pragma unroll
  for (int r = 1; r < C; ++r)
#pragma unroll
    for (int j = 0; 4 * j < r; ++j) ar[r][j] = *reinterpret_cast<const float4*>(s_A + r * AR + 4 * j);
  float bt[C];
#pragma unroll
  for (int r = 0; r < C; r += 4) {
    const float4 b = *reinterpret_cast<const float4*>(s_beta + r);
    bt[r] = b.x, bt[r + 1] = b.y, bt[r + 2] = b.z, bt[r + 3] = b.w;
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < C; ++r) {
    float x = r == t ? 1.f : 0.f;
#pragma unroll
    for (int j = 0; j < r; ++j) {
      const float4& q4 = ar[r][j / 4];
      x = fmaf(j % 4 == 0 ? -q4.x : j % 4 == 1 ? -q4.y : j % 4 == 2 ? -q4.z : -q4.w, m[j], x);
    }
    m[r] = bt[r] * x;
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float lo = g & 1 ? m[4 + v] : m[v], hi = g & 1 ? m[12 + v] : m[8 + v];
    out[L::M + (4 * g + v) * C + t] = g & 2 ? hi : lo;
  }
}

// A barrier for LDS accesses only: the wave's own are done, its global and direct loads stay in flight (a fence would
// wait for the direct ones).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 16-byte reads of LDS filled by direct loads (already waited for), waited for in the same block: for an ordinary read
// the compiler waits until no direct load is in flight.
__device__ __forceinline__ floatx4 lds_read(uint32_t p) {
  floatx4 x;
  asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(x) : "v"(p) : "memory");
  return x;
}
// The operands of a worker's chunk at p (lane's place; KdaLds offsets) but k P, which is the next chunk's, at pn.
template <int TPW>
__device__ __forceinline__ void lds_read_chunk(uint32_t p, uint32_t ppc, uint32_t pm, uint32_t pn, floatx4 (&qp)[TPW],
                                               floatx4 (&wt)[TPW], floatx4 (&pc)[TPW], floatx4& m, floatx4 (&kp)[TPW]) {
  if constexpr (TPW == 2)
    asm volatile(
        "ds_read_b128 %0, %9 offset:2048\n\tds_read_b128 %1, %9 offset:3072\n\t"
        "ds_read_b128 %6, %11\n\t"
        "ds_read_b128 %4, %10\n\tds_read_b128 %5, %10 offset:64\n\t"
        "ds_read_b128 %2, %9 offset:4096\n\tds_read_b128 %3, %9 offset:5120\n\t"
        "ds_read_b128 %7, %12\n\tds_read_b128 %8, %12 offset:1024\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(qp[0]), "=&v"(qp[1]), "=&v"(wt[0]), "=&v"(wt[1]), "=&v"(pc[0]), "=&v"(pc[1]), "=&v"(m), "=&v"(kp[0]), "=&v"(kp[1])
        : "v"(p), "v"(ppc), "v"(pm), "v"(pn)
        : "memory");
  else
    asm volatile(
        "ds_read_b128 %0, %5 offset:1024\n\tds_read_b128 %3, %7\n\tds_read_b128 %2, %6\n\t"
        "ds_read_b128 %1, %5 offset:2048\n\tds_read_b128 %4, %8\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(qp[0]), "=&v"(wt[0]), "=&v"(pc[0]), "=&v"(m), "=&v"(kp[0])
        : "v"(p), "v"(ppc), "v"(pm), "v"(pn)
        : "memory");
}

// Operands in LDS of kda_chunk_kernel: each worker wave's of kDepth chunks (its tiles of k P, q P, W, then P_{C-1} and
// M), then the output wave's B.
template <int K>
struct KdaLds {
  static constexpr int TPW = K / 64, kDepth = 4;                      // state tiles (16 rows) per wave; chunks in flight
  static constexpr int KP = 0, QP = TPW * 1024, W = 2 * TPW * 1024, PC = 3 * TPW * 1024, M = PC + 1024, STAGE = M + 1024;
  static constexpr int B = 4 * kDepth * STAGE;
  static constexpr size_t BYTES = B + kDepth * 1024;
  static constexpr int LOADS = 3 * TPW + 2;                           // direct loads per chunk of a worker, besides v
};

// Grid (H, V / 16) x 5 waves (with 8 or more heads, a head's workgroups share an XCD and its L2): 16 value columns of one
// head. Waves 0 .. 3 hold K / 4 state rows each (the matrix instruction's result layout), form their parts of a and b,
// exchange the parts of a through LDS (one barrier a chunk) and update their rows; wave 4 forms the outputs of the chunk
// before from the parts of b and wave 0's u. The operands come by direct loads into each wave's own LDS, three chunks
// ahead: a chunk's 26 KB would take longer than its products through register loads. FAR: rows of v (or o) too far apart
// for 32-bit offsets.
template <int K, bool FAR>
__global__ __launch_bounds__(320) void kda_chunk_kernel(KdaArgs a, const float* __restrict__ blk) {
  using L = KdaBlk<K>;
  using S_ = KdaLds<K>;
  constexpr int C = L::C, TPW = S_::TPW, kDepth = S_::kDepth;
  constexpr int LOADS = S_::LOADS + 4;  // and the chunk's 4 values of v
  extern __shared__ __align__(16) char s_kda[];
  // the parts of a and b and u, of two chunks: arrays of their own, or the compiler makes each store to them wait for
  // the direct loads in flight
  __shared__ float4 s_a[2][4][kWave], s_b[2][4][kWave], s_u[2][kWave];
  const int h = blockIdx.x, lane = lane_id(), t16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t V = a.V, col = static_cast<int64_t>(blockIdx.y) * 16 + t16;
  const int64_t colc = min(col, V - 1);  // columns past V (V a multiple of 8) repeat the last one and are not stored
  const int nch = (a.T + C - 1) / C;
  const int64_t cs = static_cast<int64_t>(a.H) * L::SIZE;  // between the chunks of a head
  const float* bh = blk + static_cast<int64_t>(h) * L::SIZE;
  const uint32_t lane16 = lane * 16u, row16 = t16 * (C * 4u) + g * 16u;
  auto at4 = [](const float4& x, int s) { return s == 0 ? x.x : s == 1 ? x.y : s == 2 ? x.z : x.w; };
  auto f4 = [](const floatx4& x) { return make_float4(x[0], x[1], x[2], x[3]); };
  auto sum4 = [&](const float4 (*p)[kWave]) {  // of the four waves' parts
    const float4 x = p[0][lane], y = p[1][lane], z = p[2][lane], u = p[3][lane];
    return floatx4{((x.x + y.x) + z.x) + u.x, ((x.y + y.y) + z.y) + u.y, ((x.z + y.z) + z.z) + u.z, ((x.w + y.w) + z.w) + u.w};
  };
  // chunks past the last give the last one's block
  auto block = [&](int ci) { return make_rsrc(bh + min(ci, nch - 1) * cs, L::SIZE * 4); };
  // Runs chunk(ci, j) over all chunks (j = ci % kDepth), whole groups of kDepth, then the rest, the first kDepth - 1
  // chunks' loads issued before; chunk(ci, ..) issues those of chunk ci + kDepth - 1.
  auto run = [&](auto issue, auto first, auto chunk) {
#pragma unroll
    for (int j = 0; j < kDepth - 1; ++j) issue(j, j);
    first();
    int c0 = 0;
    for (; c0 + kDepth <= nch; c0 += kDepth)
#pragma unroll
      for (int j = 0; j < kDepth; ++j) chunk(c0 + j, j);
#pragma unroll
    for (int j = 0; j < kDepth - 1; ++j)
      if (c0 + j < nch) chunk(c0 + j, j);
    lds_barrier();
  };
  if (wave < 4) {
    const int nvalid = kda_valid(a);
    const uint16_t* vh = a.v + static_cast<int64_t>(h) * V;
    uint32_t voff[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) voff[v] = static_cast<uint32_t>((4 * g + v) * a.v_ts + colc) * 2u;
    char* own = s_kda + wave * kDepth * S_::STAGE;
    floatx4 S[TPW];
    float* st = a.state + (static_cast<int64_t>(h) * K + 16 * wave * TPW + 4 * g) * V + colc;
#pragma unroll
    for (int i = 0; i < TPW; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) S[i][v] = st[(16 * i + v) * V];
    uint16_t rv[kDepth][4];
    // a chunk's loads in three parts of 4 or so, issued between the matrix instructions of another chunk: 12 at once
    // hold the wave up for longer than they are worth
    constexpr int PART1 = 2 * TPW;
    auto issue1 = [&](int ci, int j) {
      const rsrc_t b = block(ci);
      char* d = own + j * S_::STAGE;
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        const uint32_t tile = (wave * TPW + i) * 1024u + lane16;
        buf_lds16(b, L::KP * 4 + tile, d + S_::KP + i * 1024);
        buf_lds16(b, L::QP * 4 + tile, d + S_::QP + i * 1024);
      }
    };
    auto issue2 = [&](int ci, int j) {
      const rsrc_t b = block(ci);
      char* d = own + j * S_::STAGE;
#pragma unroll
      for (int i = 0; i < TPW; ++i)
        buf_lds16(b, L::W * 4 + (wave * TPW + i) * 1024u + lane16, d + S_::W + i * 1024);
      buf_lds16(b, L::PC * 4 + lane16, d + S_::PC);  // its K channels, then the start of M
      buf_lds16(b, L::M * 4 + lane16, d + S_::M);
    };
    auto issue3 = [&](int ci, int j) {
      if constexpr (FAR) {
#pragma unroll
        for (int v = 0; v < 4; ++v) rv[j][v] = vh[min(ci * C + 4 * g + v, a.T - 1) * a.v_ts + colc];
      } else {
        const int n = min(a.T - ci * C, C);
        const rsrc_t r = make_rsrc(vh + static_cast<int64_t>(ci) * C * a.v_ts, n > 0 ? ((n - 1) * a.v_ts + V) * 2 : 0);
#pragma unroll
        for (int v = 0; v < 4; ++v) rv[j][v] = __builtin_amdgcn_raw_buffer_load_b16(r, static_cast<int>(voff[v]), 0, 0);
      }
    };
    auto issue = [&](int ci, int j) {
      issue1(ci, j);
      issue2(ci, j);
      issue3(ci, j);
    };
    // The matrix pipe takes 32 cycles an instruction (28 of them a chunk), so the order is fixed: while the parts of a
    // are exchanged it works on b.
    const uint32_t mine = lds_place(own) + lane16, mpc = lds_place(own) + S_::PC + wave * TPW * 64 + g * 16,
                   mm = lds_place(own) + S_::M + row16;
    floatx4 kp[TPW];
    auto first = [&] {  // k P of chunk 0
      wait_vmcnt<(kDepth - 2) * LOADS>();
#pragma unroll
      for (int i = 0; i < TPW; ++i) kp[i] = lds_read(mine + S_::KP + i * 1024);
    };
    auto chunk = [&](int ci, int j) {
      floatx4 as[TPW], bs[TPW], sc[TPW], qp[TPW], wt[TPW], pc[TPW], kn[TPW], m;
#pragma unroll
      for (int i = 0; i < TPW; ++i) as[i] = bs[i] = sc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < TPW; ++i) as[i] = mfma4(kp[i][s], S[i][s], as[i]);
      __builtin_amdgcn_sched_barrier(0);
      const int ni = ci + kDepth - 1, nj = (j + kDepth - 1) % kDepth;  // its place was the last chunk's, all read
      issue1(ni, nj);
      __builtin_amdgcn_sched_barrier(0);
      wait_vmcnt<(kDepth - 3) * LOADS + PART1>();  // this chunk and the next are in LDS
      const uint32_t at_j = j * S_::STAGE;
      lds_read_chunk<TPW>(mine + at_j, mpc + at_j, mm + at_j, mine + (j + 1) % kDepth * S_::STAGE, qp, wt, pc, m, kn);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (TPW == 2) as[0] += as[1];
      s_a[ci & 1][wave][lane] = f4(as[0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TPW; ++i) bs[i] = mfma4(qp[i][0], S[i][0], bs[i]);
      lds_barrier();
      const floatx4 at = sum4(s_a[ci & 1]);
#pragma unroll
      for (int s = 1; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < TPW; ++i) bs[i] = mfma4(qp[i][s], S[i][s], bs[i]);
      __builtin_amdgcn_sched_barrier(0);
      issue2(ni, nj);
      __builtin_amdgcn_sched_barrier(0);
      // u = M (v - a), by every wave
      floatx4 u = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s)
        u = mfma4(m[s], 4 * g + s < nvalid - ci * C ? bf16_to_f32(rv[j][s]) - at[s] : 0.f, u);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < TPW; ++i) sc[i] = mfma4(wt[i][s], u[s], sc[i]);
      __builtin_amdgcn_sched_barrier(0);
      issue3(ni, nj);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        // the chunk's 16 terms are summed on their own, so that the state is rounded once a chunk
#pragma unroll
        for (int v = 0; v < 4; ++v) S[i][v] = fmaf(S[i][v], pc[i][v], sc[i][v]);
        kp[i] = kn[i];
      }
      if constexpr (TPW == 2) bs[0] += bs[1];
      s_b[ci & 1][wave][lane] = f4(bs[0]);
      if (wave == 0) s_u[ci & 1][lane] = f4(u);
    };
    run(issue, first, chunk);
    if (col < V) {
#pragma unroll
      for (int i = 0; i < TPW; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) st[(16 * i + v) * V] = S[i][v];
    }
  } else {
    auto issue = [&](int ci, int j) { buf_lds16(block(ci), L::B * 4 + lane16, s_kda + S_::B + j * 1024); };
    uint16_t* oh = a.o + static_cast<int64_t>(h) * V;
    uint32_t ooff[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) ooff[v] = col < V ? static_cast<uint32_t>((4 * g + v) * a.o_ts + col) * 2u : kPast;
    floatx4 b1 = floatx4{0.f, 0.f, 0.f, 0.f};  // B of the chunk before
    const uint32_t mine = lds_place(s_kda + S_::B) + row16;
    auto outputs = [&](int ci) {
      floatx4 o = sum4(s_b[ci & 1]);
      const float4 u = s_u[ci & 1][lane];
#pragma unroll
      for (int s = 0; s < 4; ++s) o = mfma4(b1[s], at4(u, s), o);
      if constexpr (FAR) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int t = ci * C + 4 * g + v;
          if (t < a.T && col < V) oh[t * a.o_ts + col] = f32_to_bf16(o[v]);
        }
      } else {  // rows past T lie past the resource
        const int n = min(a.T - ci * C, C);
        const rsrc_t r = make_rsrc(oh + static_cast<int64_t>(ci) * C * a.o_ts, ((n - 1) * a.o_ts + V) * 2);
#pragma unroll
        for (int v = 0; v < 4; ++v)
          __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(o[v]), r, static_cast<int>(ooff[v]), 0, 0);
      }
    };
    auto chunk = [&](int ci, int j) {
      issue(ci + kDepth - 1, (j + kDepth - 1) % kDepth);
      lds_barrier();
      // the chunk's B: three later blocks and, from the fourth chunk on, three chunks' stores may be in flight
      if (ci < kDepth) wait_vmcnt<kDepth - 1>();
      else wait_vmcnt<5 * (kDepth - 1)>();
      const floatx4 b = lds_read(mine + j * 1024);
      if (ci > 0) outputs(ci - 1);
      b1 = b;
    };
    run(issue, [] {}, chunk);
    outputs(nch - 1);
  }
}

// ----------------------------------------------------------------------------------------- short conv

// y[t, ch] = silu(sum_j w[ch, j] * win_t[j] + b[ch]), win_t = the inputs t - W + 1 .. t of the channel (the cache
// holds the last W before the prompt, oldest first); the cache keeps the window after the last token. fp32 math,
// one rounding of y. Grid (C / 64, T / 16) x 64: a thread takes one channel for 16 tokens, all of whose inputs it
// loads at once; only the first token chunk reads the cache (16 >= W - 1), and its threads write the new window
// after their own reads of the old one.
constexpr int kConvTokens = 16;

template <int W>
__device__ __forceinline__ void short_conv_tile(const uint16_t* __restrict__ x, int64_t xs, int T, int64_t C,
                                                uint16_t* __restrict__ cache, const uint16_t* __restrict__ w,
                                                const uint16_t* __restrict__ b, int act, uint16_t* __restrict__ y,
                                                int64_t ys, const int64_t* __restrict__ n_valid, int bx, int by) {
  static_assert(kConvTokens >= W - 1, "only the first chunk may read the cache");
  const int64_t ch = static_cast<int64_t>(bx) * kWave + threadIdx.x;
  if (ch >= C) return;
  const int t0 = by * kConvTokens;
  float wt[W], in[kConvTokens + W - 1];  // inputs t0 - W + 1 .. t0 + 15
#pragma unroll
  for (int j = 0; j < W; ++j) wt[j] = bf16_to_f32(w[ch * W + j]);
  // every load unconditional (rows clamped into range, the value chosen after), so they all issue before the
  // first wait
#pragma unroll
  for (int i = 0; i < kConvTokens + W - 1; ++i) {
    const int t = t0 - (W - 1) + i;
    const float xv = bf16_to_f32(x[static_cast<int64_t>(t < 0 ? 0 : t < T ? t : T - 1) * xs + ch]);
    if (i < W - 1) {  // only these can precede the prompt (chunk 0)
      const float cv = bf16_to_f32(cache[ch * W + W + (t < 0 ? t : -1)]);
      in[i] = t < 0 ? cv : t < T ? xv : 0.f;
    } else {
      in[i] = t < T ? xv : 0.f;
    }
  }
  const float bias = b ? bf16_to_f32(b[ch]) : 0.f;
#pragma unroll
  for (int i = 0; i < kConvTokens; ++i) {
    if (t0 + i < T) {
      float acc = bias;
#pragma unroll
      for (int j = 0; j < W; ++j) acc = fmaf(wt[j], in[i + j], acc);
      if (act) acc = silu(acc);
      y[(t0 + i) * ys + ch] = f32_to_bf16(acc);
    }
  }
  if (by == 0) {
    // the window after the prompt's real tokens (the first n_valid, clamped to [0, T], when given: the padded
    // prefill's conv_idx, engine.py:261-262): inputs nv - W .. nv - 1, from the old cache where they precede it
    int nv = T;
    if (n_valid) nv = static_cast<int>(*n_valid < 0 ? 0 : *n_valid > T ? T : *n_valid);
    uint16_t nw[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const int t = nv - W + j;
      const uint16_t cv = cache[ch * W + (t < 0 ? W + t : j)];
      const uint16_t xv = x[static_cast<int64_t>(t < 0 ? 0 : t) * xs + ch];
      nw[j] = t < 0 ? cv : xv;
    }
#pragma unroll
    for (int j = 0; j < W; ++j) cache[ch * W + j] = nw[j];
  }
}


template <int W>
__global__ __launch_bounds__(64) void short_conv_kernel(const uint16_t* __restrict__ x, int64_t xs, int T, int64_t C,
                                                        uint16_t* __restrict__ cache, const uint16_t* __restrict__ w,
                                                        const uint16_t* __restrict__ b, int act,
                                                        uint16_t* __restrict__ y, int64_t ys,
                                                        const int64_t* __restrict__ n_valid) {
  short_conv_tile<W>(x, xs, T, C, cache, w, b, act, y, ys, n_valid, blockIdx.x, blockIdx.y);
}

// Up to kConvMany convolutions over the same tokens and width in one launch (a KDA layer's q, k and v):
// grid (channel blocks of the widest, token chunks, problems); a block past its problem's channels does nothing.
constexpr int kConvMany = 4;

struct ConvMany {
  const uint16_t* x[kConvMany];
  int64_t xs[kConvMany], C[kConvMany];
  uint16_t* cache[kConvMany];
  const uint16_t* w[kConvMany];
  uint16_t* y[kConvMany];
  int64_t ys[kConvMany];
  int T, act;
  const int64_t* n_valid;
};

template <int W>
__global__ __launch_bounds__(64) void short_conv_many_kernel(ConvMany m) {
  const int z = blockIdx.z;
  short_conv_tile<W>(m.x[z], m.xs[z], m.T, m.C[z], m.cache[z], m.w[z], nullptr, m.act, m.y[z], m.ys[z], m.n_valid,
                     blockIdx.x, blockIdx.y);
}

// --------------------------------------------------------------------------------------- gated RMSNorm

// One wave per row of n (<= 512) elements: y = bf16(x * rsqrt(mean(x^2) + eps) * w * sigmoid(g)), fp32 math.
__global__ __launch_bounds__(256) void rms_norm_gated_kernel(const uint16_t* __restrict__ x, int64_t xs,
                                                             const uint16_t* __restrict__ g, int64_t gs,
                                                             const uint16_t* __restrict__ w, int64_t rows, int n,
                                                             float eps, uint16_t* __restrict__ y, int64_t ys) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (row >= rows) return;
  const int lane = lane_id();
  // x, g and w of the row all requested first, through buffer resources over the row (an element past n reads
  // zero), so the wave waits for memory once (behind the range tests, each load was waited on in turn)
  const rsrc_t xr = make_rsrc(x + row * xs, static_cast<int64_t>(n) * 2), gr = make_rsrc(g + row * gs, static_cast<int64_t>(n) * 2),
               wr = make_rsrc(w, static_cast<int64_t>(n) * 2);
  float xv[8], gv[8], wv[8], ss = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int i = lane + kWave * j;
    const uint32_t off = i < n ? static_cast<uint32_t>(i) * 2u : kPast;
    xv[j] = bf16_to_f32(static_cast<uint16_t>(buf2(xr, off)));
    gv[j] = bf16_to_f32(static_cast<uint16_t>(buf2(gr, off)));
    wv[j] = bf16_to_f32(static_cast<uint16_t>(buf2(wr, off)));
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) ss = fmaf(xv[j], xv[j], ss);
  const float rstd = rsqrtf(wave_sum(ss) / static_cast<float>(n) + eps);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int i = lane + kWave * j;
    if (i < n) y[row * ys + i] = f32_to_bf16(xv[j] * rstd * wv[j] / (1.f + __expf(-gv[j])));
  }
}

// ------------------------------------------------------------------------------ one KDA decode token, one kernel
//
// The per-token core of a KDA layer (engine.py:242-263: the q/k/v short convolutions, the gate's LoRA up-projection
// f = f_b . fa, beta, fused_recurrent_kda, then g = g_b . ga and the gated output norm) in one launch instead of
// five, on the layer's projection row pr = [q | k (H K each) | v (H V) | fa | ga (R each) | beta logits (H)].
// kda_token_kernel: one workgroup of 16 waves per head, so every step that needs the whole head (the l2 norms over
// the key channels, the output norm over the value columns, the conv windows of the head's channels) stays inside
// the workgroup:
//   - the head's K key channels and V value channels are convolved over their cached windows (SiLU, rounded to
//     bf16 as short_conv_kernel stores them) and the windows shift in this token's inputs;
//   - f = bf16(sum_r f_b[ch, r] fa[r]) per key channel and g = bf16(sum_r g_b[ch, r] ga[r]) per value column
//     (two lanes per LoRA row, each over its half of R in order, one shuffle);
//   - one token of kda_short_kernel's recurrence, column block by column block (four waves per block of 16
//     value columns, the sums over key rows in kda_short_kernel's order);
//   - y = rms_norm_gated(bf16(o), g).
// Same arithmetic as the five kernels except the order of the f and g dots (small_linear reduces over more
// lanes), so f and g can differ in the last bf16 place.

struct KdaStepArgs {
  const uint16_t* pr;         // projection row
  const uint16_t* conv_w[3];  // q, k [H K, W] and v [H V, W] conv weights
  uint16_t* cache[3];         // the q, k and v conv caches of the same shapes, shifted in place
  const uint16_t* f_b;     // [H K, R]
  const uint16_t* g_b;     // [H V, R]
  const float* A_log;      // [H]
  const float* dt_bias;    // [H K]
  float lower_bound;       // NaN: the softplus gate
  float scale;
  float* state;            // [H, K, V] fp32, updated in place
  const uint16_t* o_norm;  // [V]
  float eps;
  uint16_t* y;             // [H, V]: the normed output
  int H, V, R;
};

// SiLU of a conv channel's window after the shift (cache cw[1..3], then the new input x), rounded to bf16 as
// short_conv_kernel stores it; ww the channel's 4 weights.
__device__ __forceinline__ float conv4(uint2 cw, uint2 ww, uint16_t x) {
  const float win[4] = {__uint_as_float(cw.x & 0xffff0000u), __uint_as_float(cw.y << 16),
                        __uint_as_float(cw.y & 0xffff0000u), bf16_to_f32(x)};
  const float wt[4] = {__uint_as_float(ww.x << 16), __uint_as_float(ww.x & 0xffff0000u), __uint_as_float(ww.y << 16),
                       __uint_as_float(ww.y & 0xffff0000u)};
  float acc = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = fmaf(wt[j], win[j], acc);
  return round_bf16(silu(acc));
}

// The window after this token: the oldest input dropped, x appended.
__device__ __forceinline__ uint2 conv4_shift(uint2 cw, uint16_t x) {
  return make_uint2((cw.x >> 16) | (cw.y << 16), (cw.y >> 16) | (static_cast<uint32_t>(x) << 16));
}

constexpr int kKdaMaxR = 256;  // LoRA rank limit: one fa / ga element per thread of 256

// LoRA up-projection rows (row i at m + i * R, bf16, 16-byte aligned) times vec (fp32 in LDS, R entries):
// out[i] = bf16(sum_r m[i, r] vec[r]). R is taken in pieces of kLoraPiece; two neighbouring lanes share a row and
// a piece, each taking its half of it in r order (one wave load covers 32 rows x 256 bytes), and one shuffle adds
// the halves. lora_fetch issues a lane's loads for one piece, so that a kernel can issue its first piece with its
// other loads at the start; lora_piece does the arithmetic once vec is in LDS.
constexpr int kLoraPiece = 128;

struct LoraPart {
  uint4 v[kLoraPiece / 16];
};

__device__ __forceinline__ void lora_fetch(const uint16_t* m, int64_t i, bool ok, int R, int r0, LoraPart& lp) {
  const int rh = r0 + (threadIdx.x & 1) * (kLoraPiece / 2);
  const uint16_t* p = m + (ok ? i : 0) * R + rh;
#pragma unroll
  for (int j = 0; j < kLoraPiece / 16; ++j)
    lp.v[j] = ok && rh + 8 * j < R ? *reinterpret_cast<const uint4*>(p + 8 * j) : make_uint4(0u, 0u, 0u, 0u);
}

__device__ __forceinline__ float lora_piece(const LoraPart& lp, const float* vec, int R, int r0, float acc) {
  const int rh = r0 + (threadIdx.x & 1) * (kLoraPiece / 2);
#pragma unroll
  for (int j = 0; j < kLoraPiece / 16; ++j) {
    if (rh + 8 * j >= R) break;  // R is a multiple of 16: whole 8-element pieces
    const uint32_t u[4] = {lp.v[j].x, lp.v[j].y, lp.v[j].z, lp.v[j].w};
    const float* vv = vec + rh + 8 * j;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      acc = fmaf(__uint_as_float(u[q] << 16), vv[2 * q], acc);
      acc = fmaf(__uint_as_float(u[q] & 0xffff0000u), vv[2 * q + 1], acc);
    }
  }
  return acc;
}

// One row (i, shared by the lane pair threadIdx.x / 2) with its first piece already fetched into lp: the
// remaining pieces are fetched here. Both lanes of the pair hold the bf16-rounded result.
__device__ __forceinline__ float lora_row(const uint16_t* m, int64_t i, bool ok, int R, const float* vec,
                                          const LoraPart& first) {
  float acc = lora_piece(first, vec, R, 0, 0.f);
  for (int r0 = kLoraPiece; r0 < R; r0 += kLoraPiece) {
    LoraPart lp;
    lora_fetch(m, i, ok, R, r0, lp);
    acc = lora_piece(lp, vec, R, r0, acc);
  }
  return round_bf16(acc + __shfl_xor(acc, 1, kWave));
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// v + v of lane ^ m, element by element
__device__ __forceinline__ float4 xor_add4(float4 v, int m) {
  return make_float4(v.x + __shfl_xor(v.x, m, kWave), v.y + __shfl_xor(v.y, m, kWave), v.z + __shfl_xor(v.z, m, kWave),
                     v.w + __shfl_xor(v.w, m, kWave));
}

constexpr int kKdaThreads = 512;

// Grid H x 512 threads, K = 128, V <= 128 NP. Wave w, lane (rg = lane / 16, c4 = lane % 16): row group w4 = w % 4
// and column half hf = w / 4; in pass p the lane holds state rows r = 16 i + 4 w4 + rg (i < 8) of the four columns
// 128 p + 64 hf + 4 c4 .. + 3 (one 16-byte load per row). Each column's sums over rows keep kda_short_kernel's
// order: lane-internal over i, then over the 4 row groups of a wave (xor 16, then 32), then over the 4 waves of
// its half through LDS. Threads 0..255 take the f rows (K of them, a lane pair each), threads 256..511 the g rows,
// 128 per pass; threads < K the q and k channels, threads < V the v channels. Every global load is issued before
// the first barrier; column groups past V read zeros and write nothing (buffer bounds).
// prefetching workgroups per head: kda_token_kernel traced at 11.26 / 9.86 / 9.51 / 9.44 us per call with 0 / 3 / 7 /
// 15 of them (16 heads of 128 x 128, R = 128, inside the 28-layer hybrid step); with each helper thread's loads
// issued together (they had waited for one another) the 28-layer step took 1490 / 1484.5 / 1483 us per token with
// 3 / 7 / 15 helpers, against 1496 before
#ifndef MM_KDA_HELPERS
#define MM_KDA_HELPERS 7
#endif
constexpr int kKdaHelpers = MM_KDA_HELPERS;

// A helper workgroup of kda_token_kernel (blockIdx.x >= H): part `part` of kKdaHelpers of the head's state block
// and LoRA rows, read and dropped, so that the lines come into L2 through more CUs than the one running the head
// (whose own loads of them then find them there or in flight): one CU alone keeps too few misses outstanding to
// pull the head's 128 KB at HBM speed.
__device__ __forceinline__ void kda_token_prefetch(const KdaStepArgs& a, int h, int part) {
  constexpr int K = 128, B = 4;  // up to B pieces of each block per thread and batch, all blocks' batches at once
  const int64_t V = a.V;
  const void* blocks[3] = {a.state + static_cast<int64_t>(h) * K * V, a.f_b + static_cast<int64_t>(h) * K * a.R,
                           a.g_b + static_cast<int64_t>(h) * V * a.R};
  const int64_t bytes[3] = {K * V * 4, static_cast<int64_t>(K) * a.R * 2, V * a.R * 2};
  rsrc_t r[3];
  int64_t n[3];
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    r[b] = make_rsrc(blocks[b], bytes[b]);
    n[b] = bytes[b] / 16;  // whole 16-byte pieces (rows are 16-byte multiples)
  }
  const int64_t stride = static_cast<int64_t>(kKdaThreads) * kKdaHelpers;
  const int64_t most = n[0] > n[1] ? (n[0] > n[2] ? n[0] : n[2]) : (n[1] > n[2] ? n[1] : n[2]);
  uint32_t acc = 0;
  // every piece of a batch is requested before any is used (a load whose value the next one waits for keeps one
  // request per thread in flight); pieces past a block's end read nothing
  for (int64_t i0 = threadIdx.x + static_cast<int64_t>(part) * kKdaThreads; i0 < most; i0 += stride * B) {
    uint4 v[3][B];
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int j = 0; j < B; ++j) {
        const int64_t i = i0 + stride * j;
        v[b][j] = buf16(r[b], i < n[b] ? static_cast<uint32_t>(i) * 16u : kPast);
      }
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int j = 0; j < B; ++j) acc ^= v[b][j].x;
  }
  asm volatile("" ::"v"(acc));  // keeps the loads; nothing is written
}

template <int NP>
__global__ __launch_bounds__(kKdaThreads) void kda_token_kernel(KdaStepArgs a) {
  constexpr int K = 128, RPT = K / 16, NV = 128 * NP;
  if (kKdaHelpers > 0 && static_cast<int>(blockIdx.x) >= a.H) {  // uniform: a helper workgroup
    const int hb = static_cast<int>(blockIdx.x) - a.H;
    kda_token_prefetch(a, hb % a.H, hb / a.H);
    return;
  }
  __shared__ float s_fga[2 * kKdaMaxR], s_f[K], s_q[K], s_k[K], s_dec[K], s_g[NV], s_vc[NV], s_nr[NV];
  __shared__ float s_red[K / kWave][2];
  __shared__ float4 part_u[NP][2][4][16], part_o[NP][2][4][16];
  __shared__ uint16_t s_o[NV];
  const int h = blockIdx.x;
  const int tid = threadIdx.x, w = tid / kWave, lane = lane_id();
  const int rg = lane / 16, c4 = lane % 16, w4 = w % 4, hf = w / 4;
  const int64_t V = a.V, HK = static_cast<int64_t>(a.H) * K, HV = static_cast<int64_t>(a.H) * V;
  const int64_t fa0 = 2 * HK + HV;  // fa, then ga, then the beta logits
  // fa (threads 0..255) and ga (256..511): R <= 256, one element per thread
  const int sec = tid >> 8, j8 = tid & 255;
  const uint16_t fga = a.pr[fa0 + sec * a.R + min(j8, a.R - 1)];
  // the first piece of this lane pair's f row (threads < 256) or g row
  const bool frow = tid < 256;
  const int gi0 = (tid - 256) >> 1;
  const uint16_t* lm = frow ? a.f_b + static_cast<int64_t>(h) * K * a.R : a.g_b + static_cast<int64_t>(h) * V * a.R;
  LoraPart lp;
  lora_fetch(lm, frow ? tid >> 1 : gi0, frow || gi0 < V, a.R, 0, lp);
  // the state rows of this lane's columns, through a resource over the head's [K, V] block (32-bit offsets)
  const rsrc_t srs = make_rsrc(a.state + static_cast<int64_t>(h) * K * V, static_cast<int64_t>(K) * V * 4);
  const uint32_t rstep = 16u * static_cast<uint32_t>(V) * 4u;
  uint32_t soff[NP];
  float4 S[NP][RPT];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int col = 128 * p + 64 * hf + 4 * c4;
    soff[p] = col < V ? (static_cast<uint32_t>(4 * w4 + rg) * static_cast<uint32_t>(V) + col) * 4u : kPast;
#pragma unroll
    for (int i = 0; i < RPT; ++i) S[p][i] = __builtin_bit_cast(float4, buf16(srs, soff[p] + i * rstep));
  }
  // conv channels: q and k channel tid (tid < K), v channel tid (tid < V); indices clamped, results unused past
  // the end
  const int64_t iq = static_cast<int64_t>(h) * K + min(tid, K - 1), iv = static_cast<int64_t>(h) * V + min<int64_t>(tid, V - 1);
  const uint2 cwq = *reinterpret_cast<const uint2*>(a.cache[0] + iq * 4), wq = *reinterpret_cast<const uint2*>(a.conv_w[0] + iq * 4);
  const uint2 cwk = *reinterpret_cast<const uint2*>(a.cache[1] + iq * 4), wk = *reinterpret_cast<const uint2*>(a.conv_w[1] + iq * 4);
  const uint2 cwv = *reinterpret_cast<const uint2*>(a.cache[2] + iv * 4), wv = *reinterpret_cast<const uint2*>(a.conv_w[2] + iv * 4);
  const uint16_t xq = a.pr[iq], xk = a.pr[HK + iq], xv = a.pr[2 * HK + iv];
  const float dtb = a.dt_bias[iq], nA = __expf(a.A_log[h]);
  const uint16_t nrm = a.o_norm[min<int64_t>(tid, V - 1)];  // the output norm's weight of column tid
  float beta = bf16_to_f32(a.pr[fa0 + 2 * a.R + h]);

  const bool chan = tid < K, vchan = tid < V;
  const float qv = conv4(cwq, wq, xq), kv = conv4(cwk, wk, xk);
  if (chan) {
    *reinterpret_cast<uint2*>(a.cache[0] + iq * 4) = conv4_shift(cwq, xq);
    *reinterpret_cast<uint2*>(a.cache[1] + iq * 4) = conv4_shift(cwk, xk);
  }
  if (vchan) {
    s_vc[tid] = conv4(cwv, wv, xv);
    s_nr[tid] = bf16_to_f32(nrm);
    *reinterpret_cast<uint2*>(a.cache[2] + iv * 4) = conv4_shift(cwv, xv);
  }
  if (j8 < a.R) s_fga[sec * kKdaMaxR + j8] = bf16_to_f32(fga);
  beta = 1.f / (1.f + __expf(-beta));
  __syncthreads();
  if (frow) {
    static_assert(K == 128, "one pass of 128 f rows over 256 threads");
    const float fv = lora_row(lm, tid >> 1, true, a.R, s_fga, lp);
    if ((tid & 1) == 0) s_f[tid >> 1] = fv;
  } else {
    for (int i0 = 0; i0 < V; i0 += 128) {  // wave-uniform trip count
      const int i = i0 + gi0;
      if (i0 > 0) lora_fetch(lm, i, i < V, a.R, 0, lp);
      const float gv = lora_row(lm, i, i < V, a.R, s_fga + kKdaMaxR, lp);
      if ((tid & 1) == 0 && i < V) s_g[i] = gv;
    }
  }
  __syncthreads();
  if (chan) {
    const float x = s_f[tid] + dtb;
    const float gl = isnan(a.lower_bound) ? -nA * softplus20(x) : a.lower_bound / (1.f + __expf(-nA * x));
    s_q[tid] = qv;
    s_k[tid] = kv;
    s_dec[tid] = __expf(gl);
    const float sq = wave_sum(qv * qv), sk = wave_sum(kv * kv);
    if (lane == 0) {
      s_red[w][0] = sq;
      s_red[w][1] = sk;
    }
  }
  __syncthreads();
  float sq = s_red[0][0], sk = s_red[0][1];
#pragma unroll
  for (int j = 1; j < K / kWave; ++j) {
    sq += s_red[j][0];
    sk += s_red[j][1];
  }
  const float qs = a.scale / sqrtf(sq + 1e-6f), ks = 1.f / sqrtf(sk + 1e-6f);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    float4 pu = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = 16 * i + 4 * w4 + rg;
      const float d = s_dec[r], kk = s_k[r] * ks;
      S[p][i].x *= d;
      S[p][i].y *= d;
      S[p][i].z *= d;
      S[p][i].w *= d;
      pu.x = fmaf(kk, S[p][i].x, pu.x);
      pu.y = fmaf(kk, S[p][i].y, pu.y);
      pu.z = fmaf(kk, S[p][i].z, pu.z);
      pu.w = fmaf(kk, S[p][i].w, pu.w);
    }
    pu = xor_add4(pu, 16);
    pu = xor_add4(pu, 32);
    if (rg == 0) part_u[p][hf][w4][c4] = pu;
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int col = 128 * p + 64 * hf + 4 * c4;
    const float4 u0 = part_u[p][hf][0][c4], u1 = part_u[p][hf][1][c4], u2 = part_u[p][hf][2][c4], u3 = part_u[p][hf][3][c4];
    const float4 u = make_float4((s_vc[col] - (((u0.x + u1.x) + u2.x) + u3.x)) * beta,
                                 (s_vc[col + 1] - (((u0.y + u1.y) + u2.y) + u3.y)) * beta,
                                 (s_vc[col + 2] - (((u0.z + u1.z) + u2.z) + u3.z)) * beta,
                                 (s_vc[col + 3] - (((u0.w + u1.w) + u2.w) + u3.w)) * beta);
    float4 po = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = 16 * i + 4 * w4 + rg;
      const float kk = s_k[r] * ks, qq = s_q[r] * qs;
      S[p][i].x = fmaf(kk, u.x, S[p][i].x);
      S[p][i].y = fmaf(kk, u.y, S[p][i].y);
      S[p][i].z = fmaf(kk, u.z, S[p][i].z);
      S[p][i].w = fmaf(kk, u.w, S[p][i].w);
      po.x = fmaf(qq, S[p][i].x, po.x);
      po.y = fmaf(qq, S[p][i].y, po.y);
      po.z = fmaf(qq, S[p][i].z, po.z);
      po.w = fmaf(qq, S[p][i].w, po.w);
    }
    po = xor_add4(po, 16);
    po = xor_add4(po, 32);
    if (rg == 0) part_o[p][hf][w4][c4] = po;
#pragma unroll
    for (int i = 0; i < RPT; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, S[p][i]), srs, static_cast<int>(soff[p] + i * rstep), 0, 0);
  }
  __syncthreads();
  if (w4 == 0 && rg == 0) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int col = 128 * p + 64 * hf + 4 * c4;
      const float4 o0 = part_o[p][hf][0][c4], o1 = part_o[p][hf][1][c4], o2 = part_o[p][hf][2][c4], o3 = part_o[p][hf][3][c4];
      s_o[col] = f32_to_bf16(((o0.x + o1.x) + o2.x) + o3.x);
      s_o[col + 1] = f32_to_bf16(((o0.y + o1.y) + o2.y) + o3.y);
      s_o[col + 2] = f32_to_bf16(((o0.z + o1.z) + o2.z) + o3.z);
      s_o[col + 3] = f32_to_bf16(((o0.w + o1.w) + o2.w) + o3.w);
    }
  }
  __syncthreads();
  // y = rms_norm_gated(bf16(o), g): wave 0, 8 elements per lane (V <= 512)
  if (w == 0) {
    float xo[8], ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = lane + kWave * j;
      xo[j] = i < V ? bf16_to_f32(s_o[min(i, NV - 1)]) : 0.f;
      ss = fmaf(xo[j], xo[j], ss);
    }
    const float rstd = rsqrtf(wave_sum(ss) / static_cast<float>(V) + a.eps);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = lane + kWave * j;
      if (i < V) a.y[static_cast<int64_t>(h) * V + i] = f32_to_bf16(xo[j] * rstd * s_nr[i] / (1.f + __expf(-s_g[i])));
    }
  }
}

// ------------------------------------------------------------------------------------ MLA decode attention

constexpr int kMlaChunk = 32;  // positions per workgroup: 4 waves of 8

struct MlaArgs {
  const uint16_t* q;      // [nh, dqk]
  const uint16_t* k_new;  // [nh, dqk]
  const uint16_t* v_new;  // [nh, dv]
  uint16_t* kc;           // [nh, max_len, dqk]
  uint16_t* vc;           // [nh, max_len, dv]
  const void* pos;
  int pos_dtype;
  int nh, dqk, dv;
  int64_t max_len;
  float scale;
  float* ws;  // [nh, nc, dv + 2]: a chunk's unnormalised sum of p * v, then its max and sum of p
  int nc;
  uint16_t* out;  // [nh, dv]
};

__device__ __forceinline__ int64_t load_pos64(const void* p, int dt) {
  return dt == MM_INT64 ? *static_cast<const int64_t*>(p) : static_cast<int64_t>(*static_cast<const int32_t*>(p));
}


// Grid (chunks, heads) x 4 waves; wave w owns positions t0 .. t0 + 7 (t0 = 32 chunk + 8 w), the new row standing
// in for row pos (and stored there by the wave that holds pos). First every lane issues its loads of the wave's
// value rows (LPR lanes x 8 dims per row, 64 / LPR rows per load), then the scores: 8 lanes per position, lane
// part taking the 16-byte pieces part, part + 8, ... of the q . k dot (KP of them at most), summed over the
// 8 lanes. Softmax over the chunk (a max over the 4 waves through LDS), p . V in the lanes' 8 dims, summed over
// a wave's row groups, then over the 4 waves in LDS; wave 0 writes the chunk's [dv] sums, max and sum of p.
template <int KP, int LPR>
__global__ __launch_bounds__(256) void mla_split_kernel(MlaArgs a) {
  constexpr int RPL = kWave / LPR;  // value rows per load
  constexpr int VI = 8 / RPL;       // loads covering a wave's 8 positions
  __shared__ float s_sc[kMlaChunk], s_max[4], s_l[4];
  __shared__ float s_acc[4][8 * LPR];
  const int tid = threadIdx.x, wave = tid / kWave, lane = lane_id();
  const int h = blockIdx.y, chunk = blockIdx.x;
  const int64_t pos = load_pos64(a.pos, a.pos_dtype);
  const int64_t c0 = static_cast<int64_t>(chunk) * kMlaChunk;
  if (pos < 0 || pos >= a.max_len || c0 > pos) return;  // uniform over the workgroup
  const int64_t t0 = c0 + wave * 8;
  const int64_t hk = static_cast<int64_t>(h) * a.max_len;
  // value rows t0 + vr + RPL i, dims 8 vd .. 8 vd + 7; rows past pos are not read (zeros: the cache there may
  // hold anything, and 0 * NaN would poison the sums)
  const int vr = lane / LPR, vd = lane % LPR;
  const bool vdim = vd * 8 < a.dv;
  uint4 vv[VI];
#pragma unroll
  for (int i = 0; i < VI; ++i) {
    const int64_t tt = t0 + vr + RPL * i;
    const uint16_t* row = tt == pos ? a.v_new + static_cast<int64_t>(h) * a.dv : a.vc + (hk + tt) * a.dv;
    vv[i] = vdim && tt <= pos ? *reinterpret_cast<const uint4*>(row + vd * 8) : make_uint4(0, 0, 0, 0);
  }
  // scores: position t0 + sp, pieces part + 8 j (rows past pos are not read)
  const int sp = lane / 8, part = lane % 8;
  const int64_t t = t0 + sp;
  const int np = t <= pos ? a.dqk / 8 : 0;
  const uint16_t* krow = t == pos ? a.k_new + static_cast<int64_t>(h) * a.dqk : a.kc + (hk + t) * a.dqk;
  const uint16_t* qrow = a.q + static_cast<int64_t>(h) * a.dqk;
  uint4 kb[KP], qa[KP];
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    const int pc = part + 8 * j;
    if (pc < np) {
      kb[j] = *reinterpret_cast<const uint4*>(krow + pc * 8);
      qa[j] = *reinterpret_cast<const uint4*>(qrow + pc * 8);
    }
  }
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < KP; ++j)
    if (part + 8 * j < np) s = dot8_bf16(kb[j], qa[j], s);
  s += dpp_f32<kDppXor1>(s);
  s += dpp_f32<kDppXor2>(s);
  s += dpp_f32<kDppHalfMirror>(s);
  const float sc = t <= pos ? s * a.scale : -INFINITY;
  const float wm = wave_max(sc);
  if (part == 0) s_sc[wave * 8 + sp] = sc;
  if (lane == 0) s_max[wave] = wm;
  // the wave holding pos stores the new rows into the cache
  if (pos >= t0 && pos < t0 + 8) {
    uint16_t* kd = a.kc + (hk + pos) * a.dqk;
    uint16_t* vd_ = a.vc + (hk + pos) * a.dv;
    for (int i = lane; i < a.dqk; i += kWave) kd[i] = a.k_new[static_cast<int64_t>(h) * a.dqk + i];
    for (int i = lane; i < a.dv; i += kWave) vd_[i] = a.v_new[static_cast<int64_t>(h) * a.dv + i];
  }
  __syncthreads();
  const float m = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));  // finite: c0 <= pos is valid
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
#pragma unroll
  for (int i = 0; i < VI; ++i) {
    const int r = vr + RPL * i;
    const float p = t0 + r <= pos ? __expf(s_sc[wave * 8 + r] - m) : 0.f;
    const uint32_t x[4] = {vv[i].x, vv[i].y, vv[i].z, vv[i].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc[2 * e] = fmaf(p, bf_lo(x[e]), acc[2 * e]);
      acc[2 * e + 1] = fmaf(p, bf_hi(x[e]), acc[2 * e + 1]);
    }
  }
#pragma unroll
  for (int off = LPR; off < kWave; off *= 2)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], off, kWave);
  if (lane < LPR && vdim) {
#pragma unroll
    for (int e = 0; e < 8; ++e) s_acc[wave][vd * 8 + e] = acc[e];
  }
  // the wave's sum of p: lane i < 8 for position t0 + i
  const float pl = lane < 8 && t0 + lane <= pos ? __expf(s_sc[wave * 8 + lane] - m) : 0.f;
  const float lsum = wave_sum(pl);
  if (lane == 0) s_l[wave] = lsum;
  __syncthreads();
  if (wave != 0) return;
  float* dst = a.ws + (static_cast<int64_t>(h) * a.nc + chunk) * (a.dv + 2);
  for (int d = lane; d < a.dv; d += kWave) dst[d] = ((s_acc[0][d] + s_acc[1][d]) + s_acc[2][d]) + s_acc[3][d];
  if (lane == 0) {
    dst[a.dv] = m;
    dst[a.dv + 1] = ((s_l[0] + s_l[1]) + s_l[2]) + s_l[3];
  }
}

// One workgroup of 4 waves per head merges the chunks 0 .. pos / 32: the max of the maxima (lanes over chunks),
// then wave w rescales and sums chunks w, w + 4, ... in that order (lane = value dimension), the 4 waves' sums
// added in LDS. The chunk states a wave needs for the first kMergeBatch of its chunks and the maxima of the first
// 256 chunks are loaded before pos arrives (chunks clamped into the workspace, the ones past pos dropped by
// selects), so the kernel waits for memory about once; longer prefixes load the rest afterwards.
// A position outside [0, max_len) writes NaN (and the split kernel wrote nothing).
// Bound: load latency, since one workgroup per head leaves the chip idle. The chunks past the first batch come
// kMergeTail at a time, clamped to the last one: chunk by chunk, each waited for the one before (0.85 us a chunk), and
// the attention of 16 heads x (192, 128) took 15.1 us behind 2000 positions and 28.9 behind 4000; now 10.7 and 14.2.
constexpr int kMergeBatch = 8;  // chunks per wave loaded ahead: 4 waves x 8 x 32 positions = 1024 positions
constexpr int kMergeTail = 16;  // and per further batch: 2048 positions
constexpr int kMergeFew = 4;    // where these are all: up to 1536 positions (16 loads for a chunk or two cost 0.2-0.4 us: the
                                // attention of 16 heads x 64 at position 1100, 7.2 -> 6.7 us)

// B chunks of the wave from c0 on (c0 + 4 b) into the running sums, every load in front of its first use.
template <int NDV, int B>
__device__ __forceinline__ void mla_merge_batch(const MlaArgs& a, const float* base, int64_t cs, int c0, int n, float m,
                                                float (&acc)[NDV], float& l) {
  const int lane = lane_id();
  float tm[B], tl[B], tv[B][NDV];
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const float* p = base + static_cast<int64_t>(min(c0 + 4 * b, n - 1)) * cs;
    tm[b] = p[a.dv];
    tl[b] = p[a.dv + 1];
#pragma unroll
    for (int j = 0; j < NDV; ++j) tv[b][j] = p[min(lane + kWave * j, a.dv - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int b = 0; b < B; ++b) {
    if (c0 + 4 * b < n) {  // uniform
      const float wgt = __expf(tm[b] - m);
      l = fmaf(tl[b], wgt, l);
#pragma unroll
      for (int j = 0; j < NDV; ++j) {
        const int d = lane + kWave * j;
        if (d < a.dv) acc[j] = fmaf(tv[b][j], wgt, acc[j]);
      }
    }
  }
}

template <int NDV>
__global__ __launch_bounds__(256) void mla_merge_kernel(MlaArgs a) {
  __shared__ float s_acc[4][kWave * NDV], s_l[4], s_m[4];
  const int h = blockIdx.x, tid = threadIdx.x, wave = tid / kWave, lane = lane_id();
  const int64_t cs = a.dv + 2;
  const float* base = a.ws + static_cast<int64_t>(h) * a.nc * cs;
  // loads that do not depend on pos
  const float m_first = base[static_cast<int64_t>(min(tid, a.nc - 1)) * cs + a.dv];
  float pm[kMergeBatch], pl[kMergeBatch], pv[kMergeBatch][NDV];
#pragma unroll
  for (int b = 0; b < kMergeBatch; ++b) {
    const float* p = base + static_cast<int64_t>(min(wave + 4 * b, a.nc - 1)) * cs;
    pm[b] = p[a.dv];
    pl[b] = p[a.dv + 1];
#pragma unroll
    for (int j = 0; j < NDV; ++j) pv[b][j] = p[min(lane + kWave * j, a.dv - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);  // pos (a scalar load) after the vector loads
  const int64_t pos = load_pos64(a.pos, a.pos_dtype);
  if (pos < 0 || pos >= a.max_len) {
    for (int d = tid; d < a.dv; d += 256) a.out[static_cast<int64_t>(h) * a.dv + d] = 0x7fc0;  // NaN
    return;
  }
  const int n = static_cast<int>(pos / kMlaChunk) + 1;
  float mx = tid < n ? m_first : -INFINITY;
  for (int c = tid + 256; c < n; c += 256) mx = fmaxf(mx, base[c * cs + a.dv]);
  mx = wave_max(mx);
  if (lane == 0) s_m[wave] = mx;
  __syncthreads();
  const float m = fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3]));
  float acc[NDV], l = 0.f;
#pragma unroll
  for (int j = 0; j < NDV; ++j) acc[j] = 0.f;
#pragma unroll
  for (int b = 0; b < kMergeBatch; ++b) {
    if (wave + 4 * b < n) {  // uniform
      const float wgt = __expf(pm[b] - m);
      l = fmaf(pl[b], wgt, l);
#pragma unroll
      for (int j = 0; j < NDV; ++j) {
        const int d = lane + kWave * j;
        if (d < a.dv) acc[j] = fmaf(pv[b][j], wgt, acc[j]);
      }
    }
  }
  const int c1 = wave + 4 * kMergeBatch;
  if (n <= 4 * (kMergeBatch + kMergeFew)) {
    if (c1 < n) mla_merge_batch<NDV, kMergeFew>(a, base, cs, c1, n, m, acc, l);
  } else {
    for (int c0 = c1; c0 < n; c0 += 4 * kMergeTail) mla_merge_batch<NDV, kMergeTail>(a, base, cs, c0, n, m, acc, l);
  }
#pragma unroll
  for (int j = 0; j < NDV; ++j) s_acc[wave][lane + kWave * j] = acc[j];
  if (lane == 0) s_l[wave] = l;
  __syncthreads();
  const float lt = ((s_l[0] + s_l[1]) + s_l[2]) + s_l[3];
  for (int d = tid; d < a.dv; d += 256) {
    const float o = ((s_acc[0][d] + s_acc[1][d]) + s_acc[2][d]) + s_acc[3][d];
    a.out[static_cast<int64_t>(h) * a.dv + d] = f32_to_bf16(o / lt);
  }
}

// ------------------------------------------------------------------------------- MLA prefill (T tokens)

struct MlaPrefillArgs {
  const uint16_t* q;      // token t's heads at q + t q_ts: [nh, dqk]
  const uint16_t* k_new;  // [nh, dqk] per token (token stride k_ts)
  const uint16_t* v_new;  // [nh, dv] per token (token stride v_ts)
  int64_t q_ts, k_ts, v_ts;
  uint16_t* kc;  // [nh, max_len, dqk]
  uint16_t* vc;  // [nh, max_len, dv]
  const void* pos;  // the first token's position
  int pos_dtype;
  int T, nh, dqk, dv;
  int64_t max_len;
  float scale;
  uint16_t* out;  // [nh, dv] per token (token stride out_ts)
  int64_t out_ts;
  int stored;  // the prompt's rows are in the cache already
};

__device__ __forceinline__ bool mla_prefill_pos_ok(const MlaPrefillArgs& a, int64_t pos) {
  return pos >= 0 && pos + a.T <= a.max_len;
}

// Grid (T, nh) x 64: token t's key and value rows of head h go to cache row pos + t (engine.py:537-541,
// index_copy_ at the prompt's positions). A prompt that does not fit in [0, max_len) stores nothing.
__global__ __launch_bounds__(64) void mla_prefill_store_kernel(MlaPrefillArgs a) {
  const int t = blockIdx.x, h = blockIdx.y;
  const int64_t pos = load_pos64(a.pos, a.pos_dtype);
  if (!mla_prefill_pos_ok(a, pos)) return;
  const int64_t row = static_cast<int64_t>(h) * a.max_len + pos + t;
  const auto* ks = reinterpret_cast<const uint4*>(a.k_new + t * a.k_ts + static_cast<int64_t>(h) * a.dqk);
  const auto* vs = reinterpret_cast<const uint4*>(a.v_new + t * a.v_ts + static_cast<int64_t>(h) * a.dv);
  auto* kd = reinterpret_cast<uint4*>(a.kc + row * a.dqk);
  auto* vd = reinterpret_cast<uint4*>(a.vc + row * a.dv);
  for (int i = threadIdx.x; i < a.dqk / 8; i += kWave) kd[i] = ks[i];
  for (int i = threadIdx.x; i < a.dv / 8; i += kWave) vd[i] = vs[i];
}

constexpr int kMlaPKeys = 32;  // keys per tile

// 8 bytes per lane from LDS, transposed within groups of 16 lanes: with lane s of a group reading row s / 4, columns
// 4 (s % 4) .. + 3 of a 4 x 16 block of bf16, lane i receives column i of the 4 rows (ds_read_b64_tr_b16; the lane layout
// checked on the device). Four fragments at once, each from place p[i] and `HI` bytes on, waited for in the same block:
// the builtin makes the compiler wait for every load in flight into LDS, the next tile's among them.
template <int HI>
__device__ __forceinline__ void lds_tr4x2(const uint32_t (&p)[4], uint64_t (&lo)[4], uint64_t (&hi)[4]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %2, %9\n\tds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
      "ds_read_b64_tr_b16 %4, %10\n\tds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
      "ds_read_b64_tr_b16 %6, %11\n\tds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1]), "=&v"(lo[2]), "=&v"(hi[2]), "=&v"(lo[3]), "=&v"(hi[3])
      : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "n"(HI)
      : "memory");
}

__device__ __forceinline__ bf16x8_t lds_frag(const char* p) {
  return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(p));
}

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// Max over the 4 lanes that share lane % 16.
__device__ __forceinline__ float quarter_max(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), true, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), true, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// The shape of mla_prefill_attn_kernel: QF 16-query fragments per workgroup, NW waves, head dims up to 32 NKQ (q, k;
// FULL: exactly) and 16 NT (v).
template <int QF, int NW, int NKQ, bool FULL, int NT>
struct MlaP {
  static constexpr int BQ = 16 * QF;                     // queries per workgroup
  static constexpr int DVM = 16 * NT;
  static constexpr int KC = 4 * NKQ, VC = 2 * NT;        // 16-byte chunks of a key, value row in LDS
  static constexpr int KI = kMlaPKeys * KC / kWave, VI = kMlaPKeys * VC / kWave;  // direct loads per key, value tile
  static constexpr int K_BYTES = kMlaPKeys * KC * 16, V_BYTES = kMlaPKeys * VC * 16;
  static constexpr int OROW = DVM + 4;                   // fp32 per output row of the merge
  static constexpr int ML = BQ * OROW;                   // the wave's max and sum of each query, after its outputs
  static constexpr int O_BYTES = (ML + 2 * BQ) * 4;
  static constexpr int WAVE_BYTES = K_BYTES + V_BYTES > O_BYTES ? K_BYTES + V_BYTES : O_BYTES;
  static constexpr size_t LDS = static_cast<size_t>(NW) * WAVE_BYTES;
  static_assert(LDS <= 160 * 1024 && KI % 2 == 0, "tile shape");
};

// The chunk of a tile's row held at LDS place c of the row (an involution). Keys: the 16 rows that a fragment reads at
// one chunk fall on the 16 distinct 16-byte columns of the banks; values: the 16 rows of a transposing read, 32 bytes
// each, fall on the 8 columns twice.
template <int KC>
__device__ __forceinline__ int mla_k_chunk(int row, int c) {
  return KC % 16 == 0 ? c ^ (row & 15) : c ^ ((row >> 1) & 7);
}
template <int VC>
__device__ __forceinline__ int mla_v_chunk(int row, int c) {
  return VC == 16 ? c ^ (2 * (row & 7)) : c ^ (2 * ((row >> 1) & 3));
}

// Causal attention of T prompt tokens over the static cache: token t at position pos + t takes
// softmax(scale q_t . K[0..pos+t]^T) . V[0..pos+t] (engine.py:679-682's mask), rows below pos from the cache, the
// prompt's own from k_new / v_new, which the workgroup of a token's queries also copies to its cache row
// (engine.py:537-541; no workgroup reads those cache rows, so the copy needs no launch of its own). a.stored: the rows
// are in the cache already (mla_prefill_store_kernel) and are read there, k_new and v_new by nobody.
// Grid (nh, query blocks, the last and longest first) x NW waves: with 8 or more heads the workgroups of a head share an
// XCD, whose L2 then serves its keys and values. A workgroup holds 16 QF queries of one head, and its waves take the
// 32-key tiles round robin (wave w: tiles w, w + NW, ...; first the cached keys' tiles, then the prompt's), each keeping
// its own running max, sum and output for all the queries; they are merged through LDS at the end. Per tile, on the
// 16x16x32 bf16 MFMA:
//   S^T [32 keys, 16 queries] = K Q^T, the key rows as A fragments, which every query fragment uses, and the queries
//     held as B fragments (lane: query lane % 16, dims 32 kk + 8 (lane / 16) .. + 7);
//   the masked softmax update per query is lane-local (a lane of the S^T tiles holds 8 keys of its query
//     column: 4 (lane / 16) + v and 16 + 4 (lane / 16) + v), the tile max taken over the 4 lane quarters;
//   O^T [dv, 16 queries] += V^T P^T: the B fragment of P comes straight from the S^T registers, its 8 k slots
//     taking those 8 keys in that order, and the A fragment of V^T (dim lane % 16, the same 8 keys) by two transposing
//     reads of the value tile.
// Bound by the vector-memory path: a tile's 20 KB come by loads straight into the wave's own LDS, the next tile's keys
// requested as soon as this one's are in registers, its values as soon as this one's are. us per call, 16 heads of
// 192 / 128, at 500@611, 2000@2000 and 30@3000 (tokens @ position): 59, 588 and 74 with 16 queries per workgroup, tiles
// by loads into registers and values transposed by stores; 25, 168 and 43 with 32 queries, transposing reads and the
// next tile in flight, still by register loads (81 at 2000@2000 without the loads); 19.2, 105 and 22 as it is.
// O^T's lane layout (dims 4 (lane / 16) + v of each 16-dim tile, query lane % 16) keeps the rescaling by the
// query's exp(m_old - m_new) lane-local as well. Rows past a tile's keys read zero (the buffer resource ends there),
// and so do the keys past a fragment's last query, so that a value no query of the fragment attends never meets it;
// queries past T repeat the last token and are not stored. A prompt outside [0, max_len) writes NaN.
template <int QF, int NW, int NKQ, bool FULL, int NT>
__global__ __launch_bounds__(NW * 64, 2) void mla_prefill_attn_kernel(MlaPrefillArgs a) {
  using P = MlaP<QF, NW, NKQ, FULL, NT>;
  constexpr int BQ = P::BQ, DVM = P::DVM;
  extern __shared__ __align__(16) char s_mla[];
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15, lq = lane >> 4;
  const int h = blockIdx.x, tq0 = (static_cast<int>(gridDim.y) - 1 - static_cast<int>(blockIdx.y)) * BQ;
  const int64_t pos = load_pos64(a.pos, a.pos_dtype);
  const int n4 = a.dv / 4;
  if (!mla_prefill_pos_ok(a, pos)) {  // uniform over the workgroup
    for (int i = tid; i < BQ * a.dv; i += NW * kWave) {
      const int t = tq0 + i / a.dv;
      if (t < a.T) a.out[t * a.out_ts + static_cast<int64_t>(h) * a.dv + i % a.dv] = 0x7fc0;  // NaN
    }
    return;
  }
  const int ctx = static_cast<int>(pos);               // < max_len <= 2^24
  const int nnew = min(tq0 + BQ, a.T);                 // the prompt's keys that any query of the workgroup attends
  const int nc = (ctx + kMlaPKeys - 1) / kMlaPKeys, nt_all = nc + (nnew + kMlaPKeys - 1) / kMlaPKeys;
  // row 0 of each segment and the bytes between rows (the host keeps 32 rows within 2^31 bytes)
  const uint16_t* kc = a.kc + static_cast<int64_t>(h) * a.max_len * a.dqk;
  const uint16_t* vc = a.vc + static_cast<int64_t>(h) * a.max_len * a.dv;
  const uint16_t* kn = a.stored ? kc + pos * a.dqk : a.k_new + static_cast<int64_t>(h) * a.dqk;
  const uint16_t* vn = a.stored ? vc + pos * a.dv : a.v_new + static_cast<int64_t>(h) * a.dv;
  const int64_t kn_ts = a.stored ? a.dqk : a.k_ts, vn_ts = a.stored ? a.dv : a.v_ts;
  char* kt = s_mla + wave * P::WAVE_BYTES;
  char* vt = kt + P::K_BYTES;
  // direct load i of a key tile fills LDS chunks 64 i + lane: row krow[i] (+ 16 for the second half), dims kdim[i] ..; of
  // a value tile row vrow + (64 / VC) i, dims vdim[i % 2] ..
  constexpr int KH = P::KI / 2, VPI = kWave / P::VC;
  int krow[KH], kdim[KH], vdim[2];
#pragma unroll
  for (int i = 0; i < KH; ++i) {
    krow[i] = (kWave * i + lane) / P::KC;
    kdim[i] = 8 * mla_k_chunk<P::KC>(krow[i], (kWave * i + lane) % P::KC);
  }
  const int vrow = lane / P::VC;
#pragma unroll
  for (int i = 0; i < 2; ++i) vdim[i] = 8 * mla_v_chunk<P::VC>(vrow + VPI * i, lane % P::VC);
  static_assert(P::VC == 16 || P::VC == 8, "value rows: the swizzle repeats after two loads");

  // keys of tile it that exist (0 past the last tile: the loads write zeros and touch no memory)
  auto rows_of = [&](int it) {
    return it >= nt_all ? 0 : min(it < nc ? ctx - it * kMlaPKeys : nnew - (it - nc) * kMlaPKeys, kMlaPKeys);
  };
  auto load_k = [&](int it) {
    const bool old = it < nc;
    const int n = rows_of(it);
    const int64_t ts = old ? a.dqk : kn_ts, row = n ? static_cast<int64_t>(old ? it : it - nc) * kMlaPKeys : 0;
    const rsrc_t r = make_rsrc((old ? kc : kn) + row * ts, n ? ((n - 1) * ts + a.dqk) * 2 : 0);
    const uint32_t ts2 = static_cast<uint32_t>(ts) * 2u;
#pragma unroll
    for (int i = 0; i < P::KI; ++i) {
      const uint32_t off = krow[i % KH] * ts2 + kdim[i % KH] * 2u + (i / KH) * 16u * ts2;
      buf_lds16(r, (FULL || kdim[i % KH] < a.dqk) ? off : kPast, kt + i * 1024);
    }
  };
  auto load_v = [&](int it) {
    const bool old = it < nc;
    const int n = rows_of(it);
    const int64_t ts = old ? a.dv : vn_ts, row = n ? static_cast<int64_t>(old ? it : it - nc) * kMlaPKeys : 0;
    const rsrc_t r = make_rsrc((old ? vc : vn) + row * ts, n ? ((n - 1) * ts + a.dv) * 2 : 0);
    const uint32_t ts2 = static_cast<uint32_t>(ts) * 2u;
#pragma unroll
    for (int i = 0; i < P::VI; ++i)
      buf_lds16(r, vdim[i % 2] < a.dv ? (vrow + VPI * i) * ts2 + vdim[i % 2] * 2u : kPast, vt + i * 1024);
  };
  // LDS places of this lane's fragment pieces: key row 16 f + lr, chunk 4 kk + lq; value rows 4 lq + lr / 4 (+ 16),
  // dims 16 nt + 4 (lr % 4) .. + 3
  const char* kfrag = kt + lr * P::KC * 16;
  const int vfr = 4 * lq + lr / 4;
  const int vplace = vfr * P::VC * 16 + mla_v_chunk<P::VC>(vfr, (lr % 4) / 2) * 16 + (lr & 1) * 8;

  bf16x8_t qf[QF][NKQ];
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    const uint16_t* qrow = a.q + min(tq0 + 16 * f + lr, a.T - 1) * a.q_ts + static_cast<int64_t>(h) * a.dqk;
#pragma unroll
    for (int kk = 0; kk < NKQ; ++kk) {
      const int d = 32 * kk + 8 * lq;
      const bool ok = FULL || d < a.dqk;
      qf[f][kk] = __builtin_bit_cast(bf16x8_t, and_mask16(*reinterpret_cast<const uint4*>(qrow + (ok ? d : 0)), ok));
    }
  }
  floatx4 o[QF][NT];
  float m[QF], l[QF];
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    m[f] = -INFINITY;
    l[f] = 0.f;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) o[f][nt] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  const float sc = a.scale * 1.4426950408889634f;  // scores in units of log2: exp2 gives the weights
  wait_vmcnt<0>();  // the queries: from here on only the tiles' loads are in flight
  load_k(wave);
  load_v(wave);
  for (int it = wave; it < nt_all; it += NW) {
    const int n = rows_of(it);
    const bool old = it < nc;
    const int j0 = (it - nc) * kMlaPKeys;  // the tile's first prompt token (prompt tiles)
    wait_vmcnt<P::VI>();  // the tile's keys (its values still in flight)
    wave_lds_fence();
    bf16x8_t kx[2][NKQ];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int kk = 0; kk < NKQ; ++kk)
        kx[u][kk] = lds_frag(kfrag + u * 16 * P::KC * 16 + mla_k_chunk<P::KC>(lr, 4 * kk + lq) * 16);
    wait_lgkm0();  // read before the next tile overwrites them
    load_k(it + NW);
    floatx4 s[QF][2];
#pragma unroll
    for (int f = 0; f < QF; ++f) s[f][0] = s[f][1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NKQ; ++kk)  // 2 QF independent sums in turn
#pragma unroll
      for (int f = 0; f < QF; ++f)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          s[f][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kx[u][kk], qf[f][kk], s[f][u], 0, 0, 0);
    // masked online softmax: slot e < 4 is key 4 lq + e of the tile, slot e >= 4 key 16 + 4 lq + e - 4
    bf16x8_t pf[QF];
#pragma unroll
    for (int f = 0; f < QF; ++f) {
      const int lim = old ? n : min(n, tq0 + 16 * f + lr - j0 + 1);  // keys of the tile this lane's query attends
      float sv[8];
      float tmax = -INFINITY;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int key = e < 4 ? 4 * lq + e : 16 + 4 * lq + e - 4;
        const float x = e < 4 ? s[f][0][e] : s[f][1][e - 4];
        sv[e] = key < lim ? x * sc : -INFINITY;
        tmax = fmaxf(tmax, sv[e]);
      }
      const float mn = fmaxf(m[f], quarter_max(tmax));
      const float mu = mn == -INFINITY ? 0.f : mn;  // a query with no key yet in this wave's tiles
      const float alpha = exp2_fast(m[f] - mu);
      m[f] = mn;
      float ps = 0.f;
      uint32_t pw[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p0 = exp2_fast(sv[2 * e] - mu), p1 = exp2_fast(sv[2 * e + 1] - mu);
        ps += p0 + p1;
        pw[e] = static_cast<uint32_t>(f32_to_bf16(p0)) | (static_cast<uint32_t>(f32_to_bf16(p1)) << 16);
      }
      l[f] = fmaf(l[f], alpha, ps);
      pf[f] = __builtin_bit_cast(bf16x8_t, make_uint4(pw[0], pw[1], pw[2], pw[3]));
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) o[f][nt] *= alpha;
      }
    }
    const bool diag = QF > 1 && !old && j0 == tq0;  // keys 16 .. 31 lie past every query of the first fragment
    wait_vmcnt<P::KI>();  // the tile's values (the next tile's keys still in flight)
    wave_lds_fence();
#pragma unroll
    for (int n0 = 0; n0 < NT; n0 += 4) {
      uint32_t place[4];
      uint64_t lo[4], hi[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) place[b] = lds_place(vt) + (vplace ^ (32 * (n0 + b)));
      lds_tr4x2<16 * P::VC * 16>(place, lo, hi);
      if (n0 + 4 == NT) load_v(it + NW);  // the tile's last values are read
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int f = 0; f < QF; ++f) {
          const uint64_t hf = (f == 0 && diag) ? 0 : hi[b];
          const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, make_uint4(static_cast<uint32_t>(lo[b]), static_cast<uint32_t>(lo[b] >> 32),
                                                                      static_cast<uint32_t>(hf), static_cast<uint32_t>(hf >> 32)));
          o[f][n0 + b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[f], o[f][n0 + b], 0, 0, 0);
        }
    }
  }
  // this workgroup's tokens into their cache rows
  if (!a.stored) {
    const int kp = a.dqk / 8, np = kp + a.dv / 8, rows = nnew - tq0;
    for (int i = tid; i < rows * np; i += NW * kWave) {
      const int t = i / np, c = i % np;
      const bool isk = c < kp;
      const int64_t row = pos + tq0 + t;
      const uint16_t* src = isk ? kn + (tq0 + t) * kn_ts + 8 * c : vn + (tq0 + t) * vn_ts + 8 * (c - kp);
      uint16_t* dst = isk ? a.kc + (static_cast<int64_t>(h) * a.max_len + row) * a.dqk + 8 * c
                          : a.vc + (static_cast<int64_t>(h) * a.max_len + row) * a.dv + 8 * (c - kp);
      *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
    }
  }
  // the wave's state into its own LDS region (the loads past its last tile done), then the merge
  wait_vmcnt<0>();
  wave_lds_fence();
  float* so = reinterpret_cast<float*>(s_mla + wave * P::WAVE_BYTES);
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    l[f] += __shfl_xor(l[f], 16, kWave);
    l[f] += __shfl_xor(l[f], 32, kWave);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      *reinterpret_cast<floatx4*>(so + (16 * f + lr) * P::OROW + 16 * nt + 4 * lq) = o[f][nt];
    if (lq == 0) {
      so[P::ML + 16 * f + lr] = m[f];
      so[P::ML + BQ + 16 * f + lr] = l[f];
    }
  }
  __syncthreads();
  for (int i = tid; i < BQ * n4; i += NW * kWave) {
    const int qi = i / n4, d = 4 * (i % n4), t = tq0 + qi;
    if (t >= a.T) continue;
    auto state = [&](int w) { return reinterpret_cast<const float*>(s_mla + w * P::WAVE_BYTES); };
    float mx = state(0)[P::ML + qi];  // finite: wave 0 holds key 0
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = fmaxf(mx, state(w)[P::ML + qi]);
    float lt = 0.f;
    floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float wt = exp2_fast(state(w)[P::ML + qi] - mx);
      lt = fmaf(state(w)[P::ML + BQ + qi], wt, lt);
      acc += wt * *reinterpret_cast<const floatx4*>(state(w) + qi * P::OROW + d);
    }
    const float inv = 1.f / lt;
    uint16_t* dst = a.out + t * a.out_ts + static_cast<int64_t>(h) * a.dv + d;
    const uint32_t w0 = static_cast<uint32_t>(f32_to_bf16(acc[0] * inv)) | (static_cast<uint32_t>(f32_to_bf16(acc[1] * inv)) << 16);
    const uint32_t w1 = static_cast<uint32_t>(f32_to_bf16(acc[2] * inv)) | (static_cast<uint32_t>(f32_to_bf16(acc[3] * inv)) << 16);
    *reinterpret_cast<uint2*>(dst) = make_uint2(w0, w1);
  }
}

template <int QF, int NW, int NKQ, bool FULL, int NT>
int launch_mla_prefill(const MlaPrefillArgs& a, hipStream_t st) {
  using P = MlaP<QF, NW, NKQ, FULL, NT>;
  auto kern = mla_prefill_attn_kernel<QF, NW, NKQ, FULL, NT>;
  int rc = mm::allow_lds(kern, P::LDS, "mla_prefill_attn");
  if (rc) return rc;
  const dim3 grid(static_cast<unsigned>(a.nh), static_cast<unsigned>((a.T + P::BQ - 1) / P::BQ));
  hipLaunchKernelGGL(kern, grid, dim3(NW * kWave), P::LDS, st, a);
  return mm::check_launch("mla_prefill_attn");
}

// The workgroup's shape by how many there would be of 32 queries, against the CUs. us per call at 16 heads of 192 / 128
// (tokens @ position), 32 queries on half a CU's waves | 16 queries on half | 16 queries on all:
//   2000@2000 114 | 158 | 179, 1024@0 21.8 | 25.0 | 32.3   more than a CU each: 32 queries share every key tile read
//   500@611 20.8 | 20.5 | 23.2, 300@0 11.3 | 8.8 | 11.3    every CU still gets a workgroup of 16 queries
//   256@1000 20.2 | 14.1 | 13.1, 30@3000 37.5 | 26.5 | 22.2  few workgroups: more waves share a query block's tiles
template <int NKQ, bool FULL, int NT>
int launch_mla_prefill_shape(const MlaPrefillArgs& a, hipStream_t st) {
  constexpr int NW = NKQ <= 6 ? 8 : 6;  // waves whose tiles fill one CU's LDS
  const int64_t cus = mm::cu_count(), wgs = static_cast<int64_t>((a.T + 31) / 32) * a.nh;
  if (wgs > cus) return launch_mla_prefill<2, NW / 2, NKQ, FULL, NT>(a, st);
  if (2 * wgs > cus) return launch_mla_prefill<1, NW / 2, NKQ, FULL, NT>(a, st);
  return launch_mla_prefill<1, NW, NKQ, FULL, NT>(a, st);
}

template <int K>
int launch_kda(const KdaArgs& a, float* ws, hipStream_t st) {
  if (a.T <= kKdaShortT) {
    hipLaunchKernelGGL((kda_short_kernel<K>), dim3(static_cast<unsigned>(a.V / kKdaCols), static_cast<unsigned>(a.H)),
                       dim3(256), 0, st, a);
    return mm::check_launch("kda_recurrent");
  }
  const int64_t rows = static_cast<int64_t>(a.T) * a.H;
  hipLaunchKernelGGL((kda_prep_kernel<K>), dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(256), 0, st, a, ws);
  int rc = mm::check_launch("kda_recurrent prep");
  if (rc) return rc;
  constexpr int RPL = kKdaRpl, NWB = kKdaNwb, cols = NWB * kWave / (K / RPL);
  if (a.V % cols == 0) {
    hipLaunchKernelGGL((kda_recurrent_kernel<K, RPL, NWB>), dim3(static_cast<unsigned>(a.V / cols),
                       static_cast<unsigned>(a.H)), dim3(kWave * NWB), 0, st, a, static_cast<const float*>(ws));
  } else {  // V a multiple of 8 only: one wave of 8 rows per lane per workgroup
    hipLaunchKernelGGL((kda_recurrent_kernel<K, 8, 1>), dim3(static_cast<unsigned>(a.V / (kWave / (K / 8))),
                       static_cast<unsigned>(a.H)), dim3(kWave), 0, st, a, static_cast<const float*>(ws));
  }
  return mm::check_launch("kda_recurrent");
}

// The chunked form: the (chunk, head) blocks, then the chunks in turn.
template <int K, bool VEC, bool GF32>
int launch_kda_prep(const KdaArgs& a, float* blk, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(static_cast<int64_t>((a.T + kKdaChunk - 1) / kKdaChunk) * a.H));
  hipLaunchKernelGGL((kda_chunk_prep_kernel<K, VEC, GF32>), grid, dim3(2 * K), 0, st, a, blk);
  return mm::check_launch("kda_chunk prep");
}

template <int K>
int launch_kda_chunk(const KdaArgs& a, float* ws, hipStream_t st) {
  if (a.T <= kKdaShortT) return launch_kda<K>(a, ws, st);  // a decode step: one launch, no workspace
  // every token's channels 16-byte aligned: loads of 8 channels, else one by one
  const bool f32 = a.g_dtype == MM_FP32;
  const bool vec = mm::aligned16(a.q) && mm::aligned16(a.k) && mm::aligned16(a.g) && (!a.use_gate || mm::aligned16(a.dt_bias)) &&
                   a.q_ts % 8 == 0 && a.k_ts % 8 == 0 && a.g_ts % (f32 ? 4 : 8) == 0;
  int rc;
  if (vec) rc = f32 ? launch_kda_prep<K, true, true>(a, ws, st) : launch_kda_prep<K, true, false>(a, ws, st);
  else rc = f32 ? launch_kda_prep<K, false, true>(a, ws, st) : launch_kda_prep<K, false, false>(a, ws, st);
  if (rc) return rc;
  const dim3 grid(static_cast<unsigned>(a.H), static_cast<unsigned>((a.V + 15) / 16));
  const bool far = a.v_ts >= (1 << 25) || a.o_ts >= (1 << 25);
  auto kern = far ? kda_chunk_kernel<K, true> : kda_chunk_kernel<K, false>;
  rc = mm::allow_lds(kern, KdaLds<K>::BYTES, "kda_chunk");
  if (rc) return rc;
  hipLaunchKernelGGL(kern, grid, dim3(320), KdaLds<K>::BYTES, st, a, static_cast<const float*>(ws));
  return mm::check_launch("kda_chunk");
}

}  // namespace

extern "C" int64_t mm_kda_recurrent_workspace(int64_t T, int64_t H, int64_t K) {
  if (T < 0 || H < 1 || (K != 64 && K != 128)) return -1;
  if (T <= kKdaShortT) return 0;
  return T * H * (3 * K + 4) * static_cast<int64_t>(sizeof(float));
}

extern "C" int64_t mm_kda_chunk_workspace(int64_t T, int64_t H, int64_t K) {
  if (T < 0 || H < 1 || (K != 64 && K != 128)) return -1;
  if (T <= kKdaShortT) return 0;
  const int64_t blk = K == 64 ? KdaBlk<64>::SIZE : KdaBlk<128>::SIZE;
  return (T + kKdaChunk - 1) / kKdaChunk * H * blk * static_cast<int64_t>(sizeof(float));
}

// The argument checks and launches of mm_kda_recurrent and mm_kda_chunk (same arguments, same results up to the
// order of fp32 sums).
static int kda_entry(bool chunked, const void* q, int64_t q_ts, const void* k, int64_t k_ts, const void* v,
                     int64_t v_ts, const void* g, int g_dtype, int64_t g_ts, const void* beta, int beta_dtype,
                     int64_t beta_ts, const float* A_log, const float* dt_bias, float lower_bound, int use_qk_l2norm,
                     int use_gate, int beta_logits, float scale, int64_t T, int64_t H, int64_t K, int64_t V,
                     float* state, void* o, int64_t o_ts, const int64_t* n_valid, void* workspace,
                     int64_t workspace_bytes, void* stream) {
  const char* who = chunked ? "kda_chunk" : "kda_recurrent";
  MM_REQUIRE(T >= 0 && T <= (1 << 20) && H >= 1 && H <= 65535 && T * H <= (1LL << 31),
             "%s: bad T=%lld or H=%lld (T <= 2^20, H <= 65535, T H <= 2^31)", who, (long long)T, (long long)H);
  // a lane holds 8 state rows of one column; one wave per 64 / (K / 8) value columns
  MM_REQUIRE((K == 64 || K == 128) && V % (T <= kKdaShortT ? kKdaCols : 8) == 0 && V >= 8 && V <= 4096,
             "%s: head dims K=%lld (64 or 128), V=%lld (a multiple of 8 up to 4096; of 16 for T <= %d)", who,
             (long long)K, (long long)V, kKdaShortT);
  const int64_t need = chunked ? mm_kda_chunk_workspace(T, H, K) : mm_kda_recurrent_workspace(T, H, K);
  MM_REQUIRE(T <= kKdaShortT || (workspace && mm::aligned16(workspace) && workspace_bytes >= need),
             "%s: the workspace must be 16-byte aligned and hold mm_%s_workspace(T, H, K) bytes", who, who);
  MM_REQUIRE(g_dtype == MM_BF16 || g_dtype == MM_FP32, "%s: g must be bf16 or fp32", who);
  MM_REQUIRE(beta_dtype == MM_BF16 || beta_dtype == MM_FP32, "%s: beta must be bf16 or fp32", who);
  MM_REQUIRE(q && k && v && g && beta && state && o, "%s: null pointer", who);
  MM_REQUIRE(!use_gate || (A_log && dt_bias), "%s: the gate needs A_log and dt_bias", who);
  MM_REQUIRE(q_ts >= H * K && k_ts >= H * K && g_ts >= H * K && v_ts >= H * V && beta_ts >= H && o_ts >= H * V,
             "%s: token strides smaller than a token's heads", who);
  if (T == 0) return MM_OK;
  KdaArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.g = g;
  a.beta = beta;
  a.g_dtype = g_dtype;
  a.beta_dtype = beta_dtype;
  a.q_ts = q_ts;
  a.k_ts = k_ts;
  a.v_ts = v_ts;
  a.g_ts = g_ts;
  a.b_ts = beta_ts;
  a.A_log = A_log;
  a.dt_bias = dt_bias;
  a.lower_bound = lower_bound;
  a.use_l2norm = use_qk_l2norm;
  a.use_gate = use_gate;
  a.beta_logits = beta_logits;
  a.scale = scale;
  a.state = state;
  a.o = static_cast<uint16_t*>(o);
  a.o_ts = o_ts;
  a.T = static_cast<int>(T);
  a.H = static_cast<int>(H);
  a.V = static_cast<int>(V);
  a.n_valid = n_valid;
  hipStream_t st = MM_STREAM(stream);
  float* ws = static_cast<float*>(workspace);
  if (chunked) return K == 64 ? launch_kda_chunk<64>(a, ws, st) : launch_kda_chunk<128>(a, ws, st);
  return K == 64 ? launch_kda<64>(a, ws, st) : launch_kda<128>(a, ws, st);
}

extern "C" int mm_kda_recurrent(const void* q, int64_t q_ts, const void* k, int64_t k_ts, const void* v, int64_t v_ts,
                                const void* g, int g_dtype, int64_t g_ts, const void* beta, int beta_dtype,
                                int64_t beta_ts, const float* A_log, const float* dt_bias, float lower_bound,
                                int use_qk_l2norm, int use_gate, int beta_logits, float scale, int64_t T, int64_t H,
                                int64_t K, int64_t V, float* state, void* o, int64_t o_ts, const int64_t* n_valid,
                                void* workspace, int64_t workspace_bytes, void* stream) {
  return kda_entry(false, q, q_ts, k, k_ts, v, v_ts, g, g_dtype, g_ts, beta, beta_dtype, beta_ts, A_log, dt_bias,
                   lower_bound, use_qk_l2norm, use_gate, beta_logits, scale, T, H, K, V, state, o, o_ts, n_valid,
                   workspace, workspace_bytes, stream);
}

extern "C" int mm_kda_chunk(const void* q, int64_t q_ts, const void* k, int64_t k_ts, const void* v, int64_t v_ts,
                            const void* g, int g_dtype, int64_t g_ts, const void* beta, int beta_dtype, int64_t beta_ts,
                            const float* A_log, const float* dt_bias, float lower_bound, int use_qk_l2norm,
                            int use_gate, int beta_logits, float scale, int64_t T, int64_t H, int64_t K, int64_t V,
                            float* state, void* o, int64_t o_ts, const int64_t* n_valid, void* workspace,
                            int64_t workspace_bytes, void* stream) {
  return kda_entry(true, q, q_ts, k, k_ts, v, v_ts, g, g_dtype, g_ts, beta, beta_dtype, beta_ts, A_log, dt_bias,
                   lower_bound, use_qk_l2norm, use_gate, beta_logits, scale, T, H, K, V, state, o, o_ts, n_valid,
                   workspace, workspace_bytes, stream);
}

extern "C" int mm_short_conv(const void* x, int64_t x_ts, int64_t T, int64_t C, void* cache, int64_t W, const void* w,
                             const void* b, int act, void* y, int64_t y_ts, const int64_t* n_valid, void* stream) {
  MM_REQUIRE(T >= 0 && T <= 65535LL * kConvTokens && C >= 1 && C <= (1LL << 31) / 8, "short_conv: bad T=%lld or C=%lld",
             (long long)T, (long long)C);
  MM_REQUIRE(W >= 2 && W <= 8, "short_conv: kernel width %lld must be in [2, 8]", (long long)W);
  MM_REQUIRE(x && cache && w && y, "short_conv: null pointer");
  MM_REQUIRE(x_ts >= C && y_ts >= C, "short_conv: token strides smaller than the channels");
  if (T == 0) return MM_OK;
  const auto* xp = static_cast<const uint16_t*>(x);
  auto* cp = static_cast<uint16_t*>(cache);
  const auto* wp = static_cast<const uint16_t*>(w);
  const auto* bp = static_cast<const uint16_t*>(b);
  auto* yp = static_cast<uint16_t*>(y);
  const int64_t* nv = n_valid;
  dim3 grid(static_cast<unsigned>((C + kWave - 1) / kWave), static_cast<unsigned>((T + kConvTokens - 1) / kConvTokens));
  hipStream_t st = MM_STREAM(stream);
  switch (W) {
    case 2: hipLaunchKernelGGL(short_conv_kernel<2>, grid, dim3(kWave), 0, st, xp, x_ts, (int)T, C, cp, wp, bp, act, yp, y_ts, nv); break;
    case 3: hipLaunchKernelGGL(short_conv_kernel<3>, grid, dim3(kWave), 0, st, xp, x_ts, (int)T, C, cp, wp, bp, act, yp, y_ts, nv); break;
    case 4: hipLaunchKernelGGL(short_conv_kernel<4>, grid, dim3(kWave), 0, st, xp, x_ts, (int)T, C, cp, wp, bp, act, yp, y_ts, nv); break;
    case 5: hipLaunchKernelGGL(short_conv_kernel<5>, grid, dim3(kWave), 0, st, xp, x_ts, (int)T, C, cp, wp, bp, act, yp, y_ts, nv); break;
    case 6: hipLaunchKernelGGL(short_conv_kernel<6>, grid, dim3(kWave), 0, st, xp, x_ts, (int)T, C, cp, wp, bp, act, yp, y_ts, nv); break;
    case 7: hipLaunchKernelGGL(short_conv_kernel<7>, grid, dim3(kWave), 0, st, xp, x_ts, (int)T, C, cp, wp, bp, act, yp, y_ts, nv); break;
    default: hipLaunchKernelGGL(short_conv_kernel<8>, grid, dim3(kWave), 0, st, xp, x_ts, (int)T, C, cp, wp, bp, act, yp, y_ts, nv); break;
  }
  return mm::check_launch("short_conv");
}

extern "C" int mm_short_conv_many(int64_t n, const void* const* x, const int64_t* x_ts, const int64_t* C,
                                  void* const* cache, const void* const* w, void* const* y, const int64_t* y_ts,
                                  int64_t T, int64_t W, int act, const int64_t* n_valid, void* stream) {
  MM_REQUIRE(n >= 1 && n <= kConvMany, "short_conv_many: %lld convolutions (1 to %d)", (long long)n, kConvMany);
  MM_REQUIRE(x && x_ts && C && cache && w && y && y_ts, "short_conv_many: null array");
  MM_REQUIRE(T >= 0 && T <= 65535LL * kConvTokens, "short_conv_many: bad T=%lld", (long long)T);
  MM_REQUIRE(W >= 2 && W <= 8, "short_conv_many: kernel width %lld must be in [2, 8]", (long long)W);
  ConvMany m{};
  int64_t cmax = 0;
  for (int64_t i = 0; i < n; ++i) {
    MM_REQUIRE(C[i] >= 1 && C[i] <= (1LL << 31) / 8, "short_conv_many: bad C=%lld (convolution %lld)", (long long)C[i],
               (long long)i);
    MM_REQUIRE(x[i] && cache[i] && w[i] && y[i], "short_conv_many: null pointer (convolution %lld)", (long long)i);
    MM_REQUIRE(x_ts[i] >= C[i] && y_ts[i] >= C[i], "short_conv_many: token strides smaller than the channels "
               "(convolution %lld)", (long long)i);
    m.x[i] = static_cast<const uint16_t*>(x[i]);
    m.xs[i] = x_ts[i];
    m.C[i] = C[i];
    m.cache[i] = static_cast<uint16_t*>(cache[i]);
    m.w[i] = static_cast<const uint16_t*>(w[i]);
    m.y[i] = static_cast<uint16_t*>(y[i]);
    m.ys[i] = y_ts[i];
    cmax = C[i] > cmax ? C[i] : cmax;
  }
  if (T == 0) return MM_OK;
  m.T = static_cast<int>(T);
  m.act = act;
  m.n_valid = n_valid;
  dim3 grid(static_cast<unsigned>((cmax + kWave - 1) / kWave), static_cast<unsigned>((T + kConvTokens - 1) / kConvTokens),
            static_cast<unsigned>(n));
  hipStream_t st = MM_STREAM(stream);
  switch (W) {
    case 2: hipLaunchKernelGGL(short_conv_many_kernel<2>, grid, dim3(kWave), 0, st, m); break;
    case 3: hipLaunchKernelGGL(short_conv_many_kernel<3>, grid, dim3(kWave), 0, st, m); break;
    case 4: hipLaunchKernelGGL(short_conv_many_kernel<4>, grid, dim3(kWave), 0, st, m); break;
    case 5: hipLaunchKernelGGL(short_conv_many_kernel<5>, grid, dim3(kWave), 0, st, m); break;
    case 6: hipLaunchKernelGGL(short_conv_many_kernel<6>, grid, dim3(kWave), 0, st, m); break;
    case 7: hipLaunchKernelGGL(short_conv_many_kernel<7>, grid, dim3(kWave), 0, st, m); break;
    default: hipLaunchKernelGGL(short_conv_many_kernel<8>, grid, dim3(kWave), 0, st, m); break;
  }
  return mm::check_launch("short_conv_many");
}

extern "C" int mm_rms_norm_gated(const void* x, int64_t x_rs, const void* g, int64_t g_rs, const void* w, int64_t rows,
                                 int64_t n, float eps, void* y, int64_t y_rs, void* stream) {
  MM_REQUIRE(rows >= 0 && n >= 1 && n <= 512, "rms_norm_gated: row length %lld must be in [1, 512]", (long long)n);
  MM_REQUIRE(x && g && w && y, "rms_norm_gated: null pointer");
  MM_REQUIRE(x_rs >= n && g_rs >= n && y_rs >= n, "rms_norm_gated: row strides smaller than the row");
  if (rows == 0) return MM_OK;
  hipLaunchKernelGGL(rms_norm_gated_kernel, dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(256), 0, MM_STREAM(stream),
                     static_cast<const uint16_t*>(x), x_rs, static_cast<const uint16_t*>(g), g_rs,
                     static_cast<const uint16_t*>(w), rows, static_cast<int>(n), eps, static_cast<uint16_t*>(y), y_rs);
  return mm::check_launch("rms_norm_gated");
}

extern "C" int mm_kda_decode_step(const void* pr, int64_t pr_len, const void* const* conv_w, void* const* conv_cache,
                                  int64_t W, const void* f_b, const void* g_b, int64_t R, const float* A_log,
                                  const float* dt_bias, float lower_bound, float scale, float* state, int64_t H,
                                  int64_t K, int64_t V, const void* o_norm, float eps, void* y, void* stream) {
  MM_REQUIRE(H >= 1 && H <= 65535, "kda_decode_step: bad H=%lld", (long long)H);
  MM_REQUIRE(K == 128 && V % kKdaCols == 0 && V >= kKdaCols && V <= 512,
             "kda_decode_step: head dims K=%lld (128), V=%lld (a multiple of 16 up to 512)", (long long)K, (long long)V);
  MM_REQUIRE(W == 4, "kda_decode_step: conv window %lld (4)", (long long)W);
  MM_REQUIRE(R >= 16 && R <= kKdaMaxR && R % 16 == 0, "kda_decode_step: LoRA rank %lld (a multiple of 16 up to %d)",
             (long long)R, kKdaMaxR);
  MM_REQUIRE(pr_len == 2 * H * K + H * V + 2 * R + H,
             "kda_decode_step: projection row of %lld elements, expected 2 H K + H V + 2 R + H = %lld", (long long)pr_len,
             (long long)(2 * H * K + H * V + 2 * R + H));
  MM_REQUIRE(pr && conv_w && conv_cache && f_b && g_b && A_log && dt_bias && state && o_norm && y,
             "kda_decode_step: null pointer");
  MM_REQUIRE(mm::aligned16(f_b) && mm::aligned16(g_b) && mm::aligned16(state),
             "kda_decode_step: f_b, g_b and state must be 16-byte aligned");
  KdaStepArgs a;
  for (int i = 0; i < 3; ++i) {
    MM_REQUIRE(conv_w[i] && conv_cache[i] && (reinterpret_cast<uintptr_t>(conv_w[i]) & 7) == 0 &&
                   (reinterpret_cast<uintptr_t>(conv_cache[i]) & 7) == 0,
               "kda_decode_step: conv weight / cache %d null or not 8-byte aligned", i);
    a.conv_w[i] = static_cast<const uint16_t*>(conv_w[i]);
    a.cache[i] = static_cast<uint16_t*>(conv_cache[i]);
  }
  a.pr = static_cast<const uint16_t*>(pr);
  a.f_b = static_cast<const uint16_t*>(f_b);
  a.g_b = static_cast<const uint16_t*>(g_b);
  a.A_log = A_log;
  a.dt_bias = dt_bias;
  a.lower_bound = lower_bound;
  a.scale = scale;
  a.state = state;
  a.o_norm = static_cast<const uint16_t*>(o_norm);
  a.eps = eps;
  a.y = static_cast<uint16_t*>(y);
  a.H = static_cast<int>(H);
  a.V = static_cast<int>(V);
  a.R = static_cast<int>(R);
  hipStream_t st = MM_STREAM(stream);
  const dim3 grid(static_cast<unsigned>(H * (1 + kKdaHelpers))), block(kKdaThreads);
  if (V <= 128) hipLaunchKernelGGL(kda_token_kernel<1>, grid, block, 0, st, a);
  else if (V <= 256) hipLaunchKernelGGL(kda_token_kernel<2>, grid, block, 0, st, a);
  else hipLaunchKernelGGL(kda_token_kernel<4>, grid, block, 0, st, a);
  return mm::check_launch("kda_decode_step");
}

extern "C" int64_t mm_mla_attn_workspace(int nh, int dv, int64_t max_len) {
  if (nh < 1 || dv < 1 || max_len < 1) return 0;
  return static_cast<int64_t>(nh) * ((max_len + kMlaChunk - 1) / kMlaChunk) * (dv + 2) * 4;
}

extern "C" int mm_mla_decode_attn(const void* q, const void* k_new, const void* v_new, int nh, int dqk, int dv,
                                  void* k_cache, void* v_cache, int64_t max_len, const void* pos, int pos_dtype,
                                  float scale, void* out, void* workspace, int64_t workspace_bytes, void* stream) {
  MM_REQUIRE(nh >= 1 && nh <= 65535 && max_len >= 1 && max_len <= (1LL << 24), "mla_decode_attn: bad nh or max_len");
  MM_REQUIRE(dqk % 8 == 0 && dqk >= 8 && dqk <= 512, "mla_decode_attn: dqk=%d must be a multiple of 8 in [8, 512]",
             dqk);
  MM_REQUIRE(dv % 8 == 0 && dv >= 8 && dv <= 256, "mla_decode_attn: dv=%d must be a multiple of 8 in [8, 256]", dv);
  MM_REQUIRE(pos_dtype == MM_INT64 || pos_dtype == MM_INT32, "mla_decode_attn: pos must be int64 or int32");
  MM_REQUIRE(q && k_new && v_new && k_cache && v_cache && pos && out && workspace, "mla_decode_attn: null pointer");
  MM_REQUIRE(mm::aligned16(q) && mm::aligned16(k_new) && mm::aligned16(v_new) && mm::aligned16(k_cache) &&
                 mm::aligned16(v_cache) && mm::aligned16(workspace),
             "mla_decode_attn: q, k_new, v_new, the caches and the workspace must be 16-byte aligned");
  MM_REQUIRE(workspace_bytes >= mm_mla_attn_workspace(nh, dv, max_len), "mla_decode_attn: workspace too small");
  MlaArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.k_new = static_cast<const uint16_t*>(k_new);
  a.v_new = static_cast<const uint16_t*>(v_new);
  a.kc = static_cast<uint16_t*>(k_cache);
  a.vc = static_cast<uint16_t*>(v_cache);
  a.pos = pos;
  a.pos_dtype = pos_dtype;
  a.nh = nh;
  a.dqk = dqk;
  a.dv = dv;
  a.max_len = max_len;
  a.scale = scale;
  a.ws = static_cast<float*>(workspace);
  a.nc = static_cast<int>((max_len + kMlaChunk - 1) / kMlaChunk);
  a.out = static_cast<uint16_t*>(out);
  hipStream_t st = MM_STREAM(stream);
  dim3 grid(static_cast<unsigned>(a.nc), static_cast<unsigned>(nh));
  const int kp = (dqk / 8 + 7) / 8;  // 16-byte pieces of a k row per lane, 8 lanes per position
  if (dv <= 128) {
    if (kp <= 1) hipLaunchKernelGGL((mla_split_kernel<1, 16>), grid, dim3(256), 0, st, a);
    else if (kp <= 2) hipLaunchKernelGGL((mla_split_kernel<2, 16>), grid, dim3(256), 0, st, a);
    else if (kp <= 4) hipLaunchKernelGGL((mla_split_kernel<4, 16>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((mla_split_kernel<8, 16>), grid, dim3(256), 0, st, a);
  } else {
    if (kp <= 2) hipLaunchKernelGGL((mla_split_kernel<2, 32>), grid, dim3(256), 0, st, a);
    else if (kp <= 4) hipLaunchKernelGGL((mla_split_kernel<4, 32>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((mla_split_kernel<8, 32>), grid, dim3(256), 0, st, a);
  }
  int rc = mm::check_launch("mla_decode_attn split");
  if (rc) return rc;
  if (dv <= 64) hipLaunchKernelGGL(mla_merge_kernel<1>, dim3(static_cast<unsigned>(nh)), dim3(256), 0, st, a);
  else if (dv <= 128) hipLaunchKernelGGL(mla_merge_kernel<2>, dim3(static_cast<unsigned>(nh)), dim3(256), 0, st, a);
  else hipLaunchKernelGGL(mla_merge_kernel<4>, dim3(static_cast<unsigned>(nh)), dim3(256), 0, st, a);
  return mm::check_launch("mla_decode_attn merge");
}

extern "C" int mm_mla_prefill_attn(const void* q, int64_t q_ts, const void* k_new, int64_t k_ts, const void* v_new,
                                   int64_t v_ts, int64_t T, int nh, int dqk, int dv, void* k_cache, void* v_cache,
                                   int64_t max_len, const void* pos, int pos_dtype, float scale, void* out,
                                   int64_t out_ts, void* stream) {
  MM_REQUIRE(T >= 0 && T <= (1 << 20), "mla_prefill_attn: bad T=%lld", (long long)T);
  MM_REQUIRE(nh >= 1 && nh <= 65535 && max_len >= 1 && max_len <= (1LL << 24), "mla_prefill_attn: bad nh or max_len");
  MM_REQUIRE(dqk % 8 == 0 && dqk >= 8 && dqk <= 256, "mla_prefill_attn: dqk=%d must be a multiple of 8 in [8, 256]",
             dqk);
  MM_REQUIRE(dv % 8 == 0 && dv >= 8 && dv <= 128, "mla_prefill_attn: dv=%d must be a multiple of 8 in [8, 128]", dv);
  MM_REQUIRE(pos_dtype == MM_INT64 || pos_dtype == MM_INT32, "mla_prefill_attn: pos must be int64 or int32");
  MM_REQUIRE(q && k_new && v_new && k_cache && v_cache && pos && out, "mla_prefill_attn: null pointer");
  MM_REQUIRE(q_ts >= static_cast<int64_t>(nh) * dqk && k_ts >= static_cast<int64_t>(nh) * dqk &&
                 v_ts >= static_cast<int64_t>(nh) * dv && out_ts >= static_cast<int64_t>(nh) * dv,
             "mla_prefill_attn: token strides smaller than a token's heads");
  MM_REQUIRE(q_ts % 8 == 0 && k_ts % 8 == 0 && v_ts % 8 == 0 && out_ts % 4 == 0,
             "mla_prefill_attn: token strides must keep rows 16-byte aligned (8-byte for out)");
  MM_REQUIRE(mm::aligned16(q) && mm::aligned16(k_new) && mm::aligned16(v_new) && mm::aligned16(k_cache) &&
                 mm::aligned16(v_cache) && (reinterpret_cast<uintptr_t>(out) & 7) == 0,
             "mla_prefill_attn: q, k_new, v_new and the caches must be 16-byte aligned, out 8-byte aligned");
  if (T == 0) return MM_OK;
  MlaPrefillArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.k_new = static_cast<const uint16_t*>(k_new);
  a.v_new = static_cast<const uint16_t*>(v_new);
  a.q_ts = q_ts;
  a.k_ts = k_ts;
  a.v_ts = v_ts;
  a.kc = static_cast<uint16_t*>(k_cache);
  a.vc = static_cast<uint16_t*>(v_cache);
  a.pos = pos;
  a.pos_dtype = pos_dtype;
  a.T = static_cast<int>(T);
  a.nh = nh;
  a.dqk = dqk;
  a.dv = dv;
  a.max_len = max_len;
  a.scale = scale;
  a.out = static_cast<uint16_t*>(out);
  a.out_ts = out_ts;
  hipStream_t st = MM_STREAM(stream);
  // Two calls store the rows first and read them from the cache: token strides past 2^25 elements, since the attention
  // kernel addresses a tile's 32 rows by 32-bit offsets, and an out that meets k_new or v_new (the values' buffer used
  // again for the result: both are nh dv wide), since a workgroup reads the rows of all earlier tokens while others
  // already store their outputs. Spans are compared, so column slices of one buffer count as meeting.
  auto meets_out = [&](const void* p, int64_t ts, int d) {
    const auto b = reinterpret_cast<uintptr_t>(p), o = reinterpret_cast<uintptr_t>(out);
    const int64_t row = static_cast<int64_t>(nh) * d, orow = static_cast<int64_t>(nh) * dv;
    return b < o + static_cast<uintptr_t>((T - 1) * out_ts + orow) * 2 && o < b + static_cast<uintptr_t>((T - 1) * ts + row) * 2;
  };
  a.stored = k_ts >= (1 << 25) || v_ts >= (1 << 25) || meets_out(k_new, k_ts, dqk) || meets_out(v_new, v_ts, dv);
  if (a.stored) {
    hipLaunchKernelGGL(mla_prefill_store_kernel, dim3(static_cast<unsigned>(T), static_cast<unsigned>(nh)), dim3(kWave),
                       0, st, a);
    int rc = mm::check_launch("mla_prefill_attn store");
    if (rc) return rc;
  }
  // 192 in its 6 steps of 32; any other dqk in 8, the ones past it masked. us against a loop of dqk / 32 steps over tiles by
  // register loads, 16 heads at 500@611 and 2000@2000: 64 / 64 19.6 | 48.7 and 125 | 476, 96 / 64 19.6 | 36.9 and 124 | 307,
  // 128 / 128 23.3 | 59.8 and 147 | 579, 256 / 128 24.2 | 62.4 and 152 | 592
  if (dv <= 64)
    return dqk == 192 ? launch_mla_prefill_shape<6, true, 4>(a, st) : launch_mla_prefill_shape<8, false, 4>(a, st);
  return dqk == 192 ? launch_mla_prefill_shape<6, true, 8>(a, st) : launch_mla_prefill_shape<8, false, 8>(a, st);
}
