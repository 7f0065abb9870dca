// mcpm_kernels.hip -- gfx950 kernels of the decode path.
//
// Numerics contract (the CPU oracle follows the same sequences):
//  * Q4_K/Q6_K x Q8_K dots form, per 256-block, the eight int32 lane sums of
//    the reference's AVX2 kernels (src/ops/ops_avx2.cpp:161-181, 224-270):
//    lane m folds bytes 4m..4m+3 of every 32-byte group.  Per row, lane m then
//    runs acc_m = fma(d_x*d_w, float(isum_m), acc_m) over blocks in order,
//    Q4_K adds acc_min = fma(-(d_x*dmin_w), float(minsum), acc_min), and the
//    lanes are summed ((a0+a4)+(a2+a6)) + ((a1+a5)+(a3+a7)) (ops_avx2.cpp:43-48).
//    The result is bit-identical to the reference's compiled AVX2 GEMV.
//  * Q8_K quantization: d = amax*(1/127), v = x*(127/amax), rint or round.
//  * Sums of squares: 256 strided partials, then a pairwise tree.
//  * Everything is compiled with -ffp-contract=off; fused multiply-adds are
//    explicit.
#include "mcpm_attn.h"
#include "mcpm_device.h"

namespace mcpm {

// ------------------------------------------------------- standalone ops ----

// One wave's 256-value block (lane l: values 4l .. 4l+3) quantized into out.
__device__ __forceinline__ void store_q8k_block(const float (&v)[4], bool away, int lane, BlockQ8K* __restrict__ out) {
  uint32_t packed;
  float d;
  int gsum;
  quant_block_wave(v, away, packed, d, gsum);
  reinterpret_cast<uint32_t*>(out->qs)[lane] = packed;
  if ((lane & 3) == 0) out->bsums[lane >> 2] = static_cast<int16_t>(gsum);
  if (lane == 0) out->d = d;
}

typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));  // float vectors have no alignment of their own

// Q8_K blocks of an fp32 vector in native layout, one wave (work group) per block.
__global__ void __launch_bounds__(64) k_quantize_q8k(const float* __restrict__ x, bool away,
                                                     BlockQ8K* __restrict__ out) {
  const int b = blockIdx.x, lane = threadIdx.x;
  const f32x4_u xv = *reinterpret_cast<const f32x4_u*>(x + b * QK_K + 4 * lane);
  const float v[4] = {xv.x, xv.y, xv.z, xv.w};
  store_q8k_block(v, away, lane, out + b);
}

// Q8_K blocks of the RMS-normalised vector, a work group per block: each reads
// the whole vector (its gammas with it, so there is one trip to memory) and
// forms the sum of squares itself, then its first wave quantizes the work
// group's block.  NV: values per thread, dim <= 256 * NV.  One work group for
// all blocks ran them three deep after two more trips to memory: 4.8 -> 3.1 us
// at 2048 and 2304 values.
template <int NV>
__global__ void __launch_bounds__(256) k_norm_quantize_q8k(const float* __restrict__ x,
                                                           const float* __restrict__ gamma, float eps, int dim,
                                                           bool away, BlockQ8K* __restrict__ out) {
  __shared__ float red[256];
  const int tid = threadIdx.x, b = blockIdx.x;
  f32x4_u xb = {}, gb = {};
  if (tid < 64) {
    xb = *reinterpret_cast<const f32x4_u*>(x + b * QK_K + 4 * tid);
    gb = *reinterpret_cast<const f32x4_u*>(gamma + b * QK_K + 4 * tid);
  }
  float p = 0.0f;
  for (int i0 = 0; i0 < dim; i0 += 256 * NV) {
    float v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = x[min(i0 + tid + 256 * k, dim - 1)];
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (i0 + tid + 256 * k < dim) p = p + v[k] * v[k];
  }
  const float rms = block_rms_1sync(p, dim, eps, red);
  if (tid < 64) {
    const float v[4] = {(xb.x * rms) * gb.x, (xb.y * rms) * gb.y, (xb.z * rms) * gb.z, (xb.w * rms) * gb.w};
    store_q8k_block(v, away, tid, out + b);
  }
}

hipError_t launch_quantize_q8k(const float* x, const float* gamma, float eps, int dim, int mode, BlockQ8K* out,
                               hipStream_t s) {
  const bool norm = (mode == PRO_NORM_AWAY || mode == PRO_NORM_EVEN);
  const bool away = (mode == PRO_QUANT_AWAY || mode == PRO_NORM_AWAY);
  const dim3 grid(dim / QK_K);
  if (!norm)
    hipLaunchKernelGGL(k_quantize_q8k, grid, dim3(64), 0, s, x, away, out);
  else
    hipLaunchKernelGGL(k_norm_quantize_q8k<12>, grid, dim3(256), 0, s, x, gamma, eps, dim, away, out);
  return hipGetLastError();
}

// rmsnorm (src/ops/ops.cpp:468-481): out = (x*rms)*w.  One work group, which
// reads all of x before it writes (out may be x).  Up to NV values a thread
// stay in registers with their weights, so the vector is read once; the
// second trip to memory is for longer ones only (2304 values: 4.1 -> 3.1 us),
// whose values past those are loaded NV at a time in both passes (a load a step:
// 16384 values 13.9 us, 262144 226; now 7.4 and 93).  A batch that passes the end
// reads the thread's own first value of it again, never another thread's (which
// out may have overwritten).
template <int NV>
__global__ void __launch_bounds__(256) k_rmsnorm(const float* x, const float* __restrict__ w, float eps, int dim,
                                                 float* out) {
  __shared__ float red[256];
  const int tid = threadIdx.x;
  float v[NV], g[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    v[k] = x[min(tid + 256 * k, dim - 1)];
    g[k] = w[min(tid + 256 * k, dim - 1)];
  }
  float p = 0.0f;
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if (tid + 256 * k < dim) p = p + v[k] * v[k];
  for (int i = tid + 256 * NV; i < dim; i += 256 * NV) {
    float y[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) y[k] = x[i + 256 * k < dim ? i + 256 * k : i];
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (i + 256 * k < dim) p = p + y[k] * y[k];
  }
  const float rms = block_rms_1sync(p, dim, eps, red);
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if (tid + 256 * k < dim) out[tid + 256 * k] = (v[k] * rms) * g[k];
  for (int i = tid + 256 * NV; i < dim; i += 256 * NV) {
    float y[NV], h[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int j = i + 256 * k < dim ? i + 256 * k : i;
      y[k] = x[j];
      h[k] = w[j];
    }
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (i + 256 * k < dim) out[i + 256 * k] = (y[k] * rms) * h[k];
  }
}

hipError_t launch_rmsnorm(const float* x, const float* w, float eps, int dim, float* out, hipStream_t s) {
  hipLaunchKernelGGL(k_rmsnorm<12>, dim3(1), dim3(256), 0, s, x, w, eps, dim, out);
  return hipGetLastError();
}

// swiglu_and_quantize_q8k (src/ops/ops.cpp:725-765): dim/256 blocks, lround,
// one wave (work group) per block.  One work group for all blocks took them
// six deep, with four scalar loads of each vector: 10.0 -> 2.6 us at 5888 values.
__global__ void __launch_bounds__(64) k_swiglu_quant(const float* __restrict__ g, const float* __restrict__ u,
                                                     BlockQ8K* __restrict__ out) {
  const int b = blockIdx.x, lane = threadIdx.x;
  const f32x4_u gv = *reinterpret_cast<const f32x4_u*>(g + b * QK_K + 4 * lane);
  const f32x4_u uv = *reinterpret_cast<const f32x4_u*>(u + b * QK_K + 4 * lane);
  float v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float gg = gv[k];
    const float silu = gg / (1.0f + exp_f32(-gg));
    v[k] = silu * uv[k];
  }
  store_q8k_block(v, true, lane, out + b);
}

hipError_t launch_swiglu_quant(const float* g, const float* u, int dim, BlockQ8K* out, hipStream_t s) {
  hipLaunchKernelGGL(k_swiglu_quant, dim3(dim / QK_K), dim3(64), 0, s, g, u, out);
  return hipGetLastError();
}

// apply_rope for every head with a host-built (cos, sin) row for pos, held in
// the kernel's arguments: no copy to the device comes before the launch.
// (device, when not null, holds the row instead: rows past RopeRow::MAX pairs.)
__global__ void k_rope(float* __restrict__ vec, const RopeRow row, const float2* __restrict__ device, int n_pairs,
                       int half_hd) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_pairs) return;
  const float2 c = device ? device[p % half_hd] : row.v[p % half_hd];
  const float v0 = vec[2 * p], v1 = vec[2 * p + 1];
  vec[2 * p] = v0 * c.x - v1 * c.y;
  vec[2 * p + 1] = v0 * c.y + v1 * c.x;
}

hipError_t launch_rope(float* vec, const RopeRow& row, const float2* device, int n_heads, int head_dim,
                       hipStream_t s) {
  if (!device && head_dim / 2 > RopeRow::MAX) return hipErrorInvalidValue;
  const int n_pairs = n_heads * head_dim / 2;
  hipLaunchKernelGGL(k_rope, dim3((n_pairs + 255) / 256), dim3(256), 0, s, vec, row, device, n_pairs,
                     head_dim / 2);
  return hipGetLastError();
}

__global__ void k_kv_append(const float* __restrict__ k, const float* __restrict__ v, float* __restrict__ kc,
                            float* __restrict__ vc, int pos, int kvd) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= kvd) return;
  const size_t o = static_cast<size_t>(pos) * kvd + i;
  kc[o] = k[i];
  vc[o] = v[i];
}

hipError_t launch_kv_append(const float* k, const float* v, float* kc, float* vc, int pos, int kvd,
                            hipStream_t s) {
  hipLaunchKernelGGL(k_kv_append, dim3((kvd + 255) / 256), dim3(256), 0, s, k, v, kc, vc, pos, kvd);
  return hipGetLastError();
}


template <int HDM, bool WL>
__global__ void __launch_bounds__(256) k_attention(const float* __restrict__ q, const float* __restrict__ kc,
                                                   const float* __restrict__ vc, const int* __restrict__ state,
                                                   int n_heads, int n_kv_heads, int hd, int max_chunks,
                                                   float* __restrict__ part_o, float2* __restrict__ part_mz,
                                                   int pos) {
  __shared__ __attribute__((aligned(16))) float lds[AttnLds<HDM>::bytes / sizeof(float)];
  // the position: given (pos >= 0), or the step state's
  const int T = (pos >= 0 ? pos : state[1]) + 1;
  AttnRegs<HDM / 16> R;
  attn_split<HDM, false, WL>(q, kc, vc, T, static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y), n_heads,
                         n_kv_heads, hd, max_chunks, part_o, part_mz, AttnLds<HDM>(lds), R, false);
}

static_assert(ATTN_Q8K_MAX_CHUNKS == ATTN_CPW, "one work group holds every chunk's o_c in registers");

// Decode, contexts of at most ATTN_CPW chunks, head_dim 64: one work group of
// four 256-thread groups per kv head.  Group g runs chunks g and g + 4 (the
// splits' arithmetic, attn_token_chunk on its own staged K and V rows; the
// query rows are shared), the groups' waves sharing each SIMD; then the work
// group combines the chunks with the consumers' arithmetic (m = max m_c;
// f_c = exp(m_c - m); Z = fma(z_c, f_c, Z); O = fma(o_c, f_c, O); O / Z) and
// quantizes its heads' outputs ties-even into Q8_K blocks (the group's
// gh = group*64 values are gh/256 whole blocks: block kvh*gh/256 + r), so
// the O projection reads them as they are.  A longer context sets *err and
// writes nothing.
constexpr int AQ_GROUPS = 4;
struct AttnQ8kLds {
  static constexpr int K = ATTN_CHUNK * 68, V = ATTN_CHUNK * 64, E = ATTN_MAX_GROUP * ATTN_CHUNK;
  static constexpr int PER = K + V + E;                        // floats per group
  static constexpr int Q = ATTN_MAX_GROUP * 64;
  static constexpr int MZ = ATTN_CPW * ATTN_MAX_GROUP;        // float2
  static constexpr size_t bytes = (AQ_GROUPS * PER + Q) * sizeof(float) + MZ * sizeof(float2);
};

__global__ void __launch_bounds__(256 * AQ_GROUPS) k_attention_q8k(const float* __restrict__ q,
                                                                   const float* __restrict__ kc,
                                                                   const float* __restrict__ vc,
                                                                   const int* __restrict__ state, int n_heads,
                                                                   int n_kv_heads, BlockQ8K* __restrict__ out,
                                                                   unsigned* __restrict__ err) {
  constexpr int HDM = 64, NV = HDM / 16, OPT = ATTN_MAX_GROUP * HDM / 256, KS = HDM + 4;
  using L = AttnQ8kLds;
  __shared__ __attribute__((aligned(16))) float lds[L::bytes / sizeof(float)];
  const int T = state[1] + 1;
  const int nch = (T + ATTN_CHUNK - 1) / ATTN_CHUNK;
  if (nch > ATTN_CPW) {  // uniform: before any barrier
    if (blockIdx.x == 0 && threadIdx.x == 0) *err = 1u;
    return;
  }
  const int tid = threadIdx.x, g = tid >> 8, t = tid & 255, kvh = blockIdx.x;
  const int hd = HDM, group = n_heads / n_kv_heads, gh = group * hd, kvd = n_kv_heads * hd;
  const int r4 = hd / 4, nf4 = ATTN_CHUNK * r4;
  const float scale = 1.0f / sqrtf(static_cast<float>(hd));
  const size_t head_off = static_cast<size_t>(kvh) * hd;
  float* sK = lds + g * L::PER;
  float* sV = sK + L::K;
  float* sE = sV + L::V;
  float* sQ = lds + AQ_GROUPS * L::PER;
  float2* sMZ = reinterpret_cast<float2*>(sQ + L::Q);
  AttnRegs<NV> R;
  if (g < nch) attn_load_chunk<NV>(R, kc, vc, g, T, kvd, head_off, r4, nf4, t);  // uniform in the group
  if (g == 0) {  // group 0 stages the queries for every group
    const float* qg = q + static_cast<size_t>(kvh) * gh;
#pragma unroll
    for (int u = 0; u < OPT; ++u) {
      const int i = min(t + 256 * u, gh - 1);  // threads past the queries store query gh-1 again
      sQ[(i / hd) * HDM + i % hd] = qg[i];
    }
  }
  const int rounds = (nch + AQ_GROUPS - 1) / AQ_GROUPS;  // 1 or 2
  float oc[2][OPT];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if (r < rounds) {  // uniform
      // chunk c of group g; a group past the context (c >= nch, uniform in
      // the group) loads, stages and computes nothing and only keeps the
      // barriers
      const int c = g + AQ_GROUPS * r;
      __syncthreads();  // readers of the previous chunk are done
      if (c < nch) {
#pragma unroll
        for (int u = 0; u < NV; ++u) {
          const int f = min(t + 256 * u, nf4 - 1);
          const int j = f / r4, c4 = f - j * r4;
          *reinterpret_cast<f32x4*>(&sK[j * KS + c4 * 4]) = R.k[u];
          *reinterpret_cast<f32x4*>(&sV[j * HDM + c4 * 4]) = R.v[u];
        }
        if (c + AQ_GROUPS < nch) attn_load_chunk<NV>(R, kc, vc, c + AQ_GROUPS, T, kvd, head_off, r4, nf4, t);
      }
      __syncthreads();
      if (c < nch)
        attn_token_chunk<HDM, OPT, true>(sK, sV, sQ, sE, sMZ + c * ATTN_MAX_GROUP, c, T, group, hd, gh, scale, oc[r], t);
    }
  }
  // every chunk's o_c into the staging area (each group's own K rows: its
  // readers are done after the barrier), o_c of chunk c at sO[c*gh + oi]
  __syncthreads();
  float* sO = lds;  // ATTN_CPW * 512 floats at most: within group 0's K and V rows
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int c = g + AQ_GROUPS * r;
    if (r < rounds && c < nch) {
#pragma unroll
      for (int u = 0; u < OPT; ++u) {
        const int oi = t + 256 * u;
        if (oi < gh) sO[c * gh + oi] = oc[r][u];
      }
    }
  }
  __syncthreads();
  float* sX = lds + 2 * L::PER;  // group 2's area: gh floats
  if (tid < gh) {
    const int oi = tid, hh = oi / hd;
    float m = sMZ[hh].x;
    for (int cc = 1; cc < nch; ++cc) m = fmaxf(m, sMZ[cc * ATTN_MAX_GROUP + hh].x);
    float Z = 0.0f, O = 0.0f;
    for (int cc = 0; cc < nch; ++cc) {
      const float2 mz = sMZ[cc * ATTN_MAX_GROUP + hh];
      const float f = exp_f32(mz.x - m);
      Z = __builtin_fmaf(mz.y, f, Z);
      O = __builtin_fmaf(sO[cc * gh + oi], f, O);
    }
    sX[oi] = O / Z;
  }
  __syncthreads();
  // block r of the group on row r (16 lanes) of wave 0, lane j holding
  // values 16j .. 16j+15: the GEMV prologue's quantization
  const int row = tid >> 4, j = tid & 15;
  if (tid < 64 && 256 * row < gh) {
    float v[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4 x4 = *reinterpret_cast<const f32x4*>(&sX[256 * row + 16 * j + 4 * i]);
      v[4 * i] = x4.x;
      v[4 * i + 1] = x4.y;
      v[4 * i + 2] = x4.z;
      v[4 * i + 3] = x4.w;
    }
    u32x4 packed;
    float d;
    int gsum;
    quant_block_row16(v, false, packed, d, gsum);
    BlockQ8K* blk = out + kvh * (gh / QK_K) + row;
    uint32_t* qs = reinterpret_cast<uint32_t*>(blk->qs) + 4 * j;  // 4-byte aligned
    qs[0] = packed.x;
    qs[1] = packed.y;
    qs[2] = packed.z;
    qs[3] = packed.w;
    blk->bsums[j] = static_cast<int16_t>(gsum);
    if (j == 0) blk->d = d;
  }
}

// Prefill: chunk blockIdx.y of kv head blockIdx.x for the tile of tt
// consecutive tokens from blockIdx.z * tt (token z at position pos0 + z,
// its own q and partials).  The chunk's K and V rows are staged once; a wave
// then takes 16 rows at a time, a row being one query head of one of the
// tile's tokens whose context reaches the chunk, and writes their partials.
//
// The score chains and the weighted V chains run on v_mfma_f32_16x16x4_f32:
// its result is the chain of four fmas over k in order, each rounded to
// nearest even with denormals kept (6 million results over normal, widely
// spread, underflowing, denormal and cancelling operands, none different:
// tests/cpp/mfma_check.hip), so a token's scores and o_c have the bits of the
// decode attention's fma chains.  Positions past a
// token's context score -1e9 and weigh 0; a 0 leaves the V chain as it is if
// that V is finite, so a chunk with an infinity or NaN in V takes the plain
// chains instead.  Layouts: A lane l holds row l%16, k = l/16; B column l%16, k
// = l/16; D register i row 4*(l/16) + i, column l%16.  K, V and the softmax
// terms are stored so that the 64 lanes of an operand read hit 64 banks.
//
// Of 90 us per launch for 1023 tokens and 32 heads of 64, a SIMD spends 28 in
// MFMAs (32 cycles each, 128 per 16 rows and chunk) and 39 issuing the other
// vector instructions (softmax, addresses); the rest is waiting, for what is not
// measured.  The fma chains it replaces, one lane per (head, position) and (head,
// dim): 131 us; 16 heads of 128 over 332 tokens 51.7 -> 24.6.
template <int HDM, bool FULL>
__global__ void __launch_bounds__(256) k_attention_tile(const float* __restrict__ q, const float* __restrict__ kc,
                                                        const float* __restrict__ vc, int n_heads, int n_kv_heads,
                                                        int head_dim, int max_chunks, float* __restrict__ part_o,
                                                        float2* __restrict__ part_mz, int pos0, int n_tok, int tt,
                                                        size_t tok_q, size_t tok_o, size_t tok_mz) {
  constexpr int NV = HDM / 16, NS = HDM / 4, ND = HDM / 16;
  __shared__ __attribute__((aligned(16))) float sK[ATTN_CHUNK * HDM];
  __shared__ __attribute__((aligned(16))) float sV[ATTN_CHUNK * HDM];
  __shared__ __attribute__((aligned(16))) float s_e[4][16 * ATTN_CHUNK];
  const int hd = FULL ? HDM : head_dim;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kvh = blockIdx.x, c = blockIdx.y;
  const int z0 = static_cast<int>(blockIdx.z) * tt;
  const int zlo = max(z0, c * ATTN_CHUNK - pos0);  // first token with pos0 + z + 1 > c * ATTN_CHUNK
  const int zhi = min(z0 + tt, n_tok);
  if (zlo >= zhi) return;
  const int group = n_heads / n_kv_heads;
  const int kvd = n_kv_heads * hd;
  const int r4 = hd / 4, nf4 = ATTN_CHUNK * r4;
  const float scale = 1.0f / sqrtf(static_cast<float>(hd));
  const int rows = (zhi - zlo) * group;
  // row f is head f % group of token zlo + f / group (f < 2^13, group <= 8:
  // the product's error stays below one)
  const uint32_t inv = 65536u / static_cast<uint32_t>(group) + 1u;
  auto row_token = [&](int f) { return static_cast<int>((static_cast<uint32_t>(f) * inv) >> 16); };

  AttnRegs<NV> R;
  attn_load_chunk<NV>(R, kc, vc, c, pos0 + zhi, kvd, static_cast<size_t>(kvh) * hd, r4, nf4);
  float qa[NS];  // A operands: query row c16 of a row tile, dims 4s + g
  auto load_q = [&](int rt) {
    const int f = min(rt * 16 + c16, rows - 1), z = row_token(f);
    const float* p = q + static_cast<size_t>(zlo + z) * tok_q + static_cast<size_t>(kvh * group + f - z * group) * hd + g;
#pragma unroll
    for (int s = 0; s < NS; ++s) qa[s] = p[FULL ? 4 * s : 4 * min(s, r4 - 1)];
  };
  load_q(wave);
  // K row j's dims 4s .. 4s+3 at quad s ^ (j % 16), V row j's dims 16d ..
  // 16d+15 at 16-float group d ^ (j % 4)
  bool bad = false;
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int f = min(tid + 256 * u, nf4 - 1);
    const int j = f / r4, c4 = f - j * r4;
    *reinterpret_cast<f32x4*>(&sK[j * HDM + ((c4 ^ (j & 15)) << 2)]) = R.k[u];
    *reinterpret_cast<f32x4*>(&sV[j * HDM + (((c4 >> 2) ^ (j & 3)) << 4) + ((c4 & 3) << 2)]) = R.v[u];
#pragma unroll
    for (int i = 0; i < 4; ++i) bad = bad || !(fabsf(R.v[u][i]) <= 3.402823466e38f);
  }
  float* sE = s_e[wave];
  const bool wave_bad = __builtin_amdgcn_ballot_w64(bad) != 0;  // of every lane: outside the branch
  if (lane == 0) sE[0] = wave_bad ? 1.0f : 0.0f;
  __syncthreads();
  const bool plain = (s_e[0][0] + s_e[1][0]) + (s_e[2][0] + s_e[3][0]) != 0.0f;
  __syncthreads();
  const f32x4 zero4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int rt = wave; rt * 16 < rows; rt += 4) {
    f32x4 S[4] = {zero4, zero4, zero4, zero4};
#pragma unroll
    for (int s = 0; s < NS; ++s) {
#pragma unroll
      for (int p = 0; p < 4; ++p)
        if (FULL || s < r4)
          S[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[s], sK[(16 * p + c16) * HDM + ((s ^ c16) << 2) + g], S[p], 0, 0, 0);
    }
    if ((rt + 4) * 16 < rows) load_q(rt + 4);
    // rows 4g+i of the lane: their positions 16p + c16
    float* po[4];
    int nt[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int f = min(rt * 16 + 4 * g + i, rows - 1), z = row_token(f), h = kvh * group + f - z * group;
      const size_t pc = static_cast<size_t>(h) * max_chunks + c;
      po[i] = part_o + static_cast<size_t>(zlo + z) * tok_o + pc * hd;
      nt[i] = min(ATTN_CHUNK, pos0 + zlo + z + 1 - c * ATTN_CHUNK);
      float sv[4], e[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) sv[p] = 16 * p + c16 < nt[i] ? S[p][i] * scale : -1e9f;
      const float mc = fmaxf(row16_max(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]))), -1e9f);
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        e[p] = 16 * p + c16 < nt[i] ? exp_f32(sv[p] - mc) : 0.0f;
        // row r's positions 4s .. 4s+3 at quad s ^ r
        sE[(4 * g + i) * ATTN_CHUNK + (((4 * p + (c16 >> 2)) ^ (4 * g + i)) << 2) + (c16 & 3)] = e[p];
      }
      // wave_tree_sum's tree over the 64 positions (slots t and t+32, then
      // t+16, then within 16), whole on the row's first lane
      float zs = (e[0] + e[2]) + (e[1] + e[3]);
      zs = zs + dpp_f<0x108>(zs);
      zs = zs + dpp_f<0x104>(zs);
      zs = zs + dpp_f<0x102>(zs);
      zs = zs + dpp_f<0x101>(zs);
      if (c16 == 0 && rt * 16 + 4 * g + i < rows) part_mz[static_cast<size_t>(zlo + z) * tok_mz + pc] = make_float2(mc, zs);
    }
    wave_sync();
    const int last = pos0 + zlo + row_token(min(rt * 16 + 15, rows - 1)) + 1 - c * ATTN_CHUNK;  // the tile's longest
    if (!plain) {
      f32x4 O[ND];
#pragma unroll
      for (int d = 0; d < ND; ++d) O[d] = zero4;
      const int ns = (min(ATTN_CHUNK, last) + 3) >> 2;
#pragma unroll 4
      for (int s = 0; s < ns; ++s) {
        const float a = sE[c16 * ATTN_CHUNK + ((s ^ c16) << 2) + g];
#pragma unroll
        for (int d = 0; d < ND; ++d)
          O[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, sV[(4 * s + g) * HDM + ((d ^ g) << 4) + c16], O[d], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (rt * 16 + 4 * g + i < rows) {
#pragma unroll
          for (int d = 0; d < ND; ++d)
            if (FULL || 16 * d + c16 < hd) po[i][16 * d + c16] = O[d][i];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (rt * 16 + 4 * g + i < rows) {
          for (int d = c16; d < hd; d += 16) {
            float acc = 0.0f;
            for (int j = 0; j < nt[i]; ++j)
              acc = __builtin_fmaf(sE[(4 * g + i) * ATTN_CHUNK + (((j >> 2) ^ (4 * g + i)) << 2) + (j & 3)],
                                   sV[j * HDM + (((d >> 4) ^ (j & 3)) << 4) + (d & 15)], acc);
            po[i][d] = acc;
          }
        }
      }
    }
    wave_sync();  // the reads of sE, before the next row tile's terms
  }
}

// The combine over a head's chunks for output i (head h, dim d), in chunk
// order: m = max m_c; f_c = exp(m_c - m); Z = fma(z_c, f_c, Z);
// O = fma(o_c[d], f_c, O); out = O / Z.  One wave per 64 outputs of a head.
// Lane c holds chunk c's (m_c, z_c) and forms f_c once for the wave (each
// output formed every f_c itself before, an exp between each two loads); the
// chains read it by lane, and the o_c of COMBINE_BATCH chunks are loaded
// together, the first ones before the maximum (one chunk has nothing else to
// wait for: 64 heads of 64 at up to 64 positions, a decoded layer 51.1 -> 50.8 us,
// 50.2 with a thread per output and no lane moves).  Average over 32 heads of 64
// at 9 chunks and 16 of 128 at 63: 22.9 -> 4.5 us.
constexpr int COMBINE_BATCH = 16;

__global__ void __launch_bounds__(64) k_attn_combine(const float* __restrict__ part_o,
                                                     const float2* __restrict__ part_mz,
                                                     const int* __restrict__ state, int pos, int hd, int max_chunks,
                                                     float* __restrict__ out) {
  const int nch = (pos >= 0 ? pos : state[1]) / ATTN_CHUNK + 1;
  const int h = blockIdx.x, lane = threadIdx.x, d = blockIdx.y * 64 + lane;
  const float2* mz = part_mz + static_cast<size_t>(h) * max_chunks;
  // lanes past the head's dims repeat its last one (unused)
  const float* o = part_o + static_cast<size_t>(h) * max_chunks * hd + min(d, hd - 1);
  // lanes past the last chunk hold it again: the maximum is unchanged, and
  // the chains stop before them
  float2 cur = mz[min(lane, nch - 1)];
  float ov[COMBINE_BATCH];
  auto load_o = [&](int c) {
#pragma unroll
    for (int k = 0; k < COMBINE_BATCH; ++k) ov[k] = o[static_cast<size_t>(min(c + k, nch - 1)) * hd];
  };
  load_o(0);  // in flight beside the maximum
  float m = cur.x;
  for (int c0 = 64; c0 < nch; c0 += 64) m = fmaxf(m, mz[min(c0 + lane, nch - 1)].x);
  m = wave_max_fast(m);
  float Z = 0.0f, O = 0.0f;
  for (int c0 = 0; c0 < nch; c0 += 64) {
    if (c0 > 0) cur = mz[min(c0 + lane, nch - 1)];
    const float f = exp_f32(cur.x - m);
    const int n = min(64, nch - c0);
    for (int j0 = 0; j0 < n; j0 += COMBINE_BATCH) {
      if (c0 + j0 > 0) load_o(c0 + j0);
#pragma unroll
      for (int k = 0; k < COMBINE_BATCH; ++k) {
        if (j0 + k < n) {  // uniform
          const float fc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), j0 + k));
          const float zc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cur.y), j0 + k));
          Z = __builtin_fmaf(zc, fc, Z);
          O = __builtin_fmaf(ov[k], fc, O);
        }
      }
    }
  }
  if (d < hd) out[static_cast<size_t>(h) * hd + d] = O / Z;
}

hipError_t launch_attention(const float* q, const float* kc, const float* vc, const int* state, int n_heads,
                            int n_kv_heads, int head_dim, int max_chunks, const AttnPart& part, hipStream_t s,
                            int pos) {
  if (head_dim <= 0 || head_dim > 128 || head_dim % 4 || n_heads % n_kv_heads ||
      n_heads / n_kv_heads > ATTN_MAX_GROUP)
    return hipErrorInvalidValue;
  // a given position needs its own splits only; the step state's may be any
  const dim3 grid(n_kv_heads, pos >= 0 ? attn_splits(pos / ATTN_CHUNK + 1) : attn_max_splits(1, max_chunks));
  if (head_dim <= 64)
    launch_kernel(head_dim == 64 ? k_attention<64, true> : k_attention<64, false>, grid, dim3(256), 0, s, q, kc, vc,
                  state, n_heads, n_kv_heads, head_dim,
                  max_chunks, part.o, part.mz, pos);
  else
    launch_kernel(k_attention<128, false>, grid, dim3(256), 0, s, q, kc, vc, state, n_heads, n_kv_heads, head_dim,
                  max_chunks, part.o, part.mz, pos);
  return hipGetLastError();
}

hipError_t launch_attention_q8k(const float* q, const float* kc, const float* vc, const int* state, int n_heads,
                                int n_kv_heads, int head_dim, BlockQ8K* out, unsigned* err, hipStream_t s) {
  if (!attn_q8k_fits(n_heads, n_kv_heads, head_dim)) return hipErrorInvalidValue;
  launch_kernel(k_attention_q8k, dim3(n_kv_heads), dim3(256 * AQ_GROUPS), 0, s, q, kc, vc, state, n_heads, n_kv_heads,
                out, err);
  return hipGetLastError();
}

hipError_t launch_attention_batch(const float* q, const float* kc, const float* vc, int n_heads, int n_kv_heads,
                                  int head_dim, int max_chunks, const AttnPart& part, size_t tok_o, size_t tok_mz,
                                  int pos0, int n_tok, hipStream_t s) {
  if (head_dim <= 0 || head_dim > 128 || head_dim % 4 || n_heads % n_kv_heads ||
      n_heads / n_kv_heads > ATTN_MAX_GROUP || pos0 < 0)
    return hipErrorInvalidValue;
  if (n_tok <= 0) return hipSuccess;
  // one work group per (kv head, chunk, token tile); tiles whose tokens do
  // not reach a chunk return at once.  A tile is the whole tokens of one row tile
  // per wave, 64 rows at most: more rows per wave, to stage K and V for more
  // tokens, were slower at every length (1023 tokens, 4 heads per kv head: a
  // prompt in 18.88 ms with 16 tokens, 19.01 with 32, 19.17 with 64; 332 tokens, 8
  // heads: 7.31 with 8, 8.10 with 32), half of it too beyond 332 tokens (1023:
  // 21.0).  Rounded up instead, groups of 3, 5, 6 and 7 heads gave one wave a
  // second row tile of 1 to 6 rows (four layers, 7 heads of 128 per kv head, 1023
  // tokens: 1681 us, 1440 rounded down; 3 heads of 64: 531, 482).
  const int group = n_heads / n_kv_heads, nch = (pos0 + n_tok - 1) / ATTN_CHUNK + 1;
  const int tt = 64 / group;
  const dim3 grid(n_kv_heads, nch, (n_tok + tt - 1) / tt);
  const size_t tok_q = static_cast<size_t>(n_heads) * head_dim;
  auto kern = head_dim == 64    ? k_attention_tile<64, true>
              : head_dim == 128 ? k_attention_tile<128, true>
              : head_dim < 64   ? k_attention_tile<64, false>
                                : k_attention_tile<128, false>;
  launch_kernel(kern, grid, dim3(256), 0, s, q, kc, vc, n_heads, n_kv_heads, head_dim, max_chunks, part.o, part.mz, pos0,
                n_tok, tt, tok_q, tok_o, tok_mz);
  return hipGetLastError();
}

hipError_t launch_attn_combine(const AttnPart& part, const int* state, int n_heads, int head_dim, int max_chunks,
                               float* out, hipStream_t s, int pos) {
  hipLaunchKernelGGL(k_attn_combine, dim3(n_heads, (head_dim + 63) / 64), dim3(64), 0, s, part.o, part.mz, state,
                     pos, head_dim, max_chunks, out);
  return hipGetLastError();
}

__global__ void k_dequant_rows(const WView w, int row0, int n_rows, int cols, float* __restrict__ out) {
  const int r = row0 + blockIdx.y;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < cols; i += gridDim.x * blockDim.x) {
    float v;
    if (w.type == MCPM_TYPE_Q8_0) {
      const size_t blk = static_cast<size_t>(i / QK8_0) * w.rows + r;
      const int8_t q = static_cast<int8_t>(w.p0[blk * 32 + i % QK8_0]);
      const uint16_t dh = w.p1[blk * 2] | (w.p1[blk * 2 + 1] << 8);
      v = fp16_to_fp32(dh) * static_cast<float>(q);
    } else if (w.type == MCPM_TYPE_F32) {
      v = reinterpret_cast<const float*>(w.p0)[static_cast<size_t>(r) * cols + i];
    } else {
      v = dequant_value(w, r, i / QK_K, i % QK_K);
    }
    out[static_cast<size_t>(blockIdx.y) * cols + i] = v;
  }
}

hipError_t launch_dequant_rows(const WView& w, int row0, int n_rows, int cols, float* out, hipStream_t s) {
  hipLaunchKernelGGL(k_dequant_rows, dim3((cols + 255) / 256, n_rows), dim3(256), 0, s, w, row0, n_rows, cols, out);
  return hipGetLastError();
}

// get_embedding: row `token` (when negative: the step state's) dequantized to x; one
// work group per 256-value block, one value per thread.  epoch (optional):
// advanced by one, by one thread.
__global__ void __launch_bounds__(256) k_embedding(const WView w, const int* __restrict__ state, int token,
                                                   int dim, float* __restrict__ out, unsigned* epoch) {
  if (token < 0) token = state[0];
  const int i = blockIdx.x * QK_K + threadIdx.x;
  if (i < dim) out[i] = dequant_value(w, token, blockIdx.x, threadIdx.x);
  if (epoch && i == 0) epoch[0] = epoch[0] + 1u;
}

hipError_t launch_embedding(const WView& w, const int* state, int dim, float* out, hipStream_t s,
                            unsigned* epoch, int token) {
  hipLaunchKernelGGL(k_embedding, dim3((dim + QK_K - 1) / QK_K), dim3(QK_K), 0, s, w, state, token, dim, out, epoch);
  return hipGetLastError();
}

// ------------------------------------------------- fp32-activation GEMVs ----
// gemv_f32 (src/ops/ops.cpp:32-43): lane t sums w*x over c = t, t+64, ...
// (multiply then add), then the 64-lane pairwise tree.  One wave per row; up to
// 16 steps' loads are issued together (the sum then runs over them in order),
// so a wave keeps 2 * 16 * 256 bytes in flight where a load per step waited for
// memory every few terms.  What a row leaves past whole 16s runs as an 8, a 4
// and up to four more steps.  The split depends on the column count alone, not
// on a lane's own column: that sent lanes 0-39 of a row of 1000 through 16 steps
// together and the others through 15 one by one.  A load per step throughout,
// split by the lane's column, this: 32768 x 1000 25.5, 47.3, 21.6 us; 8192 x
// 2047 12.7, 14.2, 12.5; 2304 x 2304 5.4, 3.7, 3.7; 8192 x 5760 32.7, 29.9, 28.9
// (6.5 TB/s).
// N steps from column c on.  LAST: the row may end among them (the columns past
// it read the row's last, unused).
template <int N, bool LAST = false>
__device__ __forceinline__ float f32_steps(const float* __restrict__ wr, const float* __restrict__ x, int c, int cols,
                                           float p) {
  float wv[N], xv[N];
#pragma unroll
  for (int k = 0; k < N; ++k) wv[k] = __builtin_nontemporal_load(wr + (LAST ? min(c + 64 * k, cols - 1) : c + 64 * k));
#pragma unroll
  for (int k = 0; k < N; ++k) xv[k] = x[LAST ? min(c + 64 * k, cols - 1) : c + 64 * k];
#pragma unroll
  for (int k = 0; k < N; ++k)
    if (!LAST || c + 64 * k < cols) p = p + wv[k] * xv[k];
  return p;
}

// SHORT: rows of at most three steps, one by one (32768 x 64: 3.6 us, 3.9 with
// the batches in the kernel).
constexpr int F32_SHORT = 3 * 64;

template <bool SHORT>
__global__ void __launch_bounds__(256) k_gemv_f32(const float* __restrict__ w, const float* __restrict__ x,
                                                  float* __restrict__ out, int rows, int cols) {
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= rows) return;
  const float* wr = w + static_cast<size_t>(r) * cols;
  float p = 0.0f;
  int c = lane, left = cols;
  if constexpr (!SHORT) {
    constexpr int S = 64;  // columns a step
    const int c16 = (cols & ~(16 * S - 1)) + lane;
    for (; c < c16; c += 16 * S) p = f32_steps<16>(wr, x, c, cols, p);
    left = cols & (16 * S - 1);
    if (left >= 8 * S) {
      p = f32_steps<8>(wr, x, c, cols, p);
      c += 8 * S;
      left -= 8 * S;
    }
    if (left >= 4 * S) {
      p = f32_steps<4>(wr, x, c, cols, p);
      c += 4 * S;
      left -= 4 * S;
    }
  }
  if (!SHORT && left > 2 * 64)
    p = f32_steps<4, true>(wr, x, c, cols, p);
  else
    for (; c < cols; c += 64) p = p + wr[c] * x[c];
  p = wave_tree_sum(p);
  if (lane == 0) out[r] = p;
}

hipError_t launch_gemv_f32(const float* w, const float* x, float* out, int rows, int cols, hipStream_t s) {
  hipLaunchKernelGGL(cols <= F32_SHORT ? k_gemv_f32<true> : k_gemv_f32<false>, dim3((rows + 3) / 4), dim3(256), 0, s, w,
                     x, out, rows, cols);
  return hipGetLastError();
}

// Read-only pass: every 16-byte word of src once (non-temporal loads, as the
// GEMVs stream their weights), a grid-stride loop over `grid` work groups; one
// xor per work group goes to out so the loads stay.  Its duration is the floor
// of one launch that reads as many bytes as a GEMV class.
__global__ void __launch_bounds__(256) k_stream_read(const u32x4* __restrict__ src, size_t n16,
                                                     uint32_t* __restrict__ out) {
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  uint32_t acc = 0;
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n16; i += stride) {
    const u32x4 v = __builtin_nontemporal_load(src + i);
    acc ^= v.x ^ v.y ^ v.z ^ v.w;
  }
  __shared__ uint32_t s[256];
  s[threadIdx.x] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t a = 0;
    for (int t = 0; t < 256; ++t) a ^= s[t];
    out[blockIdx.x] = a;
  }
}

hipError_t launch_stream_read(const void* src, size_t bytes, int grid, uint32_t* out, hipStream_t s) {
  launch_kernel(k_stream_read, dim3(grid), dim3(256), 0, s, static_cast<const u32x4*>(src), bytes / 16, out);
  return hipGetLastError();
}

// gemv_q8_0 (src/ops/ops.cpp:58-79): per block s = sum over i of float(q_i)*x_i
// (i ascending, multiply then add); row = row + s*d over blocks in order.
//
// The blocks' sums s do not depend on each other, only the row chain does: a
// lane takes one (row, block), a work group ROWS rows and 256 / ROWS blocks a
// step, and leaves s*d in LDS; after up to 2048 / ROWS blocks one lane per row
// runs the chain over them.  Consecutive lanes take consecutive rows, whose
// 32-byte codes are consecutive (256-byte runs with 8 rows).  8 rows a work
// group: 288 work groups at 2304 rows.  Bound by load latency.  One lane per
// whole row gave 9 work groups at 2304 rows: 2304 x 5760 52.7 -> 7.6 us, 1000 x
// 1024 10.8 -> 3.8, 8192 x 6144 87.0 -> 20.9 (53.7 MB, 2.6 TB/s).
template <int ROWS>
__global__ void __launch_bounds__(256) k_gemv_q8_0(const WView w, const float* __restrict__ x,
                                                   float* __restrict__ out, int rows, int cols) {
  constexpr int PAR = 256 / ROWS, CHUNK = 2048 / ROWS;
  __shared__ float sp[ROWS][CHUNK + 1];
  const int tid = threadIdx.x, rr = tid % ROWS, bl = tid / ROWS;
  const int r = blockIdx.x * ROWS + rr;
  const int rc = min(r, rows - 1);  // lanes past the last row repeat it (unused)
  const int nb = cols / QK8_0;
  float row = 0.0f;
  for (int c0 = 0; c0 < nb; c0 += CHUNK) {
    const int c1 = min(c0 + CHUNK, nb);
#pragma unroll 2
    for (int b = c0 + bl; b < c1; b += PAR) {
      const size_t blk = static_cast<size_t>(b) * w.rows + rc;
      u32x4 q4[2];
      q4[0] = ld_stream4(w.p0 + blk * 32);
      q4[1] = ld_stream4(w.p0 + blk * 32 + 16);
      const uint16_t dh = ld_stream_u16(w.p1 + blk * 2);
      f32x4_u xv[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) xv[k] = *reinterpret_cast<const f32x4_u*>(x + b * QK8_0 + 4 * k);
      float s = 0.0f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t q = q4[k >> 2][k & 3];
#pragma unroll
        for (int i = 0; i < 4; ++i) s = s + static_cast<float>(static_cast<int8_t>(q >> (8 * i))) * xv[k][i];
      }
      sp[rr][b - c0] = s * fp16_to_fp32(dh);
    }
    __syncthreads();
    if (tid < ROWS) {
#pragma unroll 8
      for (int b = 0; b < c1 - c0; ++b) row = row + sp[tid][b];
    }
    __syncthreads();  // the chain's reads before the next blocks' products
  }
  if (tid < ROWS && r < rows) out[r] = row;
}

// One lane per row: no LDS, no barrier, and x by scalar loads.
__global__ void __launch_bounds__(256) k_gemv_q8_0_rows(const WView w, const float* __restrict__ x,
                                                        float* __restrict__ out, int rows, int cols) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  const int nb = cols / QK8_0;
  float row = 0.0f;
  for (int b = 0; b < nb; ++b) {
    const size_t blk = static_cast<size_t>(b) * w.rows + r;
    const int8_t* q = reinterpret_cast<const int8_t*>(w.p0 + blk * 32);
    float s = 0.0f;
    for (int i = 0; i < QK8_0; ++i) s = s + static_cast<float>(q[i]) * x[b * QK8_0 + i];
    const uint16_t dh = w.p1[blk * 2] | (w.p1[blk * 2 + 1] << 8);
    row = row + s * fp16_to_fp32(dh);
  }
  out[r] = row;
}

// The more rows, the more of the chip they fill by themselves, and the less the
// split of a row's blocks is worth its barrier.  A lane per row where that is a
// wave for every SIMD (64 rows each; 65,536 rows on 256 CUs): 130560 x 1536 31.2
// us, with 8 rows a work group 64.4, with 32 50.7; 65536 x 2304 35.7, 54.5, 44.7
// (weights in the Infinity Cache; from HBM 50.0, 55.3, 45.8).  32 rows a work
// group where 8 would take more than 12 work groups per CU: 32768 x 2304 21.9
// us, with 8 rows 27.1, a lane per row 33.9; below that short rows lose by it
// (18000 x 512 4.4 us, with 8 rows 3.7; 12000 x 1024 5.2, 4.5).
hipError_t launch_gemv_q8_0(const WView& w, const float* x, float* out, int rows, int cols, int n_cu, hipStream_t s) {
  if (rows >= 256 * n_cu)
    hipLaunchKernelGGL(k_gemv_q8_0_rows, dim3((rows + 255) / 256), dim3(256), 0, s, w, x, out, rows, cols);
  else if (rows > 96 * n_cu)
    hipLaunchKernelGGL(k_gemv_q8_0<32>, dim3((rows + 31) / 32), dim3(256), 0, s, w, x, out, rows, cols);
  else
    hipLaunchKernelGGL(k_gemv_q8_0<8>, dim3((rows + 7) / 8), dim3(256), 0, s, w, x, out, rows, cols);
  return hipGetLastError();
}

// ------------------------------------------------------------- argmax ------
__global__ void __launch_bounds__(256) k_argmax_partial(const float* __restrict__ x, int n, float2* __restrict__ part) {
  __shared__ float sv[4];
  __shared__ int si[4];
  float bv = -__builtin_inff();
  int bi = 0x7fffffff;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const float v = x[i];
    if (v > bv || (v == bv && i < bi)) {
      bv = v;
      bi = i;
    }
  }
  for (int o = 32; o >= 1; o >>= 1) {
    const float ov = __shfl_xor(bv, o);
    const int oi = __shfl_xor(bi, o);
    if (ov > bv || (ov == bv && oi < bi)) {
      bv = ov;
      bi = oi;
    }
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sv[wave] = bv;
    si[wave] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 4; ++k)
      if (sv[k] > bv || (sv[k] == bv && si[k] < bi)) {
        bv = sv[k];
        bi = si[k];
      }
    part[blockIdx.x] = make_float2(bv, __int_as_float(bi));
  }
}

hipError_t launch_argmax_partial(const float* x, int n, float2* part, int nparts, hipStream_t s) {
  hipLaunchKernelGGL(k_argmax_partial, dim3(nparts), dim3(256), 0, s, x, n, part);
  return hipGetLastError();
}

// Reduces (value, index) partials to the first index of the maximum; writes
// it to out_token, and when a step state is given, feeds it back as the next
// input token, appends it to out_tokens and advances pos.
// Final argmax over the partials (value, index) of the LM-head work groups:
// the largest value, ties to the lowest index.  256 threads, loads issued 16
// at a time; slots past nparts re-read the last partial (harmless for a max).
__global__ void __launch_bounds__(256) k_argmax_final(const float2* __restrict__ part, int nparts,
                                                      int* __restrict__ out_token, StepState* st,
                                                      int* __restrict__ out_tokens) {
  __shared__ float s_v[4];
  __shared__ int s_i[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float bv = -__builtin_inff();
  int bi = 0x7fffffff;
  for (int i0 = tid; i0 < nparts; i0 += 256 * 16) {
    float2 v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = part[min(i0 + 256 * k, nparts - 1)];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float pv = v[k].x;
      const int pi = __float_as_int(v[k].y);
      if (pv > bv || (pv == bv && pi < bi)) {
        bv = pv;
        bi = pi;
      }
    }
  }
  for (int o = 32; o >= 1; o >>= 1) {
    const float ov = __shfl_xor(bv, o);
    const int oi = __shfl_xor(bi, o);
    if (ov > bv || (ov == bv && oi < bi)) {
      bv = ov;
      bi = oi;
    }
  }
  if (lane == 0) {
    s_v[wave] = bv;
    s_i[wave] = bi;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; ++w) {
      if (s_v[w] > bv || (s_v[w] == bv && s_i[w] < bi)) {
        bv = s_v[w];
        bi = s_i[w];
      }
    }
    if (out_token) *out_token = bi;
    if (st) {
      st->token = bi;
      st->pos = st->pos + 1;
      if (out_tokens && st->step < st->n_out) out_tokens[st->step] = bi;
      st->step = st->step + 1;
    }
  }
}

hipError_t launch_argmax_final(const float2* part, int nparts, int* out_token, StepState* st, int* out_tokens,
                               hipStream_t s) {
  hipLaunchKernelGGL(k_argmax_final, dim3(1), dim3(256), 0, s, part, nparts, out_token, st, out_tokens);
  return hipGetLastError();
}

__global__ void k_fill_f32(float* p, float v, size_t n) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

hipError_t launch_fill_f32(float* p, float v, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_f32, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, s, p, v, n);
  return hipGetLastError();
}

}  // namespace mcpm
