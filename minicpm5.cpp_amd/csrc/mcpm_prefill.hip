// mcpm_prefill.hip -- batched prompt processing (prefill) for gfx950.
//
// The reference prefills by calling forward() once per prompt token
// (src/chat_session.cpp:154-160).  Here the prompt's tokens go through each
// layer together, and every number that reaches the KV cache is the one the
// per-token decode path produces:
//  * activations are quantized per token exactly as the GEMV prologues do
//    (same RMS tree, same Q8_K rounding), into fp16 copies of the int8 codes;
//  * a row dot keeps the reference's AVX2 structure: per 256-block the eight
//    integer lane sums isum[m] (lane m: bytes 4m..4m+3 of every 32-byte
//    group), then acc[m] = fma(d_x*d_w, float(isum[m]), acc[m]) over blocks in
//    order, Q4_K's min chain, and ((a0+a4)+(a2+a6))+((a1+a5)+(a3+a7));
//  * isum[m] for 16 rows x 16 tokens is one v_mfma_f32_16x16x32_f16: K runs
//    over lane m's 32 bytes (8 sub-blocks x 4), activation code times 64 (the
//    MFMA's A) against sub-block scale x weight code over 64 (its B).  Every
//    product is an integer of at most 1920 * 127 in magnitude, its factors
//    exact in fp16, and every sum stays below 2^24 (exact in fp32), so the MFMA
//    result is isum[m] itself.  Q4_K: sc*q <= 945.
//    Q6_K: the reference sums sc*q*x over lane m's bytes (q in 0..63) and
//    subtracts 32*(sc[2m]*bsums[2m] + sc[2m+1]*bsums[2m+1]) -- sub-block m's
//    offset, added into lane m -- then converts the int32 sum to float.
//    Written as S + 16*T with q = ql + 16*qh (ql the low 4 bits, qh the high
//    2): S = sum over lane m of sc*ql*x (|sc*ql| <= 1920, |S| < 2^23), T =
//    sum over lane m of sc*qh*x - 2*C (|sc*qh| <= 384), C = sub-block m's
//    sc*bsums pair, fed in as T's accumulator from one more MFMA (|T| <
//    2^22).  Three MFMAs, all exact; fma(16, T, S) rounds S + 16*T once, to
//    nearest even, as the reference's int32 -> float conversion of the same
//    integer does.
//  * Q4_K's min sum (sum over sub-blocks of mn * pair-sum of bsums) is one
//    more MFMA: mn[k/2] for k < 16 against bsums[k].
// The attention (k_attention_tile, mcpm_kernels.hip) forms the decode attention's
// chains for tiles of tokens, and its partials are combined per token.
#include <algorithm>

#include "mcpm_device.h"

namespace mcpm {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

// ------------------------------------------------------------- embedding ---
// Row tokens[t] of the embedding, dequantized into x[t] (grid: blocks x tokens).
__global__ void __launch_bounds__(256) k_embed_batch(const WView w, const int* __restrict__ tokens, int dim,
                                                     float* __restrict__ x) {
  const int t = blockIdx.y;
  const int i = blockIdx.x * QK_K + threadIdx.x;
  if (i < dim) x[static_cast<size_t>(t) * dim + i] = dequant_value(w, tokens[t], blockIdx.x, threadIdx.x);
}

// ------------------------------------------------------------- quantize ----
// Per token (one work group each): the Q8_K quantization of the GEMV
// prologues, written as the GEMM's operands (store_codes).  mode:
// PRO_QUANT_EVEN / PRO_QUANT_AWAY / PRO_NORM_AWAY / PRO_NORM_EVEN; values from
// n_valid on quantize as 0.
// The quantized activations in the order the GEMM's MFMA operands want them,
// in tiles of 16 tokens: codes [tile][block][lane group m][K-half g][token of
// the tile][8 halves], the 8 halves being elements 64g + 4m .. +3 and 64g + 32
// + 4m .. +3 of the block, each code times 64 (exact in fp16; the weights'
// operands are divided by 64); d [tile][block][token]; bsums
// [tile][block][token][16].  A GEMM wave then reads a lane group's whole
// operand (64 lanes x 16 bytes) as one run of 1 KiB, with no staging in LDS.
// lane: the block's values 4*lane .. +3.
__device__ __forceinline__ void store_codes(int t, int nb, int b, int lane, uint32_t packed, float d, int gsum,
                                            _Float16* __restrict__ xh, float* __restrict__ xd,
                                            _Float16* __restrict__ xbs) {
  typedef _Float16 h4 __attribute__((ext_vector_type(4)));
  const size_t tb = static_cast<size_t>(t >> 4) * nb + b;
  const int c = t & 15, m = lane & 7, half = (lane >> 3) & 1, g = lane >> 4;
  h4 hv;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    hv[k] = static_cast<_Float16>(64.0f * static_cast<float>(static_cast<int8_t>((packed >> (8 * k)) & 0xffu)));
  *reinterpret_cast<h4*>(xh + (tb * 8 + m) * 512 + (16 * g + c) * 8 + 4 * half) = hv;
  if ((lane & 3) == 0) xbs[(tb * 16 + c) * 16 + (lane >> 2)] = static_cast<_Float16>(gsum);
  if (lane == 0) xd[tb * 16 + c] = d;
}

// The token of a quantization work group: a tile's 16 tokens share cache lines
// of the operand layout, so they go to one XCD (work group b runs on XCD b %
// 8), whose L2 puts the lines together.
__device__ __forceinline__ int quant_token(unsigned b) {
  const int xcd = static_cast<int>(b & 7), j = static_cast<int>(b >> 3);
  return 16 * (xcd + 8 * (j >> 4)) + (j & 15);
}
static dim3 quant_grid(int n_tok) { return dim3(128 * ((n_tok + 127) / 128)); }

__global__ void __launch_bounds__(256) k_quant_batch(const float* __restrict__ x, int ld_x,
                                                     const float* __restrict__ gamma, float eps, int dim,
                                                     int n_valid, int mode, int n_tok, _Float16* __restrict__ xh,
                                                     float* __restrict__ xd, _Float16* __restrict__ xbs) {
  __shared__ float red[260];
  const int t = quant_token(blockIdx.x);
  if (t >= n_tok) return;  // uniform, before any barrier
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float* xt = x + static_cast<size_t>(t) * ld_x;
  const bool norm = (mode == PRO_NORM_AWAY || mode == PRO_NORM_EVEN);
  const bool away = (mode == PRO_QUANT_AWAY || mode == PRO_NORM_AWAY);
  float rms = 1.0f;
  if (norm) rms = block_rms_scale(xt, dim, eps, red);
  const int nb = dim / QK_K;
  for (int b = wave; b < nb; b += 4) {
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = b * QK_K + 4 * lane + k;
      v[k] = i < n_valid ? xt[i] : 0.0f;
      if (norm) v[k] = (v[k] * rms) * gamma[i];
    }
    uint32_t packed;
    float d;
    int gsum;
    quant_block_wave(v, away, packed, d, gsum);
    store_codes(t, nb, b, lane, packed, d, gsum, xh, xd, xbs);
  }
}

// k_quant_batch for up to 4*MAXB blocks per token, with every global load
// issued at the start: wave w holds blocks w, w+4, ... (lane l: values 4l ..
// 4l+3 of each, with their gamma), RMSNorm's strided partials are read
// back from an LDS copy of the row (thread t: x[t], x[t+256], ... in order,
// as block_rms_scale sums them), and each block is quantized from registers.
// Same operations and outputs as k_quant_batch.
template <int MAXB>
__global__ void __launch_bounds__(256) k_quant_batch_r(const float* __restrict__ x, int ld_x,
                                                       const float* __restrict__ gamma, float eps, int dim,
                                                       int n_valid, int mode, int n_tok, _Float16* __restrict__ xh,
                                                       float* __restrict__ xd, _Float16* __restrict__ xbs) {
  __shared__ float red[260];
  __shared__ __attribute__((aligned(16))) float sx[4 * MAXB * QK_K];
  const int t = quant_token(blockIdx.x);
  if (t >= n_tok) return;  // uniform, before any barrier
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const float* xt = x + static_cast<size_t>(t) * ld_x;
  const bool norm = (mode == PRO_NORM_AWAY || mode == PRO_NORM_EVEN);
  const bool away = (mode == PRO_QUANT_AWAY || mode == PRO_NORM_AWAY);
  const int nb = dim / QK_K;
  // x and gamma; blocks past nb re-read the last, and values at or past
  // n_valid (a multiple of 4, checked by the launch; they quantize as 0) read
  // the last valid four, unused
  f32x4 xv[MAXB], wv[MAXB];
#pragma unroll
  for (int j = 0; j < MAXB; ++j) {
    const int i = min(min(wave + 4 * j, nb - 1) * QK_K + 4 * lane, n_valid - 4);
    xv[j] = *reinterpret_cast<const f32x4*>(xt + i);
    if (norm) wv[j] = *reinterpret_cast<const f32x4*>(gamma + i);
  }
  float rms = 1.0f;
  if (norm) {
#pragma unroll
    for (int j = 0; j < MAXB; ++j)
      if (wave + 4 * j < nb) *reinterpret_cast<f32x4*>(&sx[(wave + 4 * j) * QK_K + 4 * lane]) = xv[j];
    __syncthreads();
    float p = 0.0f;
    for (int k = 0; k < nb; ++k) {
      const float v = sx[k * QK_K + tid];
      p = p + v * v;
    }
    rms = block_rms_1sync(p, dim, eps, red);
  }
#pragma unroll
  for (int j = 0; j < MAXB; ++j) {
    const int b = wave + 4 * j;
    if (b >= nb) break;
    float v[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w};
    const float w4[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (norm) v[k] = (v[k] * rms) * w4[k];
      if (b * QK_K + 4 * lane + k >= n_valid) v[k] = 0.0f;
    }
    uint32_t packed;
    float d;
    int gsum;
    quant_block_wave(v, away, packed, d, gsum);
    store_codes(t, nb, b, lane, packed, d, gsum, xh, xd, xbs);
  }
}

// ------------------------------------------------------------------ GEMM ----
struct GemmArgs {
  WView w;
  int rows, nb, n_tok;
  // quantized activations in store_codes' layout (whole tiles of 16 tokens)
  const _Float16* xh;
  const float* xd;
  const _Float16* xbs;
  float* out;           // out[t*ld_out + r]
  int ld_out;
  int add;              // 1: out += v (residual), 0: out = v
  // an optional second matrix of the same type and blocks per row on the
  // same activations (rows2 > 0), written to out2 (row stride ld_out2)
  WView w2;
  int rows2;
  float* out2;
  int ld_out2;
  // rope != nullptr: every row pair (2i, 2i+1) of a matrix is rotated as
  // apply_rope does before it is stored (head_dim rope_hd, token t at
  // position pos0 + t, table rows of rope_hd/2 (cos, sin) pairs)
  const float2* rope;
  int rope_hd, pos0;
  // swiglu: the two matrices are gate and up (rows2 == rows); a work group
  // takes the same rows of both and writes h = silu(gate)*up (decode's
  // gate/up epilogue) to out
  int swiglu;
};

__device__ __forceinline__ uint32_t h2bits(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// A raw buffer resource over p (byte offsets up to 2 GB).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gemm_rsrc(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), static_cast<short>(0), 0x7fffffff, 0x00020000);
}

// fp16 pair (1024 + byte) of the bytes of t that sel picks
__device__ __forceinline__ h2 byte_pair(uint32_t t, uint32_t sel) {
  return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, t, sel));
}
constexpr uint32_t SEL01 = 0x04010400u, SEL23 = 0x04030402u;

// Eight halves of a weight operand: the low (j < 4) and high (j >= 4)
// K-halves, each four bytes of ta / tb times sa / sb, as (1024 + byte) * s + m
// in one packed fma with m = -1024 * s, whose single rounding meets the exact
// product byte * s.  s = sc / 64 over the field's power of two: Q4_K sc <= 63
// (byte * sc <= 945), Q6_K signed sc (|byte * sc| <= 1920), so byte * sc / 64
// is exact in fp16, and the activations' factor 64 makes every MFMA product
// the integer code * scale * code.
__device__ __forceinline__ h8 w_operand(uint32_t ta, uint32_t tb, h2 sa, h2 sb, h2 ma, h2 mb) {
  const u32x4 r{h2bits(__builtin_elementwise_fma(byte_pair(ta, SEL01), sa, ma)),
                h2bits(__builtin_elementwise_fma(byte_pair(ta, SEL23), sa, ma)),
                h2bits(__builtin_elementwise_fma(byte_pair(tb, SEL01), sb, mb)),
                h2bits(__builtin_elementwise_fma(byte_pair(tb, SEL23), sb, mb))};
  return __builtin_bit_cast(h8, r);
}

__device__ __forceinline__ h2 splat2(float v) {
  const _Float16 h = static_cast<_Float16>(v);
  return h2{h, h};
}

// A work group of four waves takes 16*RT rows x 16*NT tokens over all blocks;
// wave w takes lane groups 2w and 2w+1 of every block, whose chains over the
// blocks no other lane group's touch, so the waves meet only at the end.
// MFMA operand layout (v_mfma_f32_16x16x32_f16), activations as A, weights as
// B: lane l feeds A row (token) l%16 and B column (weight row) l%16 with K =
// 8*g .. +7, g = l/16; D lane l register i is token 4g+i, weight row l%16, so
// the row whose scales a lane decodes is the row of its results.  With K index
// k = 4*s + i over sub-blocks s and bytes i, a lane's K range is sub-blocks 2g
// and 2g+1: elements 64g + 4m + i and 64g + 32 + 4m + i for lane group m.
// One wave per lane-group pair (not per row tile) lets a weight operand, whose
// build costs more than its MFMA, serve up to four token tiles in the registers
// that two took (a wave's chains are 8 floats per result where all lane groups
// in one wave need 32), and a short prompt's rows run on four waves at once.
// Against a work group of four row tiles x all lane groups with activations
// staged in LDS (a barrier per block): 1023 tokens of the 2.4B shape, gate/up 198
// -> 131 us, down 171 -> 125, the prompt 23.8 -> 20.5 ms; 44 tokens, down 30 -> 19
// us, the prompt 5.2 -> 4.0 ms.
// What bounds it: past 64 tokens no unit alone (gate/up at 1023 tokens, by
// counters: 17 TB/s of reads from the L2s, 96 % of them hits, vector instructions
// issuing 60 % of the time, matrix cores busy 17 %), though half the reads, by a
// second row tile per wave, took it from 204 us to 132.  For short prompts each wave's own chain of blocks: a launch on
// weights from HBM takes about 5 us and, per block, 0.42 us for Q6_K and 0.31 for
// Q4_K with one token tile, 0.12 more for each further one (2304 rows, down's 23
// blocks at 11, 27, 44 and 59 tokens 14.8, 17.0, 20.1 and 23.0 us, o's 8 blocks
// 7.5, 8.2, 9.3 and 10.6).
// PF: blocks in flight (loads return in order, so weights and activations are
// loaded equally far ahead).
// bid: the work group's index in the GEMM's grid; s_acc: 8*NT*64 entries,
// one row tile's chains [lane group][token tile][lane].
template <int WT, int RT, int NT, int PF>
__device__ __forceinline__ void gemm_block(const GemmArgs& a, unsigned bid, f32x4* s_acc) {
  constexpr int NM = (NT + 3) / 4;  // token tiles whose min chain and epilogue a wave takes: w, w+4, ...
  const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  // Row groups: the first matrix's, then the second's (swiglu: of RT/2 row
  // tiles of both).
  const int rpg = a.swiglu ? 8 * RT : 16 * RT;
  const int n_rg1 = (a.rows + rpg - 1) / rpg;
  const int n_rg = n_rg1 + (a.swiglu ? 0 : (a.rows2 + rpg - 1) / rpg);
  // XCD-aware tiles: work group b runs on XCD b % 8.  Of n_rg = 8q + r row
  // groups, XCD x takes rg = x + 8j (j < q) for every token tile (token
  // tiles outer, so the tile's activations serve its q row groups from one
  // L2), and then an equal share of the r remaining row groups' (row group,
  // token tile) items, so every XCD has the same work; each XCD's L2 keeps
  // about one eighth of the matrix for the whole launch.
  const int xcd = static_cast<int>(bid) & 7, loc = static_cast<int>(bid) >> 3;
  const int n_tt = (a.n_tok + 15) >> 4;
  const int n_tg = (n_tt + NT - 1) / NT;
  const int rq = n_rg >> 3, rr = n_rg & 7;
  const int share = (rr * n_tg + 7) >> 3;
  int rg, tg;
  if (loc < rq * n_tg) {
    rg = xcd + 8 * (loc % rq);
    tg = loc / rq;
  } else {
    const int li = xcd * share + (loc - rq * n_tg);
    if (loc - rq * n_tg >= share || li >= rr * n_tg) return;  // uniform in the work group, before any barrier
    rg = 8 * rq + li / n_tg;
    tg = li % n_tg;
  }
  const bool second = rg >= n_rg1;
  const int rows = second ? a.rows2 : a.rows;
  // row tile rt's first row, and its matrix (swiglu: even tiles gate, odd up)
  auto row0 = [&](int rt) {
    return a.swiglu ? (rg * (RT / 2) + rt / 2) * 16 : ((second ? rg - n_rg1 : rg) * RT + rt) * 16;
  };
  const WView& W0 = second ? a.w2 : a.w;
  const WView& W1 = second || a.swiglu ? a.w2 : a.w;
  const uint32_t rows16 = static_cast<uint32_t>(rows) * 16;

  // Every load of the block loop is a buffer load whose lane offset is fixed
  // here and whose block offset is a scalar.  Rows and token tiles past the
  // end read the last one; their results are not stored.
  struct WRaw {
    // Q4_K: d, dmin and scales; lane groups 2w and 2w+1 of chunk 2g + w/2.
    // Q6_K: scales 4g .. 4g+3, scales 4w .. 4w+3, d; ql of both 32-byte
    // halves and qh of lane groups 2w, 2w+1.
    u32x4 hdr;
    u32x2 q[WT == 0 ? 1 : 3];
  };
  const __amdgpu_buffer_rsrc_t p00 = gemm_rsrc(W0.p0), p01 = gemm_rsrc(W1.p0), p10 = gemm_rsrc(W0.p1),
                               p11 = gemm_rsrc(W1.p1), p20 = gemm_rsrc(W0.p2), p21 = gemm_rsrc(W1.p2),
                               p30 = gemm_rsrc(W0.p3), p31 = gemm_rsrc(W1.p3);
  uint32_t vr[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) vr[rt] = static_cast<uint32_t>(min(row0(rt) + c16, rows - 1));
  const uint32_t w8 = 8u * static_cast<uint32_t>(w & 1);
  auto load_w = [&](WRaw (&r)[RT], int b) {
    const uint32_t ub = static_cast<uint32_t>(b);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const bool o = rt & 1;
      if constexpr (WT == 0) {
        r[rt].hdr = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(o ? p11 : p10, vr[rt] * 16, ub * rows16, 0));
        r[rt].q[0] = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_raw_buffer_load_b64(o ? p01 : p00, vr[rt] * 16 + 2 * g * rows16 + w8,
                                                        (ub * 8 + static_cast<uint32_t>(w >> 1)) * rows16, 0));
      } else {
        const uint32_t h = static_cast<uint32_t>(g >> 1);
        r[rt].hdr.x = __builtin_amdgcn_raw_buffer_load_b32(o ? p21 : p20, vr[rt] * 16 + 4 * g, ub * rows16, 0);
        r[rt].hdr.y = __builtin_amdgcn_raw_buffer_load_b32(o ? p21 : p20, vr[rt] * 16 + 4 * w, ub * rows16, 0);
        r[rt].hdr.z = __builtin_amdgcn_raw_buffer_load_b16(o ? p31 : p30, vr[rt] * 2, ub * static_cast<uint32_t>(rows) * 2, 0);
        const uint32_t ql = vr[rt] * 16 + 4 * h * rows16 + w8;
#pragma unroll
        for (int k = 0; k < 2; ++k)
          r[rt].q[k] = __builtin_bit_cast(
              u32x2, __builtin_amdgcn_raw_buffer_load_b64(o ? p01 : p00, ql, (ub * 8 + static_cast<uint32_t>(2 * k + (w >> 1))) * rows16, 0));
        r[rt].q[2] = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_raw_buffer_load_b64(o ? p11 : p10, vr[rt] * 16 + 2 * h * rows16 + w8,
                                                        (ub * 4 + static_cast<uint32_t>(w >> 1)) * rows16, 0));
      }
    }
  };
  struct XRaw {
    u32x4 x[NT][2];            // the token tiles' operands of lane groups 2w, 2w+1
    f32x4 d[NT];               // d of tokens 4g .. 4g+3
    u32x4 bs[WT == 0 ? NM : NT];  // Q4_K: bsums of tiles w, w+4, ..; Q6_K: bsums 4w .. of every tile
    f32x4 dm[WT == 0 ? NM : 1];   // Q4_K: d of tiles w, w+4, ..
  };
  const __amdgpu_buffer_rsrc_t rxh = gemm_rsrc(a.xh), rxd = gemm_rsrc(a.xd), rxbs = gemm_rsrc(a.xbs);
  const uint32_t vx = static_cast<uint32_t>(lane) * 16, vd = static_cast<uint32_t>(g) * 16;
  const uint32_t vb = static_cast<uint32_t>(c16) * 32 + (WT == 0 ? 16u * (g & 1) : 8u * static_cast<uint32_t>(w));
  uint32_t tb[NT], tm[NM];  // first block of each token tile
#pragma unroll
  for (int n = 0; n < NT; ++n) tb[n] = static_cast<uint32_t>(min(tg * NT + n, n_tt - 1) * a.nb);
#pragma unroll
  for (int k = 0; k < NM; ++k) tm[k] = static_cast<uint32_t>(min(tg * NT + w + 4 * k, n_tt - 1) * a.nb);
  auto load_x = [&](XRaw& r, int n, int b) {
    const uint32_t ub = tb[n] + static_cast<uint32_t>(b);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      r.x[n][j] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(rxh, vx, (ub * 8 + static_cast<uint32_t>(2 * w + j)) * 1024, 0));
    r.d[n] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rxd, vd, ub * 64, 0));
    if constexpr (WT == 1) r.bs[n] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rxbs, vb, ub * 512, 0));
  };
  auto load_min = [&](XRaw& r, int b) {
    if constexpr (WT == 0) {
#pragma unroll
      for (int k = 0; k < NM; ++k) {
        const uint32_t ub = tm[k] + static_cast<uint32_t>(b);
        r.bs[k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rxbs, vb, ub * 512, 0));
        r.dm[k] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rxd, vd, ub * 64, 0));
      }
    }
  };

  f32x4 acc[RT][2][NT], accm[RT][NM];
  const f32x4 zero4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[rt][0][n] = acc[rt][1][n] = zero4;
#pragma unroll
    for (int k = 0; k < NM; ++k) accm[rt][k] = zero4;
  }
  // Q4_K, per lane: the scale bytes of sub-blocks 2g and 2g+1 as ((s0 >> sh4) &
  // m4a) | (s2 & m4b), the min bytes of K-half g (0, 1; none for 2, 3)
  // alike, so that no lane branches
  const uint32_t sh4 = g < 2 ? 0u : 2u, m4a = g < 2 ? 0x3f3f3f3fu : 0x30303030u, m4b = g < 2 ? 0u : 0x0f0f0f0fu;
  const uint32_t shm = g == 1 ? 2u : 0u, mma = g == 0 ? 0x3f3f3f3fu : g == 1 ? 0x30303030u : 0u,
                 mmb = g == 1 ? 0x0f0f0f0fu : 0u;
  const uint32_t sel4a = 0x04000400u | (0x00010001u * 2u * (g & 1)), sel4b = sel4a + 0x00010001u;
  const uint32_t mac = g == 0 ? 0xffffffffu : 0u;  // Q6_K's offset pairs sit in K-half 0
  // Q6_K, per lane (K-half g: code fields at bit 4*(g&1) of each byte, and
  // the high bits' second field 2 above): field masks and the constants of
  // the scale builds (f = 2^-p for a field at bit p; u = sc + 128):
  // sc*f/64 = (1024 + u)*f/64 - 18*f, -16*sc*f = (1024 + u)*(-16*f) + 18432*f
  const bool odd = (g & 1) != 0;
  const float fl = odd ? 0.0625f : 1.0f, fa = odd ? 0.015625f : 0.25f;
  const uint32_t ml = odd ? 0xf0f0f0f0u : 0x0f0f0f0fu, ma0 = odd ? 0x30303030u : 0x03030303u,
                 ma1 = odd ? 0xc0c0c0c0u : 0x0c0c0c0cu;
  const h2 sl1 = splat2(fl * 0.015625f), sl2 = splat2(-18.0f * fl), ol1 = splat2(-16.0f * fl), ol2 = splat2(18432.0f * fl);
  const h2 sa1 = splat2(fa * 0.015625f), sa2 = splat2(-18.0f * fa), oa1 = splat2(-16.0f * fa), oa2 = splat2(18432.0f * fa);
  const uint32_t k0 = static_cast<uint32_t>(w >> 1), k1 = 2 + k0;  // the lane groups' sub-block scales
  const uint32_t selk0 = 0x04000400u | (k0 << 16) | k0, selk1 = 0x04000400u | (k1 << 16) | k1;

  // One block: the weight operands of every row tile are built, then each
  // token tile's MFMAs and chain steps run for all of them.  Loads of block b +
  // PF are issued as the registers they go to are read out.
  auto block = [&](WRaw (&r)[RT], XRaw& x, int b) {
    const int bn = min(b + PF, a.nb - 1);
    h8 Bl[RT][2], Bh[RT][2], Bc[RT][2];
    float dw[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if constexpr (WT == 0) {
        dw[rt] = fp16_to_fp32(static_cast<uint16_t>(r[rt].hdr.x & 0xffffu));
        const uint32_t s0 = r[rt].hdr.y, s1 = r[rt].hdr.z, s2 = r[rt].hdr.w;
        // sc[2g] over 64 (low nibbles) and sc[2g+1] over 1024 (high nibbles,
        // read in place as 16*code), and the offsets -1024*s
        const uint32_t sw = ((s0 >> sh4) & m4a) | (s2 & m4b);
        const h2 ha = byte_pair(sw, sel4a), hb = byte_pair(sw, sel4b);
        const h2 sa = __builtin_elementwise_fma(ha, splat2(0.015625f), splat2(-16.0f));
        const h2 sb = __builtin_elementwise_fma(hb, splat2(0.0009765625f), splat2(-1.0f));
        const h2 ma = sa * splat2(-1024.0f), mb = sb * splat2(-1024.0f);
        const uint32_t q0 = r[rt].q[0].x, q1 = r[rt].q[0].y;
        Bl[rt][0] = w_operand(q0 & 0x0f0f0f0fu, q0 & 0xf0f0f0f0u, sa, sb, ma, mb);
        Bl[rt][1] = w_operand(q1 & 0x0f0f0f0fu, q1 & 0xf0f0f0f0u, sa, sb, ma, mb);
        // the min chain of token tiles w, w+4, ..: k = 8g + j < 16 -> mn[k/2]
        const float dmw = fp16_to_fp32(static_cast<uint16_t>(r[rt].hdr.x >> 16));
        const uint32_t mw = ((s1 >> shm) & mma) | ((s2 >> 4) & mmb);  // 0 for K-halves 2, 3
        const h2 o1024 = splat2(1024.0f);
        const u32x4 mr{h2bits(byte_pair(mw, 0x04000400u) - o1024), h2bits(byte_pair(mw, 0x04010401u) - o1024),
                       h2bits(byte_pair(mw, 0x04020402u) - o1024), h2bits(byte_pair(mw, 0x04030403u) - o1024)};
        const h8 BM = __builtin_bit_cast(h8, mr);
#pragma unroll
        for (int k = 0; k < NM; ++k) {
          const f32x4 DM = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, x.bs[k]), BM, zero4, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) accm[rt][k][i] = __builtin_fmaf(-(x.dm[k][i] * dmw), DM[i], accm[rt][k][i]);
        }
      } else {
        dw[rt] = fp16_to_fp32(static_cast<uint16_t>(r[rt].hdr.z));
        const uint32_t su = r[rt].hdr.x ^ 0x80808080u, sc = r[rt].hdr.y ^ 0x80808080u;
        const h2 ha = byte_pair(su, selk0), hb = byte_pair(su, selk1);
        const h2 sLa = __builtin_elementwise_fma(ha, sl1, sl2), oLa = __builtin_elementwise_fma(ha, ol1, ol2);
        const h2 sLb = __builtin_elementwise_fma(hb, sl1, sl2), oLb = __builtin_elementwise_fma(hb, ol1, ol2);
        const h2 sAb = __builtin_elementwise_fma(hb, sa1, sa2), oAb = __builtin_elementwise_fma(hb, oa1, oa2);
        // (qh's first field is at the bit of the low codes' field: its factor)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const uint32_t la = j ? r[rt].q[0].y : r[rt].q[0].x, lb = j ? r[rt].q[1].y : r[rt].q[1].x;
          const uint32_t hq = j ? r[rt].q[2].y : r[rt].q[2].x;
          Bl[rt][j] = w_operand(la & ml, lb & ml, sLa, sLb, oLa, oLb);
          Bh[rt][j] = w_operand(hq & ma0, hq & ma1, sLa, sAb, oLa, oAb);
          // the offset pair -2*sc of sub-blocks 2m, 2m+1 = (1024 + u)*(-2) +
          // 2304, against the bsums 2m, 2m+1 that K-half 0 holds at dword j
          const h2 hp = byte_pair(sc, 0x04000400u | ((2u * j + 1) << 16) | (2u * j));
          const uint32_t ac = h2bits(__builtin_elementwise_fma(hp, splat2(-2.0f), splat2(2304.0f))) & mac;
          Bc[rt][j] = __builtin_bit_cast(h8, j ? u32x4{0u, ac, 0u, 0u} : u32x4{ac, 0u, 0u, 0u});
        }
      }
    }
    load_w(r, bn);
    load_min(x, bn);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        f32x4 S[2], T[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const h8 A = __builtin_bit_cast(h8, x.x[n][j]);
          S[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, Bl[rt][j], zero4, 0, 0, 0);
          if constexpr (WT == 1) {
            T[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, x.bs[n]), Bc[rt][j], zero4, 0, 0, 0);
            T[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, Bh[rt][j], T[j], 0, 0, 0);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float ds = x.d[n][i] * dw[rt];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const float v = WT == 0 ? S[j][i] : __builtin_fmaf(16.0f, T[j][i], S[j][i]);
            acc[rt][j][n][i] = __builtin_fmaf(ds, v, acc[rt][j][n][i]);
          }
        }
      }
      load_x(x, n, bn);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  WRaw wr[PF][RT];
  XRaw xr[PF];
  // oldest first: a wait for a load waits for every older one
#pragma unroll
  for (int p = 0; p < PF; ++p) {
    load_w(wr[p], min(p, a.nb - 1));
    load_min(xr[p], min(p, a.nb - 1));
#pragma unroll
    for (int n = 0; n < NT; ++n) load_x(xr[p], n, min(p, a.nb - 1));
  }
  // groups of PF blocks with no branch inside (the waits for the loads then
  // count exactly), then the remainder
  int b = 0;
  for (; b + PF <= a.nb; b += PF) {
#pragma unroll
    for (int p = 0; p < PF; ++p) block(wr[p], xr[p], b + p);
  }
#pragma unroll
  for (int p = 0; p < PF - 1; ++p)
    if (b + p < a.nb) block(wr[p], xr[p], b + p);

  // Row tile by row tile, the waves put their lane groups' chains together:
  // wave w finishes token tiles w, w+4, ...
  f32x4 gate[NM];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    if (rt) __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int n = 0; n < NT; ++n) s_acc[((2 * w + j) * NT + n) * 64 + lane] = acc[rt][j][n];
    }
    __syncthreads();
    const int r = row0(rt) + c16;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
      const int n = w + 4 * k;
      if (n >= NT) break;
      f32x4 m[8], v;
#pragma unroll
      for (int j = 0; j < 8; ++j) m[j] = s_acc[(j * NT + n) * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = ((m[0][i] + m[4][i]) + (m[2][i] + m[6][i])) + ((m[1][i] + m[5][i]) + (m[3][i] + m[7][i]));
        if constexpr (WT == 0) v[i] = v[i] + accm[rt][k][i];
      }
      if (a.swiglu) {
        if ((rt & 1) == 0) {
          gate[k] = v;
          continue;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (gate[k][i] / (1.0f + exp_f32(-gate[k][i]))) * v[i];
      }
      const int t4 = 16 * (tg * NT + n) + 4 * g;  // the lane's first token
      if (a.rope) {
        // rows (2i, 2i+1) of a pair are neighbouring lanes; apply_rope's
        // products and sums (src/ops/ops.cpp:502-516)
        const int d = (r % a.rope_hd) >> 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const size_t pos = static_cast<size_t>(a.pos0 + min(t4 + i, a.n_tok - 1));
          const float2 cs = a.rope[pos * (a.rope_hd / 2) + d];
          const float o = dpp_f<DPP_XOR1>(v[i]);
          v[i] = (c16 & 1) ? o * cs.y + v[i] * cs.x : v[i] * cs.x - o * cs.y;
        }
      }
      if (r < rows) {
        float* o = (second ? a.out2 : a.out) + r;
        const size_t ld = second ? a.ld_out2 : a.ld_out;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (t4 + i < a.n_tok) o[(t4 + i) * ld] = a.add ? o[(t4 + i) * ld] + v[i] : v[i];
      }
    }
  }
}

template <int WT, int RT, int NT, int PF>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8))) k_gemm_q8k(const GemmArgs a) {
  __shared__ f32x4 s_acc[8 * NT * 64];
  gemm_block<WT, RT, NT, PF>(a, blockIdx.x, s_acc);
}

// Two GEMMs on the same activations in one launch, the first grid_a work
// groups (a multiple of 8, so both keep their XCDs) a Q4_K one (q and k), the
// rest a Q6_K one (v): v's few rows alone left most CUs idle for 9 us of each
// layer (32 work groups for 44 tokens).
template <int RT, int NT, int PF>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8)))
k_gemm_q4_q6(const GemmArgs a, const GemmArgs b, unsigned grid_a) {
  __shared__ f32x4 s_acc[8 * NT * 64];
  if (blockIdx.x < grid_a)
    gemm_block<0, RT, NT, PF>(a, blockIdx.x, s_acc);
  else
    gemm_block<1, RT, NT, PF>(b, blockIdx.x - grid_a, s_acc);
}

// ------------------------------------------------- attention combine + Q8_K --
// Per token t (one work group, position pos0 + t): the attention output from
// the per-token chunk partials -- k_attn_combine's arithmetic for each value:
// m = max m_c, then over the chunks in order f_c = exp(m_c - m),
// Z = fma(z_c, f_c, Z), O = fma(o_c, f_c, O), value O / Z -- then the O
// projection's ties-even Q8_K quantization of it (k_quant_batch's), with no
// fp32 copy of the output in between.  A lane takes 4 consecutive values of
// one head (head_dim % 4 == 0), which share m and Z.
__global__ void __launch_bounds__(256) k_quant_batch_attn(const float* __restrict__ part_o,
                                                          const float2* __restrict__ part_mz, size_t tok_stride_o,
                                                          size_t tok_stride_mz, int pos0, int dim, int hd,
                                                          int max_chunks, int n_tok, _Float16* __restrict__ xh,
                                                          float* __restrict__ xd, _Float16* __restrict__ xbs) {
  const int t = quant_token(blockIdx.x);
  if (t >= n_tok) return;  // uniform, before any barrier
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nch = (pos0 + t) / ATTN_CHUNK + 1;
  const int nb = dim / QK_K;
  for (int b = wave; b < nb; b += 4) {
    const int i0 = b * QK_K + 4 * lane;
    const int h = i0 / hd, d0 = i0 - h * hd;
    const float2* mz = part_mz + t * tok_stride_mz + static_cast<size_t>(h) * max_chunks;
    const float* o = part_o + t * tok_stride_o + static_cast<size_t>(h) * max_chunks * hd + d0;
    // the chunks' partials in batches of CB whose loads are issued together
    // (indices past the last chunk re-read it: the max is unchanged, and the
    // combine skips them)
    constexpr int CB = 8;
    float m = mz[0].x;
    for (int c0 = 0; c0 < nch; c0 += CB) {
      float mv[CB];
#pragma unroll
      for (int k = 0; k < CB; ++k) mv[k] = mz[min(c0 + k, nch - 1)].x;
#pragma unroll
      for (int k = 0; k < CB; ++k) m = fmaxf(m, mv[k]);
    }
    float Z = 0.0f;
    float O[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int c0 = 0; c0 < nch; c0 += CB) {
      float2 zc[CB];
      f32x4 oc[CB];
#pragma unroll
      for (int k = 0; k < CB; ++k) {
        const int c = min(c0 + k, nch - 1);
        zc[k] = mz[c];
        oc[k] = *reinterpret_cast<const f32x4*>(o + static_cast<size_t>(c) * hd);
      }
#pragma unroll
      for (int k = 0; k < CB; ++k) {
        if (c0 + k < nch) {
          const float f = exp_f32(zc[k].x - m);
          Z = __builtin_fmaf(zc[k].y, f, Z);
          O[0] = __builtin_fmaf(oc[k].x, f, O[0]);
          O[1] = __builtin_fmaf(oc[k].y, f, O[1]);
          O[2] = __builtin_fmaf(oc[k].z, f, O[2]);
          O[3] = __builtin_fmaf(oc[k].w, f, O[3]);
        }
      }
    }
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = O[k] / Z;
    uint32_t packed;
    float dq;
    int gsum;
    quant_block_wave(v, false, packed, dq, gsum);
    store_codes(t, nb, b, lane, packed, dq, gsum, xh, xd, xbs);
  }
}

// -------------------------------------------------------------- launchers --
hipError_t launch_embed_batch(const WView& w, const int* tokens, int n_tok, int dim, float* x, hipStream_t s) {
  hipLaunchKernelGGL(k_embed_batch, dim3((dim + QK_K - 1) / QK_K, n_tok), dim3(QK_K), 0, s, w, tokens, dim, x);
  return hipGetLastError();
}

hipError_t launch_quant_batch(const float* x, int ld_x, const float* gamma, float eps, int dim, int n_valid, int mode,
                              int n_tok, QuantBatch q, hipStream_t s) {
  if (dim % QK_K) return hipErrorInvalidValue;
  // rows of up to 24 blocks load everything up front (k_quant_batch_r)
  const int nb = dim / QK_K;
  if (n_valid < 1 || n_valid > dim || n_valid > ld_x) return hipErrorInvalidValue;
  const bool up_front = ld_x % 4 == 0 && n_valid % 4 == 0;
  auto kern = up_front && nb <= 12 ? k_quant_batch_r<3> : up_front && nb <= 24 ? k_quant_batch_r<6> : k_quant_batch;
  hipLaunchKernelGGL(kern, quant_grid(n_tok), dim3(256), 0, s, x, ld_x, gamma, eps, dim, n_valid, mode, n_tok, q.xh,
                     q.xd, q.xbs);
  return hipGetLastError();
}

hipError_t launch_gemm_q8k(const WView& w, int rows, int nb, int n_tok, const QuantBatch& q, float* out, int ld_out,
                           bool add, int n_cu, hipStream_t s, const WView* w2, int rows2, float* out2, int ld_out2,
                           const GemmRope* rope, bool swiglu, const GemmMore* v) {
  if (w.type != MCPM_TYPE_Q4_K && w.type != MCPM_TYPE_Q6_K) return hipErrorInvalidValue;
  if (rows < 1 || nb < 1 || n_tok < 1) return hipErrorInvalidValue;
  if (rows2 > 0 && (!w2 || w2->type != w.type || (!swiglu && !out2))) return hipErrorInvalidValue;
  if (swiglu && (rows2 != rows || rope || add)) return hipErrorInvalidValue;
  // a rotated pair (rows 2i, 2i+1) stays in one head and one row tile:
  // head_dim even, every matrix's rows a multiple of it
  if (rope && (!rope->table || rope->head_dim <= 0 || rope->head_dim % 2 || rows % rope->head_dim ||
               (rows2 > 0 && rows2 % rope->head_dim)))
    return hipErrorInvalidValue;
  GemmArgs a{w, rows, nb, n_tok, q.xh, q.xd, q.xbs, out, ld_out, add ? 1 : 0, rows2 > 0 ? *w2 : WView{},
             std::max(rows2, 0), out2, ld_out2, rope ? rope->table : nullptr, rope ? rope->head_dim : 0,
             rope ? rope->pos0 : 0, swiglu ? 1 : 0};
  // v: a further matrix of the other type, in the same launch
  const bool pair = v && v->rows > 0;
  if (pair && (w.type != MCPM_TYPE_Q4_K || v->w.type != MCPM_TYPE_Q6_K || swiglu || add)) return hipErrorInvalidValue;
  const GemmArgs av{pair ? v->w : WView{}, pair ? v->rows : 0, nb, n_tok, q.xh, q.xd, q.xbs, pair ? v->out : nullptr,
                    pair ? v->ld_out : 0, 0, WView{}, 0, nullptr, 0, nullptr, 0, 0, 0};
  const bool q4 = w.type == MCPM_TYPE_Q4_K;
  // Token tiles per work group: building a block's weight operands costs about
  // two tiles' chains, so NT token tiles per group cost ceil(tiles / NT) * (2 +
  // NT); the fewest, up to 4 (the registers of two waves per SIMD).  Two row
  // tiles per work group share each activation operand where that still leaves
  // a work group per CU, else one (2304 rows, 76 tokens: 144 work groups of
  // two, 5.53 ms a prompt, 5.20 with one); gate and up always pair.
  const int tiles = (n_tok + 15) / 16;
  int NT = 1;
  for (int n = 2; n <= 4; ++n)
    if ((tiles + n - 1) / n * (2 + n) < (tiles + NT - 1) / NT * (2 + NT)) NT = n;
  const int n_tg = (tiles + NT - 1) / NT;
  auto groups = [&](int rpg) { return (rows + rpg - 1) / rpg + (swiglu ? 0 : (std::max(rows2, 0) + rpg - 1) / rpg); };
  const int RT = swiglu || (groups(32) + (av.rows + 31) / 32) * n_tg >= n_cu ? 2 : 1;
  auto blocks = [&](int n_rg) { return 8u * static_cast<unsigned>((n_rg / 8) * n_tg + ((n_rg % 8) * n_tg + 7) / 8); };
  const unsigned grid_a = blocks(groups(swiglu ? 16 : 16 * RT));
  const dim3 grid(grid_a + (pair ? blocks((av.rows + 16 * RT - 1) / (16 * RT)) : 0u));
  // Blocks in flight: two where a block's work is short (few tokens, weights
  // from HBM: 2304 x 5888 Q6_K, 12 tokens, 18.9 us with one, 12.8 with two,
  // 12.6 with four), one where the other wave of the SIMD fills the wait and
  // the registers are better spent (1023 tokens: 21.4 ms a prompt with two
  // blocks of weights, 20.5 with one).
#define MCPM_GEMM(R, N, P) \
  if (RT == R && NT == N) { \
    if (pair) launch_kernel(k_gemm_q4_q6<R, N, P>, grid, dim3(256), 0, s, a, av, grid_a); \
    else if (q4) launch_kernel(k_gemm_q8k<0, R, N, P>, grid, dim3(256), 0, s, a); \
    else launch_kernel(k_gemm_q8k<1, R, N, P>, grid, dim3(256), 0, s, a); \
  }
  MCPM_GEMM(1, 1, 2) MCPM_GEMM(1, 2, 2) MCPM_GEMM(1, 3, 2) MCPM_GEMM(1, 4, 2)
  MCPM_GEMM(2, 1, 2) MCPM_GEMM(2, 2, 2) MCPM_GEMM(2, 3, 1) MCPM_GEMM(2, 4, 1)
#undef MCPM_GEMM
  return hipGetLastError();
}

hipError_t launch_quant_batch_attn(const AttnPart& part, size_t tok_stride_o, size_t tok_stride_mz, int pos0,
                                  int n_tok, int n_heads, int head_dim, int max_chunks, QuantBatch q, hipStream_t s) {
  const int dim = n_heads * head_dim;
  if (dim % QK_K || head_dim % 4) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_quant_batch_attn, quant_grid(n_tok), dim3(256), 0, s, part.o, part.mz, tok_stride_o, tok_stride_mz,
                     pos0, dim, head_dim, max_chunks, n_tok, q.xh, q.xd, q.xbs);
  return hipGetLastError();
}

}  // namespace mcpm
