// lmhead_kernel.hip - the LM head's logits for the decode head with the
// sampling step fused behind it (gfx950).
//
// The decode head of the reference is a projection of the final-normed
// hidden state onto every vocabulary row, then a topk pass that reads the
// logits back (lib/webgpu-llm/model.js:466-471, gemma-model.js:786-799).
// lmh_logits_kernel streams the head once for every row of the call
// (<= SAS_LMH_MAX_ROWS) and writes f32 logits (1 MB per row at 262,144 ids,
// against 1.3 GB of bf16 head); the sampling kernels then take them as for
// sas_sample.
//
// Eight lanes share one id: lane g of the group sums the hidden indices
// 64 c + 8 g .. + 7 (c ascending) as one f32 fused multiply-add chain, so
// each load of the group is a whole 128-byte line of the weight row; the
// eight partial sums then add in one fixed tree.  That order is the one the
// host oracle follows.  The bf16 weight widens exactly to f32 (bits << 16,
// ggml/kernels.js:31-33), so each product is the reference's f32 product.
//
// Bound by HBM (2 R flops per 2-byte weight): every wave walks the
// vocabulary in groups of 8 ids, wave w of the grid taking groups w,
// w + waves, ..., so that whatever the vocabulary every CU streams until the
// end.  (Blocks of 512 consecutive ids with the sampling pass over them in
// the same block left CUs idle below 131,072 ids, and folding their records
// took a launch of its own.  A whole call before -> now: Q4_0 32,000 x
// 4,096, one row, 91.7 -> 31.2 us; Q6_K 248,320 x 2,560, three rows, 129.2
// -> 117.9 us; bf16 262,144 x 2,560, one row, 217.1 -> 208.8 us, 7.0 TB/s
// in this kernel.)
#include "sas_device.h"
#include "sas_launch.h"

namespace sas {

constexpr int kLmhStep = 64;  // hidden values per load step: 128 bytes of a weight row

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

// ---- GGUF heads: the Q8_1 operand on chip, exact integer block dots ----

// GGUF rows are staged through LDS: 8 items of a row at a time (a stage:
// 8 blocks of Q8_0 / Q4_0, 8 units = 2 super-blocks of Q6_K), loaded as the
// 16-byte aligned chunks that cover them, so the 8 lanes of a row read 128
// contiguous bytes per load and every load is a whole aligned chunk.  A
// chunk that holds one byte of the head lies in the head's pages, so the
// few bytes it holds past either end of the stage are safe to read.
template <int kFmt>
struct QStage {
  static constexpr int bytes = kFmt == SAS_HEAD_Q6_K ? 420 : kFmt == SAS_HEAD_Q8_0 ? 272 : 144;
  static constexpr int chunks = (bytes + 14 + 15) / 16;  // the stage starts 0 .. 14 bytes into its first chunk
  static constexpr int loads = (chunks + 7) / 8;         // per lane
  static constexpr int pitch = 4 * (chunks + 1);         // LDS dwords per row (one chunk of bank skew)
  static constexpr int depth = 4;                        // stages in flight per wave
};

__device__ __forceinline__ float f16_value(uint32_t bits) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
}

// N words that start `sh` bytes (0 or 2) into u[0]: the N + 1 dwords
// read from LDS, shifted.
template <int N>
__device__ __forceinline__ void words_of(const uint32_t (&u)[N + 1], uint32_t sh, uint32_t (&out)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) out[i] = __builtin_amdgcn_alignbyte(u[i + 1], u[i], sh);
}
template <int N>
__device__ __forceinline__ void lds_dwords(const uint32_t *p, uint32_t (&u)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) u[i] = p[i];
}

// The Q8_1 operand of R hidden rows, in LDS, packed per item so that a
// lane reads its item's operand from one base address in whole 16-byte
// loads: kQOpWords dwords per item, rows one after another.
//   Q8_0 / Q4_0, per 32-value block: q (8 words, four int8 each), d8, s8
//     (the f16 d and d * sum(q), as f32), 2 words of padding;
//   Q6_K, per 64-value unit u (super-block u / 4, half h = (u / 2) % 2,
//     16-value half lh = u % 2): for its quarters qt = 0 .. 3 (the Q8_1
//     block 8 (u / 4) + 4 h + qt, its half lh): the 16 q (4 words each,
//     quarter after quarter), then -32 x each quarter's sum of q, then each
//     quarter's d8.
// Each 32-value block (q8.js:27-42): amax,
// d = amax / 127, q = round-half-even(x * (1 / d)), the f16 d and d * sum(q).
template <int kFmt>
constexpr int kQOpWords = kFmt == SAS_HEAD_Q6_K ? 24 : 12;
template <int kFmt>
__host__ __device__ constexpr int q_items(int dim) {
  return kFmt == SAS_HEAD_Q6_K ? dim / 64 : dim / 32;
}

template <int R, int kFmt>
__device__ __forceinline__ void q81_stage(const LmhArgs &L, uint32_t *U) {
  // eight lanes per 32-value block, four values each (nq is a multiple of
  // 64: every wave is whole, so the lanes of a block are together); a thread's
  // loads of a batch are in flight together, their chains overlap
  constexpr int kBatch = 4;
  const int dim = L.dim, nq = dim / 4, rw = q_items<kFmt>(dim) * kQOpWords<kFmt>;
  for (int t0 = threadIdx.x; t0 < R * nq; t0 += kBatch * kThreads) {
    f32x4u v[kBatch];
    int row[kBatch], quad[kBatch];
#pragma unroll
    for (int n = 0; n < kBatch; ++n) {
      const int t = min(t0 + n * kThreads, R * nq - 1);
      row[n] = 0;
#pragma unroll
      for (int r = 1; r < R; ++r) row[n] += t >= r * nq ? 1 : 0;
      quad[n] = t - row[n] * nq;
      v[n] = *reinterpret_cast<const f32x4u *>(L.hidden + (int64_t)row[n] * L.hidden_stride + 4 * quad[n]);
    }
#pragma unroll
    for (int n = 0; n < kBatch; ++n) {
      if (t0 + n * kThreads >= R * nq) break;  // uniform over the wave
      const int b = quad[n] >> 3, e = quad[n] & 7;
      // amax is a maximum of non-negative floats (NaNs left out): their bit
      // patterns order as the values do
      uint32_t am = __float_as_uint(
          fmaxf(fmaxf(fmaxf(0.0f, fabsf(v[n].x)), fabsf(v[n].y)), fmaxf(fabsf(v[n].z), fabsf(v[n].w))));
      am = max(am, dppx<kDppQuad1032>(am));
      am = max(am, dppx<kDppQuad2301>(am));
      am = max(am, dppx<kDppRowHalfMirror>(am));
      const float d = __uint_as_float(am) / 127.0f;
      const float inv = d > 0.0f ? 1.0f / d : 0.0f;
      uint32_t x = 0u, sum = 0u;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float xs = v[n][c] * inv;
        const float rq = xs != xs ? 0.0f : fminf(fmaxf(rintf(xs), -128.0f), 127.0f);
        const int qi = (int)rq;
        sum += (uint32_t)qi;
        x |= ((uint32_t)qi & 0xFFu) << (8 * c);
      }
      sum += dppx<kDppQuad1032>(sum);
      sum += dppx<kDppQuad2301>(sum);
      const int half = (int)sum;  // of the lane's 16 values
      const int all = (int)(sum + dppx<kDppRowHalfMirror>(sum));
      const float d16 = (float)(_Float16)d;
      uint32_t *ur = U + row[n] * rw;
      if constexpr (kFmt == SAS_HEAD_Q6_K) {
        const int sb = b >> 3, hh = (b >> 2) & 1, qt = b & 3;
        uint32_t *o = ur + (sb * 4 + hh * 2 + (e >> 2)) * 24;
        o[4 * qt + (e & 3)] = x;
        if ((e & 3) == 0) {
          o[16 + qt] = (uint32_t)(-32 * half);
          o[20 + qt] = __float_as_uint(d16);
        }
      } else {
        uint32_t *o = ur + b * 12;
        o[e] = x;
        if (e == 0) {
          o[8] = __float_as_uint(d16);
          o[9] = __float_as_uint((float)(_Float16)(d * (float)all));
        }
      }
    }
  }
}

// Where a lane's item lies in its row's staged copy: `c0` its byte offset
// from the stage's first byte, and the LDS dword index of each field for a
// stage that starts at dword 0 (the stage adds its own base).
template <int kFmt>
struct QLane {
  uint32_t c0, row;  // Q8_0 / Q4_0: the block (its f16 d, then its values)
};
template <>
struct QLane<SAS_HEAD_Q6_K> {
  uint32_t c0, la, lb, qh, sc, d;  // Q6_K: the unit's ql spans, qh span, scales, the super-block's d
  uint32_t lh8;                    // 8 lh: the bit offset of the unit's scales in a scale word
};

// Item g of a stage of the lane's row, whose copy starts at LDS dword `row`.
template <int kFmt>
__device__ __forceinline__ QLane<kFmt> q_lane(int g, uint32_t row) {
  QLane<kFmt> ln;
  if constexpr (kFmt == SAS_HEAD_Q6_K) {
    // unit g % 4 (half h, quarter pair lh) of the stage's super-block g / 4
    const uint32_t h = (uint32_t)(g & 3) >> 1, lh = (uint32_t)g & 1u;
    ln.c0 = 210u * (uint32_t)(g >> 2);
    ln.la = row + h * 16u + lh * 4u;        // byte h*64 + lh*16
    ln.lb = ln.la + 8u;                     // byte h*64 + 32 + lh*16
    ln.qh = row + 32u + h * 8u + lh * 4u;   // byte 128 + h*32 + lh*16
    ln.sc = row + 48u + h * 2u;             // byte 192 + h*8: scales h*8 .. h*8 + 7
    ln.d = row + 52u;                       // byte 208
    ln.lh8 = 8u * lh;
  } else {
    ln.c0 = (uint32_t)((kFmt == SAS_HEAD_Q8_0 ? 34 : 18) * g);
    ln.row = row;
  }
  return ln;
}

// A lane's Q8_1 operand for its item, read from LDS where it is used: `u`
// the item's words for row 0, `rw` words between rows.
struct QOp {
  const uint32_t *u;
  int rw;
  // Q8_0 / Q4_0: the block's 32 values, d and the f16 of d * sum
  __device__ __forceinline__ void block(int r, int32_t (&q)[8], float &d, float &sd) const {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 *p = reinterpret_cast<const u32x4 *>(u + r * rw);
    const u32x4 a0 = p[0], a1 = p[1], a2 = p[2];
    q[0] = (int32_t)a0.x;
    q[1] = (int32_t)a0.y;
    q[2] = (int32_t)a0.z;
    q[3] = (int32_t)a0.w;
    q[4] = (int32_t)a1.x;
    q[5] = (int32_t)a1.y;
    q[6] = (int32_t)a1.z;
    q[7] = (int32_t)a1.w;
    d = __uint_as_float(a2.x);
    sd = __uint_as_float(a2.y);
  }
  // Q6_K: quarter qt of the unit, -32 x its sum, its Q8_1 block's d
  __device__ __forceinline__ void quarter(int r, int qt, int32_t (&q4)[4], int32_t &zq, float &dq) const {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const uint32_t *b = u + r * rw;
    const u32x4 a = reinterpret_cast<const u32x4 *>(b)[qt];
    q4[0] = (int32_t)a.x;
    q4[1] = (int32_t)a.y;
    q4[2] = (int32_t)a.z;
    q4[3] = (int32_t)a.w;
    zq = (int32_t)b[16 + qt];
    dq = __uint_as_float(b[20 + qt]);
  }
};

// The dwords of a lane's item of a stage, read from its row's copy in LDS
// one stage ahead of their use (so that the LDS round trip overlaps the
// previous stage's arithmetic).
template <int kFmt>
struct QRaw {
  uint32_t w[kFmt == SAS_HEAD_Q8_0 ? 9 : 5];  // Q8_0 / Q4_0: the values' dwords
  uint32_t d;                                // the dword of the f16 d
  uint32_t x0;                               // the item's first byte in the copy
};
template <>
struct QRaw<SAS_HEAD_Q6_K> {
  uint32_t la[5], lb[5], qh[5], sc[3], d;
  uint32_t x0;
};

template <int kFmt>
__device__ __forceinline__ void q_fetch(const uint32_t *stg, const QLane<kFmt> &ln, uint32_t off, QRaw<kFmt> &x) {
  const uint32_t x0 = off + ln.c0;  // the item's first byte (even)
  x.x0 = x0;
  if constexpr (kFmt == SAS_HEAD_Q8_0 || kFmt == SAS_HEAD_Q4_0) {
    lds_dwords(stg + ln.row + ((x0 + 2u) >> 2), x.w);
    x.d = stg[ln.row + (x0 >> 2)];
  } else {
    // every field of the unit starts a multiple of 4 bytes after x0: one
    // dword base and one shift for all
    const uint32_t bdw = x0 >> 2;
    lds_dwords(stg + ln.la + bdw, x.la);
    lds_dwords(stg + ln.lb + bdw, x.lb);
    lds_dwords(stg + ln.qh + bdw, x.qh);
    lds_dwords(stg + ln.sc + bdw, x.sc);
    x.d = stg[ln.d + bdw];
  }
}

// Adds the lane's item (fetched by q_fetch) to acc[r] for every row, in the
// order of the header.
template <int R, int kFmt>
__device__ __forceinline__ void q_terms(const QRaw<kFmt> &x, const QLane<kFmt> &ln, const QOp &op, float (&acc)[R]) {
  if constexpr (kFmt == SAS_HEAD_Q8_0 || kFmt == SAS_HEAD_Q4_0) {
    constexpr int NW = kFmt == SAS_HEAD_Q8_0 ? 8 : 4;
    uint32_t wv[NW];
    words_of<NW>(x.w, (x.x0 + 2u) & 3u, wv);
    const float dw = f16_value(x.d >> (8u * (x.x0 & 2u)));
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int32_t q[8];
      float d8b, s8b;
      op.block(r, q, d8b, s8b);
      int dot = 0;
      if constexpr (kFmt == SAS_HEAD_Q8_0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) dot = __builtin_amdgcn_sdot4((int)wv[j], q[j], dot, false);
        acc[r] = acc[r] + ((float)dot * dw) * d8b;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          dot = __builtin_amdgcn_sdot4((int)(wv[j] & 0x0F0F0F0Fu), q[j], dot, false);
          dot = __builtin_amdgcn_sdot4((int)((wv[j] >> 4) & 0x0F0F0F0Fu), q[4 + j], dot, false);
        }
        acc[r] = acc[r] + (((float)dot * dw) * d8b - (8.0f * dw) * s8b);
      }
    }
  } else {
    const uint32_t sh = x.x0 & 3u;
    uint32_t la[4], lb[4], qh[4], sc[2];
    words_of<4>(x.la, sh, la);
    words_of<4>(x.lb, sh, lb);
    words_of<4>(x.qh, sh, qh);
    words_of<2>(x.sc, sh, sc);  // scales h*8 .. h*8 + 7
    const float dq = f16_value(x.d >> (8u * sh));
#pragma unroll
    for (int qt = 0; qt < 4; ++qt) {
      // the 16 six-bit values q of quarter qt, one per byte (0 .. 63): the
      // low or high nibbles of its ql span, bits 2 qt, 2 qt + 1 of qh moved
      // to bits 4, 5.  sum (q - 32) q8 = sum q q8 - 32 sum q8, exactly.
      const uint32_t *src = (qt & 1) ? lb : la;
      uint32_t raw[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t nib = qt >= 2 ? src[j] >> 4 : src[j];
        const uint32_t hi = qt == 3 ? qh[j] >> 2 : qh[j] << (4 - 2 * qt);
        raw[j] = (nib & 0x0F0F0F0Fu) | (hi & 0x30303030u);
      }
      // scale byte h*8 + lh + 2 qt: word qt >> 1, byte lh + 2 (qt & 1)
      const uint32_t sw = sc[qt >> 1];
      const float scv = (float)(int)(int8_t)(uint8_t)(sw >> (ln.lh8 + 16u * (uint32_t)(qt & 1)));
      const float ds = dq * scv;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        int32_t q4[4], zq;
        float d8q;
        op.quarter(r, qt, q4, zq, d8q);
        int dot = __builtin_amdgcn_sdot4((int)raw[0], q4[0], zq, false);
        dot = __builtin_amdgcn_sdot4((int)raw[1], q4[1], dot, false);
        dot = __builtin_amdgcn_sdot4((int)raw[2], q4[2], dot, false);
        dot = __builtin_amdgcn_sdot4((int)raw[3], q4[3], dot, false);
        acc[r] = acc[r] + (ds * d8q) * (float)dot;
      }
    }
  }
}

template <int R, int kFmt>
__global__ __launch_bounds__(kThreads, 2) void lmh_logits_kernel(const LmhArgs L) {
  // bf16: [R][dim] hidden states; GGUF: their Q8_1 operand
  extern __shared__ __attribute__((aligned(16))) float xs[];
  // GGUF: each wave's staged rows (8 rows of one stage)
  __shared__ __attribute__((aligned(16))) uint32_t stg[kFmt == SAS_HEAD_BF16 ? 4 : kWaves * 8 * QStage<kFmt>::pitch];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dim = L.dim;
  const int vocab = L.vocab;
  // ---- the wave's ids: groups of 8 consecutive ones, group gw + nw m at
  // round m; lanes 8 i .. 8 i + 7 take the group's id i.  Lane g of them
  // takes hidden indices 64 c + 8 g .. + 7 (c = 0, 1, ...; GGUF heads:
  // blocks or units g, g + 8, ... of the row).  A wave past the last group
  // computes the last id again and stores nothing. ----
  const int g = lane & 7;
  const int gw = (int)blockIdx.x * kWaves + wave, nw = (int)gridDim.x * kWaves;
  const int groups = (vocab + 7) >> 3;
  const int rounds = max((groups - gw + nw - 1) / nw, 1);
  const int idl = 8 * gw + (lane >> 3);  // this lane's id at round 0
  const int ids = 8 * nw;                // and the ids between rounds
  // the eight partial sums of a group's id, in one fixed tree: lane 0 of
  // the group holds ((p0 + p1) + (p2 + p3)) + ((p4 + p5) + (p6 + p7))
  auto id_done = [&](float (&a)[R], int id) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float v = a[r];
      v = v + __uint_as_float(dppx<kDppQuad1032>(__float_as_uint(v)));
      v = v + __uint_as_float(dppx<kDppQuad2301>(__float_as_uint(v)));
      v = v + __uint_as_float(dppx<kDppRowHalfMirror>(__float_as_uint(v)));
      if (g == 0 && id < vocab) L.logits[(int64_t)r * L.logits_stride + id] = v;
      a[r] = 0.0f;
    }
  };
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.0f;
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  if constexpr (kFmt == SAS_HEAD_BF16) {
    constexpr int kQ = 4;               // steps (128 bytes of a row) per batch of loads
    const int nb = dim / (kLmhStep * kQ);  // batches per id (dim is a multiple of 256)
    const uint16_t *W = static_cast<const uint16_t *>(L.weight);
    // batches in the flattened order (round, batch): two in flight ahead of
    // the one computed (past the last: the last again)
    u32x4 nxt[kQ], nx2[kQ];
    int ml = 0, cl = 0;
    auto load_next = [&](u32x4 (&dst)[kQ]) __attribute__((always_inline)) {
      const int id = min(idl + ids * ml, vocab - 1);  // loads stay inside the head
      const uint16_t *w = W + (int64_t)id * L.weight_stride + 8 * g + cl * (kQ * kLmhStep);
#pragma unroll
      for (int q = 0; q < kQ; ++q) dst[q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(w + q * kLmhStep));
      if (++cl == nb) {
        if (ml + 1 < rounds) {
          cl = 0;
          ++ml;
        } else {
          cl = nb - 1;
        }
      }
    };
    load_next(nxt);
    load_next(nx2);
    // while the first batches are in flight: the rows' hidden states into LDS
    for (int r = 0; r < R; ++r) {
      const float *h = L.hidden + (int64_t)r * L.hidden_stride;
      for (int i = tid; i < dim; i += kThreads) xs[r * dim + i] = h[i];
    }
    __syncthreads();  // the hidden states are in LDS
    for (int m = 0; m < rounds; ++m) {
      for (int cb = 0; cb < nb; ++cb) {
        u32x4 cur[kQ];
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
          cur[q] = nxt[q];
          nxt[q] = nx2[q];
        }
        load_next(nx2);
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
          const int k = (cb * kQ + q) * kLmhStep + 8 * g;  // hidden indices k .. k + 7
          const uint32_t w4[4] = {cur[q].x, cur[q].y, cur[q].z, cur[q].w};
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const float4 *xp = reinterpret_cast<const float4 *>(xs + r * dim + k);
            const float4 x0 = xp[0], x1 = xp[1];
            const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int h = 0; h < 4; ++h) {
              acc[r] = __builtin_fmaf(bf16_lo(w4[h]), xv[2 * h], acc[r]);
              acc[r] = __builtin_fmaf(bf16_hi(w4[h]), xv[2 * h + 1], acc[r]);
            }
          }
        }
      }
      id_done(acc, idl + ids * m);
    }
  } else {
    using St = QStage<kFmt>;
    constexpr int J = St::loads, D = St::depth;
    const uint8_t *W = static_cast<const uint8_t *>(L.weight);
    // items per id: blocks (Q8_0, Q4_0) or 64-value units (Q6_K); lane g
    // takes g, g + 8, ...: item g of each stage of its row
    const int items = q_items<kFmt>(dim);
    const int rowbytes = kFmt == SAS_HEAD_Q6_K ? 210 * (dim / 256) : (kFmt == SAS_HEAD_Q8_0 ? 34 : 18) * (dim / 32);
    const int per = (items + 7) / 8;  // stages per id
    // Stage (m, c) of the wave: items 8 c .. 8 c + 7 of round m's ids (this
    // lane: its group's id), m outer, c inner: a row's stages follow one
    // another, so the line two stages share comes from L2 the second time.
    // The loads are plain (cached) loads for that.
    const uint32_t rbi = (uint32_t)((wave * 8 + (lane >> 3)) * St::pitch);  // the lane's row copy in stg
    const QLane<kFmt> ln = q_lane<kFmt>(g, rbi);
    struct Ring {
      u32x4 v[J];
      uint32_t off;  // the stage's first byte in its first chunk; chunks in use << 8
    };
    Ring ring[D];
    // byte offsets into the head are 32-bit (the host checks that it spans
    // less than 4 GiB); the head is 16-byte aligned
    const uint32_t wstride = (uint32_t)L.weight_stride;
    int cl = 0, ml = 0;  // the next stage to load
    // Loads the next stage into a slot (past the last stage: the last one again).
    auto stage_load = [&](Ring &s) __attribute__((always_inline)) {
      const uint32_t id = (uint32_t)min(idl + ids * ml, vocab - 1);  // loads stay inside the head
      const uint32_t o = id * wstride + (uint32_t)(St::bytes * cl);  // the stage's first byte
      const uint32_t off = o & 15u;
      const uint32_t nch = (off + (uint32_t)min(St::bytes, rowbytes - St::bytes * cl) + 15u) >> 4;
      const uint32_t o16 = o - off;
      // chunks g, g + 8, ... (past the last: the last again, so that every
      // lane loads and no branch splits the loads in flight)
#pragma unroll
      for (int j = 0; j < J; ++j)
        s.v[j] = *reinterpret_cast<const u32x4 *>(W + (o16 + 16u * min((uint32_t)(g + 8 * j), nch - 1u)));
      s.off = off | (nch << 8);
      if (++cl == per) {
        if (ml + 1 < rounds) {
          cl = 0;
          ++ml;
        } else {
          cl = per - 1;
        }
      }
    };
    // the chunks of the stage in slot rs into the row's copy (the wave's LDS
    // operations run in order, so the reads that follow see them and the
    // previous stage's reads came first), then the slot loads the stage D
    // ahead; returns the stage's offset
    auto stage_take = [&](Ring &rs) __attribute__((always_inline)) {
      const uint32_t off = rs.off & 0xFFu, nch = rs.off >> 8;
      __asm__ volatile("" ::: "memory");
#pragma unroll
      for (int j = 0; j < J; ++j)
        *reinterpret_cast<u32x4 *>(stg + rbi + 4u * min((uint32_t)(g + 8 * j), nch - 1u)) = rs.v[j];
      __asm__ volatile("" ::: "memory");
      stage_load(rs);
      return off;
    };
#pragma unroll
    for (int d = 0; d < D; ++d) stage_load(ring[d]);
    uint32_t *U = reinterpret_cast<uint32_t *>(xs);
    const int rw = items * kQOpWords<kFmt>;
    q81_stage<R, kFmt>(L, U);
    __syncthreads();  // the Q8_1 operand is in LDS
    int m = 0, c = 0;  // the stage computed
    // the fields of stage t + 1 are read while stage t is computed (after
    // the last stage: the last stage's copy again, unused)
    QRaw<kFmt> cur;
    q_fetch<kFmt>(stg, ln, stage_take(ring[0]), cur);
    while (m < rounds) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        QRaw<kFmt> nxt;
        q_fetch<kFmt>(stg, ln, stage_take(ring[(d + 1) % D]), nxt);
        const int it = 8 * c + g;
        // past the wave's last stage (the ring's length does not divide the
        // stages) nothing is added: no lane holds an item
        if (m < rounds && it < items) q_terms<R, kFmt>(cur, ln, QOp{U + it * kQOpWords<kFmt>, rw}, acc);
        cur = nxt;
        if (++c == per) {
          if (m < rounds) id_done(acc, idl + ids * m);
          c = 0;
          ++m;
        }
      }
    }
  }
}

int lmh_blocks(int vocab, int cus) {
  // two blocks per CU, each wave at least one group of 8 ids (three and
  // four per CU measured within 5 % either way: bf16 262,144 x 2,560 214 /
  // 215 / 220 us, Q6_K 248,320 x 2,560 at three rows 120 / 125 / 124 us)
  const int all = (vocab + 8 * kWaves - 1) / (8 * kWaves);
  return all < 2 * cus ? all : 2 * cus;
}

template <int R, int kFmt>
static hipError_t launch_rows(const LmhArgs &a, hipStream_t stream) {
  // bf16: the f32 hidden rows; GGUF: the packed Q8_1 operand of every row
  const size_t lds = kFmt == SAS_HEAD_BF16 ? (size_t)R * a.dim * sizeof(float)
                                           : (size_t)R * q_items<kFmt>(a.dim) * kQOpWords<kFmt> * sizeof(uint32_t);
  hipLaunchKernelGGL((lmh_logits_kernel<R, kFmt>), dim3((unsigned)a.blocks), dim3(kThreads), lds, stream, a);
  return hipGetLastError();
}

template <int kFmt>
static hipError_t launch_format(const LmhArgs &a, hipStream_t stream) {
  switch (a.rows) {
    case 1: return launch_rows<1, kFmt>(a, stream);
    case 2: return launch_rows<2, kFmt>(a, stream);
    case 3: return launch_rows<3, kFmt>(a, stream);
    default: return launch_rows<4, kFmt>(a, stream);
  }
}

hipError_t launch_lm_head(const LmhArgs &a, hipStream_t stream) {
  switch (a.format) {
    case SAS_HEAD_Q8_0: return launch_format<SAS_HEAD_Q8_0>(a, stream);
    case SAS_HEAD_Q4_0: return launch_format<SAS_HEAD_Q4_0>(a, stream);
    case SAS_HEAD_Q6_K: return launch_format<SAS_HEAD_Q6_K>(a, stream);
    default: return launch_format<SAS_HEAD_BF16>(a, stream);
  }
}

}  // namespace sas
