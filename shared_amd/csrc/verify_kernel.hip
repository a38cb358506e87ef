// verify_kernel.hip - speculative verification by rejection sampling
// (Leviathan et al. 2023, "Fast Inference from Transformers via Speculative
// Decoding"; Chen et al. 2023, "Accelerating Large Language Model Decoding
// with Speculative Sampling").
//
// The reference verifies drafts by an exact-match cascade
// (lib/webgpu-llm/kernels.js:328-339, acceptSpec); this path implements the
// distribution-preserving rule the sampling API needs at temperature > 0:
//
//   p_j = softmax(target row j / T), q_j = softmax(draft row j / T), both over
//   allowed, non-NaN ids.  Position j accepts draft d_j iff
//   d_j < vocab and p_j(d_j) > 0 and U1 * q_j(d_j) <= p_j(d_j).  The first
//   rejected position a draws from max(0, p_a - q_a) (from p_a when that is
//   all zero) with U2; when every draft is accepted the bonus position L
//   draws from p_L with its U2.  A draw returns the smallest id whose
//   running weight (ascending ids) exceeds U2 * total.
//
// Three launches, each reading what the previous one wrote:
//   1. verify_stats_kernel, one block per (position, 4096-id chunk): reads
//      the target chunk, the draft chunk and the mask words once, and writes
//      the chunk's max and sum of exp((x - max) / T) for both rows.  This is
//      the pass that streams the whole input.
//   2. verify_decide_kernel, one block per (sequence, chunk): combines the
//      chunk statistics of the sequence's positions (every block the same
//      way, in the same order, so they agree bit for bit), decides the
//      accepted prefix, and for the one position that draws, writes the
//      residual mass and target mass of each run of 1024 of the chunk's ids
//      (one wave's).  Only that position's rows are read again.
//   3. verify_draw_kernel, one block per sequence: finds the run in which
//      U2 * total falls, scans its ids in ascending order, and writes the
//      tokens.
//
// The weights that are summed (softmax normalizers, residual and target
// masses, the draw's running sums) are exp_sum of (x - max) * (1 / T) and
// products with reciprocals of the normalizers: within a few ulp of the
// host oracle's fdlibm exp and divisions, a difference of the same order as
// that of the summation order, which differs from a sequential loop anyway.
// The acceptance test p(d) >= U1 q(d) uses fdlibm exp and divisions.
#include <hip/hip_runtime.h>

#include <cmath>

#include "sas_device.h"
#include "sas_launch.h"
#include "shared_amd_sampler.h"

namespace sas {
namespace {

constexpr int kPerThread = kVChunk / kThreads;  // 16 ids per thread
typedef double f64x2 __attribute__((ext_vector_type(2)));
static_assert(kPerThread == 16, "a thread owns four float4 of a chunk");

__device__ __forceinline__ double dneg_inf() { return -__longlong_as_double(0x7ff0000000000000ll); }

// 2^(j / 64), j = 0 .. 63: the nearest double and the nearest double to what
// it leaves (computed with 80 decimal digits).
constexpr int kExpTab = 64;
__device__ const f64x2 kExp2Tab[kExpTab] = {
    {0x1.p+0, 0.0}, {0x1.02c9a3e778061p+0, -0x1.19083535b085dp-56},
    {0x1.059b0d3158574p+0, 0x1.d73e2a475b465p-55}, {0x1.0874518759bc8p+0, 0x1.186be4bb284ffp-57},
    {0x1.0b5586cf9890fp+0, 0x1.8a62e4adc610bp-54}, {0x1.0e3ec32d3d1a2p+0, 0x1.03a1727c57b53p-59},
    {0x1.11301d0125b51p+0, -0x1.6c51039449b3ap-54}, {0x1.1429aaea92de0p+0, -0x1.32fbf9af1369ep-54},
    {0x1.172b83c7d517bp+0, -0x1.19041b9d78a76p-55}, {0x1.1a35beb6fcb75p+0, 0x1.e5b4c7b4968e4p-55},
    {0x1.1d4873168b9aap+0, 0x1.e016e00a2643cp-54}, {0x1.2063b88628cd6p+0, 0x1.dc775814a8495p-55},
    {0x1.2387a6e756238p+0, 0x1.9b07eb6c70573p-54}, {0x1.26b4565e27cddp+0, 0x1.2bd339940e9d9p-55},
    {0x1.29e9df51fdee1p+0, 0x1.612e8afad1255p-55}, {0x1.2d285a6e4030bp+0, 0x1.0024754db41d5p-54},
    {0x1.306fe0a31b715p+0, 0x1.6f46ad23182e4p-55}, {0x1.33c08b26416ffp+0, 0x1.32721843659a6p-54},
    {0x1.371a7373aa9cbp+0, -0x1.63aeabf42eae2p-54}, {0x1.3a7db34e59ff7p+0, -0x1.5e436d661f5e3p-56},
    {0x1.3dea64c123422p+0, 0x1.ada0911f09ebcp-55}, {0x1.4160a21f72e2ap+0, -0x1.ef3691c309278p-58},
    {0x1.44e086061892dp+0, 0x1.89b7a04ef80d0p-59}, {0x1.486a2b5c13cd0p+0, 0x1.3c1a3b69062f0p-56},
    {0x1.4bfdad5362a27p+0, 0x1.d4397afec42e2p-56}, {0x1.4f9b2769d2ca7p+0, -0x1.4b309d25957e3p-54},
    {0x1.5342b569d4f82p+0, -0x1.07abe1db13cadp-55}, {0x1.56f4736b527dap+0, 0x1.9bb2c011d93adp-54},
    {0x1.5ab07dd485429p+0, 0x1.6324c054647adp-54}, {0x1.5e76f15ad2148p+0, 0x1.ba6f93080e65ep-54},
    {0x1.6247eb03a5585p+0, -0x1.383c17e40b497p-54}, {0x1.6623882552225p+0, -0x1.bb60987591c34p-54},
    {0x1.6a09e667f3bcdp+0, -0x1.bdd3413b26456p-54}, {0x1.6dfb23c651a2fp+0, -0x1.bbe3a683c88abp-57},
    {0x1.71f75e8ec5f74p+0, -0x1.16e4786887a99p-55}, {0x1.75feb564267c9p+0, -0x1.0245957316dd3p-54},
    {0x1.7a11473eb0187p+0, -0x1.41577ee04992fp-55}, {0x1.7e2f336cf4e62p+0, 0x1.05d02ba15797ep-56},
    {0x1.82589994cce13p+0, -0x1.d4c1dd41532d8p-54}, {0x1.868d99b4492edp+0, -0x1.fc6f89bd4f6bap-54},
    {0x1.8ace5422aa0dbp+0, 0x1.6e9f156864b27p-54}, {0x1.8f1ae99157736p+0, 0x1.5cc13a2e3976cp-55},
    {0x1.93737b0cdc5e5p+0, -0x1.75fc781b57ebcp-57}, {0x1.97d829fde4e50p+0, -0x1.d185b7c1b85d1p-54},
    {0x1.9c49182a3f090p+0, 0x1.c7c46b071f2bep-56}, {0x1.a0c667b5de565p+0, -0x1.359495d1cd533p-54},
    {0x1.a5503b23e255dp+0, -0x1.d2f6edb8d41e1p-54}, {0x1.a9e6b5579fdbfp+0, 0x1.0fac90ef7fd31p-54},
    {0x1.ae89f995ad3adp+0, 0x1.7a1cd345dcc81p-54}, {0x1.b33a2b84f15fbp+0, -0x1.2805e3084d708p-57},
    {0x1.b7f76f2fb5e47p+0, -0x1.5584f7e54ac3bp-56}, {0x1.bcc1e904bc1d2p+0, 0x1.23dd07a2d9e84p-55},
    {0x1.c199bdd85529cp+0, 0x1.11065895048ddp-55}, {0x1.c67f12e57d14bp+0, 0x1.2884dff483cadp-54},
    {0x1.cb720dcef9069p+0, 0x1.503cbd1e949dbp-56}, {0x1.d072d4a07897cp+0, -0x1.cbc3743797a9cp-54},
    {0x1.d5818dcfba487p+0, 0x1.2ed02d75b3707p-55}, {0x1.da9e603db3285p+0, 0x1.c2300696db532p-54},
    {0x1.dfc97337b9b5fp+0, -0x1.1a5cd4f184b5cp-54}, {0x1.e502ee78b3ff6p+0, 0x1.39e8980a9cc8fp-55},
    {0x1.ea4afa2a490dap+0, -0x1.e9c23179c2893p-54}, {0x1.efa1bee615a27p+0, 0x1.dc7f486a4b6b0p-54},
    {0x1.f50765b6e4540p+0, 0x1.9d3e12dd8a18bp-54}, {0x1.fa7c1819e90d8p+0, 0x1.74853f3a5931ep-55},
};

// The table in LDS.  Every wave writes all of it (its lanes one entry each,
// the same values), so no barrier is needed before a wave reads it.
struct ExpTab {
  f64x2 e[kExpTab];
  __device__ __forceinline__ void fill(const f64x2 &mine) {
    e[threadIdx.x & (kExpTab - 1)] = mine;
    wave_lds_sync();
  }
};
__device__ __forceinline__ f64x2 exp_tab_entry() { return kExp2Tab[threadIdx.x & (kExpTab - 1)]; }

// e^x for sums of many weights, x <= 0, where the order of the additions
// already differs from a sequential loop (the table-driven method of P. T. P.
// Tang, ACM TOMS 15, 1989): within 0.82 ulp of the exact value (rms 0.296
// ulp, over 8 million x in [-700, 0] against 113-bit arithmetic;
// a degree-13 series without a table: 0.86 and 0.302), with no division.
// x = k ln2 / 64 + r, |r| <= ln2 / 128 (k by adding 1.5 * 2^52, ln2 / 64
// split in two parts, the high one with 21 zero bits), e^r - 1 by its Taylor
// series to degree 5 (truncation below 3.5e-17), times 2^((k mod 64) / 64)
// from the table, scaled by ldexp (subnormal results included).  x = -inf
// and NaN give 0; x > 0 is not used (but harmless).  The statistics pass
// without a mask is bound by these double operations: 15 here, 22 in the
// degree-13 series (32 x 5 positions of 151,936 ids: 106 -> 80 us a call), 17
// with 16 entries, whose reads never conflict (83 us).
__device__ __forceinline__ double exp_sum(double x, const ExpTab &tab) {
  const double magic = 6755399441055744.0;
  const double xc = fmax(x, -1100.0);
  const double kf = fma(xc, 0x1.71547652b82fep+6, magic);
  const int k = (int)(uint32_t)(uint64_t)__double_as_longlong(kf);
  const f64x2 T = tab.e[k & (kExpTab - 1)];
  const double kd = kf - magic;
  const double r = fma(-kd, 0x1.a39ef35793c76p-39, fma(-kd, 0x1.62e42fee00000p-7, xc));
  const double q = fma(fma(fma(r, 1.0 / 120.0, 1.0 / 24.0), r, 1.0 / 6.0), r, 0.5);
  const double p = fma(r * r, q, r);
  return __builtin_amdgcn_ldexp(T.x + fma(T.x, p, T.y), k >> 6);
}

// Chunk layout of passes 1 and 2: wave w owns the kWaveIds consecutive ids
// from base + w * kWaveIds on, lane l of it ids (64 f + l) * 4 + k of those
// (f, k in 0..3), loaded as four coalesced float4.
constexpr int kWaveIds = kVChunk / kWaves;
static_assert(kWaveIds == 64 * kPerThread, "four float4 per lane");
__device__ __forceinline__ int lane_id0(int f) {
  return (int)(threadIdx.x >> 6) * kWaveIds + (64 * f + (int)(threadIdx.x & 63)) * 4;
}
// (Each needs 4-byte alignment only and is loaded from min(id, vocab - 4) on,
// inside the row; the float4 that straddles the row's end is shifted into
// place by settle_chunk.  Ids past the row hold no allowed bit.)
__device__ __forceinline__ void load_chunk(const float *row, int base, int vocab, float x[kPerThread]) {
  if (vocab < 4) {
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) x[i] = i < 4 ? row[min(i, vocab - 1)] : 0.0f;
    return;
  }
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const uint32_t at = (uint32_t)min(base + lane_id0(f), vocab - 4);
    const f32x4u v = __builtin_nontemporal_load(reinterpret_cast<const f32x4u *>(row + at));
    x[f * 4 + 0] = v.x;
    x[f * 4 + 1] = v.y;
    x[f * 4 + 2] = v.z;
    x[f * 4 + 3] = v.w;
  }
}
__device__ __forceinline__ void settle_chunk(int base, int vocab, float x[kPerThread]) {
  if ((vocab & 3) == 0 || vocab < 4 || base + kVChunk < vocab) return;  // uniform over the block
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const int sh = base + lane_id0(f) - (vocab - 4);  // 1 .. 3: straddles the end
    const float y = x[f * 4 + 1], z = x[f * 4 + 2], w = x[f * 4 + 3];
    x[f * 4 + 0] = sh == 1 ? y : sh == 2 ? z : sh == 3 ? w : x[f * 4 + 0];
    x[f * 4 + 1] = sh == 1 ? z : sh == 2 ? w : y;
    x[f * 4 + 2] = sh == 1 ? w : z;
  }
}

// The mask words of the lane's four float4, loaded unconditionally (clamped
// into the row), so that they are in flight together.
template <bool kMask>
__device__ __forceinline__ void load_words(const uint32_t *mrow, int base, int vocab, uint32_t (&mw)[4]) {
  const int last_word = ((vocab + 31) >> 5) - 1;
#pragma unroll
  for (int f = 0; f < 4; ++f) mw[f] = kMask ? mrow[(uint32_t)min((base + lane_id0(f)) >> 5, last_word)] : ~0u;
}

// Bit f*4+k set: id base + lane_id0(f) + k is below vocab and its mask bit
// is set.
__device__ __forceinline__ uint32_t allow_bits(const uint32_t (&mw)[4], int base, int vocab) {
  uint32_t bits = 0;
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const int id0 = base + lane_id0(f);
    // ids of the four below vocab: 0 .. 4 (no branch, so the loads stay
    // ahead of every use)
    const int left = min(max(vocab - id0, 0), 4);
    bits |= ((mw[f] >> (uint32_t)(id0 & 31)) & ((1u << left) - 1u)) << (f * 4);
  }
  return bits;
}

// Places n items per lane in one list for the wave: `pre` the lane's first
// slot (the items of the lanes below it), `tot` the wave's total.  n < 32.
__device__ __forceinline__ void wave_place(uint32_t n, uint32_t &pre, uint32_t &tot) {
  pre = 0u;
  tot = 0u;
#pragma unroll
  for (int bit = 0; bit < 5; ++bit) {
    const uint64_t bb = __ballot((n >> bit) & 1u);
    pre += lanes_below(bb) << bit;
    tot += (uint32_t)__popcll(bb) << bit;
  }
}

// A wave's allowed values of one side, packed, when they are few.
constexpr int kCompact = 256;
// pk_n words: the wave's allowed ids' values were packed for both rows
// (a draft value may be NaN), or for the target row only (a position
// without a draft); the count in the low bits.  0: not packed (more than
// kCompact allowed, or a target value among them is NaN).
constexpr uint32_t kPkJoint = 1u << 30;
constexpr uint32_t kPkTarget = 1u << 29;
constexpr uint32_t kPkCount = 0xFFFFu;

struct StatsLds {
  double m[2][kWaves];  // each wave's maximum and sum of the target row, then of the draft row
  double z[2][kWaves];
  float cv[kWaves][2][kCompact];
  ExpTab tab;
};

__device__ __forceinline__ uint32_t nan_free(const float x[kPerThread], uint32_t ok) {
#pragma unroll
  for (int i = 0; i < kPerThread; ++i)
    if (x[i] != x[i]) ok &= ~(1u << i);
  return ok;
}

// Bound by the loads under a sparse mask (178 MB at 32 x 5 positions of
// 151,936 ids, 5 %: 32.4 us, the loads alone 28.5), by the double
// exponentials without one (there 52 us).  Five waves per SIMD, no spills: a
// wave computes while others load (six: 8 registers spilled, 54 us; seven: 61
// us, and 36 with the mask; resident blocks that looped over their items with
// the next one's loads in flight, four waves: 74 and 45 us).
template <bool kMask>
__global__ __launch_bounds__(kThreads, 5) void verify_stats_kernel(VerifyArgs a) {
  __shared__ StatsLds l;
  const int c = blockIdx.x, pos = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int P1 = a.L + 1;
  const int s = pos / P1, j = pos - s * P1;
  const int base = c * kVChunk;
  const bool has_draft = j < a.L;
  const f64x2 te = exp_tab_entry();
  float xt[kPerThread], xq[kPerThread];
  load_chunk(a.target + (int64_t)pos * a.stride, base, a.vocab, xt);
  if (has_draft) load_chunk(a.draft + ((int64_t)s * a.L + j) * a.stride, base, a.vocab, xq);
  uint32_t mw[4];
  load_words<kMask>(kMask ? a.mask + (int64_t)pos * a.mask_stride : nullptr, base, a.vocab, mw);
  if (has_draft && tid == 0) {
    // the block whose chunk holds the position's draft token records the
    // token's two logits for the acceptance test (NaN when masked)
    const uint32_t d = a.draft_ids[(int64_t)s * a.L + j];
    if (d < (uint32_t)a.vocab && (int)(d / kVChunk) == c) {
      const bool allowed = !kMask || ((a.mask[(int64_t)pos * a.mask_stride + (d >> 5)] >> (d & 31)) & 1u);
      a.dtok[2 * pos] = allowed ? a.target[(int64_t)pos * a.stride + d] : __builtin_nanf("");
      a.dtok[2 * pos + 1] = allowed ? a.draft[((int64_t)s * a.L + j) * a.stride + d] : __builtin_nanf("");
    }
  }
  l.tab.fill(te);
  const uint32_t ok = allow_bits(mw, base, a.vocab);
  // The wave's allowed ids, when at most kCompact of its 1,024 (a sparse
  // mask): both rows' values packed into the wave's LDS slots in id order,
  // NaNs included, so that the NaN tests, the maxima and the exponentials
  // run over those values only.  Otherwise every value is tested in the
  // registers.
  uint32_t pre, tot;
  wave_place((uint32_t)__popc(ok), pre, tot);
  const bool packed = tot <= (uint32_t)kCompact;  // uniform over the wave
  float *cvt = l.cv[wave][0], *cvq = l.cv[wave][1];
  // each row's maximum over the wave (allowed, not NaN) and its sum of
  // exp((x - max) / T)
  double Mt, Mq = dneg_inf(), zt = 0.0, zq = 0.0;
  uint32_t pk = 0u;  // how the wave's values were packed for the decide pass
  settle_chunk(base, a.vocab, xt);
  if (packed) {
    if (has_draft) settle_chunk(base, a.vocab, xq);
    uint32_t jj = pre;
#pragma unroll
    for (int i = 0; i < kPerThread; ++i)
      if ((ok >> i) & 1u) {
        cvt[jj] = xt[i];
        if (has_draft) cvq[jj] = xq[i];
        ++jj;
      }
    wave_lds_sync();
    bool tnan = false;  // a packed target value is NaN
    float mt = -__builtin_inff(), mq = -__builtin_inff();
    // a NaN compares false: it never becomes a maximum
    for (uint32_t e = (uint32_t)lane; e < tot; e += 64u) {
      const float t = cvt[e];
      tnan |= t != t;
      mt = t > mt ? t : mt;
      if (has_draft) {
        const float q = cvq[e];
        mq = q > mq ? q : mq;
      }
    }
    Mt = (double)wave_max(mt);
    Mq = (double)wave_max(mq);
    for (uint32_t e = (uint32_t)lane; e < tot; e += 64u) {
      const float t = cvt[e];
      if (t == t) zt += exp_sum(((double)t - Mt) * a.inv_t, l.tab);
      if (has_draft) {
        const float q = cvq[e];
        if (q == q) zq += exp_sum(((double)q - Mq) * a.inv_t, l.tab);
      }
    }
    // the decide pass takes packed target values that are not NaN (a NaN
    // draft value it tests itself)
    if (__ballot(tnan) == 0ull) pk = (has_draft ? kPkJoint : kPkTarget) | tot;
  } else {
    // a value that is masked or NaN becomes -inf: no maximum, weight 0.
    // The target row whole before the draft row, whose loads are behind it.
    auto side = [&](float (&x)[kPerThread], double &M, double &z) __attribute__((always_inline)) {
      float m = -__builtin_inff();
#pragma unroll
      for (int i = 0; i < kPerThread; ++i) {
        x[i] = ((ok >> i) & 1u) != 0u && x[i] == x[i] ? x[i] : -__builtin_inff();
        m = fmaxf(m, x[i]);
      }
      M = (double)wave_max(m);
#pragma unroll
      for (int i = 0; i < kPerThread; ++i) {
        z += exp_sum(((double)x[i] - M) * a.inv_t, l.tab);
        asm volatile("" : "+v"(z));
        if ((i & 3) == 3) __builtin_amdgcn_sched_barrier(0);
      }
    };
    side(xt, Mt, zt);
    if (has_draft) {
      settle_chunk(base, a.vocab, xq);
      side(xq, Mq, zq);
    }
  }
  zt = wave_sum_d(zt);
  zq = wave_sum_d(zq);
  if (lane == 0) {
    l.m[0][wave] = Mt;
    l.m[1][wave] = Mq;
    l.z[0][wave] = zt;
    l.z[1][wave] = zq;
  }
  // the wave's packed values (in the order the decide pass packs them from
  // the rows, so that its sums are the same) and how they were packed
  if (kMask) {
    const int64_t w = ((int64_t)pos * a.chunks + c) * kWaves + wave;
    float *pv = a.pk_v + w * (2 * kCompact);
    for (uint32_t e = (uint32_t)lane; pk && e < tot; e += 64u) {
      pv[e] = cvt[e];
      if (pk & kPkJoint) pv[kCompact + e] = cvq[e];
    }
    if (lane == 0) a.pk_n[w] = pk;
  }
  lds_barrier();
  if (tid < 2) {
    // the chunk's statistics of one row: the waves' sums brought to the
    // chunk's maximum (a wave without allowed values has sum 0)
    const double *wm = l.m[tid], *wz = l.z[tid];
    double m = wm[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) m = fmax(m, wm[w]);
    double z = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const double e = exp_sum((wm[w] - m) * a.inv_t, l.tab);
      if (wz[w] > 0.0) z += wz[w] * e;
    }
    double *o = a.stats + ((int64_t)pos * a.chunks + c) * 4 + 2 * tid;
    o[0] = m;
    o[1] = z;
  }
}

struct Decided {
  int a;         // accepted drafts; the position that draws
  double mt, zt, mq, zq;
};

struct DecideLds {
  double m[SAS_MAX_DRAFT + 1][2];
  double z[SAS_MAX_DRAFT + 1][2];
  int acc[SAS_MAX_DRAFT];
  float ct[kWaves][kCompact];  // a wave's allowed target values, packed
  float cq[kWaves][kCompact];  // and the draft values of the same ids
  ExpTab tab;
};

// Softmax statistics of every position of sequence s from the chunk
// statistics, then the accepted prefix.  Identical in every block.
__device__ Decided decide(const VerifyArgs &a, int s, DecideLds &l) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int L = a.L, P1 = L + 1;
  const double T = a.temperature;
  // the acceptance inputs (loaded with the statistics: nothing depends on them)
  uint32_t d = 0u;
  float dxt = 0.0f, dxq = 0.0f;
  double u1 = 0.0;
  if (tid < L) {
    const int pos = s * P1 + tid;
    d = a.draft_ids[(int64_t)s * L + tid];
    dxt = a.dtok[2 * pos];
    dxq = a.dtok[2 * pos + 1];
    u1 = a.uniforms[(int64_t)pos * 2];
  }
  if (a.chunks <= 64 && P1 <= 2 * kWaves) {
    // at most two positions per wave and one chunk per lane: both
    // positions' statistics are loaded at once (clamped into the existing
    // ones), then combined as below
    const bool cok = lane < a.chunks;
    const int c = min(lane, a.chunks - 1);
    f64x2 st[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int j = min(wave + kWaves * i, P1 - 1);
      const f64x2 *p = reinterpret_cast<const f64x2 *>(a.stats + ((int64_t)(s * P1 + j) * a.chunks + c) * 4);
      st[i][0] = p[0];  // (max, sum) of the target row
      st[i][1] = p[1];  // and of the draft row
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int j = wave + kWaves * i;
      if (j < P1) {
        for (int side = 0; side < (j < L ? 2 : 1); ++side) {
          const double mc = st[i][side].x, zc = cok ? st[i][side].y : 0.0;
          const double m = wave_max_d(fmax(dneg_inf(), cok ? mc : dneg_inf()));
          double z = 0.0;
          if (zc > 0.0) z += zc * exp_sum((mc - m) * a.inv_t, l.tab);
          z = wave_sum_d(z);
          if (lane == 0) {
            l.m[j][side] = m;
            l.z[j][side] = z;
          }
        }
      }
    }
  } else {
    for (int j = wave; j < P1; j += kWaves) {
      const double *st = a.stats + (int64_t)(s * P1 + j) * a.chunks * 4;
      for (int side = 0; side < (j < L ? 2 : 1); ++side) {
        double m = dneg_inf();
        for (int c = lane; c < a.chunks; c += 64) m = fmax(m, st[c * 4 + side * 2]);
        m = wave_max_d(m);
        double z = 0.0;
        for (int c = lane; c < a.chunks; c += 64) {
          const double zc = st[c * 4 + side * 2 + 1];
          if (zc > 0.0) z += zc * exp_sum((st[c * 4 + side * 2] - m) * a.inv_t, l.tab);
        }
        z = wave_sum_d(z);
        if (lane == 0) {
          l.m[j][side] = m;
          l.z[j][side] = z;
        }
      }
    }
  }
  __syncthreads();
  if (tid < L) {
    const int j = tid;
    double pd = 0.0, qd = 0.0;
    const bool in_vocab = d < (uint32_t)a.vocab;
    if (in_vocab) {
      // dtok: written by the statistics pass for every in-vocabulary draft
      // token (NaN when masked)
      const double wt = dxt == dxt ? fd_exp(((double)dxt - l.m[j][0]) / T) : 0.0;
      const double wq = dxq == dxq ? fd_exp(((double)dxq - l.m[j][1]) / T) : 0.0;
      pd = wt / l.z[j][0];
      qd = wq / l.z[j][1];
    }
    l.acc[j] = in_vocab && pd > 0.0 && u1 * qd <= pd;
  }
  __syncthreads();
  Decided r;
  r.a = L;
  for (int j = 0; j < L; ++j)
    if (!l.acc[j]) {
      r.a = j;
      break;
    }
  r.mt = l.m[r.a][0];
  r.zt = l.z[r.a][0];
  r.mq = r.a < L ? l.m[r.a][1] : 0.0;
  r.zq = r.a < L ? l.z[r.a][1] : 0.0;
  return r;
}

// Residual weight max(0, p - q) and target weight exp((x - M) / T) of one
// id whose target value is allowed and not NaN.  izt, izq: 1 / zt, 1 / zq.
struct Weights {
  double mt, izt, mq, izq, inv_t;
  bool resid;
  const ExpTab &tab;
  __device__ __forceinline__ void at(float xt, float xq, bool q_ok, double &wt, double &r) const {
    wt = exp_sum(((double)xt - mt) * inv_t, tab);
    r = 0.0;
    if (resid) {
      const double eq = exp_sum(((double)xq - mq) * inv_t, tab);
      const double wq = q_ok ? eq : 0.0;
      const double d = wt * izt - wq * izq;
      r = d > 0.0 ? d : 0.0;
    }
  }
};

template <bool kMask>
__global__ __launch_bounds__(kThreads, 5) void verify_decide_kernel(VerifyArgs a) {
  __shared__ DecideLds l;
  const int c = blockIdx.x, s = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  l.tab.fill(exp_tab_entry());
  const Decided d = decide(a, s, l);
  const int P1 = a.L + 1;
  const int pos = s * P1 + d.a;
  const bool resid = d.a < a.L;
  const int base = c * kVChunk;
  const Weights w{d.mt, 1.0 / d.zt, d.mq, resid ? 1.0 / d.zq : 0.0, a.inv_t, resid, l.tab};
  double pm = 0.0, rs = 0.0;
  // the wave's allowed ids as the statistics pass packed them (both rows,
  // or the target row where no residual is drawn); else the rows again
  const int64_t wpk = ((int64_t)pos * a.chunks + c) * kWaves + wave;
  // (without a mask no wave but the last of a row has few: not packed)
  const uint32_t pk = kMask ? a.pk_n[wpk] : 0u;
  if (resid ? (pk & kPkJoint) != 0u : (pk & (kPkJoint | kPkTarget)) != 0u) {
    const float *pv = a.pk_v + wpk * (2 * kCompact);
    const uint32_t tot = pk & kPkCount;
    for (uint32_t e = (uint32_t)lane; e < tot; e += 64u) {
      const float vq = resid ? pv[kCompact + e] : 0.0f;
      double wt, r;
      w.at(pv[e], vq, resid && vq == vq, wt, r);
      pm += wt;
      rs += r;
    }
  } else {
    float xt[kPerThread], xq[kPerThread];
    load_chunk(a.target + (int64_t)pos * a.stride, base, a.vocab, xt);
    if (resid) load_chunk(a.draft + ((int64_t)s * a.L + d.a) * a.stride, base, a.vocab, xq);
    settle_chunk(base, a.vocab, xt);
    if (resid) settle_chunk(base, a.vocab, xq);
    uint32_t mw[4];
    load_words<kMask>(kMask ? a.mask + (int64_t)pos * a.mask_stride : nullptr, base, a.vocab, mw);
    const uint32_t ok = nan_free(xt, allow_bits(mw, base, a.vocab));
    // the allowed ids' values, packed per wave when few (a sparse mask)
    uint32_t pre, tot;
    wave_place((uint32_t)__popc(ok), pre, tot);
    if (tot <= (uint32_t)kCompact) {
      uint32_t jj = pre;
#pragma unroll
      for (int i = 0; i < kPerThread; ++i)
        if ((ok >> i) & 1u) {
          l.ct[wave][jj] = xt[i];
          l.cq[wave][jj] = resid ? xq[i] : 0.0f;
          ++jj;
        }
      wave_lds_sync();
      for (uint32_t e = (uint32_t)lane; e < tot; e += 64u) {
        const float vq = l.cq[wave][e];
        double wt, r;
        w.at(l.ct[wave][e], vq, resid && vq == vq, wt, r);
        pm += wt;
        rs += r;
      }
    } else {
#pragma unroll
      for (int i = 0; i < kPerThread; ++i) {
        // no branch per value, so that exponentials overlap
        const bool in = (ok >> i) & 1u;
        const float vq = resid ? xq[i] : 0.0f;
        double wt, r;
        w.at(xt[i], vq, in && vq == vq, wt, r);
        pm += in ? wt : 0.0;
        rs += in ? r : 0.0;
        // two values' exponentials overlap, not all sixteen's (whose
        // registers would leave room for four waves per SIMD)
        asm volatile("" : "+v"(pm), "+v"(rs));
        if (i & 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  pm = wave_sum_d(pm);
  rs = wave_sum_d(rs);
  // the wave's ids are consecutive: its masses tell the draw in which of
  // the chunk's kWaves runs of ids the target falls
  if (lane == 0) {
    double *o = a.part + (((int64_t)s * a.chunks + c) * kWaves + wave) * 2;
    o[0] = rs;
    o[1] = pm;
  }
  if (c == 0 && tid == 0) {
    double *q = a.seqrec + (int64_t)s * 8;
    q[0] = (double)d.a;
    q[1] = d.mt;
    q[2] = d.zt;
    q[3] = d.mq;
    q[4] = d.zq;
  }
}

struct DrawLds {
  double wsum[kWaves];
  int chunk;       // the run of kWaveIds ids that the draw falls in: its chunk,
  int run;         // its place in the chunk,
  double before;   // and the running mass before it
  int resid;
  int last_mode;   // no running mass passes the target: the run's last id with a weight
  double target;
  uint32_t found;
  uint32_t last;
  ExpTab tab;
};

template <bool kMask>
__global__ __launch_bounds__(kThreads) void verify_draw_kernel(VerifyArgs a) {
  __shared__ DrawLds l;
  const int s = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int L = a.L, P1 = L + 1;
  const int C = a.chunks;
  const f64x2 *part = reinterpret_cast<const f64x2 *>(a.part) + (int64_t)s * C * kWaves;
  // Loads that do not wait for the accepted count come first: wave 0's run
  // masses (one chunk per lane when there are at most 64) and the second
  // uniform of every position of the sequence (P1 <= 64).
  f64x2 pc[kWaves];
#pragma unroll
  for (int v = 0; v < kWaves; ++v) pc[v] = part[min(lane, C - 1) * kWaves + v];
  const double u2c = a.uniforms[((int64_t)s * P1 + min(lane, P1 - 1)) * 2 + 1];
  l.tab.fill(exp_tab_entry());
  const double *q = a.seqrec + (int64_t)s * 8;
  const int acc = (int)q[0];
  const int pos = s * P1 + acc;
  const double u2 = __shfl(u2c, acc, 64);
  if (tid == 0) {
    l.found = SAS_NO_TOKEN;
    l.last = 0;
    l.chunk = -1;
  }
  if (tid <= L && tid != acc)
    a.out_tokens[(int64_t)s * P1 + tid] = tid < acc ? a.draft_ids[(int64_t)s * L + tid] : SAS_NO_TOKEN;
  if (tid == 0) a.out_accepted[s] = acc;

  // Which weights draw: the residual unless it is all zero, else the target.
  if (wave == 0) {
    const int R = (C + 63) / 64;
    const int c0 = lane * R, c1 = min(C, c0 + R);
    // run v's residual (col 0) or target (col 1) mass of chunk c; with one
    // chunk per lane (c == lane) from the registers
    auto wrun = [&](int c, int v, int col) __attribute__((always_inline)) -> double {
      const f64x2 x = C <= 64 ? pc[v] : part[c * kWaves + v];
      return col ? x.y : x.x;
    };
    auto wpart = [&](int c, int col) __attribute__((always_inline)) -> double {
      double x = wrun(c, 0, col);
#pragma unroll
      for (int v = 1; v < kWaves; ++v) x += wrun(c, v, col);
      return x;
    };
    bool resid = acc < L;
    if (resid) {
      double v = 0.0;
      for (int c = c0; c < c1; ++c) v += wpart(c, 0);
      resid = wave_sum_d(v) > 0.0;
    }
    const int col = resid ? 0 : 1;
    double v = 0.0;
    for (int c = c0; c < c1; ++c) v += wpart(c, col);
    const double incl = wave_scan_d(v);
    double excl = __shfl_up(incl, 1, 64);
    if (lane == 0) excl = 0.0;
    const double tot = bcast(incl, 63);
    const double target = u2 * tot;
    // the first chunk whose running total passes the target, else the last
    // with a mass
    int hit = -1;
    double cum = excl, hit_before = 0.0;
    int lastc = -1;
    double last_before = 0.0;
    for (int c = c0; c < c1; ++c) {
      const double wc = wpart(c, col);
      if (!(wc > 0.0)) continue;
      lastc = c;
      last_before = cum;
      const double nxt = cum + wc;
      if (hit < 0 && nxt > target) {
        hit = c;
        hit_before = cum;
      }
      cum = nxt;
    }
    const bool any_hit = __ballot(hit >= 0) != 0ull;
    const uint64_t cand = any_hit ? __ballot(hit >= 0) : __ballot(lastc >= 0);
    // its first run whose running total passes the target, else its last
    // with a mass (every lane looks at its own chunk)
    const int ch = any_hit ? hit : lastc;
    double b = any_hit ? hit_before : last_before, run_before = b;
    int run = 0;
    bool passed = false;
    if (ch >= 0) {
#pragma unroll
      for (int r = 0; r < kWaves; ++r) {
        const double w = wrun(ch, r, col);
        if (!passed && w > 0.0) {
          run = r;
          run_before = b;
          passed = any_hit && b + w > target;
          b += w;
        }
      }
    }
    if (tot > 0.0 && cand) {
      const int src = any_hit ? __ffsll((long long)cand) - 1 : 63 - __clzll((long long)cand);
      if (lane == src) {
        l.chunk = ch;
        l.run = run;
        l.before = run_before;
        l.last_mode = passed ? 0 : 1;
      }
    }
    if (lane == 0) {
      l.target = target;
      l.resid = resid;
    }
  }
  __syncthreads();
  if (l.chunk < 0) {
    if (tid == 0) a.out_tokens[(int64_t)s * P1 + acc] = SAS_NO_TOKEN;
    return;
  }
  const bool resid = l.resid != 0;
  const double target = l.target;
  const bool last_mode = l.last_mode != 0;

  // The run's ids in ascending order, four consecutive ones per thread: the
  // same weights whose sum the decide pass took, then their running sums.
  constexpr int kPer = kWaveIds / kThreads;
  static_assert(kPer == 4, "one mask word per thread");
  const int64_t id0 = (int64_t)l.chunk * kVChunk + l.run * kWaveIds + tid * kPer;
  const float *trow = a.target + (int64_t)pos * a.stride;
  const float *drow = a.draft + ((int64_t)s * L + min(acc, L - 1)) * a.stride;
  const int64_t last_id = (int64_t)a.vocab - 1;
  float vt[kPer], vq[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    vt[i] = trow[min(id0 + i, last_id)];
    vq[i] = drow[min(id0 + i, last_id)];
  }
  const uint32_t word = kMask ? a.mask[(int64_t)pos * a.mask_stride + (min(id0, last_id) >> 5)] >> (id0 & 31) : ~0u;
  const Weights w{q[1], 1.0 / q[2], q[3], resid ? 1.0 / q[4] : 0.0, a.inv_t, resid, l.tab};
  double wv[kPer], mine = 0.0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const bool in = ((word >> i) & 1u) && id0 + i <= last_id && vt[i] == vt[i];
    double wt, r;
    w.at(vt[i], vq[i], vq[i] == vq[i], wt, r);
    wv[i] = in ? (resid ? r : wt) : 0.0;
    mine += wv[i];
  }
  // exclusive prefix of the per-thread sums in thread order
  const double incl = wave_scan_d(mine);
  if (lane == 63) l.wsum[wave] = incl;
  double ex = __shfl_up(incl, 1, 64);
  if (lane == 0) ex = 0.0;
  __syncthreads();
  double cum = l.before;
  for (int v = 0; v < wave; ++v) cum += l.wsum[v];
  cum += ex;
  uint32_t found = SAS_NO_TOKEN, last = 0u;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    if (wv[i] > 0.0) {
      const uint32_t id = (uint32_t)(id0 + i);
      last = id + 1u;
      cum += wv[i];
      if (found == SAS_NO_TOKEN && cum > target) found = id;
    }
  }
  if (!last_mode && found != SAS_NO_TOKEN) atomicMin(&l.found, found);
  if (last) atomicMax(&l.last, last);
  __syncthreads();
  if (tid == 0) {
    uint32_t tok = l.found;
    if (last_mode || tok == SAS_NO_TOKEN) tok = l.last ? l.last - 1u : SAS_NO_TOKEN;
    a.out_tokens[(int64_t)s * P1 + acc] = tok;
  }
}

}  // namespace

size_t verify_scratch_bytes(int seqs, int L, int vocab) {
  const size_t chunks = ((size_t)vocab + kVChunk - 1) / kVChunk;
  const size_t positions = (size_t)seqs * (L + 1);
  return (positions * chunks * 4 + (size_t)seqs * chunks * kWaves * 2 + (size_t)seqs * 8) * sizeof(double) +
         positions * 2 * sizeof(float) + positions * chunks * kWaves * sizeof(uint32_t) +
         positions * chunks * kWaves * 2 * kCompact * sizeof(float);
}

hipError_t launch_verify(const VerifyArgs &a, hipStream_t stream) {
  const dim3 block(kThreads);
  const dim3 g1(a.chunks, a.seqs * (a.L + 1)), g2(a.chunks, a.seqs), g3(a.seqs);
  if (a.mask) {
    hipLaunchKernelGGL(verify_stats_kernel<true>, g1, block, 0, stream, a);
    hipLaunchKernelGGL(verify_decide_kernel<true>, g2, block, 0, stream, a);
    hipLaunchKernelGGL(verify_draw_kernel<true>, g3, block, 0, stream, a);
  } else {
    hipLaunchKernelGGL(verify_stats_kernel<false>, g1, block, 0, stream, a);
    hipLaunchKernelGGL(verify_decide_kernel<false>, g2, block, 0, stream, a);
    hipLaunchKernelGGL(verify_draw_kernel<false>, g3, block, 0, stream, a);
  }
  return hipGetLastError();
}

}  // namespace sas
