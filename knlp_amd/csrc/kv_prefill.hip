// Causal attention of fresh prompts (gfx950): every query token of a sequence
// attends to that sequence's keys up to itself, K and V straight from the
// step's fp16 / bf16 rows (the reference's prefill, F:3127-3198, which runs
// per-sequence SDPA in fp32; F = fused-quant/fused_int4.v0.1.0.py).
//
// What bounds it: the matrix cores, 4 D flops per visible (query, key) pair
// and head.  One block of 4 waves takes 128 queries of one q head, a wave 32
// of them, and walks the keys 64 at a time:
//  S^T = K Q^T by v_mfma_f32_32x32x16: fp16 / bf16 products are exact in the
//      fp32 accumulator, so the scores carry no 16-bit rounding.  With the
//      scores transposed a lane holds one query's scores of 16 keys, so the
//      softmax's max and sum are in-lane (plus one exchange between the wave's
//      halves), and the probabilities are the B operand of O^T = V^T P^T as
//      they lie: no cross-lane movement between the two products.
//  P   enters as hi + lo, two 16-bit values (fp16: p 2^12, so that the pair
//      keeps 22 bits down to 2^-14 of the largest p; bf16: 16 bits at any
//      magnitude), one product each.  Against 64 bits, prompts of 300 to 3000,
//      the error beside the output's own rounding is 2e-7 to 7e-7 in fp16
//      (rounding 2.0e-4) and 1.7e-6 to 2.3e-6 in bf16 (1.6e-3); fp32 SDPA has
//      3e-7 to 1.7e-6, and the totals agree to seven places.
//  V^T is read from row-major LDS with the transposing ds_read_b64_tr_b16.
// K and V tiles are staged through registers into two LDS buffers: tile i + 2
// is loaded from memory and tile i + 1 written to LDS while tile i computes,
// one barrier per tile; 72 KB at D = 128, two blocks per CU, so one wave's
// softmax runs under the other's products.  LDS rows are padded by 16 bytes
// (K: the 16 rows of a b128 phase then start 4 banks apart) and by 32 (V: the
// 8 rows of a transposing read 8 banks apart).
//
// The matrix units are busy 59 % of the CUs' busy cycles, at a clock of about
// 1.8 GHz under this load (busy cycles over time), and the vector units most of
// the rest.  Running
// the next 32 keys' QK products among the exponentials of these (one wave's
// units overlapped by hand) gained 3 % at D = 64 and lost 1-2 % at 128: the
// other wave of the SIMD fills the gaps already.  At D = 64 a wave raises its
// priority for its products, so that it is not the wave still short of them
// that waits: prompts of 3500 and 3000 (14 q / 2 kv heads) 83.7 -> 79.6 us.  At
// 128 that lost 0.5-2 %.
//
// Blocks are dealt out with the kv head fastest, so with 8 kv heads each XCD
// works on one head and its L2 holds that head's K and V; the query tiles with
// the most keys come first (find_tile), so the short ones fill the end.
//
// Measured: a layer's prefill of four prompts of up to 3000 tokens (32 q / 8
// kv heads of 128, bf16; 1.0e11 flops), cache writes included, took 5430 us
// with fp32 SDPA per prompt and takes 231 us; the kernel alone, one prompt of
// 8192: 718-746 us, 740-765 TFLOP/s of the visible pairs and 1.5 times that
// with lo's products (a large bf16 matmul here: 1280).  Tile order: prompts of
// 3000, 2000, 2500 and 1100 tokens took 312 us laid end to end and 302 with
// the longest tiles of all first; twelve of 1024 (12 heads of 64) 37.4 and 33.1.
#include "kv_prefill.h"

namespace knlp {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f16x __attribute__((ext_vector_type(16)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

constexpr int kBM = 128;    // queries per block (32 per wave)
constexpr int kBN = 64;     // keys per tile
constexpr int kWaves = 4;
// a row's running max is raised only when a tile exceeds it by more than 2
// (log2 units), so p <= 4 and p 2^12 <= 2^14, inside fp16
constexpr float kRaise = 2.0f;
constexpr float kPScale = 12.0f;
constexpr float kBaseMax = 1024.0f;

template <bool BF16>
__device__ __forceinline__ f16x mfma(u4 a, u4 b, f16x c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8, a),
                                                   __builtin_bit_cast(b8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a),
                                                  __builtin_bit_cast(h8, b), c, 0, 0, 0);
}

// Two probabilities as a 16-bit pair hi and the pair lo of what hi leaves.
template <bool BF16>
__device__ __forceinline__ void split2(float p0, float p1, uint32_t& hi, uint32_t& lo) {
  if constexpr (BF16) {
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{p0, p1}, b2));
    const float h0 = __builtin_bit_cast(float, hi << 16);
    const float h1 = __builtin_bit_cast(float, hi & 0xFFFF0000u);
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{p0 - h0, p1 - h1}, b2));
  } else {
    const h2 h = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(p0, p1));
    hi = __builtin_bit_cast(uint32_t, h);
    lo = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(
                                          p0 - static_cast<float>(h[0]),
                                          p1 - static_cast<float>(h[1])));
  }
}

// max / sum of a value over the wave's two halves (lanes l and l ^ 32)
__device__ __forceinline__ float half_max(float x) {
  // (one swap; the copy is opaque, else the compiler takes the two results for one)
  uint32_t a = __builtin_bit_cast(uint32_t, x), b = a;
  asm("" : "+v"(b));
  const auto w = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  return fmaxf(__builtin_bit_cast(float, static_cast<uint32_t>(w[0])),
               __builtin_bit_cast(float, static_cast<uint32_t>(w[1])));
}
__device__ __forceinline__ float half_sum(float x) { return x + __shfl_xor(x, 32, kWave); }

// Sum over the wave's lanes.
__device__ __forceinline__ int wave_total(int x) {
  return __builtin_amdgcn_readlane(static_cast<int>(wave_incl_scan(static_cast<uint32_t>(x))), 63);
}

// The sequence and query tile that the blocks numbered `t` (one per q head)
// run; false past the last.  2 to 64 sequences: the tiles of all of them from
// the highest tile number (the most keys) down, so that the longest start
// first whatever the order of the lengths.  S(h) = sum of max(0, tiles - h)
// tiles are numbered h or higher; t's number is the h with S(h + 1) <= t < S(h).
// One, or more: laid end to end, each from its last tile down.
__device__ __forceinline__ bool find_tile(const PrefillArgs& a, int t, int lane, int* start,
                                          int* len, int* tile) {
  for (int r0 = 0; r0 < a.num_seqs; r0 += kWave) {
    int s = 0, n = 0;
    if (r0 + lane < a.num_seqs) {
      s = min(max(a.starts[r0 + lane], 0), a.tokens);
      n = min(max(a.starts[r0 + lane + 1], s), a.tokens) - s;
      if (n < a.min_len) n = 0;
    }
    const int nt = (n + kBM - 1) / kBM;
    const int incl = static_cast<int>(wave_incl_scan(static_cast<uint32_t>(nt)));
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    if (t < total) {
      int c;
      if (a.num_seqs > 1 && a.num_seqs <= kWave) {
        int lo = 0, hi = total;                          // S(lo) > t >= S(hi)
        while (hi - lo > 1) {
          const int mid = (lo + hi) / 2;
          if (wave_total(max(0, nt - mid)) > t) lo = mid; else hi = mid;
        }
        const int j = t - wave_total(max(0, nt - lo - 1));       // among the sequences that have it
        const uint64_t have = __ballot(nt > lo);
        const bool mine = nt > lo && __popcll(have & ((1ull << lane) - 1)) == j;
        c = __builtin_ctzll(__ballot(mine));
        *tile = lo;
      } else {
        c = __popcll(__ballot(incl <= t));               // sequences wholly before t
        const int ntc = __builtin_amdgcn_readlane(nt, c);
        *tile = ntc - 1 - (t - (__builtin_amdgcn_readlane(incl, c) - ntc));
      }
      *start = __builtin_amdgcn_readlane(s, c);
      *len = __builtin_amdgcn_readlane(n, c);
      return true;
    }
    t -= total;
  }
  return false;
}

template <int D, bool BF16>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_kernel(PrefillArgs a) {
  constexpr int NC = D / 16;              // contraction chunks of QK
  constexpr int ND = D / 32;              // output tiles of 32 dims
  constexpr int KROW = 2 * D + 16;        // LDS row bytes
  constexpr int VROW = 2 * D + 32;
  constexpr int CH = D / 8;               // 16-byte chunks per row
  constexpr int NL = kBN * CH / (kWaves * 64);   // chunks per thread and tile
  __shared__ __attribute__((aligned(16))) uint8_t lds_k[2][kBN * KROW];
  __shared__ __attribute__((aligned(16))) uint8_t lds_v[2][kBN * VROW];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int n32 = lane & 31;
  const int half = lane >> 5;
  const int G = a.hq / a.hkv;
  const int kvh = blockIdx.x % a.hkv;
  const int rest = blockIdx.x / a.hkv;
  const int head = kvh * G + rest % G;
  int start, len, tile;
  if (!find_tile(a, rest / G, lane, &start, &len, &tile)) return;      // uniform
  start = __builtin_amdgcn_readfirstlane(start);
  len = __builtin_amdgcn_readfirstlane(len);
  tile = __builtin_amdgcn_readfirstlane(tile);

  const int q0 = tile * kBM;                       // the block's first query
  const int qw = q0 + 32 * wave;                   // the wave's first query
  const int query = qw + n32;                      // this lane's query

  // B operand of QK: this lane's query, dims 16 c + 8 half .. + 7.  The
  // softmax below needs a positive scale: a negative one enters as -q.
  u4 qf[NC];
  {
    const uint16_t* qp = a.q + static_cast<int64_t>(start + min(query, len - 1)) * a.qst +
                         head * a.qsh + 8 * half;
    const uint32_t flip = a.scale_log2 < 0.0f ? 0x80008000u : 0u;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      u4 w = *reinterpret_cast<const u4*>(qp + 16 * c);
      w ^= flip;
      // a zero scale: every score 0, uniform weights
      qf[c] = a.scale_log2 == 0.0f ? u4{0u, 0u, 0u, 0u} : w;
    }
  }
  const float sl2 = a.scale_log2 == 0.0f ? 1.0f : fabsf(a.scale_log2);
  const float thr = kRaise / sl2;

  // keys 0 .. q0 + 127 (cut at the sequence's length)
  const int keys = min(len, q0 + kBM);
  const int ntiles = (keys + kBN - 1) / kBN;
  const uint16_t* kb = a.k + static_cast<int64_t>(start) * a.kst + kvh * a.ksh;
  const uint16_t* vb = a.v + static_cast<int64_t>(start) * a.vst + kvh * a.vsh;
  // A tile's rows are read through a buffer descriptor that starts at the tile
  // and ends with the sequence's last row: the lane offsets are the same for
  // every tile, and rows past the end read as 0 (V's must not be stale: a zero
  // probability would not cancel an Inf or NaN) with no compares or selects.
  uint32_t ko[NL], vo[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int c = static_cast<int>(threadIdx.x) + i * kWaves * 64;
    ko[i] = static_cast<uint32_t>(2 * ((c / CH) * a.kst + 8 * (c % CH)));
    vo[i] = static_cast<uint32_t>(2 * ((c / CH) * a.vst + 8 * (c % CH)));
  }
  const auto rows_of = [&](const uint16_t* base, int64_t st, int t) {
    const uint32_t rows = static_cast<uint32_t>(min(kBN, len - t * kBN));     // at least 1
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(base + static_cast<int64_t>(t) * kBN * st), static_cast<short>(0),
        static_cast<int>((rows - 1) * static_cast<uint32_t>(2 * st) + 2 * D), 0x00020000);
  };
  u4 kr[NL], vr[NL];
  const auto load = [&](int t) {
    const auto kd = rows_of(kb, a.kst, t), vd = rows_of(vb, a.vst, t);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      kr[i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(kd, ko[i], 0, 0));
      vr[i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(vd, vo[i], 0, 0));
    }
  };
  const auto store = [&](int b) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = static_cast<int>(threadIdx.x) + i * kWaves * 64;
      *reinterpret_cast<u4*>(&lds_k[b][(c / CH) * KROW + 16 * (c % CH)]) = kr[i];
      *reinterpret_cast<u4*>(&lds_v[b][(c / CH) * VROW + 16 * (c % CH)]) = vr[i];
    }
  };

  f16x o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;

  load(0);
  store(0);
  if (ntiles > 1) load(1);
  __syncthreads();
  for (int t = 0; t < ntiles; ++t) {
    if (t + 1 < ntiles) store((t + 1) & 1);      // last read by tile t - 1, before the barrier
    if (t + 2 < ntiles) load(t + 2);
    const int k0 = t * kBN;
    if (k0 <= qw + 31) {                         // uniform: some query of the wave sees the tile
      const uint8_t* lk = lds_k[t & 1];
      const uint8_t* lv = lds_v[t & 1];
      if constexpr (D == 64) __builtin_amdgcn_s_setprio(1);
      f16x s[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[x][r] = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const u4 kf = *reinterpret_cast<const u4*>(lk + (32 * x + n32) * KROW + 32 * c +
                                                     16 * half);
          s[x] = mfma<BF16>(kf, qf[c], s[x]);
        }
      }
      if constexpr (D == 64) __builtin_amdgcn_s_setprio(0);
      // register r of s[x] is key k0 + 32 x + 8 (r / 4) + 4 half + r % 4
      if (k0 + kBN - 1 > qw) {                   // uniform: the diagonal
        // (keeps this a branch: as selects it was 80 operations in every tile)
        asm volatile("");
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (k0 + 32 * x + 8 * (r / 4) + 4 * half + r % 4 > query) s[x][r] = -INFINITY;
      }
      float tmax = s[0][0];
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[x][r]);
      tmax = half_max(tmax);
      if (__any(tmax > m_run + thr)) {
        const float mn = tmax > m_run + thr ? tmax : m_run;
        // (the first raise: exp2(-inf) = 0; rows that see nothing yet keep -inf)
        const float alpha = mn == m_run ? 1.0f : __builtin_amdgcn_exp2f((m_run - mn) * sl2);
        m_run = mn;
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
      }
      // p = 2^(12 + (score - max) sl2), the max's part taken out once (every
      // score so far -inf: any finite base gives p = 0)
      const float ref = m_run == -INFINITY ? 0.0f : m_run;
      float base = kPScale - ref * sl2;
      // the base is rounded to its own last bit, which is part of p's exponent:
      // where that grows past 2^-14 the max is taken from the scores instead
      if (__any(fabsf(base) > kBaseMax)) {       // uniform, rare
        asm volatile("");                        // (a branch, as above)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[x][r] -= ref;
        base = kPScale;
      }
      uint32_t hi[16], lo[16];
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const float p0 = __builtin_amdgcn_exp2f(fmaf(s[x][r], sl2, base));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(s[x][r + 1], sl2, base));
          l_run += p0;
          l_run += p1;
          split2<BF16>(p0, p1, hi[8 * x + r / 2], lo[8 * x + r / 2]);
        }
      // O^T += V^T P^T, 16 keys a product: slot e of lane half h is key
      // 16 m + 8 (e / 4) + 4 h + e % 4, on both sides
      if constexpr (D == 64) __builtin_amdgcn_s_setprio(1);
      const uint8_t* vp = lv + (4 * half + (lane & 15) / 4) * VROW + 32 * ((lane >> 4) & 1) +
                          8 * (lane & 3);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const u4 ph = {hi[4 * m], hi[4 * m + 1], hi[4 * m + 2], hi[4 * m + 3]};
        const u4 pl = {lo[4 * m], lo[4 * m + 1], lo[4 * m + 2], lo[4 * m + 3]};
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          using lp = __attribute__((address_space(3))) s4*;
          const uint8_t* p0 = vp + 16 * m * VROW + 64 * d;
          const s4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(p0));
          const s4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(p0 + 8 * VROW));
          const uint2 w0 = __builtin_bit_cast(uint2, v0), w1 = __builtin_bit_cast(uint2, v1);
          const u4 vf = {w0.x, w0.y, w1.x, w1.y};
          o[d] = mfma<BF16>(vf, ph, o[d]);
          o[d] = mfma<BF16>(vf, pl, o[d]);
        }
      }
      if constexpr (D == 64) __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
  }
  l_run = half_sum(l_run);
  if (query >= len) return;
  // (no visible score above -inf: 0, as SDPA's safe softmax)
  const float inv = l_run == 0.0f ? 0.0f : 1.0f / l_run;
  uint16_t* op = a.out + static_cast<int64_t>(start + query) * a.ost + head * a.osh;
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      uint16_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = o[d][4 * b + i] * inv;
        w[i] = BF16 ? __builtin_bit_cast(uint16_t, static_cast<__bf16>(x))
                    : float_to_half_bits(x);
      }
      *reinterpret_cast<uint2*>(op + 32 * d + 8 * b + 4 * half) =
          make_uint2(w[0] | (static_cast<uint32_t>(w[1]) << 16),
                     w[2] | (static_cast<uint32_t>(w[3]) << 16));
    }
}

}  // namespace

int launch_prefill(const PrefillArgs& a, int head_size, int bf16, hipStream_t stream) {
  // every sequence has at most one partial tile, so this many tiles hold them all
  const int64_t tiles = a.tokens / kBM + a.num_seqs;
  const int64_t blocks = tiles * a.hq;
  if (blocks > 0x7FFFFFFF) return KNLP_ERR_SHAPE;
  const dim3 grid(static_cast<uint32_t>(blocks)), block(kWaves * 64);
#define KNLP_PREFILL(D, B) hipLaunchKernelGGL((prefill_kernel<D, B>), grid, block, 0, stream, a)
  if (head_size == 128) {
    if (bf16) KNLP_PREFILL(128, true); else KNLP_PREFILL(128, false);
  } else if (head_size == 64) {
    if (bf16) KNLP_PREFILL(64, true); else KNLP_PREFILL(64, false);
  } else {
    return KNLP_ERR_SHAPE;
  }
#undef KNLP_PREFILL
  return hipGetLastError() == hipSuccess ? KNLP_OK : KNLP_ERR_LAUNCH;
}

}  // namespace knlp
