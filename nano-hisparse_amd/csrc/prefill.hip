// Causal GQA self-attention for prefill (flash-attention forward, MFMA).
//
// out[s, h] = softmax_{t <= s}(q[s, h] . k[t, h/g] * D^-1/2) . v[t, h/g] for
// one prompt of `seq` tokens, bf16 or fp16 in, fp32 accumulation. A
// workgroup of NW waves owns 32 * NW queries of one query head (32 per wave)
// and walks the key tiles of 64 up to the diagonal with an online softmax.
//
// MFMA v_mfma_f32_32x32x16 (bf16 / f16): lane l supplies row l%32 of A and
// column l%32 of B at k = (l/32)*8 .. +7, and receives D rows
// 8*(i/4) + (l/32)*4 + i%4 (i = 0..15) of column l%32. The scores are
// computed transposed, S^T = K Q^T (A = 32 key rows of the LDS K tile, B =
// the wave's 32 query rows, kept in registers), so a lane holds 16 keys of
// every 32-key block for its query column l%32 and a query's softmax
// statistics live in the lane pair l, l ^ 32. The output is accumulated
// transposed too, O^T = V^T P^T: registers 8s .. 8s+7 of a score block are
// the B operand of k step s as they stand once the step's 16 keys are taken
// in the order (l/32)*4 + 0..3, 8 + (l/32)*4 + 0..3, and the LDS V^T tile
// stores each 16 keys in that order, so its A operand is one 16-byte read.
// The rescaling by a query's max stays in its lane.
//
// Why 32 queries per wave and 32x32 tiles: a wave reads every K and V byte
// of the tile from LDS once per MFMA operand, so the LDS bytes per flop fall
// with the queries a wave holds. At 16 per wave (16x16 tiles) the LDS reads
// took twice the matrix cores' time; at 32 they take as long as it does, and
// the wave still fits 256 registers, so two waves share a SIMD and one's
// softmax runs beside the other's MFMAs. K and V^T rows are stored with their
// 16-byte chunks permuted by an XOR of the row, so that reads of 16 rows at
// one chunk meet all 64 banks.
//
// The weights are rounded to the input dtype for the P.V product and the
// denominator sums the same rounded weights, so each output is an exact
// convex combination of V rows. A tile that moves no query's max rescales
// nothing. (Moving the max only once a score exceeds it by 2^8 would skip
// more, 3% of the time at 32K tokens, but the largest weight would no longer
// be exactly 1: the error against float64 grew by 3%.)
//
// Measured (MI355X, bf16, 32/8 heads of 128): 32768 tokens 8.86 ms, 993
// TFLOP/s causal (22.37 ms with 16 queries per wave and 16x16 tiles; a large
// hipBLASLt product reaches 1342); 4000 tokens 157 us (605); 1999 tokens of
// 28/4 heads 63 us (159), where the longest workgroup's 32 tiles of ~2 us
// are the bound and the chip is half idle.
#include <math.h>

#include "nhs_common.h"

namespace nhs {

constexpr int kPfBN = 64;            // keys per tile
constexpr int kPfCUs = 256;

typedef __bf16 pf_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 pf_f16x8 __attribute__((ext_vector_type(8)));
typedef float pf_f32x16 __attribute__((ext_vector_type(16)));
typedef float pf_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 pf_bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 pf_f16x2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ pf_f32x16 mfma32x32x16(uint4 a, uint4 b, pf_f32x16 c) {
  if constexpr (T::dtype == NHS_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(pf_bf16x8, a), __builtin_bit_cast(pf_bf16x8, b),
                                                  c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pf_f16x8, a), __builtin_bit_cast(pf_f16x8, b), c,
                                                 0, 0, 0);
}

// two fp32 weights as a packed pair of the input dtype (round to nearest
// even, by the hardware conversions)
template <typename T>
__device__ __forceinline__ uint32_t pf_pack(float lo, float hi) {
  if constexpr (T::dtype == NHS_BF16)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((pf_f32x2){lo, hi}, pf_bf16x2));
  else
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((pf_f32x2){lo, hi}, pf_f16x2));
}

// acc + both halves of a packed pair, in fp32
template <typename T>
__device__ __forceinline__ float pf_add_pair(uint32_t pair, float acc) {
  if constexpr (T::dtype == NHS_BF16)
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(pf_bf16x2, pair),
                                           __builtin_bit_cast(pf_bf16x2, 0x3f803f80u), acc, false);
  else
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(pf_f16x2, pair), __builtin_bit_cast(pf_f16x2, 0x3c003c00u), acc,
                                  false);
}

__device__ __forceinline__ uint32_t pf_word(const uint4& v, int w) {
  return w == 0 ? v.x : w == 1 ? v.y : w == 2 ? v.z : v.w;
}

struct PrefillArgs {
  const char* q;
  const char* k;
  const char* v;
  int64_t q_s, q_h, k_s, k_h, v_s, v_h;  // element strides
  int seq, q_heads, group;
  float scale_log2;  // D^-1/2 * log2(e)
  char* out;
  int64_t o_s, o_h;
};

// LDS slot of 16-byte chunk c of K row r (D * 2 bytes) and of V^T row r (128 bytes): any 16 consecutive rows at one
// chunk fall on distinct banks.
template <int D>
__device__ __forceinline__ int pf_k_slot(int r, int c) {
  return D == 128 ? c ^ (r & 15) : c ^ ((r >> 1) & 7);
}
__device__ __forceinline__ int pf_v_slot(int r, int c) { return c ^ (((r >> 1) ^ (r >> 4)) & 7); }

template <typename T, int D, int NW>
__global__ __launch_bounds__(NW* kWave, 2) void prefill_attention_kernel(PrefillArgs a) {
  constexpr int kThreads = NW * kWave;
  constexpr int BM = 32 * NW;          // queries per workgroup
  constexpr int KS = D / 16;           // 16-wide k steps of Q.K
  constexpr int DB = D / 32;           // 32-wide dim blocks of the output
  constexpr int C = D / 8;             // 16-byte chunks of a K or V row
  constexpr int kVRow = kPfBN * 2;     // bytes per V^T row
  // a staging unit is four 16-byte loads: 4 keys x 8 dims of V (a 4-key piece of 8 V^T rows), or one chunk of 4 K rows
  constexpr int kUnits = kPfBN * D / 32;  // units per tile of each
  constexpr int kMine = (2 * kUnits + kThreads - 1) / kThreads;
  // two buffers per tile: tile t+1 is stored while tile t is read, one barrier per tile
  __shared__ __attribute__((aligned(16))) char k_buf[2][kPfBN * D * 2];
  __shared__ __attribute__((aligned(16))) char v_buf[2][D * kVRow];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, n = lane & 31;
  // The longest rows first; with a multiple of 8 heads each XCD (workgroup id mod 8) keeps neighbouring heads, so that
  // the heads of one KV head read its tiles from one L2.
  const int n_qblocks = (a.seq + BM - 1) / BM;
  const int id = blockIdx.x;
  const int h = a.q_heads % 8 == 0 ? (id % 8) * (a.q_heads / 8) + (id / 8) % (a.q_heads / 8) : id % a.q_heads;
  const int qb = n_qblocks - 1 - id / a.q_heads;
  const int kvh = h / a.group;
  const int q0 = qb * BM, wq0 = q0 + wave * 32;
  const int query = wq0 + n;  // this lane's query (column of S^T)

  // the wave's query rows as B operands: dims s*16 + half*8 .. +7
  uint4 qf[KS];
  {
    const int qr = min(query, a.seq - 1);
    const char* qp = a.q + ((int64_t)qr * a.q_s + (int64_t)h * a.q_h) * T::bytes + half * 16;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const uint4*>(qp + s * 32);
  }

  float m = -INFINITY, l = 0.f;  // running max (of the unscaled scores) and this lane's share of the denominator
  pf_f32x16 o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[b][i] = 0.f;

  const int last_key = min(a.seq, q0 + BM) - 1;
  const int n_tiles = last_key / kPfBN + 1;
  const char* kbase = a.k + (int64_t)kvh * a.k_h * T::bytes;
  const char* vbase = a.v + (int64_t)kvh * a.v_h * T::bytes;
  uint4 reg[kMine][4];
  auto load_tile = [&](int t0) {
#pragma unroll
    for (int u = 0; u < kMine; ++u) {
      const int unit = tid + u * kThreads;
      const bool is_v = unit < kUnits;
      if (unit >= 2 * kUnits) break;
      const int x = is_v ? unit : unit - kUnits;
      const int row = is_v ? (x / C) * 4 : x / C, step = is_v ? 1 : kPfBN / 4;
      const char* base = (is_v ? vbase : kbase) + (x % C) * 16;
      const int64_t stride = (is_v ? a.v_s : a.k_s) * T::bytes;
      if (t0 + kPfBN <= a.seq) {
        const char* p = base + (int64_t)(t0 + row) * stride;
#pragma unroll
        for (int i = 0; i < 4; ++i) reg[u][i] = *reinterpret_cast<const uint4*>(p + i * step * stride);
      } else {  // rows past the end re-read the last key (masked below)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          reg[u][i] = *reinterpret_cast<const uint4*>(base + (int64_t)min(t0 + row + i * step, a.seq - 1) * stride);
      }
    }
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int u = 0; u < kMine; ++u) {
      const int unit = tid + u * kThreads;
      if (unit >= 2 * kUnits) break;
      if (unit < kUnits) {
        const int kg = unit / C, r0 = (unit % C) * 8;  // keys 4 kg .. +3, dims r0 .. +7
        const int c = 2 * (kg >> 2) + (kg & 1), piece = (kg >> 1) & 1;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
          const uint32_t lo = __builtin_amdgcn_perm(pf_word(reg[u][1], j >> 1), pf_word(reg[u][0], j >> 1), sel);
          const uint32_t hi = __builtin_amdgcn_perm(pf_word(reg[u][3], j >> 1), pf_word(reg[u][2], j >> 1), sel);
          *reinterpret_cast<uint2*>(v_buf[buf] + (r0 + j) * kVRow + pf_v_slot(r0 + j, c) * 16 + piece * 8) =
              make_uint2(lo, hi);
        }
      } else {
        const int x = unit - kUnits, c = x % C;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = x / C + i * (kPfBN / 4);
          *reinterpret_cast<uint4*>(k_buf[buf] + r * (D * 2) + pf_k_slot<D>(r, c) * 16) = reg[u][i];
        }
      }
    }
  };

  auto stage = [&](int t) {
    store_tile((t + 1) & 1);
    if (t + 2 < n_tiles) load_tile((t + 2) * kPfBN);  // in flight during the rest of tile t's math and tile t+1's QK
  };

  load_tile(0);
  store_tile(0);
  if (n_tiles > 1) load_tile(kPfBN);
  for (int t = 0; t < n_tiles; ++t) {
    const int t0 = t * kPfBN;
    // tile t's buffer is complete and every wave is done with tile t-1's
    // buffer, which takes tile t+1 (loaded during tile t-1's math)
    __syncthreads();
    // the next tile is stored under the first MFMAs (waves without queries in this tile store it alone)
    const bool stages = t + 1 < n_tiles;
    if (t0 > wq0 + 31) {  // wholly above the wave's diagonal
      if (stages) stage(t);
      continue;
    }
    const char* kl = k_buf[t & 1] + n * (D * 2);
    const char* vl = v_buf[t & 1] + n * kVRow;

    // S^T for 2 key blocks of 32: s[kb][i] holds key t0 + kb*32 + (i/4)*8 + half*4 + i%4
    pf_f32x16 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kb][i] = 0.f;
#pragma unroll
    for (int st = 0; st < KS; ++st)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const uint4 kf =
            *reinterpret_cast<const uint4*>(kl + kb * 32 * D * 2 + pf_k_slot<D>(n, 2 * st + half) * 16);
        s[kb] = mfma32x32x16<T>(kf, qf[st], s[kb]);
      }
    if (stages) stage(t);
    // causal and past-the-end mask (a tile wholly below the wave's diagonal
    // and inside the prompt needs none)
    if (t0 + kPfBN - 1 > wq0 || t0 + kPfBN > a.seq) {  // uniform over the wave
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = t0 + kb * 32 + (i >> 2) * 8 + half * 4 + (i & 3);
          if (key > query || key >= a.seq) s[kb][i] = -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kb][i]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if (__any(mx > m)) {
      const float moved = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f((m - (moved == -INFINITY ? 0.f : moved)) * a.scale_log2);
      m = moved;
      l *= alpha;
#pragma unroll
      for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[b][i] *= alpha;
    }
    const float ref = m == -INFINITY ? 0.f : m * a.scale_log2;
    // weights rounded to the input dtype, packed as P^T B operands
    uint4 pb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t w[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float e0 = s[j >> 1][(j & 1) * 8 + 2 * x], e1 = s[j >> 1][(j & 1) * 8 + 2 * x + 1];
        w[x] = pf_pack<T>(__builtin_amdgcn_exp2f(__builtin_fmaf(e0, a.scale_log2, -ref)),
                          __builtin_amdgcn_exp2f(__builtin_fmaf(e1, a.scale_log2, -ref)));
        l = pf_add_pair<T>(w[x], l);
      }
      pb[j] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    // O^T += V^T P^T: dim block b, 16-key step j
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int b = 0; b < DB; ++b) {
        const uint4 vf =
            *reinterpret_cast<const uint4*>(vl + b * 32 * kVRow + pf_v_slot(b * 32 + n, 2 * j + half) * 16);
        o[b] = mfma32x32x16<T>(vf, pb[j], o[b]);
      }
  }
  l += __shfl_xor(l, 32);
  if (query >= a.seq) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  char* op = a.out + ((int64_t)query * a.o_s + (int64_t)h * a.o_h) * T::bytes + half * 8;
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int x = 0; x < 4; ++x) {  // dims b*32 + x*8 + half*4 .. +3 of the lane's query
      const uint32_t w0 = pf_pack<T>(o[b][4 * x] * inv, o[b][4 * x + 1] * inv);
      const uint32_t w1 = pf_pack<T>(o[b][4 * x + 2] * inv, o[b][4 * x + 3] * inv);
      *reinterpret_cast<uint2*>(op + b * 64 + x * 16) = make_uint2(w0, w1);
    }
}

template <typename T, int D, int NW>
static void launch_prefill(const PrefillArgs& a, const LaunchEvents& ev, hipStream_t s) {
  const int64_t blocks = ((int64_t)a.seq + 32 * NW - 1) / (32 * NW) * a.q_heads;
  launch(prefill_attention_kernel<T, D, NW>, dim3((unsigned)blocks), dim3(NW * kWave), 0, s, ev.start, ev.stop, a);
}

// Eight waves share each staged tile (one workgroup fills a CU) once there are
// two such workgroups per CU to balance; below, four waves and up to two
// workgroups per CU. us with eight / four waves, bf16, heads x head_dim:
// 32768 tokens 32 x 128: 8597 / 9337; 4000 tokens 32 x 128: 159 / 169;
// 4096 tokens 16 x 128 (256 eight-wave workgroups): 131 / 122; 1999 tokens
// 28 x 128: 70 / 64; 1000 tokens 32 x 128: 37 / 32. Two waves lose
// everywhere (1999 tokens: 93).
template <typename T, int D>
static void launch_prefill(const PrefillArgs& a, const LaunchEvents& ev, hipStream_t s) {
  if (((int64_t)a.seq + 255) / 256 * a.q_heads >= 2 * kPfCUs)
    launch_prefill<T, D, 8>(a, ev, s);
  else
    launch_prefill<T, D, 4>(a, ev, s);
}

}  // namespace nhs

extern "C" int nhs_prefill_attention(const void* q, int64_t q_seq_stride, int64_t q_head_stride, const void* k,
                                     int64_t k_seq_stride, int64_t k_head_stride, const void* v,
                                     int64_t v_seq_stride, int64_t v_head_stride, int32_t dtype, int32_t seq,
                                     int32_t q_heads, int32_t kv_heads, int32_t head_dim, void* out,
                                     int64_t out_seq_stride, int64_t out_head_stride, void* stream) {
  using namespace nhs;
  const LaunchEvents ev = take_launch_events();
  const char* who = "nhs_prefill_attention";
  if (!q || !k || !v || !out) return fail(NHS_ERR_INVALID, "%s: null pointer", who);
  if (dtype != NHS_BF16 && dtype != NHS_F16) return fail(NHS_ERR_UNSUPPORTED, "%s: bf16 or fp16 only", who);
  if (head_dim != 64 && head_dim != 128) return fail(NHS_ERR_UNSUPPORTED, "%s: head_dim 64 or 128", who);
  if (seq < 1 || q_heads < 1 || kv_heads < 1 || q_heads % kv_heads)
    return fail(NHS_ERR_INVALID, "%s: invalid shape", who);
  const int64_t strides[] = {q_seq_stride, q_head_stride, k_seq_stride, k_head_stride, v_seq_stride,
                             v_head_stride, out_seq_stride, out_head_stride};
  for (int64_t st : strides)
    if (st % 8) return fail(NHS_ERR_INVALID, "%s: strides must be multiples of 8 elements", who);
  if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) % 16) != 0)
    return fail(NHS_ERR_INVALID, "%s: tensors must be 16-byte aligned", who);
  PrefillArgs a;
  a.q = static_cast<const char*>(q);
  a.k = static_cast<const char*>(k);
  a.v = static_cast<const char*>(v);
  a.q_s = q_seq_stride, a.q_h = q_head_stride;
  a.k_s = k_seq_stride, a.k_h = k_head_stride;
  a.v_s = v_seq_stride, a.v_h = v_head_stride;
  a.seq = seq;
  a.q_heads = q_heads;
  a.group = q_heads / kv_heads;
  a.scale_log2 = (float)(1.4426950408889634 / sqrt((double)head_dim));
  a.out = static_cast<char*>(out);
  a.o_s = out_seq_stride, a.o_h = out_head_stride;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == NHS_BF16) {
    if (head_dim == 128)
      launch_prefill<BF16, 128>(a, ev, s);
    else
      launch_prefill<BF16, 64>(a, ev, s);
  } else {
    if (head_dim == 128)
      launch_prefill<F16, 128>(a, ev, s);
    else
      launch_prefill<F16, 64>(a, ev, s);
  }
  return launch_status(who);
}
