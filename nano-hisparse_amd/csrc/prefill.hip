// Causal GQA self-attention for prefill (flash-attention forward, MFMA).
//
// out[s, h] = softmax_{t <= s}(q[s, h] . k[t, h/g] * D^-1/2) . v[t, h/g] for
// one prompt of `seq` tokens, bf16 or fp16 in, fp32 accumulation. A
// workgroup of 8 waves takes 256 queries of one query head (32 per wave) and
// walks the key tiles of 64 up to the diagonal with an online softmax; or
// (KSPLIT 2, where that leaves the chip idle) 128 queries, the two halves of
// the workgroup taking the even and the odd tiles, whose sums meet in LDS.
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
// in the order (l/32)*4 + 0..3, 8 + (l/32)*4 + 0..3, and the transposing LDS
// read (ds_read_b64_tr_b16: four keys of one dim per lane from row-major V)
// fetches the A operand in that order. The rescaling by a query's max stays
// in its lane.
//
// Why 32 queries per wave and 32x32 tiles: a wave reads every K and V byte
// of the tile from LDS once per MFMA operand, so the LDS bytes per flop fall
// with the queries a wave holds. At 16 per wave (16x16 tiles) the LDS reads
// took twice the matrix cores' time; at 32 they take as long as it does, and
// the wave still fits 256 registers, so two waves share a SIMD and one's
// softmax runs beside the other's MFMAs. Tiles go from global memory straight
// to LDS; the 16-byte chunks of their rows are permuted by an XOR of the row
// (the lanes of a load fetch the chunks in that order), so that the rows of a
// read meet distinct banks.
//
// The weights are rounded to the input dtype for the P.V product and the
// denominator sums the same rounded weights, so each output is an exact
// convex combination of V rows. A tile that moves no query's max rescales
// nothing. (Moving the max only once a score exceeds it by 2^8 would skip
// more, 3% of the time at 32K tokens, but the largest weight would no longer
// be exactly 1: the error against float64 grew by 3%.)
//
// Measured (MI355X, bf16, 32/8 heads of 128): 32768 tokens 7.8-8.3 ms, 1060
// to 1130 TFLOP/s causal (22.37 ms with 16 queries per wave and 16x16 tiles, 8.86 with
// tiles staged through registers and V transposed by the stores; a large
// hipBLASLt product reaches 1342); 4000 tokens 146 us (605, 157); 1999 tokens
// of 28/4 heads 46 us (159, 63); 333 tokens 11.7 us (19.7, 14.9).
#include <math.h>

#include "nhs_common.h"

namespace nhs {

constexpr int kPfBN = 64;            // keys per tile
constexpr int kPfWaves = 8, kPfThreads = kPfWaves * kWave;
// Workgroups of 256 queries from which each takes every tile. us with one /
// two shares (bf16, heads x head_dim): 4096 tokens 16 x 128 (256 of them) 116
// / 88, 6000 tokens (384) 181 / 186, 8192 tokens (512) 285 / 312; 4096 tokens
// 32 x 64 (512) 102 / 90, 16384 tokens 16 x 64 (1024) 584 / 606.
constexpr int pf_whole(int head_dim) { return head_dim == 128 ? 384 : 768; }

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

// LDS slot of 16-byte chunk c of K row r: any 16 consecutive rows at one chunk fall on distinct banks
template <int D>
__device__ __forceinline__ int pf_k_slot(int r, int c) {
  return D == 128 ? c ^ (r & 15) : c ^ ((r >> 1) & 7);
}
// and of V row (key) r: the 4 rows of a transposing read fall on distinct banks
template <int D>
__device__ __forceinline__ int pf_v_slot(int r, int c) {
  return D == 128 ? c ^ (4 * (r & 3)) : c ^ (4 * ((r >> 1) & 1));
}

constexpr int kPfVmcnt0 = 0x0f70;  // s_waitcnt vmcnt(0), the other counters left alone

// 16 bytes per lane from global memory to LDS at `dst` (uniform over the wave) + 16 * lane
__device__ __forceinline__ void pf_load_lds(const char* src, char* dst) {
  __builtin_amdgcn_global_load_lds((const NHS_GLOBAL void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

typedef short pf_i16x4 __attribute__((ext_vector_type(4)));

// Transposing read: of each 16 lanes, lanes 4r .. 4r+3 name 16 elements of row r; lane i receives column i of the four
// rows.
__device__ __forceinline__ uint2 pf_read_tr(const char* p) {
  return __builtin_bit_cast(
      uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) pf_i16x4*)const_cast<char*>(p)));
}

template <typename T, int D, int KSPLIT>
__global__ __launch_bounds__(kPfThreads) void prefill_attention_kernel(PrefillArgs a) {
  constexpr int QW = kPfWaves / KSPLIT;  // waves of different queries
  constexpr int BM = 32 * QW;            // queries per workgroup
  constexpr int KS = D / 16;           // 16-wide k steps of Q.K
  constexpr int DB = D / 32;           // 32-wide dim blocks of the output
  constexpr int C = D / 8;             // 16-byte chunks of a K or V row
  // Tiles go straight to LDS (global_load_lds, 1 KB per wave and instruction: kRows rows). Two buffers of their own
  // names, used by alternate rounds: the compiler then knows that reads of one need not wait for loads into the other.
  constexpr int kRows = 1024 / (D * 2);
  constexpr int kInstr = kPfBN / kRows;             // instructions per tile
  constexpr int kMine = kInstr * KSPLIT / kPfWaves;  // of a wave, per round, for K and for V each
  constexpr int kTile = kPfBN * D * 2;              // bytes
  __shared__ __attribute__((aligned(16))) char k0[KSPLIT * kTile], k1[KSPLIT * kTile];
  __shared__ __attribute__((aligned(16))) char v0[KSPLIT * kTile], v1[KSPLIT * kTile];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wave_id % QW, share = wave_id / QW;  // the wave's queries, its tile of each round
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
  const int n_rounds = last_key / (kPfBN * KSPLIT) + 1;
  const char* kbase = a.k + (int64_t)kvh * a.k_h * T::bytes;
  const char* vbase = a.v + (int64_t)kvh * a.v_h * T::bytes;
  // this lane's part of load i: row `row` of its tile (below), chunk of the row, permuted so that the LDS slots come
  // out in lane order
  const int lrow = lane / C;
  const int k_chunk = pf_k_slot<D>(wave_id * kRows + lrow, lane % C), v_chunk = pf_v_slot<D>(lrow, lane % C);
  constexpr int kRound = kPfBN * KSPLIT;
  const int64_t k_stride = a.k_s * T::bytes, v_stride = a.v_s * T::bytes;
  const char* kp[kMine];
  const char* vp[kMine];
#pragma unroll
  for (int i = 0; i < kMine; ++i) {
    const int row = (i * kPfWaves + wave_id) * kRows + lrow;  // of the round (its tiles one after another)
    kp[i] = kbase + k_chunk * 16 + row * k_stride;
    vp[i] = vbase + v_chunk * 16 + row * v_stride;
  }
  auto load_round = [&](int t, char* kb, char* vb) {
    const bool whole = (t + 1) * kRound <= a.seq;
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
      const int dst = (i * kPfWaves + wave_id) * 1024;
      const char* ks = kp[i];
      const char* vs = vp[i];
      if (!whole) {  // rows past the end re-read the last key (masked below)
        const int row = min(t * kRound + (i * kPfWaves + wave_id) * kRows + lrow, a.seq - 1);
        ks = kbase + k_chunk * 16 + row * k_stride;
        vs = vbase + v_chunk * 16 + row * v_stride;
      }
      pf_load_lds(ks, kb + dst);
      pf_load_lds(vs, vb + dst);
      kp[i] += kRound * k_stride;
      vp[i] += kRound * v_stride;
    }
  };
  // addresses within a tile: K row n at k step st, V^T's two 4-key pieces of dim block b
  const int k_row = n * (D * 2);
  const int j = (lane & 15) >> 2;
  int v_at[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
    v_at[b] = (4 * half + j) * (D * 2) + pf_v_slot<D>(j, b * 4 + ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1)) * 16 + (lane & 1) * 8;

  auto round = [&](int t, char* kb, char* vb, char* kb_next, char* vb_next) {
    const int t0 = t * kRound + share * kPfBN;
    // this wave's loads of round t are in; after the barrier every wave's are, and every wave is done with the other
    // buffers, which take round t+1
    __builtin_amdgcn_s_waitcnt(kPfVmcnt0);
    __syncthreads();
    if (t + 1 < n_rounds) load_round(t + 1, kb_next, vb_next);
    if (t0 > min(wq0 + 31, last_key)) return;  // wholly above the wave's diagonal or past the last key
    const char* kl = kb + share * kTile + k_row;
    const char* vl = vb + share * kTile;

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
    if constexpr (D == 128) {  // keep eight K reads ahead of the MFMAs (two by default: 3% slower)
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x8, 8, 0);
    }
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
    // weights rounded to the input dtype, packed as P^T B operands; the
    // denominator takes each tile's sum (in one chain over all tiles its error
    // at 32768 keys is 6.6e-7 of it and not 3.1e-7)
    uint4 pb[4];
    float tile_sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t w[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float e0 = s[j >> 1][(j & 1) * 8 + 2 * x], e1 = s[j >> 1][(j & 1) * 8 + 2 * x + 1];
        w[x] = pf_pack<T>(__builtin_amdgcn_exp2f(__builtin_fmaf(e0, a.scale_log2, -ref)),
                          __builtin_amdgcn_exp2f(__builtin_fmaf(e1, a.scale_log2, -ref)));
        tile_sum = pf_add_pair<T>(w[x], tile_sum);
      }
      pb[j] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    l += tile_sum;
    // O^T += V^T P^T: dim block b, 16-key step j
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int b = 0; b < DB; ++b) {
        const uint2 lo = pf_read_tr(vl + v_at[b] + (16 * j) * (D * 2));
        const uint2 hi = pf_read_tr(vl + v_at[b] + (16 * j + 8) * (D * 2));
        const uint4 vf = make_uint4(lo.x, lo.y, hi.x, hi.y);
        o[b] = mfma32x32x16<T>(vf, pb[j], o[b]);
      }
  };
  load_round(0, k0, v0);
  for (int t = 0; t < n_rounds; t += 2) {
    round(t, k0, v0, k1, v1);
    if (t + 1 < n_rounds) round(t + 1, k1, v1, k0, v0);
  }
  l += __shfl_xor(l, 32);
  if constexpr (KSPLIT == 2) {
    // the waves of the second share hand their sums over through the tile buffers (registers by lane: each lane's
    // partner holds the same query and dims)
    float* part = reinterpret_cast<float*>(wave < QW / 2 ? k0 : k1) + wave % (QW / 2) * (DB * 16 * kWave) + lane;
    float* stat = reinterpret_cast<float*>(v0) + wave * 2 * kWave + lane;
    __syncthreads();
    if (share) {
#pragma unroll
      for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) part[(b * 16 + i) * kWave] = o[b][i];
      stat[0] = m;
      stat[kWave] = l;
    }
    __syncthreads();
    if (share) return;
    const float m2 = stat[0], l2 = stat[kWave];
    const float both = fmaxf(m, m2), ref = both == -INFINITY ? 0.f : both;
    const float f1 = __builtin_amdgcn_exp2f((m - ref) * a.scale_log2);
    const float f2 = __builtin_amdgcn_exp2f((m2 - ref) * a.scale_log2);
    l = l * f1 + l2 * f2;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[b][i] = o[b][i] * f1 + part[(b * 16 + i) * kWave] * f2;
  }
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

template <typename T, int D, int KSPLIT>
static void launch_prefill(const PrefillArgs& a, const LaunchEvents& ev, hipStream_t s) {
  constexpr int BM = 32 * kPfWaves / KSPLIT;
  const int64_t blocks = ((int64_t)a.seq + BM - 1) / BM * a.q_heads;
  launch(prefill_attention_kernel<T, D, KSPLIT>, dim3((unsigned)blocks), dim3(kPfThreads), 0, s, ev.start, ev.stop, a);
}

template <typename T, int D>
static void launch_prefill(const PrefillArgs& a, const LaunchEvents& ev, hipStream_t s) {
  if (((int64_t)a.seq + 255) / 256 * a.q_heads >= pf_whole(D))
    launch_prefill<T, D, 1>(a, ev, s);
  else
    launch_prefill<T, D, 2>(a, ev, s);
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
