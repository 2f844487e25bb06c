// Attention for few query rows per KV head: a token or a few against a long
// KV cache, grouped-query heads, and short or ragged sequences with a mask.
//
// The fused kernel (attention.hip) gives a (batch, query head) 128 query rows
// a workgroup and walks all keys in it: with one query row per head that is
// one workgroup per head, and every query head of a group reads its KV head
// again. Here the rows of all query heads of a KV head are packed (row r =
// query r / group of head r % group) into tiles of 16 or 32, the keys are
// dealt to the 4 waves of a workgroup, and, with a workspace, to several
// workgroups:
//
//  * A wave walks its own 32-key blocks alone, with no workgroup barrier: K
//    rows go straight from memory into MFMA fragments (S^T = K Q^T, a lane
//    holds 4 + 4 keys of one query row), V rows through the wave's own LDS
//    tile, from which the transposed reads take the very key order that the
//    S^T fragments have, so P goes from registers into O^T += V^T P. The
//    next block's K, V and mask are in flight during the current one.
//  * Online softmax in the log2 domain, the row sum over the rounded f16
//    probabilities. A wave moves its rows' reference to every new max, so
//    that the largest weight of a row is 1 and exact: letting it lag by up to
//    2^8, as the fused kernel does, ran 3 % faster and was up to 12 % further
//    from 64 bits than the kernels this one replaces.
//  * The waves' (max, sum, O) are merged through LDS, those of several
//    workgroups through f32 partials in the workspace, summed in split order
//    by the last to arrive. The result is 0 for a row that sees no key.
//
// Bound by the latency of a wave's few blocks when rows are few (one query of
// 32 heads over 8 KV heads, batch 4, 3001 keys, d 128: 13.3 us for 49 MB, 8
// splits; the fused kernel 44.0) and by each row tile reading K and V again
// when they are many, where the fused kernel takes over (abi.cpp, rows_us).
#include <type_traits>

#include "device_common.h"
#include "kernels_internal.h"

namespace ihp {

namespace {

constexpr int kRowsThreads = 256;
constexpr int kRowsWaves = kRowsThreads / 64;
constexpr int kBlockKeys = 32;
constexpr int kDeviceScope = 16;  // sc1 of a buffer instruction
constexpr float kNegInf = -__builtin_inff();
constexpr float kLog2e = 1.4426950408889634f;

typedef i32x4 __attribute__((aligned(2))) i32x4_u;
typedef i32x2 __attribute__((aligned(2))) i32x2_u;
typedef f16x4 __attribute__((aligned(2))) f16x4_u;
typedef f32x4 __attribute__((aligned(4))) f32x4_u;

// Chunk swizzle of a staged V row (key) of NCH 16-byte chunks: a transposed
// read takes 4 rows of one 32-byte window per 16-lane block, two blocks (rows
// 4 apart) at a time, and all of it must spread over the 64 banks.
template <int NCH>
__device__ __forceinline__ int v_swizzle(int k) {
  return NCH >= 16 ? (4 * (k & 3)) ^ (2 * ((k >> 2) & 1))
                   : (2 * ((k >> 1) & 1)) ^ (4 * ((k >> 2) & 1));
}

__device__ __forceinline__ float across_groups_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}
__device__ __forceinline__ float across_groups_sum(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}

}  // namespace

// DP: the head-dim bucket (64, 128 or 256, at least both head dims); RF:
// 16-row fragments a tile.
template <int DP, int RF, bool MASK, typename OutT>
__global__ __launch_bounds__(kRowsThreads, DP >= 256 ? 1 : 2) void
attention_rows_kernel(const f16 *__restrict__ Q, const f16 *__restrict__ K,
                      const f16 *__restrict__ V, OutT *__restrict__ O,
                      const f16 *__restrict__ Mask, AttentionGeneralLayout L,
                      int row_tiles, int blocks_per_split,
                      float *__restrict__ partials,
                      unsigned *__restrict__ counters) {
  constexpr int KS = DP / 32;           // head-dim steps of S
  constexpr int DB = DP / 16;           // 16-wide d blocks of O
  constexpr int NCH = DP / 8;           // 16-byte chunks of a V row
  constexpr int VROWS = 64 / NCH;       // V rows per load
  constexpr int VP = kBlockKeys / VROWS;
  constexpr int VBYTES = kBlockKeys * DP * 2;
  constexpr int OPITCH = DP + 4;        // floats, merge rows
  constexpr int MERGE = kRowsWaves * 16 * OPITCH * 4;
  constexpr int SMEM = kRowsWaves * VBYTES > MERGE ? kRowsWaves * VBYTES : MERGE;
  __shared__ __attribute__((aligned(1024))) char smem[SMEM];
  __shared__ float wave_m[kRowsWaves][RF * 16], wave_l[kRowsWaves][RF * 16];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, lg = lane >> 4;
  // One XCD's workgroups take consecutive tiles: a KV head's row tiles share
  // its L2.
  int tile, unused;
  xcd_tile_order((int)blockIdx.x, (int)gridDim.x, (int)gridDim.x, 1, 1, &tile,
                 &unused);
  const int kv_heads = L.heads / L.group;
  const int plane = tile / row_tiles;  // batch x KV head
  const int64_t b = plane / kv_heads;
  const int kvh = plane % kv_heads;
  const int rows = L.seq_q * L.group;
  const int r0 = (tile % row_tiles) * (RF * 16);
  const f16 *Kp = K + b * L.k[0] + kvh * L.k[1];
  const f16 *Vp = V + b * L.v[0] + kvh * L.v[1];

  // This lane's query rows (rows past the end repeat the last one).
  i32x4 qf[RF][KS];
  int limit[RF];  // keys the row sees
  const f16 *mrow[RF];
#pragma unroll
  for (int f = 0; f < RF; ++f) {
    int r = r0 + f * 16 + l15;
    r = r < rows ? r : rows - 1;
    const int i = r / L.group, h = kvh * L.group + r % L.group;
    limit[f] = L.causal && i + 1 < L.seq_kv ? i + 1 : L.seq_kv;
    const f16 *qp = Q + b * L.q[0] + h * L.q[1] + i * L.q[2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int c = 32 * ks + 8 * lg;
      qf[f][ks] = i32x4{0, 0, 0, 0};
      if (c < L.dqk)
        qf[f][ks] = *(const i32x4_u *)(qp + c);
    }
    mrow[f] = MASK ? Mask + b * L.mask[0] + h * L.mask[1] + i * L.mask[2]
                   : nullptr;
  }
  // Every row of the tile sees the keys below all_see; none those from
  // some_see on.
  const int i_first = r0 / L.group;
  const int r_last = r0 + RF * 16 < rows ? r0 + RF * 16 - 1 : rows - 1;
  const int i_last = r_last / L.group;
  const int all_see =
      L.causal && i_first + 1 < L.seq_kv ? i_first + 1 : L.seq_kv;
  const int some_see =
      L.causal && i_last + 1 < L.seq_kv ? i_last + 1 : L.seq_kv;

  const int blocks = (some_see + kBlockKeys - 1) / kBlockKeys;
  const int c_begin = (int)blockIdx.y * blocks_per_split;
  const int c_end =
      blocks - c_begin < blocks_per_split ? blocks : c_begin + blocks_per_split;

  // Chunks of a row past the head dim: K's are zeroed before use, V's reach
  // columns that are not stored; both are loaded from inside the row.
  const bool pad_k = L.dqk != DP;
  int koff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int c = 32 * ks + 8 * lg;
    koff[ks] = c < L.dqk ? c : L.dqk - 8;
  }
  const int vrow = lane / NCH, vch = lane % NCH;
  const int voff = 8 * vch < L.dv ? 8 * vch : L.dv - 8;

  i32x4 kf[2][KS], vf[VP];
  i32x2 mf[RF][2];
  int mshift[2];
  auto load_k = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      int key = c * kBlockKeys + f * 16 + l15;
      key = key < L.seq_kv ? key : L.seq_kv - 1;
      const f16 *p = Kp + (int64_t)key * L.k[2];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kf[f][ks] = *(const i32x4_u *)(p + koff[ks]);
    }
    if constexpr (MASK) {
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        // 4 keys from the row's last 4 on: shifted down before use
        const int key = c * kBlockKeys + f * 16 + 4 * lg;
        const int at = key + 4 <= L.seq_kv ? key : L.seq_kv - 4;
        mshift[f] = key - at < 4 ? 16 * (key - at) : 0;
#pragma unroll
        for (int r = 0; r < RF; ++r)
          mf[r][f] = *(const i32x2_u *)(mrow[r] + at);
      }
    }
  };
  auto load_v = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < VP; ++p) {
      int key = c * kBlockKeys + p * VROWS + vrow;
      key = key < L.seq_kv ? key : L.seq_kv - 1;
      vf[p] = *(const i32x4_u *)(Vp + (int64_t)key * L.v[2] + voff);
    }
  };

  f32x4 o[RF][DB];
  float m_ref[RF], l_sum[RF];
#pragma unroll
  for (int f = 0; f < RF; ++f) {
    m_ref[f] = kNegInf;
    l_sum[f] = 0.0f;
#pragma unroll
    for (int d = 0; d < DB; ++d)
      o[f][d] = f32x4{0, 0, 0, 0};
  }
  char *vs = smem + wave * VBYTES;
  const float scale = L.scale * kLog2e;
  const f16x2 ones = {(f16)1.0f, (f16)1.0f};

  int c = c_begin + wave;
  if (c < c_end) {
    load_k(c);
    load_v(c);
  }
  for (; c < c_end; c += kRowsWaves) {
    const bool more = c + kRowsWaves < c_end;
    if (pad_k) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        if (32 * ks + 8 * lg >= L.dqk)
          kf[0][ks] = kf[1][ks] = i32x4{0, 0, 0, 0};
    }
    f32x4 s[RF][2];
#pragma unroll
    for (int r = 0; r < RF; ++r)
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        s[r][f] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          s[r][f] = Mfma16<f16>::mma(kf[f][ks], qf[r][ks], s[r][f]);
      }
    float sv[RF][8];
#pragma unroll
    for (int r = 0; r < RF; ++r)
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        f16x4 mv = {0, 0, 0, 0};
        if constexpr (MASK) {
          uint64_t w = __builtin_bit_cast(uint64_t, mf[r][f]);
          w >>= mshift[f];
          mv = __builtin_bit_cast(f16x4, w);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // With a mask in natural units: a mask of the lowest f16 leaves
          // as much of the score as the f32 sum of the two holds.
          sv[r][4 * f + e] =
              MASK ? __builtin_fmaf(s[r][f][e], L.scale, (float)mv[e])
                   : s[r][f][e] * scale;
        }
      }
    if ((c + 1) * kBlockKeys > all_see) {
#pragma unroll
      for (int r = 0; r < RF; ++r)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = c * kBlockKeys + 16 * (e >> 2) + 4 * lg + (e & 3);
          sv[r][e] = key < limit[r] ? sv[r][e] : kNegInf;
        }
    }
    if (more)
      load_k(c + kRowsWaves);

    float top[RF];
    bool move = false;
#pragma unroll
    for (int r = 0; r < RF; ++r) {
      float t = sv[r][0];
#pragma unroll
      for (int e = 1; e < 8; ++e)
        t = fmaxf(t, sv[r][e]);
      if constexpr (MASK)
        t *= kLog2e;
      top[r] = t;
      move |= t > m_ref[r];
    }
    if (__any(move)) {
#pragma unroll
      for (int r = 0; r < RF; ++r) {
        const float t = fmaxf(m_ref[r], across_groups_max(top[r]));
        const float keep =
            t == kNegInf ? 1.0f : __builtin_amdgcn_exp2f(m_ref[r] - t);
        m_ref[r] = t;
        l_sum[r] *= keep;
#pragma unroll
        for (int d = 0; d < DB; ++d)
          o[r][d] *= keep;
      }
    }
    i32x4 pf[RF];
#pragma unroll
    for (int r = 0; r < RF; ++r) {
      const float ref = m_ref[r] == kNegInf ? 0.0f : m_ref[r];
      auto weight = [&](float x) {
        return (f16)__builtin_amdgcn_exp2f(
            MASK ? __builtin_fmaf(x, kLog2e, -ref) : x - ref);
      };
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f16x2 p2 = {weight(sv[r][2 * e]), weight(sv[r][2 * e + 1])};
        l_sum[r] = __builtin_amdgcn_fdot2(p2, ones, l_sum[r], false);
        pf[r][e] = __builtin_bit_cast(int, p2);
      }
    }

    // V through this wave's LDS tile; keys past the sequence are zeros.
#pragma unroll
    for (int p = 0; p < VP; ++p) {
      const int k = p * VROWS + vrow;
      if (c * kBlockKeys + k >= L.seq_kv)
        vf[p] = i32x4{0, 0, 0, 0};
      *(i32x4 *)(vs + k * (DP * 2) + ((vch ^ v_swizzle<NCH>(k)) << 4)) = vf[p];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (more)
      load_v(c + kRowsWaves);
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      typedef short s16x4 __attribute__((ext_vector_type(4)));
      const int k = 4 * lg + (l15 >> 2);
      const int byte = 2 * (16 * d + 4 * (l15 & 3));
      const IHP_LDS char *p =
          (const IHP_LDS char *)vs + k * (DP * 2) +
          (((byte >> 4) ^ v_swizzle<NCH>(k)) << 4) + (byte & 15);
      const i32x2 lo = __builtin_bit_cast(
          i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((IHP_LDS s16x4 *)p));
      const i32x2 hi = __builtin_bit_cast(
          i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                     (IHP_LDS s16x4 *)(p + 16 * (DP * 2))));
      const i32x4 v = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
      for (int r = 0; r < RF; ++r)
        o[r][d] = Mfma16<f16>::mma(v, pf[r], o[r][d]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }

  // Merge the waves: a common max per row, O scaled to it.
#pragma unroll
  for (int r = 0; r < RF; ++r) {
    const float l = across_groups_sum(l_sum[r]);
    if (lg == 0) {
      wave_m[wave][r * 16 + l15] = m_ref[r];
      wave_l[wave][r * 16 + l15] = l;
    }
  }
  __syncthreads();
  const int splits = (int)gridDim.y;
  // Thread (q, dq) of the merge: row q of a fragment, DP / 16 columns from dq.
  constexpr int CPT = DP / 16;
  const int q = tid >> 4, dq = (tid & 15) * CPT;
  constexpr int PROW = DP + 4;  // partial row: O, then max and sum
  float *part = partials + (int64_t)tile * splits * (RF * 16 * PROW);
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc(part, 0, -1, 0x00027000);
  auto store_row = [&](int row, const float *acc, float inv) {
    const int i = row / L.group, h = kvh * L.group + row % L.group;
    OutT *dst = O + b * L.o[0] + h * L.o[1] + i * L.o[2] + dq;
#pragma unroll
    for (int e = 0; e < CPT; e += 4) {
      if (dq + e >= L.dv)  // dv is a multiple of 8
        break;
      if constexpr (std::is_same<OutT, float>::value)
        *(f32x4_u *)(dst + e) = f32x4{acc[e] * inv, acc[e + 1] * inv,
                                      acc[e + 2] * inv, acc[e + 3] * inv};
      else
        *(f16x4_u *)(dst + e) =
            f16x4{(f16)(acc[e] * inv), (f16)(acc[e + 1] * inv),
                  (f16)(acc[e + 2] * inv), (f16)(acc[e + 3] * inv)};
    }
  };
#pragma unroll
  for (int r = 0; r < RF; ++r) {
    float *om = (float *)smem;
    {
      float top = kNegInf;
#pragma unroll
      for (int w = 0; w < kRowsWaves; ++w)
        top = fmaxf(top, wave_m[w][r * 16 + l15]);
      const float f =
          m_ref[r] == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(m_ref[r] - top);
#pragma unroll
      for (int d = 0; d < DB; ++d)
        *(f32x4 *)(om + (wave * 16 + l15) * OPITCH + 16 * d + 4 * lg) =
            o[r][d] * f;
    }
    __syncthreads();
    float top = kNegInf, sum = 0.0f;
#pragma unroll
    for (int w = 0; w < kRowsWaves; ++w)
      top = fmaxf(top, wave_m[w][r * 16 + q]);
#pragma unroll
    for (int w = 0; w < kRowsWaves; ++w)
      sum += wave_m[w][r * 16 + q] == kNegInf
                 ? 0.0f
                 : wave_l[w][r * 16 + q] *
                       __builtin_amdgcn_exp2f(wave_m[w][r * 16 + q] - top);
    float acc[CPT];
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
      acc[e] = 0.0f;
#pragma unroll
      for (int w = 0; w < kRowsWaves; ++w)
        acc[e] += om[(w * 16 + q) * OPITCH + dq + e];
    }
    __syncthreads();  // before the next fragment's rows
    const int row = r0 + r * 16 + q;
    if (row >= rows)
      continue;
    if (splits == 1) {
      store_row(row, acc, sum > 0.0f ? 1.0f / sum : 0.0f);
    } else {
      const int at = (((int)blockIdx.y * RF + r) * 16 + q) * PROW;
#pragma unroll
      for (int e = 0; e < CPT; e += 4)
        __builtin_amdgcn_raw_buffer_store_b128(
            __builtin_bit_cast(i32x4,
                               f32x4{acc[e], acc[e + 1], acc[e + 2],
                                     acc[e + 3]}),
            rs, (at + dq + e) * 4, 0, kDeviceScope);
      if (dq == 0)
        __builtin_amdgcn_raw_buffer_store_b128(
            __builtin_bit_cast(i32x4, f32x4{top, sum, 0.0f, 0.0f}), rs,
            (at + DP) * 4, 0, kDeviceScope);
    }
  }
  if (splits == 1)
    return;
  unsigned *last = (unsigned *)smem;
  wait_vmcnt<0>();  // published before it is counted
  __syncthreads();
  if (tid == 0) {
    const unsigned prev =
        __hip_atomic_fetch_add(&counters[tile * kCounterStride], 1u,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *last = prev == (unsigned)splits - 1;
  }
  __syncthreads();
  if (!*last)
    return;
#pragma unroll
  for (int r = 0; r < RF; ++r) {
    const int row = r0 + r * 16 + q;
    if (row >= rows)
      continue;
    // 4 splits' loads in flight; a split past the last repeats it with
    // weight 0
    float top = kNegInf, sum = 0.0f, acc[CPT];
#pragma unroll
    for (int e = 0; e < CPT; ++e)
      acc[e] = 0.0f;
    for (int s0 = 0; s0 < splits; s0 += 4) {
      f32x4 ml[4], v[4][CPT / 4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int s = s0 + u < splits ? s0 + u : splits - 1;
        const int at = ((s * RF + r) * 16 + q) * PROW;
        ml[u] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       rs, (at + DP) * 4, 0, kDeviceScope));
#pragma unroll
        for (int e = 0; e < CPT; e += 4)
          v[u][e / 4] = __builtin_bit_cast(
              f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                         rs, (at + dq + e) * 4, 0, kDeviceScope));
      }
      float t = top;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        t = fmaxf(t, ml[u][0]);
      const float keep =
          top == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(top - t);
      top = t;
      sum *= keep;
#pragma unroll
      for (int e = 0; e < CPT; ++e)
        acc[e] *= keep;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float f = s0 + u < splits && ml[u][0] != kNegInf
                            ? __builtin_amdgcn_exp2f(ml[u][0] - t)
                            : 0.0f;
        sum += f * ml[u][1];
#pragma unroll
        for (int e = 0; e < CPT; ++e)
          acc[e] += f * v[u][e / 4][e & 3];
      }
    }
    store_row(row, acc, sum > 0.0f ? 1.0f / sum : 0.0f);
  }
  if (tid == 0)  // re-arm for the next call on this workspace
    __hip_atomic_store(&counters[tile * kCounterStride], 0u, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// ----------------------------------------------------------------------------
// Host side.
// ----------------------------------------------------------------------------

namespace {

struct RowsKernel {
  const char *name;
  int dp, rf, mask, out_f32;
  const void *fn;
};
#define IHP_ROWS(DP, RF)                                                       \
  {"attention_rows_d" #DP "_r" #RF, DP, RF, 0, 0,                              \
   (const void *)&attention_rows_kernel<DP, RF, false, f16>},                  \
      {"attention_rows_d" #DP "_r" #RF "_f32", DP, RF, 0, 1,                   \
       (const void *)&attention_rows_kernel<DP, RF, false, float>},            \
      {"attention_rows_d" #DP "_r" #RF "_mask", DP, RF, 1, 0,                  \
       (const void *)&attention_rows_kernel<DP, RF, true, f16>},               \
      {"attention_rows_d" #DP "_r" #RF "_mask_f32", DP, RF, 1, 1,              \
       (const void *)&attention_rows_kernel<DP, RF, true, float>}
const RowsKernel kRowsKernels[] = {IHP_ROWS(64, 1), IHP_ROWS(64, 2),
                                   IHP_ROWS(128, 1), IHP_ROWS(128, 2),
                                   IHP_ROWS(256, 1)};
constexpr int kRowsKernelCount = sizeof(kRowsKernels) / sizeof(kRowsKernels[0]);

}  // namespace

AttentionRowsPlan plan_attention_rows(int64_t batch, int64_t kv_heads,
                                      int64_t group, int64_t seq_q,
                                      int64_t seq_kv, int64_t head_dim,
                                      int64_t head_dim_v,
                                      size_t workspace_limit) {
  AttentionRowsPlan p;
  const int64_t rows = seq_q * group;
  const int64_t d = head_dim > head_dim_v ? head_dim : head_dim_v;
  p.dp = d <= 64 ? 64 : d <= 128 ? 128 : 256;
  p.rf = rows > 16 && p.dp < 256 ? 2 : 1;
  p.row_tiles = (rows + 16 * p.rf - 1) / (16 * p.rf);
  p.tiles = p.row_tiles * kv_heads * batch;
  const int64_t blocks = (seq_kv + kBlockKeys - 1) / kBlockKeys;
  int64_t splits = kRowsTargetWgs / p.tiles;
  if (splits > blocks / kRowsSplitBlocks)
    splits = blocks / kRowsSplitBlocks;
  if (splits > kRowsMaxSplits)
    splits = kRowsMaxSplits;
  const int64_t split_bytes = p.tiles * 16 * p.rf * (p.dp + 4) * 4;
  if (p.tiles > kMaxWorkspaceCounters ||
      workspace_limit < kWorkspaceCounterBytes + 2 * (size_t)split_bytes)
    splits = 1;
  else if (kWorkspaceCounterBytes + (uint64_t)(splits * split_bytes) >
           workspace_limit)
    splits = (int64_t)(workspace_limit - kWorkspaceCounterBytes) / split_bytes;
  if (splits < 1)
    splits = 1;
  p.blocks_per_split = (blocks + splits - 1) / splits;
  p.splits = (blocks + p.blocks_per_split - 1) / p.blocks_per_split;
  if (p.splits < 1)
    p.splits = 1;
  p.workspace = p.splits > 1 ? (int64_t)kWorkspaceCounterBytes +
                                   p.splits * split_bytes
                             : 0;
  return p;
}

hipError_t launch_attention_rows(const void *q, const void *k, const void *v,
                                 void *o, const void *mask,
                                 const AttentionGeneralLayout &layout,
                                 const AttentionRowsPlan &p, int out_f32,
                                 void *workspace, void *stream) {
  const void *kernel = nullptr;
  for (const RowsKernel &c : kRowsKernels)
    if (c.dp == p.dp && c.rf == p.rf && c.mask == (mask != nullptr) &&
        c.out_f32 == out_f32)
      kernel = c.fn;
  if (!kernel || p.tiles >= ((int64_t)1 << 31))
    return hipErrorInvalidValue;
  AttentionGeneralLayout l = layout;
  int row_tiles = (int)p.row_tiles, per = (int)p.blocks_per_split;
  unsigned *counters = (unsigned *)workspace;
  float *partials = (float *)((char *)workspace + kWorkspaceCounterBytes);
  void *args[] = {&q, &k, &v, &o, &mask, &l, &row_tiles, &per, &partials,
                  &counters};
  return hipLaunchKernel(kernel, dim3((unsigned)p.tiles, (unsigned)p.splits),
                         dim3(kRowsThreads), args, 0, (hipStream_t)stream);
}

const KernelEntry *attention_rows_kernels(int *count) {
  static KernelEntry all[kRowsKernelCount];
  static const bool filled = [] {
    for (int i = 0; i < kRowsKernelCount; ++i)
      all[i] = {kRowsKernels[i].name, kRowsKernels[i].fn, kRowsThreads,
                kExportAttention};
    return true;
  }();
  (void)filled;
  *count = kRowsKernelCount;
  return all;
}

}  // namespace ihp
