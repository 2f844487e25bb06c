// gfx950 matmul kernels for shapes and operands the macro-tile path does not
// take: any extents, strides, alignment and layout of A and B, f16, int8 and
// int8 weights under f16 activations (W8A16).
//
// The macro-tile kernel (gemm.hip) copies HBM straight into LDS, which needs
// 16-byte aligned rows and exact tiles. Here each lane loads 16 bytes at any
// element-aligned address into registers, one K stage ahead, and writes them
// to LDS in the same swizzled layouts, so that the MFMA side is the same:
// K-contiguous operands are read with ds_read_b128, row-major B and
// transposed A with the transposed LDS reads. int8 weights are widened to
// f16 (exactly) on their way into LDS, once per element, in either layout.
//
//  * A chunk that runs past the end of its row is loaded from the row's last
//    16 bytes and shifted down, which leaves zeros past the end: no element
//    loads, no branch in whole stages, nothing read outside the operand.
//    Rows past M (N) repeat the last row; their results are not stored.
//  * Two LDS slots and one barrier a stage: the registers of stage t+1 go to
//    the other slot while stage t is multiplied, then the loads of stage t+2
//    are issued.
//  * MFMAs are issued with their operands swapped (C^T fragments), so a lane
//    holds 4 consecutive columns of one row: bias, multiplier, C and the
//    result move 4 columns at a time, at any alignment.
//  * With a workspace K is split over grid y: partial tiles are published in
//    fragment order (16 bytes a lane, no edges) with device-scope stores and
//    summed in split order by the last workgroup to arrive, as the macro-tile
//    kernel does.
#include <type_traits>
#include <vector>

#include "device_common.h"
#include "kernels_internal.h"

namespace ihp {

namespace {

constexpr int kStageBytes = 128;  // K bytes of a staged K-contiguous row

// 16 bytes at any address (the compiler emits one global_load_dwordx4: gfx950
// loads vectors at any alignment).
typedef i32x4 __attribute__((aligned(1))) i32x4_u;
typedef f16x4 __attribute__((aligned(2))) f16x4_u;
typedef f32x4 __attribute__((aligned(4))) f32x4_u;
typedef i32x4 __attribute__((aligned(4))) i32x4_u4;

// v >> 8 * bytes over the 16 bytes, zeros shifted in; bytes in [0, 16].
__device__ __forceinline__ i32x4 shift_down(i32x4 v, int bytes) {
  if (bytes & 16)
    v = i32x4{0, 0, 0, 0};
  if (bytes & 8)
    v = i32x4{v[2], v[3], 0, 0};
  if (bytes & 4)
    v = i32x4{v[1], v[2], v[3], 0};
  const unsigned r = bytes & 3;
  const unsigned a = v[0], b = v[1], c = v[2], d = v[3];
  return i32x4{(int)__builtin_amdgcn_alignbyte(b, a, r),
               (int)__builtin_amdgcn_alignbyte(c, b, r),
               (int)__builtin_amdgcn_alignbyte(d, c, r),
               (int)__builtin_amdgcn_alignbyte(0u, d, r)};
}

// The `E` elements from position `pos` of a row of `extent` < E elements.
template <typename T, int E>
__device__ __forceinline__ i32x4 load_short(const T *row, int64_t pos,
                                            int64_t extent) {
  T v[E];
#pragma unroll
  for (int e = 0; e < E; ++e)
    v[e] = pos + e < extent ? row[pos + e] : (T)0;
  i32x4 out;
  __builtin_memcpy(&out, v, 16);
  return out;
}

// Swizzle of a staged row-major (N-contiguous) row k of NCH 16-byte chunks:
// the transposed reads of two 16-lane blocks (4 f16 or 8 int8 rows each at
// one 32- or 16-byte window, blocks 8 or 16 rows apart) must cover all 64
// banks. Rows narrower than the 256-byte bank line differ in their place on
// it already; the rest of the row index is XORed into the chunk index.
template <int ELEM_BYTES, int NCH>
__device__ __forceinline__ int row_swizzle(int k) {
  if constexpr (ELEM_BYTES == 2)
    return NCH >= 16 ? (4 * (k & 3)) ^ (2 * ((k >> 3) & 1))
                     : (2 * ((k >> 1) & 1)) ^ (4 * ((k >> 3) & 1));
  else
    return (NCH >= 16 ? 2 * (k & 7)
                      : NCH == 8 ? 2 * ((k >> 1) & 3) : 2 * ((k >> 2) & 1)) ^
           ((k >> 4) & 1);
}

// One operand's way from memory to LDS: TS its stored type, TM the MFMA
// type, KC whether its rows run along K (else along M / N), R its tile
// extent along M / N, DEPTH the stages its registers hold. A load's address
// is a wave-uniform base, one scalar add a stage, and a 32-bit lane offset.
// ANY takes what that does not: 64-bit lane addresses for pitches whose
// offsets pass 32 bits, and rows shorter than one load, element by element.
template <typename TS, typename TM, bool KC, int R, int NT, int DEPTH,
          bool ANY>
struct Stager {
  static constexpr int KE = kStageBytes / (int)sizeof(TM);
  static constexpr int E = 16 / (int)sizeof(TS);  // elements per load
  static constexpr int ROWS = KC ? R : KE;
  static constexpr int CPR = (KC ? KE : R) / E;  // loads per staged row
  static constexpr int RPP = NT / CPR;           // rows per pass
  static constexpr int PASSES = ROWS / RPP;
  static constexpr int LDS_ROW = KC ? kStageBytes : R * (int)sizeof(TM);
  static constexpr int NCH = LDS_ROW / 16;
  static constexpr int BYTES = ROWS * LDS_ROW;
  static constexpr bool kWiden = sizeof(TS) != sizeof(TM);
  static_assert(CPR >= 1 && NT % CPR == 0 && ROWS % RPP == 0 && PASSES >= 1,
                "staging shape");
  static_assert(!KC || RPP % 16 == 0 || 16 % RPP == 0, "swizzle");

  typedef typename std::conditional<ANY, const char *, uint32_t>::type Lane;
  const char *base;  // this stage's wave-uniform base (ANY: in the lanes)
  Lane lane[PASSES];
  i32x4 reg[DEPTH][PASSES];
  int shift[DEPTH];       // bytes the chunks are shifted down at a row's end
  int64_t ld, extent, K;  // extent: M or N
  int row, pos;           // this lane's staged row (pass 0) and position
  bool edge;              // !KC: the tile runs past the row's end

  __device__ __forceinline__ void init(const TS *p, int64_t ld_, int64_t r0,
                                       int64_t extent_, int64_t k_begin,
                                       int64_t k_total) {
    ld = ld_;
    extent = extent_;
    K = k_total;
    const int tid = threadIdx.x;
    row = tid / CPR;
    pos = (tid % CPR) * E;
    int64_t start = pos;  // this lane's first element, from the base's column
    if constexpr (KC) {
      base = (const char *)(p + r0 * ld + k_begin);
    } else {
      base = (const char *)(p + k_begin * ld);
      edge = r0 + R > extent;
      const int64_t c = r0 + pos;
      start = c + E <= extent ? c : extent < E ? 0 : extent - E;
#pragma unroll
      for (int d = 0; d < DEPTH; ++d)
        shift[d] = c - start < E ? (int)(c - start) * (int)sizeof(TS) : 16;
    }
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      int64_t r = i * RPP + row;
      if (KC && r0 + r >= extent)
        r = extent - 1 - r0;
      const int64_t off = (r * ld + start) * (int64_t)sizeof(TS);
      if constexpr (ANY)
        lane[i] = base + off;
      else
        lane[i] = (uint32_t)off;
    }
  }

  __device__ __forceinline__ const char *addr(int i) const {
    if constexpr (ANY)
      return lane[i];
    else
      return base + lane[i];
  }

  __device__ __forceinline__ void advance() {
    const int64_t step = (KC ? (int64_t)KE : KE * ld) * (int64_t)sizeof(TS);
    if constexpr (ANY) {
#pragma unroll
      for (int i = 0; i < PASSES; ++i)
        lane[i] += step;
    } else {
      base += step;
    }
  }

  // The stage at k0 into register set `d`.
  __device__ __forceinline__ void load(int d, int64_t k0) {
    if constexpr (KC) {
      shift[d] = 0;
      if (k0 + KE <= K) {
#pragma unroll
        for (int i = 0; i < PASSES; ++i)
          reg[d][i] = *(const i32x4_u *)addr(i);
      } else if (!ANY || K >= E) {  // the K tail: zeros past K
        const int64_t kp = k0 + pos;
        const int64_t start = kp + E <= K ? kp : K - E;
        shift[d] = kp - start < E ? (int)(kp - start) * (int)sizeof(TS) : 16;
#pragma unroll
        for (int i = 0; i < PASSES; ++i)
          reg[d][i] = *(const i32x4_u *)(addr(i) -
                                         (kp - start) * (int64_t)sizeof(TS));
      } else if constexpr (ANY) {
#pragma unroll
        for (int i = 0; i < PASSES; ++i)
          reg[d][i] = load_short<TS, E>((const TS *)addr(i) - (k0 + pos),
                                        k0 + pos, K);
      }
    } else {
      if (ANY && extent < E) {
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
          reg[d][i] = i32x4{0, 0, 0, 0};
          if (k0 + i * RPP + row < K)  // the tile starts at the row's start
            reg[d][i] = load_short<TS, E>((const TS *)addr(i), pos, extent);
        }
        shift[d] = 0;
      } else if (k0 + KE <= K) {
#pragma unroll
        for (int i = 0; i < PASSES; ++i)
          reg[d][i] = *(const i32x4_u *)addr(i);
      } else {  // rows past K: zeros
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
          reg[d][i] = i32x4{0, 0, 0, 0};
          if (k0 + i * RPP + row < K)
            reg[d][i] = *(const i32x4_u *)addr(i);
        }
      }
    }
    advance();
  }

  __device__ __forceinline__ int lds_offset(int r, int chunk) const {
    const int sw = KC ? (r / 2) % 8 : row_swizzle<(int)sizeof(TM), NCH>(r);
    return r * LDS_ROW + ((chunk ^ sw) << 4);
  }

  // Register set `d`, loaded from k0, to a slot of the LDS ring. Chunks at a
  // row's end are shifted here and not at the load, which stays in flight.
  __device__ __forceinline__ void store(int d, int64_t k0, char *slot) {
    const int chunk = threadIdx.x % CPR;
    if (KC ? k0 + KE > K : edge) {
#pragma unroll
      for (int i = 0; i < PASSES; ++i)
        reg[d][i] = shift_down(reg[d][i], shift[d]);
    }
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int r = i * RPP + row;
      if constexpr (kWiden) {
        *(i32x4 *)(slot + lds_offset(r, 2 * chunk)) =
            i8x8_to_f16x8(i32x2{reg[d][i][0], reg[d][i][1]});
        *(i32x4 *)(slot + lds_offset(r, 2 * chunk + 1)) =
            i8x8_to_f16x8(i32x2{reg[d][i][2], reg[d][i][3]});
      } else {
        *(i32x4 *)(slot + lds_offset(r, chunk)) = reg[d][i];
      }
    }
  }
};

// One MFMA operand fragment (16 rows x 64 bytes of K) of a staged slot, from
// tile row (column) w0.
template <typename S, typename TM, bool KC>
__device__ __forceinline__ i32x4 read_frag(const char *slot, int w0, int ks,
                                           int lane) {
  const int l15 = lane & 15, lg = lane >> 4;
  if constexpr (KC) {
    const int off =
        (w0 + l15) * kStageBytes + (((4 * ks + lg) ^ (l15 / 2)) << 4);
    return *(const i32x4 *)(slot + off);
  } else if constexpr (sizeof(TM) == 2) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    const int k = 32 * ks + 8 * lg + (l15 >> 2);
    const int byte = 2 * (w0 + 4 * (l15 & 3));
    const int off = k * S::LDS_ROW +
                    (((byte >> 4) ^ row_swizzle<2, S::NCH>(k)) << 4) +
                    (byte & 15);
    const IHP_LDS char *p = (const IHP_LDS char *)slot + off;
    const i32x2 lo = __builtin_bit_cast(
        i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((IHP_LDS s16x4 *)p));
    const i32x2 hi = __builtin_bit_cast(
        i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                   (IHP_LDS s16x4 *)(p + 4 * S::LDS_ROW)));
    return i32x4{lo[0], lo[1], hi[0], hi[1]};
  } else {
    const int k = 64 * ks + 16 * lg + (l15 >> 1);
    const int byte = w0 + 8 * (l15 & 1);
    const int off = k * S::LDS_ROW +
                    (((byte >> 4) ^ row_swizzle<1, S::NCH>(k)) << 4) +
                    (byte & 15);
    const IHP_LDS char *p = (const IHP_LDS char *)slot + off;
    const i32x2 lo =
        __builtin_amdgcn_ds_read_tr8_b64_v2i32((IHP_LDS i32x2 *)p);
    const i32x2 hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
        (IHP_LDS i32x2 *)(p + 8 * S::LDS_ROW));
    return i32x4{lo[0], lo[1], hi[0], hi[1]};
  }
}

// Barrier ordering LDS only: the global loads of the next stage stay in
// flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int kDeviceScope = 16;  // sc1 of a buffer instruction

}  // namespace

struct RaggedArgs {
  const void *a, *b;
  void *c;
  const f16 *scale;
  int64_t M, N, K, lda, ldb, ldc, sa, sb, sc, s_mul;
  Epi epi;
  int accumulate;
  int through;         // store the result past the L2 (kStoreThroughBytes)
  int k_split;         // K elements per split, a multiple of the stage
  float *partials;     // split-K: f32 / i32 partial tiles, else unused
  unsigned *counters;
};

template <typename TA, typename TB, typename OutT, bool AT, bool BT, int BM,
          int BN, int WM, int WN, int WGS, int DEPTH, bool ANY>
__global__ __launch_bounds__(64 * WM *WN, WGS) void gemm_ragged_kernel(
    RaggedArgs p) {
  typedef typename MfmaInput<TA, TB>::type TM;
  typedef Mfma16<TM> MF;
  typedef typename MF::Acc Acc;
  constexpr int NT = 64 * WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int FM = WTM / 16, FN = WTN / 16;
  typedef Stager<TA, TM, !AT, BM, NT, DEPTH, ANY> SA;
  typedef Stager<TB, TM, BT, BN, NT, DEPTH, ANY> SB;
  constexpr int KE = SA::KE;
  constexpr int SLOT = SA::BYTES + SB::BYTES;
  constexpr bool kScale = !std::is_same<TA, TB>::value;
  __shared__ __attribute__((aligned(1024))) char smem[2 * SLOT];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int64_t z = blockIdx.z;
  const int tiles_m = (int)((p.M + BM - 1) / BM);
  const int tiles_n = (int)((p.N + BN - 1) / BN);
  int tm, tn;
  xcd_tile_order((int)blockIdx.x, (int)gridDim.x, tiles_m, tiles_n, 4, &tm,
                 &tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int64_t k_begin = (int64_t)blockIdx.y * p.k_split;
  const int64_t k_end =
      p.K - k_begin < p.k_split ? p.K : k_begin + p.k_split;
  const int nk = (int)((k_end - k_begin + KE - 1) / KE);

  Acc acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[i][j][r] = 0;

  if (nk > 0) {
    SA sa;
    SB sb;
    sa.init((const TA *)p.a + z * p.sa, p.lda, m0, p.M, k_begin, p.K);
    sb.init((const TB *)p.b + z * p.sb, p.ldb, n0, p.N, k_begin, p.K);
    auto load = [&](int d, int t) {
      const int64_t k0 = k_begin + (int64_t)t * KE;
      sa.load(d, k0);
      sb.load(d, k0);
    };
    auto store = [&](int d, int t) {
      const int64_t k0 = k_begin + (int64_t)t * KE;
      char *slot = smem + (t & 1) * SLOT;
      sa.store(d, k0, slot);
      sb.store(d, k0, slot + SA::BYTES);
    };
    load(0, 0);
    store(0, 0);
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (1 + d < nk)
        load(d, 1 + d);
    lds_barrier();
    // Fragments of K step 0 and 1. Each is read half a stage ahead, so the
    // reads (and the barrier) run under the other step's MFMAs: a CU with one
    // workgroup has no other wave to hide them.
    i32x4 fa[2][FM], fb[2][FN];
    auto read = [&](int ks, int t) __attribute__((always_inline)) {
      const char *slot = smem + (t & 1) * SLOT;
#pragma unroll
      for (int i = 0; i < FM; ++i)
        fa[ks][i] = read_frag<SA, TM, !AT>(slot, wm * WTM + i * 16, ks, lane);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        fb[ks][j] = read_frag<SB, TM, BT>(slot + SA::BYTES, wn * WTN + j * 16,
                                          ks, lane);
    };
    auto mma = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = MF::mma(fb[ks][j], fa[ks][i], acc[i][j]);
    };
    read(0, 0);
    // Stage t; register set d holds stage t + 1.
    auto stage = [&](int d, int t) __attribute__((always_inline)) {
      read(1, t);
      if (t + 1 < nk)
        store(d, t + 1);
      if (t + 1 + DEPTH < nk)
        load(d, t + 1 + DEPTH);
      mma(0);
      lds_barrier();
      if (t + 1 < nk)
        read(0, t + 1);
      mma(1);
    };
    int t = 0;
    for (; t + DEPTH <= nk; t += DEPTH)
#pragma unroll
      for (int d = 0; d < DEPTH; ++d)
        stage(d, t + d);
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
      if (t + d < nk)
        stage(d, t + d);
  }

  const int splits = (int)gridDim.y;
  if (splits > 1) {
    // Partial tiles of one output tile: [split][fragment][lane] x 16 bytes.
    const int64_t tile = z * gridDim.x + blockIdx.x;
    char *tile_parts =
        (char *)p.partials + tile * splits * (int64_t)(BM * BN * 4);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(tile_parts, 0, -1, 0x00027000);
    const int voff = (wave * FM * FN * 64 + lane) * 16;
    // Fragments of rows past M are neither published nor summed.
    const int frags = (int)((p.M - m0 - wm * WTM + 15) / 16);
#pragma unroll
    for (int i = 0; i < FM; ++i)
      if (i < frags)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(
              __builtin_bit_cast(i32x4, acc[i][j]), rs,
              voff + (i * FN + j) * 1024, (int)blockIdx.y * (BM * BN * 4),
              kDeviceScope);
    __shared__ unsigned last_split;
    unsigned *last = &last_split;
    wait_vmcnt<0>();  // published before it is counted
    __syncthreads();
    if (tid == 0) {
      const unsigned prev = __hip_atomic_fetch_add(
          &p.counters[tile * kCounterStride], 1u, __ATOMIC_RELAXED,
          __HIP_MEMORY_SCOPE_AGENT);
      *last = prev == (unsigned)splits - 1;
    }
    __syncthreads();
    if (!*last)
      return;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[i][j][r] = 0;
    // 32 loads a lane in flight (the sum is a chain of memory latencies): U
    // splits at a time, the last one again where they run out.
    constexpr int U = 32 / (FM * FN);
    for (int s0 = 0; s0 < splits; s0 += U) {
      i32x4 v[U][FM][FN];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int s = s0 + u < splits ? s0 + u : splits - 1;
#pragma unroll
        for (int i = 0; i < FM; ++i)
          if (i < frags)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              v[u][i][j] = __builtin_amdgcn_raw_buffer_load_b128(
                  rs, voff + (i * FN + j) * 1024, s * (BM * BN * 4),
                  kDeviceScope);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s0 + u < splits)
#pragma unroll
          for (int i = 0; i < FM; ++i)
            if (i < frags)
#pragma unroll
              for (int j = 0; j < FN; ++j)
                acc[i][j] += __builtin_bit_cast(Acc, v[u][i][j]);
    }
    if (tid == 0)  // re-arm for the next call on this workspace
      __hip_atomic_store(&p.counters[tile * kCounterStride], 0u,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // out = [C +] mul * act(acc [* scale] + bias), 4 columns a lane. i32 and
  // f32 results are stored from there, 64 bytes of a row an instruction; f16
  // ones (32 bytes) go through the wave's part of the idle LDS ring, row
  // chunks swizzled, and leave as whole rows of the wave's tile: short sums
  // with large results are bound by these stores (int8 weights, 1500 x 4096 x
  // 256: 17.9 us without the staging).
  constexpr bool kIntOut = std::is_same<OutT, int32_t>::value;
  constexpr bool kStage = sizeof(OutT) == 2;
  constexpr int OROW = WTN * (int)sizeof(OutT);  // bytes of a staged row
  constexpr int OCH = OROW / 16;
  static_assert(!kStage || (WM * WN * WTM * OROW <= 2 * SLOT &&
                            (OCH & (OCH - 1)) == 0),
                "staging");
  char *const stage = smem + wave * (WTM * OROW);
  OutT *C = (OutT *)p.c + z * p.sc;
  const f16 *mul = p.epi.mul ? p.epi.mul + z * p.s_mul : nullptr;
  const int64_t row0 = m0 + wm * WTM, col0 = n0 + wn * WTN;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int64_t col = col0 + j * 16 + 4 * (lane >> 4);
    const int valid = (int)(p.N - col < 4 ? p.N - col : 4);
    if (valid <= 0)
      continue;
    float sc[4] = {1.0f, 1.0f, 1.0f, 1.0f}, bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (!kIntOut) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r < valid) {
          if (kScale)
            sc[r] = (float)p.scale[col + r];
          if (p.epi.bias)
            bias[r] = (float)p.epi.bias[col + r];
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int64_t row = row0 + i * 16 + (lane & 15);
      if (row >= p.M)
        continue;
      OutT *dst = C + row * p.ldc + col;
      if constexpr (kIntOut) {
        if (valid == 4) {
          i32x4 v = acc[i][j];
          if (p.accumulate) {
            const i32x4 old = *(const i32x4_u4 *)dst;
#pragma unroll
            for (int r = 0; r < 4; ++r)
              v[r] = (int)((unsigned)old[r] + (unsigned)v[r]);
          }
          if (p.through)
            store_through16(dst, v);
          else
            *(i32x4_u4 *)dst = v;
        } else {
#pragma unroll
          for (int r = 0; r < 3; ++r)
            if (r < valid)
              store_out(dst + r, acc[i][j][r],
                        p.accumulate ? kStoreAccumulate : kStorePlain);
        }
      } else {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] = acc[i][j][r];
          if (kScale)
            v[r] *= sc[r];
          v[r] = epi_act(v[r] + bias[r], p.epi.act);
        }
        if (mul) {
          const f16 *g = mul + row * p.epi.ld_mul + col;
          f16x4 gv = {0, 0, 0, 0};
          if (valid == 4)
            gv = *(const f16x4_u *)g;
          else
#pragma unroll
            for (int r = 0; r < 3; ++r)
              if (r < valid)
                gv[r] = g[r];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] *= (float)gv[r];
        }
        if (p.accumulate) {
          if (valid == 4) {
            if constexpr (kStage) {
              const f16x4 old = *(const f16x4_u *)dst;
#pragma unroll
              for (int r = 0; r < 4; ++r)
                v[r] += (float)old[r];
            } else {
              const f32x4 old = *(const f32x4_u *)dst;
#pragma unroll
              for (int r = 0; r < 4; ++r)
                v[r] += old[r];
            }
          } else {
#pragma unroll
            for (int r = 0; r < 3; ++r)
              if (r < valid)
                v[r] += (float)dst[r];
          }
        }
        if constexpr (kStage) {
          const int srow = i * 16 + (lane & 15);
          const int byte = (j * 16 + 4 * (lane >> 4)) * 2;
          *(f16x4 *)(stage + srow * OROW +
                     (((byte >> 4) ^ (srow & (OCH - 1))) << 4) + (byte & 15)) =
              f16x4{(f16)v[0], (f16)v[1], (f16)v[2], (f16)v[3]};
        } else if (valid == 4) {
          const f32x4 o = {v[0], v[1], v[2], v[3]};
          if (p.through)
            store_through16(dst, __builtin_bit_cast(i32x4, o));
          else
            *(f32x4_u *)dst = o;
        } else {
#pragma unroll
          for (int r = 0; r < 3; ++r)
            if (r < valid)
              dst[r] = (OutT)v[r];
        }
      }
    }
  }
  if constexpr (kStage) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < WTM * OCH / 64; ++t) {
      const int srow = (t * 64 + lane) / OCH, ch = (t * 64 + lane) % OCH;
      const int64_t row = row0 + srow, col = col0 + ch * 8;
      if (row >= p.M || col >= p.N)
        continue;
      const i32x4 v = *(const i32x4 *)(stage + srow * OROW +
                                       ((ch ^ (srow & (OCH - 1))) << 4));
      OutT *dst = C + row * p.ldc + col;
      if (col + 8 <= p.N) {
        if (p.through)
          store_through16(dst, v);
        else
          *(i32x4_u *)dst = v;
      } else {
        const f16x8 h = __builtin_bit_cast(f16x8, v);
#pragma unroll
        for (int r = 0; r < 7; ++r)
          if (col + r < p.N)
            dst[r] = h[r];
      }
    }
  }
}

// ----------------------------------------------------------------------------
// Host side: the configurations and their launch.
// ----------------------------------------------------------------------------

template <typename TA, typename TB, typename OutT, bool AT, bool BT, int BM,
          int BN, int WM, int WN, int WGS, int DEPTH, bool ANY>
static hipError_t launch_ragged(const MatmulArgs &a, int splits, int k_split) {
  const int64_t tiles_m = (a.m + BM - 1) / BM, tiles_n = (a.n + BN - 1) / BN;
  if (tiles_m * tiles_n >= ((int64_t)1 << 31))
    return hipErrorInvalidValue;
  RaggedArgs p;
  p.a = a.a;
  p.b = a.b;
  p.c = a.c;
  p.scale = (const f16 *)a.scale;
  p.M = a.m;
  p.N = a.n;
  p.K = a.k;
  p.lda = a.lda;
  p.ldb = a.ldb;
  p.ldc = a.ldc;
  p.sa = a.sa;
  p.sb = a.sb;
  p.sc = a.sc;
  p.s_mul = epi_batch_stride(a);
  p.epi = make_epi(a);
  p.accumulate = a.accumulate;
  p.through = a.m * a.n * a.batch * (int64_t)sizeof(OutT) >= kStoreThroughBytes;
  p.k_split = k_split;
  p.counters = (unsigned *)a.workspace;
  p.partials = (float *)((char *)a.workspace + kWorkspaceCounterBytes);
  hipLaunchKernelGGL(
      (gemm_ragged_kernel<TA, TB, OutT, AT, BT, BM, BN, WM, WN, WGS,
                          DEPTH, ANY>),
      dim3((unsigned)(tiles_m * tiles_n), (unsigned)splits, (unsigned)a.batch),
      dim3(64 * WM * WN), 0, (hipStream_t)a.stream, p);
  return hipGetLastError();
}

// One configuration of every layout a kind has. Names: general_<types>, then
// the layout unless it is A [M,K], B [K,N], then the tile unless it is 64x64.
#define IHP_RAGGED(KIND, NAME, TA, TB, OUT, AT, BT, BM, BN, WM, WN, WGS, D, W)\
  {NAME, KIND, AT, BT, BM, BN, WGS, W, 64 * WM * WN, 2 * 128 * (BM + BN),     \
   (const void *)&gemm_ragged_kernel<TA, TB, OUT, AT, BT, BM, BN, WM, WN,     \
                                     WGS, D, W>,                                     \
   &launch_ragged<TA, TB, OUT, AT, BT, BM, BN, WM, WN, WGS, D, W>}
#define IHP_RAGGED_B(KIND, PRE, TA, TB, OUT, TILE, ...)                       \
  IHP_RAGGED(KIND, PRE TILE, TA, TB, OUT, false, false, __VA_ARGS__),         \
      IHP_RAGGED(KIND, PRE "_tn" TILE, TA, TB, OUT, false, true, __VA_ARGS__)
#define IHP_RAGGED_AB(KIND, PRE, TA, TB, OUT, TILE, ...)                      \
  IHP_RAGGED_B(KIND, PRE, TA, TB, OUT, TILE, __VA_ARGS__),                    \
      IHP_RAGGED(KIND, PRE "_at" TILE, TA, TB, OUT, true, false,              \
                 __VA_ARGS__),                                                 \
      IHP_RAGGED(KIND, PRE "_at_tn" TILE, TA, TB, OUT, true, true, __VA_ARGS__)
#define IHP_RAGGED_ALL(TILE, ...)                                             \
  IHP_RAGGED_AB(kGeneralF16F16, "general_f16", f16, f16, f16, TILE,           \
                __VA_ARGS__),                                                  \
      IHP_RAGGED_AB(kGeneralF16F32, "general_f16f32", f16, f16, float, TILE,  \
                    __VA_ARGS__),                                              \
      IHP_RAGGED_B(kGeneralI8I32, "general_i8", int8_t, int8_t, int32_t,      \
                   TILE, __VA_ARGS__),                                         \
      IHP_RAGGED_B(kGeneralW8A16, "general_w8a16", f16, int8_t, f16, TILE,    \
                   __VA_ARGS__)

static const GeneralConfig kGeneralConfigs[] = {
    IHP_RAGGED_ALL("", 64, 64, 2, 2, 3, 2, false),
    IHP_RAGGED_ALL("_64x128", 64, 128, 2, 2, 2, 2, false),
    IHP_RAGGED_ALL("_128x128", 128, 128, 2, 2, 2, 1, false),
    IHP_RAGGED_ALL("_any", 64, 64, 2, 2, 3, 1, true),
};

const GeneralConfig *general_configs(int *count) {
  *count = (int)(sizeof(kGeneralConfigs) / sizeof(kGeneralConfigs[0]));
  return kGeneralConfigs;
}

hipError_t launch_general(const MatmulArgs &a, const GeneralPlan &plan) {
  int count = 0;
  return general_configs(&count)[plan.index].launch(a, plan.splits,
                                                    plan.k_split);
}

}  // namespace ihp
