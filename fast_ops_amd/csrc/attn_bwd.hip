// FlashAttention backward for gfx950 (MI355X): dQ, dK, dV from Q, K, V, O, dO and the forward's logsumexp.
//
// Replaces the backward the reference leaves unimplemented behind its CUDA forward (fast_ops/flash_attention/
// flash_attention.py:40-45) with what its Triton backward computes (flash_attention_triton.py:273-315 delta pre-pass,
// :322-638 kernel, :832-958 host): with P = exp(scale * Q K^T - LSE) (masked entries 0),
//     delta_i = sum_d dO_id O_id      dV = P^T dO      dP = dO V^T      dS = P * (dP - delta) * scale
//     dQ = dS K                       dK = dS^T Q
// fp32 scores and accumulators; P and dS are rounded to the operand type before the second GEMMs, as the reference
// does (:515,:562-563).
//
// Two launches, no atomics, no scratch beyond the caller's [2, B, H, Sq] fp32 workspace (delta and -LSE / scale), or, where the caller
// gives memory for it, dS kept by the dK/dV kernel and dQ computed from that (attn_bwd.hpp, attn_bwd_dq_of_ds.hip). The two:
//   1. attn_bwd_dq_kernel: one workgroup per 128 query rows (4 waves x 32), walks the key tiles like the forward
//      kernel. Scores are computed transposed, S^T = K Q^T and dP^T = V dO^T (A operands = K / V rows from LDS, B
//      operands = Q^T / dO^T held in registers), so a lane owns one query: LSE and delta are per-lane scalars and
//      dS^T is, as it stands, the B operand of dQ^T = K^T dS^T (A operand via the transposing LDS read of the K tile).
//      It also computes delta (negated) from the dO fragments it holds and the same pieces of O, and stores it.
//   2. attn_bwd_dkdv_kernel: one workgroup per 128 keys (4 waves x 32), walks the query tiles. Here the scores are
//      computed untransposed, S = Q K^T and dP = dO V^T (A operands = Q / dO rows from LDS, B operands = K^T / V^T
//      held in registers), so a lane owns one key and P, dS are the B operands of dV^T = dO^T P and dK^T = Q^T dS
//      (A operands via the transposing LDS read of the dO and Q tiles); per-row LSE and delta come from LDS.
//      Mostly this runs as attn_bwd_dkdv_pipe_kernel, the same computation laid out by hand as a software pipeline (described
//      there); attn_bwd_dkdv_kernel is the plain, compiler-scheduled form for what that one does not take: a bias with a query
//      stride whose tiles cannot be copied or that comes with dropout, other head dims with dropout or a bias.
// Both recompute the scores (seven GEMMs in total instead of the five of an atomics-based single pass). softmax_scale
// is applied once to the finished dQ and dK accumulators rather than to every dS.
// Tiles of 64 rows go global -> LDS with the direct-to-LDS loads, double buffered (three buffers in the pipelined
// kernel), one barrier per tile, 16-byte chunks XOR-swizzled inside a row (no bank conflicts), exactly as in the
// 128-row forward kernel.
#include <type_traits>

#include <mutex>

#include "attn_bwd.hpp"

namespace fo {

// acc += A B with the accumulator pinned in AGPRs. Left to the compiler, the 128 accumulator registers of dK and dV are
// kept elsewhere between uses and copied in and out around every MFMA (eight extra VALU instructions per MFMA). Inside
// an asm statement the compiler's hazard recognizer does not see the MFMA: no source may have been written by a VALU
// instruction (a register copy, say) in the two instructions before it, and nothing but such an MFMA may touch an
// accumulator before acc_fence(). The build checks the generated assembly for both (fast_ops_amd/asm_lint.py) and
// falls back to FO_MFMA_NOPS=1, the builtin, if it finds a violation.
#ifndef FO_MFMA_NOPS
#define FO_MFMA_NOPS 0
#endif
// pipelined dK/dV kernel: the copies of the tile after next are issued between the MFMAs of phase 4 (1) or in one batch
// at the hand-over (0)
#ifndef FO_BWD_SPREAD
#define FO_BWD_SPREAD 1
#endif
template <typename T>
__device__ __forceinline__ void mfma_acc_agpr(f32x16& acc, typename Ops<T>::vec8 a, typename Ops<T>::vec8 b) {
#if defined(__HIP_DEVICE_COMPILE__) && !FO_MFMA_NOPS
  if constexpr (std::is_same<T, __bf16>::value)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
#else
  acc = Ops<T>::mfma(a, b, acc);
#endif
}
// S / dP of the pipelined dK/dV kernel: result pinned in VGPRs (the softmax gradient reads it element by element; from
// AGPRs every read is an extra instruction); the accumulator is given its start values before the first call. A VALU
// instruction may read the result 11 wait states after the last MFMA was issued: the kernel's schedule sees to that.
template <typename T>
__device__ __forceinline__ void mfma_scores_vgpr(f32x16& acc, typename Ops<T>::vec8 a, typename Ops<T>::vec8 b) {
#if defined(__HIP_DEVICE_COMPILE__) && !FO_MFMA_NOPS
  if constexpr (std::is_same<T, __bf16>::value) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
#else
  acc = Ops<T>::mfma(a, b, acc);
#endif
}
// the first of a chain, started from zero or from registers that stay as they are
template <typename T>
__device__ __forceinline__ void mfma_scores_vgpr_first(f32x16& acc, typename Ops<T>::vec8 a, typename Ops<T>::vec8 b, const f32x16& start) {
#if defined(__HIP_DEVICE_COMPILE__) && !FO_MFMA_NOPS
  if constexpr (std::is_same<T, __bf16>::value) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(acc) : "v"(a), "v"(b), "v"(start));
  else asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %3" : "=&v"(acc) : "v"(a), "v"(b), "v"(start));
#else
  acc = Ops<T>::mfma(a, b, start);
#endif
}
template <typename T>
__device__ __forceinline__ void mfma_scores_vgpr_first(f32x16& acc, typename Ops<T>::vec8 a, typename Ops<T>::vec8 b) {
#if defined(__HIP_DEVICE_COMPILE__) && !FO_MFMA_NOPS
  if constexpr (std::is_same<T, __bf16>::value) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));
#else
  f32x16 zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.0f;
  acc = Ops<T>::mfma(a, b, zero);
#endif
}
template <int N>
__device__ __forceinline__ void acc_fence(f32x16 (&acc)[N]) {
#if defined(__HIP_DEVICE_COMPILE__) && !FO_MFMA_NOPS
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+a"(acc[i]));
#endif
}

// ---------------------------------------------------------------------------------------------------------------------
// ---------------------------------------------------------------------------------------------------------------------
// Copy of a 64-row tile (rows row0 .. row0+63 of a [S, D] matrix with row stride `stride`) into LDS by the whole
// workgroup: per wave D/32 direct-to-LDS instructions. Each instruction fills 1 KiB of LDS with the 64 lanes' pieces
// back to back, so the swizzle is applied by choosing which global chunk a lane fetches. Rows past the end re-read
// the last row (callers mask them); columns from the true head_dim `d` on read zeros.
template <typename T, int D>
__device__ __forceinline__ void copy_tile64(const T* base, int64_t stride, int row0, int S, int d, FO_LDS char* dst, int wave_s, int lane_in) {
  // (an opaque copy of the lane index: this is the path of tiles that cross the end of the matrix, taken once per
  // workgroup at most; its address arithmetic must not be hoisted out of it into registers that live across the loop)
  int lane = lane_in;
  asm volatile("" : "+v"(lane));
  constexpr int ROW_BYTES = D * 2;
  constexpr int CHUNKS = ROW_BYTES / 16;
  constexpr int ROWS_PER_DMA = 1024 / ROW_BYTES;
  constexpr int DMA_PER_WAVE = kBwdTile * ROW_BYTES / 1024 / kBwdWaves;
#pragma unroll
  for (int i = 0; i < DMA_PER_WAVE; ++i) {
    const int row = (wave_s * DMA_PER_WAVE + i) * ROWS_PER_DMA + lane / CHUNKS;
    const int col = ((lane % CHUNKS) ^ swz<D>(row)) * 8;
    const int r = min(row0 + row, S - 1);
    dma16_lane_ptr(live_or_zero(base + (int64_t)r * stride + col, col, d), dst + (wave_s * DMA_PER_WAVE + i) * 1024);
  }
}

// The same copy for a tile that lies wholly inside the matrix, with the address split into a wave-uniform base (the
// tile's first row: scalar arithmetic, once per tile) and per-lane byte offsets that never change (TileLaneOffsets,
// computed once per kernel): two instructions per 1 KiB piece instead of a 64-bit multiply-add per lane and piece.
template <typename T, int D>
struct TileLaneOffsets {
  static constexpr int N = kBwdTile * D * 2 / 1024 / kBwdWaves;   // pieces per wave and tile
  uint32_t off[N];
  bool ok;                                                        // 32-bit offsets suffice for this row stride, and the rows have all D columns
  __device__ __forceinline__ void init(int64_t stride, int d, int wave_s, int lane) {
    constexpr int ROW_BYTES = D * 2, CHUNKS = ROW_BYTES / 16, ROWS_PER_DMA = 1024 / ROW_BYTES;
    ok = stride < (1 << 23) && d == D;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int row = (wave_s * N + i) * ROWS_PER_DMA + lane / CHUNKS;
      const int col = ((lane % CHUNKS) ^ swz<D>(row)) * 8;
      off[i] = (uint32_t)(row * (int)stride + col) * 2u;
    }
  }
};
template <typename T, int D>
__device__ __forceinline__ void copy_tile64_inside(const T* base, int64_t stride, int row0, const TileLaneOffsets<T, D>& lo,
                                                   FO_LDS char* dst, int wave_s) {
  const char* tile = (const char*)(base + (int64_t)row0 * stride);
#pragma unroll
  for (int i = 0; i < TileLaneOffsets<T, D>::N; ++i) dma16_uniform_base(tile, lo.off[i], dst + (wave_s * TileLaneOffsets<T, D>::N + i) * 1024);
}

// A head_dim d below D: the lanes whose piece of a tile lies inside the d columns. Copies by those lanes alone leave the
// rest of the tile's rows in LDS untouched, which therefore stays zero once it is (copy_tile64 writes zeros there): a tile
// inside the matrix then costs what it costs at d == D, where copy_tile64 takes a 64-bit address per lane and piece.
template <typename T, int D>
struct TileLiveLanes {
  static constexpr int N = kBwdTile * D * 2 / 1024 / kBwdWaves;
  uint64_t lanes[N];
  __device__ __forceinline__ void init(int d, int wave_s, int lane) {
    constexpr int CHUNKS = D * 2 / 16, ROWS_PER_DMA = 1024 / (D * 2);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int row = (wave_s * N + i) * ROWS_PER_DMA + lane / CHUNKS;
      lanes[i] = __builtin_amdgcn_ballot_w64(((lane % CHUNKS) ^ swz<D>(row)) * 8 < d);
    }
  }
};
template <typename T, int D>
__device__ __forceinline__ void copy_tile64_inside(const T* base, int64_t stride, int row0, const TileLaneOffsets<T, D>& lo,
                                                   const TileLiveLanes<T, D>& live, FO_LDS char* dst, int wave_s) {
  const char* tile = (const char*)(base + (int64_t)row0 * stride);
  const uint32_t dst_s = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)dst) + (uint32_t)(wave_s * TileLaneOffsets<T, D>::N * 1024);
#pragma unroll
  for (int i = 0; i < TileLaneOffsets<T, D>::N; ++i) dma16_uniform_base_of_lanes(tile, lo.off[i], dst_s + i * 1024, live.lanes[i]);
}

// The same offsets kept as two registers per matrix instead of one per piece, for a kernel that has none to spare: the
// byte offset of the lane's row of piece 0 and of its 16-byte chunk in that row. Piece i lies ROWS_PER_DMA * i rows
// further (added to the uniform base) and its rows' swizzle differs from piece 0's in fixed bits (i for 256-byte rows,
// 2 i for 128-byte rows: the bits of the row number that the swizzle takes and the piece index changes), so a piece's
// offset is an XOR with a constant and an addition.
template <typename T, int D>
struct TileLaneOffsetsCompact {
  static constexpr int N = kBwdTile * D * 2 / 1024 / kBwdWaves;
  static constexpr int ROW_BYTES = D * 2, CHUNKS = ROW_BYTES / 16, ROWS_PER_DMA = 1024 / ROW_BYTES;
  uint32_t row_bytes0, chunk_bytes0;
  bool ok;
  __device__ __forceinline__ void init(int64_t stride, int d, int wave_s, int lane) {
    ok = stride < (1 << 23) && d == D;
    const int row = (wave_s * N) * ROWS_PER_DMA + lane / CHUNKS;
    row_bytes0 = (uint32_t)(row * (int)stride) * 2u;
    chunk_bytes0 = (uint32_t)(((lane % CHUNKS) ^ swz<D>(row)) * 16);
  }
  static constexpr uint32_t flip(int i) { return (uint32_t)((D == 128 ? i : 2 * i) * 16); }
  // (wave_s * N is a multiple of N = 4 or 2, so the piece index occupies bits of the row number that are zero in piece 0)
  static_assert((D == 128 && N == 4) || (D == 64 && N == 2), "which bits of the swizzle a piece index changes");
};
// Two tiles (K and V) at once: every offset is computed before the first copy goes out. (Should the compiler have parked
// one of the four registers in scratch memory, its reload - which it waits for with vmcnt(0) - then comes before the
// copies and finds nothing in flight; between two copies it would wait for the first one to land.)
template <typename T, int D>
__device__ __forceinline__ void copy_two_tiles64_inside(const T* base_a, int64_t stride_a, const TileLaneOffsetsCompact<T, D>& lo_a, FO_LDS char* dst_a,
                                                        const T* base_b, int64_t stride_b, const TileLaneOffsetsCompact<T, D>& lo_b, FO_LDS char* dst_b,
                                                        int row0, int wave_s) {
  typedef TileLaneOffsetsCompact<T, D> L;
  const char* tile_a = (const char*)(base_a + (int64_t)row0 * stride_a);
  const char* tile_b = (const char*)(base_b + (int64_t)row0 * stride_b);
  uint32_t ra = lo_a.row_bytes0, ca = lo_a.chunk_bytes0, rb = lo_b.row_bytes0, cb = lo_b.chunk_bytes0;
  // (recomputed per tile: hoisted out of the loop they would be 2 N registers again)
  asm volatile("" : "+v"(ra), "+v"(ca), "+v"(rb), "+v"(cb));
  uint32_t off_a[L::N], off_b[L::N];
#pragma unroll
  for (int i = 0; i < L::N; ++i) {
    off_a[i] = ra + (ca ^ L::flip(i));
    off_b[i] = rb + (cb ^ L::flip(i));
    asm volatile("" : "+v"(off_a[i]), "+v"(off_b[i]));
  }
#pragma unroll
  for (int i = 0; i < L::N; ++i) {
    dma16_uniform_base(tile_a + (int64_t)i * L::ROWS_PER_DMA * stride_a * 2, off_a[i], dst_a + (wave_s * L::N + i) * 1024);
    dma16_uniform_base(tile_b + (int64_t)i * L::ROWS_PER_DMA * stride_b * 2, off_b[i], dst_b + (wave_s * L::N + i) * 1024);
  }
}

template <int TBIAS, int D>
constexpr int tile_bias_bytes() { return TBIAS == 4 && D == 128 ? 3 * 32 * 32 * 4 : 2 * kBwdTile * 32 * TBIAS; }   // per wave of the dK/dV kernel: its tiles of a bias

// ---------------------------------------------------------------------------------------------------------------------
// KBIAS (without BIAS): a bias that is the same for every query (query stride 0), at no cost per score. Its 64
// values of a key tile, divided by softmax_scale, are what the accumulators of S^T start from - register r of a lane
// holds a key that depends on r and the half of the wave only - so that the MFMAs deliver S + b / scale and everything
// after them is the code without bias. Wave 0 fetches the values of tile t+2 while tile t is worked on (a plain load: it
// is waited for at the top of the next tile, where every copy in flight is waited for anyway), converts those of tile
// t+1 and puts them into LDS, where every wave reads them after the next barrier.
// PAD: a head_dim below D. The products run over LIVE columns, the next multiple of 32 (live_columns); the columns of a
// tile from head_dim on are zeroed by the copies of the first two tiles, and the later ones leave them alone.
// TBIAS: a bias with a query stride, of so many bytes per element, whose tiles can be copied (BiasRows): it too is what the
// score accumulators start from.
template <typename T, int D, bool CAUSAL, bool DROP, bool BIAS, bool KBIAS = false, bool PAD = false, int LIVE = D, int TBIAS = 0>
__global__ void __launch_bounds__(kBwdWaves * 64, 2) attn_bwd_dq_kernel(const AttnBwdParams prm) {
  static_assert(KBIAS + BIAS + (TBIAS != 0) <= 1, "one bias form at a time");
  typedef typename Ops<T>::vec8 vec8;
  constexpr int TILE_BYTES = kBwdTile * D * 2;
  constexpr int KSTEPS = LIVE / 16;
  constexpr int DBLK = LIVE / 32;
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  FO_LDS char* smem = (FO_LDS char*)smem_raw;   // K0 | K1 | V0 | V1 | bias of the tile's 64 keys, two buffers (BIAS)
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int n_qblk = (prm.Sq + kBwdRows - 1) / kBwdRows;
  int bh, qblk;
  bwd_item(prm, n_qblk, bh, qblk);
  qblk = n_qblk - 1 - qblk;                          // heaviest causal blocks first
  const int b = bh / prm.H, h = bh % prm.H;
  const int q0 = qblk * kBwdRows, q0w = q0 + wave * 32;
  const int Sq = prm.Sq, Sk = prm.Sk;
  const T* kbase = (const T*)prm.k + b * prm.ks[0] + h * prm.ks[1];
  const T* vbase = (const T*)prm.v + b * prm.vs[0] + h * prm.vs[1];
  const int n_tiles = CAUSAL ? (min(Sk, q0 + kBwdRows) + kBwdTile - 1) / kBwdTile : (Sk + kBwdTile - 1) / kBwdTile;

  // (one register per piece where the kernel has them - head_dim 64, and the plain causal form at head_dim 128, which
  // were 0.4-0.6 % faster that way - and two per matrix where it would otherwise park some in scratch memory)
  constexpr bool ROOMY = D == 64 || PAD || (CAUSAL && !DROP && !BIAS && !KBIAS && TBIAS == 0);
  typename std::conditional<ROOMY, TileLaneOffsets<T, D>, TileLaneOffsetsCompact<T, D>>::type klo, vlo;
  klo.init(prm.ks[2], PAD ? D : prm.d, wave_s, lane);
  vlo.init(prm.vs[2], PAD ? D : prm.d, wave_s, lane);
  TileLiveLanes<T, D> live;
  if constexpr (PAD) live.init(prm.d, wave_s, lane);
  // A bias that is the same for every query (query stride 0) is 64 values per key tile, the same for all lanes: wave 0
  // copies them into LDS with the tile (4 bytes per lane: one key in fp32, two in the operand type), and every lane
  // reads its registers' keys from there. (Loaded from global memory where they are used, the compiler waits for
  // them together with the tile copies in flight.) Keys past the end re-read the last ones and are masked below.
  FO_LDS char* bias_keys = smem + 4 * TILE_BYTES;
  bool bias_keys_staged = false;
  const char* bias_keys_src = nullptr;
  if constexpr (BIAS) {
    const int64_t at = b * prm.bias.strides[0] + h * prm.bias.strides[1];
    bias_keys_src = (const char*)prm.bias.ptr + at * (prm.bias.is_f32 ? 4 : 2);
    bias_keys_staged = prm.bias.strides[2] == 0 && ((uintptr_t)bias_keys_src % 4) == 0 && (prm.bias.is_f32 || Sk % 2 == 0);   // (pairs of keys: an even count)
  }
  auto issue = [&](int tile, int buf) {
    if constexpr (BIAS) {
      if (bias_keys_staged && wave_s == 0) {
        if (prm.bias.is_f32) dma4_lane_ptr(bias_keys_src + (int64_t)min(tile * kBwdTile + lane, Sk - 1) * 4, bias_keys + buf * 256);
        else if (lane < 32) dma4_lane_ptr(bias_keys_src + (int64_t)min(tile * kBwdTile + 2 * lane, Sk - 2) * 2, bias_keys + buf * 256);
      }
    }
    if (tile * kBwdTile + kBwdTile <= Sk && klo.ok && vlo.ok && (!PAD || tile >= 2)) {
      if constexpr (PAD) {
        copy_tile64_inside<T, D>(kbase, prm.ks[2], tile * kBwdTile, klo, live, smem + buf * TILE_BYTES, wave_s);
        copy_tile64_inside<T, D>(vbase, prm.vs[2], tile * kBwdTile, vlo, live, smem + (2 + buf) * TILE_BYTES, wave_s);
      } else if constexpr (ROOMY) {
        copy_tile64_inside<T, D>(kbase, prm.ks[2], tile * kBwdTile, klo, smem + buf * TILE_BYTES, wave_s);
        copy_tile64_inside<T, D>(vbase, prm.vs[2], tile * kBwdTile, vlo, smem + (2 + buf) * TILE_BYTES, wave_s);
      } else {
        copy_two_tiles64_inside<T, D>(kbase, prm.ks[2], klo, smem + buf * TILE_BYTES, vbase, prm.vs[2], vlo, smem + (2 + buf) * TILE_BYTES,
                                      tile * kBwdTile, wave_s);
      }
    } else {
      copy_tile64<T, D>(kbase, prm.ks[2], tile * kBwdTile, Sk, prm.d, smem + buf * TILE_BYTES, wave_s, lane);
      copy_tile64<T, D>(vbase, prm.vs[2], tile * kBwdTile, Sk, prm.d, smem + (2 + buf) * TILE_BYTES, wave_s, lane);
    }
  };
  issue(0, 0);
  FO_LDS float* key_bias = (FO_LDS float*)(smem + 4 * TILE_BYTES);      // KBIAS: [2][64], bias / scale of the keys of a tile
  float key_bias_next = 0.0f;                                           // (wave 0) this lane's key of the tile after next
  // (wave-uniform, and told so: this kernel has no vector register to spare)
  const float per_scale = KBIAS || TBIAS ? __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, kLog2e / prm.scale_log2e))) : 0.0f;
  const int64_t key_bias_row = KBIAS || TBIAS ? b * prm.bias.strides[0] + h * prm.bias.strides[1] : 0;
  if constexpr (KBIAS) {
    if (wave_s == 0) {
      key_bias[lane] = load_bias<T>(prm.bias, key_bias_row + min(lane, Sk - 1)) * per_scale;
      key_bias_next = load_bias<T>(prm.bias, key_bias_row + min(kBwdTile + lane, Sk - 1));
    }
  }
  typedef BiasRows<T, TBIAS == 4 ? 4 : 2> BR;
  // (TBIAS 4 at head_dim 128: half a tile at a time, 32 keys, or two workgroups of this kernel do not fit a compute unit)
  constexpr bool HALVES = TBIAS == 4 && D == 128;
  typedef BiasRows<T, 4, 32> BRH;
  FO_LDS char* row_bias = smem + 4 * TILE_BYTES + wave_s * (HALVES ? BRH::BYTES : BR::BYTES);      // TBIAS: the wave's own
  if constexpr (HALVES) BRH::copy(prm.bias, key_bias_row, q0 + wave_s * 32, Sq, Sk, 0, row_bias, lane);
  else if constexpr (TBIAS != 0) BR::copy(prm.bias, key_bias_row, q0 + wave_s * 32, Sq, Sk, 0, row_bias, lane);

  // B operands held for the whole kernel: Q^T and dO^T fragments of this lane's query row; its LSE and delta
  const int qrow = min(q0w + l32, Sq - 1);
  vec8 qf[KSTEPS], gf[KSTEPS];
  {
    const T* qp = (const T*)prm.q + b * prm.qs[0] + h * prm.qs[1] + (int64_t)qrow * prm.qs[2] + 8 * hh;
    const T* gp = (const T*)prm.d_o + b * prm.dos[0] + h * prm.dos[1] + (int64_t)qrow * prm.dos[2] + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      qf[ks] = *(const vec8*)live_or_zero(qp + 16 * ks, 16 * ks + 8 * hh, prm.d);
      gf[ks] = *(const vec8*)live_or_zero(gp + 16 * ks, 16 * ks + 8 * hh, prm.d);
    }
  }
  // (dropout: P comes out times k = 1 / (1 - p), so that it and dS are rounded to the operand type with that factor, as the
  // reference's are: without it fp16 gradients at p = 0.9 reach the subnormal numbers ten times earlier)
  const float lse2 = prm.lse[(int64_t)bh * Sq + qrow] * kLog2e - (DROP ? prm.drop.keep_log2 : 0.0f);
  // TBIAS: -LSE / scale starts the scores together with the bias, its rounding error (times c) takes the LSE's place in the exponent.
  // (The products of a row whose whole bias is large are otherwise summed at the ulp of bias / scale: at -1e5 an error of 1 % of dQ.
  // (bias - LSE) / scale instead is an instruction more per score: 107 -> 125 us at 12 heads x 3072 causal. The dK/dV kernel has no
  // room for a row's second value; its error there is that of -LSE / scale, rounded once: the same as of LSE * log2 e elsewhere.)
  const float row_start = -prm.lse[(int64_t)bh * Sq + qrow] * per_scale;
  const float row_shift = TBIAS ? __builtin_fmaf(-prm.lse[(int64_t)bh * Sq + qrow], per_scale, -row_start) * prm.scale_log2e : -lse2;
  // delta_i = sum_d dO_id O_id (flash_attention_triton.py:273-315), negated: this lane holds half of its row's dO
  // already, so it reads the same pieces of O, and the two halves of the wave add up. Stored for the dK/dV kernel,
  // which runs after this one (a pass of its own over O and dO would be a launch more: 5 of 83 us at B=8 H=12 S=1024).
  float delta = 0.0f;
  {
    const T* op = (const T*)prm.o + b * prm.os[0] + h * prm.os[1] + (int64_t)qrow * prm.os[2] + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      const vec8 ov = *(const vec8*)live_or_zero(op + 16 * ks, 16 * ks + 8 * hh, prm.d);
#pragma unroll
      for (int e = 0; e < 8; ++e) delta -= (float)ov[e] * (float)gf[ks][e];
    }
    delta += half_swap(delta);
    // dropout: with Z = 0 or 1 per element, dS = P (k Z dP - delta) = (k P) (Z dP - delta (1 - p))
    if constexpr (DROP) delta *= prm.drop.keep_prob;
    if (hh == 0 && q0w + l32 < Sq) prm.delta[(int64_t)bh * Sq + q0w + l32] = delta;
  }
  // (consumed here so that the compiler waits for these loads before the loop: a vmcnt wait inside the loop would
  // also wait for the tile copies in flight, which it does not see)
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) asm volatile("" ::"v"(qf[ks]), "v"(gf[ks]));
  asm volatile("" ::"v"(row_start), "v"(row_shift), "v"(delta));

  f32x16 acc[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
  const float c = prm.scale_log2e, scale = prm.scale;
  DropRows<1> drop;
  // head_dim 64: the products of dP start from -delta, sixteen registers that hold it, so that an element's dS takes an instruction less:
  // whole backward, 8 x 12 heads x 1024 causal 77.8 -> 75.5 us, 16 x 16 171 -> 166, 4 x 16 x 2048 233 -> 229. (At head_dim 128 every register
  // is taken; with dropout, which clears dP before delta joins it, 113 -> 116 us.) delta is a mean of the row's dP, so that no partial sum
  // is larger for it: fp32 error of P (dP - delta), modelled over softmax peaks and means of V, 1.2 to 1.8 times smaller.
  constexpr bool DP_FROM_DELTA = D == 64 && !DROP;
  f32x16 dp_start;
  if constexpr (DP_FROM_DELTA) {
#pragma unroll
    for (int r = 0; r < 16; ++r) dp_start[r] = delta;
    asm volatile("" : "+v"(dp_start));
  }

  for (int tile = 0; tile < n_tiles; ++tile) {
    const int buf = tile & 1;
    const int key0 = tile * kBwdTile;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if constexpr (KBIAS) {
      // (the value fetched one tile ago is used before this tile's copies go out: the wait the compiler puts in front
      // of its use then finds nothing in flight)
      if (wave_s == 0) {
        asm volatile("" : "+v"(key_bias_next));                                  // (the use starts here, not earlier)
        key_bias[(buf ^ 1) * kBwdTile + lane] = key_bias_next * per_scale;       // tile + 1: read after the next barrier
      }
    }
    if (tile + 1 < n_tiles) issue(tile + 1, buf ^ 1);
    if constexpr (KBIAS) {
      if (wave_s == 0) key_bias_next = load_bias<T>(prm.bias, key_bias_row + min((tile + 2) * kBwdTile + lane, Sk - 1));
    }
    if (CAUSAL && key0 > q0w + 31) continue;
    if constexpr (DROP) {
      drop.look(prm.drop, bh, Sq, Sk, q0 + wave_s * 32, tile);
    }
    FO_LDS const char* kt = smem + buf * TILE_BYTES;
    FO_LDS const char* vt = smem + (2 + buf) * TILE_BYTES;

    f32x16 sacc[2], dpacc[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) { sacc[kb][r] = 0.0f; dpacc[kb][r] = DP_FROM_DELTA ? dp_start[r] : 0.0f; }
    if constexpr (KBIAS) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int jv = 0; jv < 4; ++jv) {
          const f32x4 b4 = *(FO_LDS const f32x4*)(key_bias + buf * kBwdTile + 32 * kb + 8 * jv + 4 * hh);
#pragma unroll
          for (int u = 0; u < 4; ++u) sacc[kb][4 * jv + u] = b4[u];
        }
    }
    if constexpr (HALVES) {
      BRH::each(row_bias, 0, l32, hh, [&](int r, float v) { sacc[0][r] = __builtin_fmaf(v, per_scale, row_start); });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // read: the buffer is free for the tile's other half
      BRH::copy(prm.bias, key_bias_row, q0 + wave_s * 32, Sq, Sk, key0 + 32, row_bias, lane);
    } else if constexpr (TBIAS != 0) {
      BR::each(row_bias, 0, l32, hh, [&](int r, float v) { sacc[0][r] = __builtin_fmaf(v, per_scale, row_start); });
      BR::each(row_bias, 1, l32, hh, [&](int r, float v) { sacc[1][r] = __builtin_fmaf(v, per_scale, row_start); });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // read: the buffer is free for the next tile's
      if (tile + 1 < n_tiles) BR::copy(prm.bias, key_bias_row, q0 + wave_s * 32, Sq, Sk, key0 + kBwdTile, row_bias, lane);
    }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        sacc[kb] = Ops<T>::mfma(row_frag<T, D>(kt, kb, ks, l32, hh), qf[ks], sacc[kb]);      // S^T = K Q^T
        dpacc[kb] = Ops<T>::mfma(row_frag<T, D>(vt, kb, ks, l32, hh), gf[ks], dpacc[kb]);    // dP^T = V dO^T
      }
    if constexpr (HALVES) {
      // (behind the products, which cover most of the copy's way; what else is in flight was issued before it)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      BRH::each(row_bias, 0, l32, hh, [&](int r, float v) { sacc[1][r] += __builtin_fmaf(v, per_scale, row_start); });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (tile + 1 < n_tiles) BRH::copy(prm.bias, key_bias_row, q0 + wave_s * 32, Sq, Sk, key0 + kBwdTile, row_bias, lane);
    }
    // register r of block kb holds key key0 + 32*kb + 4*hh + koff(r), koff(r) = (r & 3) + 8 * (r >> 2); dead iff
    // key > q or key >= Sk
    vec8 dsf[4];
    // dropout (flash_attention_triton.py:524-532,599): dP reaches only the kept probabilities
    if constexpr (DROP) {
      if (__builtin_expect(drop.state != kKeepAll, 0)) drop.apply(dpacc);
    }
    // bias row of this lane's query (flash_attention_triton.py:497-509); keys past the end re-read the last one
    const int64_t bias_row = BIAS ? b * prm.bias.strides[0] + h * prm.bias.strides[1] + (int64_t)qrow * prm.bias.strides[2] : 0;
    // (the factor softmax_scale of dS is applied once, to the finished accumulators; tiles that no mask touches - most -
    // go without the comparisons)
    auto softmax_grad = [&](auto masked) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int key_base = key0 + 32 * kb + 4 * hh;
        int lim = key_base - Sk + 1;
        if (CAUSAL) lim = max(lim, key_base - (q0w + l32));
        // registers 4*j .. 4*j + 3 (four consecutive keys), given their bias
        auto four = [&](int j, const float* b4) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int r = 4 * j + u;
            const bool dead = decltype(masked)::value && lim > -(u + 8 * j);
            float shift = row_shift;
            if constexpr (BIAS) shift = __builtin_fmaf(b4[u], kLog2e, -lse2);
            const float p = dead ? 0.0f : __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][r], c, shift));
            dsf[kb * 2 + (r >> 3)][r & 7] = (T)(p * (DP_FROM_DELTA ? dpacc[kb][r] : dpacc[kb][r] + delta));
          }
        };
        // The bias of four keys at a time (few values in flight: this kernel has no registers to spare). From the
        // per-key values staged in LDS; else with one load of four consecutive keys when the tile is complete and the
        // bias is laid out for it; else key by key. Every lane reads its own row, so a load instruction touches 32
        // cache lines either way, and fewer instructions is what counts. The bias type is decided around the loops.
        float b4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (!BIAS) {
#pragma unroll
          for (int j = 0; j < 4; ++j) four(j, b4);
        } else if (bias_keys_staged) {
          FO_LDS const char* bk = bias_keys + buf * 256;
          if (prm.bias.is_f32) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const f32x4 t4 = *(FO_LDS const f32x4*)(bk + (32 * kb + 4 * hh + 8 * j) * 4);
#pragma unroll
              for (int u = 0; u < 4; ++u) b4[u] = t4[u];
              four(j, b4);
            }
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              typedef __attribute__((ext_vector_type(4))) T vec4;
              const vec4 t4 = *(FO_LDS const vec4*)(bk + (32 * kb + 4 * hh + 8 * j) * 2);
#pragma unroll
              for (int u = 0; u < 4; ++u) b4[u] = (float)t4[u];
              four(j, b4);
            }
          }
        } else if (prm.bias.vec_ok && key0 + kBwdTile <= Sk) {
          if (prm.bias.is_f32) {
#pragma unroll
            for (int j = 0; j < 4; ++j) { load_bias4<float>((const float*)prm.bias.ptr + bias_row + key_base + 8 * j, b4); four(j, b4); }
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) { load_bias4<T>((const T*)prm.bias.ptr + bias_row + key_base + 8 * j, b4); four(j, b4); }
          }
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int u = 0; u < 4; ++u) b4[u] = load_bias<T>(prm.bias, bias_row + min(key_base + u + 8 * j, Sk - 1));
            four(j, b4);
          }
        }
      }
    };
    if (key0 + kBwdTile > Sk || (CAUSAL && key0 + kBwdTile - 1 > q0w)) softmax_grad(std::true_type{});
    else softmax_grad(std::false_type{});
    // dQ^T += K^T dS^T : four 16-key steps x DBLK d-blocks
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int db = 0; db < DBLK; ++db) acc[db] = Ops<T>::mfma(col_frag<T, D>(kt, t, db, lane), dsf[t], acc[db]);
  }

  // (straight from the registers, 8 bytes per lane: with two workgroups per CU the other one covers the time these
  // stores take, and staging the rows in LDS as the dK/dV kernels do made this kernel 5-10 % slower)
  const int qi = q0w + l32;
  if (qi < Sq) {
    // -LSE / softmax_scale for the dK/dV kernel, whose score accumulators start from it: P = exp2((QK^T - LSE / scale)
    // * scale * log2 e) is then one multiplication and the exponential per element. (Stored here, from the scaled LSE
    // the loop used, and not beside delta: every register is taken while the loop runs.)
    // (TBIAS: by the factor that kernel scales the bias with)
    if (hh == 0) prm.nlse[(int64_t)bh * Sq + qi] = TBIAS ? row_start : lse2 * prm.neg_inv_scale_log2e;
    T* op = (T*)prm.dq + b * prm.dqs[0] + h * prm.dqs[1] + (int64_t)qi * prm.dqs[2];
#pragma unroll
    for (int db = 0; db < DBLK; ++db)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        typedef __attribute__((ext_vector_type(4))) T vec4;
        vec4 o4;
#pragma unroll
        for (int u = 0; u < 4; ++u) o4[u] = (T)(acc[db][rg * 4 + u] * scale);
        if (32 * db + 8 * rg + 4 * hh < prm.d) *(vec4*)(op + 32 * db + 8 * rg + 4 * hh) = o4;
      }
  }
}

// ---------------------------------------------------------------------------------------------------------------------
template <typename T, int D, bool CAUSAL, bool DROP, bool BIAS>
__global__ void __launch_bounds__(kBwdWaves * 64) attn_bwd_dkdv_kernel(const AttnBwdParams prm) {
  typedef typename Ops<T>::vec8 vec8;
  constexpr int TILE_BYTES = kBwdTile * D * 2;
  constexpr int KSTEPS = D / 16;
  constexpr int DBLK = D / 32;
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  FO_LDS char* smem = (FO_LDS char*)smem_raw;   // Q0 | Q1 | dO0 | dO1 | lse[2][64] | delta[2][64] | bias tiles (BIAS)
  FO_LDS float* rowvals = (FO_LDS float*)(smem + 4 * TILE_BYTES);
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  int bh, kblk;                                       // key block 0 has the most queries when causal: heaviest first
  bwd_item(prm, (prm.Sk + kBwdRows - 1) / kBwdRows, bh, kblk);
  const int b = bh / prm.H, h = bh % prm.H;
  const int k0 = kblk * kBwdRows, k0w = k0 + wave * 32;
  const int Sq = prm.Sq, Sk = prm.Sk;
  const T* qbase = (const T*)prm.q + b * prm.qs[0] + h * prm.qs[1];
  const T* gbase = (const T*)prm.d_o + b * prm.dos[0] + h * prm.dos[1];
  const int n_qt = (Sq + kBwdTile - 1) / kBwdTile;
  const int qt0 = CAUSAL ? min(k0 / kBwdTile, n_qt) : 0;   // queries before the block's first key never attend it

  TileLaneOffsets<T, D> qlo, glo;
  qlo.init(prm.qs[2], prm.d, wave_s, lane);
  glo.init(prm.dos[2], prm.d, wave_s, lane);
  // ---- bias. A lane owns a key and its registers run over queries, so a bias that is the same for every query (query
  // stride 0) is one value per lane for the whole kernel. Otherwise the wave's 64 queries x 32 keys of a tile are
  // copied straight into LDS together with the tile (a load the compiler can see is waited for right where it is
  // issued, together with the tile copies in flight, which then no longer overlap the arithmetic): two buffers of
  // kBiasWaveBytes per wave. A row of the wave's part is 128 bytes (fp32) or 64 bytes (operand type), so one copy
  // instruction of 64 x 16 bytes holds 8 or 16 rows; inside it, row 4*hh + u (+ 8 for the second eight) sits in
  // slot 2*u + hh (+ 8), so that a lane reads register u at a fixed distance from its base and the two halves of
  // a wave, four rows apart, read different banks. Only complete tiles of suitably aligned tensors; the rest reads
  // the bias element by element.
  constexpr int kBiasWaveBytes = kBwdTile * 32 * 4;
  FO_LDS char* bias_lds = (FO_LDS char*)(rowvals + 4 * kBwdTile) + wave_s * 2 * kBiasWaveBytes;
  const bool bias_per_key = BIAS && prm.bias.strides[2] == 0;
  const bool bias_staged = BIAS && !bias_per_key && prm.bias.dma_ok && k0 + wave_s * 32 + 32 <= Sk &&
                           prm.bias.strides[2] > 0 && prm.bias.strides[2] < (1 << 24);   // (32-bit offsets inside a copy instruction)
  float bias_lane = 0.0f;
  if (bias_per_key) bias_lane = load_bias<T>(prm.bias, b * prm.bias.strides[0] + h * prm.bias.strides[1] + min(k0w + l32, Sk - 1)) * kLog2e;
  // (per lane: the byte offset of its piece inside the rows of one copy instruction, added to a uniform base per
  // instruction. Handing base and offset to the copy separately, as a scalar base plus a 32-bit lane offset, left the
  // GPU faulted in this kernel for a reason not found; the per-lane 64-bit pointer is the form that is tested.)
  uint32_t bias_lane_off = 0;
  const char* bias_src = nullptr;
  int64_t bias_row_bytes = 0;
  if (bias_staged) {
    const int elt = prm.bias.is_f32 ? 4 : 2;
    const int g = prm.bias.is_f32 ? lane >> 3 : lane >> 2, piece = prm.bias.is_f32 ? lane & 7 : lane & 3;
    const int row_in = 8 * (g >> 3) + 4 * (g & 1) + ((g >> 1) & 3);   // the row kept in slot g
    bias_row_bytes = prm.bias.strides[2] * elt;
    bias_lane_off = (uint32_t)(row_in * bias_row_bytes + piece * 16);
    bias_src = (const char*)prm.bias.ptr + (b * prm.bias.strides[0] + h * prm.bias.strides[1] + k0 + wave_s * 32) * elt;   // wave-uniform
  }
  auto issue_bias = [&](int qt, int buf) {
    if (!bias_staged || qt * kBwdTile + kBwdTile > Sq) return;
    const int rows_per_dma = prm.bias.is_f32 ? 8 : 16, n_dma = prm.bias.is_f32 ? 8 : 4;
    FO_LDS char* dst = bias_lds + buf * kBiasWaveBytes;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < n_dma) dma16_lane_ptr(bias_src + (int64_t)(qt * kBwdTile + i * rows_per_dma) * bias_row_bytes + bias_lane_off, dst + i * 1024);
  };
  auto issue = [&](int qt, int buf) {
    if constexpr (BIAS) issue_bias(qt, buf);
    if (qt * kBwdTile + kBwdTile <= Sq && qlo.ok && glo.ok) {
      copy_tile64_inside<T, D>(qbase, prm.qs[2], qt * kBwdTile, qlo, smem + buf * TILE_BYTES, wave_s);
      copy_tile64_inside<T, D>(gbase, prm.dos[2], qt * kBwdTile, glo, smem + (2 + buf) * TILE_BYTES, wave_s);
    } else {
      copy_tile64<T, D>(qbase, prm.qs[2], qt * kBwdTile, Sq, prm.d, smem + buf * TILE_BYTES, wave_s, lane);
      copy_tile64<T, D>(gbase, prm.dos[2], qt * kBwdTile, Sq, prm.d, smem + (2 + buf) * TILE_BYTES, wave_s, lane);
    }
    // per-row LSE and delta of the tile, 4 bytes per lane, also straight into LDS (a load the compiler can see would
    // make it wait for the tile copies as well); rows past the end re-read the last row and are masked below
    if (wave_s < 2) {
      const int64_t at = (int64_t)bh * Sq + min(qt * kBwdTile + lane, Sq - 1);
      dma4_lane_ptr((wave_s == 0 ? prm.lse : (const float*)prm.delta) + at, rowvals + (2 * wave_s + buf) * kBwdTile);
    }
  };
  if (qt0 < n_qt) issue(qt0, 0);

  // B operands held for the whole kernel: K^T and V^T fragments of this lane's key
  const int key = k0w + l32;
  const int krow = min(key, Sk - 1);
  vec8 kf[KSTEPS], vf[KSTEPS];
  {
    const T* kp = (const T*)prm.k + b * prm.ks[0] + h * prm.ks[1] + (int64_t)krow * prm.ks[2] + 8 * hh;
    const T* vp = (const T*)prm.v + b * prm.vs[0] + h * prm.vs[1] + (int64_t)krow * prm.vs[2] + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      kf[ks] = *(const vec8*)live_or_zero(kp + 16 * ks, 16 * ks + 8 * hh, prm.d);
      vf[ks] = *(const vec8*)live_or_zero(vp + 16 * ks, 16 * ks + 8 * hh, prm.d);
    }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) asm volatile("" ::"v"(kf[ks]), "v"(vf[ks]));
  }

  f32x16 dkacc[DBLK], dvacc[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) { dkacc[i][r] = 0.0f; dvacc[i][r] = 0.0f; }
  const float c = prm.scale_log2e, scale = prm.scale;

  for (int qt = qt0; qt < n_qt; ++qt) {
    const int buf = (qt - qt0) & 1;
    const int q0t = qt * kBwdTile;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (qt + 1 < n_qt) issue(qt + 1, buf ^ 1);
    FO_LDS const char* qtile = smem + buf * TILE_BYTES;
    FO_LDS const char* gtile = smem + (2 + buf) * TILE_BYTES;
    FO_LDS const float* lse_t = rowvals + buf * kBwdTile;
    FO_LDS const float* del_t = rowvals + (2 + buf) * kBwdTile;
    // dropout: a lane looks at one of the tile's 64 rows, the wave's 32 keys of it as a whole (dropout_run)
    uint64_t rows_keep = ~0ull, rows_mixed = 0;
    if constexpr (DROP) {
      const int run = dropout_run<5>(DropRows<1>::index(prm.drop, bh, Sq, Sk, q0t + lane, k0w), 32, prm.drop.seed, prm.drop.threshold);
      rows_keep = __builtin_amdgcn_ballot_w64(run == kKeepAll);
      rows_mixed = __builtin_amdgcn_ballot_w64(run == kDropMixed);
    }
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      if (CAUSAL && q0t + 32 * qb + 31 < k0w) continue;   // every query of the block is before every key of this wave
      f32x16 sacc, dpacc;
#pragma unroll
      for (int r = 0; r < 16; ++r) { sacc[r] = 0.0f; dpacc[r] = 0.0f; }
      // the staged bias of this block's 16 registers, read ahead of the MFMAs below (read where it is used, each
      // value is waited for on its own): row 32*qb + 8*j + 4*hh + u of the tile sits in copy instruction 4*qb + j
      // (fp32) or 2*qb + j/2 (operand type)
      float bias_reg[BIAS ? 16 : 1];
      const bool bias_from_lds = BIAS && bias_staged && q0t + kBwdTile <= Sq;
      if constexpr (BIAS) {
        if (bias_from_lds) {
          FO_LDS const char* bias_t = bias_lds + buf * kBiasWaveBytes + (prm.bias.is_f32 ? hh * 128 + l32 * 4 : hh * 64 + l32 * 2);
          // (one decision on the bias type around all 16 reads: decided per element, every read gets its own branch
          // and its own wait)
          if (prm.bias.is_f32) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
              for (int u = 0; u < 4; ++u) bias_reg[4 * j + u] = *(FO_LDS const float*)(bias_t + (4 * qb + j) * 1024 + u * 256);
          } else {
            T raw[16];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
              for (int u = 0; u < 4; ++u) raw[4 * j + u] = *(FO_LDS const T*)(bias_t + (2 * qb + (j >> 1)) * 1024 + (j & 1) * 512 + u * 128);
#pragma unroll
            for (int r = 0; r < 16; ++r) bias_reg[r] = (float)raw[r];
          }
        }
      }
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        sacc = Ops<T>::mfma(row_frag<T, D>(qtile, qb, ks, l32, hh), kf[ks], sacc);      // S = Q K^T
        dpacc = Ops<T>::mfma(row_frag<T, D>(gtile, qb, ks, l32, hh), vf[ks], dpacc);    // dP = dO V^T
      }
      // register r holds query q0t + 32*qb + 4*hh + koff(r), koff(r) = (r & 3) + 8 * (r >> 2); dead iff key > query
      // or the query is past the end
      const int lim = CAUSAL ? key - (q0t + 32 * qb + 4 * hh) : 0;
      const int lim_end = Sq - (q0t + 32 * qb + 4 * hh);
      vec8 pf[2], dsf[2];
      // dropout (flash_attention_triton.py:524-532,551-552): dV sees the kept probabilities, dP reaches them only. Where all
      // or none of the block's elements are kept (nearly always) that is one factor, else a bit per register.
      uint32_t keep_bits = 0xFFFFFFFFu;
      float keep_all = 1.0f;
      bool keep_each = false;
      if constexpr (DROP) {
        const uint32_t k32 = (uint32_t)(rows_keep >> (32 * qb)), m32 = (uint32_t)(rows_mixed >> (32 * qb));
        keep_each = m32 != 0 || (k32 != 0 && k32 != 0xFFFFFFFFu);
        keep_all = k32 != 0 ? 1.0f : 0.0f;
        if (keep_each) {
          const uint32_t first = DropRows<1>::index(prm.drop, bh, Sq, Sk, q0t + 32 * qb + 4 * hh, key);
          keep_bits = 0;
#pragma unroll
          for (int r = 0; r < 16; ++r)
            keep_bits |= (dropout_keep(first + (uint32_t)((r & 3) + 8 * (r >> 2)) * (uint32_t)Sk, prm.drop.seed, prm.drop.threshold) ? 1u : 0u) << r;
        }
      }
      // bias column of this lane's key; queries past the end re-read the last one
      const int64_t bias_col = BIAS ? b * prm.bias.strides[0] + h * prm.bias.strides[1] + krow : 0;
      // where the bias comes from: 0 global memory, element by element; 1 the lane's own value; 2 the staged tile
      auto softmax_grad_of = [&](auto masked, auto bias_mode, auto each) {
      constexpr int BM = decltype(bias_mode)::value;
      constexpr bool EACH = decltype(each)::value;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 l4 = *(FO_LDS const f32x4*)(lse_t + 32 * qb + 8 * j + 4 * hh);
        const f32x4 d4 = *(FO_LDS const f32x4*)(del_t + 32 * qb + 8 * j + 4 * hh);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int r = 4 * j + u;
          const bool dead = decltype(masked)::value && ((u + 8 * j) < lim || (u + 8 * j) >= lim_end);
          float shift = DROP ? __builtin_fmaf(-l4[u], kLog2e, prm.drop.keep_log2) : -l4[u] * kLog2e;      // (P times 1 / (1 - p): see the dQ kernel)
          if constexpr (BIAS && BM == 0) {
            const int qi = min(q0t + 32 * qb + 4 * hh + u + 8 * j, Sq - 1);
            shift = __builtin_fmaf(load_bias<T>(prm.bias, bias_col + (int64_t)qi * prm.bias.strides[2]), kLog2e, shift);
          }
          if constexpr (BIAS && BM == 1) shift += bias_lane;
          if constexpr (BIAS && BM == 2) shift = __builtin_fmaf(bias_reg[r], kLog2e, shift);
          const float p = dead ? 0.0f : __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[r], c, shift));
          float pd = p, dp = dpacc[r];
          if constexpr (DROP) {
            const float z = EACH ? (float)((keep_bits >> r) & 1u) : keep_all;
            pd = p * z;
            dp = dp * z;
          }
          pf[r >> 3][r & 7] = (T)pd;
          dsf[r >> 3][r & 7] = (T)(p * (dp + d4[u]));   // (d4 = -delta) softmax_scale is applied to the finished dK
        }
      }
      };
      auto softmax_grad = [&](auto masked, auto bias_mode) {
        if constexpr (DROP) {
          if (keep_each) { softmax_grad_of(masked, bias_mode, std::true_type{}); return; }
        }
        softmax_grad_of(masked, bias_mode, std::false_type{});
      };
      const bool needs_mask = q0t + 32 * qb + 32 > Sq || (CAUSAL && k0w + 31 > q0t + 32 * qb);
      typedef std::integral_constant<int, 0> BM0;
      typedef std::integral_constant<int, 1> BM1;
      typedef std::integral_constant<int, 2> BM2;
      if constexpr (!BIAS) {
        if (needs_mask) softmax_grad(std::true_type{}, BM0{}); else softmax_grad(std::false_type{}, BM0{});
      } else if (bias_per_key) {
        if (needs_mask) softmax_grad(std::true_type{}, BM1{}); else softmax_grad(std::false_type{}, BM1{});
      } else if (bias_from_lds) {
        if (needs_mask) softmax_grad(std::true_type{}, BM2{}); else softmax_grad(std::false_type{}, BM2{});
      } else {
        if (needs_mask) softmax_grad(std::true_type{}, BM0{}); else softmax_grad(std::false_type{}, BM0{});
      }
      // dV^T += dO^T P and dK^T += Q^T dS : two 16-query steps x DBLK d-blocks
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int db = 0; db < DBLK; ++db) {
          dvacc[db] = Ops<T>::mfma(col_frag<T, D>(gtile, 2 * qb + t, db, lane), pf[t], dvacc[db]);
          dkacc[db] = Ops<T>::mfma(col_frag<T, D>(qtile, 2 * qb + t, db, lane), dsf[t], dkacc[db]);
        }
    }
  }

  // (the tile buffers are free once every wave is past its last tile; dK, then dV, through the wave's own piece of them)
  __syncthreads();
  {
    FO_LDS char* stage = smem + wave_s * stage_bytes(D);
    const int k0w_s = k0 + wave_s * 32;
    store_rows_via_lds<T, D>(dkacc, scale, stage, (T*)prm.dk + b * prm.dks[0] + h * prm.dks[1], prm.dks[2], k0w_s, Sk, prm.d, lane);
    store_rows_via_lds<T, D>(dvacc, 1.0f, stage, (T*)prm.dv + b * prm.dvs[0] + h * prm.dvs[1], prm.dvs[2], k0w_s, Sk, prm.d, lane);
  }
}

// 16 bytes per lane to a wave-uniform address + byte_off + IMM. (Inline assembly: nothing waits for it. A VALU instruction that
// writes the data registers may not follow a store of more than 8 bytes at once, which the compiler does not see here: hence the wait states.)
template <int IMM, typename V>
__device__ __forceinline__ void store16_uniform_base(char* base, uint32_t byte_off, V data) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("global_store_dwordx4 %0, %1, %2 offset:%3 nt\n\ts_nop 1" ::"v"(byte_off), "v"(data), "s"(base), "n"(IMM) : "memory");
#endif
}

// ---------------------------------------------------------------------------------------------------------------------
// The softmax-gradient jobs of one tile of the pipelined dK/dV kernel (see its tile_body): 48 slots, slot s = eight per
// half-phase from the second half of phase 1 on. stage 0 = A of element r (P = exp2(S c)), stage 1 = B of elements r and
// r + 1 (dS = P dP, both rounded) of query block qb.
struct SoftmaxGradJob { int stage, qb, r; };
constexpr SoftmaxGradJob softmax_grad_job(int s) {
  const int h = s / 8, u = s % 8;
  if (h == 0) return {0, 0, u};
  if (h == 1) return {0, 0, 8 + u};
  if (h == 2) return u < 4 ? SoftmaxGradJob{1, 0, 2 * u} : SoftmaxGradJob{0, 1, u - 4};
  if (h == 3) return u < 4 ? SoftmaxGradJob{1, 0, 8 + 2 * u} : SoftmaxGradJob{0, 1, u};
  if (h == 4) return u < 4 ? SoftmaxGradJob{1, 1, 2 * u} : SoftmaxGradJob{0, 1, 4 + u};
  return u < 4 ? SoftmaxGradJob{0, 1, 12 + u} : SoftmaxGradJob{1, 1, 8 + 2 * (u - 4)};
}
// Every element gets each stage once; a job runs behind the MFMA of its group, so stage A of block qb needs a group
// after the block's last S MFMA, stage B one after its last dP MFMA and a slot after the A jobs of its two elements, and
// the B operands of elements 8t .. 8t+7 must be complete in a group before the first gradient MFMA that reads them.
// (The wait states these distances need in instructions are checked on the generated code, fast_ops_amd/asm_lint.py.)
// the group of a half-phase (of nmf / 2 groups) in which its slot u of eight runs
constexpr int softmax_grad_slot_group(int u, int nmf) { return u * (nmf / 2) / 8; }
constexpr bool softmax_grad_jobs_fit(int nmf) {
  const int half = nmf / 2, ksteps = nmf / 2;
  int slot_a[2][16] = {}, slot_b[2][16] = {}, n_a[2][16] = {}, n_b[2][16] = {};
  for (int s = 0; s < 48; ++s) {
    const SoftmaxGradJob j = softmax_grad_job(s);
    if (j.qb < 0 || j.qb > 1 || j.r < 0 || j.r + j.stage > 15) return false;
    if (j.stage == 0) { slot_a[j.qb][j.r] = s; ++n_a[j.qb][j.r]; }
    else { slot_b[j.qb][j.r] = slot_b[j.qb][j.r + 1] = s; ++n_b[j.qb][j.r]; ++n_b[j.qb][j.r + 1]; }
  }
  for (int qb = 0; qb < 2; ++qb)
    for (int r = 0; r < 16; ++r) {
      if (n_a[qb][r] != 1 || n_b[qb][r] != 1) return false;
      // the groups the jobs run in
      const int ga = half + slot_a[qb][r] / 8 * half + softmax_grad_slot_group(slot_a[qb][r] % 8, nmf);
      const int gb = half + slot_b[qb][r] / 8 * half + softmax_grad_slot_group(slot_b[qb][r] % 8, nmf);
      if (ga < qb * nmf + ksteps) return false;                                          // S complete
      if (gb < (qb + 1) * nmf || slot_b[qb][r] <= slot_a[qb][r]) return false;           // dP complete, P there
      if (gb >= (2 + qb) * nmf + (r / 8) * half) return false;                           // before its first reader
    }
  return true;
}
static_assert(softmax_grad_jobs_fit(16) && softmax_grad_jobs_fit(12) && softmax_grad_jobs_fit(8), "128, 96 and 64 columns");

// ---------------------------------------------------------------------------------------------------------------------
// dK/dV as a software pipeline. The accumulators of dK and dV, the K^T and V^T fragments and
// two blocks of scores leave room for one wave per SIMD only, and a lone wave issues in order: whatever arithmetic sits
// between two MFMAs keeps the matrix pipe waiting unless it is laid out to run beside them. A 64-query tile is two
// 32-query blocks and four phases of NMF MFMAs each:
//   1: S, then dP of block 0 | 2: S, then dP of block 1 | 3: dV, dK of block 0 | 4: dV, dK of block 1
// as micro-groups of one MFMA, the LDS read of the A operand needed kFragAhead groups later and a share of the tile's
// softmax-gradient arithmetic (see tile_body), fenced so that the compiler keeps the groups apart. The accumulators of
// S and dP do not start from zero but from -LSE / scale and -delta of their rows (written by the launch before, read from
// LDS straight into the registers while they are idle), so that P = exp2((QK^T - LSE / scale) c) and dS = P (dP - delta)
// are two multiplications and the exponential.
// KBIAS: with a bias that is the same for every query (query stride 0): a lane owns a key, so the bias is one value per
// lane for the whole kernel, and P = exp2(S c + b log2 e) is a fused multiply-add where the form without bias multiplies.
// DROP (flash_attention_triton.py:524-532,551-552): dV sees the kept probabilities only, and dP reaches only them: where a
// query's elements of the workgroup's 128 keys are all dropped, its row of the dO tile in LDS is set to zero, which is both
// (dP = dO V^T and dV = dO^T P), and where they are all kept there is nothing to do; 1 / (1 - p) is part of P (-LSE / scale
// comes with it, and delta multiplied by 1 - p: see the dQ kernel). Each lane looks at one of the next tile's 64 rows as a
// whole (dropout_run) in the first groups of a tile, which carry no other arithmetic. A row that is neither (a few in a
// million) counts as dropped at first. At the end the workgroup's rows of this kind, up to 64 at a time, are gathered into
// one tile, which goes through the body once more with P of dropped elements set to zero and dP taken without delta: that
// adds just what is missing. (DS: dS of those elements is written anew, whole and rounded once, for dQ.) (A tile for each of them: 232 us at 12 heads x 4096 keys, of which 30 us were waited for.)
// Whole backward at p = 0.1, with every element hashed in the plain kernel -> this: 12 heads x 4096 keys at head_dim 128
// 631 -> 391 us (no dropout 387), x 8192 1957 -> 1290 (1209), x 2048 causal 187 -> 119 (105); head_dim 64, 8 x 12 heads x
// 1024 causal 139 -> 74 (71).
// PAD, LIVE: a head_dim below D, as in the dQ kernel (96 columns: the phases are 12 groups long, with one or two slots each).
// TBIAS: a bias with a query stride, of so many bytes per element (2 or 4). The wave's 64 queries x 32 keys of tile j+2 are
// copied into LDS with that tile, two buffers; a block's values, read transposed (a lane owns a key), are added to the start
// of its S accumulators in groups that carry little else: S + (b - LSE) / scale then comes out of the MFMAs. Two fp32 tiles per
// wave do not fit beside the rings of head_dim 128 (by 1.5 KiB of 160): there it is three buffers of half a tile (32 queries),
// of which tile j+2's second half takes the one that held the first half of tile j+1, half a phase after that was read.
// DS: dS is kept for attn_bwd_dq_of_ds_kernel (ds_chunk), and several workgroups may share a block's query tiles (prm.items). A tile's four pieces per wave are stored in the first groups of the next
// tile, which carry no other arithmetic and come behind every copy that the next hand-over waits for: that one then waits
// for all but the last four of the wave's memory operations, which complete in order. The stores carry nt: nothing of this kernel
// reads them, and they would push Q and dO out of the cache (12 heads x 4096 not causal: 204 us without DS, 230 with plain stores, 217
// with nt; 64 heads x 2048 causal 143, 166, 155).
// SHIFT (DS without TBIAS): dQ is made of this kernel's P then, and P has to be as exact as the dQ kernel's own. So S starts from zero (KBIAS: from
// bias / scale, sixteen registers that stay as they are), and -LSE log2 e, read from LDS where -LSE / scale is otherwise, joins in the exponent:
// P = exp2(S c + shift), a fused multiply-add in the place of the multiplication. Started from -LSE / scale, S is summed at the ulp of the LSE: fp32
// error of P at 4096 unit normal keys 7.4e-7 rms instead of 3.0e-7. (This kernel alone, start values -> shift, over several runs in turn: 12 heads x
// 4096 with key bias and dropout 269-291 -> 272-283 us, without 224-237 -> 227-234, 12 x 3072 causal 70-73 -> 72-74, 48 x 1450 x 1100 at head_dim 96 83 -> 84.)
template <typename T, int D, bool CAUSAL, bool KBIAS = false, bool DROP = false, bool PAD = false, int LIVE = D, int TBIAS = 0, bool DS = false>
__global__ void __launch_bounds__(kBwdWaves * 64) attn_bwd_dkdv_pipe_kernel(const AttnBwdParams prm) {
  static_assert(TBIAS == 0 || !(KBIAS || DROP || PAD), "not combined");
  static_assert(!(PAD && (DROP || KBIAS)), "the second visit of dropout's rows copies whole rows");
  constexpr bool SHIFT = DS && TBIAS == 0;
  typedef typename Ops<T>::vec8 vec8;
  constexpr int TILE_BYTES = kBwdTile * D * 2;
  constexpr int KSTEPS = LIVE / 16;
  constexpr int DBLK = LIVE / 32;
  constexpr int NMF = 2 * KSTEPS;           // MFMAs per phase (= 4 * DBLK)
  static_assert(4 * DBLK == NMF, "phases of equal length");
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  constexpr int NBUF = 3;                   // tile buffers: see hand_over()
  FO_LDS char* smem = (FO_LDS char*)smem_raw;   // Q[NBUF] | dO[NBUF] | -LSE/scale[NBUF][64] | -delta[NBUF][64]
  FO_LDS float* rowvals = (FO_LDS float*)(smem + 2 * NBUF * TILE_BYTES);
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  int bh, kblk;                                       // key block 0 has the most queries when causal: heaviest first
  [[maybe_unused]] uint32_t item = kWholeBlock;       // DS: the piece of the block's query tiles this workgroup takes
  if (DS && prm.n_items > 0) {
    const int n_bh = prm.B * prm.H, e = blockIdx.x / n_bh;
    bh = blockIdx.x - e * n_bh;
    item = prm.items[e];
    kblk = item & 255u;
  } else {
    bwd_item(prm, (prm.Sk + kBwdRows - 1) / kBwdRows, bh, kblk);
  }
  const int b = bh / prm.H, h = bh % prm.H;
  const int k0 = kblk * kBwdRows, k0w = k0 + wave_s * 32;
  const int Sq = prm.Sq, Sk = prm.Sk;
  const T* qbase = (const T*)prm.q + b * prm.qs[0] + h * prm.qs[1];
  const T* gbase = (const T*)prm.d_o + b * prm.dos[0] + h * prm.dos[1];
  int n_qt = (Sq + kBwdTile - 1) / kBwdTile;                 // the workgroup's query tiles are [qt0, n_qt)
  int qt0 = CAUSAL ? min(k0 / kBwdTile, n_qt) : 0;           // queries before the block's first key never attend it
  if constexpr (DS) {
    const int pieces = (item >> 12) & 15, piece = (item >> 8) & 15, len = n_qt - qt0;
    n_qt = qt0 + len * (piece + 1) / pieces;
    qt0 += len * piece / pieces;
  }
  const int ja = CAUSAL ? min(max(k0w / kBwdTile, qt0), n_qt) : qt0;     // ... and this wave's keys start later still

  TileLaneOffsets<T, D> qlo, glo;
  qlo.init(prm.qs[2], PAD ? D : prm.d, wave_s, lane);
  glo.init(prm.dos[2], PAD ? D : prm.d, wave_s, lane);
  // (PAD: the first tile, and the K and V rows that go through the other two buffers below, zero the columns past head_dim)
  TileLiveLanes<T, D> live;
  if constexpr (PAD) live.init(prm.d, wave_s, lane);
  // TBIAS: the wave's tile of the bias, 64 rows x 32 keys, as it lies in memory; needs what BiasRows needs
  constexpr int BELT = TBIAS == 4 ? 4 : 2, BROW = 32 * BELT, BTILE = kBwdTile * BROW, BPIECES = BTILE / 1024, BROWS = 1024 / BROW, BLANES = BROW / 16;
  constexpr bool HALVES = TBIAS == 4 && D == 128;
  FO_LDS char* bias_lds = (FO_LDS char*)(rowvals + 2 * NBUF * kBwdTile) + wave_s * tile_bias_bytes<TBIAS, D>();
  // where the 32 queries qb of tile qt lie
  auto bias_half = [&](int qt, int qb) -> FO_LDS char* {
    return bias_lds + (HALVES ? (uint32_t)(2 * qt + qb) % 3u * (BTILE / 2) : (uint32_t)(qt & 1) * BTILE + qb * (BTILE / 2));
  };
  const char* bias_lane_ptr = nullptr;       // the lane's piece of row lane / BLANES
  int64_t bias_row_bytes = 0;
  if constexpr (TBIAS != 0) {
    bias_row_bytes = prm.bias.strides[2] * BELT;
    const int col = min(k0w + (lane % BLANES) * (16 / BELT), (Sk - 1) / (16 / BELT) * (16 / BELT));
    bias_lane_ptr = (const char*)prm.bias.ptr + (b * prm.bias.strides[0] + h * prm.bias.strides[1] + col) * BELT + (lane / BLANES) * bias_row_bytes;
  }
  auto issue_bias_half = [&](int qt, int qb) {
    FO_LDS char* dst = bias_half(qt, qb);
    if (qt * kBwdTile + kBwdTile <= Sq) {
#pragma unroll
      for (int i = 0; i < BPIECES / 2; ++i) dma16_lane_ptr(bias_lane_ptr + (int64_t)(qt * kBwdTile + 32 * qb + i * BROWS) * bias_row_bytes, dst + i * 1024);
    } else {
      // (queries past the end re-read the last one; masked)
#pragma unroll
      for (int i = 0; i < BPIECES / 2; ++i)
        dma16_lane_ptr(bias_lane_ptr + (int64_t)(min(qt * kBwdTile + 32 * qb + i * BROWS + lane / BLANES, Sq - 1) - lane / BLANES) * bias_row_bytes, dst + i * 1024);
    }
  };
  auto issue_bias = [&](int qt) {
    if (qt < ja) return;                     // (causal: this wave's keys start later)
    issue_bias_half(qt, 0);
    if (!HALVES || qt == ja) issue_bias_half(qt, 1);      // HALVES: see where the first half of the tile before is read
  };
  auto issue = [&](int qt, int buf) {
    if constexpr (TBIAS != 0) issue_bias(qt);
    if (PAD && qt > qt0 && qt * kBwdTile + kBwdTile <= Sq && qlo.ok && glo.ok) {
      copy_tile64_inside<T, D>(qbase, prm.qs[2], qt * kBwdTile, qlo, live, smem + buf * TILE_BYTES, wave_s);
      copy_tile64_inside<T, D>(gbase, prm.dos[2], qt * kBwdTile, glo, live, smem + (NBUF + buf) * TILE_BYTES, wave_s);
    } else if (!PAD && qt * kBwdTile + kBwdTile <= Sq && qlo.ok && glo.ok) {
      copy_tile64_inside<T, D>(qbase, prm.qs[2], qt * kBwdTile, qlo, smem + buf * TILE_BYTES, wave_s);
      copy_tile64_inside<T, D>(gbase, prm.dos[2], qt * kBwdTile, glo, smem + (NBUF + buf) * TILE_BYTES, wave_s);
    } else {
      copy_tile64<T, D>(qbase, prm.qs[2], qt * kBwdTile, Sq, prm.d, smem + buf * TILE_BYTES, wave_s, lane);
      copy_tile64<T, D>(gbase, prm.dos[2], qt * kBwdTile, Sq, prm.d, smem + (NBUF + buf) * TILE_BYTES, wave_s, lane);
    }
    if (wave_s < 2) {
      const int64_t at = (int64_t)bh * Sq + min(qt * kBwdTile + lane, Sq - 1);
      dma4_lane_ptr((wave_s == 0 ? (const float*)prm.nlse : (const float*)prm.delta) + at, rowvals + (NBUF * wave_s + buf) * kBwdTile);
    }
  };
  if (qt0 < n_qt) issue(qt0, 0);
  // hand-over j, between phases 3 and 4 of tile j: tile j+1 (copy started one tile ago) has landed for everyone, and
  // since everyone is past phase 3 of tile j nobody reads tile j-1 any more, whose buffer - the third one - takes the
  // copy of tile j+2. Phase 4 still reads tile j, and already fetches the first fragments of tile j+1, so the fragment
  // pipeline never drains. Every wave runs hand-overs qt0-1 .. n_qt-2, each exactly once.
  // Dropout: the rows of tile j+1 that are kept (one bit each) when tile j is handed over, and the tiles that have rows
  // which are neither kept nor dropped, one bit for every 2^again_shift tiles.
  uint64_t next_keep = ~0ull, next_mixed = 0, again = 0;
  int again_shift = 0;
  if constexpr (DROP) { while ((n_qt >> again_shift) >= 64) ++again_shift; }
  auto drop_verdict = [&](int a, int b) {
    next_keep = __builtin_amdgcn_ballot_w64(a == kKeepAll && b == kKeepAll);
    next_mixed = ~(next_keep | __builtin_amdgcn_ballot_w64(a == kDropAll && b == kDropAll));
  };
  auto drop_index = [&](int j) -> uint32_t { return DropRows<1>::index(prm.drop, bh, Sq, Sk, j * kBwdTile + lane, k0); };
  auto drop_look = [&](int j) {          // (outside the tile bodies)
    const uint32_t first = drop_index(j);
    drop_verdict(dropout_block<7>(first, prm.drop.seed, prm.drop.threshold), dropout_block<7>(first + 127u, prm.drop.seed, prm.drop.threshold));
  };
  // this wave's pieces of tile j+1 (in buffer `buf`) have landed, nobody reads it yet: rows of dO that are not kept become zero
  auto drop_rows = [&](int j, int buf) {
    if (__builtin_expect(next_keep != ~0ull, 0)) {
      constexpr int N = TileLaneOffsets<T, D>::N, CHUNKS = D * 2 / 16, ROWS_PER_DMA = 1024 / (D * 2);
      typedef __attribute__((ext_vector_type(4))) int i32x4;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int row = (wave_s * N + i) * ROWS_PER_DMA + lane / CHUNKS;
        if (!((next_keep >> row) & 1)) *(FO_LDS i32x4*)(smem + (NBUF + buf) * TILE_BYTES + (wave_s * N + i) * 1024 + lane * 16) = i32x4{0, 0, 0, 0};
      }
      if (next_mixed != 0) again |= 1ull << ((j + 1) >> again_shift);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  };
  auto hand_over = [&](int j, auto behind) {      // `behind`: memory operations of this wave that nobody waits for yet
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(behind)::value) : "memory");
    if constexpr (DROP) drop_rows(j, (j + 1 - qt0) % NBUF);
    __builtin_amdgcn_s_barrier();
    if (j + 2 < n_qt) issue(j + 2, (j + 2 - qt0) % NBUF);
  };

  // B operands held for the whole kernel: K^T and V^T fragments of this lane's key. The block's 128 rows of K and of V
  // come in like tiles - 16-byte pieces straight into LDS, into the buffers of the second and third tile, which are
  // still free - and each lane takes its row's pieces from there. (Read from global memory row by row, 32 rows per
  // instruction, this took 4.4 us, a quarter of a workgroup's time at 512 queries.) Rows past the end re-read the
  // last one, as the masks below expect. The barrier of the first hand-over comes after every wave has its fragments.
  vec8 kf[KSTEPS], vf[KSTEPS];
  {
    const T* kbase = (const T*)prm.k + b * prm.ks[0] + h * prm.ks[1];
    const T* vbase = (const T*)prm.v + b * prm.vs[0] + h * prm.vs[1];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      copy_tile64<T, D>(kbase, prm.ks[2], k0 + 64 * half, Sk, prm.d, smem + (1 + half) * TILE_BYTES, wave_s, lane);
      copy_tile64<T, D>(vbase, prm.vs[2], k0 + 64 * half, Sk, prm.d, smem + (NBUF + 1 + half) * TILE_BYTES, wave_s, lane);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    FO_LDS const char* kt = smem + (1 + (wave_s >> 1)) * TILE_BYTES;
    FO_LDS const char* vt = smem + (NBUF + 1 + (wave_s >> 1)) * TILE_BYTES;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) { kf[ks] = row_frag<T, D>(kt, wave_s & 1, ks, l32, hh); vf[ks] = row_frag<T, D>(vt, wave_s & 1, ks, l32, hh); }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) asm volatile("" ::"v"(kf[ks]), "v"(vf[ks]));
  }
  const int key = k0w + l32;
  float bias_lane = 0.0f;
  if constexpr (KBIAS) {
    bias_lane = load_bias<T>(prm.bias, b * prm.bias.strides[0] + h * prm.bias.strides[1] + min(key, Sk - 1)) * (SHIFT ? kLog2e / prm.scale_log2e : kLog2e);
    asm volatile("" : "+v"(bias_lane));      // (waited for here, not inside the loops, where copies are in flight)
  }
  f32x16 dkacc[DBLK], dvacc[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) { dkacc[i][r] = 0.0f; dvacc[i][r] = 0.0f; }
  const float c = prm.scale_log2e, scale = prm.scale;

  // Per-lane byte offsets of the fragment reads inside a tile, swizzle included (what row_frag / col_frag compute; the
  // swizzle of a row does not depend on the 32-row block or 16-row step it is in). With the tile's base added once
  // per tile every read is register + immediate: block, step and the dO tiles (NBUF tiles behind the Q tiles) are
  // immediates.
  constexpr int ROW = D * 2;
  constexpr int G_OFF = NBUF * TILE_BYTES;
  uint32_t row_off[KSTEPS], col_off[DBLK][2];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) row_off[ks] = (uint32_t)(l32 * ROW + (((2 * ks + hh) ^ swz<D>(l32)) * 16));
  {
    const int L16 = lane & 15, g16 = (lane >> 4) & 1;
    const int r0 = 4 * hh + (L16 >> 2), r1 = r0 + 8, sub = (L16 & 1) * 8;
#pragma unroll
    for (int db = 0; db < DBLK; ++db) {
      const int chunk = 4 * db + 2 * g16 + ((L16 & 3) >> 1);
      col_off[db][0] = (uint32_t)(r0 * ROW + ((chunk ^ swz<D>(r0)) * 16) + sub);
      col_off[db][1] = (uint32_t)(r1 * ROW + ((chunk ^ swz<D>(r1)) * 16) + sub);
    }
  }
  // A operand of MFMA i of a scores phase (i < KSTEPS: Q rows for S, then dO rows for dP) / of a gradient phase (even i:
  // dO^T for dV, odd i: Q^T for dK); rq / cq = the offsets above plus the byte offset of the tile's Q buffer
  auto scores_frag_sd = [&](const uint32_t* rq, int qb, int i) -> vec8 {
    return *(FO_LDS const vec8*)(smem + rq[i % KSTEPS] + (i >= KSTEPS ? G_OFF : 0) + qb * 32 * ROW);
  };
  auto grads_frag = [&](const uint32_t (*cq)[2], int qb, int i) -> vec8 {
    const int tp = 2 * qb + i / (2 * DBLK), db = (i >> 1) % DBLK;
    const int imm = ((i & 1) ? 0 : G_OFF) + 16 * tp * ROW;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FO_LDS s16x4*)(smem + cq[db][0] + imm));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FO_LDS s16x4*)(smem + cq[db][1] + imm));
    return __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  constexpr int kFragAhead = 4;
  static_assert((4 * NMF) % kFragAhead == 0, "the fragment ring runs on across tiles");
  vec8 fr[kFragAhead];         // A operands, fetched kFragAhead micro-groups ahead of their MFMA
  f32x16 sacc[2], dpacc[2];
  [[maybe_unused]] f32x16 shift[2];       // SHIFT: what the exponent of the rows of a block starts from
  [[maybe_unused]] f32x16 bias_start;     // ... and the key's bias / softmax_scale, from which S does, in every register (as in the dQ kernel)
  if constexpr (SHIFT && KBIAS) {
#pragma unroll
    for (int r = 0; r < 16; ++r) bias_start[r] = bias_lane;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(bias_start));   // (sixteen registers, not one)
#endif
  }
  // P and dS as B operands: pairs of 16-bit values, kept as 32-bit words so that a finished pair can be pinned
  typedef __attribute__((ext_vector_type(4))) int i32x4;
  typedef __attribute__((ext_vector_type(2))) T vec2;
  i32x4 pf[2][2], dsf[2][2];
  // DS: this wave's chunks (of tile 0 on), and the lane's place in the two kinds of pieces of one (see ds_chunk)
  char* ds_wave = nullptr;
  uint32_t ds_off[2] = {0, 0};
  [[maybe_unused]] const int64_t ds_tile_bytes = ds_key_blocks(Sk) * kDsChunk;
  if constexpr (DS) {
    ds_wave = prm.ds + ds_chunk(prm, bh, k0w / 32, 0);
#pragma unroll
    for (int t = 0; t < 2; ++t) ds_off[t] = (uint32_t)(1024 * t + ((l32 ^ (4 * t)) * 32) + 16 * hh);
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int t = 0; t < 2; ++t) dsf[qb][t] = i32x4{0, 0, 0, 0};
  }

  [[maybe_unused]] auto zero_acc = [](f32x16& acc) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_nop 1" : "+v"(acc));       // (pinned here: sunk to the first MFMA, the moves would be too close to it)
#endif
  };

  // TBIAS: the lane's 16 values of a block, then, times 1 / softmax_scale, added to the block's S accumulator one by one (the same
  // factor, to the last bit, as in the dQ kernel: -LSE / scale comes times it)
  const float per_scale = TBIAS ? __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, kLog2e / prm.scale_log2e))) : 0.0f;
  s16x4 bias16[4];
  f32x16 bias32;
  auto bias_read = [&](int jt, int qb) {
    FO_LDS const char* src = bias_half(jt, qb);
#pragma unroll
    for (int jv = 0; jv < 4; ++jv) {
      if constexpr (BELT == 2) {
        bias16[jv] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FO_LDS s16x4*)(src + (8 * jv + 4 * hh + ((lane & 15) >> 2)) * BROW + ((lane >> 4) & 1) * 32 + (lane & 3) * 8));
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) bias32[4 * jv + u] = *(FO_LDS const float*)(src + (8 * jv + 4 * hh + u) * BROW + l32 * 4);
      }
    }
  };
  auto bias_add = [&](f32x16& acc, int e) {
    float v;
    if constexpr (BELT == 2) {
      const short raw = bias16[e >> 2][e & 3];
      v = (float)__builtin_bit_cast(T, raw);
    } else {
      v = bias32[e];
    }
    float sum = __builtin_fmaf(v, per_scale, acc[e]);
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(sum));            // (pinned to its group, see stage_b)
#endif
    acc[e] = sum;
  };

  const uint32_t lane4 = (uint32_t)lane * 4u;
  // One tile. `buf`: the tile's buffer, (j - qt0) % NBUF, which the caller counts along. `spread`: tile j+2 lies wholly
  // inside Q and dO (and the lane offsets fit): its copy is not issued in one batch at the hand-over but one instruction
  // at a time between the MFMAs of phase 4 (a batch of direct-to-LDS copies holds the wave's issue port for hundreds of
  // cycles while the matrix pipe runs dry; one copy per two MFMAs hides behind them).
  // The softmax-gradient arithmetic is spread evenly over the tile's micro-groups: a lone wave hides about five VALU
  // instructions behind a 32-cycle MFMA (an exponential counts as four) and pays in full for every further one, and with
  // a whole score element (multiply, exponential, multiply, rounding) beside each MFMA of phases 2 and 3 and nothing
  // beside those of phases 1 and 4, half of the groups ran at 1.7-2x the MFMA time. So the scores of a block come first
  // (S: KSTEPS MFMAs, then dP: KSTEPS MFMAs), an element is split into stage A (P = exp2(S c), needs S only) and stage B
  // (dS = P dP, both rounded to B operands; two elements at a time), and the 32 A and 16 B jobs of a tile fill 48 slots
  // laid over the groups from the middle of phase 1 to the middle of phase 4 (one slot per group at head_dim 128, two at
  // 64) in an order that meets every producer and consumer (dK/dV kernel: -12 % cycles, -5.5 % time at head_dim 128):
  //   half-phase   MFMAs            slots
  //   0            S0               -
  //   1            dP0              A0[0..7]
  //   2            S1               A0[8..15]
  //   3            dP1              B0[0..7], A1[0..3]
  //   4            dV0,dK0 (t=0)    B0[8..15], A1[4..7]
  //   5            dV0,dK0 (t=1)    B1[0..7], A1[8..11]
  //   6            dV1,dK1 (t=0)    A1[12..15], B1[8..15]
  //   7            dV1,dK1 (t=1)    -
  [[maybe_unused]] FO_LDS int* gathered = (FO_LDS int*)(rowvals + kBwdTile);       // (in the place of the second tile's -LSE / scale)
  auto tile_body = [&](int j, int buf, auto masked, auto spread, auto once_more) __attribute__((always_inline)) {
    constexpr bool SPREAD = decltype(spread)::value;
    constexpr bool AGAIN = decltype(once_more)::value;      // dropout: only the kept elements of rows that are partly dropped
    int drop_a = kKeepAll, drop_b = kKeepAll;
    uint32_t drop_first = 0;
    constexpr int HALF = NMF / 2, NG = 4 * NMF;      // groups per half-phase / per tile
    static_assert(kFragAhead <= KSTEPS && softmax_grad_jobs_fit(NMF), "48 slots over the groups of six half-phases");
    const int nbuf = buf == NBUF - 1 ? 0 : buf + 1;
    const int q0t = j * kBwdTile;
    uint32_t rq[KSTEPS], cq[DBLK][2], rq_next[kFragAhead];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) { rq[ks] = row_off[ks] + (uint32_t)(buf * TILE_BYTES); asm volatile("" : "+v"(rq[ks])); }
#pragma unroll
    for (int db = 0; db < DBLK; ++db)
#pragma unroll
      for (int u = 0; u < 2; ++u) { cq[db][u] = col_off[db][u] + (uint32_t)(buf * TILE_BYTES); asm volatile("" : "+v"(cq[db][u])); }
#pragma unroll
    for (int ks = 0; ks < kFragAhead; ++ks) { rq_next[ks] = row_off[ks] + (uint32_t)(nbuf * TILE_BYTES); asm volatile("" : "+v"(rq_next[ks])); }
    auto frag = [&](int g) -> vec8 {
      const int ph = g / NMF, i = g % NMF;
      return ph < 2 ? scores_frag_sd(rq, ph, i) : grads_frag(cq, ph - 2, i);
    };
    auto refill = [&](int g) {
      fr[g % kFragAhead] = g + kFragAhead < NG ? frag(g + kFragAhead) : scores_frag_sd(rq_next, 0, g + kFragAhead - NG);
    };
    // an accumulator's start values, straight from LDS into its registers
    auto start_acc = [&](f32x16& acc, FO_LDS const float* rows, int qb) {
#pragma unroll
      for (int jv = 0; jv < 4; ++jv) {
        const f32x4 d4 = *(FO_LDS const f32x4*)(rows + 32 * qb + 8 * jv + 4 * hh);
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[4 * jv + u] = d4[u];
      }
    };
    // AGAIN: the tile's rows are `j` gathered ones (see below); which of the lane's 32 elements count, one bit each
    uint32_t alive = 0;
    if constexpr (AGAIN) {
#pragma unroll 1
      for (int e = 0; e < 32; ++e) {
        const int at = 32 * (e >> 4) + 4 * hh + (e & 3) + 8 * ((e & 15) >> 2), row = gathered[at];
        const bool dead = (at >= j) | (CAUSAL & (key > row)) | !dropout_keep(DropRows<1>::index(prm.drop, bh, Sq, Sk, row, key), prm.drop.seed, prm.drop.threshold);
        alive |= (dead ? 0u : 1u) << e;
      }
    }
    float pv[2][16];            // P of a block between its two stages
    [[maybe_unused]] int full[2][8];      // AGAIN, DS: pairs of dS with delta
    auto stage_a = [&](int qb, int r) {
      const int koff = (r & 3) + 8 * (r >> 2);
      bool dead = false;
      if constexpr (decltype(masked)::value) {
        const int lim = CAUSAL ? key - (q0t + 32 * qb + 4 * hh) : 0;
        const int lim_end = Sq - (q0t + 32 * qb + 4 * hh);
        dead = koff < lim || koff >= lim_end;
      }
      if constexpr (AGAIN) dead = !((alive >> (16 * qb + r)) & 1u);
      float sv = sacc[qb][r];
#if defined(__HIP_DEVICE_COMPILE__)
      if constexpr (AGAIN) asm volatile("" : "+v"(sv));      // (read here, not earlier: see the wait states at the end of tile_body)
#endif
      pv[qb][r] = dead ? 0.0f : __builtin_amdgcn_exp2f(SHIFT ? __builtin_fmaf(sv, c, shift[qb][r]) : KBIAS ? __builtin_fmaf(sv, c, bias_lane) : sv * c);
    };
    auto stage_b = [&](int qb, int r) {          // elements r and r + 1
      const float ds0 = pv[qb][r] * dpacc[qb][r], ds1 = pv[qb][r + 1] * dpacc[qb][r + 1];
      const vec2 p2 = {(T)pv[qb][r], (T)pv[qb][r + 1]}, ds2 = {(T)ds0, (T)ds1};
      int pw = __builtin_bit_cast(int, p2), dsw = __builtin_bit_cast(int, ds2);
      // (pinned to its micro-group: left alone, the compiler moves the multiplications and the rounding down to the MFMA
      // that reads them, which may not read a register that a VALU instruction has just written)
      asm volatile("" : "+v"(pw), "+v"(dsw));
      pf[qb][r >> 3][(r & 7) >> 1] = pw;
      dsf[qb][r >> 3][(r & 7) >> 1] = dsw;
      if constexpr (AGAIN && DS) {
        FO_LDS const float* d2 = rowvals + NBUF * kBwdTile + 32 * qb + 4 * hh + (r & 3) + 8 * (r >> 2);
        const vec2 full2 = {(T)(pv[qb][r] * (dpacc[qb][r] + d2[0])), (T)(pv[qb][r + 1] * (dpacc[qb][r + 1] + d2[1]))};
        full[qb][r >> 1] = __builtin_bit_cast(int, full2);
      }
    };
    auto slot = [&](int s) {
      const SoftmaxGradJob job = softmax_grad_job(s);      // (s is a constant once the loop is unrolled)
      if (job.stage == 0) stage_a(job.qb, job.r); else stage_b(job.qb, job.r);
    };
    const char* next_q = nullptr;
    const char* next_g = nullptr;
    const char* next_rows = nullptr;
    const char* next_bias = nullptr;
    [[maybe_unused]] char* ds_prev = nullptr;
    uint32_t next_q_dst = 0;
    FO_LDS char* next_rows_dst = nullptr;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int ph = g / NMF, i = g % NMF;
      if (g == 3 * NMF) {
        // the hand-over, between phases 3 and 4 (see hand_over)
        if constexpr (SPREAD) {
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DS ? 4 : 0) : "memory");
          if constexpr (DROP) drop_rows(j, nbuf);
          __builtin_amdgcn_s_barrier();
          const int b2 = buf == 0 ? NBUF - 1 : buf - 1, which = wave_s & 1;   // (waves 2 and 3 repeat the row values of waves 0 and 1)
          next_q = (const char*)(qbase + (int64_t)(j + 2) * kBwdTile * prm.qs[2]);
          next_g = (const char*)(gbase + (int64_t)(j + 2) * kBwdTile * prm.dos[2]);
          next_rows = (const char*)((which ? (const float*)prm.delta : (const float*)prm.nlse) + (int64_t)bh * Sq + (j + 2) * kBwdTile);
          next_q_dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(smem + b2 * TILE_BYTES + wave_s * (TileLaneOffsets<T, D>::N * 1024)));
          next_rows_dst = (FO_LDS char*)(rowvals + (NBUF * which + b2) * kBwdTile);
          if constexpr (TBIAS != 0) next_bias = bias_lane_ptr + (int64_t)(j + 2) * kBwdTile * bias_row_bytes;
        } else if constexpr (!AGAIN) {
          if (j + 1 < n_qt) hand_over(j, std::integral_constant<int, DS ? 4 : 0>{});
        }
      }
      // (two wait states where an MFMA may follow the VALU instruction that wrote its B operand: behind the hand-over,
      // whose paths join here, and where the last B job of the tile ends right before its first reader)
      if (AGAIN || g == 3 * NMF || g == 3 * NMF + HALF) asm volatile("s_nop 1");
      if (ph < 2) {
        if (SHIFT && KBIAS && i == 0) mfma_scores_vgpr_first<T>(sacc[ph], fr[g % kFragAhead], kf[i], bias_start);
        else if (SHIFT && i == 0) mfma_scores_vgpr_first<T>(sacc[ph], fr[g % kFragAhead], kf[i]);
        else if (i < KSTEPS) mfma_scores_vgpr<T>(sacc[ph], fr[g % kFragAhead], kf[i]);
        else mfma_scores_vgpr<T>(dpacc[ph], fr[g % kFragAhead], vf[i - KSTEPS]);
      } else {
        const int t = i / (2 * DBLK), db = (i >> 1) % DBLK;
        if (i & 1) mfma_acc_agpr<T>(dkacc[db], fr[g % kFragAhead], __builtin_bit_cast(vec8, dsf[ph - 2][t]));
        else mfma_acc_agpr<T>(dvacc[db], fr[g % kFragAhead], __builtin_bit_cast(vec8, pf[ph - 2][t]));
      }
      refill(g);
      if constexpr (DS && !AGAIN) {
        // dS of the tile before. (The wave's first tile has none: what it stores, in its own place, it stores anew after it.)
        if (g == 0) ds_prev = ds_wave + (int64_t)max(j - 1, ja) * ds_tile_bytes;
        if (g < 2) store16_uniform_base<0>(ds_prev, ds_off[g], dsf[0][g]);
        else if (g < 4) store16_uniform_base<2048>(ds_prev, ds_off[g - 2], dsf[1][g - 2]);
      }
      if constexpr (DROP && !AGAIN) {
        // (pieces of drop_look(j + 1), pinned to their groups)
        if (g == 1) { drop_first = drop_index(j + 1); asm volatile("" : "+v"(drop_first)); }
        if (g == 2) { drop_a = dropout_block<7>(drop_first, prm.drop.seed, prm.drop.threshold); asm volatile("" : "+v"(drop_a)); }
        if (g == 3) { drop_b = dropout_block<7>(drop_first + 127u, prm.drop.seed, prm.drop.threshold); asm volatile("" : "+v"(drop_b)); }
        if (g == HALF - 1) drop_verdict(drop_a, drop_b);
      }
      // start values of the accumulators while they are idle: block 1 of this tile, block 0 of the next (visible since
      // the hand-over; after the last tile: read, unused)
      if (g == 0) {
        if constexpr (AGAIN) zero_acc(dpacc[1]);
        else start_acc(dpacc[1], rowvals + (NBUF + buf) * kBwdTile, 1);
      }
      if (g == 1) start_acc(SHIFT ? shift[1] : sacc[1], rowvals + buf * kBwdTile, 1);
      if (g == 3 * NMF) start_acc(dpacc[0], rowvals + (NBUF + nbuf) * kBwdTile, 0);
      if (g == 3 * NMF + 1) start_acc(SHIFT ? shift[0] : sacc[0], rowvals + nbuf * kBwdTile, 0);
      if constexpr (TBIAS != 0) {
        // (block 1: from group 2 to two groups before its first MFMA; block 0 of the next tile: in the last half-phase but
        // for its last group - the groups without, or with the least, softmax-gradient arithmetic)
        constexpr int N1 = NMF - 4, N0 = HALF - 1;
        if (g == 1) bias_read(j, 1);
        if (g == 3 * NMF + 1) bias_read(j + 1, 0);
        if constexpr (HALVES) {
          // (the values of tile j+1's first half are in registers from here on: its buffer is free)
          if (g == 3 * NMF + HALF) {
            asm volatile("" ::"v"(bias32) : "memory");
            if constexpr (!SPREAD) { if (j + 2 < n_qt) issue_bias_half(j + 2, 1); }
          }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          if (g == 2 + e * N1 / 16) bias_add(sacc[1], e);
          if (g == 3 * NMF + HALF + e * N0 / 16) bias_add(sacc[0], e);
        }
      }
      if constexpr (SPREAD) {
        if (ph == 3) {
          constexpr int N = TileLaneOffsets<T, D>::N;
          static_assert(2 * N <= NMF && 2 * N <= 8, "at most one copy per micro-group");
          auto copy_piece = [&](auto pc) {
            constexpr int piece = decltype(pc)::value;
            if constexpr (PAD && piece < 2 * N)
              dma16_uniform_base_of_lanes(piece < N ? next_q : next_g, piece < N ? qlo.off[piece % N] : glo.off[piece % N],
                                          next_q_dst + (piece < N ? 0 : NBUF * TILE_BYTES) + (piece % N) * 1024, live.lanes[piece % N]);
            else if constexpr (piece < N) dma16_uniform_base_lds_imm<piece * 1024>(next_q, qlo.off[piece], next_q_dst);
            else if constexpr (piece < 2 * N) dma16_uniform_base_lds_imm<NBUF * TILE_BYTES + (piece - N) * 1024>(next_g, glo.off[piece - N], next_q_dst);
          };
          // (piece p goes out in group (p + 1) NMF / 2N - 1; constants once the loop is unrolled)
          if ((i + 1) * 2 * N / NMF != i * 2 * N / NMF) {
            switch ((i + 1) * 2 * N / NMF - 1) {
              case 0: copy_piece(std::integral_constant<int, 0>{}); break;
              case 1: copy_piece(std::integral_constant<int, 1>{}); break;
              case 2: copy_piece(std::integral_constant<int, 2>{}); break;
              case 3: copy_piece(std::integral_constant<int, 3>{}); break;
              case 4: copy_piece(std::integral_constant<int, 4>{}); break;
              case 5: copy_piece(std::integral_constant<int, 5>{}); break;
              case 6: copy_piece(std::integral_constant<int, 6>{}); break;
              default: copy_piece(std::integral_constant<int, 7>{}); break;
            }
          }
          if (i == 0) dma4_uniform_base(next_rows, lane4, next_rows_dst);
          if constexpr (TBIAS != 0) {
            // (two buffers: tile j's values have been read in the first groups)
            constexpr int EVERY = BPIECES == NMF ? 1 : 2;
            static_assert(BPIECES * EVERY <= NMF, "at most one piece per micro-group");
            static_assert(!HALVES || (BPIECES / 2) * EVERY >= HALF, "the second half's pieces go out once its buffer is free");
            if (i % EVERY == 0 && i / EVERY < BPIECES)
              dma16_lane_ptr(next_bias + (i / EVERY) * BROWS * bias_row_bytes,
                             bias_half(j + 2, i / EVERY / (BPIECES / 2)) + (i / EVERY) % (BPIECES / 2) * 1024);
          }
        }
      }
      if (g >= HALF && g < NG - HALF) {
        // (S of block 0 was finished by the MFMA before this group's: that one and four wait states cover the 11 its
        // result needs before a VALU instruction may read it; every later first read is several MFMAs behind)
        if (g == HALF) asm volatile("s_nop 3" : "+v"(sacc[0]));
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (softmax_grad_slot_group(u, NMF) == (g - HALF) % HALF) slot((g - HALF) / HALF * 8 + u);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (AGAIN && DS) {
      // dS of the kept elements of the gathered rows, whole, in the place of what the tiles left (by this wave, and complete: see
      // the wait in add_slots), which holds -P delta for them as for the dropped ones
#pragma unroll
      for (int e = 0; e < 32; ++e) {
        const int row = gathered[32 * (e >> 4) + 4 * hh + (e & 3) + 8 * ((e & 15) >> 2)], x = row & 15, t2 = (row >> 4) & 1;
        if ((alive >> e) & 1u)
          *(T*)(ds_wave + (int64_t)(row / kBwdTile) * ds_tile_bytes + ((row >> 5) & 1) * 2048 + t2 * 1024 + ((l32 ^ (4 * t2)) * 32) + ((x >> 2) & 1) * 16 +
                ((x & 3) + 4 * (x >> 3)) * 2) = __builtin_bit_cast(vec2, full[e >> 4][(e & 15) >> 1])[e & 1];
      }
    }
  };

  int j = qt0 - 1;
  for (; j <= min(ja, n_qt) - 1 && j <= n_qt - 2; ++j) {
    if constexpr (DROP) drop_look(j + 1);
    hand_over(j, std::integral_constant<int, 0>{});
  }
  // Tiles that need the mask are a prefix (the causal diagonal) and possibly the last tile (queries past the end).
  // One loop per kind, each with a single body: with alternatives inside one loop the compiler moves the 128
  // accumulator registers between homes at every tile.
  auto needs_mask = [&](int jt) { return jt * kBwdTile + kBwdTile > Sq || (CAUSAL && k0w + 31 > jt * kBwdTile); };
  j = ja;
  // the first fragments of the tile in buffer `buf`, and what the accumulators of its block 0 start from (as every later
  // tile gets them at the end of the tile before it)
  auto start_tile = [&](int buf) {
    uint32_t rq0[kFragAhead];
#pragma unroll
    for (int ks = 0; ks < kFragAhead; ++ks) rq0[ks] = row_off[ks < KSTEPS ? ks : 0] + (uint32_t)(buf * TILE_BYTES);
#pragma unroll
    for (int i = 0; i < kFragAhead; ++i) fr[i] = scores_frag_sd(rq0, 0, i);
#pragma unroll
    for (int jv = 0; jv < 4; ++jv) {
      const f32x4 d4 = *(FO_LDS const f32x4*)(rowvals + (NBUF + buf) * kBwdTile + 8 * jv + 4 * hh);
#pragma unroll
      for (int u = 0; u < 4; ++u) dpacc[0][4 * jv + u] = d4[u];
      const f32x4 n4 = *(FO_LDS const f32x4*)(rowvals + buf * kBwdTile + 8 * jv + 4 * hh);
#pragma unroll
      for (int u = 0; u < 4; ++u) (SHIFT ? shift[0] : sacc[0])[4 * jv + u] = n4[u];
    }
    if constexpr (TBIAS != 0) {
      bias_read(ja, 0);
#pragma unroll
      for (int e = 0; e < 16; ++e) bias_add(sacc[0], e);
      if constexpr (HALVES) { if (ja + 1 < n_qt) issue_bias_half(ja + 1, 1); }
    }
  };
  if (j < n_qt) start_tile((j - qt0) % NBUF);
  int buf = j < n_qt ? (j - qt0) % NBUF : 0;
  auto next_buf = [&]() { buf = buf == NBUF - 1 ? 0 : buf + 1; };
  for (; j < n_qt && needs_mask(j); ++j, next_buf()) tile_body(j, buf, std::true_type{}, std::false_type{}, std::false_type{});
#if FO_BWD_SPREAD
  // (from here on only a last tile that crosses the end of Q needs the mask; tiles j with tile j+2 wholly inside Q)
  if (qlo.ok && glo.ok)
    for (const int end = (DS ? min(Sq / kBwdTile, n_qt) : Sq / kBwdTile) - 2; j < end; ++j, next_buf()) tile_body(j, buf, std::false_type{}, std::true_type{}, std::false_type{});
#endif
  for (; j < n_qt && !needs_mask(j); ++j, next_buf()) tile_body(j, buf, std::false_type{}, std::false_type{}, std::false_type{});
  for (; j < n_qt; ++j, next_buf()) tile_body(j, buf, std::true_type{}, std::false_type{}, std::false_type{});

  if constexpr (DS) {
    if (ja < n_qt) {                         // the last tile's
      char* last = ds_wave + (int64_t)(n_qt - 1) * ds_tile_bytes;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        store16_uniform_base<0>(last, ds_off[t], dsf[0][t]);
        store16_uniform_base<2048>(last, ds_off[t], dsf[1][t]);
      }
    }
  }
  if constexpr (DROP) {
    // rows that are partly dropped (`again` and what follows from it is the same for every wave)
    int slot_row = 0, n_slots = 0;           // lane i holds the row of slot i
    auto add_slots = [&]() {
      __syncthreads();                       // everyone is done with the buffers
      constexpr int N = TileLaneOffsets<T, D>::N, CHUNKS = D * 2 / 16, ROWS_PER_DMA = 1024 / (D * 2);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int at = (wave_s * N + i) * ROWS_PER_DMA + lane / CHUNKS, col = ((lane % CHUNKS) ^ swz<D>(at)) * 8;
        const int64_t row = __shfl(slot_row, at);
        dma16_lane_ptr(qbase + row * prm.qs[2] + col, smem + (wave_s * N + i) * 1024);
        dma16_lane_ptr(gbase + row * prm.dos[2] + col, smem + NBUF * TILE_BYTES + (wave_s * N + i) * 1024);
      }
      if (wave_s == 0) {
        dma4_lane_ptr((const float*)prm.nlse + (int64_t)bh * Sq + slot_row, rowvals);
        if constexpr (DS) dma4_lane_ptr((const float*)prm.delta + (int64_t)bh * Sq + slot_row, rowvals + NBUF * kBwdTile);
        gathered[lane] = slot_row;
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      start_tile(0);
      zero_acc(dpacc[0]);
      tile_body(n_slots, 0, std::false_type{}, std::false_type{}, std::true_type{});
      n_slots = 0;
    };
    int jt = qt0 - 1;
    next_mixed = 0;
    while (again != 0) {
      if (next_mixed == 0) {
        ++jt;
        if (jt < n_qt && ((again >> (jt >> again_shift)) & 1)) drop_look(jt);
      }
      while (next_mixed != 0 && n_slots < 64) {
        const int row = jt * kBwdTile + __builtin_ctzll(next_mixed);
        next_mixed &= next_mixed - 1;
        if (row < Sq) { slot_row = lane == n_slots ? row : slot_row; ++n_slots; }
      }
      if (jt >= n_qt) again = 0;
      if (n_slots == 64 || (again == 0 && n_slots > 0)) add_slots();
    }
  }

  acc_fence(dkacc);
  acc_fence(dvacc);
  if constexpr (DS) {
    if ((item >> 16) != kWholeBlock >> 16) {
      // a piece of a block: the accumulators as they stand, for the dQ kernel's last workgroups (merge_dkdv) to add
      char* part = dkdv_part(prm, item >> 16, bh, wave_s) + lane * 16;
#pragma unroll
      for (int db = 0; db < DBLK; ++db)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          f32x4 dk4, dv4;
#pragma unroll
          for (int u = 0; u < 4; ++u) { dk4[u] = dkacc[db][4 * rg + u]; dv4[u] = dvacc[db][4 * rg + u]; }
          *(f32x4*)(part + (4 * db + rg) * 1024) = dk4;
          *(f32x4*)(part + kPartBytes / 8 + (4 * db + rg) * 1024) = dv4;
        }
      return;
    }
  }
  // (the tile buffers are free once every wave is past its last tile; dK, then dV, through the wave's own piece of them)
  __syncthreads();
  {
    FO_LDS char* stage = smem + wave_s * stage_bytes(D);
    const int k0w_s = k0 + wave_s * 32;
    store_rows_via_lds<T, LIVE>(dkacc, scale, stage, (T*)prm.dk + b * prm.dks[0] + h * prm.dks[1], prm.dks[2], k0w_s, Sk, prm.d, lane);
    store_rows_via_lds<T, LIVE>(dvacc, 1.0f, stage, (T*)prm.dv + b * prm.dvs[0] + h * prm.dvs[1], prm.dvs[2], k0w_s, Sk, prm.d, lane);
  }
}

// rows, dK/dV with dS kept, dQ of dS
template <typename T, bool CAUSAL, bool KBIAS, bool DROP, bool PAD, int LIVE, int TBIAS>
static int launch_bwd_ds(const AttnBwdParams& q, unsigned g_dkdv, size_t lds_kv, hipStream_t s) {
  static const hipError_t a = hipFuncSetAttribute((const void*)attn_bwd_dkdv_pipe_kernel<T, 128, CAUSAL, KBIAS, DROP, PAD, LIVE, TBIAS, true>,
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_kv);
  if (a != hipSuccess) return FO_ERR_LAUNCH;
  const int st = launch_bwd_rows<T>(q, DROP, TBIAS != 0, s);
  if (st != FO_OK) return st;
  const unsigned grid = q.n_items > 0 ? (unsigned)(q.n_items * q.B * q.H) : g_dkdv;
  attn_bwd_dkdv_pipe_kernel<T, 128, CAUSAL, KBIAS, DROP, PAD, LIVE, TBIAS, true><<<grid, kBwdWaves * 64, lds_kv, s>>>(q);
  return launch_dq_of_ds<T>(q, CAUSAL, TBIAS != 0, s);
}

// A head_dim below the D columns the kernels are laid out for, without bias and dropout: the pipelined dK/dV kernel, and
// products over the next multiple of 32 columns. B=4 H=16, 777 x 1250, head_dim 80, bf16: dQ 67.5 -> 55.4 us, dK/dV 137 ->
// 72.6 us (plain kernel over 128 columns, every tile copied with lane addresses -> this).
template <typename T, int D, bool CAUSAL, int LIVE>
static int launch_bwd_pad(const AttnBwdParams& q, unsigned g_dq, unsigned g_dkdv, size_t lds_dq, size_t lds_pipe, hipStream_t s) {
  constexpr int LIVE_KV = LIVE < 64 ? 64 : LIVE;      // (the pipeline's phases are at least eight MFMAs long)
  static const hipError_t a1 = hipFuncSetAttribute((const void*)attn_bwd_dq_kernel<T, D, CAUSAL, false, false, false, true, LIVE>,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_dq);
  static const hipError_t a2 = hipFuncSetAttribute((const void*)attn_bwd_dkdv_pipe_kernel<T, D, CAUSAL, false, false, true, LIVE_KV>,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_pipe);
  if (a1 != hipSuccess || a2 != hipSuccess) return FO_ERR_LAUNCH;
  if constexpr (D == 128) {
    if (q.ds != nullptr) return launch_bwd_ds<T, CAUSAL, false, false, true, LIVE, 0>(q, g_dkdv, lds_pipe, s);
  }
  attn_bwd_dq_kernel<T, D, CAUSAL, false, false, false, true, LIVE><<<g_dq, kBwdWaves * 64, lds_dq, s>>>(q);
  attn_bwd_dkdv_pipe_kernel<T, D, CAUSAL, false, false, true, LIVE_KV><<<g_dkdv, kBwdWaves * 64, lds_pipe, s>>>(q);
  return launch_status();
}

// A bias with a query stride whose tiles can be copied, without dropout: what the score accumulators start from in both
// kernels. (An fp32 bias at head_dim 128 goes through half a tile's buffer in the dQ kernel, so that two of its workgroups still
// fit a compute unit, and three in the dK/dV kernel.) General form -> this, bias [1, H, S, S]:
// 12 heads x 3072 causal at head_dim 128 bf16 bias: dQ 156 -> 111 us, dK/dV 147 -> 90; whole backward not causal 540 -> 320;
// at head_dim 64 235 -> 131 causal, 347 -> 209 not, with an fp32 bias 258 -> 151 and 384 -> 270.
// fp32 bias at head_dim 128, whole backward: 12 heads x 3072 345 -> 218 causal (290 with the general dQ kernel), 585 -> 384 not (468);
// x 1024 111 -> 88; x 512 the same (87); 16 x 4096 510 -> 371 and 803 -> 626.
template <typename T, int D, bool CAUSAL, int ELT>
static int launch_bwd_tile_bias(const AttnBwdParams& q, unsigned g_dq, unsigned g_dkdv, size_t lds_tiles, size_t lds_pipe, hipStream_t s) {
  const size_t lds_dq = lds_tiles + kBwdWaves * (D == 128 && ELT == 4 ? BiasRows<T, 4, 32>::BYTES : BiasRows<T, ELT>::BYTES), lds_kv = lds_pipe + kBwdWaves * tile_bias_bytes<ELT, D>();
  static const hipError_t a1 = hipFuncSetAttribute((const void*)attn_bwd_dq_kernel<T, D, CAUSAL, false, false, false, false, D, ELT>,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_dq);
  static const hipError_t a2 = hipFuncSetAttribute((const void*)attn_bwd_dkdv_pipe_kernel<T, D, CAUSAL, false, false, false, D, ELT>,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_kv);
  if (a1 != hipSuccess || a2 != hipSuccess) return FO_ERR_LAUNCH;
  if constexpr (D == 128) {
    if (q.ds != nullptr) return launch_bwd_ds<T, CAUSAL, false, false, false, D, ELT>(q, g_dkdv, lds_kv, s);
  }
  attn_bwd_dq_kernel<T, D, CAUSAL, false, false, false, false, D, ELT><<<g_dq, kBwdWaves * 64, lds_dq, s>>>(q);
  attn_bwd_dkdv_pipe_kernel<T, D, CAUSAL, false, false, false, D, ELT><<<g_dkdv, kBwdWaves * 64, lds_kv, s>>>(q);
  return launch_status();
}

template <typename T, int D, bool CAUSAL, bool DROP, bool BIAS>
static int launch_bwd(const AttnBwdParams& p, hipStream_t s) {
  const int64_t n_bh = (int64_t)p.B * p.H;
  const int64_t g_dq = ((p.Sq + kBwdRows - 1) / kBwdRows) * n_bh;
  const int64_t g_dkdv = ((p.Sk + kBwdRows - 1) / kBwdRows) * n_bh;
  if (g_dq > 0x7FFFFFFFll || g_dkdv > 0x7FFFFFFFll) return FO_ERR_BAD_SHAPE;
  const size_t lds_tiles = 4 * (size_t)kBwdTile * D * 2;
  const size_t lds_dq = lds_tiles + (BIAS ? 512 : 0);   // + the per-key bias of two tiles (both bias forms)
  const size_t lds_dkdv = lds_tiles + 4 * kBwdTile * sizeof(float) + (BIAS ? kBwdWaves * 2 * kBwdTile * 32 * 4 : 0);   // + bias tiles
  static const hipError_t a1 = hipFuncSetAttribute((const void*)attn_bwd_dq_kernel<T, D, CAUSAL, DROP, BIAS>,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_dq);
  static const hipError_t a2 = hipFuncSetAttribute((const void*)attn_bwd_dkdv_kernel<T, D, CAUSAL, DROP, BIAS>,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_dkdv);
  const size_t lds_pipe = 6 * (size_t)kBwdTile * D * 2 + 6 * kBwdTile * sizeof(float);   // three tile buffers
  static const hipError_t a3 = hipFuncSetAttribute((const void*)attn_bwd_dkdv_pipe_kernel<T, D, CAUSAL, false, DROP>,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_pipe);
  if (a1 != hipSuccess || a2 != hipSuccess || a3 != hipSuccess) return FO_ERR_LAUNCH;
  // a bias without a query stride: the forms of the dQ kernel and of the pipelined dK/dV kernel that
  // take it at no cost per score (attn_bwd.variant 0 keeps the general bias kernels, which tests compare them with)
  const bool key_bias = BIAS && p.bias.strides[2] == 0 && tune(g_attn_bwd_variant) != 0;
  if constexpr (BIAS) {
    static const hipError_t a4 = hipFuncSetAttribute((const void*)attn_bwd_dq_kernel<T, D, CAUSAL, DROP, false, true>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_dq);
    static const hipError_t a5 = hipFuncSetAttribute((const void*)attn_bwd_dkdv_pipe_kernel<T, D, CAUSAL, true, DROP>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_pipe);
    if (a4 != hipSuccess || a5 != hipSuccess) return FO_ERR_LAUNCH;
  }
  // one group while the Q, dO, K and V of all heads fit the memory-side cache (256 MiB), else groups of heads whose
  // operands stay within a quarter of it; multiples of 8 so that a head's workgroups keep landing on one XCD
  // (B=16 H=32 S=2048 D=128 causal: 2.61 ms in one group, 2.23 ms in groups of 32; the headline shape, 256 MiB: 1.80 ms
  // in one group, 1.90 ms in groups of 8)
  AttnBwdParams q = p;
  {
    const int64_t bytes_head = 2 * ((int64_t)p.Sq + p.Sk) * D * 2;
    const int order = tune(g_attn_bwd_order);
    int64_t group = order >= 0 ? order : bytes_head * n_bh <= (256ll << 20) ? n_bh : ((64ll << 20) / bytes_head) & ~7ll;
    if (order < 0 && group < 8) group = 8;
    if (group <= 0 || group > n_bh) group = n_bh;
    q.head_group = (int)group;
  }
  // (delta is computed by the dQ kernel, which the dK/dV kernel follows; where dS is kept, by the rows' kernel before both)
  if constexpr (BIAS) {
    if (key_bias) {
      if constexpr (D == 128) {
        if (q.ds != nullptr) return launch_bwd_ds<T, CAUSAL, true, DROP, false, D, 0>(q, (unsigned)g_dkdv, lds_pipe, s);
      }
      attn_bwd_dq_kernel<T, D, CAUSAL, DROP, false, true><<<(unsigned)g_dq, kBwdWaves * 64, lds_dq, s>>>(q);
      if (p.d == D) attn_bwd_dkdv_pipe_kernel<T, D, CAUSAL, true, DROP><<<(unsigned)g_dkdv, kBwdWaves * 64, lds_pipe, s>>>(q);
      else attn_bwd_dkdv_kernel<T, D, CAUSAL, DROP, BIAS><<<(unsigned)g_dkdv, kBwdWaves * 64, lds_dkdv, s>>>(q);
      return launch_status();
    }
  }
  if constexpr (BIAS && !DROP) {
    // (dma_ok: base and strides are multiples of 16 bytes, the query stride is not zero)
    if (p.d == D && p.bias.dma_ok && tune(g_attn_bwd_variant) != 0) {
      if (!p.bias.is_f32) return launch_bwd_tile_bias<T, D, CAUSAL, 2>(q, (unsigned)g_dq, (unsigned)g_dkdv, lds_tiles, lds_pipe, s);
      return launch_bwd_tile_bias<T, D, CAUSAL, 4>(q, (unsigned)g_dq, (unsigned)g_dkdv, lds_tiles, lds_pipe, s);
    }
  }
  if constexpr (!DROP && !BIAS) {
    if (p.d != D && tune(g_attn_bwd_variant) != 0) {
      constexpr int NARROW = live_columns(D, 8);
      return p.d <= NARROW ? launch_bwd_pad<T, D, CAUSAL, NARROW>(q, (unsigned)g_dq, (unsigned)g_dkdv, lds_dq, lds_pipe, s)
                           : launch_bwd_pad<T, D, CAUSAL, D>(q, (unsigned)g_dq, (unsigned)g_dkdv, lds_dq, lds_pipe, s);
    }
  }
  if constexpr (!BIAS && D == 128) {
    if (q.ds != nullptr && p.d == D)
      return launch_bwd_ds<T, CAUSAL, false, DROP, false, D, 0>(q, (unsigned)g_dkdv, lds_pipe, s);
  }
  attn_bwd_dq_kernel<T, D, CAUSAL, DROP, BIAS><<<(unsigned)g_dq, kBwdWaves * 64, lds_dq, s>>>(q);
  // attn_bwd.variant 0 selects the plain dK/dV kernel everywhere (tests compare the two)
  // (and other head dims with dropout)
  if (!BIAS && p.d == D && tune(g_attn_bwd_variant) != 0) attn_bwd_dkdv_pipe_kernel<T, D, CAUSAL, false, DROP><<<(unsigned)g_dkdv, kBwdWaves * 64, lds_pipe, s>>>(q);
  else attn_bwd_dkdv_kernel<T, D, CAUSAL, DROP, BIAS><<<(unsigned)g_dkdv, kBwdWaves * 64, lds_dkdv, s>>>(q);
  return launch_status();
}

// every kernel of one operand type and head_dim behind one function, which one translation unit defines (see below)
template <typename T, int D>
int launch_bwd_of(const AttnBwdParams& p, bool causal, bool drop, bool has_bias, hipStream_t s) {
  if (has_bias) {
    if (drop) return causal ? launch_bwd<T, D, true, true, true>(p, s) : launch_bwd<T, D, false, true, true>(p, s);
    return causal ? launch_bwd<T, D, true, false, true>(p, s) : launch_bwd<T, D, false, false, true>(p, s);
  }
  if (drop) return causal ? launch_bwd<T, D, true, true, false>(p, s) : launch_bwd<T, D, false, true, false>(p, s);
  return causal ? launch_bwd<T, D, true, false, false>(p, s) : launch_bwd<T, D, false, false, false>(p, s);
}
// This file is compiled several times, in parallel: as it stands it is the C ABI and holds no kernel;
// attn_bwd_bf16_d64.hip ... attn_bwd_f16_d128.hip include it with FO_ATTN_UNIT set and instantiate launch_bwd_of<T, D>.
#ifndef FO_ATTN_UNIT
#define FO_ATTN_UNIT 0
#endif
#define FO_ATTN_LAUNCH(UNIT, T, D) \
  FO_ATTN_EXTERN_##UNIT template int launch_bwd_of<T, D>(const AttnBwdParams&, bool, bool, bool, hipStream_t);
#if FO_ATTN_UNIT == 1
#define FO_ATTN_EXTERN_1
#else
#define FO_ATTN_EXTERN_1 extern
#endif
#if FO_ATTN_UNIT == 2
#define FO_ATTN_EXTERN_2
#else
#define FO_ATTN_EXTERN_2 extern
#endif
#if FO_ATTN_UNIT == 3
#define FO_ATTN_EXTERN_3
#else
#define FO_ATTN_EXTERN_3 extern
#endif
#if FO_ATTN_UNIT == 4
#define FO_ATTN_EXTERN_4
#else
#define FO_ATTN_EXTERN_4 extern
#endif
FO_ATTN_LAUNCH(1, __bf16, 64)
FO_ATTN_LAUNCH(2, __bf16, 128)
FO_ATTN_LAUNCH(3, _Float16, 64)
FO_ATTN_LAUNCH(4, _Float16, 128)

}  // namespace fo

#if FO_ATTN_UNIT == 0
using namespace fo;

// ---- the same without a workspace argument and without any allocation: the workspace is a device array of this library.
// The array's name is only a host-side handle for the device symbol; its address on a device comes from
// hipGetSymbolAddress, asked once per device with that device current, and only that pointer is handed to the kernels.
constexpr int64_t kStaticDeltaFloats = FO_ATTN_BWD_STATIC_ROWS;
static __device__ __align__(256) float scratch[2 * kStaticDeltaFloats];   // two values per row: see AttnBwdParams
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static float* g_scratch_ptr[kMaxDevices];   // per device; null until that device's first call

static int scratch_of_current_device(float** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return FO_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr) return FO_ERR_LAUNCH;
    g_scratch_ptr[dev] = static_cast<float*>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return FO_OK;
}

// The workspace of fo_attn_bwd_ws: the two values per query row, then dS where it is kept.
static int64_t rows_ws_bytes(int B, int H, int Sq) { return ((int64_t)B * H * Sq * 2 * (int64_t)sizeof(float) + 255) & ~255ll; }
static int64_t ds_bytes_of(int B, int H, int Sq, int Sk) { return (int64_t)B * H * ds_key_blocks(Sk) * ds_query_tiles(Sq) * kDsChunk; }
// When dS is kept. Not at head_dim 64 and below, where computing the scores again costs half as much and reading dS the same: 8 x 12
// heads x 1024 causal 77 us -> 82, 16 x 16 x 1024 157 -> 223. At head_dim 128, whole backward, scores again -> dS kept:
//   12 heads x 4096, per-key bias, dropout 440 -> 347 us; x 3072 causal, bf16 bias with a query stride 200 -> 144; x 6144 853 -> 713
//   4 heads x 2048 .. 8192 causal: the dQ kernel's workgroups walk their keys 2.2 us per 64 alone on their CU, reading dS 0.8 us:
//   2 x 4 x 4096 217 -> 159; so from 1536 keys whatever the size
//   fewer keys: with the rows' kernel and a third launch it takes 96 MiB of dS to gain: 192 heads x 512 125 -> 115, 64 x 1024 125 -> 114,
//   64 x 768 not causal 90 -> 89, 16 x 1024 72 -> 76, 4 heads x 128 70 -> 73 (these wait for their host);
//   half as much again up to head_dim 96, whose scores cost 3/4, forward and backward: 96 heads x 700 x 1100 at 72 (149 MiB) 146 -> 139, 48 x 1450 x
//   1100 at 96 (155) 144 -> 133, 128 x 600 x 900 at 80 (160) 137 -> 132; 64 x 777 x 1250 at 80 (130) 113.2 -> 113.3, 64 x 1024 at 96 causal (128) 86 -> 88
//   up to 2 GiB, what a caller's memory is asked for; beyond, the gain shrinks with the traffic that no cache holds: 12 x 8192
//   causal (1.6 GiB) 639 -> 594, 64 x 4096 causal (2 GiB) 877 -> 846, 512 x 2048 (4 GiB) 3402 -> 3392.
// With many heads (B H) the launches fill the chip without it, the operands come from memory as well, and dS pays only while the caches hold it:
//   head_dim above 96: to 96 heads at any size (96 x 3072 x 2048 978 -> 925, x 2048 x 4096, 1.5 GiB, 1285 -> 1291); to 192 not causal to 2048 keys (192 x
//   1024 x 2048 715 -> 702, x 2048 x 2048 1351 -> 1325), else to 384 MiB (192 x 1024 causal 252 -> 249, 128 x 384 x 4096 456 -> 454; not 192 x 384 x 4096,
//   576 MiB, 678 -> 688, 160 x 256 x 8192, 640, 911 -> 938, 192 x 1536 x 2048 causal, 1152, 504 -> 518); more heads to 512 keys (384 x 512 248 -> 238,
//   768 x 2048 x 512 1634 -> 1544), not beyond: 256 x 128 x 4096 476 -> 516, 256 x 256 x 2048 337 -> 350, 384 x 384 x 2048 658 -> 682, 512 x 128 x
//   1024 256 -> 261, 768 x 1024 causal 993 -> 1025; between lie gains as well (320 x 320 x 1024 292 -> 280)
//   with dropout, or a bias with a query stride, which the other dQ kernel pays for a second time, with any number of heads: 384 x 1536, dropout
//   1615 -> 1564, causal 991 -> 987; 384 x 1536 with a bf16 bias 1706 -> 1644, causal 1096 -> 1034; 384 x 128 x 2048 404 -> 404
//   up to 96: to 64 heads at any size (48 x 3072 x 4096 801 -> 785, 24 x 4096 281 -> 266), to 128 to 192 MiB (128 x 128 x 4096 248 -> 237, 96 x 1024 163 -> 160;
//   not 128 x 384 x 4096, 384 MiB, 392 -> 407, 96 x 2048 x 4096 1061 -> 1157), not with more: 160 x 256 x 2048 208 -> 217, 256 x 128 x 2048 211 ->
//   230, 192 x 2048 x 1024 594 -> 636, 384 x 1024 633 -> 687, 768 x 1024 causal 845 -> 933
constexpr int64_t kDsFromBytes = 96ll << 20, kDsMaxBytes = 2ll << 30;
constexpr int kDsFromKeys = 1536;
struct BwdCall { bool causal, drop; BiasParams bias; };
static int64_t ds_bytes_that_pay(int64_t heads, int Sk, int D, const BwdCall& c) {
  if (D <= 96) return heads <= 64 ? kDsMaxBytes : heads <= 128 ? 192ll << 20 : 0;
  if (heads <= 96 || Sk <= 512 || c.drop || (c.bias.ptr != nullptr && c.bias.strides[2] != 0)) return kDsMaxBytes;
  return heads > 192 ? 0 : !c.causal && Sk <= 2048 ? kDsMaxBytes : 384ll << 20;
}
// The calls that can keep it are those that launch_bwd gives to the pipelined dK/dV kernel. The others (a bias with a query stride whose tiles
// cannot be copied, or together with dropout; head dims off 128 with any bias or dropout) have no use for the memory.
static bool bwd_keeps_ds(int B, int H, int Sq, int Sk, int D, const BwdCall& c) {
  const int asked = tune(g_attn_bwd_keep_ds);
  if (asked == 0 || D <= 64 || tune(g_attn_bwd_variant) == 0 || (int64_t)B * H > (1 << 20) || ds_key_blocks(Sk) * ds_query_tiles(Sq) > kDsMaxBytes / kDsChunk) return false;
  if (D != 128 && (c.drop || c.bias.ptr != nullptr)) return false;
  if (c.bias.ptr != nullptr && c.bias.strides[2] != 0 && (!c.bias.dma_ok || c.drop)) return false;
  const int64_t bytes = ds_bytes_of(B, H, Sq, Sk);
  if (asked == 1) return bytes <= kDsMaxBytes;
  return bytes <= ds_bytes_that_pay((int64_t)B * H, Sk, D, c) && (Sk >= kDsFromKeys || bytes >= (D > 96 ? kDsFromBytes : kDsFromBytes + kDsFromBytes / 2));
}
static BiasParams make_bias(const void* bias, const int64_t* strides, bool is_f32) {
  BiasParams b;
  b.ptr = bias;
  for (int i = 0; i < 3; ++i) b.strides[i] = bias ? strides[i] : 0;
  b.is_f32 = is_f32;
  const uintptr_t elt = is_f32 ? 4 : 2;
  // (dK/dV kernel: tiles of the bias are copied into LDS in 16-byte pieces)
  b.dma_ok = bias && b.strides[2] != 0 && ((uintptr_t)bias % 16) == 0 && (b.strides[0] * elt) % 16 == 0 && (b.strides[1] * elt) % 16 == 0 &&
             (b.strides[2] * elt) % 16 == 0;
  b.vec_ok = bias && ((uintptr_t)bias % (4 * elt)) == 0 && b.strides[0] % 4 == 0 && b.strides[1] % 4 == 0 && b.strides[2] % 4 == 0;
  return b;
}

// (A step of a model asks for the same few over and over, and a plan takes 2 to 40 us: the last ones are kept per thread. With one place,
// layers of two shapes in turn worked theirs out at every call.)
static const DkdvPlan& dkdv_plan(int B, int H, int Sq, int Sk, bool causal) {
  struct Place { int n_bh, Sq, Sk, causal, asked, cus; DkdvPlan plan; };
  constexpr int kPlaces = 8;
  static thread_local Place places[kPlaces];      // (n_bh 0: empty)
  static thread_local int oldest = 0;
  const int asked = tune(g_attn_bwd_order) >= 0 ? 0 : tune(g_attn_bwd_split), cus = device_cus();
  for (const Place& p : places)
    if (p.n_bh == B * H && p.Sq == Sq && p.Sk == Sk && p.causal == (int)causal && p.asked == asked && p.cus == cus) return p.plan;
  Place& p = places[oldest];
  oldest = (oldest + 1) % kPlaces;
  p.n_bh = B * H; p.Sq = Sq; p.Sk = Sk; p.causal = (int)causal; p.asked = asked; p.cus = cus;
  p.plan = make_dkdv_plan(B * H, Sq, Sk, causal, asked, cus);
  return p.plan;
}
static int64_t part_bytes_of(int B, int H, int Sq, int Sk, bool causal) {
  return dkdv_plan(B, H, Sq, Sk, causal).n_parts * (int64_t)B * H * kPartBytes;
}

// What a call does with its workspace: where dS lies in it (0: not kept), and the sums of shared key blocks (plan null: none are shared).
struct BwdForm { int64_t ds_at, part_at; const DkdvPlan* plan; };
static BwdForm bwd_form(int B, int H, int Sq, int Sk, int D, const BwdCall& c, const void* ws, int64_t ws_bytes) {
  BwdForm f = {0, 0, nullptr};
  if (ws_bytes <= 0 || ((uintptr_t)ws & 15u) || !bwd_keeps_ds(B, H, Sq, Sk, D, c)) return f;
  const int64_t rows = rows_ws_bytes(B, H, Sq), end = rows + ds_bytes_of(B, H, Sq, Sk);
  if (ws_bytes < end) return f;
  f.ds_at = rows;
  const DkdvPlan& plan = dkdv_plan(B, H, Sq, Sk, c.causal);
  if (plan.n_items > 0 && ws_bytes >= end + plan.n_parts * (int64_t)B * H * kPartBytes) { f.part_at = end; f.plan = &plan; }
  return f;
}

static int attn_bwd_impl(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                         float* delta_ws, void* dq, void* dk, void* dv, int B, int H, int Sq, int Sk, int D,
                         const int64_t* const* strides_host, float softmax_scale, int causal, int dtype, float dropout_p,
                         uint32_t seed, uint64_t rng_offset, const void* bias, const int64_t* bias_strides, int bias_dtype,
                         void* stream, bool static_ws = false, int64_t ws_bytes = -1) {
  // ws_bytes: how much memory delta_ws points to where the caller says so (fo_attn_bwd_ws; else -1); dS is kept behind its two rows of values
  // static_ws: delta_ws is ignored and the library's own per-device array takes its place (fo_attn_bwd_static_ws)
  if (!q || !k || !v || !o || !d_o || !lse || (!delta_ws && !static_ws) || !dq || !dk || !dv || !strides_host) return FO_ERR_NULL_POINTER;
  for (int t = 0; t < 8; ++t)
    if (!strides_host[t]) return FO_ERR_NULL_POINTER;
  if (dtype != FO_DTYPE_F16 && dtype != FO_DTYPE_BF16) return FO_ERR_BAD_DTYPE;
  if (D < 8 || D > 128 || D % 8 != 0) return FO_ERR_BAD_HEAD_DIM;
  if (B <= 0 || H <= 0 || Sq <= 0 || Sk <= 0 || (int64_t)B * H > (1ll << 40) / Sq) return FO_ERR_BAD_SHAPE;
  if (ws_bytes != -1 && ws_bytes < (int64_t)B * H * Sq * 2 * (int64_t)sizeof(float)) return FO_ERR_BAD_SHAPE;
  for (int t = 0; t < 8; ++t) {
    // rows start on 16-byte boundaries (8 elements); only the inputs K and V may repeat a head (stride 0 = multi-query)
    for (int i = 0; i < 3; ++i)
      if (strides_host[t][i] < 0 || (strides_host[t][i] % 8) != 0) return FO_ERR_BAD_STRIDE;
    if (strides_host[t][2] < D) return FO_ERR_BAD_STRIDE;
    const bool output = t >= 5;
    if (output && ((strides_host[t][0] == 0 && B > 1) || (strides_host[t][1] == 0 && H > 1))) return FO_ERR_BAD_STRIDE;
  }
  const uintptr_t all = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o | (uintptr_t)d_o | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv;
  if (all & 15u) return FO_ERR_MISALIGNED;
  if (((uintptr_t)lse | (static_ws ? 0 : (uintptr_t)delta_ws)) & 3u) return FO_ERR_MISALIGNED;
  if (!(softmax_scale > 0.0f) || softmax_scale > 3.0e38f) return FO_ERR_BAD_SHAPE;
  if (!(dropout_p >= 0.0f) || dropout_p >= 1.0f) return FO_ERR_BAD_SHAPE;
  if (bias) {
    if (!bias_strides) return FO_ERR_NULL_POINTER;
    if (bias_dtype != FO_DTYPE_F32 && bias_dtype != dtype) return FO_ERR_BAD_DTYPE;
    if (bias_strides[0] < 0 || bias_strides[1] < 0 || bias_strides[2] < 0) return FO_ERR_BAD_STRIDE;
    if ((uintptr_t)bias & (bias_dtype == FO_DTYPE_F32 ? 3u : 1u)) return FO_ERR_MISALIGNED;
  }
  if (static_ws) {
    // (after every argument check: a rejected call has made no HIP call)
    if ((int64_t)B * H * Sq > kStaticDeltaFloats) return FO_ERR_BAD_SHAPE;
    const int st = scratch_of_current_device(&delta_ws);
    if (st != FO_OK) return st;
  }

  AttnBwdParams p;
  p.q = q; p.k = k; p.v = v; p.o = o; p.d_o = d_o; p.lse = lse; p.delta = delta_ws; p.nlse = delta_ws + (int64_t)B * H * Sq; p.dq = dq; p.dk = dk; p.dv = dv;
  p.B = B; p.H = H; p.Sq = Sq; p.Sk = Sk; p.d = D;
  p.bias = make_bias(bias, bias_strides, bias_dtype == FO_DTYPE_F32);
  const BwdForm form = bwd_form(B, H, Sq, Sk, D, BwdCall{causal != 0, dropout_p > 0.0f, p.bias}, delta_ws, ws_bytes);
  p.ds = form.ds_at > 0 ? (char*)delta_ws + form.ds_at : nullptr;
  p.n_items = p.n_merges = 0;
  p.part = nullptr;
  if (form.plan != nullptr) {
    const DkdvPlan& plan = *form.plan;
    p.part = (char*)delta_ws + form.part_at;
    p.n_items = plan.n_items; p.n_merges = plan.n_merges;
    for (int i = 0; i < plan.n_items; ++i) p.items[i] = plan.items[i];
    for (int i = 0; i < plan.n_merges; ++i) p.merges[i] = plan.merges[i];
  }
  int64_t* dst[8] = {p.qs, p.ks, p.vs, p.os, p.dos, p.dqs, p.dks, p.dvs};
  for (int t = 0; t < 8; ++t)
    for (int i = 0; i < 3; ++i) dst[t][i] = strides_host[t][i];
  p.scale = softmax_scale;
  p.scale_log2e = softmax_scale * kLog2e;
  p.neg_inv_scale_log2e = -1.0f / p.scale_log2e;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool c = causal != 0, drop = dropout_p > 0.0f;
  p.drop = make_dropout(dropout_p, seed, rng_offset);
  // kernels are compiled for 64 and 128 columns; a head_dim in between runs on the next one with zero columns
  const bool has_bias = bias != nullptr;
  if (dtype == FO_DTYPE_BF16) return D > 64 ? launch_bwd_of<__bf16, 128>(p, c, drop, has_bias, s) : launch_bwd_of<__bf16, 64>(p, c, drop, has_bias, s);
  return D > 64 ? launch_bwd_of<_Float16, 128>(p, c, drop, has_bias, s) : launch_bwd_of<_Float16, 64>(p, c, drop, has_bias, s);
}

extern "C" int fo_attn_bwd(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                           float* delta_ws, void* dq, void* dk, void* dv, int B, int H, int Sq, int Sk, int D,
                           const int64_t* const* strides_host, float softmax_scale, int causal, int dtype, void* stream) {
  return attn_bwd_impl(q, k, v, o, d_o, lse, delta_ws, dq, dk, dv, B, H, Sq, Sk, D, strides_host, softmax_scale, causal, dtype,
                       0.0f, 0u, 0ull, nullptr, nullptr, 0, stream);
}

extern "C" int fo_attn_bwd_static_ws(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                                     void* dq, void* dk, void* dv, int B, int H, int Sq, int Sk, int D,
                                     const int64_t* const* strides_host, float softmax_scale, int causal, int dtype, void* stream) {
  // Every delta element the dK/dV kernel reads (rows below Sq of each head) is written by the dQ kernel of the same
  // call, so what an earlier call left in the array does not matter and nothing has to be cleared.
  return attn_bwd_impl(q, k, v, o, d_o, lse, nullptr, dq, dk, dv, B, H, Sq, Sk, D, strides_host, softmax_scale, causal, dtype,
                       0.0f, 0u, 0ull, nullptr, nullptr, 0, stream, true);
}

extern "C" int fo_attn_bwd_dropout(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                                   float* delta_ws, void* dq, void* dk, void* dv, int B, int H, int Sq, int Sk, int D,
                                   const int64_t* const* strides_host, float softmax_scale, int causal, int dtype,
                                   float dropout_p, uint32_t seed, uint64_t rng_offset, void* stream) {
  return attn_bwd_impl(q, k, v, o, d_o, lse, delta_ws, dq, dk, dv, B, H, Sq, Sk, D, strides_host, softmax_scale, causal, dtype,
                       dropout_p, seed, rng_offset, nullptr, nullptr, 0, stream);
}

extern "C" int fo_attn_bwd_ex(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                              float* delta_ws, void* dq, void* dk, void* dv, int B, int H, int Sq, int Sk, int D,
                              const int64_t* const* strides_host, float softmax_scale, int causal, int dtype,
                              const fo_attn_extras* extras, void* stream) {
  if (!extras)
    return attn_bwd_impl(q, k, v, o, d_o, lse, delta_ws, dq, dk, dv, B, H, Sq, Sk, D, strides_host, softmax_scale, causal, dtype,
                         0.0f, 0u, 0ull, nullptr, nullptr, 0, stream);
  return attn_bwd_impl(q, k, v, o, d_o, lse, delta_ws, dq, dk, dv, B, H, Sq, Sk, D, strides_host, softmax_scale, causal, dtype,
                       extras->dropout_p, extras->dropout_seed, extras->dropout_offset, extras->bias, extras->bias_strides,
                       extras->bias_dtype, stream);
}
static bool bwd_ws_shape_ok(int B, int H, int Sq, int Sk, int D) {
  return B > 0 && H > 0 && Sq > 0 && Sk > 0 && D >= 8 && D <= 128 && D % 8 == 0 && (int64_t)B * H <= (1ll << 40) / Sq;
}
static BwdCall bwd_call(int causal, const fo_attn_extras* x) {
  if (!x) return BwdCall{causal != 0, false, make_bias(nullptr, nullptr, false)};
  return BwdCall{causal != 0, x->dropout_p > 0.0f, make_bias(x->bias, x->bias_strides, x->bias_dtype == FO_DTYPE_F32)};
}
static int64_t bwd_ws_bytes(int B, int H, int Sq, int Sk, int D, const BwdCall& c) {
  if (!bwd_ws_shape_ok(B, H, Sq, Sk, D)) return 0;
  if (!bwd_keeps_ds(B, H, Sq, Sk, D, c)) return rows_ws_bytes(B, H, Sq);
  return rows_ws_bytes(B, H, Sq) + ds_bytes_of(B, H, Sq, Sk) + part_bytes_of(B, H, Sq, Sk, c.causal);
}
extern "C" int64_t fo_attn_bwd_workspace_ex(int B, int H, int Sq, int Sk, int D, int causal, const fo_attn_extras* extras) {
  return bwd_ws_bytes(B, H, Sq, Sk, D, bwd_call(causal, extras));
}
extern "C" int64_t fo_attn_bwd_workspace(int B, int H, int Sq, int Sk, int D) {
  int64_t most = 0;
  for (int i = 0; i < 4; ++i) {        // (whatever keeps dS at a shape: one of these does, and a bias asks for no more)
    const int64_t n = bwd_ws_bytes(B, H, Sq, Sk, D, BwdCall{(i & 1) != 0, (i & 2) != 0, make_bias(nullptr, nullptr, false)});
    most = n > most ? n : most;
  }
  return most;
}
extern "C" int fo_attn_bwd_kernels(int B, int H, int Sq, int Sk, int D, int causal, const fo_attn_extras* extras, int64_t ws_bytes) {
  if (!bwd_ws_shape_ok(B, H, Sq, Sk, D)) return FO_ERR_BAD_SHAPE;
  const BwdForm f = bwd_form(B, H, Sq, Sk, D, bwd_call(causal, extras), nullptr, ws_bytes);
  if (f.ds_at == 0) return 0;
  return FO_ATTN_BWD_KEEPS_DS | (f.plan != nullptr ? FO_ATTN_BWD_SHARES_BLOCKS : 0) |
         (dq_two_teams((int64_t)B * H, Sq, Sk, causal != 0, f.plan != nullptr ? f.plan->n_merges : 0) ? FO_ATTN_BWD_DQ_TWO_TEAMS : 0);
}

extern "C" int fo_attn_bwd_ws(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse,
                              void* dq, void* dk, void* dv, int B, int H, int Sq, int Sk, int D,
                              const int64_t* const* strides_host, float softmax_scale, int causal, int dtype,
                              const fo_attn_extras* extras, void* ws, int64_t ws_bytes, void* stream) {
  if (ws_bytes < 0) return FO_ERR_BAD_SHAPE;
  const fo_attn_extras none = {};
  const fo_attn_extras& x = extras ? *extras : none;
  return attn_bwd_impl(q, k, v, o, d_o, lse, (float*)ws, dq, dk, dv, B, H, Sq, Sk, D, strides_host, softmax_scale, causal, dtype,
                       x.dropout_p, x.dropout_seed, x.dropout_offset, x.bias, x.bias_strides, x.bias_dtype, stream, false, ws_bytes);
}
#endif  // FO_ATTN_UNIT == 0
