// dQ of the attention backward from stored dS (see attn_bwd.hpp), and the two values per query row that the dK/dV kernel needs first.
#include <type_traits>

#include "attn_bwd.hpp"

namespace fo {

// (read once: kept out of the way of K, which the workgroups of a head share in the cache)
__device__ __forceinline__ void dma16_uniform_base_nt(const void* base, uint32_t byte_off, FO_LDS void* dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)dst)), "v"(byte_off), "s"(base) : "memory", "m0");
#endif
}

constexpr int kD = 128;      // columns the kernels are laid out for

// -delta and the value of the LSE (AttnBwdParams::nlse) of every query row, for the dK/dV kernel where the dQ kernel runs after it (which
// otherwise computes both): delta_i = sum_d dO_id O_id (flash_attention_triton.py:273-315). 16 lanes per row, 16 bytes each of O and dO.
constexpr int kRowsPerWg = 64;
template <typename T, bool DROP, bool TBIAS>
__global__ void __launch_bounds__(256) attn_bwd_rows_kernel(const AttnBwdParams prm) {
  typedef typename Ops<T>::vec8 vec8;
  constexpr int N = kRowsPerWg / 16;
  const int n_blk = (prm.Sq + kRowsPerWg - 1) / kRowsPerWg, bh = blockIdx.x / n_blk, q0 = (blockIdx.x - bh * n_blk) * kRowsPerWg;
  const int b = bh / prm.H, h = bh - b * prm.H, col = 8 * (threadIdx.x & 15), row = q0 + (threadIdx.x >> 4);
  const T* o = (const T*)prm.o + b * prm.os[0] + h * prm.os[1] + col;
  const T* g = (const T*)prm.d_o + b * prm.dos[0] + h * prm.dos[1] + col;
  vec8 ov[N], gv[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int64_t qi = min(row + 16 * i, prm.Sq - 1);
    ov[i] = *(const vec8*)live_or_zero(o + qi * prm.os[2], col, prm.d);
    gv[i] = *(const vec8*)live_or_zero(g + qi * prm.dos[2], col, prm.d);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float delta = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) delta -= (float)ov[i][e] * (float)gv[i][e];
#pragma unroll
    for (int s = 1; s < 16; s <<= 1) delta += __shfl_xor(delta, s);
    if (col != 0 || row + 16 * i >= prm.Sq) continue;
    const int64_t at = (int64_t)bh * prm.Sq + row + 16 * i;
    const float lse = prm.lse[at];
    prm.delta[at] = DROP ? delta * prm.drop.keep_prob : delta;      // (the factors: see the dQ kernel of attn_bwd.hip)
    prm.nlse[at] = TBIAS ? -lse * (kLog2e / prm.scale_log2e) : -(lse * kLog2e - (DROP ? prm.drop.keep_log2 : 0.0f));
  }
}

// dK and dV of a key block whose query tiles several workgroups of the dK/dV kernel shared: their sums added, in order, in the lanes that
// held them. By the last workgroups of the dQ launch, beside its others (they have what the launch before left, as those do).
template <typename T, int LIVE, int TEAMS>
__device__ __forceinline__ void merge_dkdv(const AttnBwdParams& prm, int at, FO_LDS char* smem) {
  const int n_bh = prm.B * prm.H, m = at / n_bh, bh = at - m * n_bh, b = bh / prm.H, h = bh - b * prm.H;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave_s = wave_all % kBwdWaves, lane = threadIdx.x & 63;
  FO_LDS char* stage = smem + wave_all * stage_bytes(kD);
  const uint32_t w = prm.merges[m];
  const int k0w = (int)(w & 255u) * kBwdRows + wave_s * 32, pieces = (w >> 12) & 15;
#pragma unroll 1
  for (int mat = wave_all / kBwdWaves; mat < 2; mat += TEAMS) {
    f32x16 acc[LIVE / 32];
#pragma unroll
    for (int i = 0; i < LIVE / 32; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
    for (int i = 0; i < pieces; ++i) {
      const char* part = dkdv_part(prm, (w >> 16) + i, bh, wave_s) + mat * (kPartBytes / 8) + lane * 16;
#pragma unroll
      for (int g = 0; g < LIVE / 8; ++g) {
        const f32x4 v = *(const f32x4*)(part + g * 1024);
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[g >> 2][4 * (g & 3) + u] += v[u];
      }
    }
    if (mat == 0) store_rows_via_lds<T, LIVE>(acc, prm.scale, stage, (T*)prm.dk + b * prm.dks[0] + h * prm.dks[1], prm.dks[2], k0w, prm.Sk, prm.d, lane);
    else store_rows_via_lds<T, LIVE>(acc, 1.0f, stage, (T*)prm.dv + b * prm.dvs[0] + h * prm.dvs[1], prm.dvs[2], k0w, prm.Sk, prm.d, lane);
  }
}

// dQ^T = K^T dS^T: a wave owns 32 query rows and walks 32-key tiles of K (shared by the workgroup's four waves) and dS
// (its own) through a ring of four LDS buffers, one barrier per tile; both operands by transposing reads. Bound by reading dS where there
// are workgroups enough, else by a workgroup's chain per tile (0.4 us, the unit's LDS: 12 heads x 3072 causal 40 us; with reads, conditions and products in
// the order they come to mind 48). 12 heads x 4096 (0.4 GB of dS) 98 us = 4.1 TB/s of dS: the dQ kernel that computes the scores again takes
// 172; copied without nt, dS pushes K out of the cache: 131. Five or eight buffers, or 64 rows per wave, gain nothing (131, 131 / 108-170).
// TEAMS 2: eight waves, the second four with the odd tiles and a ring of their own; the two teams' sums are added at the end (see dq_two_teams).
// TBIAS: P of a row whose bias is large as a whole is off by the rounding of -LSE / scale, one factor per row, made good here.
template <typename T, bool CAUSAL, int LIVE, bool PAD, bool TBIAS, int SLOTS, int TEAMS>
__global__ void __launch_bounds__(TEAMS * kBwdWaves * 64, 2) attn_bwd_dq_of_ds_kernel(const AttnBwdParams prm) {
  typedef typename Ops<T>::vec8 vec8;
  constexpr int D = kD, TILE = 32, ROW_BYTES = D * 2, CHUNKS = ROW_BYTES / 16, ROWS_PER_DMA = 1024 / ROW_BYTES;
  constexpr int K_BYTES = TILE * ROW_BYTES, DS_BYTES = 2048, SLOT = K_BYTES + kBwdWaves * DS_BYTES;
  constexpr int NK = K_BYTES / 1024 / kBwdWaves, ND = DS_BYTES / 1024, NI = NK + ND;
  constexpr int DBLK = LIVE / 32;
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), team = wave_all / kBwdWaves, wave_s = wave_all % kBwdWaves;
  FO_LDS char* smem = (FO_LDS char*)smem_raw + team * SLOTS * SLOT;      // the team's slots: K tile | dS of each wave
  const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5, L16 = lane & 15, g16 = (lane >> 4) & 1;
  const int Sq = prm.Sq, Sk = prm.Sk, n_qblk = (Sq + kBwdRows - 1) / kBwdRows, n_qt = (int)ds_query_tiles(Sq);
  const int n_dq = prm.B * prm.H * n_qblk;
  if ((int)blockIdx.x >= n_dq) return merge_dkdv<T, LIVE, TEAMS>(prm, (int)blockIdx.x - n_dq, (FO_LDS char*)smem_raw);
  int bh, qblk;
  bwd_item(prm, n_qblk, bh, qblk);
  qblk = n_qblk - 1 - qblk;                        // heaviest causal blocks first
  const int b = bh / prm.H, h = bh % prm.H;
  const T* kbase = (const T*)prm.k + b * prm.ks[0] + h * prm.ks[1];
  const int block32 = qblk * kBwdWaves + wave_s;                      // the wave's block of 32 queries
  const int qt = min(block32 >> 1, n_qt - 1);                         // (rows past the end: the chunk exists, nothing is stored)
  const char* ds = prm.ds + ds_chunk(prm, bh, 0, qt) + (wave_s & 1) * 2048;
  const int all_tiles = (Sk + TILE - 1) / TILE;
  // (causal: key blocks past a 64-query tile's last query left no dS for it)
  const int n_tiles = CAUSAL ? min(all_tiles, 4 * (qblk + 1)) : all_tiles, my_tiles = CAUSAL ? min(n_tiles, 2 * qt + 2) : n_tiles;

  uint32_t k_off[NK];
#pragma unroll
  for (int i = 0; i < NK; ++i) {
    const int row = (wave_s * NK + i) * ROWS_PER_DMA + lane / CHUNKS;
    // (a column past the head_dim re-reads the last 8: a column of K makes that column of dQ alone, which is not stored. So other head dims take
    // the straight loop too: 8 x 500 x 1600 at 104 30.1 -> 17.7 us, 64 x 1500 x 3000 at 96 129 -> 112)
    const int col = ((lane % CHUNKS) ^ swz<D>(row)) * 8;
    k_off[i] = (uint32_t)(row * (int)prm.ks[2] + (PAD ? min(col, prm.d - 8) : col)) * 2u;
  }
  const bool k_off_ok = prm.ks[2] < (1 << 23);
  const uint32_t lane16 = (uint32_t)lane * 16u;
  auto issue = [&](int tile, int slot_i, auto inside) {
    FO_LDS char* slot = smem + slot_i * SLOT;
    if (decltype(inside)::value || (k_off_ok && tile * TILE + TILE <= Sk)) {
      const char* src = (const char*)(kbase + (int64_t)(tile * TILE) * prm.ks[2]);
#pragma unroll
      for (int i = 0; i < NK; ++i) dma16_uniform_base(src, k_off[i], slot + (wave_s * NK + i) * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        const int row = (wave_s * NK + i) * ROWS_PER_DMA + lane / CHUNKS, col = ((lane % CHUNKS) ^ swz<D>(row)) * 8;
        // (keys past the end re-read the last one; their dS counts as zero below)
        dma16_lane_ptr(live_or_zero(kbase + (int64_t)min(tile * TILE + row, Sk - 1) * prm.ks[2] + col, col, prm.d), slot + (wave_s * NK + i) * 1024);
      }
    }
    const char* src = ds + (int64_t)tile * kDsChunk;
#pragma unroll
    for (int t = 0; t < ND; ++t) dma16_uniform_base_nt(src + 1024 * t, lane16, slot + K_BYTES + wave_s * DS_BYTES + 1024 * t);
  };
  f32x16 acc[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
#pragma unroll
  for (int i = 0; i < SLOTS - 1; ++i)
    if (TEAMS * i + team < n_tiles) issue(TEAMS * i + team, i, std::false_type{});

  // Byte offsets of the fragment reads inside a slot (K as col_frag computes them; dS: keys r and r + 8 of a 16-key step, four
  // queries' worth of 8 bytes). A 16-key step further is an immediate.
  const int r0 = 4 * hh + (L16 >> 2), sub = (L16 & 1) * 8;
  uint32_t k_at[DBLK][2], ds_at[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = r0 + 8 * u;
#pragma unroll
    for (int db = 0; db < DBLK; ++db) k_at[db][u] = (uint32_t)(r * ROW_BYTES + ((4 * db + 2 * g16 + ((L16 & 3) >> 1)) ^ swz<D>(r)) * 16 + sub);
    ds_at[u] = (uint32_t)(K_BYTES + wave_s * DS_BYTES + g16 * 1024 + ((r ^ (4 * g16)) * 32) + (L16 & 3) * 8);
  }
  auto tr_read = [&](uint32_t at, int imm) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((FO_LDS s16x4*)(smem + at + imm)); };
  auto joined = [](s16x4 lo, s16x4 hi) { return __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)); };
  // every fragment of a tile is asked for before its first product
  auto products = [&](int tile, int slot_i, auto ragged) {
    const uint32_t slot = (uint32_t)(slot_i * SLOT);
    vec8 kv[2][DBLK], dsv[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      s16x4 lo = tr_read(ds_at[0] + slot, 512 * t), hi = tr_read(ds_at[1] + slot, 512 * t);
      if constexpr (decltype(ragged)::value) {
        const int left = Sk - (tile * TILE + 16 * t + 4 * hh);      // element e of lo (hi) is key e (8 + e) from there
#pragma unroll
        for (int e = 0; e < 4; ++e) { lo[e] = e < left ? lo[e] : (short)0; hi[e] = 8 + e < left ? hi[e] : (short)0; }
      }
      dsv[t] = joined(lo, hi);
#pragma unroll
      for (int db = 0; db < DBLK; ++db) kv[t][db] = joined(tr_read(k_at[db][0] + slot, 16 * t * ROW_BYTES), tr_read(k_at[db][1] + slot, 16 * t * ROW_BYTES));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int db = 0; db < DBLK; ++db) acc[db] = Ops<T>::mfma(kv[t][db], dsv[t], acc[db]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (every read is back before the next barrier)
  };
  int slot_i = 0, it = 0;                               // the team's tiles are TEAMS it + team; every wave meets the same barriers
  const int n_it = (n_tiles + TEAMS - 1) / TEAMS;
  // Its tile `it` has landed when all but the copies of the SLOTS - 2 tiles after it have; behind the barrier that holds for everyone,
  // and nobody reads the tile before it any more, whose slot takes the tile SLOTS - 1 further on.
  // (one straight loop for the tiles that copy a whole one ahead; causal: they count for every wave, whose last tiles differ by two)
  static_assert(SLOTS > 2, "");
  if (k_off_ok)
    for (const int end = min(n_tiles, Sk / TILE) / TEAMS - (SLOTS - 1); it < end; ++it, slot_i = slot_i == SLOTS - 1 ? 0 : slot_i + 1) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SLOTS - 2) * NI) : "memory");
      __builtin_amdgcn_s_barrier();
      issue(TEAMS * (it + SLOTS - 1) + team, slot_i == 0 ? SLOTS - 1 : slot_i - 1, std::true_type{});
      products(TEAMS * it + team, slot_i, std::false_type{});
    }
  for (; it < n_it; ++it, slot_i = slot_i == SLOTS - 1 ? 0 : slot_i + 1) {
    const int tile = TEAMS * it + team;
    if (tile + TEAMS * (SLOTS - 2) < n_tiles) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SLOTS - 2) * NI) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (tile + TEAMS * (SLOTS - 1) < n_tiles) issue(tile + TEAMS * (SLOTS - 1), slot_i == 0 ? SLOTS - 1 : slot_i - 1, std::false_type{});
    if ((CAUSAL || TEAMS > 1) && tile >= my_tiles) continue;
    if (tile * TILE + TILE > Sk) products(tile, slot_i, std::true_type{});
    else products(tile, slot_i, std::false_type{});
  }
  if constexpr (TEAMS > 1) {
    // the second team's sums, through its slots (which its waves are past), added by the first
    static_assert(TEAMS == 2 && kBwdWaves * DBLK * 4096 <= SLOTS * SLOT, "");
    FO_LDS char* sums = (FO_LDS char*)smem_raw + SLOTS * SLOT + wave_s * (DBLK * 4096) + lane * 16;
    __syncthreads();
    if (team == 1) {
#pragma unroll
      for (int g = 0; g < 4 * DBLK; ++g) {
        f32x4 v;
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = acc[g >> 2][4 * (g & 3) + u];
        *(FO_LDS f32x4*)(sums + g * 1024) = v;
      }
    }
    __syncthreads();
    if (team == 1) return;
#pragma unroll
    for (int g = 0; g < 4 * DBLK; ++g) {
      const f32x4 v = *(FO_LDS const f32x4*)(sums + g * 1024);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[g >> 2][4 * (g & 3) + u] += v[u];
    }
  }
  // column l32 of the result is position l32 of the block (see attn_bwd.hpp)
  const int qi = block32 * 32 + 16 * (l32 >> 4) + (l32 & 3) + 8 * ((l32 >> 2) & 1) + 4 * ((l32 >> 3) & 1);
  if (qi >= Sq) return;
  float mul = prm.scale;
  if constexpr (TBIAS) {
    const float per_scale = kLog2e / prm.scale_log2e, lse = prm.lse[(int64_t)bh * Sq + qi];
    mul *= __builtin_amdgcn_exp2f(__builtin_fmaf(-lse, per_scale, lse * per_scale) * prm.scale_log2e);
  }
  T* op = (T*)prm.dq + b * prm.dqs[0] + h * prm.dqs[1] + (int64_t)qi * prm.dqs[2];
#pragma unroll
  for (int db = 0; db < DBLK; ++db)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      typedef __attribute__((ext_vector_type(4))) T vec4;
      vec4 o4;
#pragma unroll
      for (int u = 0; u < 4; ++u) o4[u] = (T)(acc[db][rg * 4 + u] * mul);
      if (32 * db + 8 * rg + 4 * hh < prm.d) *(vec4*)(op + 32 * db + 8 * rg + 4 * hh) = o4;
    }
}

template <typename T>
int launch_bwd_rows(const AttnBwdParams& p, bool drop, bool tile_bias, hipStream_t s) {
  const unsigned grid = (unsigned)((int64_t)p.B * p.H * ((p.Sq + kRowsPerWg - 1) / kRowsPerWg));
  if (drop) attn_bwd_rows_kernel<T, true, false><<<grid, 256, 0, s>>>(p);
  else if (tile_bias) attn_bwd_rows_kernel<T, false, true><<<grid, 256, 0, s>>>(p);
  else attn_bwd_rows_kernel<T, false, false><<<grid, 256, 0, s>>>(p);
  return launch_status();
}

template <typename T, bool CAUSAL, int LIVE, bool PAD, bool TBIAS, int SLOTS, int TEAMS>
static int launch_one(const AttnBwdParams& p, hipStream_t s) {
  constexpr int lds = TEAMS * SLOTS * (32 * kD * 2 + kBwdWaves * 2048);
  static const hipError_t a = hipFuncSetAttribute((const void*)attn_bwd_dq_of_ds_kernel<T, CAUSAL, LIVE, PAD, TBIAS, SLOTS, TEAMS>,
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (a != hipSuccess) return FO_ERR_LAUNCH;
  const unsigned grid = (unsigned)((int64_t)p.B * p.H * ((p.Sq + kBwdRows - 1) / kBwdRows + p.n_merges));
  attn_bwd_dq_of_ds_kernel<T, CAUSAL, LIVE, PAD, TBIAS, SLOTS, TEAMS><<<grid, TEAMS * kBwdWaves * 64, lds, s>>>(p);
  return launch_status();
}
template <typename T, bool CAUSAL, int LIVE, bool PAD, bool TBIAS>
static int launch_form(const AttnBwdParams& p, hipStream_t s) {
  const bool two = dq_two_teams((int64_t)p.B * p.H, p.Sq, p.Sk, CAUSAL, p.n_merges);
  return two ? launch_one<T, CAUSAL, LIVE, PAD, TBIAS, 4, 2>(p, s) : launch_one<T, CAUSAL, LIVE, PAD, TBIAS, 4, 1>(p, s);
}
template <typename T>
int launch_dq_of_ds(const AttnBwdParams& p, bool causal, bool tile_bias, hipStream_t s) {
  if (p.d == kD) {
    if (tile_bias) return causal ? launch_form<T, true, 128, false, true>(p, s) : launch_form<T, false, 128, false, true>(p, s);
    return causal ? launch_form<T, true, 128, false, false>(p, s) : launch_form<T, false, 128, false, false>(p, s);
  }
  if (p.d <= 96) return causal ? launch_form<T, true, 96, true, false>(p, s) : launch_form<T, false, 96, true, false>(p, s);
  return causal ? launch_form<T, true, 128, true, false>(p, s) : launch_form<T, false, 128, true, false>(p, s);
}
template int launch_bwd_rows<__bf16>(const AttnBwdParams&, bool, bool, hipStream_t);
template int launch_bwd_rows<_Float16>(const AttnBwdParams&, bool, bool, hipStream_t);
template int launch_dq_of_ds<__bf16>(const AttnBwdParams&, bool, bool, hipStream_t);
template int launch_dq_of_ds<_Float16>(const AttnBwdParams&, bool, bool, hipStream_t);

}  // namespace fo
