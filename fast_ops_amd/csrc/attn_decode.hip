// Attention forward of a few query rows over many keys (generation against a K/V cache): O and LSE as in attn_fwd.hip, same
// numerics (fp32 scores and online softmax, P rounded to the operand type before P V, flash_attention_triton.py:128-255).
//
// What bounds it is reading K and V once. The kernels of attn_fwd.hip give a head one workgroup whose four waves share
// every key tile and own 32 query rows each: with one row, three waves idle, a barrier per tile keeps the copies of one
// tile in flight at a time, and with fewer heads than compute units part of the chip reads nothing. Here
//   * a row block is up to 32 query rows that read the same keys (one MFMA column each): the rows of one head, or, with
//     multi-query K/V (head stride 0), the rows of all heads, whose keys are then read once and not once per head;
//   * the keys of a row block are dealt to the four waves of a workgroup, and, where that leaves compute units without
//     work, to n_split workgroups. A wave streams its own 32-key tiles through its own two LDS buffers: no barrier in
//     the loop, 64 KiB of copies in flight per compute unit at head_dim 128;
//   * row maxima, row sums and O of the waves are merged in LDS at the end, those of several workgroups by a second kernel
//     from fp32 partial results in the caller's workspace.
// One query per head, bf16, the better one of the 128-row kernels -> this, us per call, keys that no cache holds (a GiB of K/V taken
// in turn; in brackets the same K/V again and again): B=4 H=32, 4001 keys at head_dim 128 69 -> 53 (62 -> 44; the kernel alone
// 41 us = 6.4 TB/s, the merge 4.6), B=1 H=32, 4096 keys 64 -> 20 (54 -> 17), 16384 keys 239 -> 57 (195 -> 51), B=16 H=32, 2048 keys 98 -> 96
// (98 -> 96), B=1 H=12, 8192 keys at head_dim 64 81 -> 15 (81 -> 14). The same K/V: 16 queries, B=16 H=32, 9000 keys at 64
// 348 -> 201; multi-query B=14 H=32, 1697 keys at 128 96 -> 15.
#include <type_traits>

#include "attn_common.hpp"

namespace fo {

constexpr int kDecWaves = 4;
constexpr int kDecTile = 32;                     // keys per tile
constexpr float kDecLazyLog2 = 8.0f;             // how far (in log2 units) a tile maximum may exceed the reference before a rescale

template <typename T, int D>
__global__ void __launch_bounds__(kDecWaves * 64) attn_decode_kernel(const DecodeParams prm) {
  typedef typename Ops<T>::vec8 vec8;
  constexpr int ROW_BYTES = D * 2, CHUNKS = ROW_BYTES / 16, ROWS_PER_DMA = 1024 / ROW_BYTES;
  constexpr int TILE_BYTES = kDecTile * ROW_BYTES, N = TILE_BYTES / 1024;      // copies per tile and matrix
  constexpr int KSTEPS = D / 16, DBLK = D / 32;
  constexpr int OROW = D + 4;                    // floats per staged row of O
  static_assert(32 * OROW * 4 <= 4 * TILE_BYTES, "a wave stages its O where its tiles were");
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  FO_LDS char* smem = (FO_LDS char*)smem_raw;    // per wave: K0 | V0 | K1 | V1; then (max, sum) of 4 waves x 32 rows
  const int tid = threadIdx.x;
  const int wave_s = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;

  // ---- work item: (batch, key head, split), row block. Row blocks of one item sit on one XCD (8 ids apart), whose cache
  // then holds the keys they share.
  const int rows = decode_rows(prm.H, prm.n_kv, prm.Sq), n_rb = (rows + 31) / 32;
  const int x = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int rb = j % n_rb, item = (j / n_rb) * 8 + x;
  if (item >= prm.B * prm.n_kv * prm.n_split) return;
  const int split = item % prm.n_split, pair = item / prm.n_split;
  const int b = pair / prm.n_kv, hk = pair % prm.n_kv;
  const int Sk = prm.Sk;
  const T* kbase = (const T*)prm.k + b * prm.ks[0] + hk * prm.ks[1];
  const T* vbase = (const T*)prm.v + b * prm.vs[0] + hk * prm.vs[1];
  auto row_of = [&](int r, int& h, int& s) { if (prm.n_kv == 1) { h = r / prm.Sq; s = r - h * prm.Sq; } else { h = hk; s = r; } };

  // ---- this wave's tiles
  const int n_tiles = (Sk + kDecTile - 1) / kDecTile, n_chunks = prm.n_split * kDecWaves, chunk = split * kDecWaves + wave_s;
  const int t0 = (int)((int64_t)n_tiles * chunk / n_chunks), t1 = (int)((int64_t)n_tiles * (chunk + 1) / n_chunks);
  FO_LDS char* mine = smem + wave_s * 4 * TILE_BYTES;

  // (piece i holds rows ROWS_PER_DMA * i + lane / CHUNKS, 16-byte chunks XOR-swizzled inside a row: see swz)
  uint32_t k_off[N], v_off[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int a = lane / CHUNKS, col = ((lane % CHUNKS) ^ swz<D>(ROWS_PER_DMA * i + a)) * 8;
    k_off[i] = (uint32_t)(a * (int)prm.ks[2] + col) * 2u;
    v_off[i] = (uint32_t)(a * (int)prm.vs[2] + col) * 2u;
  }
  auto issue = [&](int tile, int buf) {
    FO_LDS char* kdst = mine + buf * 2 * TILE_BYTES;
    FO_LDS char* vdst = kdst + TILE_BYTES;
    const int key0 = tile * kDecTile;
    if (key0 + kDecTile <= Sk) {
#pragma unroll
      for (int i = 0; i < N; ++i) dma16_uniform_base((const char*)(kbase + (int64_t)(key0 + ROWS_PER_DMA * i) * prm.ks[2]), k_off[i], kdst + i * 1024);
#pragma unroll
      for (int i = 0; i < N; ++i) dma16_uniform_base((const char*)(vbase + (int64_t)(key0 + ROWS_PER_DMA * i) * prm.vs[2]), v_off[i], vdst + i * 1024);
    } else {
      // rows past the end re-read the last key (masked below)
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int row = ROWS_PER_DMA * i + lane / CHUNKS, col = ((lane % CHUNKS) ^ swz<D>(row)) * 8;
        const int64_t key = min(key0 + row, Sk - 1);
        dma16_lane_ptr(kbase + key * prm.ks[2] + col, kdst + i * 1024);
        dma16_lane_ptr(vbase + key * prm.vs[2] + col, vdst + i * 1024);
      }
    }
  };
  if (t0 < t1) issue(t0, 0);

  // ---- Q^T fragments: lane holds row 32 rb + l32, d = 16 ks + 8 hh ..
  vec8 qf[KSTEPS];
  {
    int h, s;
    row_of(min(32 * rb + l32, rows - 1), h, s);
    const T* qp = (const T*)prm.q + b * prm.qs[0] + h * prm.qs[1] + (int64_t)s * prm.qs[2] + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) qf[ks] = *(const vec8*)(qp + 16 * ks);
    // (waited for here and not inside the loop, where the wait would cover the copies in flight)
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) asm volatile("" ::"v"(qf[ks]));
  }
  f32x16 oacc[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[i][r] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;
  const float c = prm.scale_log2e;

  for (int t = t0; t < t1; ++t) {
    const int buf = (t - t0) & 1;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // this wave has read the other buffer
    if (t + 1 < t1) {
      issue(t + 1, buf ^ 1);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * N) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    FO_LDS const char* kt = mine + buf * 2 * TILE_BYTES;
    FO_LDS const char* vt = kt + TILE_BYTES;
    f32x16 sacc;
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[r] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) sacc = Ops<T>::mfma(row_frag<T, D>(kt, 0, ks, l32, hh), qf[ks], sacc);      // S^T = K Q^T
    if (t * kDecTile + kDecTile > Sk) {
      // register r holds key key_base + (r & 3) + 8 (r >> 2)
      const int lim = t * kDecTile + 4 * hh - Sk + 1;
#pragma unroll
      for (int r = 0; r < 16; ++r) sacc[r] = (lim > -((r & 3) + 8 * (r >> 2))) ? -INFINITY : sacc[r];
    }
    float mloc = sacc[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mloc = fmaxf(mloc, sacc[r]);
    mloc = fmaxf(mloc, half_swap(mloc));
    // (scores of -inf - K may hold it to take keys out - can fill all of a wave's tiles so far, whatever the other waves'
    // keys score: its reference then stays 0 until a key counts, and its sums 0)
    if (__builtin_amdgcn_ballot_w64(mloc * c > m_run * c + kDecLazyLog2) != 0) {
      const float m_new = fmaxf(m_run, mloc);
      const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f((m_run - m_new) * c);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < DBLK; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] *= alpha;
    }
    const float mc = m_run == -INFINITY ? 0.0f : m_run * c;
    vec8 pf[2];
    float psum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[r], c, -mc));
      psum += p;                                                           // in fp32 before rounding (flash_attention_triton.py:203)
      pf[r >> 3][r & 7] = (T)p;
    }
    l_run += psum;
#pragma unroll
    for (int ts = 0; ts < 2; ++ts)
#pragma unroll
      for (int db = 0; db < DBLK; ++db) oacc[db] = Ops<T>::mfma(col_frag<T, D>(vt, ts, db, lane), pf[ts], oacc[db]);
  }

  // ---- merge the four waves
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  FO_LDS float* st = (FO_LDS float*)mine;
  FO_LDS float* ml = (FO_LDS float*)(smem + kDecWaves * 4 * TILE_BYTES);
  const float l_tot = l_run + half_swap(l_run);
  if (hh == 0) { ml[(wave_s * 32 + l32) * 2] = m_run; ml[(wave_s * 32 + l32) * 2 + 1] = l_tot; }
  const int n_here = min(32, rows - 32 * rb);
  if (l32 < n_here) {
#pragma unroll
    for (int db = 0; db < DBLK; ++db)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const f32x4 o4 = {oacc[db][4 * rg], oacc[db][4 * rg + 1], oacc[db][4 * rg + 2], oacc[db][4 * rg + 3]};
        *(FO_LDS f32x4*)(st + l32 * OROW + 32 * db + 8 * rg + 4 * hh) = o4;
      }
  }
  __syncthreads();
  const int64_t row0 = (int64_t)pair * rows + 32 * rb, all_rows = (int64_t)prm.B * prm.H * prm.Sq;
  for (int idx = tid; idx < n_here * (D / 4); idx += kDecWaves * 64) {
    const int r = idx / (D / 4), d4 = idx % (D / 4);
    float m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) m = fmaxf(m, ml[(w * 32 + r) * 2]);
    f32x4 o4 = {0.0f, 0.0f, 0.0f, 0.0f};
    // (no key of this workgroup counts, those of another may: sums of 0. A row without any such key comes out as NaN.)
    const bool none = prm.n_split > 1 && m == -INFINITY;
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) {
      const float f = none ? 0.0f : __builtin_amdgcn_exp2f((ml[(w * 32 + r) * 2] - m) * c);      // (a wave without tiles: 0)
      l += f * ml[(w * 32 + r) * 2 + 1];
      const f32x4 part = *(FO_LDS const f32x4*)((FO_LDS float*)(smem + w * 4 * TILE_BYTES) + r * OROW + 4 * d4);
#pragma unroll
      for (int u = 0; u < 4; ++u) o4[u] += f * part[u];
    }
    if (prm.n_split == 1) {
      int h, s;
      row_of(32 * rb + r, h, s);
      typedef __attribute__((ext_vector_type(4))) T vec4;
      const float inv = 1.0f / l;
      const vec4 out = {(T)(o4[0] * inv), (T)(o4[1] * inv), (T)(o4[2] * inv), (T)(o4[3] * inv)};
      *(vec4*)((T*)prm.o + b * prm.os[0] + h * prm.os[1] + (int64_t)s * prm.os[2] + 4 * d4) = out;
      if (prm.lse != nullptr && d4 == 0) prm.lse[row0 + r] = (m * c + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
    } else {
      *(f32x4*)(prm.ws + (split * all_rows + row0 + r) * D + 4 * d4) = o4;
      if (d4 == 0) {
        f32x2* mlw = (f32x2*)(prm.ws + prm.n_split * all_rows * D) + split * all_rows + row0 + r;
        *mlw = f32x2{m, l};
      }
    }
  }
}

// Partial results of n_split workgroups per row -> O and LSE. One wave per row; lane s first looks after split s (at most 64).
template <typename T, int D>
__global__ void __launch_bounds__(256) attn_decode_merge_kernel(const DecodeParams prm) {
  const int64_t all_rows = (int64_t)prm.B * prm.H * prm.Sq, row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= all_rows) return;
  const int lane = threadIdx.x & 63, n = prm.n_split;
  const f32x2* mlw = (const f32x2*)(prm.ws + n * all_rows * D);
  const f32x2 mine = lane < n ? mlw[lane * all_rows + row] : f32x2{-INFINITY, 0.0f};
  // What bounds this kernel is one latency behind another. So the first splits' sums are asked for together with the references and not
  // behind them, the others eight at a time, and the reductions go over the splits' lanes alone; whole calls, head_dim 128: B=4 H=32,
  // one query x 4001 keys (2 splits) 51.2 -> 50.5 us, B=8 H=32 over one K/V head x 8000 (32 splits) 17.1 -> 15.9, B=1 H=16 over one,
  // 16 queries x 2048 14.1 -> 12.8; head_dim 64: B=1 H=12 x 16000 (21 splits) 19.3 -> 17.1.
  constexpr int PER = D / 64, kEager = 4;
  typedef __attribute__((ext_vector_type(PER))) float vecf;
  auto part = [&](int s) { return *(const vecf*)(prm.ws + (s * all_rows + row) * D + PER * lane); };
  vecf first[kEager];
#pragma unroll
  for (int s = 0; s < kEager; ++s) first[s] = part(s < n ? s : 0);
  float m = mine[0];
  for (int i = 1; i < n; i <<= 1) m = fmaxf(m, __shfl_xor(m, i));      // (lanes from n on hold nothing: lane 0 has all of them)
  m = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, m)));
  const float f = lane < n ? __builtin_amdgcn_exp2f((mine[0] - m) * prm.scale_log2e) : 0.0f;
  float l = f * mine[1];
  for (int i = 1; i < n; i <<= 1) l += __shfl_xor(l, i);
  l = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, l)));
  float o[PER] = {};
  auto add = [&](int s, const vecf& v) {
    const float fs = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), s));
#pragma unroll
    for (int u = 0; u < PER; ++u) o[u] += fs * v[u];
  };
#pragma unroll
  for (int s = 0; s < kEager; ++s)
    if (s < n) add(s, first[s]);
  for (int s0 = kEager; s0 < n; s0 += 8) {                             // (eight at a time, past the end the last one again)
    vecf next[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) next[u] = part(s0 + u < n ? s0 + u : n - 1);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < n) add(s0 + u, next[u]);
  }
  const float inv = 1.0f / l;
  const int64_t bh = row / prm.Sq, s = row - bh * prm.Sq, b = bh / prm.H, h = bh - b * prm.H;
  typedef __attribute__((ext_vector_type(PER))) T vec;
  vec out;
#pragma unroll
  for (int u = 0; u < PER; ++u) out[u] = (T)(o[u] * inv);
  *(vec*)((T*)prm.o + b * prm.os[0] + h * prm.os[1] + s * prm.os[2] + PER * lane) = out;
  if (prm.lse != nullptr && lane == 0) prm.lse[row] = (m * prm.scale_log2e + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
}

int64_t decode_workspace_bytes(int B, int H, int Sq, int D, int n_split) {
  return n_split > 1 ? (int64_t)n_split * B * H * Sq * (D + 2) * (int64_t)sizeof(float) : 0;
}

// How many workgroups share the keys of a row block: as many as make one round of workgroups on the chip, if that gains
// more than the second launch costs. A workgroup by itself streams about 42 bytes per ns, all of them together about
// 6200, the merge takes 3.5 us (B=1 H=32, one query, head_dim 128, 4096 keys: 43 us with one workgroup per head, 30 / 21 /
// 21 / 26 with 2 / 4 / 8 / 16; B=8 H=16, 1024 keys at head_dim 64: 11.0 us with one, 13.8 with two; B=4 H=32, 4001 keys
// at 128: 54 with one, 53 with two). A wave gets at least four tiles.
int decode_split(int B, int H, int n_kv, int Sq, int Sk, int D, int n_cu) {
  const int64_t items = (int64_t)B * n_kv * ((decode_rows(H, n_kv, Sq) + 31) / 32);
  const int tiles = (Sk + kDecTile - 1) / kDecTile;
  const int asked = tune(g_attn_decode_split);
  if (asked > 0) return asked < tiles ? asked : 1;
  int64_t n = n_cu / items;
  if (n > tiles / (4 * kDecWaves)) n = tiles / (4 * kDecWaves);
  if (n > 64) n = 64;
  if (n <= 1) return 1;
  const double bytes = (double)Sk * D * 4, ns_chip = bytes * B * n_kv / 6200.0, ns_one = bytes / 42.0;
  const double one = ns_one > ns_chip ? ns_one : ns_chip, split = (ns_one / n > ns_chip ? ns_one / n : ns_chip) + 3500.0;
  return split < one ? (int)n : 1;
}

template <typename T, int D>
int launch_decode(const DecodeParams& p, hipStream_t stream) {
  constexpr size_t lds = kDecWaves * 4 * kDecTile * D * 2 + kDecWaves * 32 * 2 * sizeof(float);
  static const hipError_t attr = hipFuncSetAttribute((const void*)attn_decode_kernel<T, D>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return FO_ERR_LAUNCH;
  const int64_t items = (int64_t)p.B * p.n_kv * p.n_split, n_rb = (decode_rows(p.H, p.n_kv, p.Sq) + 31) / 32;
  attn_decode_kernel<T, D><<<(unsigned)((items + 7) / 8 * 8 * n_rb), kDecWaves * 64, lds, stream>>>(p);
  if (p.n_split > 1) {
    const int64_t all_rows = (int64_t)p.B * p.H * p.Sq;
    attn_decode_merge_kernel<T, D><<<(unsigned)((all_rows + 3) / 4), 256, 0, stream>>>(p);
  }
  return launch_status();
}
template int launch_decode<__bf16, 64>(const DecodeParams&, hipStream_t);
template int launch_decode<__bf16, 128>(const DecodeParams&, hipStream_t);
template int launch_decode<_Float16, 64>(const DecodeParams&, hipStream_t);
template int launch_decode<_Float16, 128>(const DecodeParams&, hipStream_t);

}  // namespace fo
