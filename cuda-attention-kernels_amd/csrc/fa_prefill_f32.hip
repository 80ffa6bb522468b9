// fp32 FlashAttention-2 prefill on the fp32 matrix cores of MI355X (gfx950), D in {32, 64, 128, 256}.
//
// Serves fp32 Q/K/V: the role of the reference's SIMT kernel attn_fwd_kernel
// (csrc/flash_attn.cu:54-187) and of its Triton kernel's fp32 inputs
// (fused_attn/triton_fwd.py:85-172, 210-222), dense and varlen, with the natural-log LSE
// (triton_fwd.py:169-172).  Both products run on v_mfma_f32_32x32x2_f32, so every product
// and sum is an fp32 operation, and P stays fp32.
//
// A workgroup of 4 waves covers 128 queries of one q-head; wave w owns 32 of them (in small grids 32 queries,
// the key tiles shared out among the waves: KS below).  K and V
// stream through LDS in 32-key fp32 tiles, double-buffered and filled straight from memory.
//
// Operand layout per 32-key block and wave (lane l: j = l % 32, g = l / 32):
//  - S^T = K Q^T over D/2 steps of k = 2.  Step s pairs d = s (lanes g = 0) with d = D/2 + s
//    (lanes g = 1): A = K (lane: key j, that d), B = Q^T (lane: query j, that d).  A lane
//    thus reads four steps of its K row with one 16-byte LDS read and keeps half of its Q row
//    in registers for the whole kernel.
//  - The C fragment gives lane (j, g) query j's scores of keys 8(r/4) + 4g + r%4, r = 0..15.
//  - O^T += V^T P^T over 16 steps of k = 2.  Step r uses, in lane (j, g), the key
//    8(r/4) + 4g + r%4: the one whose probability the lane holds in register r, so P never
//    moves between lanes.  A = V^T, where row i of d block b is d = DB*i + b (DB = D/32
//    blocks), so one LDS read of a V row (32 bytes at D=256 down to 4 at D=32) feeds the
//    step's DB MFMAs.  At D=256 the fp32 accumulators and half a Q row take 256 registers, so
//    that variant runs one wave per SIMD.
//  - K tiles keep 16-byte chunk c of row n at c ^ swz(n), swz(n) = n % 16 (D >= 64) or
//    (n / 2) % 8 (D = 32, whose 128-byte rows put two rows on one bank line): the 16 rows of
//    one read pass hit 16 different bank groups.  A pass over V reads whole rows, so V needs
//    no swizzle (at D=32 the two row halves of a wave share banks: a 2-way conflict on
//    4-byte reads, small beside the 64-cycle MFMAs they feed).
#include <float.h>

#include <algorithm>
#include <cmath>

#include <type_traits>

#include "fa_device.hpp"
#include "fa_internal.hpp"

namespace fa {

namespace {

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// KS (D <= 128): a workgroup covers 32 queries and its waves share out the key tiles, wave w taking tiles w,
// w + 4, ... through LDS of its own, without barriers; the four partial results are merged through LDS at
// the end.  Four times the workgroups with a quarter of the serial chain each (run_fwd_f32 says when).
template <int D, bool KS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 256 || (KS && D >= 64) ? 1 : 2)))
attn_fwd_f32_kernel(const TileArgs a) {
  constexpr int NW = 4;
  constexpr int BN = 32;                      // keys per tile: one 32-key MFMA block
  constexpr int TILE = BN * D;                // floats per K (or V) tile
  constexpr int RPB = KS ? 32 : NW * 32;      // queries per workgroup
  constexpr int QPW = TILE * 4 / 1024 / (KS ? 1 : NW);  // 1-KiB DMA blocks per wave per tile
  constexpr int DB = D / 32;                  // 32-row d blocks of O^T
  constexpr int HS = D / 2;                   // k = 2 steps of S^T
  static_assert(D == 32 || D == 64 || D == 128 || D == 256, "head dim");
  static_assert(TILE * 4 % (1024 * NW) == 0, "direct loads must split evenly over the waves");
  constexpr float NEG_INF = -__builtin_inff();

  // separate arrays so that the compiler can tell a DMA into one buffer from reads of another
  // (KS: a buffer holds one tile per wave; at D=128 one stage of them fills 128 KiB)
  static_assert(!KS || D <= 128, "a tile per wave must fit LDS");
  constexpr bool TWO_STAGES = !KS || D <= 64;
  constexpr int BUF = KS ? NW * TILE : TILE;
  __shared__ __align__(16) float k_buf0[BUF];
  __shared__ __align__(16) float k_buf1[TWO_STAGES ? BUF : 4];
  __shared__ __align__(16) float v_buf0[BUF];
  __shared__ __align__(16) float v_buf1[TWO_STAGES ? BUF : 4];

  // ---- work item: (batch or sequence, q-head, 128-query block), rank-major ---------------
  // All (batch, q-head) pairs at one rank run together (heaviest causal blocks first), the
  // q-heads of one kv-head side by side; xcd_remap gives each XCD a contiguous range.  The ranks of a
  // dense causal call are dealt to the XCDs instead: a contiguous range gave the first XCD all the heaviest
  // (us, B=4 H=16 N=1024 D=32 / 64 / 128 / 256: 79 / 141 / 266 / 650 -> 57 / 104 / 190 / 354).  A varlen grid's
  // heaviest ranks are mostly empty, and dealing spreads a sequence's K/V over all XCDs: 4 sequences up to
  // 1500 tokens, 16 heads, D=64: 177 us in order and 197 dealt.
  const int nbh = a.total / a.n_rowblk;
  const int logical = a.causal && !a.varlen ? (int)blockIdx.x : xcd_remap((int)blockIdx.x, a.total);
  const int mrev = logical / nbh;
  const int item = logical % nbh;
  const int hq = item % a.hq;
  const int b = item / a.hq;
  const int kvh = hq / a.group;
  const int rb = a.causal ? (a.n_rowblk - 1 - mrev) : mrev;

  int seq_q = a.nq, seq_k = a.nk;
  int64_t qtok0 = 0, ktok0 = 0;
  if (a.varlen) {
    const int qs = __builtin_amdgcn_readfirstlane(a.cu_q[b]);
    const int ks = __builtin_amdgcn_readfirstlane(a.cu_k[b]);
    seq_q = __builtin_amdgcn_readfirstlane(a.cu_q[b + 1]) - qs;
    seq_k = __builtin_amdgcn_readfirstlane(a.cu_k[b + 1]) - ks;
    qtok0 = qs;
    ktok0 = ks;
  }
  const int r0 = rb * RPB;
  if (r0 >= seq_q) return;  // uniform over the workgroup (zero-length sequences exit here)
  const int offset = seq_k - seq_q;  // bottom-right causal alignment (reference.py:24-33)
  int khi = seq_k;
  if (a.causal) khi = min(khi, min(r0 + RPB, seq_q) + offset);
  const int n_tiles = khi > 0 ? (khi + BN - 1) / BN : 0;

  // ---- lane roles --------------------------------------------------------------------
  const int tid = (int)threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 5, j = lane & 31;
  const int wr0 = KS ? r0 : r0 + wave * 32;
  const int qi = wr0 + j;
  const bool row_ok = qi < seq_q;
  const bool wave_active = wr0 < seq_q;
  // keys at or beyond mask_from are not visible to every row of this wave
  int mask_from = khi;
  if (a.causal && wave_active) mask_from = min(khi, wr0 + offset + 1);
  // keys below wave_khi are visible to some row of this wave; later tiles only take part in
  // the DMA and the barriers
  const int wave_khi = !wave_active ? 0 : (a.causal ? min(khi, min(wr0 + 32, seq_q) + offset) : khi);
  const int qlim = qi + offset;  // last key this lane's row may see (causal)

  // A negative scale is applied by negating Q (exact); c = |scale| * log2(e) > 0.
  const float c = fmaxf(fabsf(a.qk_scale), kMinScale);
  const uint32_t qsign = a.qk_scale < 0.f ? 0x80000000u : 0u;

  // ---- Q: half of this lane's row, resident (rows past the end read row 0, zeroed) ----
  float qreg[HS];
  {
    const int64_t qrow = qtok0 + (row_ok ? qi : 0);
    const float* qp = (const float*)a.q + (int64_t)b * a.sqb + (int64_t)hq * a.sqh + qrow * a.sqn + g * HS;
    const uint32_t keep = row_ok ? 0xffffffffu : 0u;
#pragma unroll
    for (int i = 0; i < HS / 4; ++i) {
      const u32x4 w = ld16(qp + 4 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) qreg[4 * i + e] = __builtin_bit_cast(float, (w[e] ^ qsign) & keep);
    }
  }

  auto swz = [](int n) __attribute__((always_inline)) { return D >= 64 ? n % 16 : (n >> 1) & 7; };

  // ---- K/V tiles: global -> LDS (loads past the tile's last valid key return zeros) -----
  const uint8_t* kbase = (const uint8_t*)a.k + ((int64_t)b * a.skb + (int64_t)kvh * a.skh + ktok0 * a.skn) * 4;
  const uint8_t* vbase = (const uint8_t*)a.v + ((int64_t)b * a.svb + (int64_t)kvh * a.svh + ktok0 * a.svn) * 4;
  const int64_t krow_bytes = a.skn * 4, vrow_bytes = a.svn * 4;
  auto limit = [&](int n0, int64_t row_bytes) __attribute__((always_inline)) {
    const int valid = min(khi - n0, BN);
    return __builtin_amdgcn_readfirstlane(valid > 0 ? (uint32_t)(valid - 1) * (uint32_t)row_bytes + (uint32_t)(D * 4)
                                                    : 0u);
  };
  auto load_tiles = [&](int n0, float* kd, float* vd) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kbase + (int64_t)n0 * krow_bytes, limit(n0, krow_bytes));
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vbase + (int64_t)n0 * vrow_bytes, limit(n0, vrow_bytes));
#pragma unroll
    for (int i = 0; i < QPW; ++i) {
      const int blk = (KS ? 0 : wave * QPW) + i;  // within the tile (KS: the wave's own)
      const int byte = blk * 1024 + lane * 16;
      const int r = byte / (D * 4), p = (byte % (D * 4)) / 16;
      lds_dma16<false>(rk, (uint8_t*)kd + blk * 1024, r * (int)krow_bytes + ((p ^ swz(r)) * 16));
      lds_dma16<false>(rv, (uint8_t*)vd + blk * 1024, r * (int)vrow_bytes + p * 16);
    }
  };

  f32x16 oacc[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d) oacc[d] = f32x16{};
  float m_run = NEG_INF, l_run = 0.f;  // running max (scaled log2 domain), this lane's row-sum share

  // ---- one 32-key tile --------------------------------------------------------------------
  auto tile = [&](const float* Ks, const float* Vs, int n0) __attribute__((always_inline)) {
    // S^T, in two accumulators so that consecutive MFMAs do not depend on each other
    f32x16 s0 = f32x16{}, s1 = f32x16{};
#pragma unroll
    for (int s4 = 0; s4 < HS / 4; ++s4) {
      const int chunk = (g * (HS / 4) + s4) ^ swz(j);
      const f32x4 kv = __builtin_bit_cast(f32x4, ld16(Ks + j * D + chunk * 4));
      s0 = mfma_f32(kv[0], qreg[4 * s4 + 0], s0);
      s1 = mfma_f32(kv[1], qreg[4 * s4 + 1], s1);
      s0 = mfma_f32(kv[2], qreg[4 * s4 + 2], s0);
      s1 = mfma_f32(kv[3], qreg[4 * s4 + 3], s1);
    }
    f32x16 sc;
#pragma unroll
    for (int r = 0; r < 16; ++r) sc[r] = s0[r] + s1[r];
    if (n0 + BN > mask_from) {
      __asm__ volatile("");  // keep the rare masking branch out of the common path
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = n0 + 8 * (r >> 2) + 4 * g + (r & 3);
        const bool ok = (n < khi) & ((a.causal == 0) | (n <= qlim));
        sc[r] = ok ? sc[r] : NEG_INF;
      }
    }
    float mx = sc[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = vmax(mx, sc[r]);
    const float m_new = vmax(m_run, max_xor32(mx * c));
    const float m_safe = (m_new == NEG_INF) ? 0.f : m_new;
    const float alpha = fast_exp2(m_run - m_safe);
    m_run = m_new;
    float p[16];
    float rs = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      p[r] = fast_exp2(__builtin_fmaf(sc[r], c, -m_safe));
      rs += p[r];
    }
    l_run = l_run * alpha + rs;
#pragma unroll
    for (int d = 0; d < DB; ++d) oacc[d] *= alpha;
    // O^T += V^T P^T
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float* vp = Vs + (8 * (r >> 2) + 4 * g + (r & 3)) * D + DB * j;
      if constexpr (DB == 8) {
        const f32x4 w0 = __builtin_bit_cast(f32x4, ld16(vp)), w1 = __builtin_bit_cast(f32x4, ld16(vp + 4));
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          oacc[d] = mfma_f32(w0[d], p[r], oacc[d]);
          oacc[d + 4] = mfma_f32(w1[d], p[r], oacc[d + 4]);
        }
      } else if constexpr (DB == 4) {
        const f32x4 w = __builtin_bit_cast(f32x4, ld16(vp));
#pragma unroll
        for (int d = 0; d < 4; ++d) oacc[d] = mfma_f32(w[d], p[r], oacc[d]);
      } else if constexpr (DB == 2) {
        const f32x2 w = __builtin_bit_cast(f32x2, ld8(vp));
#pragma unroll
        for (int d = 0; d < 2; ++d) oacc[d] = mfma_f32(w[d], p[r], oacc[d]);
      } else {
        oacc[0] = mfma_f32(*vp, p[r], oacc[0]);
      }
    }
  };

  // ---- main loop, unrolled by 2 so that every buffer is named at compile time ------------
  if constexpr (KS) {
    const int own = wave * TILE;
    if constexpr (TWO_STAGES) {
      if (wave < n_tiles) load_tiles(wave * BN, k_buf0 + own, v_buf0 + own);
      auto step = [&](auto stage_tag, int t) __attribute__((always_inline)) {
        constexpr int ST = decltype(stage_tag)::value;
        lds_dma_wait();
        __asm__ volatile("" ::: "memory");
        // (the stage of tile t - 4 was read before that tile's last MFMAs issued)
        if (t + NW < n_tiles) load_tiles((t + NW) * BN, (ST == 0 ? k_buf1 : k_buf0) + own, (ST == 0 ? v_buf1 : v_buf0) + own);
        tile((ST == 0 ? k_buf0 : k_buf1) + own, (ST == 0 ? v_buf0 : v_buf1) + own, t * BN);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage has been read
        __asm__ volatile("" ::: "memory");
      };
      for (int t = wave; t < n_tiles; t += 2 * NW) {
        step(std::integral_constant<int, 0>{}, t);
        if (t + NW < n_tiles) step(std::integral_constant<int, 1>{}, t + NW);
      }
    } else {
      for (int t = wave; t < n_tiles; t += NW) {
        load_tiles(t * BN, k_buf0 + own, v_buf0 + own);
        lds_dma_wait();
        __asm__ volatile("" ::: "memory");
        tile(k_buf0 + own, v_buf0 + own, t * BN);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage has been read
        __asm__ volatile("" ::: "memory");
      }
    }
  } else {
    if (n_tiles > 0) load_tiles(0, k_buf0, v_buf0);
    auto step = [&](auto stage_tag, int t) __attribute__((always_inline)) {
      constexpr int ST = decltype(stage_tag)::value;
      const float* kc = ST == 0 ? k_buf0 : k_buf1;  // holds tile t
      const float* vc = ST == 0 ? v_buf0 : v_buf1;
      float* kn = ST == 0 ? k_buf1 : k_buf0;  // held tile t-1 (every wave is done with it), takes t+1
      float* vn = ST == 0 ? v_buf1 : v_buf0;
      lds_dma_wait();
      __syncthreads();
      if (t + 1 < n_tiles) load_tiles((t + 1) * BN, kn, vn);
      if (t * BN < wave_khi) tile(kc, vc, t * BN);
    };
    for (int t = 0; t < n_tiles; t += 2) {
      step(std::integral_constant<int, 0>{}, t);
      if (t + 1 < n_tiles) step(std::integral_constant<int, 1>{}, t + 1);
    }
  }

  if constexpr (KS) {
    // ---- merge: O = sum_w 2^(m_w - m) O_w / sum_w 2^(m_w - m) l_w over the waves ------------
    // O_w goes to the wave's own K buffer as rows of D floats, 16-byte chunks XOR-swizzled by row: lane
    // (j, g) holds columns DB*(8q + 4g) .. + 4*DB - 1 of row j in registers 4q..4q+3 of its DB blocks.
    constexpr int NCH = D / 4;
    __shared__ f32x2 ml[NW][32];
    const float l_w = sum_xor32(l_run);
    float* part = k_buf0 + wave * TILE;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
#pragma unroll
      for (int cc = 0; cc < DB; ++cc) {
        f32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = oacc[(4 * cc + e) % DB][4 * q4 + (4 * cc + e) / DB];
        *(f32x4*)(part + j * D + (((DB * (2 * q4 + g) + cc) ^ (j & (NCH - 1))) * 4)) = w;
      }
    }
    if (g == 0) ml[wave][j] = f32x2{m_run, l_w};
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32 * NCH / 256; ++i) {
      const int idx = tid + 256 * i, row = idx / NCH, ch = idx % NCH;
      f32x2 st[NW];
#pragma unroll
      for (int w = 0; w < NW; ++w) st[w] = ml[w][row];
      const float m = vmax(vmax(st[0][0], st[1][0]), vmax(st[2][0], st[3][0]));
      const float m_ref = (m == NEG_INF) ? 0.f : m;
      float l = 0.f;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float f = fast_exp2(st[w][0] - m_ref);  // 0 for a wave that saw no key of this row
        l += f * st[w][1];
        o += f * *(const f32x4*)(k_buf0 + w * TILE + row * D + ((ch ^ (row & (NCH - 1))) * 4));
      }
      if (r0 + row >= seq_q) continue;
      const float l_safe = (l == 0.f) ? 1.f : l;
      const float inv = 1.f / l_safe;
      float* op = (float*)a.o + (int64_t)b * a.sob + (int64_t)hq * a.soh + (qtok0 + r0 + row) * a.son + 4 * ch;
      st8(op, __builtin_bit_cast(u32x2, f32x2{o[0] * inv, o[1] * inv}));
      st8(op + 2, __builtin_bit_cast(u32x2, f32x2{o[2] * inv, o[3] * inv}));
      if (a.lse != nullptr && ch == 0)
        a.lse[(int64_t)b * a.slb + (int64_t)hq * a.slh + (qtok0 + r0 + row)] = (m + __log2f(l_safe)) * kLn2;
    }
    return;
  }

  // ---- epilogue ------------------------------------------------------------------------
  if (!wave_active) return;
  const float l_tot = sum_xor32(l_run);
  if (!row_ok) return;
  // rows that saw no key have l == 0 and emit zeros (triton_fwd.py:163-165)
  const float l_safe = (l_tot == 0.f) ? 1.f : l_tot;
  const float inv = 1.f / l_safe;
  float* op = (float*)a.o + (int64_t)b * a.sob + (int64_t)hq * a.soh + (qtok0 + qi) * a.son;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int i = 8 * (r >> 2) + 4 * g + (r & 3);  // O^T row of register r: d = DB*i + block
    if constexpr (DB == 1) {
      op[i] = oacc[0][r] * inv;
    } else {
#pragma unroll
      for (int d = 0; d < DB; d += 2) {
        st8(op + DB * i + d, u32x2{__builtin_bit_cast(uint32_t, oacc[d][r] * inv),
                                   __builtin_bit_cast(uint32_t, oacc[d + 1][r] * inv)});
      }
    }
  }
  if (a.lse != nullptr && g == 0) {
    a.lse[(int64_t)b * a.slb + (int64_t)hq * a.slh + (qtok0 + qi)] = (m_run + __log2f(l_safe)) * kLn2;
  }
}

template <int D>
hipError_t launch_f32(const TileArgs& a, bool key_split, hipStream_t stream) {
  if constexpr (D <= 128) {
    if (key_split) {
      hipLaunchKernelGGL((attn_fwd_f32_kernel<D, true>), dim3((unsigned)a.total), dim3(256), 0, stream, a);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((attn_fwd_f32_kernel<D, false>), dim3((unsigned)a.total), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace

// Whether a workgroup per 32 queries with the keys shared out among its waves (KS) beats one per 128 queries.
// Both in units of one 32-key tile of a 4-wave workgroup, per compute unit: the plain kernel takes its
// heaviest row block or the mean load of the 256 CUs, whichever is longer; KS takes a quarter of the tiles, 10%
// more for K/V that four times as many workgroups fetch, and 1.1 tiles to start and merge each workgroup.
// At D=128 a CU runs one KS workgroup with a single stage, so a started round counts whole (not causal, B=11 H=8
// N=151, 440 workgroups: 31.8 and 36.6).  D=64, causal unless said, us plain and KS: B=2 H=4 N=256 22.3 and 10.0; 8
// heads N=1000 74.9 and 25.2; B=4 H=8 N=1000 78.2 and 59.6 (not causal 84.4 and 95.9); B=8 H=16 N=256 24.6 and 29.4;
// B=8 H=16 N=2048 570 and 725.
static bool f32_key_split_pays(const fa_fwd_params& p) {
  constexpr double kCus = 256;
  const double heads = (double)p.batch * p.heads_q, tiles = (p.seqlen_k + 31) / 32;
  auto mean_tiles = [&](int rows) {  // over the row blocks; a causal first block sees nk - nq + rows keys
    if (!p.causal) return tiles;
    return 0.5 * (tiles + std::min(tiles, std::max(1.0, (double)(p.seqlen_k - p.seqlen_q + rows) / 32)));
  };
  const double plain_wgs = heads * ((p.seqlen_q + 127) / 128), ks_wgs = heads * ((p.seqlen_q + 31) / 32);
  const double plain = std::max(tiles, plain_wgs * mean_tiles(128) / kCus);
  const double rounds = p.head_dim == 128 && ks_wgs > kCus ? std::ceil(ks_wgs / kCus) : ks_wgs / kCus;
  const double ks = std::max(1.1 * tiles / 4 + 1.1, rounds * (1.1 * (mean_tiles(32) + 1.5) / 4 + 1.1));
  return ks < plain;
}

fa_status run_fwd_f32(const fa_fwd_params& p, bool varlen, hipStream_t stream, const char** err) {
  TileArgs a = common_args(p);
  a.o = p.o;
  a.sob = p.o_stride_b;
  a.soh = p.o_stride_h;
  a.son = p.o_stride_n;
  a.lse = p.lse;
  a.slb = p.lse_stride_b;
  a.slh = p.lse_stride_h;
  a.varlen = varlen ? 1 : 0;
  if (varlen) {
    a.cu_q = p.cu_seqlens_q;
    a.cu_k = p.cu_seqlens_k;
    a.nq = p.max_seqlen_q;
    a.nk = p.max_seqlen_k;
    a.sqb = a.skb = a.svb = a.sob = a.slb = 0;  // rows are addressed by packed token index
  }
  if (a.nq <= 0 || p.batch <= 0) return FA_OK;
  const bool key_split = !varlen && p.head_dim <= 128 && f32_key_split_pays(p);
  const int rpb = key_split ? 32 : 128;
  a.n_rowblk = (a.nq + rpb - 1) / rpb;
  const int64_t total = (int64_t)p.batch * p.heads_q * a.n_rowblk;
  if (total > INT32_MAX) {
    *err = "grid too large";
    return FA_ERR_UNSUPPORTED;
  }
  a.total = (int32_t)total;
  const hipError_t e = p.head_dim == 256 ? launch_f32<256>(a, key_split, stream)
                       : p.head_dim == 128 ? launch_f32<128>(a, key_split, stream)
                       : p.head_dim == 64 ? launch_f32<64>(a, key_split, stream)
                                          : launch_f32<32>(a, key_split, stream);
  return hip_status(e, err);
}

}  // namespace fa
