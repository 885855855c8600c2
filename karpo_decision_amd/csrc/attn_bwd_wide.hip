// The backward at head size 512 for one sequence (a training sequence's global layer) as two matrix-product kernels
// per chunk of query rows, with P and dS of the chunk held in the workspace as bf16 (the precision at which they enter
// the matrix products in every backward kernel here):
//   1. bwd_wide_ds_kernel: S = Q K^T and dP = dO V^T of a tile of 256 rows x 128 keys, then P and dS, stored;
//   2. bwd_wide_grad_kernel: dQ = dS K, dK = dS^T Q and dV = P^T dO, 256 x 256 outputs per workgroup.
// Why: at this head size a wave cannot hold the operands and accumulators of a fused tile (attn_bwd_pair.hip: pairs
// of waves that exchange partial sums through LDS, one wave per SIMD, three barriers per 32-row step, 24-26% of the
// MFMA rate), and it computes S and dP twice (seven products). P and dS cost 10 bytes of traffic per visible pair and
// 5,120 FLOPs need them, so keeping them takes less time than either the recomputation or the exchange: five products,
// each a plain tiled matrix product with every accumulator in one wave's registers. Measured against the wave pairs as
// they are now (32 / 4 heads, causal, MI355X): 838 -> 253 us at 1,024 rows, 1.80 -> 0.63 ms at 2,048, 10.7 -> 6.1 ms at
// 8,192, 41 -> 23 ms at 16,384. In one chunk it is faster at every size tried (1 to 16,384 rows over 1 to 65,536 keys,
// groups 1 to 16), in several where they are long enough (wide_chunks_pay, capi.cpp); such calls take this path when the
// workspace has room for it.
//
// P and dS in the workspace: per head [key block of 16][chunk of 8 rows][16 keys][8 rows] bf16, the 16 keys of a
// 256-byte run XOR-swizzled by the chunk index (key ^ 4 (chunk % 4): free of bank conflicts read either way), the layout
// in which a tile is read from LDS: a copy instruction moves 1 KiB of consecutive bytes. A lane of kernel 1 holds one
// key's scores of 8 consecutive rows (the MFMA's A rows are taken in key_row order) and stores them as one 16-byte
// chunk; dK and dV read those chunks directly as MFMA operands, dQ reads the same tile transposed.
//
// Chunks of rows run in ascending order. dQ of a chunk's rows is complete within it; dK and dV go on from one chunk to
// the next in fp32 (workspace, in the accumulators' register order) and are rounded once, in the last chunk.
// Every sum has a fixed order (no atomics): repeated calls with the same chunk size are bitwise equal (it sets where dK's
// and dV's sums pass from one head of a group to the next).
//
// Outside the mask P and dS are exact zeros, and those enter the products with whatever the other operand holds: a NaN or
// infinity in a K row reaches dQ of every row of the 256-row tiles that visit its 32-key step, one in a Q or dO row
// dK or dV of the 256-key tiles that visit its 32-row step (the wave pairs: tiles of 64 query vectors, and of 64
// keys). One in a V row reaches only dQ of the rows that see it. Rows past the sequence are never read.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "bwd_common.h"
#include "internal.h"
#include "karpo_attn.h"
#include "mfma_common.h"
#include "plan_common.h"

namespace karpo {

constexpr int kWideD = 512;
constexpr int kWideThreads = 512;               // kernel 1: eight waves
constexpr int kGradThreads = 256;               // kernel 2: four waves
constexpr int kDsRows = 256, kDsKeys = 128;     // kernel 1's tile
constexpr int kDsStep = 32;                     // elements of D per step
constexpr int kGradTile = 256, kGradStep = 32;  // kernel 2's outputs (both ways) and contraction step
constexpr int kRing = 4;                        // buffers: three steps of copies ahead

// The sequence's bounds, clamped to the call's rows.
struct WideSeq {
  int qa, lq, ka, lk;
  __device__ __forceinline__ explicit WideSeq(const BwdWideParams& w) {
    qa = w.b.q_cu[0];
    ka = w.b.k_cu[0];
    lq = min(w.b.q_cu[1], (int)w.b.total_q) - qa;
    lk = min(w.b.k_cu[1], w.total_k) - ka;
  }
  // The first query row that sees `key` (no left bound): key - right <= row + lk - lq.
  __device__ __forceinline__ int first_row(int right, int key) const {
    if (right < 0) return 0;
    const int64_t r = (int64_t)key - right - (lk - lq);
    return r < 0 ? 0 : (int)min(r, (int64_t)INT32_MAX);
  }
};

// Transposed read of a P or dS tile (chunks as columns): the lane's address in its first 16 keys and 32 rows.
__device__ __forceinline__ int x_tr_base(int lane, int rr) {
  const int g = lane >> 4, jl = lane & 15;
  const int c = 2 * (g & 1) + ((jl >> 1) & 1);
  return c * 256 + (((4 * rr + 8 * (g >> 1) + (jl >> 2)) ^ (c << 2)) * 16) + (jl & 1) * 8;
}

// Work index -> head with XCD w % 8 given heads that are neighbours (the same key/value head) where the count allows.
__device__ __forceinline__ int spread_head(int i, int n) { return n % 8 == 0 ? (i % 8) * (n / 8) + i / 8 : i; }

// s_barrier after the wave's own LDS accesses, without the fence of __syncthreads (which waits for every copy in
// flight): the copies a step needs are waited for by count.
__device__ __forceinline__ void step_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---- kernel 1: P and dS of 256 rows x 128 keys of one head (eight waves of 64 x 64), for a run of key tiles: the next
// tile's first copies are in flight while this one's P and dS are formed and stored, and a tile's exponentials run
// beside its dP products. 770 TFLOP/s over the eight chunks of 16,384 rows (32 / 4 heads), 40% MFMA-busy: bound by its
// copies and stores, which overlap the products badly (the last chunk: 2.5 ms; without its copies 1.67, its copies alone
// 1.71). Besides the waits below the compiler adds its own before the LDS reads of a tile's first three steps after
// another tile (vmcnt 19, 12, 11: it does not follow which copy fills which buffer), so most of the 16 stores are waited for
// there; and 176 SGPRs are spilled to VGPR lanes (171 lane moves in the tile loop).
__global__ __launch_bounds__(kWideThreads, 2) void bwd_wide_ds_kernel(BwdWideParams w) {
  constexpr int STEPS = kWideD / kDsStep;  // per product
  constexpr int ALL = 2 * STEPS;           // S, then dP
  static_assert(ALL % kRing == 0 && STEPS == 16, "a tile starts in buffer 0; four exponentials per dP step");
  constexpr int AT = kDsRows * kDsStep * 2, BT = kDsKeys * kDsStep * 2;
  constexpr int COPIES = 3, STORES = 16;  // vector-memory operations of a wave per step and per tile's end
  __shared__ __attribute__((aligned(1024))) char a0_s[AT], a1_s[AT], a2_s[AT], a3_s[AT];
  __shared__ __attribute__((aligned(1024))) char b0_s[BT], b1_s[BT], b2_s[BT], b3_s[BT];
  __shared__ __attribute__((aligned(16))) float st_s[2][kDsRows];  // the rows' log2 LSE and -D

  const BwdParams& p = w.b;
  const WideSeq s(w);
  const int key_tiles = w.keys / kDsKeys, runs = (key_tiles + w.run - 1) / w.run;
  const int head = spread_head(blockIdx.x % p.heads, p.heads);
  const int rest = blockIdx.x / p.heads;
  const int rt = rest / runs;
  const int r0 = w.r_begin + rt * kDsRows;
  int kt = (rest - rt * runs) * w.run;
  // the tiles that kernel 2 reads (keys in tiles of 256), and of those the ones that a row of this tile sees
  if (r0 >= s.lq) return;
  const int top = (int)min((int64_t)r0 + kDsRows - 1 + (s.lk - s.lq) + (p.right < 0 ? 0 : p.right), (int64_t)s.lk - 1);
  const int seen = p.right < 0 ? s.lk : top + 1;  // keys
  const int last = min((seen + kDsKeys - 1) / kDsKeys, kt + w.run);
  const int read = min((seen + kGradTile - 1) / kGradTile * (kGradTile / kDsKeys), kt + w.run);
  if (seen <= 0 || kt >= read) return;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int wr = wave >> 1, wc = wave & 1;
  // this lane's chunk (rows rt*256 + wr*64 + rb*32 + kc*16 + half*8 .. +8) of key kt*128 + wc*64 + cb*32 + col
  char* const out_p = (char*)(w.p + (int64_t)head * w.keys * w.rows);
  char* const out_s = (char*)(w.ds + (int64_t)head * w.keys * w.rows);
  const uint32_t run = (uint32_t)(w.rows / 8) * 256u;  // bytes per block of 16 keys
  uint32_t out_base = (uint32_t)(kt * 8 + wc * 4 + (col >> 4)) * run + (uint32_t)(rt * 32 + wr * 8 + half) * 256u;
  const uint32_t out_key[2] = {(uint32_t)((col & 15) ^ (half << 2)) * 16u,
                               (uint32_t)((col & 15) ^ ((2 + half) << 2)) * 16u};
  if (kt < last) {
    {
      const int row = r0 + (tid & 255), which = tid >> 8;
      st_s[which][tid & 255] = row < s.lq ? p.stats[((int64_t)head * 2 + which) * p.total_q + s.qa + row]
                                          : (which ? 0.f : INFINITY);  // a row past the sequence has P = 0
    }
    const int kvh = head / p.group;
    const uint16_t* const q = p.q + (int64_t)(s.qa + r0) * p.sq_t + (int64_t)head * p.sq_h;
    const uint16_t* const o = p.dout + (int64_t)(s.qa + r0) * p.sdo_t + (int64_t)head * p.sdo_h;
    const uint16_t* k = p.k + (int64_t)(s.ka + kt * kDsKeys) * p.sk_t + (int64_t)kvh * p.sk_h;
    const uint16_t* v = p.v + (int64_t)(s.ka + kt * kDsKeys) * p.sv_t + (int64_t)kvh * p.sv_h;
    const int64_t k_tile = (int64_t)kDsKeys * p.sk_t, v_tile = (int64_t)kDsKeys * p.sv_t;
    const int rows = min(s.lq - r0, kDsRows);
    // tiles in the S layout of 32 columns (16 rows x 64 B per copy): wave w copies A rows 32w .. +32, B rows 16w .. +16
    int lrow, lcol;
    s_dma_source<kDsStep>(0, lane, &lrow, &lcol);
    const uint32_t q_off = (uint32_t)((wave * 32 + lrow) * (int)p.sq_t + lcol) * 2u;
    const uint32_t o_off = (uint32_t)((wave * 32 + lrow) * (int)p.sdo_t + lcol) * 2u;
    const uint32_t k_off = (uint32_t)((wave * 16 + lrow) * (int)p.sk_t + lcol) * 2u;
    const uint32_t v_off = (uint32_t)((wave * 16 + lrow) * (int)p.sv_t + lcol) * 2u;
    // step i of the tile at k, v (with `keys` of its keys in the sequence)
    auto copy = [&](int i, const uint16_t* kb, const uint16_t* vb, int keys, KA_LDS char* a, KA_LDS char* b) {
      const bool second = i >= STEPS;
      const int at = (second ? i - STEPS : i) * kDsStep;
      const int a_t = (int)(second ? p.sdo_t : p.sq_t) * 2, b_t = (int)(second ? p.sv_t : p.sk_t) * 2;
      const uint32_t a_off = second ? o_off : q_off;
#pragma unroll
      for (int r = 0; r < 2; ++r)
        dma_16b((second ? o : q) + at, rows * a_t, a + (wave * 2 + r) * 1024, a_off + (uint32_t)(r * 16 * a_t));
      dma_16b((second ? vb : kb) + at, keys * b_t, b + wave * 1024, second ? v_off : k_off);
    };
    const int arow = key_row(col);
    const int a_read[2] = {s_offset<kDsStep>(wr * 64 + arow, half), s_offset<kDsStep>(wr * 64 + arow, 2 + half)};
    const int b_read[2] = {s_offset<kDsStep>(wc * 64 + col, half), s_offset<kDsStep>(wc * 64 + col, 2 + half)};
    KA_LDS char* const at[kRing] = {(KA_LDS char*)a0_s, (KA_LDS char*)a1_s, (KA_LDS char*)a2_s, (KA_LDS char*)a3_s};
    KA_LDS char* const bt[kRing] = {(KA_LDS char*)b0_s, (KA_LDS char*)b1_s, (KA_LDS char*)b2_s, (KA_LDS char*)b3_s};
    const float c = p.c;

    int keys = min(s.lk - kt * kDsKeys, kDsKeys);
#pragma unroll
    for (int i = 0; i < kRing - 1; ++i) copy(i, k, v, keys, at[i], bt[i]);
    wait_vmcnt<2 * COPIES>();
    step_barrier();
    for (bool start = true;; start = false) {
      const bool more = kt + 1 < last;
      const int k0 = kt * kDsKeys, keys_next = min(s.lk - k0 - kDsKeys, kDsKeys);
      f32x16 st[2][2], dp[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          st[i][j] = f32x16{};
          dp[i][j] = f32x16{};
        }
#pragma unroll
      for (int i = 0; i < ALL; ++i) {
        constexpr int AHEAD = kRing - 1;
        KA_LDS char* const an = at[(i + AHEAD) % kRing];
        KA_LDS char* const bn = bt[(i + AHEAD) % kRing];
        if (i + AHEAD < ALL) copy(i + AHEAD, k, v, keys, an, bn);
        else if (more) copy(i + AHEAD - ALL, k + k_tile, v + v_tile, keys_next, an, bn);
        __builtin_amdgcn_sched_barrier(0);  // the copies are issued first
        const KA_LDS char* const a = at[i % kRing];
        const KA_LDS char* const b = bt[i % kRing];
#pragma unroll
        for (int kk = 0; kk < kDsStep / 16; ++kk) {
          bf16x8 x[2], y[2];
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            x[m] = *(const KA_LDS bf16x8*)(a + a_read[kk] + m * 2048);
            y[m] = *(const KA_LDS bf16x8*)(b + b_read[kk] + m * 2048);
          }
#pragma unroll
          for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int n = 0; n < 2; ++n) {
              f32x16& acc = i < STEPS ? st[m][n] : dp[m][n];
              acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[m], y[n], acc, 0, 0, 0);
            }
        }
        if (i >= STEPS) {  // four exponentials of P beside the dP products
          const int e = i - STEPS, rb = e >> 3, kc = (e >> 2) & 1, th = (e >> 1) & 1, cb = e & 1;
          const f32x4 l = *(const f32x4*)&st_s[0][wr * 64 + rb * 32 + kc * 16 + half * 8 + th * 4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int at4 = kc * 8 + th * 4 + t;
            st[rb][cb][at4] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[rb][cb][at4], c, -l[t]));
          }
        }
        if (i + 1 < ALL) {
          // the next step's copies are done; the last tile's stores were issued between the copies of steps 2 and 3
          if (i + AHEAD >= ALL && !more) wait_vmcnt<0>();
          else if (i < 2 && !start) wait_vmcnt<2 * COPIES + STORES>();
          else wait_vmcnt<2 * COPIES>();
          step_barrier();
        }
      }
      const bool whole = k0 + kDsKeys <= s.lk && r0 >= s.first_row(p.right, k0 + kDsKeys - 1);
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
          const int lr = wr * 64 + rb * 32 + kc * 16 + half * 8;  // the chunk's first row in the tile
          const f32x4 d0 = *(const f32x4*)&st_s[1][lr], d1 = *(const f32x4*)&st_s[1][lr + 4];
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) {
            float x[8], y[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
              x[t] = st[rb][cb][kc * 8 + t];
              y[t] = x[t] * (dp[rb][cb][kc * 8 + t] + (t < 4 ? d0[t] : d1[t - 4]));
            }
            if (!whole) {
              const int key = k0 + wc * 64 + cb * 32 + col;
              const int first = key < s.lk ? s.first_row(p.right, key) : INT32_MAX;
#pragma unroll
              for (int t = 0; t < 8; ++t) {
                const bool vis = r0 + lr + t >= first;
                x[t] = vis ? x[t] : 0.f;
                y[t] = vis ? y[t] : 0.f;
              }
            }
            const uint32_t to = out_base + (uint32_t)cb * 2u * run + (uint32_t)(rb * 4 + kc * 2) * 256u + out_key[kc];
            u32x4 px, dx;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              px[t] = pack_bf16(x[2 * t], x[2 * t + 1]);
              dx[t] = pack_bf16(y[2 * t], y[2 * t + 1]);
            }
            __builtin_nontemporal_store(px, (u32x4*)(out_p + to));
            __builtin_nontemporal_store(dx, (u32x4*)(out_s + to));
          }
        }
      out_base += 8u * run;
      ++kt;
      if (!more) break;
      k += k_tile;
      v += v_tile;
      keys = keys_next;
      wait_vmcnt<2 * COPIES + STORES>();  // the copies of the next tile's first step
      step_barrier();
    }
  }
  if (kt < read) {  // the second half of a 256-key tile whose first half is seen: kernel 2 reads it
    const u32x4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
          const uint32_t to = out_base + (uint32_t)cb * 2u * run + (uint32_t)(rb * 4 + kc * 2) * 256u + out_key[kc];
          *(u32x4*)(out_p + to) = zero;
          *(u32x4*)(out_s + to) = zero;
        }
  }
}

// ---- kernel 2: a 256 x 256 output (256 columns of D, and 256 query rows of dQ or 256 keys of dK or dV) per workgroup,
// four waves of 128 x 128 (one per SIMD, 256 accumulators in AGPRs): each operand read from LDS feeds four MFMAs. The
// operands of a half step (16 of the contraction) are read during the MFMAs of the half step before it; the barrier
// that publishes a step's copies is passed halfway through the step before, when every wave has read the whole of
// that step's buffer, so the copies of three to four steps are in flight. (dQ's loop drains them once in four steps: the
// compiler puts a vmcnt(0) of its own before the first LDS read of the unrolled four; the dK / dV loop has none.) The
// 65 spilled VGPRs are outside the loops. The chunk of the last 2,048 of 16,384 rows
// (32 / 4 heads): 3.13 ms with eight waves of 128 x 64, 2.88 ms so, 2.50 ms with the reads and copies spread between the
// MFMAs (sched_group_barrier); 1.4 ms at the nominal MFMA rate.
template <bool DQ>
__device__ __forceinline__ void wide_grad(const BwdWideParams& w, const WideSeq& s, int item,
                                          KA_LDS char* const (&at)[kRing], KA_LDS char* const (&bt)[kRing]) {
  constexpr int W = kGradThreads / 64, INSTS = kGradStep * kGradTile * 2 / 1024 / W;
  constexpr int COPIES = 2 * INSTS;  // a wave's copies per step
  const BwdParams& p = w.b;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int wd = wave >> 1, wn = wave & 1;
  const int64_t run = (int64_t)(w.rows / 8) * 256;  // bytes per block of 16 keys of P or dS
  const int r_end = min(s.lq, w.r_begin + w.rows);

  int head, dhalf, n0, which = 0, steps, first = 0;  // n0: the first query row (dQ, from the chunk's first) or key
  bool carry = false, last = true;
  if constexpr (DQ) {
    head = spread_head(item % p.heads, p.heads);
    const int rest = item / p.heads;
    dhalf = rest & 1;
    n0 = (w.rows / kGradTile - 1 - (rest >> 1)) * kGradTile;  // the rows that see most keys first
    const int row = w.r_begin + n0;
    if (row >= s.lq) return;
    const int top = min(row + kGradTile, s.lq) - 1;
    const int64_t seen = p.right < 0 ? s.lk : (int64_t)top + (s.lk - s.lq) + p.right + 1;
    const int khi = (int)max((int64_t)0, min(seen, (int64_t)s.lk));
    steps = (khi + kGradStep - 1) / kGradStep;
  } else {
    const int kinds = 2 * (p.heads / p.group);
    const int kind = item % kinds, rest = item / kinds;
    head = kind >> 1;  // the key/value head
    which = kind & 1;  // 0: dK, 1: dV
    dhalf = rest & 1;
    n0 = (rest >> 1) * kGradTile;
    if (n0 >= s.lk) return;
    last = s.lq <= w.r_begin + w.rows && (s.lq > w.r_begin || w.r_begin == 0);
    const int seen = s.first_row(p.right, n0);
    first = max(seen, w.r_begin) & ~(kGradStep - 1);
    carry = seen < w.r_begin;
    steps = first < r_end ? (r_end - first + kGradStep - 1) / kGradStep : 0;
    if (steps == 0 && !(last && !carry)) return;  // no row of the chunk sees these keys
  }

  // copies: the A tile (32 keys or query rows x 256 columns of D, S layout): wave w copies columns (w & 1) * 128 .. of
  // rows (w >> 1) * 16 .. +16; the B tile: dQ 32 keys x 256 rows, dK / dV 256 keys x 32 rows of P or dS
  const int64_t a_t = DQ ? p.sk_t : which ? p.sdo_t : p.sq_t;
  const int64_t a_h = which ? p.sdo_h : p.sq_h;
  const uint32_t a_off = s_block_base<kGradTile, INSTS>(wave, lane, a_t), b_off = (uint32_t)lane * 16u;
  const int64_t head_bytes = (int64_t)w.keys * w.rows * 2;
  const uint16_t* a_src;
  const char* b_src;
  int left_rows, in_head = 0;
  if constexpr (DQ) {
    a_src = p.k + (int64_t)s.ka * a_t + (int64_t)(head / p.group) * p.sk_h + dhalf * 256;
    left_rows = s.lk;
    b_src = (const char*)w.ds + head * head_bytes + (int64_t)(n0 / 8) * 256 + (wave >> 1) * run + (wave & 1) * 4096;
  } else {
    a_src = (which ? p.dout : p.q) + (int64_t)(s.qa + first) * a_t + (int64_t)head * p.group * a_h + dhalf * 256;
    left_rows = s.lq - first;
    b_src = (const char*)(which ? w.p : w.ds) + (int64_t)head * p.group * head_bytes +
            (int64_t)(n0 / 16 + wave * INSTS) * run + (int64_t)((first - w.r_begin) / 8) * 256;
  }
  const int64_t a_step = (int64_t)kGradStep * a_t;
  const int64_t b_step = DQ ? (kGradStep / 16) * run : (int64_t)(kGradStep / 8) * 256;
  const int64_t b_block = DQ ? 1024 : run;
  const int64_t a_wrap = a_h - (steps - 1) * a_step, b_wrap = head_bytes - (steps - 1) * b_step;
  const int top_rows = left_rows;
  auto copy = [&](KA_LDS char* a, KA_LDS char* b) {
    const int bytes = min(left_rows, kGradStep) * (int)a_t * 2;
#pragma unroll
    for (int r = 0; r < INSTS; ++r) {
      dma_16b(a_src, bytes, a + (wave * INSTS + r) * 1024, s_block(a_off, r));
      dma_16b((const uint16_t*)(b_src + r * b_block), 1024, b + (wave * INSTS + r) * 1024, b_off);
    }
    const bool wrap = !DQ && in_head + 1 == steps;  // the group's next head
    in_head = wrap ? 0 : in_head + 1;
    a_src += wrap ? a_wrap : a_step;
    b_src += wrap ? b_wrap : b_step;
    left_rows = wrap ? top_rows : left_rows - kGradStep;
  };
  // transposed reads: + kc * 8192 + 32-column block * 1024
  const int t_read[2] = {s_tr_base(lane, 0) + wd * 4096, s_tr_base(lane, 1) + wd * 4096};
  const int xt_read[2] = {x_tr_base(lane, 0) + wn * 4096, x_tr_base(lane, 1) + wn * 4096};
  // dK / dV: chunk kc*2 + half of key wn*128 + j*32 + col
  const int x_read[2] = {((wn * 8 + (col >> 4)) * 4 + half) * 256 + ((col & 15) ^ (half << 2)) * 16,
                         ((wn * 8 + (col >> 4)) * 4 + 2 + half) * 256 + ((col & 15) ^ ((2 + half) << 2)) * 16};

  f32x16 acc[4][4];
  f32x4* const kept = (f32x4*)w.acc + (int64_t)item * 64 * kGradThreads + tid;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x16{};
  if (!DQ && carry) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 x = kept[((i * 4 + j) * 4 + g) * kGradThreads];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][g * 4 + e] = x[e];
        }
  }

  auto tr = [&](const KA_LDS char* t, const int (&base)[2], int at) {
    bf16x4 x[2];
#pragma unroll
    for (int rr = 0; rr < 2; ++rr)
      x[rr] = __builtin_bit_cast(bf16x4,
                                 __builtin_amdgcn_ds_read_tr16_b64_v4i16((KA_LDS s16x4*)(t + base[rr] + at)));
    return __builtin_shufflevector(x[0], x[1], 0, 1, 2, 3, 4, 5, 6, 7);
  };
  bf16x8 x[2][4], y[2][4];  // the operands of the two half steps
  auto read = [&](int kc, const KA_LDS char* a, const KA_LDS char* b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (DQ) y[kc][i] = tr(b, xt_read, kc * 8192 + i * 1024);
      else y[kc][i] = *(const KA_LDS bf16x8*)(b + x_read[kc] + i * 2048);
      x[kc][i] = tr(a, t_read, kc * 8192 + i * 1024);
    }
  };
  auto multiply = [&](int kc) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[kc][i], y[kc][j], acc[i][j], 0, 0, 0);
  };
  const int total = DQ ? steps : steps * p.group;
  // step n in buffer a, b (an, bn: step n + 1's); its first half's operands are read
  // (FULL: so are steps n + 1 to n + 4 there)
  auto step = [&](auto full, int n, KA_LDS char* a, KA_LDS char* b, const KA_LDS char* an, const KA_LDS char* bn) {
    constexpr bool FULL = decltype(full)::value;
    read(1, a, b);
    multiply(0);
    if constexpr (FULL) {  // LDS reads (0x100) and copies (0x020) issued between the MFMAs (0x008)
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (FULL || n + 3 < total) wait_vmcnt<2 * COPIES>();  // step n + 1's copies; two later steps' may be in flight
    else if (n + 2 < total) wait_vmcnt<COPIES>();
    else wait_vmcnt<0>();
    step_barrier();
    if (FULL || n + kRing < total) copy(a, b);
    if (FULL || n + 1 < total) read(0, an, bn);
    multiply(1);
    if constexpr (FULL) {
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < kRing; ++i)
    if (i < total) copy(at[i], bt[i]);
  if (total > 3) wait_vmcnt<3 * COPIES>();
  else wait_vmcnt<0>();
  step_barrier();
  if (total > 0) read(0, at[0], bt[0]);
  int n = 0;
  const std::true_type full;
  const std::false_type tail;
  for (; n + 2 * kRing <= total; n += kRing) {
    step(full, n, at[0], bt[0], at[1], bt[1]);
    step(full, n + 1, at[1], bt[1], at[2], bt[2]);
    step(full, n + 2, at[2], bt[2], at[3], bt[3]);
    step(full, n + 3, at[3], bt[3], at[0], bt[0]);
  }
  for (; n < total; n += kRing) {
    step(tail, n, at[0], bt[0], at[1], bt[1]);
    if (n + 1 < total) step(tail, n + 1, at[1], bt[1], at[2], bt[2]);
    if (n + 2 < total) step(tail, n + 2, at[2], bt[2], at[3], bt[3]);
    if (n + 3 < total) step(tail, n + 3, at[3], bt[3], at[0], bt[0]);
  }

  if (!DQ && !last) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          kept[((i * 4 + j) * 4 + g) * kGradThreads] =
              f32x4{acc[i][j][g * 4], acc[i][j][g * 4 + 1], acc[i][j][g * 4 + 2], acc[i][j][g * 4 + 3]};
    return;
  }
  // lane (col, half) holds d = dhalf*256 + wd*128 + i*32 + (reg/4)*8 + half*4 + reg%4 of row / key wn*128 + j*32 + col
  const float scale = DQ || which == 0 ? p.scale : 1.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int at_n = n0 + wn * 128 + j * 32 + col;
    const bool valid = DQ ? w.r_begin + at_n < s.lq : at_n < s.lk;
    uint16_t* to;
    if constexpr (DQ) to = p.dq + (int64_t)(s.qa + w.r_begin + at_n) * p.sdq_t + (int64_t)head * p.sdq_h;
    else to = which ? p.dv + (int64_t)(s.ka + at_n) * p.sdv_t + (int64_t)head * p.sdv_h
                    : p.dk + (int64_t)(s.ka + at_n) * p.sdk_t + (int64_t)head * p.sdk_h;
    to += dhalf * 256 + wd * 128 + half * 4;
    if (!valid) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        u32x2 o;
        o[0] = pack_bf16(acc[i][j][g * 4] * scale, acc[i][j][g * 4 + 1] * scale);
        o[1] = pack_bf16(acc[i][j][g * 4 + 2] * scale, acc[i][j][g * 4 + 3] * scale);
        *(u32x2*)(to + i * 32 + g * 8) = o;
      }
  }
}

__global__ __launch_bounds__(kGradThreads, 1) void bwd_wide_grad_kernel(BwdWideParams w) {
  constexpr int TILE = kGradStep * kGradTile * 2;
  __shared__ __attribute__((aligned(1024))) char a0_s[TILE], a1_s[TILE], a2_s[TILE], a3_s[TILE];
  __shared__ __attribute__((aligned(1024))) char b0_s[TILE], b1_s[TILE], b2_s[TILE], b3_s[TILE];
  KA_LDS char* const at[kRing] = {(KA_LDS char*)a0_s, (KA_LDS char*)a1_s, (KA_LDS char*)a2_s, (KA_LDS char*)a3_s};
  KA_LDS char* const bt[kRing] = {(KA_LDS char*)b0_s, (KA_LDS char*)b1_s, (KA_LDS char*)b2_s, (KA_LDS char*)b3_s};
  const WideSeq s(w);
  // dK and dV first where the group is large: their items are then the longer ones (rows / 32 steps of every head of the
  // group, against the visible keys / 32 of dQ), and early chunks have few of them, so dQ fills the CUs that they leave
  // free. Backward in us, dQ first and dK / dV first (medians of seven in turn), at 1,024, 2,048, 4,096, 8,192 rows:
  //   group 16 (32 / 2 heads): 394 379, 981 916, 2493 2318, 6948 6697     8 (32 / 4): 270 255, 706 639, 1942 1734, 6323 6013
  //   4 (32 / 8): 209 196, 576 517, 1711 1699, 6032 6025                   4 (4 / 1): 112 112, 217 216, 447 447, 1334 1319
  //   3 (24 / 8): 146 145, 426 390, 1368 1364, 4762 4725                   3 (6 / 2): 101 100, 204 205, 473 483, 1573 1507
  //   2 (32 / 16): 184 180, 542 538, 1764 1768, 6452 6482                  1 (32 / 32): 203 205, 635 629, 2045 2073, 7443 7485
  const int dkdv_items = w.keys / kGradTile * 4 * (w.b.heads / w.b.group);
  const int dq_items = w.rows / kGradTile * 2 * w.b.heads;
  const bool dkdv_first = w.b.group >= 4;
  const int at_dkdv = (int)blockIdx.x - (dkdv_first ? 0 : dq_items);
  const int at_dq = (int)blockIdx.x - (dkdv_first ? dkdv_items : 0);
  if (at_dkdv >= 0 && at_dkdv < dkdv_items) wide_grad<false>(w, s, at_dkdv, at, bt);
  else wide_grad<true>(w, s, at_dq, at, bt);
}

hipError_t launch_bwd_wide(BwdWideParams w, hipStream_t stream) {
  const int kv_heads = w.b.heads / w.b.group;
  // key tiles per workgroup of kernel 1: at least 1,024 workgroups (four per CU), at most eight tiles. The backward of
  // 16,384 rows at 32 / 4 heads with at most 1, 2, 4, 8, 16: 24.1, 22.9, 22.6, 22.8, 23.4 ms; 32 / 16: 27.1, 26.1, 25.8, 26.0,
  // 26.7. At least 256, 512, 1,024, 2,048 workgroups: 264, 264, 251, 252 us at 1,024 rows (32 / 4), 995, 995, 932, 903 at 4,096
  // (8 / 1), no difference where there are plenty.
  const int64_t row_tiles = (int64_t)(w.rows / kDsRows) * w.b.heads, key_tiles = w.keys / kDsKeys;
  const int64_t per = row_tiles * key_tiles / 1024;
  w.run = (int32_t)(per < 1 ? 1 : per > 8 ? 8 : per);
  const int64_t ds_items = row_tiles * ((key_tiles + w.run - 1) / w.run);
  const int64_t grad_items =
      (int64_t)(w.rows / kGradTile) * 2 * w.b.heads + (int64_t)(w.keys / kGradTile) * 4 * kv_heads;
  for (int64_t r = 0; r < w.b.total_q; r += w.rows) {
    w.r_begin = (int32_t)r;
    hipLaunchKernelGGL(bwd_wide_ds_kernel, dim3((unsigned)ds_items), dim3(kWideThreads), 0, stream, w);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(bwd_wide_grad_kernel, dim3((unsigned)grad_items), dim3(kGradThreads), 0, stream, w);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace karpo
