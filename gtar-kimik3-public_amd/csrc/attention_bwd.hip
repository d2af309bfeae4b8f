// Backward of the causal grouped-query attention (gdr_attention_bwd; src/ops/flash_attention_2.py:180-207).
//
//   P = 2^(c S - lse)  (S = Q K^T, c = scale log2 e, lse the forward's row log-sum-exp in log2 units)
//   delta = rowsum(O (x) dO),  dP = dO V^T,  dS = P (x) (dP - delta)
//   dQ = scale dS K,  dK = scale dS^T Q,  dV = P^T dO                  (per (sequence, query head); key/value head
//                                                                       h / (H / Hkv) sums its group's terms)
//
// Two launches of four-wave workgroups on v_mfma_f32_16x16x32_{bf16,f16} with fp32 accumulation; P and dS enter
// their products rounded to the input type, as the reference's probs.to(dtype) and dscores.to(dtype) do:
//   * attention_dq_kernel -- 128 query rows of one (sequence, query head), two 16-row blocks per wave, the q and dO
//     rows held in registers as B operands.  It first forms delta from the out and dO rows (and stores it for the
//     second launch), then streams the 64-row key and value tiles up to the diagonal through double-buffered LDS
//     (LDS DMA).  Per tile S^T = K Q^T and dP^T = V dO^T take the tile rows as A operands, so a lane holds 16
//     entries of one query row; dS^T then feeds dQ^T += K^T dS^T straight from the accumulators, K^T coming from the
//     transposing LDS read.
//   * attention_dkdv_kernel -- 64 keys of one (sequence, key/value head), the k rows held in registers as B operands,
//     the v rows in LDS.  Query and dO tiles of 64 rows stream through double-buffered LDS for every query head of the
//     group, from the tile holding the diagonal on.  The four waves split each 64 x 64 tile two by two, 32 queries by
//     32 keys each, so a wave reads only its half of the Q and dO rows: S = Q K^T and dP = dO V^T (a lane holds 16
//     entries of two key columns), then dV^T += dO^T P and dK^T += Q^T dS with the transposing read, 44 KB of LDS
//     reads for 64 MFMAs where a 64 x 16 split took 72 KB.  The two query waves of a key half add their sums once, at
//     the end.  Two workgroups share a CU (80 KB of LDS each, the CU's 160 together, which is why lse and delta travel
//     in a register).
// A step is bound by its own chain (LDS read, score MFMAs, exponentials, LDS read, gradient MFMAs) at two waves per
// SIMD, so what helps is less of everything in it: tile copies with one 32-bit lane offset instead of 64-bit address
// arithmetic per copy, no mask selects in whole tiles, exponentials issued beside dP's MFMAs.  Measured (72,292 packed
// tokens, 16 / 8 heads, D = 128, before -> after): dQ 1,445 -> 1,277 us, dK/dV 2,284 -> 2,069 us; D = 64 773 -> 700 and
// 1,187 -> 1,150.  Sequences of one or two tiles pay 1 to 2 us per call for the exchange at the end and the spread of lse
// and delta (33 tokens, D = 128, 16 / 8 heads: dK/dV 7.1 -> 9.3 us; 60 sequences of 64 24.0 -> 26.4; 300 tokens 53.4 ->
// 52.6); the split by keys is not kept for them, because a packed sequence has to equal its own call bit for bit.  Tried
// for dK/dV and slower: 128-row tiles split over eight waves (2,337), two four-wave sets taking
// alternate tiles in one workgroup (2,397; faster only for a single long sequence, 179 against 217 us at 4,096 tokens).
// Only tiles crossing the diagonal or the sequence end are masked.  No atomics: every output element has one
// owning lane, so the result does not depend on scheduling.
#include "attention_common.h"
#include "varlen_index.h"
#include "gdr_internal.h"

namespace gdr {
namespace {

using attn::cat;
using attn::kTile;
using attn::Mma;
using attn::short4;
using chunk::kLog2e;

constexpr int kQB = 128;  // query rows per dq workgroup
constexpr int kKB = 64;   // keys per dk/dv workgroup
constexpr int kRB = 2;    // 16-row query blocks per wave in the dq kernel
static_assert(kKB == kTile && attn::kWaves == (kKB / 32) * (kTile / 32), "dk/dv wave split");

// Lane l < 32 of `rows` holds the lse of query row l, lane 32 + l its delta: those of rows kFirst / 4 + 4 g4 .. + 3 for
// `at` = 16 g4.  Inline assembly so that the constant parts of the lane indexes are instruction offsets.
template <int kFirst>
__device__ __forceinline__ void spread_rows(int at, float rows, float (&l)[4], float (&d)[4]) {
  asm volatile(
      "ds_bpermute_b32 %0, %8, %9 offset:%10\n\t"
      "ds_bpermute_b32 %1, %8, %9 offset:%11\n\t"
      "ds_bpermute_b32 %2, %8, %9 offset:%12\n\t"
      "ds_bpermute_b32 %3, %8, %9 offset:%13\n\t"
      "ds_bpermute_b32 %4, %8, %9 offset:%14\n\t"
      "ds_bpermute_b32 %5, %8, %9 offset:%15\n\t"
      "ds_bpermute_b32 %6, %8, %9 offset:%16\n\t"
      "ds_bpermute_b32 %7, %8, %9 offset:%17\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(l[0]), "=&v"(l[1]), "=&v"(l[2]), "=&v"(l[3]), "=&v"(d[0]), "=&v"(d[1]), "=&v"(d[2]), "=&v"(d[3])
      : "v"(at), "v"(rows), "i"(kFirst), "i"(kFirst + 4), "i"(kFirst + 8), "i"(kFirst + 12), "i"(kFirst + 128),
        "i"(kFirst + 132), "i"(kFirst + 136), "i"(kFirst + 140));
}

template <typename V4, typename V8>
__device__ __forceinline__ V8 tr_pair(const short4 (&r)[4], int s2) {
  return cat<V4, V8>(__builtin_bit_cast(V4, r[2 * s2]), __builtin_bit_cast(V4, r[2 * s2 + 1]));
}

template <int D, typename T>
__global__ __launch_bounds__(attn::kThreads, 2) void attention_dq_kernel(const gdr_attention_args a,
                                                                      const gdr_attention_grads g, int nqb) {
  using M = Mma<T>;
  using V8 = typename M::v8;
  using V4 = typename M::v4;
  constexpr int DS = D / 32;  // 32-wide k steps of the score products
  constexpr int DT = D / 16;  // 16-column tiles of dQ^T
  constexpr int TILE = kTile * D;
  extern __shared__ __align__(16) unsigned char smem[];
  T* ks = reinterpret_cast<T*>(smem);             // [2][kTile][D] swizzled
  T* vs = reinterpret_cast<T*>(smem) + 2 * TILE;  // [2][kTile][D] swizzled

  // ---- workgroup -> (sequence, query block, head), the latest query blocks (the most keys) first ----
  const int H = a.heads;
  const int h = blockIdx.x % H, slot = blockIdx.x / H;
  int n, qb, bos = 0, len = a.seq_len;
  if (a.cu_seqlens) {
    n = packed_slot_seq(a.cu_seqlens, a.n_seqs, a.seq_len, kQB, slot);
    bos = packed_begin(a.cu_seqlens, n, a.seq_len);
    len = packed_end(a.cu_seqlens, n, a.seq_len) - bos;
    const int nb = (len + kQB - 1) / kQB;
    const int r = slot - packed_slot_base(a.cu_seqlens, n, a.seq_len, kQB);
    if (r < 0 || r >= nb) return;  // gap slot: uniform over the workgroup, before any barrier
    qb = nb - 1 - r;
  } else {
    n = slot / nqb;
    qb = nqb - 1 - slot % nqb;
  }
  const int bidx = a.cu_seqlens ? 0 : n;
  const int hk = h / (H / a.kv_heads);
  auto at = [&](const gdr_tensor& t, int head) {
    return static_cast<const T*>(t.ptr) + bidx * t.stride_b + head * t.stride_h + int64_t(bos) * t.stride_t;
  };
  const T* qp = at(a.q, h);
  const T* kp = at(a.k, hk);
  const T* vp = at(a.v, hk);
  const T* op = at(a.out, h);
  const T* dop = at(g.d_out, h);
  T* dqp = const_cast<T*>(at(g.d_q, h));
  const int64_t row0 = (int64_t(bidx) * H + h) * a.seq_len + bos;  // lse / delta index of the sequence's row 0

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g4 = lane >> 4;
  const int q0 = qb * kQB;

  // This lane's query rows (l16 of each block) as B operands: q and dO columns 32 ds + 8 g4 .. + 7.  delta =
  // rowsum(out (x) dO) from the same fragments, summed over the four lane groups.
  int qpos[kRB];
  V8 qf[kRB][DS], df[kRB][DS];
  float lse[kRB], dlt[kRB];
#pragma unroll
  for (int b = 0; b < kRB; ++b) {
    qpos[b] = q0 + 16 * (kRB * wave + b) + l16;
    const int qrow = min(qpos[b], len - 1);
    float part = 0.f;
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) {
      const int col = 32 * ds + 8 * g4;
      qf[b][ds] = *reinterpret_cast<const V8*>(qp + int64_t(qrow) * a.q.stride_t + col);
      df[b][ds] = *reinterpret_cast<const V8*>(dop + int64_t(qrow) * g.d_out.stride_t + col);
      const V8 of = *reinterpret_cast<const V8*>(op + int64_t(qrow) * a.out.stride_t + col);
#pragma unroll
      for (int j = 0; j < 8; ++j) part += static_cast<float>(of[j]) * static_cast<float>(df[b][ds][j]);
    }
    part = xor_sum(part, 16);
    dlt[b] = xor_sum(part, 32);
    lse[b] = a.lse[row0 + qrow];
    if (g4 == 0 && qpos[b] < len) g.delta[row0 + qpos[b]] = dlt[b];
  }

  attn::TileDma<D> dma;
  dma.init(__builtin_amdgcn_readfirstlane(wave), lane);
  const uint32_t kdoff = dma.offset(a.k.stride_t), vdoff = dma.offset(a.v.stride_t);
  const int kend = min(len, q0 + kQB);  // keys this block can see
  const int nkb = (kend + kTile - 1) / kTile;
  int koff[DS], toff[DT];
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) koff[ds] = attn::row_frag<D>(ds, l16, g4);
#pragma unroll
  for (int t = 0; t < DT; ++t) toff[t] = attn::tr_frag<D>(t, l16, g4);
  const float c = a.scale * kLog2e;
  const uint32_t klds = attn::lds_addr(ks);

  dma.issue(kp, a.k.stride_t, kdoff, 0, len, ks);
  dma.issue(vp, a.v.stride_t, vdoff, 0, len, vs);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  floatx4 dq[kRB][DT];  // dQ^T: lane holds columns 16 t + 4 g4 + i of query row qpos[b]
#pragma unroll
  for (int b = 0; b < kRB; ++b)
#pragma unroll
    for (int t = 0; t < DT; ++t) dq[b][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int kb = 0; kb < nkb; ++kb) {
    const int cur = kb & 1;
    if (kb + 1 < nkb) {  // the other buffers were released by the barrier that ended the previous step
      dma.issue(kp, a.k.stride_t, kdoff, (kb + 1) * kTile, len, ks + (cur ^ 1) * TILE);
      dma.issue(vp, a.v.stride_t, vdoff, (kb + 1) * kTile, len, vs + (cur ^ 1) * TILE);
    }
    const T* kt = ks + cur * TILE;
    const T* vt = vs + cur * TILE;
    // S^T and dP^T: lane holds key kb kTile + 16 t + 4 g4 + i of query row qpos[b]
    floatx4 s[kRB][4], dp[kRB][4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int b = 0; b < kRB; ++b) s[b][t] = dp[b][t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) {
        const V8 kf = *reinterpret_cast<const V8*>(kt + 16 * t * D + koff[ds]);
        const V8 vf = *reinterpret_cast<const V8*>(vt + 16 * t * D + koff[ds]);
#pragma unroll
        for (int b = 0; b < kRB; ++b) {
          s[b][t] = M::run(kf, qf[b][ds], s[b][t]);
          dp[b][t] = M::run(vf, df[b][ds], dp[b][t]);
        }
      }
    }
    // dS^T = P^T (x) (dP^T - delta); only a tile crossing this wave's diagonal or the sequence end is masked
    const bool full = (kb + 1) * kTile - 1 <= q0 + 32 * wave && (kb + 1) * kTile <= len;
    V8 dsf[kRB][2];
#pragma unroll
    for (int b = 0; b < kRB; ++b) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][t][i], c, -lse[b]));
          s[b][t][i] = p * (dp[b][t][i] - dlt[b]);
        }
      if (!full) {  // a branch of its own, so that whole tiles pay no selects
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = kb * kTile + 16 * t + 4 * g4 + i;
            if (!(key <= qpos[b] && key < len)) s[b][t][i] = 0.f;
          }
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) dsf[b][s2] = cat<V4, V8>(M::pack(s[b][2 * s2]), M::pack(s[b][2 * s2 + 1]));
    }
    // dQ^T += K^T dS^T: K^T of column tile t through the transposing read, one tile ahead of its MFMAs
    const uint32_t kaddr = klds + 2 * cur * TILE;
    short4 x[2][4];
    attn::tr_read4<D>(kaddr + 2 * toff[0], x[0]);
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      short4(&r)[4] = x[t & 1];
      if (t + 1 < DT) {
        attn::tr_read4<D>(kaddr + 2 * toff[t + 1], x[(t + 1) & 1]);
        asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]));
      } else {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]));
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const V8 kf = tr_pair<V4, V8>(r, s2);
#pragma unroll
        for (int b = 0; b < kRB; ++b) dq[b][t] = M::run(kf, dsf[b][s2], dq[b][t]);
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's copies of the next tiles have landed
    __syncthreads();                 // ... everyone's, and every wave is done with this step's buffers
  }

#pragma unroll
  for (int b = 0; b < kRB; ++b) {
    if (qpos[b] < len) {
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        floatx4 y = dq[b][t];
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] *= a.scale;
        *reinterpret_cast<V4*>(dqp + int64_t(qpos[b]) * g.d_q.stride_t + 16 * t + 4 * g4) = M::pack(y);
      }
    }
  }
}

template <int D, typename T>
__global__ __launch_bounds__(attn::kThreads, D == 64 ? 3 : 2) void attention_dkdv_kernel(const gdr_attention_args a,
                                                                    const gdr_attention_grads g, int nkb) {
  using M = Mma<T>;
  using V8 = typename M::v8;
  using V4 = typename M::v4;
  constexpr int DS = D / 32;
  constexpr int DT = D / 16;  // 16-column tiles of dK^T and dV^T
  constexpr int TILE = kTile * D;
  extern __shared__ __align__(16) unsigned char smem[];
  T* qs = reinterpret_cast<T*>(smem);              // [2][kTile][D] swizzled query rows
  T* dos = reinterpret_cast<T*>(smem) + 2 * TILE;  // [2][kTile][D] swizzled dO rows
  T* vs = dos + 2 * TILE;                          // [kKB][D] swizzled value rows

  // ---- workgroup -> (sequence, key block, key/value head); the first key blocks (the most queries) first ----
  const int H = a.heads, Hk = a.kv_heads, G = H / Hk;
  const int hk = blockIdx.x % Hk, slot = blockIdx.x / Hk;
  int n, kb, bos = 0, len = a.seq_len;
  if (a.cu_seqlens) {
    n = packed_slot_seq(a.cu_seqlens, a.n_seqs, a.seq_len, kKB, slot);
    bos = packed_begin(a.cu_seqlens, n, a.seq_len);
    len = packed_end(a.cu_seqlens, n, a.seq_len) - bos;
    const int nb = (len + kKB - 1) / kKB;
    kb = slot - packed_slot_base(a.cu_seqlens, n, a.seq_len, kKB);
    if (kb < 0 || kb >= nb) return;  // gap slot: uniform over the workgroup, before any barrier
  } else {
    n = slot % a.batch;
    kb = slot / a.batch;
  }
  const int bidx = a.cu_seqlens ? 0 : n;
  auto at = [&](const gdr_tensor& t, int head) {
    return static_cast<const T*>(t.ptr) + bidx * t.stride_b + head * t.stride_h + int64_t(bos) * t.stride_t;
  };
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g4 = lane >> 4;
  const int uwave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = uwave & 1, wq = uwave >> 1;  // this wave's 32 keys of the block, 32 query rows of each tile
  const int key0 = kb * kKB, wkey0 = key0 + 32 * wk;

  // Iterations over (query head of the group, query tile from the diagonal on).  Lane l of a wave also fetches one of
  // its 32 query rows' lse (l < 32) or delta, a step ahead, into a register: two workgroups' tiles fill the LDS
  // exactly.  Rows past the sequence end read its last row.
  const int per = (len + kTile - 1) / kTile - kb, total = G * per;
  attn::TileDma<D> dma;
  dma.init(uwave, lane);
  const uint32_t qoff = dma.offset(a.q.stride_t), dooff = dma.offset(g.d_out.stride_t);
  const float* row_vals = (lane < 32 ? a.lse : g.delta) + int64_t(bidx) * H * a.seq_len + bos;
  auto issue = [&](int it, int buf) {
    const int hq = hk * G + it / per, r0 = (kb + it % per) * kTile;
    dma.issue(at(a.q, hq), a.q.stride_t, qoff, r0, len, qs + buf * TILE);
    dma.issue(at(g.d_out, hq), g.d_out.stride_t, dooff, r0, len, dos + buf * TILE);
    return row_vals[int64_t(hq) * a.seq_len + min(r0 + 32 * wq + (lane & 31), len - 1)];
  };
  float rows_next = issue(0, 0);
  dma.issue(at(a.v, hk), a.v.stride_t, dma.offset(a.v.stride_t), key0, len, vs);

  // The wave's key rows of k as B operands: columns 32 ds + 8 g4 .. + 7 of keys wkey0 + 16 c + l16.
  V8 kf[2][DS];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const T* kp = at(a.k, hk) + int64_t(min(wkey0 + 16 * c + l16, len - 1)) * a.k.stride_t;
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) kf[c][ds] = *reinterpret_cast<const V8*>(kp + 32 * ds + 8 * g4);
  }
  // Byte offsets in the LDS array of this lane's fragments: the row fragment of k step 0 of the wave's query rows and
  // of its value rows, and the transposing read of column tile 0.  The swizzle makes k step ds the offset ^ 64 ds and
  // column tile t the offset ^ 32 t, so one register serves each; formed inside the loop (opaque below), they leave
  // the accumulators their registers.
  const uint32_t row0 = 2 * (32 * wq * D + attn::row_frag<D>(0, l16, g4));
  const uint32_t vrow0 = 2 * (4 * TILE + 32 * wk * D + attn::row_frag<D>(0, l16, g4));
  const uint32_t tr0 = attn::lds_addr(smem) + 2 * (32 * wq * D + attn::tr_frag<D>(0, l16, g4));
  constexpr int kDo = 2 * 2 * TILE;  // bytes from a query tile to its dO tile
  const float c2 = a.scale * kLog2e;

  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  floatx4 dk[2][DT], dv[2][DT];  // dK^T, dV^T: lane holds columns 16 t + 4 g4 + i of key wkey0 + 16 c + l16
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int t = 0; t < DT; ++t) dk[c][t] = dv[c][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int it = 0; it < total; ++it) {
    const int cur = it & 1;
    const float rows = rows_next;
    if (it + 1 < total) rows_next = issue(it + 1, cur ^ 1);  // the other buffers were released by the last barrier
    const int qbase = (kb + it % per) * kTile + 32 * wq;
    uint32_t rowc = row0 + 2 * cur * TILE, vrowc = vrow0, trc = tr0 + 2 * cur * TILE;
    asm volatile("" : "+v"(rowc), "+v"(vrowc), "+v"(trc));
    // S, P and dP: lane holds query qbase + 16 r + 4 g4 + i of key wkey0 + 16 c + l16.  One block up to the mask, so
    // that the exponentials run beside dP's MFMAs.
    floatx4 s[2][2], dp[2][2];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 2; ++c) s[r][c] = dp[r][c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ds = 0; ds < DS; ++ds)
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const V8 qa = *reinterpret_cast<const V8*>(smem + (rowc ^ (64 * ds)) + 32 * r * D);
#pragma unroll
        for (int c = 0; c < 2; ++c) s[r][c] = M::run(qa, kf[c][ds], s[r][c]);
      }
    float lr[2][4], dr[2][4];
    spread_rows<0>(16 * g4, rows, lr[0], dr[0]);
    spread_rows<64>(16 * g4, rows, lr[1], dr[1]);
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[r][c][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r][c][i], c2, -lr[r][i]));
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) {
      V8 vf[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) vf[c] = *reinterpret_cast<const V8*>(smem + (vrowc ^ (64 * ds)) + 32 * c * D);
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const V8 da = *reinterpret_cast<const V8*>(smem + (rowc ^ (64 * ds)) + 32 * r * D + kDo);
#pragma unroll
        for (int c = 0; c < 2; ++c) dp[r][c] = M::run(da, vf[c], dp[r][c]);
      }
    }
    // Only a tile crossing this wave's diagonal or the sequence end is masked; then dS = P (x) (dP - delta)
    if (!(qbase >= wkey0 + 31 && qbase + 32 <= len)) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int q = qbase + 16 * r + 4 * g4 + i;
            if (!(wkey0 + 16 * c + l16 <= q && q < len)) s[r][c][i] = 0.f;
          }
    }
    V8 pf[2], dsf[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) dp[r][c][i] = s[r][c][i] * (dp[r][c][i] - dr[r][i]);
      pf[c] = cat<V4, V8>(M::pack(s[0][c]), M::pack(s[1][c]));
      dsf[c] = cat<V4, V8>(M::pack(dp[0][c]), M::pack(dp[1][c]));
    }
    // dV^T += dO^T P and dK^T += Q^T dS: column tile t of the wave's dO and Q rows through the transposing read, one
    // tile ahead of its MFMAs (four reads in flight: lgkmcnt(4) covers the current tile's)
    short4 xd[2][2], xq[2][2];
    attn::tr_read2<D, kDo>(trc, xd[0]);
    attn::tr_read2<D, 0>(trc, xq[0]);
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      short4(&rd)[2] = xd[t & 1];
      short4(&rq)[2] = xq[t & 1];
      if (t + 1 < DT) {
        attn::tr_read2<D, kDo>(trc ^ (32 * (t + 1)), xd[(t + 1) & 1]);
        attn::tr_read2<D, 0>(trc ^ (32 * (t + 1)), xq[(t + 1) & 1]);
        asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(rd[0]), "+v"(rd[1]), "+v"(rq[0]), "+v"(rq[1]));
      } else {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(rd[0]), "+v"(rd[1]), "+v"(rq[0]), "+v"(rq[1]));
      }
      const V8 df = cat<V4, V8>(__builtin_bit_cast(V4, rd[0]), __builtin_bit_cast(V4, rd[1]));
      const V8 qf = cat<V4, V8>(__builtin_bit_cast(V4, rq[0]), __builtin_bit_cast(V4, rq[1]));
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        dv[c][t] = M::run(df, pf[c], dv[c][t]);
        dk[c][t] = M::run(qf, dsf[c], dk[c][t]);
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's copies of the next tiles have landed
    __syncthreads();                 // ... everyone's, and every wave is done with this step's buffers
  }

  // The two query waves of a key half add their partial sums through LDS (the tile buffers, free now); each of them
  // finishes half of the columns.
  floatx4* part = reinterpret_cast<floatx4*>(smem);  // [wave][c][t][lane], 16 D bytes per lane and wave
  T* dkp = const_cast<T*>(at(g.d_k, hk));
  T* dvp = const_cast<T*>(at(g.d_v, hk));
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    if (which) __syncthreads();  // the first sums are read
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int t = 0; t < DT; ++t) part[((uwave * 2 + c) * DT + t) * kWave + lane] = which ? dk[c][t] : dv[c][t];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int key = wkey0 + 16 * c + l16;
#pragma unroll
      for (int j = 0; j < DT / 2; ++j) {
        const int t = wq * (DT / 2) + j;
        floatx4 y = part[((wk * 2 + c) * DT + t) * kWave + lane];
        const floatx4 z = part[(((2 + wk) * 2 + c) * DT + t) * kWave + lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] += z[i];
        if (which) {
#pragma unroll
          for (int i = 0; i < 4; ++i) y[i] *= a.scale;
        }
        if (key < len) {
          T* row = which ? dkp + int64_t(key) * g.d_k.stride_t : dvp + int64_t(key) * g.d_v.stride_t;
          *reinterpret_cast<V4*>(row + 16 * t + 4 * g4) = M::pack(y);
        }
      }
    }
  }
}

template <int D, typename T>
hipError_t launch_attention_bwd_typed(const gdr_attention_args& a, const gdr_attention_grads& g, hipStream_t stream) {
  constexpr int dq_lds = 4 * kTile * D * int(sizeof(T));                      // K and V, double-buffered
  constexpr int kv_lds = (4 * kTile + kKB) * D * int(sizeof(T));              // q and dO, double-buffered; v
  hipError_t e = configure_lds<&attention_dq_kernel<D, T>>(dq_lds);
  if (e != hipSuccess) return e;
  e = configure_lds<&attention_dkdv_kernel<D, T>>(kv_lds);
  if (e != hipSuccess) return e;
  const int nqb = (a.seq_len + kQB - 1) / kQB, nkb = (a.seq_len + kKB - 1) / kKB;
  const int64_t qslots = a.cu_seqlens ? int64_t(nqb) + a.n_seqs : int64_t(a.batch) * nqb;
  const int64_t kslots = a.cu_seqlens ? int64_t(nkb) + a.n_seqs : int64_t(a.batch) * nkb;
  if (qslots * a.heads > 0)
    hipLaunchKernelGGL((attention_dq_kernel<D, T>), dim3(unsigned(qslots * a.heads)), dim3(attn::kThreads), dq_lds,
                       stream, a, g, nqb);
  if (kslots * a.kv_heads > 0)
    hipLaunchKernelGGL((attention_dkdv_kernel<D, T>), dim3(unsigned(kslots * a.kv_heads)), dim3(attn::kThreads),
                       kv_lds, stream, a, g, nkb);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_attention_bwd(const gdr_attention_args& a, const gdr_attention_grads& g, hipStream_t stream) {
  if (a.q.dtype == GDR_BF16)
    return a.head_dim == 64 ? launch_attention_bwd_typed<64, __bf16>(a, g, stream)
                            : launch_attention_bwd_typed<128, __bf16>(a, g, stream);
  return a.head_dim == 64 ? launch_attention_bwd_typed<64, _Float16>(a, g, stream)
                          : launch_attention_bwd_typed<128, _Float16>(a, g, stream);
}

}  // namespace gdr
