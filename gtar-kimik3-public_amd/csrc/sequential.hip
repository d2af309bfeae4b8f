// The chunk op's sequential path on gfx950: every token of each (packed) sequence one after another, the state, every
// product and every sum in fp32 (fp32 q, k, v, and key dims the chunk kernels are not built for).
//
// Same recurrence as recurrent.hip, for calls of many tokens.  There a workgroup's waves share each column's rows, so
// every token costs two workgroup barriers and two LDS round trips (0.76 us per token measured); that is the right
// split when the state stream is the cost, at a token or a few per call.  Here the chain over the tokens is the cost,
// so a wave owns its columns whole: CW value columns per wave, 64 / CW lanes per column, K * CW / 64 state rows per
// lane in registers.  A token is then the decay, the product k S, one DPP reduction over the column's lanes, the
// update and the readout q S (whose reduction nothing waits for), with no barrier.  The four waves of a workgroup
// share the token vectors: q, k, e^g, beta and v of kGroup tokens are staged in LDS (fp32, the exponentials taken
// once per workgroup) while the previous group runs, loaded into registers a group ahead, so one barrier per group
// remains.  A lane keeps the outputs of "its" tokens of the group and stores them at the group's end.
//
// CW trades the chain's length against the work: 2 columns per wave have the shortest chain (4 rows per lane at
// K = 128) and fill the 1,024 SIMDs from 2,048 columns on; 8 columns need half the instructions per column (the
// reduction and the token's scalars are shared by more rows) once there are waves enough without the narrow split.
//
// Measured (fp32 KDA, K = V = 128; recurrent kernel -> here): B = 2, H = 8, T = 777 588 -> 152 us, 0.2 us per token,
// the chain's own latency (some 50 dependent instructions); B = 8, H = 24, T = 512 539 -> 286 us, where the vector ALU
// and the LDS reads of q, k, e^g (48 floats a lane and token) share the time.  Error against fp64 as before: 9.5e-8.
#include "gdr_common.h"
#include "gdr_internal.h"
#include "varlen_index.h"

namespace gdr {

namespace {

constexpr int kSeqWaves = 4;
constexpr int kSeqThreads = kSeqWaves * kWave;

// Sum over the RL consecutive lanes (aligned) a lane belongs to, in every one of them.  Within a row of 16 lanes the
// partners come by DPP: quad_perm for 1 and 2, then the mirrored half row for 4 (its lanes hold the other quad's sum,
// all four equal by then) and the row rotated by 8; 16 by the permlane swap.  No LDS round trip, unlike xor_sum's 4.
template <int RL>
__device__ __forceinline__ float lanes_sum(float x) {
  if constexpr (RL >= 2) x = xor_sum(x, 1);
  if constexpr (RL >= 4) x = xor_sum(x, 2);
  if constexpr (RL >= 8)
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xf, 0xf, false));  // row_half_mirror
  if constexpr (RL >= 16) x = xor_sum(x, 8);
  if constexpr (RL >= 32) x = xor_sum(x, 16);
  return x;
}

template <int N>
__device__ __forceinline__ float tree_sum(const float (&x)[N]) {
  if constexpr (N == 1) {
    return x[0];
  } else {
    float y[(N + 1) / 2];
#pragma unroll
    for (int i = 0; i < N / 2; ++i) y[i] = x[2 * i] + x[2 * i + 1];
    if constexpr (N % 2) y[N / 2] = x[N - 1];
    return tree_sum(y);
  }
}

template <int VARIANT, int K, int CW, typename InT>
__global__ __launch_bounds__(kSeqThreads) void sequential_fwd_kernel(const gdr_args a, int n_slices) {
  constexpr int RL = kWave / CW;                         // lanes per column
  constexpr int RPL = K / RL;                            // state rows per lane
  constexpr int VW = RPL % 4 == 0 ? 4 : RPL % 2 == 0 ? 2 : 1;  // consecutive rows of a lane, one LDS read each
  constexpr int NJ = RPL / VW;                           // row j * RL * VW + rl * VW + i for j < NJ, i < VW
  constexpr int WC = kSeqWaves * CW;                     // columns per workgroup
  constexpr int kGroup = K <= 128 ? 16 : 8;              // tokens staged at a time (two buffers in 64 KB of LDS)
  constexpr int kHeld = (kGroup + RL - 1) / RL;          // outputs a lane keeps per group
  constexpr int NK = kGroup * K / kSeqThreads;           // q / k / gate elements per thread and group
  constexpr int NV = (kGroup * WC + kSeqThreads - 1) / kSeqThreads;
  static_assert(RL >= 1 && K % RL == 0 && (kGroup * K) % kSeqThreads == 0 && kGroup % 4 == 0, "bad tiling");
  constexpr bool kDelta = VARIANT != GDR_GLA;
  constexpr bool kChannelGate = VARIANT == GDR_KDA || VARIANT == GDR_GLA;
  constexpr bool kScalarGate = VARIANT == GDR_GDN;

  // The slices of one head read the same token vectors: consecutive logical blocks go to one XCD (block x runs on
  // XCD x mod 8) when the grid divides evenly.
  const int nb = gridDim.x;
  const int block = nb % 8 == 0 ? (blockIdx.x % 8) * (nb / 8) + blockIdx.x / 8 : blockIdx.x;
  const int slice = block % n_slices, bh = block / n_slices;  // bh: (batch entry or packed sequence) * H + head
  const int H = a.heads, V = a.value_dim, h = bh % H;
  int b = bh / H, bos = 0, T = a.seq_len;
  if (a.cu_seqlens) {
    bos = packed_begin(a.cu_seqlens, b, a.seq_len);
    T = packed_end(a.cu_seqlens, b, a.seq_len) - bos;
    b = 0;
  }
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int rl = lane % RL, wcol = wave * CW + lane / RL;  // lane's place in its column, column of the workgroup
  const int v0 = slice * WC;

  __shared__ __align__(16) float s_q[2][kGroup][K], s_k[2][kGroup][K], s_eg[2][kChannelGate ? kGroup : 1][K];
  __shared__ float s_v[2][kGroup][WC], s_beta[2][kGroup], s_dec[2][kGroup];

  const InT* qp = static_cast<const InT*>(a.q.ptr) + b * a.q.stride_b + h * a.q.stride_h + bos * a.q.stride_t;
  const InT* kp = static_cast<const InT*>(a.k.ptr) + b * a.k.stride_b + h * a.k.stride_h + bos * a.k.stride_t;
  const InT* vp = static_cast<const InT*>(a.v.ptr) + b * a.v.stride_b + h * a.v.stride_h + bos * a.v.stride_t + v0;
  const int64_t ob = b * a.out.stride_b + h * a.out.stride_h + bos * a.out.stride_t + v0 + wcol;
  const float* gp = static_cast<const float*>(a.gate.ptr) + b * a.gate.stride_b + h * a.gate.stride_h +
                    bos * a.gate.stride_t;
  const float* bp = static_cast<const float*>(a.beta.ptr) + b * a.beta.stride_b + h * a.beta.stride_h +
                    bos * a.beta.stride_t;

  InT raw_q[NK], raw_k[NK], raw_v[NV];
  float raw_g[kChannelGate ? NK : 1], raw_beta = 0.f, raw_sg = 0.f;
  auto fetch = [&](int t0) {  // element i of the group's [kGroup][K] block goes to thread i % kSeqThreads
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int i = tid + j * kSeqThreads, t = t0 + i / K, c = i % K;
      if (t < T) {
        raw_q[j] = qp[t * a.q.stride_t + c];
        raw_k[j] = kp[t * a.k.stride_t + c];
        if constexpr (kChannelGate) raw_g[j] = gp[t * a.gate.stride_t + c];
      }
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = tid + j * kSeqThreads, t = t0 + i / WC;
      if (i < kGroup * WC && t < T) raw_v[j] = vp[t * a.v.stride_t + i % WC];
    }
    if (tid < kGroup && t0 + tid < T) {
      if constexpr (kDelta) raw_beta = bp[(t0 + tid) * a.beta.stride_t];
      if constexpr (kScalarGate) raw_sg = gp[(t0 + tid) * a.gate.stride_t];
    }
  };
  auto stage = [&](int t0, int buf) {
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int i = tid + j * kSeqThreads, tt = i / K, c = i % K;
      if (t0 + tt < T) {
        s_q[buf][tt][c] = static_cast<float>(raw_q[j]);
        s_k[buf][tt][c] = static_cast<float>(raw_k[j]);
        if constexpr (kChannelGate) s_eg[buf][tt][c] = exp_fast(raw_g[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = tid + j * kSeqThreads, tt = i / WC;
      if (i < kGroup * WC && t0 + tt < T) s_v[buf][tt][i % WC] = static_cast<float>(raw_v[j]);
    }
    if (tid < kGroup && t0 + tid < T) {
      if constexpr (kDelta) s_beta[buf][tid] = raw_beta;
      if constexpr (kScalarGate) s_dec[buf][tid] = exp_fast(raw_sg);
    }
  };

  const size_t state_base = size_t(bh) * K * V + v0 + wcol;
  float st[NJ][VW];
  fetch(0);
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int i = 0; i < VW; ++i)
      st[j][i] = a.h0 ? a.h0[state_base + size_t(j * RL * VW + rl * VW + i) * V] : 0.f;
  stage(0, 0);
  __syncthreads();

  float held[kHeld];
  auto token = [&](int buf, int tt) {
    const float *kr = &s_k[buf][tt][rl * VW], *qr = &s_q[buf][tt][rl * VW];
    const float* er = &s_eg[buf][kChannelGate ? tt : 0][rl * VW];
    float k[NJ][VW], q[NJ][VW], e[NJ][VW];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < VW; ++i) {
        k[j][i] = kr[j * RL * VW + i];
        q[j][i] = qr[j * RL * VW + i];
        if constexpr (kChannelGate) e[j][i] = er[j * RL * VW + i];
      }
    const float v = s_v[buf][tt][wcol];
    const float beta = kDelta ? s_beta[buf][tt] : 1.f, dec = kScalarGate ? s_dec[buf][tt] : 1.f;
    float ks[NJ], qs[NJ];  // chains of VW rows, then a tree: shorter, and rounding no worse than the wave-split sums
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      ks[j] = 0.f;
#pragma unroll
      for (int i = 0; i < VW; ++i) {
        if constexpr (kChannelGate) st[j][i] *= e[j][i];
        if constexpr (kScalarGate) st[j][i] *= dec;
        if constexpr (kDelta) ks[j] = __builtin_fmaf(k[j][i], st[j][i], ks[j]);
      }
    }
    const float u = kDelta ? beta * (v - lanes_sum<RL>(tree_sum(ks))) : v;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      qs[j] = 0.f;
#pragma unroll
      for (int i = 0; i < VW; ++i) {
        st[j][i] = __builtin_fmaf(k[j][i], u, st[j][i]);
        qs[j] = __builtin_fmaf(q[j][i], st[j][i], qs[j]);
      }
    }
    const float o = lanes_sum<RL>(tree_sum(qs));
#pragma unroll
    for (int s = 0; s < kHeld; ++s) held[s] = tt == s * RL + rl ? o : held[s];
  };

  for (int t0 = 0, buf = 0; t0 < T; t0 += kGroup, buf ^= 1) {
    const int n = min(kGroup, T - t0);
    if (t0 + kGroup < T) fetch(t0 + kGroup);
    int tt = 0;
    for (; tt + 4 <= n; tt += 4)
#pragma unroll
      for (int s = 0; s < 4; ++s) token(buf, tt + s);
    for (; tt < n; ++tt) token(buf, tt);
#pragma unroll
    for (int s = 0; s < kHeld; ++s) {
      const int t = s * RL + rl;
      if (t < n) store_any(const_cast<void*>(a.out.ptr), ob + (t0 + t) * a.out.stride_t, a.out.dtype, a.scale * held[s]);
    }
    // The other buffer's last readers passed the barrier that ended the previous group.
    if (t0 + kGroup < T) stage(t0 + kGroup, buf ^ 1);
    __syncthreads();
  }

  if (a.ht) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < VW; ++i) a.ht[state_base + size_t(j * RL * VW + rl * VW + i) * V] = st[j][i];
  }
}

template <int VARIANT, int K, int CW, typename InT>
hipError_t launch_cw(const gdr_args& a, hipStream_t stream) {
  const int n_slices = a.value_dim / (kSeqWaves * CW);  // value dims are multiples of 32
  const dim3 grid((a.cu_seqlens ? a.n_seqs : a.batch) * a.heads * n_slices);
  hipLaunchKernelGGL((sequential_fwd_kernel<VARIANT, K, CW, InT>), grid, dim3(kSeqThreads), 0, stream, a, n_slices);
  return hipGetLastError();
}

// Columns per wave, narrow (the shortest chain) and wide (the least work per column), and the most columns of a call
// that the narrow split still serves best (us, narrow / wide, fp32 KDA: K = 128 T = 777 197 / 265 at 4,096 columns and
// 247 / 266 at 6,144, T = 512 230 / 176 at 8,192; K = 64 T = 777 219 / 232 at 16,384; K = 256 T = 777 308 / 324 at
// 1,024, 385 / 316 at 2,048).
template <int K>
struct SeqSplit;
template <> struct SeqSplit<32> { static constexpr int narrow = 2, wide = 8; static constexpr int64_t most = 6144; };
template <> struct SeqSplit<64> { static constexpr int narrow = 4, wide = 8; static constexpr int64_t most = 20480; };
template <> struct SeqSplit<128> { static constexpr int narrow = 2, wide = 8; static constexpr int64_t most = 6144; };
template <> struct SeqSplit<192> { static constexpr int narrow = 2, wide = 4; static constexpr int64_t most = 2048; };
template <> struct SeqSplit<256> { static constexpr int narrow = 2, wide = 4; static constexpr int64_t most = 1536; };

template <int VARIANT, int K, typename InT>
hipError_t launch_k(const gdr_args& a, hipStream_t stream) {
  using S = SeqSplit<K>;
  const int64_t columns = int64_t(a.cu_seqlens ? a.n_seqs : a.batch) * a.heads * a.value_dim;
  return columns <= S::most ? launch_cw<VARIANT, K, S::narrow, InT>(a, stream)
                            : launch_cw<VARIANT, K, S::wide, InT>(a, stream);
}

template <int VARIANT, typename InT>
hipError_t launch_v(const gdr_args& a, hipStream_t stream) {
  switch (a.key_dim) {
    case 32: return launch_k<VARIANT, 32, InT>(a, stream);
    case 64: return launch_k<VARIANT, 64, InT>(a, stream);
    case 128: return launch_k<VARIANT, 128, InT>(a, stream);
    case 192: return launch_k<VARIANT, 192, InT>(a, stream);
    default: return launch_k<VARIANT, 256, InT>(a, stream);
  }
}

template <typename InT>
hipError_t launch_t(const gdr_args& a, hipStream_t stream) {
  switch (a.variant) {
    case GDR_KDA: return launch_v<GDR_KDA, InT>(a, stream);
    case GDR_GDN: return launch_v<GDR_GDN, InT>(a, stream);
    case GDR_GLA: return launch_v<GDR_GLA, InT>(a, stream);
    default: return launch_v<GDR_DELTANET, InT>(a, stream);
  }
}

}  // namespace

// The recurrent kernel keeps the calls it serves better (us per call, recurrent / here, fp32 KDA, V = 128):
//   * few tokens: its state loads and stores are whole rows, where a wave here touches CW columns of every row.  From
//     8 tokens on this kernel wins (B = 2, H = 16, K = 128, T = 8: 8.5 / 6.2), at K = 256 from 16 (B = 4, H = 16: T = 12
//     16.8 / 17.3, T = 16 20.5 / 17.5), for key dims above 128 (more state per column) and more than 8,192 columns from
//     about 64 (B = 8, H = 24, K = 256: T = 16 32.5 / 38.2, T = 200 308 / 259);
//   * calls that fill the chip with its workgroups: at K = 128 the 128-column ones, where both are bound by the vector ALU
//     and q, k and e^g cost those fewer LDS reads (H = 16, 16 / 100 tokens: B = 24 28.7 / 26.6 and 130 / 115, B = 32
//     30.5 / 33.9 and 132 / 145, B = 64 53.8 / 61.1 and 259 / 296); at K = 192 the scalar gate, whose decay costs those one
//     multiplication by a register (GDN, H = 16, 100 tokens: B = 16 156 / 160, B = 31 276 / 309; KDA 176 / 144 and
//     327 / 277).  At K = 32 and 64 the wide split stays ahead (B = 64, K = 64: 16 tokens 38.1 / 33.9, 100 tokens
//     186 / 161).
// A packed call is judged by its average sequence, the offsets being on the device: among many short sequences the recurrent
// kernel is faster (H = 16, K = 128, 128 sequences of 4 tokens 51 / 91), but one long prompt among them takes it 0.95 us a
// token (250 sequences of one token and one of 1,500: 1,421 / 922).
hipError_t launch_sequential(const gdr_args& a, hipStream_t stream) {
  const int64_t n = a.cu_seqlens ? a.n_seqs : a.batch, columns = n * a.heads * a.value_dim;
  const int64_t tokens = a.cu_seqlens ? a.seq_len / n : a.seq_len;  // of an average sequence
  const int enough = a.key_dim > 128 && columns > 8192 ? 64 : a.key_dim == 256 && columns > 4096 ? 16 : 8;
  const bool few = tokens < enough;
  const bool full = a.key_dim == 128   ? a.value_dim % 128 == 0 && columns >= 65536
                    : a.key_dim == 192 ? a.variant == GDR_GDN && columns >= 32768
                                       : false;
  if (few || full) return launch_recurrent(a, stream);
  return a.q.dtype == GDR_BF16 ? launch_t<__bf16>(a, stream) : launch_t<float>(a, stream);
}

}  // namespace gdr
