// The camera head's small kernels for gfx950: attention over one pose token a
// frame (head_dim 128, fp32 arithmetic), the adaLN modulation of the pose
// tokens, and the pose update that ends an iteration.
//
// The head is a chain of launches on a few hundred KB, so each kernel is bound
// by its launch and by one or two memory latencies, not by bytes or
// arithmetic; what pays is doing in one launch what the chain did in several.
// As torch ops the attention took 9 launches, the modulation 7, the pose update
// 5: the eager head at 8 frames went from 4.0 to 2.3 ms; with its own linears
// here too (below) and the trunk's norms in their linears, to 1.15 ms and from
// ~400 launches to 102.
#include <type_traits>

#include "common.h"

namespace qv {

// ------------------------------------------------- attention, head_dim 128
// softmax(q k^T * scale) v for S tokens of a fused (S, 3, H, 128) fp16 qkv,
// scores, softmax and sums in fp32 (no fp16 probabilities, so no MFMA).  A
// workgroup takes 4 queries of one head, one a wave, and walks the keys in
// tiles of 64 staged in LDS (K rows padded to 272 bytes: lane = key reads 16
// bytes a row on distinct banks).  QK^T: lane = key, q broadcast from LDS; PV:
// lane = two dims, the probabilities broadcast.  One query a wave is the most
// waves and the shortest chain: 2 or 4 (K / V reads shared) measured 5.6 / 8.8
// us against 3.9 at 8 tokens, 7.0 / 10.5 against 4.9 at 64, 23.8 / 33.6
// against 23.6 at 256.  The torch ops it replaces took 22, 26 and 96 us.
constexpr int PA_KT = 64;
constexpr int PA_KROW = 272;   // bytes of a staged K row

__global__ __launch_bounds__(256) void pose_attention_kernel(const uint16_t* __restrict__ qkv,
                                                             uint16_t* __restrict__ out, int S, int H, float scale) {
  __shared__ __attribute__((aligned(16))) uint8_t kl[PA_KT * PA_KROW];
  __shared__ __attribute__((aligned(16))) uint8_t vl[PA_KT * 256];
  __shared__ __attribute__((aligned(16))) float ql[4][128];
  __shared__ __attribute__((aligned(16))) float pl[4][PA_KT];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int head = blockIdx.x % H;
  const int qi = (blockIdx.x / H) * 4 + wave;
  const size_t ts = (size_t)3 * H * 128;   // halves a token

  // K / V tile rows: thread t copies 16-byte chunk t % 16 of rows t / 16 + 16 i
  const int ch = tid & 15, r0 = tid >> 4;
  uint4 kr[4], vr[4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = k0 + r0 + 16 * i;
      kr[i] = vr[i] = make_uint4(0, 0, 0, 0);
      if (key < S) {
        const uint16_t* p = qkv + key * ts + (size_t)(H + head) * 128 + ch * 8;
        kr[i] = *reinterpret_cast<const uint4*>(p);
        vr[i] = *reinterpret_cast<const uint4*>(p + (size_t)H * 128);
      }
    }
  };
  fetch(0);
  {
    const int qc = qi < S ? qi : S - 1;
    const uint32_t w = *reinterpret_cast<const uint32_t*>(qkv + qc * ts + (size_t)head * 128 + 2 * lane);
    ql[wave][2 * lane] = to_f32((uint16_t)(w & 0xFFFF), false);
    ql[wave][2 * lane + 1] = to_f32((uint16_t)(w >> 16), false);
  }
  float m = -INFINITY, l = 0.f, o0 = 0.f, o1 = 0.f;
  for (int k0 = 0; k0 < S; k0 += PA_KT) {
    if (k0) __syncthreads();   // every wave is done with the last tile
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = r0 + 16 * i;
      *reinterpret_cast<uint4*>(kl + r * PA_KROW + ch * 16) = kr[i];
      *reinterpret_cast<uint4*>(vl + r * 256 + ch * 16) = vr[i];
    }
    __syncthreads();
    if (k0 + PA_KT < S) fetch(k0 + PA_KT);   // lands under this tile's arithmetic
    float s = 0.f;
#pragma unroll 4
    for (int c = 0; c < 16; ++c) {
      const uint4 u = *reinterpret_cast<const uint4*>(kl + lane * PA_KROW + c * 16);
      const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s = __builtin_fmaf(ql[wave][8 * c + 2 * e], to_f32((uint16_t)(w[e] & 0xFFFF), false), s);
        s = __builtin_fmaf(ql[wave][8 * c + 2 * e + 1], to_f32((uint16_t)(w[e] >> 16), false), s);
      }
    }
    s = k0 + lane < S ? s * scale : -INFINITY;
    float mx = s;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) mx = fmaxf(mx, __shfl_xor(mx, d));
    mx = fmaxf(m, mx);
    const float p = expf(s - mx), alpha = expf(m - mx);   // alpha 0 on the first tile
    m = mx;
    l = l * alpha + p;   // this lane's share; summed over lanes at the end
    o0 *= alpha;
    o1 *= alpha;
    pl[wave][lane] = p;
    __builtin_amdgcn_wave_barrier();   // pl[wave] is the wave's own: its LDS operations are in order
    const int nk = S - k0 < PA_KT ? S - k0 : PA_KT;
    for (int k = 0; k < nk; k += 4) {   // rows past nk hold zeros and p = 0
      const float4 p4 = *reinterpret_cast<const float4*>(&pl[wave][k]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t w = *reinterpret_cast<const uint32_t*>(vl + (k + j) * 256 + 4 * lane);
        const float pj = j == 0 ? p4.x : j == 1 ? p4.y : j == 2 ? p4.z : p4.w;
        o0 = __builtin_fmaf(pj, to_f32((uint16_t)(w & 0xFFFF), false), o0);
        o1 = __builtin_fmaf(pj, to_f32((uint16_t)(w >> 16), false), o1);
      }
    }
  }
#pragma unroll
  for (int d = 1; d < 64; d *= 2) l += __shfl_xor(l, d);
  const float inv = 1.0f / l;
  if (qi < S)
    *reinterpret_cast<uint32_t*>(out + ((size_t)qi * H + head) * 128 + 2 * lane) = pack2<false>(o0 * inv, o1 * inv);
}

// ------------------------------------------------------- adaLN modulation
// x = gate * (adaln * (1 + scale) + shift) + pose in fp32, one rounding; mod
// holds (shift | scale | gate), D each, a row.  8 columns a thread.
__global__ __launch_bounds__(256) void adaln_modulate_kernel(const uint16_t* __restrict__ mod,
                                                             const uint16_t* __restrict__ adaln,
                                                             const uint16_t* __restrict__ pose,
                                                             uint16_t* __restrict__ x, long n8, int D) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const int d8 = D / 8;
  const long row = i / d8;
  const int c = (int)(i % d8) * 8;
  const uint16_t* mp = mod + row * 3 * D + c;
  const uint4 u[5] = {*reinterpret_cast<const uint4*>(mp), *reinterpret_cast<const uint4*>(mp + D),
                      *reinterpret_cast<const uint4*>(mp + 2 * D), *reinterpret_cast<const uint4*>(adaln + row * D + c),
                      *reinterpret_cast<const uint4*>(pose + row * D + c)};
  uint32_t w[5][4], r[4];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    w[k][0] = u[k].x;
    w[k][1] = u[k].y;
    w[k][2] = u[k].z;
    w[k][3] = u[k].w;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float y[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float f[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) f[k] = to_f32((uint16_t)(h ? w[k][e] >> 16 : w[k][e] & 0xFFFF), false);
      y[h] = __builtin_fmaf(f[2], __builtin_fmaf(f[3], 1.0f + f[1], f[0]), f[4]);
    }
    r[e] = pack2<false>(y[0], y[1]);
  }
  *reinterpret_cast<uint4*>(x + row * D + c) = make_uint4(r[0], r[1], r[2], r[3]);
}

// ------------------------------------------------------------ pose update
// One iteration's end: pred (fp32, in place) takes the fp16 delta -- added, or
// stored when first --, act = pred with its columns from n_linear on through
// ReLU (NaN stays), half = pred rounded to fp16, the next iteration's input.
__global__ __launch_bounds__(256) void pose_update_kernel(const uint16_t* __restrict__ delta, float* __restrict__ pred,
                                                          float* __restrict__ act, uint16_t* __restrict__ half, long n,
                                                          int cols, int n_linear, int first) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float d = to_f32(delta[i], false);
  const float p = first ? d : pred[i] + d;
  pred[i] = p;
  act[i] = (int)(i % cols) >= n_linear && p < 0.f ? 0.f : p;
  half[i] = from_f32<false>(p);
}

// ------------------------------------------------ fp16 linears of the head
// silu(src w^T + b) for src (S, C <= 16) and w (N, C): the embedded pose.
// One output a thread.
__global__ __launch_bounds__(256) void pose_embed_kernel(const uint16_t* __restrict__ src, long src_stride,
                                                         const uint16_t* __restrict__ w,
                                                         const uint16_t* __restrict__ b, uint16_t* __restrict__ out,
                                                         int S, int N, int C) {
  const int n = blockIdx.x * 256 + threadIdx.x, s = blockIdx.y;
  if (n >= N) return;
  float e = to_f32(b[n], false);
  for (int c = 0; c < C; ++c)
    e = __builtin_fmaf(to_f32(src[s * src_stride + c], false), to_f32(w[(long)n * C + c], false), e);
  out[(long)s * N + n] = from_f32<false>(e / (1.0f + expf(-e)));
}

// x w^T of up to 16 tokens a workgroup row (blockIdx.y) and 16 channels of each
// of PARTS weight blocks (N rows apart): 8 waves split K in steps of 32, the
// weights are the A operand and the tokens the B operand of
// v_mfma_f32_16x16x32_f16, partial sums meet in LDS and wave 0 finishes:
//  MODE 0: out = gelu(sum + b)
//  MODE 1: PARTS = 3 (shift, scale, gate): out = gate * (adaln * (1 + scale)
//          + shift) + pose
//  MODE 2: the pose update of pose_update_kernel with delta = sum + b
// Bound by latency and the weight stream (25 MB at 2048 -> 3 x 2048).  As
// library products with torch's passes between them an iteration's four
// linears took ~35 us of GPU time and ~25 us of host time each.
struct PoseTail {
  const uint16_t *adaln, *pose;
  float *pred, *act;
  uint16_t* half;
  int n_linear, first;
};

template <int MODE, int PARTS>
__global__ __launch_bounds__(512) void pose_linear_kernel(const uint16_t* __restrict__ x,
                                                          const uint16_t* __restrict__ w,
                                                          const uint16_t* __restrict__ bias,
                                                          uint16_t* __restrict__ out, int S, int N, int K, PoseTail tail) {
  constexpr int W = 8;
  __shared__ float4 part[W][PARTS][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int n_a = blockIdx.x * 16 + c, t_b = blockIdx.y * 16 + c;
  // rows past N and tokens past S repeat the last one; their results are not stored
  const uint16_t* wp = w + (long)(n_a < N ? n_a : N - 1) * K + 8 * g;
  const uint16_t* xp = x + (long)(t_b < S ? t_b : S - 1) * K + 8 * g;
  f32x4 acc[PARTS];
#pragma unroll
  for (int p = 0; p < PARTS; ++p) acc[p] = f32x4{0.f, 0.f, 0.f, 0.f};
  // U steps' loads are issued together, then their products
  auto steps = [&](int k, auto uc) __attribute__((always_inline)) {
    constexpr int U = decltype(uc)::value;
    uint4 b[U], a[U][PARTS];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      b[u] = *reinterpret_cast<const uint4*>(xp + k + 32 * W * u);
#pragma unroll
      for (int p = 0; p < PARTS; ++p) a[u][p] = *reinterpret_cast<const uint4*>(wp + (long)p * N * K + k + 32 * W * u);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int p = 0; p < PARTS; ++p)
        acc[p] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[u][p]),
                                                        __builtin_bit_cast(f16x8, b[u]), acc[p], 0, 0, 0);
  };
  int k = 32 * wave;
  for (; k + 32 * W * 3 < K; k += 32 * W * 4) steps(k, std::integral_constant<int, 4>());
  for (; k < K; k += 32 * W) steps(k, std::integral_constant<int, 1>());
#pragma unroll
  for (int p = 0; p < PARTS; ++p) part[wave][p][lane] = make_float4(acc[p][0], acc[p][1], acc[p][2], acc[p][3]);
  __syncthreads();
  if (wave) return;
  // lane (g, c): channels 16 bx + 4 g + r (r = 0..3) of token 16 by + c
  const int t = t_b, n0 = blockIdx.x * 16 + 4 * g;
  float y[PARTS][4];
#pragma unroll
  for (int p = 0; p < PARTS; ++p) {
#pragma unroll
    for (int r = 0; r < 4; ++r) y[p][r] = n0 + r < N ? to_f32(bias[p * N + n0 + r], false) : 0.f;
#pragma unroll
    for (int v = 0; v < W; ++v) {
      const float4 q = part[v][p][lane];
      y[p][0] += q.x;
      y[p][1] += q.y;
      y[p][2] += q.z;
      y[p][3] += q.w;
    }
  }
  if (t >= S) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = n0 + r;
    if (n >= N) break;
    const long i = (long)t * N + n;
    if constexpr (MODE == 0) {
      out[i] = from_f32<false>(gelu_erf_fine(y[0][r]));
    } else if constexpr (MODE == 1) {
      out[i] = from_f32<false>(__builtin_fmaf(
          y[2][r], __builtin_fmaf(to_f32(tail.adaln[i], false), 1.0f + y[1][r], y[0][r]), to_f32(tail.pose[i], false)));
    } else {
      const float p = tail.first ? y[0][r] : tail.pred[i] + y[0][r];
      tail.pred[i] = p;
      tail.act[i] = n >= tail.n_linear && p < 0.f ? 0.f : p;
      tail.half[i] = from_f32<false>(p);
    }
  }
}

static int pose_linear_check(const void* x, const void* w, const void* bias, int64_t S, int64_t N, int64_t K) {
  QV_CHECK_ARG(S >= 0 && S <= 65535 * 16 && N > 0 && K > 0 && K % 32 == 0 && N <= INT32_MAX / 4 && K <= INT32_MAX / 4,
               "bad shape S=%lld N=%lld K=%lld (K a multiple of 32)", (long long)S, (long long)N, (long long)K);
  QV_CHECK_ARG(S == 0 || (x && w && bias), "null pointer argument");
  QV_CHECK_ARG((((uintptr_t)x | (uintptr_t)w) % 16) == 0, "x and w must be 16-byte aligned");
  return QV_OK;
}

}  // namespace qv

extern "C" int qv_pose_embed(const void* src, int64_t src_stride, const void* w, const void* bias, void* out, int64_t S,
                             int64_t N, int64_t C, void* stream) {
  QV_CHECK_ARG(S >= 0 && S <= 65535 && N > 0 && N <= INT32_MAX - 256 && C > 0 && C <= 16 && src_stride >= 0,
               "bad shape S=%lld N=%lld C=%lld", (long long)S, (long long)N, (long long)C);
  if (S == 0) return QV_OK;
  QV_CHECK_ARG(src && w && bias && out, "null pointer argument");
  hipLaunchKernelGGL(qv::pose_embed_kernel, dim3((unsigned)((N + 255) / 256), (unsigned)S), dim3(256), 0,
                     (hipStream_t)stream, (const uint16_t*)src, (long)src_stride, (const uint16_t*)w,
                     (const uint16_t*)bias, (uint16_t*)out, (int)S, (int)N, (int)C);
  return qv::check_launch("pose_embed");
}

extern "C" int qv_pose_linear_gelu(const void* x, const void* w, const void* bias, void* out, int64_t S, int64_t N,
                                   int64_t K, void* stream) {
  if (const int rc = qv::pose_linear_check(x, w, bias, S, N, K)) return rc;
  if (S == 0) return QV_OK;
  QV_CHECK_ARG(out, "null pointer argument");
  hipLaunchKernelGGL((qv::pose_linear_kernel<0, 1>), dim3((unsigned)((N + 15) / 16), (unsigned)((S + 15) / 16)),
                     dim3(512), 0, (hipStream_t)stream, (const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias,
                     (uint16_t*)out, (int)S, (int)N, (int)K, qv::PoseTail());
  return qv::check_launch("pose_linear_gelu");
}

extern "C" int qv_pose_modulate(const void* e, const void* w, const void* bias, const void* adaln, const void* pose,
                                void* x, int64_t S, int64_t D, int64_t K, void* stream) {
  if (const int rc = qv::pose_linear_check(e, w, bias, S, D, K)) return rc;
  if (S == 0) return QV_OK;
  QV_CHECK_ARG(adaln && pose && x, "null pointer argument");
  qv::PoseTail tail = {(const uint16_t*)adaln, (const uint16_t*)pose, nullptr, nullptr, nullptr, 0, 0};
  hipLaunchKernelGGL((qv::pose_linear_kernel<1, 3>), dim3((unsigned)((D + 15) / 16), (unsigned)((S + 15) / 16)),
                     dim3(512), 0, (hipStream_t)stream, (const uint16_t*)e, (const uint16_t*)w, (const uint16_t*)bias,
                     (uint16_t*)x, (int)S, (int)D, (int)K, tail);
  return qv::check_launch("pose_modulate");
}

extern "C" int qv_pose_delta(const void* x, const void* w, const void* bias, float* pred, float* act, void* half,
                             int64_t S, int64_t cols, int64_t K, int64_t n_linear, int first, void* stream) {
  if (const int rc = qv::pose_linear_check(x, w, bias, S, cols, K)) return rc;
  if (S == 0) return QV_OK;
  QV_CHECK_ARG(pred && act && half && n_linear >= 0, "null pointer argument");
  qv::PoseTail tail = {nullptr, nullptr, pred, act, (uint16_t*)half, (int)(n_linear < cols ? n_linear : cols), first};
  hipLaunchKernelGGL((qv::pose_linear_kernel<2, 1>), dim3((unsigned)((cols + 15) / 16), (unsigned)((S + 15) / 16)),
                     dim3(512), 0, (hipStream_t)stream, (const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias,
                     (uint16_t*)nullptr, (int)S, (int)cols, (int)K, tail);
  return qv::check_launch("pose_delta");
}

extern "C" int qv_pose_attention(const void* qkv, void* out, int64_t S, int64_t H, int64_t head_dim, float scale,
                                 void* stream) {
  QV_CHECK_ARG(head_dim == 128, "only head_dim 128 is supported (got %lld)", (long long)head_dim);
  QV_CHECK_ARG(S >= 0 && H > 0, "bad shape S=%lld H=%lld", (long long)S, (long long)H);
  if (S == 0) return QV_OK;
  QV_CHECK_ARG(qkv && out, "null pointer argument");
  QV_CHECK_ARG(((uintptr_t)qkv % 16) == 0 && ((uintptr_t)out % 4) == 0,
               "qkv must be 16-byte and out 4-byte aligned");
  const int64_t nwg = (S + 3) / 4 * H;
  QV_CHECK_ARG(S <= INT32_MAX / 128 && H <= INT32_MAX && nwg <= INT32_MAX, "too many tokens");
  hipLaunchKernelGGL(qv::pose_attention_kernel, dim3((unsigned)nwg), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t*)qkv, (uint16_t*)out, (int)S, (int)H, scale);
  return qv::check_launch("pose_attention");
}

extern "C" int qv_adaln_modulate(const void* mod, const void* adaln, const void* pose, void* x, int64_t S, int64_t D,
                                 void* stream) {
  QV_CHECK_ARG(S >= 0 && D > 0 && D % 8 == 0 && D <= INT32_MAX, "bad shape S=%lld D=%lld (D a multiple of 8)",
               (long long)S, (long long)D);
  if (S == 0) return QV_OK;
  QV_CHECK_ARG(mod && adaln && pose && x, "null pointer argument");
  QV_CHECK_ARG((((uintptr_t)mod | (uintptr_t)adaln | (uintptr_t)pose | (uintptr_t)x) % 16) == 0,
               "mod, adaln, pose and x must be 16-byte aligned");
  QV_CHECK_ARG(S <= (int64_t)INT32_MAX * 256 / (D / 8), "too many rows");
  const long n8 = S * (D / 8);
  hipLaunchKernelGGL(qv::adaln_modulate_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t*)mod, (const uint16_t*)adaln, (const uint16_t*)pose, (uint16_t*)x, n8, (int)D);
  return qv::check_launch("adaln_modulate");
}

extern "C" int qv_pose_update(const void* delta, float* pred, float* act, void* half, int64_t S, int64_t cols,
                              int64_t n_linear, int first, void* stream) {
  QV_CHECK_ARG(S >= 0 && cols > 0 && cols <= INT32_MAX && n_linear >= 0, "bad shape S=%lld cols=%lld", (long long)S,
               (long long)cols);
  if (S == 0) return QV_OK;
  QV_CHECK_ARG(delta && pred && act && half, "null pointer argument");
  QV_CHECK_ARG(S <= (int64_t)INT32_MAX * 256 / cols, "too many rows");
  const long n = S * cols;
  hipLaunchKernelGGL(qv::pose_update_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t*)delta, pred, act, (uint16_t*)half, n, (int)cols,
                     (int)(n_linear < cols ? n_linear : cols), first);
  return qv::check_launch("pose_update");
}
