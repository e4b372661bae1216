// The camera head's small kernels for gfx950: attention over one pose token a
// frame (head_dim 128, fp32 arithmetic), the adaLN modulation of the pose
// tokens, and the pose update that ends an iteration.
//
// The head is a chain of launches on a few hundred KB, so each kernel is bound
// by its launch and by one or two memory latencies, not by bytes or
// arithmetic; what pays is doing in one launch what the chain did in several.
// As torch ops the attention took 9 launches, the modulation 7, the pose update
// 5: the eager head at 8 frames went from 4.0 to 2.3 ms, ~400 launches to ~150.
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

}  // namespace qv

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
