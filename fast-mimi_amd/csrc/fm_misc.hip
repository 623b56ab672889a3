// Small memory-bound kernels of the Mimi hot path and library identity.

#include <initializer_list>

#include "fm_common.h"

namespace {

// Depthwise causal ConvTranspose1d (groups == channels), trimmed to L*stride:
// y[b, q*s + r, c] = sum_{j} x[b, q - j, c] * w[c, r + j*s],  j = 0..k/s-1, q-j >= 0.
// The sum runs j = taps-1 .. 0 (earliest input first), each product rounded.
__global__ __launch_bounds__(256) void upsample_depthwise_kernel(const float* __restrict__ x,
                                                                 const float* __restrict__ w,
                                                                 int B, int L, int C, int k, int s,
                                                                 float* __restrict__ y) {
  const long total = (long)B * L * s * C;
  const int taps = k / s;
  for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const int c = (int)(e % C);
    const long o = e / C;  // output position within all batches
    const long b = o / ((long)L * s);
    const int tout = (int)(o - b * (long)L * s);
    const int q = tout / s, r = tout - q * s;
    float acc = 0.0f;
    bool first = true;
    for (int j = taps - 1; j >= 0; --j) {
      const int qi = q - j;
      if (qi < 0) continue;
      const float prod = __fmul_rn(x[(b * L + qi) * C + c], w[(long)c * k + r + j * s]);
      acc = first ? prod : __fadd_rn(acc, prod);
      first = false;
    }
    y[e] = acc;
  }
}

// Up to two byte buffers copied in one launch: 16-byte vectors where the
// pointers allow, bytes otherwise.
struct CopyPair {
  const unsigned char* src[2];
  unsigned char* dst[2];
  long bytes[2];
  long vec[2];  // 16-byte vectors copied as such (the rest byte by byte)
};

__global__ __launch_bounds__(256) void copy_buffers_kernel(CopyPair a) {
  const long stride = (long)gridDim.x * 256, first = (long)blockIdx.x * 256 + threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint4* s = reinterpret_cast<const uint4*>(a.src[i]);
    uint4* d = reinterpret_cast<uint4*>(a.dst[i]);
    for (long e = first; e < a.vec[i]; e += stride) d[e] = s[e];
    for (long e = a.vec[i] * 16 + first; e < a.bytes[i]; e += stride) a.dst[i][e] = a.src[i][e];
  }
}

// Streaming convolution input: buf[b] = context[b] (pad rows) ++ x[b] (length
// rows), and the next context (buf's last pad rows) in the same pass.  A null
// context is a stream's start: zeros, or the first row repeated.  One launch
// per layer where concatenations and a crop took three (a streamed 80 ms chunk
// is bound by its launches: about 9 us of host time each).
template <typename V>
__global__ __launch_bounds__(256) void stream_append_kernel(const V* __restrict__ ctx, const V* __restrict__ x,
                                                            int pad, int length, int C, bool replicate, long total,
                                                            V* __restrict__ buf, V* __restrict__ next) {
  const long per = (long)(pad + length) * C;
  for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const long b = e / per;
    const long o = e - b * per;
    const int t = (int)(o / C), c = (int)(o - (long)t * C);
    V v{};
    if (t >= pad) v = x[(b * length + t - pad) * C + c];
    else if (ctx) v = ctx[(b * pad + t) * C + c];
    else if (replicate) v = x[b * length * C + c];
    buf[e] = v;
    if (t >= length) next[(b * pad + t - length) * C + c] = v;
  }
}

// Streaming attention operand: comb[b] = cached ++ new rows of (q | k | v)
// columns (q only in the new rows; nothing reads it in the cached ones), with
// the new rows from the chunk's projection, and the `keep` newest key / value
// rows as the next cache.  One launch per layer for two concatenations, two
// crops and three strided copies.
template <typename V>
__global__ __launch_bounds__(256) void kv_append_kernel(const V* __restrict__ qkv, const V* __restrict__ keys,
                                                        const V* __restrict__ values, int q_cols, int kv_cols,
                                                        int cached, int length, int keep, long total,
                                                        V* __restrict__ comb, V* __restrict__ next_keys,
                                                        V* __restrict__ next_values) {
  const int ld = q_cols + 2 * kv_cols, rows = cached + length;
  for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const long m = e / ld;
    const int c = (int)(e - m * ld);
    const long b = m / rows;
    const int t = (int)(m - b * rows);
    if (c < q_cols) {
      if (t >= cached) comb[e] = qkv[(b * length + t - cached) * ld + c];
      continue;
    }
    const bool is_v = c >= q_cols + kv_cols;
    const int kc = c - q_cols - (is_v ? kv_cols : 0);
    const V v = t >= cached ? qkv[(b * length + t - cached) * ld + c]
                            : (is_v ? values : keys)[(b * cached + t) * kv_cols + kc];
    comb[e] = v;
    const int kept = t - (rows - keep);
    if (kept >= 0) (is_v ? next_values : next_keys)[(b * keep + kept) * kv_cols + kc] = v;
  }
}

bool aligned16(std::initializer_list<const void*> ps) {
  uintptr_t u = 0;
  for (const void* p : ps) u |= reinterpret_cast<uintptr_t>(p);
  return (u & 15) == 0;
}

}  // namespace

extern "C" {

int fm_stream_append(const float* context, const float* x, int batch, int pad, int length, int channels,
                     int replicate, float* buf, float* next, hipStream_t stream) {
  if (!x || !buf || !next || batch < 0 || pad <= 0 || length <= 0 || channels <= 0) return FM_BAD_ARGUMENT;
  const int vec = channels % 4 == 0 && aligned16({context, x, buf, next}) ? 4 : 1;
  const long total = (long)batch * (pad + length) * (channels / vec);
  if (total == 0) return FM_OK;
  const dim3 grid((unsigned)std::min<long>((total + 255) / 256, 4096));
  if (vec == 4)
    hipLaunchKernelGGL((stream_append_kernel<floatx4>), grid, dim3(256), 0, stream,
                       reinterpret_cast<const floatx4*>(context), reinterpret_cast<const floatx4*>(x), pad, length,
                       channels / 4, replicate != 0, total, reinterpret_cast<floatx4*>(buf),
                       reinterpret_cast<floatx4*>(next));
  else
    hipLaunchKernelGGL((stream_append_kernel<float>), grid, dim3(256), 0, stream, context, x, pad, length, channels,
                       replicate != 0, total, buf, next);
  return (int)hipGetLastError();
}

int fm_kv_append(const float* qkv, int q_cols, int kv_cols, int batch, int length, const float* keys,
                 const float* values, int cached, int keep, float* comb, float* next_keys, float* next_values,
                 hipStream_t stream) {
  if (!qkv || !comb || batch < 0 || length <= 0 || q_cols < 0 || kv_cols <= 0 || cached < 0 || keep < 0 ||
      keep > cached + length || (cached > 0 && (!keys || !values)) || (keep > 0 && (!next_keys || !next_values)))
    return FM_BAD_ARGUMENT;
  const int vec = (q_cols | kv_cols) % 4 == 0 && aligned16({qkv, keys, values, comb, next_keys, next_values}) ? 4 : 1;
  const long total = (long)batch * (cached + length) * ((q_cols + 2 * kv_cols) / vec);
  if (total == 0) return FM_OK;
  const dim3 grid((unsigned)std::min<long>((total + 255) / 256, 4096));
  if (vec == 4)
    hipLaunchKernelGGL((kv_append_kernel<floatx4>), grid, dim3(256), 0, stream,
                       reinterpret_cast<const floatx4*>(qkv), reinterpret_cast<const floatx4*>(keys),
                       reinterpret_cast<const floatx4*>(values), q_cols / 4, kv_cols / 4, cached, length, keep, total,
                       reinterpret_cast<floatx4*>(comb), reinterpret_cast<floatx4*>(next_keys),
                       reinterpret_cast<floatx4*>(next_values));
  else
    hipLaunchKernelGGL((kv_append_kernel<float>), grid, dim3(256), 0, stream, qkv, keys, values, q_cols, kv_cols,
                       cached, length, keep, total, comb, next_keys, next_values);
  return (int)hipGetLastError();
}

int fm_copy_buffers(const void* src0, void* dst0, size_t bytes0, const void* src1, void* dst1,
                    size_t bytes1, hipStream_t stream) {
  if ((bytes0 && (!src0 || !dst0)) || (bytes1 && (!src1 || !dst1))) return FM_BAD_ARGUMENT;
  if ((long)bytes0 < 0 || (long)bytes1 < 0) return FM_BAD_ARGUMENT;
  CopyPair a{};
  const void* src[2] = {src0, src1};
  void* dst[2] = {dst0, dst1};
  const size_t bytes[2] = {bytes0, bytes1};
  long most = 0;
  for (int i = 0; i < 2; ++i) {
    a.src[i] = static_cast<const unsigned char*>(src[i]);
    a.dst[i] = static_cast<unsigned char*>(dst[i]);
    a.bytes[i] = bytes[i] ? (long)bytes[i] : 0;
    const bool aligned = ((reinterpret_cast<uintptr_t>(src[i]) | reinterpret_cast<uintptr_t>(dst[i])) & 15) == 0;
    a.vec[i] = aligned ? a.bytes[i] / 16 : 0;
    const long work = a.vec[i] + (a.bytes[i] - 16 * a.vec[i]);
    most = work > most ? work : most;
  }
  if (most == 0) return FM_OK;
  const long blocks = (most + 255) / 256;
  hipLaunchKernelGGL(copy_buffers_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(256), 0,
                     stream, a);
  return (int)hipGetLastError();
}

int fm_upsample_depthwise(const float* x, int batch, int length, int channels,
                          const float* weight, int kernel, int stride, float* y,
                          hipStream_t stream) {
  if (!x || !weight || !y || batch < 0 || length < 0 || channels <= 0 || stride <= 0 ||
      kernel <= 0 || kernel % stride)
    return FM_BAD_ARGUMENT;
  const long total = (long)batch * length * stride * channels;
  if (total == 0) return FM_OK;
  const long blocks = (total + 255) / 256;
  hipLaunchKernelGGL(upsample_depthwise_kernel, dim3((unsigned)(blocks < 65536 ? blocks : 65536)),
                     dim3(256), 0, stream, x, weight, batch, length, channels, kernel, stride, y);
  return (int)hipGetLastError();
}

// ABI version of this library (bumped when an entry point's contract changes).
int fm_abi_version(void) { return 1; }

}  // extern "C"
