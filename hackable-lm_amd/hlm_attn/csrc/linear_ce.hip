// Cross-entropy rows of the LM head's fused linear + cross-entropy: for each
// row of logits x (V values) and its target t,
//   lse     = log sum_j exp(x_j)
//   loss    = (lse - x_t) / n_tokens
//   x_j    <- (exp(x_j - lse) - [j == t]) / n_tokens      (in place)
// i.e. the per-row loss and the gradient of the mean loss with respect to the
// logits, which the caller multiplies into the two GEMMs of the backward.
// This is hackable-lm's Triton _linear_ce_kernel (kernels.py:286-316, op
// :320-336), computed in fp32 from bf16 or fp32 logits.  A target equal to
// ignore_index (-100, F.cross_entropy's default, as the torch path of
// model.py:333-341 uses) contributes a zero loss and a zero gradient row; any
// other target outside [0, V) yields NaN for the row's loss and gradient (the
// kernel cannot raise).
//
// Memory-bound: one workgroup per row.  The row is read once into registers in
// the aligned 16-byte chunks that hold it (chunk k of thread i is the row's
// chunk i + 256 k), reduced (max, then sum of exponentials) with wave shuffles
// and one LDS exchange between the 4 waves, and written once: 2 * V * sizeof(T)
// bytes per row.  A row may begin and end inside a chunk (V or the row stride
// no multiple of 16 / sizeof(T)): the elements of a chunk that are not the
// row's read as -inf, which neither the maximum nor the sum sees, and are not
// written.  4096 rows of V = 50257 bf16 at a row stride of 50257: 529 us when
// such rows were read three times, one element per lane; 169 us now (4.9 TB/s).  Rows
// of more than 32 chunks per thread (V above 65536 bf16 or 32768 fp32; rows
// that are not aligned, above 65529 or 32765) keep that path.
#include "attn_common.h"

namespace hlm {

struct CeArgs {
  void* logits;            // (n_rows, >= V) rows at row_stride elements
  int64_t row_stride;
  const int64_t* targets;  // n_rows
  float* loss;             // n_rows
  int n_rows, V;
  float inv_n;             // 1 / n_tokens
  int ignore_index;
};

template <typename T>
__device__ __forceinline__ float to_f32(T x) {
  return (float)x;
}

// Block-wide reductions over 256 threads (4 waves): every thread gets the result.
__device__ __forceinline__ float block_max(float v, float* red) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m));
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  v = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  return v;
}

__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  v = (red[0] + red[1]) + (red[2] + red[3]);
  __syncthreads();
  return v;
}

// Row status from its target: 0 = valid, 1 = ignored, 2 = out of range.
__device__ __forceinline__ int target_status(int64_t t, int V, int ignore_index) {
  if (t >= 0 && t < V) return 0;
  return t == ignore_index ? 1 : 2;
}

// ALIGNED: every row begins and ends on a 16-byte boundary.
template <typename T, int K, bool ALIGNED>
__global__ __launch_bounds__(256) void ce_rows_vec_kernel(CeArgs a) {
  constexpr int E = 16 / sizeof(T);  // elements per 16-byte chunk
  // LEAN: one buffer resource and offset register for all chunks, and nothing
  // derived from a chunk is kept over the reductions (they cost 11 VGPRs a
  // chunk otherwise: one wave per SIMD from K = 24 on).  4096 rows of bf16, us
  // without / with: V = 65536 273 / 213, V = 50264 216 / 167, V = 50257
  // (unaligned) 231 / 169, V = 16381 64.5 / 52.5.  Aligned rows of up to 16
  // chunks run best without, at two waves per SIMD: V = 32768 95 / 108.
  constexpr bool LEAN = !ALIGNED || K > 16;
  typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
  __shared__ float red[4];
  const int row = blockIdx.x, tid = threadIdx.x;
  T* base = static_cast<T*>(a.logits) + (int64_t)row * a.row_stride;
  const int V = a.V;
  const int64_t tgt = a.targets[row];
  const int status = target_status(tgt, V, a.ignore_index);
  // The row's elements are E * chunk - lead + e, 0 <= lead < E.
  const int lead = ALIGNED ? 0 : (int)((reinterpret_cast<uintptr_t>(base) & 15u) / sizeof(T));
  auto first_of = [&](int k) __attribute__((always_inline)) { return E * (tid + 256 * k) - lead; };
  // Buffer over the row from its first chunk to its last 4 bytes (reads past
  // them return zeros).
  [[maybe_unused]] const __amdgpu_buffer_rsrc_t chunks =
      bytes_rsrc(base - lead, ((V + lead) * (int)sizeof(T) + 3) & ~3);
  // The target's logit, read before any thread of the block stores (the
  // stores follow two block barriers).
  float xt = 0.f;
  if (tid == 0 && status == 0) xt = to_f32(base[tgt]);

  u32x4 raw[K];
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int idx = first_of(k);
    raw[k] = u32x4{};
    if (idx >= V) continue;
    if constexpr (LEAN)
      raw[k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(chunks, 16 * tid, 4096 * k, 0));
    else
      raw[k] = *reinterpret_cast<const u32x4*>(base + idx);
  }
  if constexpr (!ALIGNED) {
    // The first chunk and the one that holds the row's end: what is not the
    // row's (a neighbouring row's elements, possibly being written) goes out.
    auto trim = [&](u32x4& w, int idx) __attribute__((always_inline)) {
      T* v = reinterpret_cast<T*>(&w);
#pragma unroll
      for (int e = 0; e < E; ++e)
        if ((unsigned)(idx + e) >= (unsigned)V) v[e] = (T)-INFINITY;
    };
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int idx = first_of(k);
      if (idx < 0 || (idx < V && idx + E > V)) trim(raw[k], idx);
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (first_of(k) >= V) continue;
    const T* v = reinterpret_cast<const T*>(&raw[k]);
#pragma unroll
    for (int e = 0; e < E; ++e) m = fmaxf(m, to_f32(v[e]));
  }
  if constexpr (LEAN) {
#pragma unroll
    for (int k = 0; k < K; ++k) asm volatile("" : "+v"(raw[k]));
  }
  const float M = block_max(m, red);
  const float c = M * kLog2e;
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (first_of(k) >= V) continue;
    const T* v = reinterpret_cast<const T*>(&raw[k]);
#pragma unroll
    for (int e = 0; e < E; ++e) s += fast_exp2(fmaf(to_f32(v[e]), kLog2e, -c));
  }
  if constexpr (LEAN) {
#pragma unroll
    for (int k = 0; k < K; ++k) asm volatile("" : "+v"(raw[k]));
  }
  const float S = block_sum(s, red);
  const float lse = M + __log2f(S) * kLn2;
  if (tid == 0) a.loss[row] = status == 0 ? (lse - xt) * a.inv_n : status == 1 ? 0.f : NAN;
  // gradient: (p_j - [j == t]) / n, p_j = 2^(x_j log2e - c) / S
  const float scale = status == 0 ? a.inv_n / S : status == 1 ? 0.f : NAN;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int idx = first_of(k);
    if (idx >= V) continue;
    const T* v = reinterpret_cast<const T*>(&raw[k]);
    u32x4 outw;
    T* o = reinterpret_cast<T*>(&outw);
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] = (T)(fast_exp2(fmaf(to_f32(v[e]), kLog2e, -c)) * scale);
    // The target's gradient, p_t / S - 1 / n, rounded once as above: one test
    // per chunk instead of one per element (the lane holding the target redoes
    // its element; the others skip the branch).
    if (status == 0 && (uint64_t)(tgt - idx) < (uint64_t)E) {
      const int et = (int)(tgt - idx);
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (e == et) o[e] = (T)(fast_exp2(fmaf(to_f32(v[e]), kLog2e, -c)) * scale - a.inv_n);
    }
    if (ALIGNED || (idx >= 0 && idx + E <= V)) {
      if constexpr (LEAN)
        __builtin_amdgcn_raw_buffer_store_b128(outw, chunks, 16 * tid, 4096 * k, 0);
      else
        *reinterpret_cast<u32x4*>(base + idx) = outw;
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if ((unsigned)(idx + e) < (unsigned)V) base[idx + e] = o[e];
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void ce_rows_generic_kernel(CeArgs a) {
  __shared__ float red[4];
  const int row = blockIdx.x, tid = threadIdx.x;
  T* base = static_cast<T*>(a.logits) + (int64_t)row * a.row_stride;
  const int V = a.V;
  const int64_t tgt = a.targets[row];
  const int status = target_status(tgt, V, a.ignore_index);
  float xt = 0.f;
  if (tid == 0 && status == 0) xt = to_f32(base[tgt]);
  float m = -INFINITY;
  for (int j = tid; j < V; j += 256) m = fmaxf(m, to_f32(base[j]));
  const float M = block_max(m, red);
  const float c = M * kLog2e;
  float s = 0.f;
  for (int j = tid; j < V; j += 256) s += fast_exp2(fmaf(to_f32(base[j]), kLog2e, -c));
  const float S = block_sum(s, red);  // its barriers order every read above before the stores below
  const float lse = M + __log2f(S) * kLn2;
  if (tid == 0) a.loss[row] = status == 0 ? (lse - xt) * a.inv_n : status == 1 ? 0.f : NAN;
  const float scale = status == 0 ? a.inv_n / S : status == 1 ? 0.f : NAN;
  for (int j = tid; j < V; j += 256) {
    float g = fast_exp2(fmaf(to_f32(base[j]), kLog2e, -c)) * scale;
    if (status == 0 && j == tgt) g -= a.inv_n;
    base[j] = (T)g;
  }
}

template <typename T, int K>
void launch_ce_rows_vec(const CeArgs& a, bool aligned, hipStream_t stream) {
  const dim3 grid((unsigned)a.n_rows), block(256);
  if (aligned)
    hipLaunchKernelGGL((ce_rows_vec_kernel<T, K, true>), grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL((ce_rows_vec_kernel<T, K, false>), grid, block, 0, stream, a);
}

template <typename T>
hipError_t launch_ce_rows_typed(const CeArgs& a, hipStream_t stream) {
  constexpr int E = 16 / sizeof(T);
  const bool aligned = (reinterpret_cast<uintptr_t>(a.logits) & 15u) == 0 && a.V % E == 0 && a.row_stride % E == 0;
  // 16-byte chunks per thread; a row that is not aligned may reach into one more.
  const int chunks = (int)(((int64_t)a.V + (aligned ? 0 : E - 1) + 256 * E - 1) / (256 * E));
  if (chunks <= 1)
    launch_ce_rows_vec<T, 1>(a, aligned, stream);
  else if (chunks <= 2)
    launch_ce_rows_vec<T, 2>(a, aligned, stream);
  else if (chunks <= 4)
    launch_ce_rows_vec<T, 4>(a, aligned, stream);
  else if (chunks <= 8)
    launch_ce_rows_vec<T, 8>(a, aligned, stream);
  else if (chunks <= 16)
    launch_ce_rows_vec<T, 16>(a, aligned, stream);
  else if (chunks <= 20)
    launch_ce_rows_vec<T, 20>(a, aligned, stream);
  else if (chunks <= 24)
    launch_ce_rows_vec<T, 24>(a, aligned, stream);
  else if (chunks <= 28)
    launch_ce_rows_vec<T, 28>(a, aligned, stream);
  else if (chunks <= 32)
    launch_ce_rows_vec<T, 32>(a, aligned, stream);
  else
    hipLaunchKernelGGL((ce_rows_generic_kernel<T>), dim3((unsigned)a.n_rows), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_ce_rows(void* logits, bool bf16_logits, int64_t row_stride, const int64_t* targets, float* loss,
                          int n_rows, int V, float inv_n, int ignore_index, hipStream_t stream) {
  CeArgs a{logits, row_stride, targets, loss, n_rows, V, inv_n, ignore_index};
  if (n_rows == 0) return hipSuccess;
  return bf16_logits ? launch_ce_rows_typed<bf16>(a, stream) : launch_ce_rows_typed<float>(a, stream);
}

}  // namespace hlm
