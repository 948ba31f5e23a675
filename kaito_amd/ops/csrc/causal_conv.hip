// Depthwise causal short convolution over time with a carried tail, for
// batches of chunks (prompt portions and single decode tokens alike).
//
//   out[t, c] = act( bias[c] + sum_j w[c, j] * in(t - (taps-1-j), c) )
//
// where in(.) is the chunk's own rows, the sequence's last taps-1 inputs
// kept in its state slot for offsets before the chunk, and zero before
// the start of the sequence. The tail is advanced after every read of the
// old one.
//
// Bound by memory in prompts and by launches in decode steps. A thread owns
// 16 bytes of channels and walks rows with the last inputs in registers, so
// that every input is read once:
//   - prompts: CONV_ROWS rows per workgroup, the tail in a second launch
//     (8192 rows of 2048 channels, 4 taps: 136 us with one thread per output
//     and 2-byte loads, 35 now);
//   - decode steps: a sequence's row, then its tail, in one launch.
// Channels that 16 bytes do not divide, more than 4 taps, and prompts too small
// to hide a workgroup's walk of 16 rows: one thread per (row, channel).
#include "mix_common.h"

namespace kaito {

namespace {

template <typename T>
__global__ void causal_conv_out_kernel(
    T* __restrict__ out, const T* __restrict__ x, const int64_t x_stride,
    const float* __restrict__ w, const float* __restrict__ bias,
    const T* __restrict__ state, const int* __restrict__ cu,
    const int* __restrict__ slots, const int* __restrict__ starts,
    const int* __restrict__ token_seq, const int C, const int taps,
    const int tail, const int act) {
  const int t = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int b = token_seq[t];
  if (b < 0) return;
  const int slot = slots[b];
  if (slot < 0) return;
  const int r0 = cu[b];
  const int off = t - r0;
  const bool carried = starts[b] > 0;
  float acc = bias ? bias[c] : 0.0f;
  for (int j = 0; j < taps; j++) {
    const int o = off - (taps - 1 - j);
    float xv = 0.0f;
    if (o >= 0) {
      xv = act_ld(x + (int64_t)(r0 + o) * x_stride + c);
    } else if (carried) {
      // the tail keeps inputs at offsets -(taps-1) .. -1 in rows 0 .. taps-2
      xv = act_ld(state + ((int64_t)slot * tail + (taps - 1 + o)) * C + c);
    }
    acc += w[c * taps + j] * xv;
  }
  if (act == 1) acc = silu_f(acc);
  act_st(out + (int64_t)t * C + c, acc);
}

template <typename T>
__global__ void causal_conv_tail_kernel(
    const T* __restrict__ x, const int64_t x_stride, T* __restrict__ state,
    const int* __restrict__ cu, const int* __restrict__ slots,
    const int* __restrict__ starts, const int C, const int taps,
    const int tail) {
  const int b = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int slot = slots[b];
  const int r0 = cu[b];
  const int n = cu[b + 1] - r0;
  if (slot < 0 || n <= 0) return;
  const bool carried = starts[b] > 0;
  T* st = state + (int64_t)slot * tail * C + c;
  // ascending s reads row s+n (> s) of the old tail before it is overwritten
  for (int s = 0; s < taps - 1; s++) {
    const int o = n - (taps - 1) + s;
    float v = 0.0f;
    if (o >= 0) v = act_ld(x + (int64_t)(r0 + o) * x_stride + c);
    else if (carried) v = act_ld(st + (int64_t)(taps - 1 + o) * C);
    act_st(st + (int64_t)s * C, v);
  }
}

constexpr int CONV_ROWS = 16;       // per workgroup
constexpr int AHEAD = 4;            // rows whose loads are under way at once

// VEC channels of a row
template <typename T, int VEC>
KAITO_DEV void ld_vec(const T* p, float* v) {
#pragma unroll
  for (int i = 0; i < VEC; i += 4) {
    const float4_t x = act_ld4(p + i);
#pragma unroll
    for (int e = 0; e < 4; e++) v[i + e] = x[e];
  }
}

template <typename T, int VEC>
KAITO_DEV void st_vec(T* p, const float* v) {
#pragma unroll
  for (int i = 0; i < VEC; i += 4)
    act_st4(p + i, float4_t{v[i], v[i + 1], v[i + 2], v[i + 3]});
}

// WHOLE: workgroup per chunk, which also advances the tail; otherwise
// workgroup per CONV_ROWS rows
template <typename T, int TAPS, bool WHOLE>
__global__ __launch_bounds__(256)
void causal_conv_rows_kernel(
    T* __restrict__ out, const T* __restrict__ x, const int64_t x_stride,
    const float* __restrict__ w, const float* __restrict__ bias,
    T* __restrict__ state, const int* __restrict__ cu,
    const int* __restrict__ slots, const int* __restrict__ starts,
    const int* __restrict__ token_seq, const int T_total, const int C,
    const int tail, const int act) {
  constexpr int VEC = 16 / sizeof(T), LAST = TAPS - 1;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * VEC;
  if (c >= C) return;
  const int t0 = WHOLE ? cu[blockIdx.x] : blockIdx.x * CONV_ROWS;
  const int t1 = WHOLE ? cu[blockIdx.x + 1] : min(T_total, t0 + CONV_ROWS);
  if (t0 >= t1 || (WHOLE && slots[blockIdx.x] < 0)) return;

  float wt[VEC][TAPS], bs[VEC];
#pragma unroll
  for (int e = 0; e < VEC; e++) {
    bs[e] = bias ? bias[c + e] : 0.0f;
#pragma unroll
    for (int j = 0; j < TAPS; j++) wt[e][j] = w[(c + e) * TAPS + j];
  }
  // win[j]: input LAST - j rows before the next one
  float win[LAST > 0 ? LAST : 1][VEC];
  int seq = -1, slot = -1;
  T* st = nullptr;
  for (int tb = t0; tb < t1; tb += AHEAD) {
    float in[AHEAD][VEC];
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
      ld_vec<T, VEC>(x + (int64_t)min(tb + i, t1 - 1) * x_stride + c, in[i]);
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      const int t = tb + i;
      if (t >= t1) break;
      const int b = WHOLE ? (int)blockIdx.x : token_seq[t];
      if (b != seq) {                         // uniform
        seq = b;
        slot = b < 0 ? -1 : slots[b];
        if (slot >= 0) {
          const int off = t - cu[b];
          const bool carried = starts[b] > 0;
          st = state + (int64_t)slot * tail * C + c;
#pragma unroll
          for (int j = 0; j < LAST; j++) {
            const int o = off - LAST + j;
            if (o >= 0) {
              ld_vec<T, VEC>(x + (int64_t)(t - LAST + j) * x_stride + c, win[j]);
            } else if (carried) {
              ld_vec<T, VEC>(st + (int64_t)(LAST + o) * C, win[j]);
            } else {
#pragma unroll
              for (int e = 0; e < VEC; e++) win[j][e] = 0.0f;
            }
          }
        }
      }
      if (slot < 0) continue;
      float acc[VEC];
#pragma unroll
      for (int e = 0; e < VEC; e++) {
        acc[e] = bs[e];
#pragma unroll
        for (int j = 0; j < LAST; j++) acc[e] += wt[e][j] * win[j][e];
        acc[e] += wt[e][LAST] * in[i][e];
        if (act == 1) acc[e] = silu_f(acc[e]);
#pragma unroll
        for (int j = 0; j + 1 < LAST; j++) win[j][e] = win[j + 1][e];
        if constexpr (LAST > 0) win[LAST - 1][e] = in[i][e];
      }
      st_vec<T, VEC>(out + (int64_t)t * C + c, acc);
    }
  }
  if constexpr (WHOLE) {
#pragma unroll
    for (int j = 0; j < LAST; j++) st_vec<T, VEC>(st + (int64_t)j * C, win[j]);
  }
}

}  // namespace

void causal_conv_update(at::Tensor out, at::Tensor x, at::Tensor weight,
                        at::Tensor bias, at::Tensor conv_state,
                        at::Tensor cu_seqlens, at::Tensor state_slots,
                        at::Tensor seq_starts, at::Tensor token_seq,
                        int64_t act) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1);
  TORCH_CHECK(out.is_contiguous() && out.sizes() == x.sizes() &&
              out.dtype() == x.dtype());
  const int T = x.size(0), C = x.size(1);
  KAITO_CHECK_F32(weight);
  TORCH_CHECK(weight.dim() == 2 && weight.size(0) == C);
  const int taps = weight.size(1);
  TORCH_CHECK(taps >= 1);
  const bool has_bias = bias.numel() > 0;
  if (has_bias) { KAITO_CHECK_F32(bias); TORCH_CHECK(bias.numel() == C); }
  TORCH_CHECK(conv_state.is_contiguous() && conv_state.dim() == 3 &&
              conv_state.dtype() == x.dtype() && conv_state.size(2) == C &&
              conv_state.size(1) >= std::max(taps - 1, 1));
  const int tail = conv_state.size(1);
  KAITO_CHECK_I32(cu_seqlens); KAITO_CHECK_I32(state_slots);
  KAITO_CHECK_I32(seq_starts); KAITO_CHECK_I32(token_seq);
  const int B = state_slots.size(0);
  TORCH_CHECK(cu_seqlens.size(0) == B + 1 && seq_starts.size(0) == B &&
              token_seq.size(0) == T);
  if (T == 0 || B == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  const int threads = 256;
  const dim3 gc((C + threads - 1) / threads);
  auto wide = [](const at::Tensor& t) {
    return (uintptr_t)t.data_ptr() % 16 == 0;
  };
  const int vec = 16 / x.element_size();
  const bool whole = T <= B;        // a row per sequence: one launch
  // The walk takes 19 us (bf16) or 12 (f32) however short the prompt, a thread
  // per output 6 us and more with its size (4 taps; 200 x 2048 bf16: 18.9, 6.9;
  // 500 x 6144: 19.7, 22.6; 2000 x 1024: 18.9, 14.5; 2000 x 2048: 21.1, 31.4; f32,
  // 500 x 2048: 13.0, 10.3; 1000 x 2048: 14.0, 17.1).
  const int64_t least = x.element_size() == 2 ? 11ll << 18 : 3ll << 19;
  const bool rows = C % vec == 0 && x.stride(0) % vec == 0 && taps <= 4 &&
      wide(x) && wide(out) && wide(conv_state) &&
      (whole || (int64_t)T * C >= least);
  if (rows) {
    // threads for the channels there are
    const int lanes = C / vec;
    const int block = lanes >= 256 ? 256 : (lanes + 63) / 64 * 64;
    const dim3 grid(whole ? B : (T + CONV_ROWS - 1) / CONV_ROWS,
                    (lanes + block - 1) / block);
#define CONV_ROWS_LAUNCH(TAPS_, WHOLE_)                                       \
      hipLaunchKernelGGL((causal_conv_rows_kernel<act_t, TAPS_, WHOLE_>),     \
          grid, dim3(block), 0, stream, (act_t*)out.data_ptr(),               \
          (const act_t*)x.data_ptr(), x.stride(0), weight.data_ptr<float>(),  \
          has_bias ? bias.data_ptr<float>() : nullptr,                        \
          (act_t*)conv_state.data_ptr(), cu_seqlens.data_ptr<int>(),          \
          state_slots.data_ptr<int>(), seq_starts.data_ptr<int>(),            \
          token_seq.data_ptr<int>(), T, C, tail, (int)act)
#define CONV_TAPS(TAPS_)                                                      \
      if (taps == TAPS_) {                                                    \
        if (whole) { CONV_ROWS_LAUNCH(TAPS_, true); }                         \
        else { CONV_ROWS_LAUNCH(TAPS_, false); }                              \
      }
    KAITO_DISPATCH_ACT(x, {
      CONV_TAPS(1) CONV_TAPS(2) CONV_TAPS(3) CONV_TAPS(4)
    });
#undef CONV_TAPS
#undef CONV_ROWS_LAUNCH
    if (whole || taps == 1) return;
  }
  KAITO_DISPATCH_ACT(x, {
    if (!rows) {
      hipLaunchKernelGGL((causal_conv_out_kernel<act_t>),
          dim3(T, gc.x), dim3(threads), 0, stream,
          (act_t*)out.data_ptr(), (const act_t*)x.data_ptr(), x.stride(0),
          weight.data_ptr<float>(),
          has_bias ? bias.data_ptr<float>() : nullptr,
          (const act_t*)conv_state.data_ptr(), cu_seqlens.data_ptr<int>(),
          state_slots.data_ptr<int>(), seq_starts.data_ptr<int>(),
          token_seq.data_ptr<int>(), C, taps, tail, (int)act);
    }
    if (taps > 1) {
      hipLaunchKernelGGL((causal_conv_tail_kernel<act_t>),
          dim3(B, gc.x), dim3(threads), 0, stream,
          (const act_t*)x.data_ptr(), x.stride(0),
          (act_t*)conv_state.data_ptr(), cu_seqlens.data_ptr<int>(),
          state_slots.data_ptr<int>(), seq_starts.data_ptr<int>(), C, taps,
          tail);
    }
  });
}

}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("causal_conv_update(Tensor(a!) out, Tensor x, Tensor weight, Tensor bias, Tensor(b!) conv_state, Tensor cu_seqlens, Tensor state_slots, Tensor seq_starts, Tensor token_seq, int act) -> ()");
}
TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("causal_conv_update", &kaito::causal_conv_update);
}
