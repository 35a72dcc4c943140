// Row softmax over the last dimension for gfx950 (reference.py:14-17).
//
// HBM-bound: each row is read once into registers, reduced for its max and
// for sum(exp(x - max)) in fp32 with wave64 DPP reductions, then normalised
// and written once, with nontemporal accesses. Rows of up to 128 16-byte
// vectors are owned by one wave (no barriers), wider rows by up to 1024
// threads holding two to four vectors each (up to 16 past 4096 vectors). Rows are
// indexed with 64-bit arithmetic and walked by grid stride on a capped grid,
// so every row is written whatever the row count.
//
// -inf logits give exp2(-inf) = 0 exactly; a row with a single finite entry
// returns exactly 1.0 there. The file is built without fast-math so those
// IEEE special cases are honoured.
#include "ak_common.h"

namespace ak {
namespace {

// TPR threads own a row (TPR / 64 waves; 256 / TPR rows per workgroup when
// TPR < 256); rows are walked with a workgroup-uniform grid stride so the
// cross-wave reductions' barriers are reached by every wave.
//
// RAG: rows at any address and of any width (an odd vocabulary, an odd number
// of tokens). The vectors start at the row's first 16-byte boundary and the
// few elements before the first and behind the last one go one to a thread,
// so the row still crosses HBM once, in whole vectors. [4096, 50257] fp16:
// 152 us, 5.4 TB/s, as a copy runs here (523 us with element accesses and two
// passes); [98304, 777] fp16 56.7 us, 5.4 TB/s.
//
// PACKED, from 4 vectors a thread on: the row stays packed between
// the passes and exp(x - max) is formed twice: 32 registers for 8 vectors
// instead of 64, so two 1024-thread workgroups fit a CU and one's loads run
// under the other's arithmetic ([4096, 50256] fp16: 179 -> 151 us). Rows too few
// for that keep their exponentials ([8, 32000] bf16: 4.9 us, packed 5.7).
template <typename T, int VPT, int TPR, bool RAG, bool PACKED>
__global__ void __launch_bounds__(TPR >= 256 ? TPR : 256, VPT == 8 && PACKED ? 8 : 1)
softmax_vec_kernel(const T* __restrict__ x, T* __restrict__ y, int64_t rows, int cols,
                   int64_t ld_x, int64_t ld_y) {
  constexpr int VE = Vec16<T>::VE;
  constexpr int RPW = TPR >= 256 ? 1 : 256 / TPR;
  constexpr int WPR = TPR / 64;
  static_assert(TPR % 64 == 0, "rows are owned by whole waves");
  __shared__ float part[RPW][WPR];
  const int t = threadIdx.x % TPR;
  const int rl = threadIdx.x / TPR;

  for (int64_t base = (int64_t)blockIdx.x * RPW; base < rows; base += (int64_t)gridDim.x * RPW) {
    const int64_t row = RPW == 1 ? base : base + rl;
    const bool live = RPW == 1 || row < rows;
    const T* xr = x + row * ld_x;
    int head = 0, nvec = cols / VE, ex = -1;  // ex: this thread's single element, if any
    if constexpr (RAG) {
      const RowSplit<T> sp(xr, cols);
      head = sp.head;
      nvec = sp.nvec;
      if (live && t < sp.nx) ex = sp.extra(t);
    }
    if (!live) nvec = 0;  // a row slot past the last row touches nothing
    Vec16<T> raw[PACKED ? VPT : 1];
    float v[PACKED ? 1 : VPT][VE];
    float xe = -INFINITY;
    float m = -INFINITY;
    // vector t + k TPR, from a workgroup-uniform address and one lane offset
    const unsigned to = t * VE;
    auto ld = [&](int k) {
      const T* xk = xr + head + k * TPR * VE;
      return RAG ? load16_any_nt(xk + to) : load16_nt(xk + to);
    };
    if constexpr (PACKED) {
#pragma unroll
      for (int k = 0; k < VPT; ++k) {  // vectors past the row stay -inf
        raw[k].u = vec_neg_inf<T>();
        if (t + k * TPR < nvec) raw[k] = ld(k);
      }
    } else {
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
        if (t + k * TPR < nvec) {
          const Vec16<T> xv = ld(k);
#pragma unroll
          for (int e = 0; e < VE; ++e) {
            v[k][e] = to_f32(xv.e[e]);
            m = fmaxf(m, v[k][e]);
          }
        }
      }
    }
    if constexpr (RAG) {
      if (ex >= 0) m = fmaxf(m, xe = to_f32(xr[ex]));
    }
    if constexpr (PACKED) {
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
#pragma unroll
        for (int e = 0; e < VE; ++e) m = fmaxf(m, to_f32(raw[k].e[e]));
        keep_packed(raw[k]);
      }
    }
    m = wave_max(m);
    if constexpr (WPR > 1) {
      if ((threadIdx.x & 63) == 0) part[rl][t / 64] = m;
      __syncthreads();
      m = part[rl][0];
#pragma unroll
      for (int i = 1; i < WPR; ++i) m = fmaxf(m, part[rl][i]);
      __syncthreads();
    }

    // exp(x - m): the max element gives exp2(0) = 1 exactly.
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      if constexpr (PACKED) {
#pragma unroll
        for (int e = 0; e < VE; ++e) s += fast_exp(to_f32(raw[k].e[e]) - m);
        keep_packed(raw[k]);
      } else if (t + k * TPR < nvec) {
#pragma unroll
        for (int e = 0; e < VE; ++e) {
          v[k][e] = fast_exp(v[k][e] - m);
          s += v[k][e];
        }
      }
    }
    if constexpr (RAG) {
      if (ex >= 0) s += (xe = fast_exp(xe - m));
    }
    s = wave_sum(s);
    if constexpr (WPR > 1) {
      if ((threadIdx.x & 63) == 0) part[rl][t / 64] = s;
      __syncthreads();
      s = 0.0f;
#pragma unroll
      for (int i = 0; i < WPR; ++i) s += part[rl][i];
      __syncthreads();
    }
    const float inv = 1.0f / s;

    T* yr = y + row * ld_y;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int c = t + k * TPR;
      if (c < nvec) {
        Vec16<T> o;
#pragma unroll
        for (int e = 0; e < VE; ++e) {
          if constexpr (PACKED) o.e[e] = from_f32<T>(fast_exp(to_f32(raw[k].e[e]) - m) * inv);
          else o.e[e] = from_f32<T>(v[k][e] * inv);
        }
        T* yk = yr + head + k * TPR * VE;
        if constexpr (RAG) store16_any_nt(yk + to, o);
        else store16_nt(yk + to, o);
      }
    }
    if constexpr (RAG) {
      if (ex >= 0) yr[ex] = from_f32<T>(xe * inv);
    }
  }
}

// Online (max, sum) state: sum is relative to max.
struct MaxSum {
  float m, s;
};

__device__ __forceinline__ MaxSum combine(MaxSum a, MaxSum b) {
  const float m = fmaxf(a.m, b.m);
  if (m == -INFINITY) return {m, 0.0f};
  const float sa = a.m == -INFINITY ? 0.0f : a.s * fast_exp(a.m - m);
  const float sb = b.m == -INFINITY ? 0.0f : b.s * fast_exp(b.m - m);
  return {m, sa + sb};
}

// Rows of more than 16384 vectors: a 256-thread workgroup per row (rows
// by grid stride), two passes over global memory (online max/sum, then
// normalise).
template <typename T>
__device__ void softmax_generic_row(const T* __restrict__ xr, T* __restrict__ yr, int cols,
                                    MaxSum* part) {
  MaxSum st{-INFINITY, 0.0f};
  for (int c = threadIdx.x; c < cols; c += 256) {
    const float v = to_f32(xr[c]);
    if (v > st.m) {
      // exp(v - v) is 1, or NaN for v = +inf, as in the reference op.
      st.s = st.s * fast_exp(st.m - v) + fast_exp(v - v);
      st.m = v;
    } else if (v != v) {
      st = {v, v};  // NaN poisons the row
    } else if (v != -INFINITY) {
      st.s += fast_exp(v - st.m);
    }
  }
  // wave-level combine through shuffles
  for (int off = 1; off < 64; off <<= 1) {
    MaxSum o{__shfl_xor(st.m, off, 64), __shfl_xor(st.s, off, 64)};
    st = (st.m != st.m || o.m != o.m) ? MaxSum{NAN, NAN} : combine(st, o);
  }
  if ((threadIdx.x & 63) == 0) part[threadIdx.x / 64] = st;
  __syncthreads();
  st = part[0];
  for (int i = 1; i < 4; ++i) {
    st = (st.m != st.m || part[i].m != part[i].m) ? MaxSum{NAN, NAN} : combine(st, part[i]);
  }
  __syncthreads();  // part is rewritten for the next row
  const float inv = 1.0f / st.s;
  for (int c = threadIdx.x; c < cols; c += 256) {
    yr[c] = from_f32<T>(fast_exp(to_f32(xr[c]) - st.m) * inv);
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
softmax_generic_kernel(const T* __restrict__ x, T* __restrict__ y, int64_t rows, int cols,
                       int64_t ld_x, int64_t ld_y) {
  __shared__ MaxSum part[4];
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    softmax_generic_row(x + row * ld_x, y + row * ld_y, cols, part);
  }
}

template <typename T, int VPT, int TPR>
void launch_vec(bool aligned, const T* x, T* y, int64_t rows, int cols, int64_t ld_x, int64_t ld_y,
                hipStream_t s) {
  constexpr int RPW = TPR >= 256 ? 1 : 256 / TPR;
  const dim3 grid(row_grid((rows + RPW - 1) / RPW)), block(TPR * RPW);
  if (aligned)
    softmax_vec_kernel<T, VPT, TPR, false, (VPT >= 4)><<<grid, block, 0, s>>>(x, y, rows, cols, ld_x, ld_y);
  else
    softmax_vec_kernel<T, VPT, TPR, true, (VPT >= 4)><<<grid, block, 0, s>>>(x, y, rows, cols, ld_x, ld_y);
}

// Few aligned rows: most threads a row, what each holds converted once.
template <typename T, int VPT, int TPR>
void launch_few(const T* x, T* y, int64_t rows, int cols, int64_t ld_x, int64_t ld_y, hipStream_t s) {
  softmax_vec_kernel<T, VPT, TPR, false, false><<<dim3(row_grid(rows)), dim3(TPR), 0, s>>>(x, y, rows, cols, ld_x, ld_y);
}

template <typename T>
int dispatch(const void* xv, void* yv, int64_t rows, int64_t cols, int64_t ld_x, int64_t ld_y,
             hipStream_t s) {
  const T* x = static_cast<const T*>(xv);
  T* y = static_cast<T*>(yv);
  constexpr int VE = Vec16<T>::VE;
  const bool aligned = cols % VE == 0 && ld_x % VE == 0 && ld_y % VE == 0 && aligned16(x) &&
                       aligned16(y);
  const int64_t nvec = cols / VE;
  const int c = (int)cols;
#define AK_LAUNCH(VPT, TPR) launch_vec<T, VPT, TPR>(aligned, x, y, rows, c, ld_x, ld_y, s)
  // Two 16-byte vectors a thread (four in rows off the 16-byte grid and in narrow
  // fp32 rows) past one wave's 128: with one a thread, half of a workgroup's time
  // went to its reductions. [16384, 8192] bf16 103 -> 84 us, [24000, 3001] fp16
  // 68.9 -> 49.4, [32768, 777] fp32 47.8 -> 36.8, [8192, 4097] fp32 59.6 -> 46.4.
  // Up to about one workgroup a SIMD the latency of one row counts: one vector a
  // thread (two and four past 1024 and 2048), unpacked. us, so and as below: [1536,
  // 2048] bf16 3.8 and 4.3 ([3072, 2048] 7.0 and 5.3), [512, 1536] fp32 3.5 and 3.6,
  // [64, 16384] bf16 4.1 and 4.4, [512, 32000] 11.3 and 12.0, [8, 65536] 7.1 and 8.9
  // ([64, 65536] 10.9 and 10.5).
  auto few = [&](int64_t most) { return aligned && rows <= most; };
#define AK_FEW(VPT, TPR) launch_few<T, VPT, TPR>(x, y, rows, c, ld_x, ld_y, s)
  if (nvec <= 64) AK_LAUNCH(1, 64);
  else if (nvec <= 128) AK_LAUNCH(2, 64);
  else if (nvec <= 256 && few(VE == 8 ? 2048 : 256)) AK_FEW(1, 256);
  else if (nvec > 256 && nvec <= 512 && few(512)) AK_FEW(1, 512);
  else if (nvec > 1024 && nvec <= 2048 && few(512)) AK_FEW(2, 1024);
  else if (nvec > 2048 && nvec <= 4096 && few(512)) AK_FEW(4, 1024);
  else if (nvec > 4096 && nvec <= 8192 && few(32)) AK_FEW(8, 1024);
  else if (nvec <= 256) {
    if (VE == 4) AK_LAUNCH(4, 64);
    else AK_LAUNCH(2, 128);
  } else if (nvec <= 512) {
    if (aligned) AK_LAUNCH(2, 256);
    else AK_LAUNCH(4, 128);
  } else if (nvec <= 1024) {
    if (aligned) AK_LAUNCH(2, 512);
    else AK_LAUNCH(4, 256);
  } else if (nvec <= 2048) AK_LAUNCH(4, 512);
  else if (nvec <= 4096) AK_LAUNCH(4, 1024);
  else if (nvec <= 8192) AK_LAUNCH(8, 1024);
  else if (nvec <= 16384) AK_LAUNCH(16, 1024);
  else softmax_generic_kernel<T><<<dim3(row_grid(rows)), dim3(256), 0, s>>>(x, y, rows, c, ld_x, ld_y);
#undef AK_FEW
#undef AK_LAUNCH
  return ak_check_launch("ak_softmax_fwd");
}

}  // namespace
}  // namespace ak

extern "C" int ak_softmax_fwd(const void* x, void* y, int64_t rows, int64_t cols, int64_t ld_x,
                              int64_t ld_y, int dtype, void* stream) {
  const char* name = "ak_softmax_fwd";
  if (ak_dtype_size(dtype) == 0) return ak_set_error(AK_ERR_UNSUPPORTED, "%s: unsupported dtype code %d", name, dtype);
  if (rows < 0 || cols <= 0 || cols > (int64_t)1 << 30)
    return ak_set_error(AK_ERR_INVALID_ARG, "%s: bad shape rows=%lld cols=%lld", name, (long long)rows, (long long)cols);
  if (ld_x < cols || ld_y < cols) return ak_set_error(AK_ERR_INVALID_ARG, "%s: row pitch smaller than cols", name);
  if (!ak_extent_ok(rows, ld_x, cols, ak_dtype_size(dtype)) || !ak_extent_ok(rows, ld_y, cols, ak_dtype_size(dtype)))
    return ak_set_error(AK_ERR_INVALID_ARG, "%s: rows=%lld x pitch exceed 64-bit addressing", name, (long long)rows);
  if (rows == 0) return AK_OK;
  if (!x || !y) return ak_set_error(AK_ERR_INVALID_ARG, "%s: null pointer", name);
  hipStream_t s = ak_stream(stream);
  switch (dtype) {
    case AK_DTYPE_F32: return ak::dispatch<float>(x, y, rows, cols, ld_x, ld_y, s);
    case AK_DTYPE_F16: return ak::dispatch<ak::f16>(x, y, rows, cols, ld_x, ld_y, s);
    default: return ak::dispatch<ak::bf16>(x, y, rows, cols, ld_x, ld_y, s);
  }
}
