// Cross-entropy over materialised logits [rows, vocab] for gfx950.
//
// Semantics of kernels/ce_fused.py:122-329 (forward) and :405-488 (tiny-mode
// backward) of the reference:
//   x      = softcap > 0 ? softcap * tanh(logit / softcap) : logit
//   lse    = max + log(sum(exp(x - max)))                 (always written)
//   loss   = ignored ? 0 : lse - (1 - a) * x[t] - a * mean(x)   (a = smoothing)
//   grad_i = (p_i (1 + 2 w lse) - [i == t](1 - a) - a / V)
//            * (softcap ? 1 - tanh^2 : 1) * scale
//   (w = z-loss weight: the gradient of loss + w lse^2); ignored rows get a
//   zero gradient row.
// The forward holds a row of up to 16384 16-byte vectors in registers, packed,
// so that it crosses HBM once whether or not the gradient is written; wider
// rows are streamed (the gradient pass re-reads the row). Row addresses and
// widths are free: vectors start at the row's first 16-byte boundary. The
// gradient scale can come from device memory (scale_dev), so the mean's 1 /
// #counted-rows and the upstream gradient never need a host read.
// ce_count_kernel and ce_mean_kernel reduce the targets and per-row results in
// one workgroup in a fixed order (deterministic).
#include <algorithm>

#include "ak_common.h"

namespace ak {
namespace {

constexpr int kCeThreads = 256;

struct CeParams {
  float softcap, inv_softcap, ls, ls_uniform, scale, zw2;  // zw2 = 2 * z-loss weight
  float tcoeff, vocab;  // 1 - ls (1 without smoothing), the vocabulary as a float
  const float* scale_dev;  // optional device factor of scale
  int64_t ignore_index;
  bool use_softcap, use_ls;
  bool nt;  // the logits (and their gradient) pass the last-level cache
};

__device__ __forceinline__ float cap(const CeParams& p, float x) {
  return p.use_softcap ? p.softcap * tanh_f32(x * p.inv_softcap) : x;
}

struct MS {
  float m, s;
};

// Merge two online (max, sum-relative-to-max) states.
__device__ __forceinline__ MS merge(MS a, MS b) {
  if (a.m != a.m || b.m != b.m) return {NAN, NAN};
  const float m = fmaxf(a.m, b.m);
  if (m == -INFINITY) return {m, 0.0f};
  float s = 0.0f;
  if (a.m != -INFINITY) s += a.s * fast_exp(a.m - m);
  if (b.m != -INFINITY) s += b.s * fast_exp(b.m - m);
  return {m, s};
}

// Workgroup-wide merge; every thread returns the row result.
__device__ MS block_merge(MS st, float& sum_x) {
  for (int off = 1; off < 64; off <<= 1) {
    MS o{__shfl_xor(st.m, off, 64), __shfl_xor(st.s, off, 64)};
    st = merge(st, o);
  }
  sum_x = wave_sum(sum_x);
  __shared__ float sm[kCeThreads / 64], ss[kCeThreads / 64], sx[kCeThreads / 64];
  const int w = threadIdx.x / 64;
  if ((threadIdx.x & 63) == 0) {
    sm[w] = st.m;
    ss[w] = st.s;
    sx[w] = sum_x;
  }
  __syncthreads();
  st = {sm[0], ss[0]};
  sum_x = sx[0];
#pragma unroll
  for (int i = 1; i < kCeThreads / 64; ++i) {
    st = merge(st, MS{sm[i], ss[i]});
    sum_x += sx[i];
  }
  __syncthreads();  // sm / ss / sx are rewritten for the workgroup's next row
  return st;
}

// What the gradient elements of one row share. zf = 1 + 2 w lse folds the
// z-loss term into the softmax part.
struct RowGrad {
  float m, inv_s, zf, scale;
  __device__ __forceinline__ RowGrad(const CeParams& p, float m_, float s) : m(m_) {
    inv_s = 1.0f / s;
    zf = p.zw2 != 0.0f ? fmaf(p.zw2, m + fast_log(s), 1.0f) : 1.0f;
    scale = p.scale_dev ? p.scale * p.scale_dev[0] : p.scale;
  }
};

// Gradient of one element from its logit; CAP: the softcap is on.
template <bool CAP>
__device__ __forceinline__ float grad_value(const CeParams& p, const RowGrad& r, float xo, bool is_tgt) {
  float th = 0.0f;
  if constexpr (CAP) th = tanh_f32(xo * p.inv_softcap);
  float g = fast_exp((CAP ? p.softcap * th : xo) - r.m) * r.inv_s * r.zf;
  if (is_tgt) g -= p.tcoeff;
  if (p.use_ls) g -= p.ls_uniform;
  if constexpr (CAP) g *= 1.0f - th * th;
  return g * r.scale;
}

// One vector of gradients; te: the target's place in it, or anything outside
// [0, VE). RARE: only the wave that holds the target compares element by
// element, at the price of a second copy of the arithmetic.
template <typename T, bool CAP, bool RARE>
__device__ __forceinline__ Vec16<T> grad_vec(const CeParams& p, const RowGrad& r, const Vec16<T>& xv, int te) {
  constexpr int VE = Vec16<T>::VE;
  Vec16<T> o;
  if (!RARE || (unsigned)te < (unsigned)VE) {
#pragma unroll
    for (int e = 0; e < VE; ++e) o.e[e] = from_f32<T>(grad_value<CAP>(p, r, to_f32(xv.e[e]), e == te));
  } else {
#pragma unroll
    for (int e = 0; e < VE; ++e) o.e[e] = from_f32<T>(grad_value<CAP>(p, r, to_f32(xv.e[e]), false));
  }
  return o;
}

// Gradient of the row's elements [v0, v1) (vectors) and, where `ends` is set,
// of the elements around the vectors: zero for ignored rows, NaN for
// out-of-range targets, otherwise the softmax gradient. U vectors of a thread
// are loaded before the first is used. NT: past the caches. RAG: rows at any
// address and of any width; otherwise whole aligned vectors.
template <typename T, bool CAP, bool NT, bool RAG, int U, typename I>
__device__ void write_grad_row(const CeParams& p, const T* __restrict__ row, T* __restrict__ grow,
                               I vocab, I tgt, bool ignored, bool bad, float m,
                               float s, I v0, I v1, bool ends, int threads) {
  constexpr int VE = Vec16<T>::VE;
  const int t = threadIdx.x;
  I nvec = vocab / VE, ex = -1, head = 0;
  if constexpr (RAG) {
    const RowSplit<T, I> sp(row, vocab);
    nvec = sp.nvec;
    head = sp.head;
    if (ends && t < sp.nx) ex = sp.extra(t);
  }
  auto ld = [](const T* q) { return NT ? load16_any_nt(q) : load16_any(q); };
  auto st = [](T* q, const Vec16<T>& w) {
    if (NT) store16_any_nt(q, w);
    else store16_any(q, w);
  };
  row += head;  // row / grow: the vectors' first element
  T* const gv = grow + head;
  if (v1 > nvec) v1 = nvec;
  if (ignored || bad) {
    const T c = from_f32<T>(ignored ? 0.0f : NAN);
    Vec16<T> o;
#pragma unroll
    for (int e = 0; e < VE; ++e) o.e[e] = c;
    for (I v = v0 + t; v < v1; v += threads) st(gv + (int64_t)v * VE, o);
    if (RAG && ex >= 0) grow[ex] = c;
    return;
  }
  float xe = 0.0f;
  if (RAG && ex >= 0) xe = to_f32(row[ex - head]);
  const I tv = tgt - head;  // relative to the vectors
  auto place = [&](I v) {
    const I d = tv - v * VE;
    return d >= 0 && d < VE ? (int)d : -1;
  };
  I v = v0 + t;
  const RowGrad r(p, m, s);
  for (; U > 1 && v + (U - 1) * threads < v1; v += U * threads) {
    Vec16<T> x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = ld(row + (int64_t)(v + u * threads) * VE);
#pragma unroll
    for (int u = 0; u < U; ++u)
      st(gv + (int64_t)(v + u * threads) * VE, grad_vec<T, CAP, true>(p, r, x[u], place(v + u * threads)));
  }
  for (; v < v1; v += threads)
    st(gv + (int64_t)v * VE, grad_vec<T, CAP, (U > 1)>(p, r, ld(row + (int64_t)v * VE), place(v)));
  if (RAG && ex >= 0) grow[ex] = from_f32<T>(grad_value<CAP>(p, r, xe, ex == tgt));
}

// A row held in registers: TPR threads, VPT vectors each, packed between the
// passes (max, sum, gradient) and converted again in each, plus the elements
// around the vectors one to a thread. HBM-bound: 4 VPT registers hold the row,
// so up to 8 vectors two 1024-thread workgroups fit a CU and one's loads and
// stores run under the other's exponentials. [4096, 32768] bf16 with its
// gradient 155 -> 104 us, 5.2 TB/s (256 threads streamed the row and read it
// again for the gradient); [4096, 50257] fp16 without one 334 -> 74 us, 5.6 TB/s,
// and the backward from saved statistics 315 -> 168 us (both had element
// accesses).
template <typename T, int VPT, int TPR, bool CAP>
__global__ void __launch_bounds__(TPR, VPT == 8 ? 8 : 1)
ce_row_kernel(const T* __restrict__ logits, const int64_t* __restrict__ targets,
              float* __restrict__ losses, float* __restrict__ lse_out,
              float* __restrict__ max_out, float* __restrict__ sum_out,
              T* __restrict__ grad, int64_t rows, int vocab, int64_t ld, int64_t ld_g,
              CeParams p) {
  constexpr int VE = Vec16<T>::VE;
  constexpr int W = TPR / 64;
  __shared__ float part_m[W], part_s[W], part_x[W];
  for (int64_t b = blockIdx.x; b < rows; b += gridDim.x) {
    // The thread's index, opaque to the compiler in each pass: the VPT offsets
    // and bounds derived from it would otherwise be held from pass to pass
    // (and row to row) beside the row, and spill.
    auto thread = [] {
      int t = threadIdx.x;
      asm volatile("" : "+v"(t));
      return t;
    };
    int t = thread();
    const T* row = logits + b * ld;
    const RowSplit<T> sp(row, vocab);
    const T* rv = row + sp.head;
    const int64_t tgt = targets[b];
    const bool ignored = tgt == p.ignore_index;
    const bool bad = !ignored && (tgt < 0 || tgt >= vocab);
    T xe = T(0.0f), xt = T(0.0f);  // this thread's single element, the target's logit
    if (t < sp.nx) xe = row[sp.extra(t)];
    if (t == 0 && !ignored && !bad) xt = row[tgt];
    Vec16<T> raw[VPT];
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      raw[k].u = u32x4{0, 0, 0, 0};
      if (t + k * TPR < sp.nvec) raw[k] = load16_any_nt(rv + k * TPR * VE + (unsigned)(t * VE));
    }

    // max; the cap is monotonic, so the largest capped logit is the cap of the largest
    t = thread();
    float m = t < sp.nx ? to_f32(xe) : -INFINITY;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      if (t + k * TPR < sp.nvec) {
#pragma unroll
        for (int e = 0; e < VE; ++e) m = fmaxf(m, to_f32(raw[k].e[e]));
      }
      keep_packed(raw[k]);
    }
    m = wave_max(m);
    if ((t & 63) == 0) part_m[t / 64] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < W; ++i) m = fmaxf(m, part_m[i]);
    if constexpr (CAP) m = cap(p, m);

    // sum of exp(x - m) (and of x); a row of -inf alone sums to 0, a NaN stays one
    const float off = m == -INFINITY ? 0.0f : m;
    float s = 0.0f, sx = 0.0f;
    t = thread();
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      if (t + k * TPR < sp.nvec) {
#pragma unroll
        for (int e = 0; e < VE; ++e) {
          const float x = CAP ? cap(p, to_f32(raw[k].e[e])) : to_f32(raw[k].e[e]);
          s += fast_exp(x - off);
          if (p.use_ls) sx += x;
        }
      }
      keep_packed(raw[k]);
    }
    if (t < sp.nx) {
      const float x = CAP ? cap(p, to_f32(xe)) : to_f32(xe);
      s += fast_exp(x - off);
      sx += x;
    }
    s = wave_sum(s);
    if (p.use_ls) sx = wave_sum(sx);
    if ((t & 63) == 0) {
      part_s[t / 64] = s;
      part_x[t / 64] = sx;
    }
    __syncthreads();  // part_m has been read by all, so the next row may write it
    s = part_s[0];
    sx = part_x[0];
#pragma unroll
    for (int i = 1; i < W; ++i) {
      s += part_s[i];
      sx += part_x[i];
    }
    if (s != s && m != INFINITY) m = NAN;  // the row holds a NaN

    if (t == 0) {
      const float lse = m + fast_log(s);
      lse_out[b] = lse;
      if (max_out) max_out[b] = m;
      if (sum_out) sum_out[b] = s;
      const float x = CAP ? cap(p, to_f32(xt)) : to_f32(xt);
      float loss = p.use_ls ? lse - p.tcoeff * x - p.ls * (sx / p.vocab) : lse - x;
      if (ignored) loss = 0.0f;
      if (bad) loss = NAN;
      losses[b] = loss;
    }
    if (grad) {
      T* grow = grad + b * ld_g;
      T* gv = grow + sp.head;
      t = thread();
      const int ex = t < sp.nx ? sp.extra(t) : -1;
      if (!ignored && !bad) {
        const RowGrad r(p, m, s);
        const int tv = (int)tgt - sp.head;
#pragma unroll
        for (int k = 0; k < VPT; ++k)
          if (t + k * TPR < sp.nvec)
            store16_any_nt(gv + k * TPR * VE + (unsigned)(t * VE),
                           grad_vec<T, CAP, true>(p, r, raw[k], tv - (t + k * TPR) * VE));
        if (ex >= 0) grow[ex] = from_f32<T>(grad_value<CAP>(p, r, to_f32(xe), ex == (int)tgt));
      } else {
        Vec16<T> o;
#pragma unroll
        for (int e = 0; e < VE; ++e) o.e[e] = from_f32<T>(ignored ? 0.0f : NAN);
#pragma unroll
        for (int k = 0; k < VPT; ++k)
          if (t + k * TPR < sp.nvec) store16_any_nt(gv + k * TPR * VE + (unsigned)(t * VE), o);
        if (ex >= 0) grow[ex] = o.e[0];
      }
    }
    __syncthreads();  // part_s / part_x are rewritten for the workgroup's next row
  }
}

template <typename T, bool VEC>
__device__ void ce_fwd_row(const T* __restrict__ row, int64_t b, const int64_t* __restrict__ targets,
                           float* __restrict__ losses, float* __restrict__ lse_out,
                           float* __restrict__ max_out, float* __restrict__ sum_out,
                           T* __restrict__ grow, int64_t vocab, const CeParams& p) {
  constexpr int VE = Vec16<T>::VE;
  const int64_t tgt = targets[b];
  const bool ignored = tgt == p.ignore_index;
  const bool bad = !ignored && (tgt < 0 || tgt >= vocab);

  MS st{-INFINITY, 0.0f};
  float sum_x = 0.0f;
  auto consume = [&](const float* xs, int n) {
    float vm = -INFINITY;
    for (int e = 0; e < n; ++e) vm = fmaxf(vm, xs[e]);
    if (vm > st.m) {
      st.s = st.s * fast_exp(st.m - vm);
      st.m = vm;
    }
    if (st.m != -INFINITY) {
      for (int e = 0; e < n; ++e) st.s += fast_exp(xs[e] - st.m);
    }
  };
  if (VEC) {
    const int64_t nvec = vocab / VE;
    for (int64_t v = threadIdx.x; v < nvec; v += kCeThreads) {
      const Vec16<T> xv = p.nt ? load16_nt(row + v * VE) : load16(row + v * VE);
      float xs[VE];
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        xs[e] = cap(p, to_f32(xv.e[e]));
        if (p.use_ls) sum_x += xs[e];
        if (xs[e] != xs[e]) st = {NAN, NAN};
      }
      if (st.m == st.m) consume(xs, VE);
    }
  } else {
    for (int64_t i = threadIdx.x; i < vocab; i += kCeThreads) {
      float xv = cap(p, to_f32(row[i]));
      if (p.use_ls) sum_x += xv;
      if (xv != xv) st = {NAN, NAN};
      if (st.m == st.m) consume(&xv, 1);
    }
  }
  st = block_merge(st, sum_x);
  const float lse = st.m + fast_log(st.s);

  if (threadIdx.x == 0) {
    lse_out[b] = lse;
    if (max_out) max_out[b] = st.m;
    if (sum_out) sum_out[b] = st.s;
    float loss;
    if (ignored) {
      loss = 0.0f;
    } else if (bad) {
      loss = NAN;
    } else {
      const float xt = cap(p, to_f32(row[tgt]));
      loss = p.use_ls ? lse - (1.0f - p.ls) * xt - p.ls * (sum_x / (float)vocab) : lse - xt;
    }
    losses[b] = loss;
  }
  if (grow) {
    if (p.use_softcap)
      write_grad_row<T, true, true, true, 4, int64_t>(p, row, grow, vocab, tgt, ignored, bad, st.m, st.s, 0, vocab, true, kCeThreads);
    else
      write_grad_row<T, false, true, true, 4, int64_t>(p, row, grow, vocab, tgt, ignored, bad, st.m, st.s, 0, vocab, true, kCeThreads);
  }
}

// One 256-thread workgroup per row, rows by grid stride (the loop bound is
// uniform per workgroup, so block_merge's barriers are reached by all waves).
template <typename T, bool VEC>
__global__ void __launch_bounds__(kCeThreads)
ce_fwd_kernel(const T* __restrict__ logits, const int64_t* __restrict__ targets,
              float* __restrict__ losses, float* __restrict__ lse_out,
              float* __restrict__ max_out, float* __restrict__ sum_out,
              T* __restrict__ grad, int64_t rows, int64_t vocab, int64_t ld, int64_t ld_g,
              CeParams p) {
  for (int64_t b = blockIdx.x; b < rows; b += gridDim.x)
    ce_fwd_row<T, VEC>(logits + b * ld, b, targets, losses, lse_out, max_out, sum_out,
                       grad ? grad + b * ld_g : nullptr, vocab, p);
}

// The gradient from the saved row statistics: blockIdx.y takes `span` vectors
// of the row, so that few rows still fill the GPU.
template <typename T, bool CAP, bool NT, bool RAG, int U, typename I>
__global__ void __launch_bounds__(kCeThreads)
ce_bwd_tiny_kernel(const T* __restrict__ logits, const int64_t* __restrict__ targets,
                   const float* __restrict__ row_max, const float* __restrict__ row_sum,
                   T* __restrict__ grad, int64_t rows, I vocab, int64_t ld, int64_t ld_g,
                   I span, CeParams p) {
  const I v0 = (I)blockIdx.y * span;
  for (int64_t b = blockIdx.x; b < rows; b += gridDim.x) {
    const int64_t tgt = targets[b];
    const bool ignored = tgt == p.ignore_index;
    const bool bad = !ignored && (tgt < 0 || tgt >= vocab);
    write_grad_row<T, CAP, NT, RAG, U, I>(p, logits + b * ld, grad + b * ld_g, vocab, (I)tgt, ignored, bad, row_max[b],
                              row_sum[b], v0, v0 + span, blockIdx.y == 0, kCeThreads);
  }
}

constexpr int kCeReduceThreads = 1024;

// Sum of per-thread values over one 1024-thread workgroup in a fixed order
// (wave DPP / shuffle tree, then the 16 wave sums in index order). Every
// thread returns the total.
template <typename V>
__device__ V workgroup_sum_fixed(V v, V* lds) {
  if constexpr (std::is_same<V, float>::value) {
    v = wave_sum(v);
  } else {
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  }
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x / 64] = v;
  __syncthreads();
  V t = lds[0];
  for (int i = 1; i < kCeReduceThreads / 64; ++i) t += lds[i];
  return t;
}

// denom[0] = max(1, #rows whose target is not ignore_index), denom[1] = 1 / denom[0].
__global__ void __launch_bounds__(kCeReduceThreads)
ce_count_kernel(const int64_t* __restrict__ targets, int64_t rows, int64_t ignore_index,
                float* __restrict__ denom) {
  __shared__ long long lds[kCeReduceThreads / 64];
  long long n = 0;
  for (int64_t i = threadIdx.x; i < rows; i += kCeReduceThreads) n += targets[i] != ignore_index;
  n = workgroup_sum_fixed<long long>(n, lds);
  if (threadIdx.x == 0) {
    const float d = n > 0 ? (float)n : 1.0f;
    denom[0] = d;
    denom[1] = 1.0f / d;
  }
}

// loss[0] = (sum over counted rows of losses + w * sum of lse^2) / max(1, #counted),
// per-thread partials in row order, then workgroup_sum_fixed. n_valid (nullable)
// receives the count.
__global__ void __launch_bounds__(kCeReduceThreads)
ce_mean_kernel(const float* __restrict__ losses, const float* __restrict__ lse,
               const int64_t* __restrict__ targets, int64_t rows, int64_t ignore_index,
               float zw, float* __restrict__ loss, int64_t* __restrict__ n_valid) {
  __shared__ float lds_f[kCeReduceThreads / 64];
  __shared__ long long lds_n[kCeReduceThreads / 64];
  float s = 0.0f;
  long long n = 0;
  for (int64_t i = threadIdx.x; i < rows; i += kCeReduceThreads) {
    if (targets[i] == ignore_index) continue;
    float v = losses[i];
    if (zw != 0.0f) v = fmaf(zw * lse[i], lse[i], v);
    s += v;
    ++n;
  }
  s = workgroup_sum_fixed<float>(s, lds_f);
  n = workgroup_sum_fixed<long long>(n, lds_n);
  if (threadIdx.x == 0) {
    loss[0] = s / (n > 0 ? (float)n : 1.0f);
    if (n_valid) n_valid[0] = n;
  }
}

// x *= round_T(scale[0]), each product rounded once. A scale of exactly 1 (the
// plain loss.backward()) costs one scalar read instead of a pass over x, the
// bits being those of the product either way.
template <typename T>
__global__ void __launch_bounds__(kCeThreads)
scale_kernel(T* __restrict__ x, int64_t n, const float* __restrict__ scale) {
  const float g = to_f32(from_f32<T>(scale[0]));
  if (g == 1.0f) return;
  constexpr int VE = Vec16<T>::VE;
  const RowSplit<T, int64_t> sp(x, n);
  const int64_t at = (int64_t)blockIdx.x * kCeThreads + threadIdx.x;
  T* const xv = x + sp.head;
  for (int64_t v = at; v < sp.nvec; v += (int64_t)gridDim.x * kCeThreads) {
    Vec16<T> a = load16(xv + v * VE);
#pragma unroll
    for (int e = 0; e < VE; ++e) a.e[e] = from_f32<T>(to_f32(a.e[e]) * g);
    store16(xv + v * VE, a);
  }
  if (at < sp.nx) x[sp.extra((int)at)] = from_f32<T>(to_f32(x[sp.extra((int)at)]) * g);
}

template <typename T>
void launch_scale(void* x, int64_t n, const float* scale, hipStream_t s) {
  // 8 workgroups a CU: few enough that the launch of a scale of 1 stays cheap
  const int64_t units = (n / Vec16<T>::VE + kCeThreads - 1) / kCeThreads;
  const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>(units, 2048));
  scale_kernel<T><<<dim3(grid), dim3(kCeThreads), 0, s>>>(static_cast<T*>(x), n, scale);
}

CeParams make_params(float softcap, int64_t ignore_index, float ls, float scale, int64_t vocab,
                     float zw = 0.0f, const float* scale_dev = nullptr) {
  CeParams p;
  p.use_softcap = softcap > 0.0f;
  p.softcap = softcap;
  p.inv_softcap = p.use_softcap ? 1.0f / softcap : 0.0f;
  p.use_ls = ls > 0.0f;
  p.ls = ls;
  p.ls_uniform = ls / (float)vocab;
  p.tcoeff = p.use_ls ? 1.0f - ls : 1.0f;
  p.vocab = (float)vocab;
  p.scale = scale;
  p.zw2 = 2.0f * zw;
  p.scale_dev = scale_dev;
  p.ignore_index = ignore_index;
  return p;
}

// Rows are walked by grid stride and indexed in 64 bits; the one limit is
// that the last row's end must be addressable.
int check(const void* logits, const int64_t* targets, void* grad, int64_t rows, int64_t vocab,
          int64_t ld, int64_t ld_g, int dtype, const char* name) {
  if (ak_dtype_size(dtype) == 0) return ak_set_error(AK_ERR_UNSUPPORTED, "%s: unsupported dtype code %d", name, dtype);
  if (rows < 0 || vocab <= 0) return ak_set_error(AK_ERR_INVALID_ARG, "%s: bad shape rows=%lld vocab=%lld", name, (long long)rows, (long long)vocab);
  if (ld < vocab || (grad && ld_g < vocab)) return ak_set_error(AK_ERR_INVALID_ARG, "%s: row pitch smaller than vocab", name);
  if (!ak_extent_ok(rows, ld, vocab, ak_dtype_size(dtype)) ||
      (grad && !ak_extent_ok(rows, ld_g, vocab, ak_dtype_size(dtype))))
    return ak_set_error(AK_ERR_INVALID_ARG, "%s: rows=%lld x pitch exceed 64-bit addressing", name, (long long)rows);
  if (rows > 0 && (!logits || !targets)) return ak_set_error(AK_ERR_INVALID_ARG, "%s: null pointer", name);
  return AK_OK;
}

// Whether that many bytes pass the 256 MiB last-level cache, so that nothing of
// them would be found there again.
bool past_cache(int64_t bytes) { return bytes > (int64_t)300 << 20; }

// The row-resident forward with the fewest vectors a thread that its workgroup
// sizes allow (256 threads up to 1024 vectors, for more rows in flight; 512 up to
// 4096, since 4 vectors in each of 1024 threads took 122 us for [4096, 32768] bf16 with a
// softcap, where 8 in 512 take 72). Returns false for the streaming kernel: past 16384
// vectors, and past 8192 without a gradient in many whole rows, where one held row
// a CU leaves its loads and its exponentials in turn ([1024, 65536] fp32 54.7 us held,
// 42.6 streamed, [1024, 131072] bf16 69 and 52; 512 rows 28.4 and 33.5).
template <typename T, bool CAP>
bool launch_row(const T* lg, const int64_t* targets, float* losses, float* lse, float* mx,
                float* sm, T* g, int64_t rows, int64_t vocab, int64_t ld, int64_t ld_g,
                const CeParams& p, bool stream_ok, hipStream_t s) {
  const int64_t nvec = vocab / Vec16<T>::VE;
  if (nvec > 16384 || (nvec > 8192 && !g && rows >= 1024 && stream_ok)) return false;
#define AK_LAUNCH(VPT, TPR)                                                                   \
  ce_row_kernel<T, VPT, TPR, CAP><<<dim3(row_grid(rows)), dim3(TPR), 0, s>>>(                 \
      lg, targets, losses, lse, mx, sm, g, rows, (int)vocab, ld, ld_g, p)
  if (nvec <= 256) AK_LAUNCH(1, 256);
  else if (nvec <= 512) AK_LAUNCH(2, 256);
  else if (nvec <= 1024) AK_LAUNCH(4, 256);
  else if (nvec <= 2048) AK_LAUNCH(4, 512);
  else if (nvec <= 4096) AK_LAUNCH(8, 512);
  else if (nvec <= 8192) AK_LAUNCH(8, 1024);
  else AK_LAUNCH(16, 1024);
#undef AK_LAUNCH
  return true;
}

template <typename T>
void launch_fwd(const void* logits, const int64_t* targets, float* losses, float* lse, float* mx,
                float* sm, void* grad, int64_t rows, int64_t vocab, int64_t ld, int64_t ld_g,
                CeParams p, hipStream_t s) {
  const T* lg = static_cast<const T*>(logits);
  T* g = static_cast<T*>(grad);
  p.nt = past_cache((grad ? 2 : 1) * rows * vocab * (int64_t)sizeof(T));
  constexpr int VE = Vec16<T>::VE;
  const bool aligned = vocab % VE == 0 && ld % VE == 0 && aligned16(logits);
  const bool done = p.use_softcap
      ? launch_row<T, true>(lg, targets, losses, lse, mx, sm, g, rows, vocab, ld, ld_g, p, aligned, s)
      : launch_row<T, false>(lg, targets, losses, lse, mx, sm, g, rows, vocab, ld, ld_g, p, aligned, s);
  if (done) return;
  const dim3 grid(row_grid(rows)), block(kCeThreads);
  if (aligned)
    ce_fwd_kernel<T, true><<<grid, block, 0, s>>>(lg, targets, losses, lse, mx, sm, g, rows, vocab, ld, ld_g, p);
  else
    ce_fwd_kernel<T, false><<<grid, block, 0, s>>>(lg, targets, losses, lse, mx, sm, g, rows, vocab, ld, ld_g, p);
}

template <typename T>
void launch_bwd(const void* logits, const int64_t* targets, const float* mx, const float* sm,
                void* grad, int64_t rows, int64_t vocab, int64_t ld, int64_t ld_g,
                const CeParams& p, hipStream_t s) {
  const T* lg = static_cast<const T*>(logits);
  T* g = static_cast<T*>(grad);
  // workgroups of one round of 4 vectors a thread where the row is that wide:
  // [4096, 50257] fp16 takes 168 us so and 179 us with one workgroup a row
  const int64_t nvec = vocab / Vec16<T>::VE;
  const int64_t ny = std::min<int64_t>(nvec / (4 * kCeThreads), 65535);
  const int64_t span = ny > 1 ? (nvec + ny - 1) / ny : nvec;
  const dim3 grid(row_grid(rows), ny > 1 ? (unsigned)ny : 1), block(kCeThreads);
  auto go = [&](auto nt, auto rag, auto unroll, auto index) {
    using I = decltype(index);
    constexpr bool NT = decltype(nt)::value, RAG = decltype(rag)::value;
    constexpr int U = decltype(unroll)::value;
    if (p.use_softcap)
      ce_bwd_tiny_kernel<T, true, NT, RAG, U, I><<<grid, block, 0, s>>>(lg, targets, mx, sm, g, rows, (I)vocab, ld, ld_g, (I)span, p);
    else
      ce_bwd_tiny_kernel<T, false, NT, RAG, U, I><<<grid, block, 0, s>>>(lg, targets, mx, sm, g, rows, (I)vocab, ld, ld_g, (I)span, p);
  };
  // One vector at a time where a row has no round of four (fewer registers, more
  // rows in flight: [4096, 1024] fp32 8.1 -> 6.6 us). Nontemporal accesses where the logits
  // and their gradient pass the 256 MiB last-level cache ([4096, 32768] bf16 90.8 us
  // so, 100.8 without; [2048, 16384] fp32, 268 MB: 45.5 and 41.3, as the forward's
  // logits are still there). 32-bit columns, a shorter chain of address arithmetic,
  // up to 2^30 of them.
  using One = std::integral_constant<int, 1>;
  using Four = std::integral_constant<int, 4>;
  const bool big = past_cache(2 * rows * vocab * (int64_t)sizeof(T));
  using Yes = std::true_type;
  using No = std::false_type;
  const bool aligned = vocab % Vec16<T>::VE == 0 && ld % Vec16<T>::VE == 0 && aligned16(logits);
  if (vocab >= (int64_t)1 << 30) go(Yes{}, Yes{}, Four{}, int64_t{});
  else if (nvec < 4 * kCeThreads && aligned) go(No{}, No{}, One{}, int{});
  else if (nvec < 4 * kCeThreads) go(No{}, Yes{}, One{}, int{});
  else if (big) go(Yes{}, Yes{}, Four{}, int64_t{});
  else go(No{}, Yes{}, Four{}, int64_t{});
}

}  // namespace
}  // namespace ak

extern "C" int ak_ce_fwd(const void* logits, const int64_t* targets, float* losses, float* lse,
                         float* row_max, float* row_sum, void* grad_logits, int64_t rows,
                         int64_t vocab, int64_t ld_logits, int64_t ld_grad, float softcap,
                         int64_t ignore_index, float label_smoothing, float scale_grad,
                         float z_loss_weight, const float* scale_dev, int dtype, void* stream) {
  const char* name = "ak_ce_fwd";
  int rc = ak::check(logits, targets, grad_logits, rows, vocab, ld_logits, ld_grad, dtype, name);
  if (rc) return rc;
  if (!(z_loss_weight >= 0.0f)) return ak_set_error(AK_ERR_INVALID_ARG, "%s: z_loss_weight must be >= 0", name);
  if (rows > 0 && (!losses || !lse)) return ak_set_error(AK_ERR_INVALID_ARG, "%s: null losses/lse", name);
  if (rows == 0) return AK_OK;
  const ak::CeParams p = ak::make_params(softcap, ignore_index, label_smoothing, scale_grad, vocab,
                                         z_loss_weight, scale_dev);
  hipStream_t s = ak_stream(stream);
  switch (dtype) {
    case AK_DTYPE_F32: ak::launch_fwd<float>(logits, targets, losses, lse, row_max, row_sum, grad_logits, rows, vocab, ld_logits, ld_grad, p, s); break;
    case AK_DTYPE_F16: ak::launch_fwd<ak::f16>(logits, targets, losses, lse, row_max, row_sum, grad_logits, rows, vocab, ld_logits, ld_grad, p, s); break;
    default: ak::launch_fwd<ak::bf16>(logits, targets, losses, lse, row_max, row_sum, grad_logits, rows, vocab, ld_logits, ld_grad, p, s); break;
  }
  return ak_check_launch(name);
}

extern "C" int ak_ce_bwd_tiny(const void* logits, const int64_t* targets, const float* row_max,
                              const float* row_sum, void* grad_logits, int64_t rows, int64_t vocab,
                              int64_t ld_logits, int64_t ld_grad, float softcap,
                              int64_t ignore_index, float label_smoothing, float scale_grad,
                              float z_loss_weight, const float* scale_dev, int dtype,
                              void* stream) {
  const char* name = "ak_ce_bwd_tiny";
  int rc = ak::check(logits, targets, grad_logits, rows, vocab, ld_logits, ld_grad, dtype, name);
  if (rc) return rc;
  if (!(z_loss_weight >= 0.0f)) return ak_set_error(AK_ERR_INVALID_ARG, "%s: z_loss_weight must be >= 0", name);
  if (rows > 0 && (!row_max || !row_sum || !grad_logits)) return ak_set_error(AK_ERR_INVALID_ARG, "%s: null pointer", name);
  if (rows == 0) return AK_OK;
  const ak::CeParams p = ak::make_params(softcap, ignore_index, label_smoothing, scale_grad, vocab,
                                         z_loss_weight, scale_dev);
  hipStream_t s = ak_stream(stream);
  switch (dtype) {
    case AK_DTYPE_F32: ak::launch_bwd<float>(logits, targets, row_max, row_sum, grad_logits, rows, vocab, ld_logits, ld_grad, p, s); break;
    case AK_DTYPE_F16: ak::launch_bwd<ak::f16>(logits, targets, row_max, row_sum, grad_logits, rows, vocab, ld_logits, ld_grad, p, s); break;
    default: ak::launch_bwd<ak::bf16>(logits, targets, row_max, row_sum, grad_logits, rows, vocab, ld_logits, ld_grad, p, s); break;
  }
  return ak_check_launch(name);
}

extern "C" int ak_ce_count_valid(const int64_t* targets, int64_t rows, int64_t ignore_index,
                                 float* denom, void* stream) {
  const char* name = "ak_ce_count_valid";
  if (rows < 0) return ak_set_error(AK_ERR_INVALID_ARG, "%s: rows < 0", name);
  if (!denom || (rows > 0 && !targets)) return ak_set_error(AK_ERR_INVALID_ARG, "%s: null pointer", name);
  ak::ce_count_kernel<<<dim3(1), dim3(ak::kCeReduceThreads), 0, ak_stream(stream)>>>(
      targets, rows, ignore_index, denom);
  return ak_check_launch(name);
}

extern "C" int ak_ce_mean(const float* losses, const float* lse, const int64_t* targets,
                          int64_t rows, int64_t ignore_index, float z_loss_weight, float* loss,
                          int64_t* n_valid, void* stream) {
  const char* name = "ak_ce_mean";
  if (rows < 0) return ak_set_error(AK_ERR_INVALID_ARG, "%s: rows < 0", name);
  if (!(z_loss_weight >= 0.0f)) return ak_set_error(AK_ERR_INVALID_ARG, "%s: z_loss_weight must be >= 0", name);
  if (!loss || (rows > 0 && (!losses || !targets || (z_loss_weight > 0.0f && !lse))))
    return ak_set_error(AK_ERR_INVALID_ARG, "%s: null pointer", name);
  ak::ce_mean_kernel<<<dim3(1), dim3(ak::kCeReduceThreads), 0, ak_stream(stream)>>>(
      losses, lse, targets, rows, ignore_index, z_loss_weight, loss, n_valid);
  return ak_check_launch(name);
}

extern "C" int ak_scale_inplace(void* x, int64_t n, const float* scale, int dtype, void* stream) {
  const char* name = "ak_scale_inplace";
  const int esz = ak_dtype_size(dtype);
  if (esz == 0) return ak_set_error(AK_ERR_UNSUPPORTED, "%s: unsupported dtype code %d", name, dtype);
  if (n < 0 || n > INT64_MAX / esz) return ak_set_error(AK_ERR_INVALID_ARG, "%s: bad element count", name);
  if (n == 0) return AK_OK;
  if (!x || !scale) return ak_set_error(AK_ERR_INVALID_ARG, "%s: null pointer", name);
  if (reinterpret_cast<uintptr_t>(x) % esz) return ak_set_error(AK_ERR_INVALID_ARG, "%s: misaligned x", name);
  hipStream_t s = ak_stream(stream);
  switch (dtype) {
    case AK_DTYPE_F32: ak::launch_scale<float>(x, n, scale, s); break;
    case AK_DTYPE_F16: ak::launch_scale<ak::f16>(x, n, scale, s); break;
    default: ak::launch_scale<ak::bf16>(x, n, scale, s); break;
  }
  return ak_check_launch(name);
}
