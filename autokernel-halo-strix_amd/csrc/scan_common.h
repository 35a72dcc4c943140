// Definitions shared by the Mamba-1 selective-scan translation units
// (selective_scan.hip: the dstate <= 16 kernels and the C-ABI entry points;
// selective_scan_wide.hip: the general kernels for dstate <= 256 and
// input-independent B / C): the parameter block, the lane-broadcast
// arithmetic and the workspace layout of the backward.
#pragma once

#include "ak_common.h"

namespace ak {

constexpr int kScanT = 64;          // steps per LDS tile
constexpr int kScanCh = 16;         // channels per workgroup (4 waves x 4)
constexpr int kBStride = kScanT + 4; // Bs[n][l] row pitch (floats)
constexpr int kCStride = 20;        // Cs[l][n] row pitch (floats)
constexpr int kHJ = 20;             // hbuf[c][j][n] step pitch (floats)
constexpr int kHC = 16 * kHJ + 16;  // hbuf channel pitch: 336 = 16 mod 64
constexpr int kCk = 16;             // steps between the states saved for the backward
constexpr int kXChunk = 2048;       // steps per chunk-state entry (the reference's chunk)

struct ScanParams {
  const void* u;
  const void* delta;
  const float* A;
  const void* B;
  const void* C;
  const float* D;
  const void* z;
  const float* delta_bias;
  void* out;
  float* last_state;
  void* out_prez;              // optional: y + D u before the gate (strides of out)
  float* chunk_states;         // optional: [batch, dim, xchunks, dstate, 2] (decay product, state)
  int xchunks;                 // 2048-step chunks of chunk_states
  int batch, dim, seqlen, dstate, ngroups, ch_per_group, tiles_per_group;
  int64_t u_bs, u_ds, d_bs, d_ds, A_ds, B_bs, B_gs, B_ns, C_bs, C_gs, C_ns, z_bs, z_ds, o_bs, o_ds;
  int softplus;
  // backward only (the preparation pass and the reverse pass)
  const void* dout;            // [batch, dim, seqlen], element type of u, strides go_bs / go_ds
  void* dz;                    // [batch, dim, seqlen], strides of out
  void* du;                    // [batch, dim, seqlen], strides of out
  void* ddelta;                // [batch, dim, seqlen] in delta's type, strides of out
  float* ck;                   // [batch, nchunks, dim, dstate] states before each 16-step block
                               // (the forward writes them when non-null)
  float* dB_part;              // [tiles, batch, ngroups, dstate, seqlen]
  float* dC_part;              // [tiles, batch, ngroups, dstate, seqlen]
  float* dA_part;              // [batch, dim, dstate]
  float* dD_part;              // [batch, dim]
  float* dbias_part;           // [batch, dim]
  int64_t go_bs, go_ds;
  int nchunks;
  // input-independent B / C ([dim, dstate] fp32, the reference's
  // !is_variable_B / !is_variable_C): flag, channel stride (B_ns / C_ns stay
  // the state strides), and in the backward the per-batch partial sums
  // [batch, dim, dstate] of their gradients
  int b_const, c_const;
  int64_t B_ds, C_ds;
  float* dBc_part;
  float* dCc_part;
  // sequence segments (scan_segments): segs segments of seg_tiles 64-step tiles,
  // and what the segment pass leaves: per segment the state from zero (the
  // adjoint, in the backward) and the sum of delta' over it
  int segs, seg_tiles;
  float* seg_state;            // [batch, segs, dim, dstate]
  float* seg_dsum;             // [batch, segs, dim]
};

// A scan whose (channel, state) lanes leave most of the GPU empty is cut into
// segments of the sequence, a workgroup each. A segment pass first forms each
// segment's state from zero and its sum of delta' (all of its decay: the
// product of exp(delta' A) is exp(A sum delta')); the scan's workgroups then
// fold the segments before theirs into their entering state. The recurrence's
// exponentials are paid twice and a launch is added, so what pays depends on the
// pass (us, uncut -> cut, bf16, 64-step tiles x workgroups of 16 channels):
// * forward, about 512 segments in all (two workgroups a CU). Up to 64 workgroups
//   from 6 tiles on (6 x 64: 11.5 -> 11.4, x 24: 11.5 -> 9.4; 4 x 24 would go
//   8.6 -> 9.4); up to 128 from 16 on (16 x 96: 25.9 -> 24.1, x 128: 26.1 -> 24.4;
//   12 x 128 20.4 -> 20.5), from 12 on with a partial tile, whose kernel is the
//   slower one (12 x 128: 22.7 -> 21.1); about 1024 segments up to 144 from 64 tiles
//   (64 x 144: 95.9 -> 88; 32 x 144 49.6 -> 52), with a partial tile from 32 (57.3
//   -> 54). 64 x 160 would go 96.5 -> 99, 24 x 192 38.4 -> 49. Channels that do not
//   fill groups of 16 run the general kernel, slower still: as the reverse pass (4 x
//   128: 14.7 -> 11.9, 24 x 188 72 -> 62).
// * reverse pass, whose steps cost several times the segment pass's: about 512
//   segments up to 128 workgroups from 4 tiles on (4 x 128: 32.0 -> 27.4, with its
//   preparation pass 41 -> 39), about 1024 up to 192 from 24 on (24 x 192: 128 -> 103,
//   169 -> 152; 24 x 144 126 -> 89).
// A function of the shape alone: the bits of a result depend on it. Where the
// forward is cut, the reverse pass is cut alike.
struct ScanSegs {
  int n, tiles;
};
inline ScanSegs scan_segments(bool reverse, int64_t batch, int64_t dim, int64_t seqlen, int64_t dstate,
                              int64_t ngroups, int bc_flags) {
  const int64_t tiles = (seqlen + kScanT - 1) / kScanT;
  const int64_t groups = batch * ngroups * ((dim / ngroups + kScanCh - 1) / kScanCh);
  const bool whole = seqlen % kScanT == 0;
  const bool early = reverse || (dim / ngroups) % kScanCh != 0;
  int64_t n = 1;
  if (dstate <= 16 && !(bc_flags & (AK_SCAN_B_CONST | AK_SCAN_C_CONST)) && groups > 0) {
    const int64_t few = early ? 4 : groups <= 64 ? 6 : whole ? 16 : 12;  // tiles from which on a cut pays
    const int64_t many = early ? 24 : whole ? 64 : 32;
    if (groups <= 128 && tiles >= few) n = (512 + groups / 2) / groups;
    else if (groups <= (early ? 192 : 144) && tiles >= many) n = 1024 / groups;
    if (n > 32) n = 32;
    if (n > tiles) n = tiles;
    if (n < 1) n = 1;
  }
  const int64_t per = (tiles + n - 1) / n;
  return {per > 0 ? (int)((tiles + per - 1) / per) : 1, per > 0 ? (int)per : 1};
}

// Bytes of the segment pass's states and sums, each region 256-byte aligned.
struct ScanSegWs {
  size_t state, dsum;
};
inline ScanSegWs scan_seg_ws(const ScanSegs& sg, int64_t batch, int64_t dim, int64_t dstate) {
  if (sg.n <= 1) return {0, 0};
  auto a256 = [](int64_t v) { return (size_t)((v + 255) & ~(int64_t)255); };
  return {a256(batch * sg.n * dim * dstate * 4), a256(batch * sg.n * dim * 4)};
}

// v * m, with v taken from lane K of each 16-lane row (DPP row_newbcast:K
// fused into the multiply). The DPP source must not have been written by a
// VALU instruction in the two preceding cycles; callers write it once per
// tile and separate that write from the first use with an s_nop 1.
template <int K>
__device__ __forceinline__ float mul_bcast(float v, float m) {
  float r;
  asm("v_mul_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "=v"(r)
               : "v"(v), "v"(m), "i"(K));
  return r;
}

// torch.nn.functional.softplus with beta=1, threshold=20: x above 20, else
// log1p(e^x). e^x and log2 come from the hardware (about 1 ulp each);
// log1p(t) = log(1 + t) * t / ((1 + t) - 1) corrects the rounding of 1 + t
// (D. Goldberg, "What every computer scientist should know about
// floating-point arithmetic", 1991, Theorem 4), so small results keep their
// relative accuracy. About 8 instructions instead of a library log1p / exp.
__device__ __forceinline__ float softplus_f32(float x) {
  const float t = __builtin_amdgcn_exp2f(fminf(x, 20.0f) * kLog2e);
  const float u = 1.0f + t;
  const float lp = u == 1.0f ? t : __builtin_amdgcn_logf(u) * kLn2 * (t * __builtin_amdgcn_rcpf(u - 1.0f));
  return x > 20.0f ? x : lp;
}

// silu(z) = z / (1 + exp(-z)) with the hardware exp2 and reciprocal (about
// 1 ulp each), evaluated once per output element.
__device__ __forceinline__ float silu_fast(float z) {
  return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-z * kLog2e));
}


constexpr int kTJ = 36;             // tbuf[c][j][n] step pitch: float pairs, b128 reads conflict-free
constexpr int kTC = 16 * kTJ + 16;  // tbuf channel pitch: 592 = 16 mod 64 (1.5% faster than 576 or 608)
constexpr int kWP = 33;             // wbuf[lane][pair] lane pitch

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// a + b over lanes i and i ^ 32 for x, and the same for y, with x's sums
// landing in lanes 0..31 and y's in lanes 32..63.
__device__ __forceinline__ float swap32_sum(float x, float y) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Row pairs (0, 1) and (2, 3): x's sums land in rows 0 and 2, y's in rows 1 and 3.
__device__ __forceinline__ float swap16_sum(float x, float y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// acc + v * m, v from lane K of each 16-lane row (DPP as in mul_bcast).
template <int K>
__device__ __forceinline__ float fma_bcast(float v, float m, float acc) {
  asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+v"(acc)
      : "v"(v), "v"(m), "i"(K));
  return acc;
}

__device__ __forceinline__ float sigmoid_f32(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * kLog2e));
}


// The workgroup's batch, segment and tiles [first, end) of the sequence. An uncut
// scan has them at compile time (kSeg = false): read at run time the bounds cost
// every kernel 1-3% ([4, 2048, 4096] bf16 inference 143.5 -> 148.2 us, the reverse
// pass with dz 440 -> 450).
template <bool kSeg>
struct ScanSeg {
  int b, seg, first, end;
  bool last;
  __device__ __forceinline__ ScanSeg(const ScanParams& p, int bk) {
    b = bk / p.segs;
    seg = bk - b * p.segs;
    const int all = (p.seqlen + kScanT - 1) / kScanT;
    first = seg * p.seg_tiles;
    end = min(first + p.seg_tiles, all);
    last = end == all;
  }
};
template <>
struct ScanSeg<false> {
  static constexpr int seg = 0, first = 0;
  static constexpr bool last = true;
  int b, end;
  __device__ __forceinline__ ScanSeg(const ScanParams& p, int bk) : b(bk), end((p.seqlen + kScanT - 1) / kScanT) {}
};

// The state that enters the segment: the segments before it (kBwd: the adjoint
// that enters it from those behind it), folded in order. A segment's decay may
// leave fp32's range although what it carries does not (a growing recurrence:
// A > 0, or a negative delta'), and an infinite state meets only decays above
// zero step by step: past 2^126 the decay's whole powers of two go to the state's
// exponent, so that the product alone over- or underflows.
template <bool kBwd, bool kSeg>
__device__ __forceinline__ float seg_enter(const ScanParams& p, const ScanSeg<kSeg>& sg, int d, int n, float a_scaled) {
  float h = 0.0f;
  if constexpr (!kSeg) return h;
  const int count = kBwd ? p.segs - 1 - sg.seg : sg.seg;
  auto fold = [&](int i0, auto batch) {  // segments i0 .. i0 + U - 1, loaded at once
    constexpr int U = decltype(batch)::value;
    float in[U], t[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int i = min(i0 + j, count - 1);
      const int64_t at = ((int64_t)sg.b * p.segs + (kBwd ? p.segs - 1 - i : i)) * p.dim + d;
      in[j] = p.seg_state[at * p.dstate + n];
      t[j] = a_scaled * p.seg_dsum[at];
    }
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const float c = fminf(fmaxf(t[j], -1000.0f), 1000.0f);  // 2^1000 takes any fp32 to its end
      const float k = fabsf(c) < 126.0f ? 0.0f : truncf(c);
      const float next = fmaf(__builtin_amdgcn_exp2f(c - k), ldexpf(h, (int)k), in[j]);
      h = i0 + j < count ? next : h;
    }
  };
  int i = 0;
  for (; count - i > 4; i += 8) fold(i, std::integral_constant<int, 8>{});
  if (i < count) fold(i, std::integral_constant<int, 4>{});
  return h;
}

// Workspace of the Mamba-1 backward, each region 256-byte aligned: the states
// before every 16-step block, the per-channel-tile partial rows of a
// variable dB / dC, the per-batch partials of dA / dD / ddelta_bias and of a
// constant dB / dC.
struct ScanBwdWs {
  size_t ck, partB, partC, dA, dD, dBc, dCc, total;
  ScanSegWs seg;
};

inline ScanBwdWs scan_bwd_ws(int64_t batch, int64_t dim, int64_t seqlen, int64_t dstate,
                             int64_t ngroups, int bc_flags) {
  auto a256 = [](int64_t v) { return (size_t)((v + 255) & ~(int64_t)255); };
  const int64_t tiles = (dim / ngroups + kScanCh - 1) / kScanCh;
  const int64_t nck = (seqlen + kCk - 1) / kCk;
  const bool bc = bc_flags & AK_SCAN_B_CONST, cc = bc_flags & AK_SCAN_C_CONST;
  ScanBwdWs w;
  w.ck = a256(batch * nck * dim * dstate * 4);
  w.partB = bc ? 0 : a256(tiles * batch * ngroups * dstate * seqlen * 4);
  w.partC = cc ? 0 : a256(tiles * batch * ngroups * dstate * seqlen * 4);
  const ScanSegs sg = scan_segments(true, batch, dim, seqlen, dstate, ngroups, bc_flags);
  w.seg = scan_seg_ws(sg, batch, dim, dstate);
  w.dA = a256(batch * sg.n * dim * dstate * 4);  // a partial per batch and segment
  w.dD = a256(batch * sg.n * dim * 4);
  w.dBc = bc ? a256(batch * dim * dstate * 4) : 0;
  w.dCc = cc ? a256(batch * dim * dstate * 4) : 0;
  w.total = w.ck + w.partB + w.partC + w.dA + 2 * w.dD + w.dBc + w.dCc + w.seg.state + w.seg.dsum;
  return w;
}

// Complex-A scan (selective_scan_complex.hip). Workspace of its backward,
// each region 256-byte aligned: the complex states every 16 steps and the
// pre-gate output (used when the caller gives no saved states), the
// per-4-channel-tile partial rows of a variable dB / dC, the per-batch
// partials of dA / dD / ddelta_bias and of a constant dB / dC.
struct ZWs {
  size_t ck, prez, partB, partC, dA, dD, dBc, dCc, total;
};
ZWs scan_complex_bwd_ws(int64_t batch, int64_t dim, int64_t seqlen, int64_t dstate, int64_t ngroups,
                        int bc_flags);
// The forward writes out / out_prez / last_state / chunk_states / checkpoints
// (complex where the real forward writes fp32). The backward restarts from
// p.ck / p.out_prez when saved, else re-runs the forward into the workspace,
// and writes every gradient. Both return nonzero for unsupported dtypes.
int launch_scan_complex_fwd(ScanParams p, int u_dtype, int delta_dtype, int bc_dtype, hipStream_t s);
int launch_scan_complex_bwd(ScanParams p, const ZWs& ws, void* workspace, bool saved, int u_dtype,
                            int delta_dtype, int bc_dtype, void* dB, void* dC, float* dA, float* dD,
                            float* ddelta_bias, hipStream_t s);
// Zero-step complex backward: dA, dD, ddelta_bias and a constant dB / dC are
// sums over nothing.
void launch_scan_complex_zero(int dim, int dstate, float* dA, float* dD, float* ddelta_bias,
                              float* dBc, float* dCc, hipStream_t s);

// Whether the general kernels (selective_scan_wide.hip) take the call:
// more than 16 states, or an input-independent B or C.
inline bool scan_needs_wide(const ScanParams& p) {
  return p.dstate > 16 || p.b_const || p.c_const;
}

// Launchers of the general kernels (selective_scan_wide.hip). The forward
// writes out / out_prez / last_state / chunk_states / checkpoints as
// ak_selective_scan_fwd describes; with prep it is instead the backward's
// preparation pass (checkpoints and dz). The reverse pass fills the
// workspace partials that scan_bwd_finish sums.
int launch_scan_wide_fwd(const ScanParams& p, bool prep, int u_dtype, int delta_dtype,
                         int bc_dtype, hipStream_t s);
int launch_scan_wide_bwd(const ScanParams& p, int u_dtype, int delta_dtype, int bc_dtype,
                         hipStream_t s);
// The whole-tile reverse pass (selective_scan_bwd_fast.hip): launches it and
// returns true when the shape and layout qualify, else launches nothing. It
// may take 32 channels per workgroup, and then sets p.tiles_per_group to the
// number of dB / dC partial rows it wrote per group (the sums that follow
// read that many).
bool launch_scan_bwd_fast(ScanParams& p, int u_dtype, int delta_dtype, int bc_dtype,
                          hipStream_t s);

}  // namespace ak
