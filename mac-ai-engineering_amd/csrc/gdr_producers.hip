// The producers of the rule's inputs in the Qwen3.5 / Qwen3-Next linear-attention layer, for MI355X (gfx950):
//
//   convolution path  u[t, c] = sum_j w[c, j] x[t - 3 + j, c] (depthwise, causal, 4 taps, zero before the start),
//                     y = u sigmoid(u) rounded once, split into q, k (key_dim channels each) and v (value_dim);
//   gates             beta = sigmoid(b), g = -exp(A_log) softplus(a + dt_bias) (softplus's threshold 20).
//   (The reference's layer/_conv.py:1-24 and layer/_gates.py:1-13 state the same functions.)
//
// The convolution is an HBM stream: every input and output byte crosses once (the 3-row halos come again through L2).
// A lane owns a channel vector over consecutive time steps, all its input rows loaded at once, a wave 64 consecutive
// vectors: 4 channels over 8 steps in the forward (conv_fwd_kernel), 2 over 16 in the backward (conv_bwd_kernel; over few
// tiles 2 over 4, conv_bwd_few_kernel), which forms du = dy silu'(u) for its steps and the 3 after them in registers, dx
// from du's windows (one writer an element) and the taps' gradient's sums over its steps; a tile of 64 rows adds its
// blocks' sums in order through LDS, sum_columns_kernel the tiles' partials in tile order: deterministic.
// The gates are one pass each way, an element a lane; over many rows the backward's also forms its workgroups' sums of
// A_log's and dt_bias's gradients, which a second launch adds in a fixed order, over few a second pass takes a workgroup
// a head (gate_direct_rows).
#include <hip/hip_runtime.h>

#include "gdr_abi.h"
#include "gdr_common.h"

namespace gdr {

typedef _Float16 f16;

// ---- vectors of 2- or 4-byte elements, as floats ------------------------------------------------------------------
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

// The 32-bit words of N values of T (N * sizeof(T) a multiple of 4), and back.
template <typename T, int N>
__device__ __forceinline__ void to_words(const float (&x)[N], unsigned (&wd)[N * sizeof(T) / 4]) {
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < N; ++i) wd[i] = __float_as_uint(x[i]);
  } else {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      typedef T T2 __attribute__((ext_vector_type(2)));
      wd[i] = __builtin_bit_cast(unsigned, T2{(T)x[2 * i], (T)x[2 * i + 1]});   // one packed conversion
    }
  }
}
template <typename T, int N>
__device__ __forceinline__ void from_words(const unsigned (&wd)[N * sizeof(T) / 4], float (&x)[N]) {
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = __uint_as_float(wd[i]);
  } else {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      x[2 * i] = (float)__builtin_bit_cast(T, (unsigned short)(wd[i] & 0xffffu));
      x[2 * i + 1] = (float)__builtin_bit_cast(T, (unsigned short)(wd[i] >> 16));
    }
  }
}
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
// N floats written as T: N * sizeof(T) bytes (4, 8, 16 or 32) in 16-byte stores and at most one narrower one.
template <typename T, int N>
__device__ __forceinline__ void store_as(T* p, const float (&x)[N]) {
  constexpr int NW = N * (int)sizeof(T) / 4;
  static_assert(NW == 1 || NW % 2 == 0, "one word or whole 8-byte pieces");
  unsigned wd[NW];
  to_words<T, N>(x, wd);
  unsigned* q = reinterpret_cast<unsigned*>(p);
#pragma unroll
  for (int s = 0; s + 4 <= NW; s += 4)
    *reinterpret_cast<u32x4_t*>(q + s) = u32x4_t{wd[s], wd[s + 1], wd[s + 2], wd[s + 3]};
  if constexpr (NW % 4 == 2) *reinterpret_cast<u32x2_t*>(q + NW - 2) = u32x2_t{wd[NW - 2], wd[NW - 1]};
  if constexpr (NW == 1) *q = wd[0];
}
// N values of T from memory as floats, in one load of N * sizeof(T) bytes.
template <typename T, int N>
__device__ __forceinline__ void load_as(const T* p, float (&x)[N]) {
  constexpr int NW = N * (int)sizeof(T) / 4;
  typedef unsigned words_t __attribute__((ext_vector_type(NW)));
  const words_t r = *reinterpret_cast<const words_t*>(p);
  unsigned wd[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) wd[i] = r[i];
  from_words<T, N>(wd, x);
}

// ---- the convolution path ----------------------------------------------------------------------------------------
constexpr int CV_TAPS = 4;
constexpr int CV_ROWS = 64;       // time steps a tile of the backward
constexpr int CV_HALO = CV_TAPS - 1;

struct ConvArgs {
  const void* x;                  // [B, T, C] in T
  const void* w;                  // [C, 4] taps: the forward's in TW, the backward's float32
  float* taps;                    // forward: the taps' float32 copy for the backward, or null
  void *q, *k, *v;                // forward outputs: q, k [B, T, KD * REP] in T, v [B, T, C - 2 KD] in TV
  const void *dq, *dk, *dv;       // backward inputs, same layouts
  void* dx;                       // [B, T, C] in T
  float* part;                    // [B * ntiles, C * 4] per-tile taps' gradient, or null
  int B, T, C, KD, DK, REP, ntiles;
};

// Where a lane's channel vector (2 or 4 channels) lives among the outputs: q, k (key heads, each written REP times: REP =
// 1 keeps key heads only) or v.  A vector never straddles a head (head widths are multiples of 8).
struct Dest {
  int which;                      // 0 q, 1 k, 2 v
  unsigned pitch;                 // row pitch of the destination (elements)
  unsigned col;                   // the vector's first column there (copy 0)
  __device__ Dest(int c, int KD, int DK, int REP, int C) {
    if (c < 2 * KD) {
      which = c < KD ? 0 : 1;
      const int cc = c - which * KD;
      pitch = (unsigned)(KD * REP);
      col = (unsigned)((cc / DK) * REP * DK + cc % DK);
    } else {
      which = 2;
      pitch = (unsigned)(C - 2 * KD);
      col = (unsigned)(c - 2 * KD);
    }
  }
};

// The lane's taps, tap-major: tw[j][i] = w[c + i, j] for its N channels, w in TW.
template <typename TW, int N>
__device__ __forceinline__ void tile_taps(const void* w, int c, float (&tw)[CV_TAPS][N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float r[CV_TAPS];
    load_as<TW, CV_TAPS>((const TW*)w + (size_t)(c + i) * CV_TAPS, r);
#pragma unroll
    for (int j = 0; j < CV_TAPS; ++j) tw[j][i] = r[j];
  }
}

// sum_j tw[j][i] win[j][i], j = 3 first.  float32 inputs (EXACT) sum in double and round once, so that the result is
// within an ulp of the exact value (their error bar is twice PyTorch's fp32 path); 2-byte inputs sum in float, whose
// rounding is far below the output's.
template <bool EXACT, int N>
__device__ __forceinline__ float tap_dot(const float (&tw)[CV_TAPS][N], int i, float w0, float w1, float w2, float w3) {
  if constexpr (EXACT) {
    double s = (double)tw[3][i] * (double)w3;
    s = fma((double)tw[2][i], (double)w2, s);
    s = fma((double)tw[1][i], (double)w1, s);
    return (float)fma((double)tw[0][i], (double)w0, s);
  } else {
    return fmaf(tw[0][i], w0, fmaf(tw[1][i], w1, fmaf(tw[2][i], w2, tw[3][i] * w3)));
  }
}
// 1 / (1 + e) for e >= 0 (or NaN): the hardware reciprocal (1 ulp) and one Newton step, r + r (1 - d r), which rounds as
// the division does but for rare ties.  Formed at 1/16 of the scale: the instruction flushes subnormal results, and past
// e = 2^126 (u below -87.3) the quotient is one while u times it is not.  d is held finite, so an overflowed exponential
// still gives 0.  The division took a fifth of the backward's instructions; the results' errors against float64 are the
// same to four digits.
__device__ __forceinline__ float recip1p(float e) {
  const float d = fminf(fmaf(0.0625f, e, 0.0625f), 3.0e38f);
  const float r = __builtin_amdgcn_rcpf(d);
  return 0.0625f * fmaf(fmaf(-d, r, 1.0f), r, r);
}
template <bool EXACT>
__device__ __forceinline__ float logistic(float u) {
  if constexpr (EXACT) return 1.0f / (1.0f + expf(-u));
  else return recip1p(__expf(-u));
}
// u sigmoid(u) with one rounding after the exponential for float32 inputs (a division, not u times a rounded
// reciprocal, whose two roundings put the float32 output past twice PyTorch's silu error)
template <bool EXACT>
__device__ __forceinline__ float silu(float u) {
  if constexpr (EXACT) return u / (1.0f + expf(-u));
  else return u * recip1p(__expf(-u));
}

constexpr int CV_VE = 4;          // channels a lane
// The forward needs no staging: a lane owns 4 channels over 8 consecutive time steps and issues the loads of all its 11
// input rows at once (the 3 halo rows come again through L2), then forms each output from them.  A wave spans 64
// consecutive vectors of one block of steps (a wave-uniform start: row addresses are scalar and the ends of the row
// cost the other waves nothing), a workgroup four consecutive blocks.  Bound by its bytes once the chip is full: at
// B = 4, T = 1024, C = 6144 in bf16 (101 MB, 18 us at the card's copy rate) 19.9 us, at C = 8192 and T = 2048 (268 MB)
// 43.5 us, 6.2 TB/s.  Lanes of 8 channels (16-byte loads) took 25.0 and 51.5 us (half the waves, twice the registers),
// 4 or 16 steps 22.9-23.7 and 50.9-52.8; with a correctly rounded division in silu 28.8 and 61 us (of 23.0 and 49.9
// then).  The taps' type is a template argument: behind branches on its code 2-byte taps were waited for after all of x,
// 24.1 and 54.1 us (float32 x 39.7 against 34.6, 103 against 96).
constexpr int CV_FWD_STEPS = 8;
template <typename T, typename TV, typename TW>
__global__ void __launch_bounds__(256) conv_fwd_kernel(ConvArgs a) {
  constexpr int VE = CV_VE;
  constexpr bool EXACT = sizeof(T) == 4;
  constexpr int S = CV_FWD_STEPS, NR = S + CV_HALO;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = (blockIdx.x * 64 + lane) * VE;
  const int t0 = (blockIdx.y * 4 + wave) * S, b = blockIdx.z, Tn = a.T;   // t0: uniform in a wave
  if (c >= a.C || t0 >= Tn) return;
  typedef unsigned wordx_t __attribute__((ext_vector_type(VE * sizeof(T) / 4)));
  const int row0 = b * Tn;                 // B T C < 2^31
  float tw[CV_TAPS][VE];                   // the taps first: loads arrive in order, and every output needs them
  tile_taps<TW, VE>(a.w, c, tw);
  wordx_t xr[NR];                          // x[t0 - 3 + i], zero outside the sequence (see conv_bwd_kernel)
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int t = t0 - CV_HALO + i;
    const size_t row = (unsigned)(row0 + (t < 0 ? 0 : t < Tn ? t : Tn - 1));
    xr[i] = *reinterpret_cast<const wordx_t*>((const T*)a.x + row * a.C + c);
  }
  if (a.taps && t0 == 0 && b == 0)         // one wave a channel range
#pragma unroll
    for (int e = 0; e < VE; ++e)
      *reinterpret_cast<f4*>(a.taps + (size_t)(c + e) * CV_TAPS) = f4{tw[0][e], tw[1][e], tw[2][e], tw[3][e]};
  if (t0 < CV_HALO || t0 + S > Tn)
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (t0 - CV_HALO + i < 0 || t0 - CV_HALO + i >= Tn) xr[i] = wordx_t{};
  const Dest d(c, a.KD, a.DK, a.REP, a.C);
  float xw[CV_TAPS][VE];                   // x[t - 3 .. t], oldest first
#pragma unroll
  for (int i = 0; i < NR; ++i) {
#pragma unroll
    for (int j = 0; j + 1 < CV_TAPS; ++j)
#pragma unroll
      for (int e = 0; e < VE; ++e) xw[j][e] = xw[j + 1][e];
    unsigned wd[VE * sizeof(T) / 4];
#pragma unroll
    for (int e = 0; e < (int)(VE * sizeof(T) / 4); ++e) wd[e] = xr[i][e];
    from_words<T, VE>(wd, xw[3]);
    const int t = t0 + i - CV_HALO;
    if (i < CV_HALO || t >= Tn) continue;
    float y[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) y[e] = silu<EXACT>(tap_dot<EXACT, VE>(tw, e, xw[0][e], xw[1][e], xw[2][e], xw[3][e]));
    const size_t row = (unsigned)(row0 + t);
    if (d.which == 2) {
      store_as<TV, VE>((TV*)a.v + row * d.pitch + d.col, y);
    } else {
      T* dst = (T*)(d.which == 0 ? a.q : a.k) + row * d.pitch + d.col;
      for (int rep = 0; rep < a.REP; ++rep) store_as<T, VE>(dst + (size_t)rep * a.DK, y);
    }
  }
}

// du = dy s (1 + u (1 - s)), s = sigmoid(u).
template <bool EXACT>
__device__ __forceinline__ float silu_grad(float u, float dy) {
  const float sg = logistic<EXACT>(u);
  return dy * (sg * (1.0f + u * (1.0f - sg)));
}

// A tile's share of the taps' gradient: the blocks' double sums (block, then the tile's channels' taps) added in block
// order.  `out` is the tile's [C, 4]; o0 the workgroup's first element of it, n the elements there.
template <int SPAN, int BLOCKS, int THREADS>
__device__ __forceinline__ void add_blocks(const double (&red)[BLOCKS][SPAN], float* out, int o0, int n) {
  for (int o = threadIdx.x; o < SPAN && o0 + o < n; o += THREADS) {
    double sum = red[0][o];
#pragma unroll
    for (int w = 1; w < BLOCKS; ++w) sum += red[w][o];
    out[o0 + o] = (float)sum;
  }
}

// The backward, like the forward, streams: a lane owns 2 channels over S consecutive time steps t0 .. t0 + S - 1 and
// issues all its loads at once -- x[t0 - 3 .. t0 + S + 2] and the upstream gradient dy[t0 .. t0 + S + 2] (q's and k's
// copies summed in copy order) -- then walks the rows with everything in registers:
//   du[t] = dy s (1 + u (1 - s)), s = sigmoid(u)   (0 past the end), for its S rows and the 3 after them,
//   dx[t] = w0 du[t + 3] + w1 du[t + 2] + w2 du[t + 1] + w3 du[t],
//   part[tile][c, j] = sum over the tile's t of du[t] x[t - 3 + j], in double.
// A workgroup is one tile of 64 rows: 64 / S waves, a time block each, over the same 64 vectors, whose sums meet in
// LDS in wave order (deterministic).  S + 3 rows of du for S of dx: at S = 16 the recomputed rows cost a fifth of the
// activations.  Bound by its bytes and its VALU work, about as long: 151 MB at B = 4, T = 1024, C = 6144 in bf16 are 27
// us at the card's copy rate.  Measured there: 30.8 us, 35.9 with the taps' gradient; at C = 8192 and T = 2048 82 and 91;
// in float32 54 and 59 at the first size.  Lanes of 4 channels took 33.5 and 43.2, 84 and 107 in bf16 (239 registers, two
// waves a SIMD, against 124 and four), 8 steps of 2 channels 30.7 and 41.5, 90 and 111, in float32 61 and 68; a form that
// staged tiles of x and dy in LDS (three barriers, every row through LDS as float32 twice) 40.6 and 60.2, 109 and 160,
// in float32 63 and 75.
constexpr int CV_BWD_STEPS = 16, CV_BWD_VE = 2;
template <typename T, typename TV, bool TAPS>
__global__ void __launch_bounds__(64 * (CV_ROWS / CV_BWD_STEPS), 2) conv_bwd_kernel(ConvArgs a) {
  constexpr int VE = CV_BWD_VE, S = CV_BWD_STEPS, BLOCKS = CV_ROWS / S;
  constexpr bool EXACT = sizeof(T) == 4;
  constexpr int XR = S + 2 * CV_HALO, DR = S + CV_HALO;
  constexpr int SPAN = CV_TAPS * VE * 64;      // the taps' gradients of the tile's channels
  __shared__ __attribute__((aligned(16))) double red[TAPS ? BLOCKS : 1][TAPS ? SPAN : 1];   // a wave's sums a row
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cl = (blockIdx.x * 64 + lane) * VE;
  const bool on = cl < a.C;                // lanes past the channels repeat the last vector and store nothing
  const int c = on ? cl : a.C - VE;
  const int t0 = blockIdx.y * CV_ROWS + wave * S, b = blockIdx.z, Tn = a.T;   // t0: uniform in a wave
  const int row0 = b * Tn;                 // B T C < 2^31
  typedef unsigned wordx_t __attribute__((ext_vector_type(VE * sizeof(T) / 4)));
  typedef unsigned wordv_t __attribute__((ext_vector_type(VE * sizeof(TV) / 4)));
  double acc[VE][CV_TAPS];
#pragma unroll
  for (int i = 0; i < VE; ++i)
#pragma unroll
    for (int j = 0; j < CV_TAPS; ++j) acc[i][j] = 0.0;
  if (t0 < Tn) {                           // the waves past the end only join the sums
    // rows outside the sequence read a row inside it, so that every load is unconditional; the waves that have such
    // rows (their first or last block) zero them after
    const bool edge = t0 < CV_HALO || t0 + DR > Tn;
    auto row_of = [&](int t) { return (size_t)(unsigned)(row0 + (t < 0 ? 0 : t < Tn ? t : Tn - 1)); };
    wordx_t xr[XR];                        // x[t0 - 3 + i]
#pragma unroll
    for (int i = 0; i < XR; ++i)
      xr[i] = *reinterpret_cast<const wordx_t*>((const T*)a.x + row_of(t0 - CV_HALO + i) * a.C + c);
    const Dest d(c, a.KD, a.DK, a.REP, a.C);
    float g[DR][VE];                       // dy[t0 + i]
    if (d.which == 2) {
      const TV* src = (const TV*)a.dv + d.col;
      wordv_t r[DR];
#pragma unroll
      for (int i = 0; i < DR; ++i) r[i] = *reinterpret_cast<const wordv_t*>(src + row_of(t0 + i) * d.pitch);
#pragma unroll
      for (int i = 0; i < DR; ++i) {
        unsigned wd[VE * sizeof(TV) / 4];
#pragma unroll
        for (int e = 0; e < (int)(VE * sizeof(TV) / 4); ++e) wd[e] = r[i][e];
        from_words<TV, VE>(wd, g[i]);
      }
    } else {
      const T* src = (const T*)(d.which == 0 ? a.dq : a.dk) + d.col;
      for (int rep = 0; rep < a.REP; ++rep, src += a.DK) {   // a repeated key head's copies, added in copy order
        wordx_t r[DR];
#pragma unroll
        for (int i = 0; i < DR; ++i) r[i] = *reinterpret_cast<const wordx_t*>(src + row_of(t0 + i) * d.pitch);
#pragma unroll
        for (int i = 0; i < DR; ++i) {
          unsigned wd[VE * sizeof(T) / 4];
          float h[VE];
#pragma unroll
          for (int e = 0; e < (int)(VE * sizeof(T) / 4); ++e) wd[e] = r[i][e];
          from_words<T, VE>(wd, h);
#pragma unroll
          for (int e = 0; e < VE; ++e) g[i][e] = rep ? g[i][e] + h[e] : h[e];
        }
      }
    }
    if (edge) {
#pragma unroll
      for (int i = 0; i < XR; ++i)
        if (t0 - CV_HALO + i < 0 || t0 - CV_HALO + i >= Tn) xr[i] = wordx_t{};
#pragma unroll
      for (int i = 0; i < DR; ++i)
        if (t0 + i >= Tn)
#pragma unroll
          for (int e = 0; e < VE; ++e) g[i][e] = 0.f;
    }
    float tw[CV_TAPS][VE];
    tile_taps<float, VE>(a.w, c, tw);
    T* dxb = (T*)a.dx + (size_t)row0 * a.C + c;
    float xw[CV_TAPS][VE], dw[CV_TAPS][VE];   // x[t - 3 .. t] and du[t - 3 .. t], oldest first
#pragma unroll
    for (int j = 1; j < CV_TAPS; ++j) {       // x[t0 - 3 .. t0 - 1] in places 1 .. 3
      unsigned wd[VE * sizeof(T) / 4];
#pragma unroll
      for (int e = 0; e < (int)(VE * sizeof(T) / 4); ++e) wd[e] = xr[j - 1][e];
      from_words<T, VE>(wd, xw[j]);
    }
#pragma unroll
    for (int s = 0; s < DR; ++s) {
      if (t0 + s - CV_HALO >= Tn) break;   // past the end: du is 0 and there is no dx
#pragma unroll
      for (int j = 0; j + 1 < CV_TAPS; ++j)
#pragma unroll
        for (int i = 0; i < VE; ++i) {
          xw[j][i] = xw[j + 1][i];
          if (s) dw[j][i] = dw[j + 1][i];
        }
      unsigned wd[VE * sizeof(T) / 4];
#pragma unroll
      for (int e = 0; e < (int)(VE * sizeof(T) / 4); ++e) wd[e] = xr[s + CV_HALO][e];
      from_words<T, VE>(wd, xw[3]);
#pragma unroll
      for (int i = 0; i < VE; ++i) {
        const float uu = tap_dot<EXACT, VE>(tw, i, xw[0][i], xw[1][i], xw[2][i], xw[3][i]);
        dw[3][i] = silu_grad<EXACT>(uu, g[s][i]);
      }
      if (TAPS && s < S)
#pragma unroll
        for (int i = 0; i < VE; ++i) {
          const double dd = (double)dw[3][i];
#pragma unroll
          for (int j = 0; j < CV_TAPS; ++j) acc[i][j] = fma(dd, (double)xw[j][i], acc[i][j]);
        }
      if (s >= CV_HALO && on) {
        float o[VE];
#pragma unroll
        for (int i = 0; i < VE; ++i) o[i] = tap_dot<EXACT, VE>(tw, i, dw[3][i], dw[2][i], dw[1][i], dw[0][i]);
        store_as<T, VE>(dxb + (size_t)(t0 + s - CV_HALO) * a.C, o);
      }
    }
  }
  if constexpr (TAPS) {
    double* mine = &red[wave][lane * VE * CV_TAPS];
#pragma unroll
    for (int i = 0; i < VE; ++i)
#pragma unroll
      for (int j = 0; j < CV_TAPS; ++j) mine[i * CV_TAPS + j] = acc[i][j];
    __syncthreads();
    add_blocks<SPAN, BLOCKS, 64 * BLOCKS>(red, a.part + (size_t)(b * a.ntiles + blockIdx.y) * a.C * CV_TAPS,
                                          blockIdx.x * SPAN, a.C * CV_TAPS);
  }
}

// The same over few tiles (conv_few), where the form above leaves compute units idle and a lane's 19 rows in turn are the
// time: a workgroup is a tile of 64 rows by 16 vectors, a lane 4 steps of one, and the 3 rows of du after a lane's own
// come through LDS from the lanes that own them (the rows after the tile are formed by its first three blocks of steps).
// Every element's arithmetic is the form's above: dx has the same bits; the taps' sums group by 4 rows.  Bound by
// latency: one row of 64 tokens, C = 6144, with the taps' gradient 6.4 us in bf16 and 6.8 in float32, of which the second
// stage's launch is 2.3, against 8.5 and 10.2 of the form above (the LDS form 9.3 and 7.6).  Tiles 8 or 32 vectors wide
// and 8 steps a lane are slower over few tiles.
constexpr int CV_FEW_STEPS = 4, CV_FEW_WIDE = 16;
template <typename T, typename TV, bool TAPS>
__global__ void __launch_bounds__(CV_FEW_WIDE * (CV_ROWS / CV_FEW_STEPS)) conv_bwd_few_kernel(ConvArgs a) {
  constexpr int VE = CV_BWD_VE, S = CV_FEW_STEPS, WIDE = CV_FEW_WIDE, BLOCKS = CV_ROWS / S;
  constexpr bool EXACT = sizeof(T) == 4;
  constexpr int XR = S + CV_HALO, SPAN = CV_TAPS * VE * WIDE;
  static_assert(S > CV_HALO && BLOCKS > CV_HALO, "a block holds the next one's halo, the first blocks the tile's");
  __shared__ __attribute__((aligned(16))) double red[TAPS ? BLOCKS : 1][TAPS ? SPAN : 1];
  __shared__ float head[BLOCKS + 1][CV_HALO][WIDE][VE];   // du of each block's first rows; then the rows after the tile
  const int vec = threadIdx.x % WIDE, block = threadIdx.x / WIDE;
  const int cl = (blockIdx.x * WIDE + vec) * VE;
  const bool on = cl < a.C;                // lanes past the channels repeat the last vector and store nothing
  const int c = on ? cl : a.C - VE;
  const int b = blockIdx.z, Tn = a.T, end = (blockIdx.y + 1) * CV_ROWS, t0 = blockIdx.y * CV_ROWS + block * S;
  const int row0 = b * Tn;                 // B T C < 2^31
  auto row_of = [&](int t) { return (size_t)(unsigned)(row0 + (t < 0 ? 0 : t < Tn ? t : Tn - 1)); };
  const Dest d(c, a.KD, a.DK, a.REP, a.C);
  // x[t0 - 3 + i], dy[t0 + i] and the row after the tile that the first blocks form, du[end + block]; loads are of rows
  // inside the sequence, masked after
  float xr[XR][VE], g[S][VE], ex[CV_TAPS][VE], eg[VE];
  const bool extra = block < CV_HALO;
  auto load_x = [&](int t, float (&r)[VE]) { load_as<T, VE>((const T*)a.x + row_of(t) * a.C + c, r); };
  auto mask = [&](int t, float (&r)[VE]) {
#pragma unroll
    for (int i = 0; i < VE; ++i) r[i] = t >= 0 && t < Tn ? r[i] : 0.f;
  };
  float du[S + CV_HALO][VE], tw[CV_TAPS][VE];
#pragma unroll
  for (int i = 0; i < XR; ++i) load_x(t0 - CV_HALO + i, xr[i]);
  if (extra)
#pragma unroll
    for (int j = 0; j < CV_TAPS; ++j) load_x(end + block - CV_HALO + j, ex[j]);
  if (d.which == 2) {
    const TV* src = (const TV*)a.dv + d.col;
#pragma unroll
    for (int i = 0; i < S; ++i) load_as<TV, VE>(src + row_of(t0 + i) * d.pitch, g[i]);
    if (extra) load_as<TV, VE>(src + row_of(end + block) * d.pitch, eg);
  } else {
    const T* src = (const T*)(d.which == 0 ? a.dq : a.dk) + d.col;
#pragma unroll
    for (int i = 0; i < S; ++i) load_as<T, VE>(src + row_of(t0 + i) * d.pitch, g[i]);
    if (extra) load_as<T, VE>(src + row_of(end + block) * d.pitch, eg);
    for (int rep = 1; rep < a.REP; ++rep) {   // a repeated key head's copies, added in copy order
      float h[S][VE], eh[VE];
      src += a.DK;
#pragma unroll
      for (int i = 0; i < S; ++i) load_as<T, VE>(src + row_of(t0 + i) * d.pitch, h[i]);
      if (extra) load_as<T, VE>(src + row_of(end + block) * d.pitch, eh);
#pragma unroll
      for (int e = 0; e < VE; ++e) {
#pragma unroll
        for (int i = 0; i < S; ++i) g[i][e] += h[i][e];
        if (extra) eg[e] += eh[e];
      }
    }
  }
  tile_taps<float, VE>(a.w, c, tw);
#pragma unroll
  for (int i = 0; i < XR; ++i) mask(t0 - CV_HALO + i, xr[i]);
#pragma unroll
  for (int i = 0; i < S; ++i) mask(t0 + i, g[i]);
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int i = 0; i < VE; ++i) {
      du[s][i] = silu_grad<EXACT>(tap_dot<EXACT, VE>(tw, i, xr[s][i], xr[s + 1][i], xr[s + 2][i], xr[s + 3][i]), g[s][i]);
      if (s < CV_HALO) head[block][s][vec][i] = du[s][i];
    }
  if (extra) {
#pragma unroll
    for (int j = 0; j < CV_TAPS; ++j) mask(end + block - CV_HALO + j, ex[j]);
    mask(end + block, eg);
#pragma unroll
    for (int i = 0; i < VE; ++i) {
      const float u = tap_dot<EXACT, VE>(tw, i, ex[0][i], ex[1][i], ex[2][i], ex[3][i]);
      head[BLOCKS][block][vec][i] = silu_grad<EXACT>(u, eg[i]);
    }
  }
  if constexpr (TAPS) {
#pragma unroll
    for (int i = 0; i < VE; ++i)
#pragma unroll
      for (int j = 0; j < CV_TAPS; ++j) {
        double sum = 0.0;
#pragma unroll
        for (int s = 0; s < S; ++s) sum = fma((double)du[s][i], (double)xr[s + j][i], sum);
        red[block][(vec * VE + i) * CV_TAPS + j] = sum;
      }
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < CV_HALO; ++s)
#pragma unroll
    for (int i = 0; i < VE; ++i) du[S + s][i] = head[block + 1][s][vec][i];
  T* dxb = (T*)a.dx + (size_t)row0 * a.C + c;
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (on && t0 + s < Tn) {
      float o[VE];
#pragma unroll
      for (int i = 0; i < VE; ++i) o[i] = tap_dot<EXACT, VE>(tw, i, du[s + 3][i], du[s + 2][i], du[s + 1][i], du[s][i]);
      store_as<T, VE>(dxb + (size_t)(t0 + s) * a.C, o);
    }
  if constexpr (TAPS)
    add_blocks<SPAN, BLOCKS, WIDE * BLOCKS>(red, a.part + (size_t)(b * a.ntiles + blockIdx.y) * a.C * CV_TAPS,
                                            blockIdx.x * SPAN, a.C * CV_TAPS);
}

// x at element i of an array in the type of code t (uniform), and back.
__device__ __forceinline__ void store_code(void* p, int t, size_t i, float x) {
  if (t == MACAI_GDR_F32) ((float*)p)[i] = x;
  else if (t == MACAI_GDR_BF16) ((bf16*)p)[i] = (bf16)x;
  else ((f16*)p)[i] = (f16)x;
}
__device__ __forceinline__ float load_code(const void* p, int t, size_t i) {
  if (t == MACAI_GDR_F32) return ((const float*)p)[i];
  if (t == MACAI_GDR_BF16) return (float)((const bf16*)p)[i];
  return (float)((const f16*)p)[i];
}

// out[i] = the sum over rows p = 0 .. P - 1 of in[p * n + i], in double, rounded to float32 and then to the type of code
// ot: the fixed-order second stage of the taps' gradient.  A workgroup takes 64 outputs; each of its waves sums a quarter
// of the rows in row order, eight rows' loads in flight together, and the quarters add in order.
__global__ void __launch_bounds__(256) sum_columns_kernel(const float* in, void* out, int ot, int P, int n) {
  __shared__ double quarter[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
  const int per = (P + 3) / 4, hi = min(P, (w + 1) * per);
  double s = 0.0;
  if (i < n) {
    int p = w * per;
    for (; p + 8 <= hi; p += 8) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = in[(size_t)(p + e) * n + i];
#pragma unroll
      for (int e = 0; e < 8; ++e) s += (double)v[e];
    }
    for (; p < hi; ++p) s += (double)in[(size_t)p * n + i];
  }
  quarter[w][lane] = s;
  __syncthreads();
  if (w == 0 && i < n)
    store_code(out, ot, i, (float)(((quarter[0][lane] + quarter[1][lane]) + quarter[2][lane]) + quarter[3][lane]));
}

// ---- the gates -----------------------------------------------------------------------------------------------------
// PyTorch's softplus with threshold 20: x above it, log1p(exp(x)) below; and its derivative with the same
// threshold: 1 above it, sigmoid(x) below.  The gates compute in double, a + dt_bias included, and round each result
// once: they are a few elements a token-head, so the kernels are bound by latency, and in float32 the sums', the
// exponentials' and the quotients' roundings put the gradients at up to twice the PyTorch path's error on short
// rows.
__device__ __forceinline__ double softplus_t20(double x) { return x > 20.0 ? x : log1p(exp(x)); }
__device__ __forceinline__ double softplus_t20_grad(double x) { return x > 20.0 ? 1.0 : 1.0 / (1.0 + exp(-x)); }

// The gates move under a megabyte per layer, so they are bound by latency, not bandwidth: one element a lane, so
// that a layer's elements spread over every lane of the chip and each lane runs one exponential chain.  TYPED: A_log and
// dt_bias are read in the types of codes ta, td, and with `params` non-null the first lanes write their float32 copies
// ([2, H]) there; otherwise both are float32 (the branches on the codes cost 0.1 us of 2.4).
constexpr int GATE_THREADS = 256;
struct GateParams {
  const void *alog, *dtb;
  int ta, td;                                // dtype codes
};
template <typename T, bool TYPED>
__global__ void __launch_bounds__(GATE_THREADS) gates_fwd_kernel(const T* b, const T* a, GateParams p, float* params,
                                                                 float* beta, float* g, int64_t n, int H) {
  const int64_t i = (int64_t)blockIdx.x * GATE_THREADS + threadIdx.x;
  if (i >= n) return;
  const int head = (int)(i % H);             // heads run fastest: element i is head i mod H
  float alog, dtb;
  if constexpr (TYPED) {
    alog = load_code(p.alog, p.ta, head);
    dtb = load_code(p.dtb, p.td, head);
    if (params && i < H) {                   // n is a multiple of H
      params[i] = alog;
      params[H + i] = dtb;
    }
  } else {
    alog = ((const float*)p.alog)[head];
    dtb = ((const float*)p.dtb)[head];
  }
  const double rate = -exp((double)alog);
  beta[i] = (float)(1.0 / (1.0 + exp(-(double)(float)b[i])));
  g[i] = (float)(rate * softplus_t20((double)(float)a[i] + (double)dtb));
}

// db = dbeta s (1 - s), s = sigmoid(b); da = dg (-exp(A_log)) softplus'(a + dt_bias).
template <typename T>
__global__ void __launch_bounds__(GATE_THREADS) gates_bwd_kernel(const T* b, const T* a, const float* alog,
                                                                 const float* dtb, const float* dbeta,
                                                                 const float* dg, T* db, T* da, int64_t n, int H) {
  const int64_t i = (int64_t)blockIdx.x * GATE_THREADS + threadIdx.x;
  if (i >= n) return;
  const int head = (int)(i % H);
  const double rate = -exp((double)alog[head]);
  const double sig = 1.0 / (1.0 + exp(-(double)(float)b[i]));
  db[i] = (T)(float)((double)dbeta[i] * (sig - sig * sig));          // d sigmoid = s (1 - s)
  da[i] = (T)(float)((double)dg[i] * rate * softplus_t20_grad((double)(float)a[i] + (double)dtb[head]));
}

// The same pass with each workgroup's sums, per head, of the parameters' gradients' terms (dA_log: dg g; ddt_bias: da
// before its rounding), in double, to part[group][2][H].  A workgroup takes `per` whole rows of min(H, 256) heads
// (block % hblocks says which heads): thread i takes head i % H of row i / H and then every rpp-th row (rpp = 256 / H
// rows at once), its own sums in row order, and the rpp sums of a head add in order through LDS: deterministic.
// gates_params_kernel adds the groups' in order.  Bound by the chain of double exponentials, so it is spread over every
// CU: see gate_direct_rows for what it is measured against.
template <typename T>
__global__ void __launch_bounds__(GATE_THREADS) gates_bwd_sums_kernel(const T* b, const T* a, const float* alog,
                                                                      const float* dtb, const float* dbeta,
                                                                      const float* dg, T* db, T* da, double* part,
                                                                      int64_t rows, int H, int per, int hblocks) {
  __shared__ double red[2][GATE_THREADS];
  const int64_t group = blockIdx.x / hblocks;
  const int64_t r0 = group * per, r1 = r0 + per < rows ? r0 + per : rows;
  const int rpp = H < GATE_THREADS ? GATE_THREADS / H : 1;   // rows at once
  const int sub = H < GATE_THREADS ? threadIdx.x / H : 0;
  const int h = H < GATE_THREADS ? threadIdx.x % H : blockIdx.x % hblocks * GATE_THREADS + threadIdx.x;
  double s_a = 0.0, s_d = 0.0;
  if (sub < rpp && h < H) {
    const double rate = -exp((double)alog[h]), bias = (double)dtb[h];
    for (int64_t r = r0 + sub; r < r1; r += rpp) {
      const int64_t i = r * H + h;
      const double sig = 1.0 / (1.0 + exp(-(double)(float)b[i]));
      db[i] = (T)(float)((double)dbeta[i] * (sig - sig * sig));
      const double x = (double)(float)a[i] + bias, gr = (double)dg[i] * rate, dx = gr * softplus_t20_grad(x);
      da[i] = (T)(float)dx;
      s_a = fma(gr, softplus_t20(x), s_a);
      s_d += dx;
    }
  }
  red[0][threadIdx.x] = s_a;
  red[1][threadIdx.x] = s_d;
  __syncthreads();
  if (sub == 0 && h < H) {
    for (int k = 1; k < rpp; ++k) {
      s_a += red[0][k * H + h];
      s_d += red[1][k * H + h];
    }
    double* out = part + (size_t)group * 2 * H;
    out[h] = s_a;
    out[H + h] = s_d;
  }
}

// dA_log[h] and ddt_bias[h]: the groups' sums of gates_bwd_sums_kernel added in double, rounded to float32 and then to
// the gradients' types.  A wave a head: lane l adds groups l, l + 64, ... in order, then the lanes add by a fixed
// butterfly.
__global__ void __launch_bounds__(64) gates_params_kernel(const double* part, void* dA, void* ddt, int ta, int td,
                                                          int groups, int H) {
  const int h = blockIdx.x;
  double s_a = 0.0, s_d = 0.0;
  for (int w = threadIdx.x; w < groups; w += 64) {
    s_a += part[(size_t)w * 2 * H + h];
    s_d += part[(size_t)w * 2 * H + H + h];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s_a += __shfl_xor(s_a, off, 64);
    s_d += __shfl_xor(s_d, off, 64);
  }
  if (threadIdx.x == 0) {
    store_code(dA, ta, h, (float)s_a);
    store_code(ddt, td, h, (float)s_d);
  }
}

// The parameters' gradients without scratch, beside gates_bwd_kernel: one workgroup a head; thread i takes rows i,
// i + 256, ... in order, then a wave sums its lanes by a fixed butterfly and the four waves add in order.
// Deterministic.  Terms and sums in double, rounded to float32 and then to the gradients' types: a head's rows of dg
// carry both signs, so the sums can cancel.
template <typename T>
__global__ void __launch_bounds__(256) gates_params_direct_kernel(const T* a, const float* alog, const float* dtb,
                                                                  const float* dg, void* dA, void* ddt, int ta, int td,
                                                                  int64_t rows, int H) {
  const int h = blockIdx.x;
  const double rate = -exp((double)alog[h]), bias = (double)dtb[h];
  double s_a = 0.0, s_d = 0.0;
  for (int64_t r = threadIdx.x; r < rows; r += 256) {
    const int64_t i = r * H + h;
    const double x = (double)(float)a[i] + bias, gv = (double)dg[i];
    s_a = fma(gv, rate * softplus_t20(x), s_a);
    s_d = fma(gv, rate * softplus_t20_grad(x), s_d);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s_a += __shfl_xor(s_a, off, 64);
    s_d += __shfl_xor(s_d, off, 64);
  }
  __shared__ double wa[4], wd[4];
  if ((threadIdx.x & 63) == 0) {
    wa[threadIdx.x >> 6] = s_a;
    wd[threadIdx.x >> 6] = s_d;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    store_code(dA, ta, h, (float)(((wa[0] + wa[1]) + wa[2]) + wa[3]));
    store_code(ddt, td, h, (float)(((wd[0] + wd[1]) + wd[2]) + wd[3]));
  }
}

}  // namespace gdr

using namespace gdr;

namespace {

int check_conv(const char* what, int64_t B, int64_t T, int64_t C, int64_t KD, int64_t DK, int64_t REP, int64_t DV,
               int32_t dtype, int32_t vdtype) {
  constexpr int64_t T_MAX = (int64_t)65535 * 4 * CV_FWD_STEPS;   // the forward's grid rows of time blocks
  if (B < 1 || T < 1 || B > 65535 || T > T_MAX)
    return fail(MACAI_GDR_EINVAL, "%s: B in [1, 65535] and T in [1, %lld] (got %lld, %lld)", what, (long long)T_MAX,
                (long long)B, (long long)T);
  if (dtype < MACAI_GDR_F32 || dtype > MACAI_GDR_F16 || vdtype < MACAI_GDR_F32 || vdtype > MACAI_GDR_F16)
    return fail(MACAI_GDR_EUNSUP, "%s: dtype codes must be F32, BF16 or F16", what);
  const int64_t VD = C - 2 * KD;
  if (KD < 1 || DK < 1 || DV < 1 || REP < 1 || VD < 1 || KD % DK || VD % DV || KD % 8 || DK % 8 || DV % 8 || C % 8)
    return fail(MACAI_GDR_EINVAL,
                "%s: need key_dim a multiple of the key head width, value_dim = C - 2 key_dim a multiple of the value "
                "head width, all multiples of 8 (got C %lld, key_dim %lld, DK %lld, DV %lld, REP %lld)",
                what, (long long)C, (long long)KD, (long long)DK, (long long)DV, (long long)REP);
  if (REP != 1 && (KD / DK) * REP != VD / DV)
    return fail(MACAI_GDR_EINVAL, "%s: REP must be 1 (key heads only) or value heads / key heads (%lld)", what,
                (long long)(VD / DV / (KD / DK)));
  if (B * T * C >= (int64_t)1 << 31 || B * T * KD * REP >= (int64_t)1 << 31)
    return fail(MACAI_GDR_EINVAL, "%s: tensors past 2^31 elements are not supported", what);
  return MACAI_GDR_OK;
}

// Up to this many rows the parameters' gradients come from gates_params_direct_kernel (a workgroup a head), whose
// chain is then the shorter one; past them from gates_bwd_sums_kernel and gates_params_kernel.  Where the two cross, with
// the pass over the elements in each: at 8 to 64 heads 500 to 650 rows (16 heads: 5.7 against 6.2 us at 64, 7.6 against
// 6.4 at 1,024, 14.6 against 7.6 at 4,096).  Few heads make the sums' LDS chain of 256 / H rows long: 1 head crosses at
// 2,050 rows, 2 at 1,050, 3 to 7 at 500 to 750.  Many spread the direct form over the chip: 65 cross at 2,050, 96 and 128 at
// 2,600, 192 and 256 at 2,900 to 3,300, more than 256 between 2,500 and 4,100.
int64_t gate_direct_rows(int64_t H) {
  if (H <= 2) return 2048 / H;
  return H <= 64 ? 576 : H <= 256 ? 2560 : 4096;
}

// The groups of rows that gates_bwd_sums_kernel's workgroups take, `per` rows each: one pass of rows a workgroup (an
// element a lane) up to 512 groups, then as many passes as keep to that (the second stage adds the groups' sums).
int64_t gate_groups(int64_t rows, int64_t H, int64_t* per) {
  const int64_t rpp = H < GATE_THREADS ? GATE_THREADS / H : 1;
  *per = rpp * ((rows + rpp * 512 - 1) / (rpp * 512));
  return (rows + *per - 1) / *per;
}

int64_t conv_tiles(int64_t T) { return (T + CV_ROWS - 1) / CV_ROWS; }

// Up to this many workgroups of conv_bwd_kernel the backward takes conv_bwd_few_kernel.  Where the two cross, without and
// with the taps' gradient, at 64 rows or more: in bf16 7.3 against 8.1 us and 11.1 against 11.8 at 384 workgroups, 9.6
// against 8.3 and 14.2 against 11.9 at 512; in float32 (more arithmetic a byte: the recomputed rows weigh more) 20.0
// against 22.0 and 24.7 against 25.4 at 1,024, 35.0 against 36.0 and 39 against 40 at 2,048, 71 against 54 and 75 against
// 59 at 3,072.  Rows shorter than a tile leave its lanes idle in the one form and only waves that exit at once in the
// other: in float32 at T = 16 5.0 against 7.0 at 128 workgroups, 10.0 against 8.1 at 512; at T = 1 about even up to 128.
int64_t conv_few(int64_t T, int32_t dtype) {
  if (dtype != MACAI_GDR_F32) return 384;
  return 256 * (T >= CV_ROWS ? CV_ROWS / CV_BWD_STEPS : (T + CV_BWD_STEPS - 1) / CV_BWD_STEPS);
}

}  // namespace

#define DISPATCH_PT(code, ...)                                             \
  switch (code) {                                                          \
    case MACAI_GDR_F32: { using PT = float; __VA_ARGS__; } break;          \
    case MACAI_GDR_BF16: { using PT = gdr::bf16; __VA_ARGS__; } break;     \
    default: { using PT = gdr::f16; __VA_ARGS__; } break;                  \
  }
#define DISPATCH_PV(code, ...)                                             \
  switch (code) {                                                          \
    case MACAI_GDR_F32: { using PV = float; __VA_ARGS__; } break;          \
    case MACAI_GDR_BF16: { using PV = gdr::bf16; __VA_ARGS__; } break;     \
    default: { using PV = gdr::f16; __VA_ARGS__; } break;                  \
  }
#define DISPATCH_PW(code, ...)                                             \
  switch (code) {                                                          \
    case MACAI_GDR_F32: { using PW = float; __VA_ARGS__; } break;          \
    case MACAI_GDR_BF16: { using PW = gdr::bf16; __VA_ARGS__; } break;     \
    default: { using PW = gdr::f16; __VA_ARGS__; } break;                  \
  }

extern "C" {

int macai_gdr_conv_fwd(const void* x, const float* w, void* q, void* k, void* v, int64_t B, int64_t T, int64_t C,
                       int64_t KD, int64_t DK, int64_t REP, int64_t DV, int32_t dtype, int32_t vdtype, void* stream) {
  return macai_gdr_conv_fwd_typed(x, w, MACAI_GDR_F32, nullptr, q, k, v, B, T, C, KD, DK, REP, DV, dtype, vdtype, stream);
}

int macai_gdr_conv_fwd_typed(const void* x, const void* w, int32_t wdtype, float* taps, void* q, void* k, void* v,
                             int64_t B, int64_t T, int64_t C, int64_t KD, int64_t DK, int64_t REP, int64_t DV,
                             int32_t dtype, int32_t vdtype, void* stream) {
  const char* what = "macai_gdr_conv_fwd";
  if (wdtype < MACAI_GDR_F32 || wdtype > MACAI_GDR_F16)
    return fail(MACAI_GDR_EUNSUP, "%s: dtype codes must be F32, BF16 or F16", what);
  if (int rc = check_conv(what, B, T, C, KD, DK, REP, DV, dtype, vdtype)) return rc;
  if (!x || !w || !q || !k || !v) return fail(MACAI_GDR_EINVAL, "%s: null pointer", what);
  const void* ps[] = {x, w, taps, q, k, v};
  for (const void* p : ps)
    if (!aligned16(p)) return fail(MACAI_GDR_EINVAL, "%s: pointers must be 16-byte aligned", what);
  ConvArgs a{x, w, taps, q, k, v, nullptr, nullptr, nullptr, nullptr, nullptr, (int)B, (int)T, (int)C, (int)KD, (int)DK,
             (int)REP, (int)conv_tiles(T)};
  hipStream_t st = (hipStream_t)stream;
  const int64_t steps = 4 * CV_FWD_STEPS, span = 64 * CV_VE;
  const dim3 grid((unsigned)((C + span - 1) / span), (unsigned)((T + steps - 1) / steps), (unsigned)B);
  DISPATCH_PT(dtype, DISPATCH_PV(vdtype, DISPATCH_PW(wdtype, hipLaunchKernelGGL((conv_fwd_kernel<PT, PV, PW>), grid,
                                                                                dim3(256), 0, st, a))))
  return launched(what);
}

int macai_gdr_conv_bwd(const void* x, const float* w, const void* dq, const void* dk, const void* dv, void* dx,
                       float* dwp, float* dw, int64_t B, int64_t T, int64_t C, int64_t KD, int64_t DK, int64_t REP,
                       int64_t DV, int32_t dtype, int32_t vdtype, void* stream) {
  return macai_gdr_conv_bwd_typed(x, w, dq, dk, dv, dx, dwp, dw, MACAI_GDR_F32, B, T, C, KD, DK, REP, DV, dtype, vdtype,
                                  stream);
}

int macai_gdr_conv_bwd_typed(const void* x, const float* w, const void* dq, const void* dk, const void* dv, void* dx,
                             float* dwp, void* dw, int32_t wdtype, int64_t B, int64_t T, int64_t C, int64_t KD,
                             int64_t DK, int64_t REP, int64_t DV, int32_t dtype, int32_t vdtype, void* stream) {
  const char* what = "macai_gdr_conv_bwd";
  if (wdtype < MACAI_GDR_F32 || wdtype > MACAI_GDR_F16)
    return fail(MACAI_GDR_EUNSUP, "%s: dtype codes must be F32, BF16 or F16", what);
  if (int rc = check_conv(what, B, T, C, KD, DK, REP, DV, dtype, vdtype)) return rc;
  if (!x || !w || !dq || !dk || !dv || !dx) return fail(MACAI_GDR_EINVAL, "%s: null pointer", what);
  if (!dwp != !dw) return fail(MACAI_GDR_EINVAL, "%s: dwp and dw go together (both or neither)", what);
  const void* ps[] = {x, w, dq, dk, dv, dx, dwp};
  for (const void* p : ps)
    if (!aligned16(p)) return fail(MACAI_GDR_EINVAL, "%s: pointers must be 16-byte aligned", what);
  const int ntiles = (int)conv_tiles(T);
  ConvArgs a{x, w, nullptr, nullptr, nullptr, nullptr, dq, dk, dv, dx, dwp, (int)B, (int)T, (int)C, (int)KD, (int)DK,
             (int)REP, ntiles};
  hipStream_t st = (hipStream_t)stream;
  const int64_t wide = 64 * CV_BWD_VE;     // channels a workgroup of the streaming form takes
  const bool few = (C + wide - 1) / wide * ntiles * B <= conv_few(T, dtype);
  const int64_t span = few ? CV_FEW_WIDE * CV_BWD_VE : wide;
  const dim3 grid((unsigned)((C + span - 1) / span), (unsigned)ntiles, (unsigned)B);
  const dim3 threads(few ? CV_FEW_WIDE * (CV_ROWS / CV_FEW_STEPS) : 64 * (CV_ROWS / CV_BWD_STEPS));
#define CONV_BWD(TAPS)                                                                          \
  DISPATCH_PT(dtype, DISPATCH_PV(vdtype, {                                                      \
    if (few) hipLaunchKernelGGL((conv_bwd_few_kernel<PT, PV, TAPS>), grid, threads, 0, st, a);  \
    else hipLaunchKernelGGL((conv_bwd_kernel<PT, PV, TAPS>), grid, threads, 0, st, a);          \
  }))
  if (dwp) {
    CONV_BWD(true)
  } else {
    CONV_BWD(false)
  }
#undef CONV_BWD
  if (int rc = launched(what)) return rc;
  if (dw) {
    const int n = (int)(C * CV_TAPS);
    hipLaunchKernelGGL(sum_columns_kernel, dim3((unsigned)((n + 63) / 64)), dim3(256), 0, st, dwp, dw,
                       wdtype, (int)(B * ntiles), n);
    return launched(what);
  }
  return MACAI_GDR_OK;
}

int64_t macai_gdr_conv_partials(int64_t B, int64_t T, int64_t C) { return B * conv_tiles(T) * C * CV_TAPS; }

static bool param_type_ok(int32_t t) { return t >= MACAI_GDR_F32 && t <= MACAI_GDR_F16; }

int macai_gdr_gates_fwd_typed(const void* b, const void* a, const void* A_log, int32_t atype, const void* dt_bias,
                              int32_t dtype_bias, float* params, float* beta, float* g, int64_t n, int64_t H,
                              int32_t dtype, void* stream) {
  const char* what = "macai_gdr_gates_fwd";
  if (n < 1 || H < 1 || n % H) return fail(MACAI_GDR_EINVAL, "%s: need n >= 1 a multiple of H >= 1", what);
  if (dtype < MACAI_GDR_F32 || dtype > MACAI_GDR_F16 || !param_type_ok(atype) || !param_type_ok(dtype_bias))
    return fail(MACAI_GDR_EUNSUP, "%s: dtype code", what);
  if (!b || !a || !A_log || !dt_bias || !beta || !g) return fail(MACAI_GDR_EINVAL, "%s: null pointer", what);
  const void* ps[] = {b, a, beta, g};
  for (const void* p : ps)
    if (!aligned16(p)) return fail(MACAI_GDR_EINVAL, "%s: pointers must be 16-byte aligned", what);
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)((n + GATE_THREADS - 1) / GATE_THREADS));
  const GateParams gp{A_log, dt_bias, atype, dtype_bias};
  if (atype != MACAI_GDR_F32 || dtype_bias != MACAI_GDR_F32 || params) {
    DISPATCH_PT(dtype, hipLaunchKernelGGL((gates_fwd_kernel<PT, true>), grid, dim3(GATE_THREADS), 0, st, (const PT*)b,
                                          (const PT*)a, gp, params, beta, g, n, (int)H))
  } else {
    DISPATCH_PT(dtype, hipLaunchKernelGGL((gates_fwd_kernel<PT, false>), grid, dim3(GATE_THREADS), 0, st, (const PT*)b,
                                          (const PT*)a, gp, params, beta, g, n, (int)H))
  }
  return launched(what);
}

int macai_gdr_gates_fwd(const void* b, const void* a, const float* A_log, const float* dt_bias, float* beta, float* g,
                        int64_t n, int64_t H, int32_t dtype, void* stream) {
  return macai_gdr_gates_fwd_typed(b, a, A_log, MACAI_GDR_F32, dt_bias, MACAI_GDR_F32, nullptr, beta, g, n, H, dtype,
                                   stream);
}

int64_t macai_gdr_gates_partials(int64_t n, int64_t H) {
  if (n < 1 || H < 1 || n % H) return 0;
  int64_t per;
  return gate_groups(n / H, H, &per) * 2 * H;
}

static int check_gates_bwd(const char* what, const void* b, const void* a, const float* A_log, const float* dt_bias,
                           const float* dbeta, const float* dg, void* db, void* da, int64_t n, int64_t H,
                           int32_t dtype) {
  if (n < 1 || H < 1 || n % H) return fail(MACAI_GDR_EINVAL, "%s: need n >= 1 a multiple of H >= 1", what);
  if (dtype < MACAI_GDR_F32 || dtype > MACAI_GDR_F16) return fail(MACAI_GDR_EUNSUP, "%s: dtype code", what);
  if (!b || !a || !A_log || !dt_bias || !dbeta || !dg || !db || !da)
    return fail(MACAI_GDR_EINVAL, "%s: null pointer", what);
  const void* ps[] = {b, a, dbeta, dg, db, da};
  for (const void* p : ps)
    if (!aligned16(p)) return fail(MACAI_GDR_EINVAL, "%s: pointers must be 16-byte aligned", what);
  return MACAI_GDR_OK;
}

// gates_bwd_kernel and, with dA_log non-null, gates_params_direct_kernel.
static int gates_bwd_direct(const char* what, const void* b, const void* a, const float* A_log, const float* dt_bias,
                            const float* dbeta, const float* dg, void* db, void* da, void* dA_log, int32_t atype,
                            void* ddt_bias, int32_t dtype_bias, int64_t n, int64_t H, int32_t dtype, hipStream_t st) {
  const dim3 grid((unsigned)((n + GATE_THREADS - 1) / GATE_THREADS));
  DISPATCH_PT(dtype, hipLaunchKernelGGL((gates_bwd_kernel<PT>), grid, dim3(GATE_THREADS), 0, st, (const PT*)b,
                                        (const PT*)a, A_log, dt_bias, dbeta, dg, (PT*)db, (PT*)da, n, (int)H))
  if (int rc = launched(what)) return rc;
  if (!dA_log) return MACAI_GDR_OK;
  DISPATCH_PT(dtype, hipLaunchKernelGGL((gates_params_direct_kernel<PT>), dim3((unsigned)H), dim3(256), 0, st,
                                        (const PT*)a, A_log, dt_bias, dg, dA_log, ddt_bias, atype, dtype_bias, n / H,
                                        (int)H))
  return launched(what);
}

int macai_gdr_gates_bwd(const void* b, const void* a, const float* A_log, const float* dt_bias, const float* dbeta,
                        const float* dg, void* db, void* da, float* dA_log, float* ddt_bias, int64_t n, int64_t H,
                        int32_t dtype, void* stream) {
  const char* what = "macai_gdr_gates_bwd";
  if (!dA_log != !ddt_bias) return fail(MACAI_GDR_EINVAL, "%s: dA_log and ddt_bias go together", what);
  if (int rc = check_gates_bwd(what, b, a, A_log, dt_bias, dbeta, dg, db, da, n, H, dtype)) return rc;
  return gates_bwd_direct(what, b, a, A_log, dt_bias, dbeta, dg, db, da, dA_log, MACAI_GDR_F32, ddt_bias, MACAI_GDR_F32,
                          n, H, dtype, (hipStream_t)stream);
}

int macai_gdr_gates_bwd_typed(const void* b, const void* a, const float* A_log, const float* dt_bias,
                              const float* dbeta, const float* dg, void* db, void* da, double* part, void* dA_log,
                              int32_t atype, void* ddt_bias, int32_t dtype_bias, int64_t n, int64_t H, int32_t dtype,
                              void* stream) {
  const char* what = "macai_gdr_gates_bwd";
  if (!part || !dA_log || !ddt_bias) return fail(MACAI_GDR_EINVAL, "%s: null pointer", what);
  if (!param_type_ok(atype) || !param_type_ok(dtype_bias)) return fail(MACAI_GDR_EUNSUP, "%s: dtype code", what);
  if (((uintptr_t)part & 7u) != 0) return fail(MACAI_GDR_EINVAL, "%s: the partial sums must be 8-byte aligned", what);
  if (int rc = check_gates_bwd(what, b, a, A_log, dt_bias, dbeta, dg, db, da, n, H, dtype)) return rc;
  hipStream_t st = (hipStream_t)stream;
  const int64_t rows = n / H;
  if (rows <= gate_direct_rows(H))
    return gates_bwd_direct(what, b, a, A_log, dt_bias, dbeta, dg, db, da, dA_log, atype, ddt_bias, dtype_bias, n, H,
                            dtype, st);
  int64_t per;
  const int64_t groups = gate_groups(rows, H, &per), hblocks = (H + GATE_THREADS - 1) / GATE_THREADS;
  DISPATCH_PT(dtype, hipLaunchKernelGGL((gates_bwd_sums_kernel<PT>), dim3((unsigned)(groups * hblocks)),
                                        dim3(GATE_THREADS), 0, st, (const PT*)b, (const PT*)a, A_log, dt_bias, dbeta, dg,
                                        (PT*)db, (PT*)da, part, rows, (int)H, (int)per, (int)hblocks))
  if (int rc = launched(what)) return rc;
  hipLaunchKernelGGL(gates_params_kernel, dim3((unsigned)H), dim3(64), 0, st, part, dA_log, ddt_bias, atype, dtype_bias,
                     (int)groups, (int)H);
  return launched(what);
}

}  // extern "C"
