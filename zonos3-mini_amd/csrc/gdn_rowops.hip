// Row-local operators of the GDN layer: depthwise causal conv1d (+ SiLU) with a rolling history over packed
// sequences, q/k L2-norm, beta sigmoid and the gated RMSNorm of the output. All are HBM-streaming kernels:
// consecutive threads own consecutive channels / elements, so every global access is coalesced.
#include <type_traits>

#include "gdn_common.h"

namespace zgdn {
namespace {

constexpr int CONV_CH = 64;       // tokens per chunk of the chunk table
constexpr int CONV_TT = 8;        // tokens per conv workgroup (16 measured 14 % slower at 4096 x 1536)
constexpr int CONV_SPLIT = CONV_CH / CONV_TT;  // workgroups per chunk
constexpr int CONV_THREADS = 256;
constexpr int CONV_WMAX = 4;

template <typename T>
__device__ __forceinline__ float rnd(float x) {
  if constexpr (sizeof(T) == 2) return bf16_to_f32(f32_to_bf16(x));
  else return x;
}

// CPT consecutive channels as loaded / stored by one thread (one 4-byte word for two bf16, a float2 for two
// floats).
__device__ __forceinline__ float as_float(float x) { return x; }
__device__ __forceinline__ float as_float(bf16 x) { return bf16_to_f32(x.bits); }

template <typename T, int CPT>
struct chans;
// ``raw`` is the loaded word(s), converted to floats by ``unpack`` where the values are used (so issuing a
// load never waits for its data).
template <typename T>
struct chans<T, 1> {
  using raw = T;
  __device__ __forceinline__ static raw load(const T* p) { return *p; }
  __device__ __forceinline__ static void unpack(raw w, float* v) { v[0] = as_float(w); }
  __device__ __forceinline__ static void store(T* p, const float* v) { io<T>::store(p, v[0]); }
};
template <>
struct chans<bf16, 2> {
  using raw = uint32_t;
  __device__ __forceinline__ static raw load(const bf16* p) { return *reinterpret_cast<const uint32_t*>(p); }
  __device__ __forceinline__ static void unpack(raw w, float* v) {
    v[0] = __uint_as_float(w << 16);
    v[1] = __uint_as_float(w & 0xffff0000u);
  }
  __device__ __forceinline__ static void store(bf16* p, const float* v) {
    *reinterpret_cast<uint32_t*>(p) = pack_bf16x2(v[0], v[1]);
  }
};
template <>
struct chans<float, 2> {
  using raw = float2;
  __device__ __forceinline__ static raw load(const float* p) { return *reinterpret_cast<const float2*>(p); }
  __device__ __forceinline__ static void unpack(raw w, float* v) {
    v[0] = w.x;
    v[1] = w.y;
  }
  __device__ __forceinline__ static void store(float* p, const float* v) {
    *reinterpret_cast<float2*>(p) = make_float2(v[0], v[1]);
  }
};

// y[t, c] = act(sum_j w[c, j] * x_{t - W + 1 + j}[c] + bias[c]) over CONV_TT tokens of one chunk of one
// sequence (x rows x_ld elements apart, y rows dense), CPT channels per thread, with x_{<0} taken from the sequence's history (the last W-1 columns of
// its state row, oldest first); the first tile of a sequence also writes the new state row = the last SW raw
// inputs of [history | x]. The accumulation is fp32; like F.conv1d and F.silu on `T` tensors, the conv
// result is rounded to T before the activation and the activation after. A tile issues all its token loads
// before the arithmetic, so its latency is one load round trip rather than one per token.
template <typename T, int CPT, int WK>
__global__ __launch_bounds__(CONV_THREADS) void conv_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const T* __restrict__ bias, const T* init, T* fin,
    T* __restrict__ y, const int32_t* __restrict__ cu, const int32_t* __restrict__ chunk_idx, int n_seqs,
    int n_chunks, int T_len, int D, long x_ld, int W_arg, int SW, int act) {
  const int W = WK > 0 ? WK : W_arg;  // WK: the width as a constant (the model's 4), 0: taken at run time
  const int c0 = (blockIdx.y * CONV_THREADS + threadIdx.x) * CPT;
  if (c0 >= D) return;
  int seq, j;
  const int tile = blockIdx.x / CONV_SPLIT, sub = blockIdx.x % CONV_SPLIT;
  if (cu != nullptr && (int)blockIdx.x >= n_chunks * CONV_SPLIT) {
    // trailing workgroups, one per sequence: empty packed sequences pass their state row through (zeros
    // without one)
    seq = blockIdx.x - n_chunks * CONV_SPLIT;
    int sb, se;
    seq_bounds(cu, seq, T_len, sb, se);
    if (fin == nullptr || se != sb) return;
    for (int k = 0; k < CPT; ++k) {
      T* frow = fin + ((size_t)seq * D + c0 + k) * SW;
      const T* hrow = init != nullptr ? init + ((size_t)seq * D + c0 + k) * SW : nullptr;
      for (int i = 0; i < SW; ++i) io<T>::store(frow + i, hrow != nullptr ? io<T>::load(hrow + i) : 0.f);
    }
    return;
  }
  if (cu != nullptr) {
    seq = chunk_idx[2 * tile];
    j = chunk_idx[2 * tile + 1];
    if (seq < 0 || seq >= n_seqs || j < 0) return;
  } else {
    const int nt = max(1, (T_len + CONV_CH - 1) / CONV_CH);
    seq = tile / nt;
    j = tile % nt;
  }
  int bos = seq * T_len, len = T_len;
  if (cu != nullptr) {
    int eos;
    seq_bounds(cu, seq, T_len, bos, eos);
    len = eos - bos;
  }
  const bool writes_state = fin != nullptr && j == 0 && sub == 0;
  if (len == 0) {  // an empty sequence (a batch of T = 0) passes its state row through
    if (writes_state)
      for (int k = 0; k < CPT; ++k) {
        T* frow = fin + ((size_t)seq * D + c0 + k) * SW;
        const T* hrow = init != nullptr ? init + ((size_t)seq * D + c0 + k) * SW : nullptr;
        for (int i = 0; i < SW; ++i) io<T>::store(frow + i, hrow != nullptr ? io<T>::load(hrow + i) : 0.f);
      }
    return;
  }
  if (j >= (len + CONV_CH - 1) / CONV_CH) return;  // a table row past the sequence's chunks
  const int t0 = j * CONV_CH + sub * CONV_TT;
  const int t1 = min(len, t0 + CONV_TT);
  if (t0 >= len) return;

  // Every load below is unconditional (indices clamped into the sequence / state row, a missing state row
  // replaced by x) and its value selected afterwards, so all of them issue back to back: a value written on
  // one side of a branch and loaded on the other would make the compiler wait for each load in turn.
  using C = chans<T, CPT>;
  const int last = len - 1;
  // Weights, bias, the tile's inputs and its history inside the sequence, all issued back to back with no
  // condition (indices clamped into the sequence). Only a sequence's first tile needs the old state row
  // (history before token 0) and the inputs of the new one; those loads come after, under conditions that
  // are false for every other tile. Raw words are converted when used.
  T wr[CPT][CONV_WMAX], br[CPT], hx[CPT][CONV_WMAX], hs[CPT][CONV_WMAX] = {}, nx[CPT][CONV_WMAX] = {},
      ns[CPT][CONV_WMAX] = {};
  typename C::raw xr[CONV_TT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int c = c0 + k;
#pragma unroll
    for (int i = 0; i < CONV_WMAX; ++i) wr[k][i] = w[(size_t)c * W + min(i, W - 1)];
    br[k] = (bias != nullptr ? bias : w)[bias != nullptr ? c : 0];
  }
#pragma unroll
  for (int i = 0; i < CONV_TT; ++i) xr[i] = C::load(x + ((size_t)(bos + min(t0 + i, last))) * x_ld + c0);
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const T* xc = x + (size_t)bos * x_ld + c0 + k;
#pragma unroll
    for (int i = 0; i < CONV_WMAX; ++i) hx[k][i] = xc[(size_t)min(max(t0 - (W - 1) + i, 0), last) * x_ld];
  }
  if (init != nullptr && (t0 < W - 1 || writes_state)) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const T* hrow = init + ((size_t)seq * D + c0 + k) * SW;
#pragma unroll
      for (int i = 0; i < CONV_WMAX; ++i) {
        hs[k][i] = hrow[min(max(SW + t0 - (W - 1) + i, 0), SW - 1)];  // the input W-1-i steps before t0
        ns[k][i] = hrow[min(max(SW + len - SW + i, 0), SW - 1)];      // the new row's i-th input
      }
    }
  }
  if (writes_state) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const T* xc = x + (size_t)bos * x_ld + c0 + k;
#pragma unroll
      for (int i = 0; i < CONV_WMAX; ++i) nx[k][i] = xc[(size_t)min(max(len - SW + i, 0), last) * x_ld];
    }
  }
  // values used (a missing state row reads as zeros)
  float wc[CPT][CONV_WMAX], hist[CPT][CONV_WMAX], nv[CPT][CONV_WMAX], bc[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    bc[k] = bias != nullptr ? as_float(br[k]) : 0.f;
#pragma unroll
    for (int i = 0; i < CONV_WMAX; ++i) {
      wc[k][i] = i < W ? as_float(wr[k][i]) : 0.f;
      const int th = t0 - (W - 1) + i, tn = len - SW + i;
      hist[k][i] = i >= W - 1 ? 0.f : th >= 0 ? as_float(hx[k][i]) : as_float(hs[k][i]);
      nv[k][i] = tn >= 0 ? as_float(nx[k][i]) : as_float(ns[k][i]);
    }
  }
  // full tiles (all but a sequence's last) run without a per-token guard
  auto run = [&](auto full) {
#pragma unroll
    for (int i = 0; i < CONV_TT; ++i) {
      if (!decltype(full)::value && t0 + i >= t1) continue;  // (not a break: the loop stays unrolled)
      float xv[CPT], out[CPT];
      C::unpack(xr[i], xv);
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        float acc = bc[k];
#pragma unroll
        for (int m = 0; m < CONV_WMAX - 1; ++m)
          if (m < W - 1) acc = fmaf(wc[k][m], hist[k][m], acc);
        out[k] = fmaf(wc[k][W - 1], xv[k], acc);
#pragma unroll
        for (int m = 0; m < CONV_WMAX - 2; ++m)
          if (m < W - 2) hist[k][m] = hist[k][m + 1];
        if (W >= 2) hist[k][W - 2] = xv[k];
      }
      // the conv rounded to T (two bf16 values with one conversion), then the activation; its result is rounded
      // to T by the store
      if constexpr (sizeof(T) == 2 && CPT == 2) {
        const uint32_t pk = pack_bf16x2(out[0], out[1]);
        out[0] = __uint_as_float(pk << 16);
        out[1] = __uint_as_float(pk & 0xffff0000u);
      } else {
#pragma unroll
        for (int k = 0; k < CPT; ++k) out[k] = rnd<T>(out[k]);
      }
      if (act) {
#pragma unroll
        for (int k = 0; k < CPT; ++k) out[k] = silu_fast(out[k]);
      }
      chans<T, CPT>::store(y + ((size_t)(bos + t0 + i)) * D + c0, out);
    }
  };
  if (t1 - t0 == CONV_TT)
    run(std::true_type{});
  else
    run(std::false_type{});
  // the tile holding the sequence start writes the new state row (it alone reads the old one, so the state
  // may be updated in place)
  if (writes_state) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      T* frow = fin + ((size_t)seq * D + c0 + k) * SW;
#pragma unroll
      for (int i = 0; i < CONV_WMAX; ++i)
        if (i < SW) io<T>::store(frow + i, nv[k][i]);
    }
  }
}

// Rows of 128 (the head size): 16 lanes per row, each with 8 consecutive elements in one 16-byte access
// (two for fp32; element by element where some row is not 16-byte aligned, ALIGNED false, with the same
// arithmetic, so results do not depend on where the rows sit; every D = 128 call runs these kernels), and the row sum over the 16 lanes by DPP;
// four rows per wave.
template <typename T>
struct oct;
template <>
struct oct<bf16> {
  using raw = uint4;
  __device__ __forceinline__ static raw load(const bf16* p) { return *reinterpret_cast<const uint4*>(p); }
  __device__ __forceinline__ static raw load_unaligned(const bf16* p) {
    uint32_t u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = (uint32_t)p[2 * i].bits | ((uint32_t)p[2 * i + 1].bits << 16);
    return make_uint4(u[0], u[1], u[2], u[3]);
  }
  __device__ __forceinline__ static void unpack(const raw& w, float* v) {
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(u[i] << 16);
      v[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
    }
  }
  __device__ __forceinline__ static void store(bf16* p, const float* v) {
    *reinterpret_cast<uint4*>(p) = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                                              pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
  }
  __device__ __forceinline__ static void store_unaligned(bf16* p, const float* v) {
#pragma unroll
    for (int i = 0; i < 8; ++i) io<bf16>::store(p + i, v[i]);
  }
};
template <>
struct oct<float> {
  struct raw {
    float4 a, b;
  };
  __device__ __forceinline__ static raw load(const float* p) {
    return {reinterpret_cast<const float4*>(p)[0], reinterpret_cast<const float4*>(p)[1]};
  }
  __device__ __forceinline__ static raw load_unaligned(const float* p) {
    return {make_float4(p[0], p[1], p[2], p[3]), make_float4(p[4], p[5], p[6], p[7])};
  }
  __device__ __forceinline__ static void unpack(const raw& w, float* v) {
    v[0] = w.a.x, v[1] = w.a.y, v[2] = w.a.z, v[3] = w.a.w;
    v[4] = w.b.x, v[5] = w.b.y, v[6] = w.b.z, v[7] = w.b.w;
  }
  __device__ __forceinline__ static void store(float* p, const float* v) {
    reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
  }
  __device__ __forceinline__ static void store_unaligned(float* p, const float* v) {
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = v[i];
  }
};
constexpr int R128_ROWS = 16;  // rows per 256-thread workgroup

// A whole 16-lane group exits together, so the DPP sums read active lanes only.
template <typename TI, typename TO, bool ALIGNED>
__global__ __launch_bounds__(256) void l2norm128_kernel(const TI* __restrict__ x, TO* __restrict__ y,
                                                        float* __restrict__ rstd, int rows, int x_group,
                                                        long x_ld, float eps) {
  const int row = blockIdx.x * R128_ROWS + (threadIdx.x >> 4), sub = threadIdx.x & 15;
  if (row >= rows) return;
  const TI* xr = x + (size_t)(row / x_group) * x_ld + (size_t)(row % x_group) * 128 + 8 * sub;
  float v[8];
  oct<TI>::unpack(ALIGNED ? oct<TI>::load(xr) : oct<TI>::load_unaligned(xr), v);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
  const float r = rsqrtf(group_sum<16>(ss) + eps);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] *= r;
  TO* yr = y + (size_t)row * 128 + 8 * sub;
  if constexpr (ALIGNED) oct<TO>::store(yr, v);
  else oct<TO>::store_unaligned(yr, v);
  if (rstd != nullptr && sub == 0) rstd[row] = r;
}

template <typename T, bool ALIGNED>
__global__ __launch_bounds__(256) void gated_rmsnorm128_kernel(const T* __restrict__ x, const T* __restrict__ g,
                                                               const T* __restrict__ w, T* __restrict__ y,
                                                               float* __restrict__ rstd, int rows, int g_group,
                                                               long g_ld, float eps) {
  const int row = blockIdx.x * R128_ROWS + (threadIdx.x >> 4), sub = threadIdx.x & 15;
  if (row >= rows) return;
  const T* xp = x + (size_t)row * 128 + 8 * sub;
  const T* gp = g + (size_t)(row / g_group) * g_ld + (size_t)(row % g_group) * 128 + 8 * sub;
  const typename oct<T>::raw xr = ALIGNED ? oct<T>::load(xp) : oct<T>::load_unaligned(xp);
  const typename oct<T>::raw gr = ALIGNED ? oct<T>::load(gp) : oct<T>::load_unaligned(gp);
  const typename oct<T>::raw wr = ALIGNED ? oct<T>::load(w + 8 * sub) : oct<T>::load_unaligned(w + 8 * sub);
  float v[8], gv[8], wv[8];
  oct<T>::unpack(xr, v);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
  const float r = rsqrtf(group_sum<16>(ss) / 128.f + eps);
  oct<T>::unpack(gr, gv);
  oct<T>::unpack(wr, wv);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = rnd<T>(v[i] * r * wv[i]) * silu(gv[i]);
  T* yr = y + (size_t)row * 128 + 8 * sub;
  if constexpr (ALIGNED) oct<T>::store(yr, v);
  else oct<T>::store_unaligned(yr, v);
  if (rstd != nullptr && sub == 0) rstd[row] = r;
}

// Whether rows of 128 at base p, ld elements apart, suit the 16-byte accesses of the 128-wide kernels.
__host__ inline bool rows128(const void* p, long ld, size_t esz) {
  return (uintptr_t)p % 16 == 0 && (ld * (long)esz) % 16 == 0;
}

// y = x * rsqrt(sum x^2 + eps) over rows of D <= 1024 elements; one wave per row. y is dense; row r of x
// starts at x + (r / x_group) * x_ld + (r % x_group) * D (a token's per-head rows inside a wider row).
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void l2norm_kernel(const TI* __restrict__ x, TO* __restrict__ y,
                                                     float* __restrict__ rstd, int rows, int D, int x_group,
                                                     long x_ld, float eps) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const TI* xr = x + (size_t)(row / x_group) * x_ld + (size_t)(row % x_group) * D;
  float v[16];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int c = lane + 64 * i;
    v[i] = c < D ? io<TI>::load(xr + c) : 0.f;
    ss = fmaf(v[i], v[i], ss);
  }
  const float r = rsqrtf(wave_sum(ss) + eps);
  TO* yr = y + (size_t)row * D;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int c = lane + 64 * i;
    if (c < D) io<TO>::store(yr + c, v[i] * r);
  }
  if (rstd != nullptr && lane == 0) rstd[row] = r;
}

template <typename TI, typename TO>
__global__ __launch_bounds__(256) void sigmoid_kernel(const TI* __restrict__ x, TO* __restrict__ y, size_t n,
                                                      float scale) {
  const size_t i = blockIdx.x * (size_t)256 + threadIdx.x;
  if (i < n) io<TO>::store(y + i, sigmoid(io<TI>::load(x + i)) * scale);
}

// y = (rms_norm(x) * w).to(T) * silu(g), product in fp32, cast to T; one wave per row of D <= 1024. x and y
// are dense; row r's gate starts at g + (r / g_group) * g_ld + (r % g_group) * D (per-head rows of a token's
// gate, read in place from a wider row).
template <typename T>
__global__ __launch_bounds__(256) void gated_rmsnorm_kernel(const T* __restrict__ x, const T* __restrict__ g,
                                                            const T* __restrict__ w, T* __restrict__ y,
                                                            float* __restrict__ rstd, int rows, int D, int g_group,
                                                            long g_ld, float eps) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const T* xr = x + (size_t)row * D;
  float v[16];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int c = lane + 64 * i;
    v[i] = c < D ? io<T>::load(xr + c) : 0.f;
    ss = fmaf(v[i], v[i], ss);
  }
  const float r = rsqrtf(wave_sum(ss) / (float)D + eps);
  const T* gr = g + (size_t)(row / g_group) * g_ld + (size_t)(row % g_group) * D;
  T* yr = y + (size_t)row * D;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int c = lane + 64 * i;
    if (c < D) io<T>::store(yr + c, rnd<T>(v[i] * r * io<T>::load(w + c)) * silu(io<T>::load(gr + c)));
  }
  if (rstd != nullptr && lane == 0) rstd[row] = r;
}

// ------------------------------------------------------------------------------- the serving layer's eager call
//
// An eager prefill / extend of the serving layer (servers/sgl/src/zonos3_sgl/models/gdn.py:271-327) runs every
// request's joined run -- its slot's unfinished chunk, then its new rows -- as one packed sequence, reading and
// writing the slots' caches in place. The kernels below are its row-local parts; each workgroup finds its rows
// from the run tables (a few dozen integers), so the host lists no rows. Six requests, 1,067 new rows, hidden 1024:
// 102 us a call, 61 us of it kernels (two GEMMs 26.0, phase 1 10.6, state pass 9.5, conv 6.3, gather 4.5, norm 4.1);
// through index lists of every row, two passes and some 45 launches of index_select / index_copy / index_fill and
// the operators 1,074-1,127 us, nearly all of it the host.

constexpr int SV_W = 4;     // conv width, and the width of a slot's conv history
constexpr int SV_ROWS = 8;  // rows per gather workgroup

// rows of the packed pass from the windows (replayed rows) and the call's rows; hidden elements in 16-byte pieces
__global__ __launch_bounds__(256) void serve_gather_kernel(const ServeRuns r, const uint4* __restrict__ x,
                                                           const uint4* __restrict__ window, int row16,
                                                           uint4* __restrict__ out) {
  constexpr int SPLIT = CHUNK_LEN / SV_ROWS;
  int run, j, bos, len, slot;
  if (!serve_chunk(r, blockIdx.x / SPLIT, run, j, bos, len, slot)) return;
  const int t0 = j * CHUNK_LEN + (blockIdx.x % SPLIT) * SV_ROWS, n = min(SV_ROWS, len - t0);
  const int replay = min(max(r.replay[run], 0), CHUNK_LEN), xoff = r.xoff[run];
  for (int e = threadIdx.x; e < n * row16; e += 256) {
    const int i = e / row16, c = e - i * row16, t = t0 + i;
    const int xr = min(max(xoff + t - replay, 0), r.new_rows - 1);
    const uint4* src = t < replay ? window + ((size_t)slot * CHUNK_LEN + t) * row16 : x + (size_t)xr * row16;
    out[(size_t)(bos + t) * row16 + c] = src[c];
  }
}

// The conv + SiLU of CONV_TT rows of a chunk for 512 channels (two a thread, one head of 128 a wave), with the
// arithmetic and rounding of conv_kernel; q and k (channels below 2 x 128 H) then L2-normalised in the wave with
// l2norm128_kernel's order of summation (a quad of lanes holds its eight elements), so both are bit-identical to
// those two kernels. The tile holding a run's start writes the slot's new histories: the last 4 raw rows of the
// run (live) and of its complete chunks (committed; untouched when it has none, zeros for a fresh slot).
__global__ __launch_bounds__(256) void serve_conv_kernel(const ServeRuns r, const bf16* __restrict__ mixed, long ld,
                                                         const bf16* __restrict__ w, bf16* conv_commit,
                                                         bf16* __restrict__ conv_live, bf16* __restrict__ qkv, int H) {
  const int C = 3 * H * 128;
  const int c0 = (blockIdx.y * 256 + threadIdx.x) * 2;
  if (c0 >= C) return;  // (whole waves: C is a multiple of 128)
  int run, j, bos, len, slot;
  if (!serve_chunk(r, blockIdx.x / CONV_SPLIT, run, j, bos, len, slot)) return;
  const int t0 = j * CONV_CH + (blockIdx.x % CONV_SPLIT) * CONV_TT;
  if (t0 >= len) return;
  const int n = min(CONV_TT, len - t0), last = len - 1;
  const bool fresh = r.fresh[run] != 0;
  const uint32_t* col = reinterpret_cast<const uint32_t*>(mixed + (size_t)bos * ld + c0);
  const long ld2 = ld / 2;  // (rows in channel pairs)
  auto raw = [&](int t) { return col[(size_t)min(max(t, 0), last) * ld2]; };
  uint32_t xr[CONV_TT], hx[3];
#pragma unroll
  for (int i = 0; i < CONV_TT; ++i) xr[i] = raw(t0 + i);
#pragma unroll
  for (int i = 0; i < 3; ++i) hx[i] = raw(t0 - 3 + i);
  const uint2 w0 = *reinterpret_cast<const uint2*>(w + (size_t)c0 * SV_W);
  const uint2 w1 = *reinterpret_cast<const uint2*>(w + (size_t)(c0 + 1) * SV_W);
  if (t0 == 0) {
    // the rows before the run: the slot's committed history [C][4], oldest first; then the new histories
    bf16* hc = conv_commit + ((size_t)slot * C + c0) * SV_W;
    uint2 h0 = *reinterpret_cast<const uint2*>(hc), h1 = *reinterpret_cast<const uint2*>(hc + SV_W);
    if (fresh) h0 = h1 = make_uint2(0, 0);
    // old[i]: both channels' history column i
    const uint32_t old[SV_W] = {(h0.x & 0xffffu) | (h1.x << 16), (h0.x >> 16) | (h1.x & 0xffff0000u),
                                (h0.y & 0xffffu) | (h1.y << 16), (h0.y >> 16) | (h1.y & 0xffff0000u)};
#pragma unroll
    for (int i = 0; i < 3; ++i) hx[i] = old[i + 1];
    auto put = [&](bf16* dst, int end) {  // the last 4 rows of [history | first `end` rows]
      uint32_t v[SV_W];
#pragma unroll
      for (int i = 0; i < SV_W; ++i) {
        const int t = end - SV_W + i;
        uint32_t o = old[SV_W - 1];
#pragma unroll
        for (int e = 0; e < SV_W - 1; ++e)
          if (t + SV_W == e) o = old[e];
        v[i] = t >= 0 ? raw(t) : o;
      }
      bf16* d = dst + ((size_t)slot * C + c0) * SV_W;
      *reinterpret_cast<uint4*>(d) =
          make_uint4((v[0] & 0xffffu) | (v[1] << 16), (v[2] & 0xffffu) | (v[3] << 16),
                     (v[0] >> 16) | (v[1] & 0xffff0000u), (v[2] >> 16) | (v[3] & 0xffff0000u));
    };
    put(conv_live, len);
    const int whole = len - len % CONV_CH;
    if (whole > 0 || fresh) put(conv_commit, whole);
  }
  const float k0[4] = {__uint_as_float(w0.x << 16), __uint_as_float(w0.x & 0xffff0000u), __uint_as_float(w0.y << 16),
                       __uint_as_float(w0.y & 0xffff0000u)};
  const float k1[4] = {__uint_as_float(w1.x << 16), __uint_as_float(w1.x & 0xffff0000u), __uint_as_float(w1.y << 16),
                       __uint_as_float(w1.y & 0xffff0000u)};
  const bool norm = c0 < 2 * H * 128;  // (wave-uniform)
  uint32_t win[3] = {hx[0], hx[1], hx[2]};
#pragma unroll
  for (int i = 0; i < CONV_TT; ++i) {
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      a = fmaf(k0[m], __uint_as_float(win[m] << 16), a);
      b = fmaf(k1[m], __uint_as_float(win[m] & 0xffff0000u), b);
    }
    a = fmaf(k0[3], __uint_as_float(xr[i] << 16), a);
    b = fmaf(k1[3], __uint_as_float(xr[i] & 0xffff0000u), b);
    win[0] = win[1];
    win[1] = win[2];
    win[2] = xr[i];
    uint32_t pk = pack_bf16x2(a, b);
    pk = pack_bf16x2(silu_fast(__uint_as_float(pk << 16)), silu_fast(__uint_as_float(pk & 0xffff0000u)));
    if (norm) {
      const float y0 = __uint_as_float(pk << 16), y1 = __uint_as_float(pk & 0xffff0000u);
      // sum of squares of the quad's 8 elements in order, then over the 16 quads
      float ss = 0.f;
      ss = fmaf(dpp<0x00>(y0), dpp<0x00>(y0), ss);  // quad_perm broadcasts of lanes 0 .. 3
      ss = fmaf(dpp<0x00>(y1), dpp<0x00>(y1), ss);
      ss = fmaf(dpp<0x55>(y0), dpp<0x55>(y0), ss);
      ss = fmaf(dpp<0x55>(y1), dpp<0x55>(y1), ss);
      ss = fmaf(dpp<0xAA>(y0), dpp<0xAA>(y0), ss);
      ss = fmaf(dpp<0xAA>(y1), dpp<0xAA>(y1), ss);
      ss = fmaf(dpp<0xFF>(y0), dpp<0xFF>(y0), ss);
      ss = fmaf(dpp<0xFF>(y1), dpp<0xFF>(y1), ss);
      ss += dpp<DPP_ROW_HALF_MIRROR>(ss);
      ss += dpp<DPP_ROW_MIRROR>(ss);
      auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(ss), __float_as_uint(ss), false, false);
      ss = __uint_as_float(p[0]) + __uint_as_float(p[1]);
      p = __builtin_amdgcn_permlane32_swap(__float_as_uint(ss), __float_as_uint(ss), false, false);
      ss = __uint_as_float(p[0]) + __uint_as_float(p[1]);
      const float rn = rsqrtf(ss + 1e-6f);
      pk = pack_bf16x2(y0 * rn, y1 * rn);
    }
    if (i < n) *reinterpret_cast<uint32_t*>(qkv + (size_t)(bos + t0 + i) * C + c0) = pk;
  }
}

// The gated norm (gated_rmsnorm128_kernel's arithmetic) of a chunk's rows, 16 head rows a workgroup, written in the
// order of the call's new rows (replayed rows are dropped), so that wo runs on the new rows alone; the open chunk's
// new rows also go to the slot's window, and the run's first workgroup sets the window's length.
__global__ __launch_bounds__(256) void serve_norm_kernel(const ServeRuns r, const bf16* __restrict__ o,
                                                         const bf16* __restrict__ z, long z_ld,
                                                         const bf16* __restrict__ w, float eps, bf16* __restrict__ gated,
                                                         const uint4* __restrict__ x, int row16, uint4* window,
                                                         int32_t* win_len, int H) {
  const int per = 16 / H;  // tokens a workgroup (H = 1, 2, 4, 8 or 16)
  const int split = CHUNK_LEN / per;
  int run, j, bos, len, slot;
  if (!serve_chunk(r, blockIdx.x / split, run, j, bos, len, slot)) return;
  const int t0 = j * CHUNK_LEN + (blockIdx.x % split) * per;
  const int replay = min(max(r.replay[run], 0), CHUNK_LEN), xoff = r.xoff[run];
  const int fill = len % CHUNK_LEN, whole = len - fill;
  if (t0 == 0 && threadIdx.x == 0) win_len[slot] = fill;
  if (t0 >= len) return;
  if (t0 >= whole) {
    const int n = min(per, len - t0);
    for (int e = threadIdx.x; e < n * row16; e += 256) {
      const int i = e / row16, c = e - i * row16, t = t0 + i, xr = xoff + t - replay;
      if (t >= replay && xr >= 0 && xr < r.new_rows)
        window[((size_t)slot * CHUNK_LEN + t - whole) * row16 + c] = x[(size_t)xr * row16 + c];
    }
  }
  const int hr = threadIdx.x >> 4, sub = threadIdx.x & 15, t = t0 + hr / H, h = hr % H;
  const int dst = xoff + t - replay;
  if (t >= len || t < replay || dst < 0 || dst >= r.new_rows) return;  // (whole 16-lane groups)
  const size_t row = (size_t)(bos + t);
  const oct<bf16>::raw xw = oct<bf16>::load(o + (row * H + h) * 128 + 8 * sub);
  const oct<bf16>::raw gw = oct<bf16>::load(z + row * z_ld + h * 128 + 8 * sub);
  const oct<bf16>::raw ww = oct<bf16>::load(w + 8 * sub);
  float v[8], gv[8], wv[8];
  oct<bf16>::unpack(xw, v);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
  const float rn = rsqrtf(group_sum<16>(ss) / 128.f + eps);
  oct<bf16>::unpack(gw, gv);
  oct<bf16>::unpack(ww, wv);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = rnd<bf16>(v[i] * rn * wv[i]) * silu(gv[i]);
  oct<bf16>::store(gated + ((size_t)dst * H + h) * 128 + 8 * sub, v);
}

}  // namespace

void serve_gather(const ServeRuns& r, const void* x, const void* window, int hidden, void* out, hipStream_t s) {
  hipLaunchKernelGGL(serve_gather_kernel, dim3(r.n_chunks * (CHUNK_LEN / SV_ROWS)), dim3(256), 0, s, r, (const uint4*)x,
                     (const uint4*)window, hidden / 8, (uint4*)out);
}
void serve_conv(const ServeRuns& r, const void* mixed, long mixed_ld, const void* conv_w, void* conv_commit,
                void* conv_live, void* qkv, int H, hipStream_t s) {
  hipLaunchKernelGGL(serve_conv_kernel, dim3(r.n_chunks * CONV_SPLIT, (3 * H * 128 + 511) / 512), dim3(256), 0, s, r,
                     (const bf16*)mixed, mixed_ld, (const bf16*)conv_w, (bf16*)conv_commit, (bf16*)conv_live, (bf16*)qkv, H);
}
void serve_norm(const ServeRuns& r, const void* o, const void* z, long z_ld, const void* norm_w, float eps, void* gated,
                const void* x, int hidden, void* window, int32_t* win_len, int H, hipStream_t s) {
  hipLaunchKernelGGL(serve_norm_kernel, dim3(r.n_chunks * CHUNK_LEN * H / 16), dim3(256), 0, s, r, (const bf16*)o,
                     (const bf16*)z, z_ld, (const bf16*)norm_w, eps, (bf16*)gated, (const uint4*)x, hidden / 8,
                     (uint4*)window, win_len, H);
}
}  // namespace zgdn

extern "C" int zgdn_causal_conv1d_fwd(const void* x, const void* weight, const void* bias, int dtype,
                                      const void* initial_state, void* final_state, int state_width, void* y,
                                      const int32_t* cu_seqlens, const int32_t* chunk_indices, int n_seqs,
                                      int n_chunks, int B, int T, int D, int W, int activation, long x_ld,
                                      void* stream) {
  using namespace zgdn;
  const char* fn = "zgdn_causal_conv1d_fwd";
  if (!x || !weight || !y) return fail(ZGDN_EINVAL, "%s: null pointer", fn);
  if (x_ld < D) return fail(ZGDN_EINVAL, "%s: x row stride %ld < D=%d", fn, x_ld, D);
  if (W < 1 || W > CONV_WMAX) return fail(ZGDN_EUNSUPPORTED, "%s: width %d (supported: 1..4)", fn, W);
  if (state_width < W - 1 || state_width > CONV_WMAX)
    return fail(ZGDN_EINVAL, "%s: state width %d for conv width %d (need W-1 .. 4)", fn, state_width, W);
  if (B < 1 || T < 0 || D < 1) return fail(ZGDN_EINVAL, "%s: bad sizes B=%d T=%d D=%d", fn, B, T, D);
  if (dtype != ZGDN_F32 && dtype != ZGDN_BF16) return fail(ZGDN_EINVAL, "%s: dtype code %d", fn, dtype);
  int grid_x;
  if (cu_seqlens != nullptr) {
    if (B != 1 || chunk_indices == nullptr || n_seqs < 1 || n_chunks < 0)
      return fail(ZGDN_EINVAL, "%s: packed sequences need B == 1, chunk_indices and n_seqs >= 1", fn);
    grid_x = n_chunks * CONV_SPLIT + n_seqs;  // + one workgroup column per sequence for empty ones
  } else {
    n_seqs = B;
    grid_x = B * ((T + CONV_CH - 1) / CONV_CH) * CONV_SPLIT;
    if (T == 0) grid_x = B * CONV_SPLIT;  // empty sequences still pass their state through
  }
  if (grid_x == 0) return check_launch(fn);
  hipStream_t s = (hipStream_t)stream;
  auto go = [&](auto* tag, auto cpt) {
    using TT = std::remove_pointer_t<decltype(tag)>;
    constexpr int CPT = decltype(cpt)::value;
    const int per_wg = CONV_THREADS * CPT;
    dim3 grid(grid_x, (D + per_wg - 1) / per_wg);
    auto kernel = W == 4 ? conv_kernel<TT, CPT, 4> : conv_kernel<TT, CPT, 0>;
    hipLaunchKernelGGL(kernel, grid, dim3(CONV_THREADS), 0, s, (const TT*)x, (const TT*)weight, (const TT*)bias,
                       (const TT*)initial_state, (TT*)final_state, (TT*)y, cu_seqlens, chunk_indices, n_seqs,
                       n_chunks, T, D, x_ld, W, state_width, activation);
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  // two channels per thread where every pair of x and y stays 4- or 8-byte aligned (four bf16 channels a thread,
  // 8-byte accesses in 128-thread workgroups, measured 13 % slower at 4096 x 1536: more registers, fewer waves)
  const size_t esz = dtype == ZGDN_F32 ? 4 : 2;
  const bool pairs = D % 2 == 0 && x_ld % 2 == 0 && (uintptr_t)x % (2 * esz) == 0 && (uintptr_t)y % (2 * esz) == 0;
  if (dtype == ZGDN_F32) {
    if (pairs) go((float*)nullptr, Two{});
    else go((float*)nullptr, One{});
  } else {
    if (pairs) go((bf16*)nullptr, Two{});
    else go((bf16*)nullptr, One{});
  }
  return check_launch(fn);
}

extern "C" int zgdn_l2norm_fwd(const void* x, int x_dtype, void* y, int y_dtype, float* rstd, int rows, int D,
                               int x_group, long x_ld, float eps, void* stream) {
  using namespace zgdn;
  const char* fn = "zgdn_l2norm_fwd";
  if (!x || !y) return fail(ZGDN_EINVAL, "%s: null pointer", fn);
  if (rows < 0 || D < 1 || D > 1024) return fail(ZGDN_EUNSUPPORTED, "%s: rows=%d D=%d (D <= 1024)", fn, rows, D);
  if (x_group < 1 || x_ld < (long)x_group * D)
    return fail(ZGDN_EINVAL, "%s: x rows: group %d, stride %ld (need group >= 1, stride >= group * D)", fn,
                x_group, x_ld);
  for (int dt : {x_dtype, y_dtype})
    if (dt != ZGDN_F32 && dt != ZGDN_BF16) return fail(ZGDN_EINVAL, "%s: dtype code %d", fn, dt);
  if (rows == 0) return check_launch(fn);
  hipStream_t s = (hipStream_t)stream;
  if (D == 128) {
    const bool al = rows128(x, x_ld, x_dtype == ZGDN_F32 ? 4 : 2) && rows128(y, 128, y_dtype == ZGDN_F32 ? 4 : 2);
    dim3 grid((rows + R128_ROWS - 1) / R128_ROWS), block(256);
    auto go = [&](auto* ti, auto* to) {
      using TI = std::remove_const_t<std::remove_pointer_t<decltype(ti)>>;
      using TO = std::remove_pointer_t<decltype(to)>;
      auto kernel = al ? l2norm128_kernel<TI, TO, true> : l2norm128_kernel<TI, TO, false>;
      hipLaunchKernelGGL(kernel, grid, block, 0, s, (const TI*)x, (TO*)y, rstd, rows, x_group, x_ld, eps);
    };
    if (x_dtype == ZGDN_F32 && y_dtype == ZGDN_F32) go((float*)nullptr, (float*)nullptr);
    else if (x_dtype == ZGDN_F32) go((float*)nullptr, (bf16*)nullptr);
    else if (y_dtype == ZGDN_F32) go((bf16*)nullptr, (float*)nullptr);
    else go((bf16*)nullptr, (bf16*)nullptr);
    return check_launch(fn);
  }
  dim3 grid((rows + 3) / 4), block(256);
  if (x_dtype == ZGDN_F32 && y_dtype == ZGDN_F32)
    hipLaunchKernelGGL((l2norm_kernel<float, float>), grid, block, 0, s, (const float*)x, (float*)y, rstd, rows, D, x_group, x_ld, eps);
  else if (x_dtype == ZGDN_F32)
    hipLaunchKernelGGL((l2norm_kernel<float, bf16>), grid, block, 0, s, (const float*)x, (bf16*)y, rstd, rows, D, x_group, x_ld, eps);
  else if (y_dtype == ZGDN_F32)
    hipLaunchKernelGGL((l2norm_kernel<bf16, float>), grid, block, 0, s, (const bf16*)x, (float*)y, rstd, rows, D, x_group, x_ld, eps);
  else
    hipLaunchKernelGGL((l2norm_kernel<bf16, bf16>), grid, block, 0, s, (const bf16*)x, (bf16*)y, rstd, rows, D, x_group, x_ld, eps);
  return check_launch(fn);
}

extern "C" int zgdn_sigmoid_fwd(const void* x, int x_dtype, void* y, int y_dtype, size_t n, float scale,
                                void* stream) {
  using namespace zgdn;
  const char* fn = "zgdn_sigmoid_fwd";
  if (!x || !y) return fail(ZGDN_EINVAL, "%s: null pointer", fn);
  for (int dt : {x_dtype, y_dtype})
    if (dt != ZGDN_F32 && dt != ZGDN_BF16) return fail(ZGDN_EINVAL, "%s: dtype code %d", fn, dt);
  if (n == 0) return check_launch(fn);
  dim3 grid((unsigned)((n + 255) / 256)), block(256);
  hipStream_t s = (hipStream_t)stream;
  if (x_dtype == ZGDN_F32 && y_dtype == ZGDN_F32)
    hipLaunchKernelGGL((sigmoid_kernel<float, float>), grid, block, 0, s, (const float*)x, (float*)y, n, scale);
  else if (x_dtype == ZGDN_F32)
    hipLaunchKernelGGL((sigmoid_kernel<float, bf16>), grid, block, 0, s, (const float*)x, (bf16*)y, n, scale);
  else if (y_dtype == ZGDN_F32)
    hipLaunchKernelGGL((sigmoid_kernel<bf16, float>), grid, block, 0, s, (const bf16*)x, (float*)y, n, scale);
  else
    hipLaunchKernelGGL((sigmoid_kernel<bf16, bf16>), grid, block, 0, s, (const bf16*)x, (bf16*)y, n, scale);
  return check_launch(fn);
}

extern "C" int zgdn_gated_rmsnorm_fwd(const void* x, const void* g, const void* weight, int dtype, void* y,
                                      float* rstd, int rows, int D, int g_group, long g_ld, float eps,
                                      void* stream) {
  using namespace zgdn;
  const char* fn = "zgdn_gated_rmsnorm_fwd";
  if (!x || !g || !weight || !y) return fail(ZGDN_EINVAL, "%s: null pointer", fn);
  if (g_group < 1 || g_ld < (long)g_group * D)
    return fail(ZGDN_EINVAL, "%s: gate rows: group %d, stride %ld (need group >= 1, stride >= group * D)", fn,
                g_group, g_ld);
  if (rows < 0 || D < 1 || D > 1024) return fail(ZGDN_EUNSUPPORTED, "%s: rows=%d D=%d (D <= 1024)", fn, rows, D);
  if (dtype != ZGDN_F32 && dtype != ZGDN_BF16) return fail(ZGDN_EINVAL, "%s: dtype code %d", fn, dtype);
  if (rows == 0) return check_launch(fn);
  hipStream_t s = (hipStream_t)stream;
  const size_t esz = dtype == ZGDN_F32 ? 4 : 2;
  if (D == 128) {
    const bool al = rows128(x, 128, esz) && rows128(g, g_ld, esz) && rows128(weight, 0, esz) && rows128(y, 128, esz);
    dim3 grid((rows + R128_ROWS - 1) / R128_ROWS), block(256);
    auto go = [&](auto* tag) {
      using T = std::remove_pointer_t<decltype(tag)>;
      auto kernel = al ? gated_rmsnorm128_kernel<T, true> : gated_rmsnorm128_kernel<T, false>;
      hipLaunchKernelGGL(kernel, grid, block, 0, s, (const T*)x, (const T*)g, (const T*)weight, (T*)y, rstd, rows,
                         g_group, g_ld, eps);
    };
    if (dtype == ZGDN_F32) go((float*)nullptr);
    else go((bf16*)nullptr);
    return check_launch(fn);
  }
  dim3 grid((rows + 3) / 4), block(256);
  if (dtype == ZGDN_F32)
    hipLaunchKernelGGL(gated_rmsnorm_kernel<float>, grid, block, 0, s, (const float*)x, (const float*)g,
                       (const float*)weight, (float*)y, rstd, rows, D, g_group, g_ld, eps);
  else
    hipLaunchKernelGGL(gated_rmsnorm_kernel<bf16>, grid, block, 0, s, (const bf16*)x, (const bf16*)g,
                       (const bf16*)weight, (bf16*)y, rstd, rows, D, g_group, g_ld, eps);
  return check_launch(fn);
}
