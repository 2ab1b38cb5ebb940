// Chunked (WY / UT form) gated delta rule in fp32 arithmetic: q/k/v in fp32 or bf16, head sizes K == V of 64
// or 128, 64-token chunks. The path zgdn_chunk_fwd takes for everything but bf16 inputs at K == V == 128 (which
// gdn_chunk.hip runs on bf16 MFMA): the fp32 model dtype of lm.py:556-602, and 64-wide heads.
//
// Per chunk of L <= 64 tokens and value head h, with in-chunk cumulative log decay G (G_t = g_1 + .. + g_t; rows
// past L carry g = 0, beta = 0 and zero q, k, v, so G_L is G at row 63), start state S [V, K] (value-major) and
// scale s:
//   A   = strictly-lower( beta_i exp(G_i - G_j) k_i.k_j ),   T = (I + A)^-1             (unit lower triangular)
//   P   = s lower-incl( exp(G_i - G_j) q_i.k_j ),            R = P T diag(beta e^G)
//   W'  = diag(Fk) T diag(beta e^G) K,   Ub' = diag(Fk) T diag(beta) V,   Fk_t = exp(G_L - G_t)
//   Q'  = s diag(e^G) Q - R K,           Ob  = P T diag(beta) V
//   then, chunk after chunk:  U' = Ub' - W' S^T,  O = Ob + Q' S^T,  S <- e^{G_L} S + U'^T K
// (O = s diag(e^G) Q S^T + P (Ub - W S^T) and S_end = e^{G_L} S + sum_t e^{G_L - G_t} u_t k_t^T, the chunked
// statement of the token loop of lm.py:574-583.) Phase 1 (chunk32_prep_kernel) forms W', Q', K, Ub', Ob and G_L
// of every (chunk, value head) item at once; phase 2 (chunk32_state_kernel) walks each sequence's chunks in
// order. Every product runs on v_mfma_f32_16x16x4_f32 (fp32 operands and accumulation) and the q/k L2 norm,
// the gate and sigmoid(beta) are fp32, so the results follow the fp32 token loop to fp32 rounding.
//
// v_mfma_f32_16x16x4_f32, lane l = 16 g + m: A[m][g], B[g][m]; D[4 g + i][m] in element i. Four products
// i = 0..3 take the contraction indices 16 n + 4 g + i of a 16-wide block n, so that one 16-byte read of
// columns 16 n + 4 g .. + 3 of a row serves a lane for all four (for both operands when both are rows of
// row-major matrices), and a D tile is the B operand of the next product as it stands (a lane's element i
// is row 4 g + i of column m, the B element of product i).
//
// Matrices in LDS are fp32 row-major with the 16-byte chunk c of row r stored at chunk c ^ (r % 16): a
// 16-byte read of 16 consecutive rows at one column (the A operands) then meets every bank once, and so
// does a 4-byte read of 4 rows x 16 columns (the B operands read as columns).
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "gdn_common.h"

namespace zgdn {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// log(1 + e^x) with torch's threshold (identity above 20), full-precision exp and log1p.
__device__ __forceinline__ float softplus_exact(float x) { return x > 20.f ? x : log1pf(expf(x)); }

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Byte offset of element (r, c) of a swizzled fp32 matrix with rows of RB bytes.
template <int RB>
__device__ __forceinline__ int swz(int r, int c) {
  return r * RB + ((((c >> 2) ^ (r & 15))) << 4) + ((c & 3) << 2);
}
__device__ __forceinline__ f32x4 ld4(const uint8_t* b, int off) { return *reinterpret_cast<const f32x4*>(b + off); }
__device__ __forceinline__ float ld1(const uint8_t* b, int off) { return *reinterpret_cast<const float*>(b + off); }
__device__ __forceinline__ void st4(uint8_t* b, int off, f32x4 v) { *reinterpret_cast<f32x4*>(b + off) = v; }
__device__ __forceinline__ void st1(uint8_t* b, int off, float v) { *reinterpret_cast<float*>(b + off) = v; }

// Workspace of one (chunk, value head) item, fp32, every block in the order phase 2 reads it (lane l = 16 g + m,
// token tile tt, key tile n, value tile vb, 64 lanes x 16 bytes = 1 KiB per block):
//   W'  [tt][n][l]: W'[16 tt + m][16 n + 4 g + i], i = 0..3       (A operands of W' S^T)
//   Q'  [tt][n][l]: Q'[16 tt + m][16 n + 4 g + i]                  (A operands of Q' S^T)
//   K^T [n][tt][l]: K[16 tt + 4 g + i][16 n + m]                    (A operands of the update U'^T K)
//   Ub' [vb][tt][l]: Ub'[16 tt + 4 g + i][16 vb + m]                 (D tiles: U' starts from them)
//   Ob  [vb][tt][l]: Ob[16 tt + 4 g + i][16 vb + m]                  (D tiles: O starts from them)
//   G_L (one float), padding to 256 bytes.
template <int D>
struct Ws32 {
  static constexpr int NK = D / 16;  // 16-wide key (and value) tiles
  static constexpr size_t BLK = (size_t)CHUNK_LEN * D * 4;
  static constexpr size_t W = 0, Q = BLK, K = 2 * BLK, U = 3 * BLK, O = 4 * BLK, G = 5 * BLK;
  static constexpr size_t ITEM = G + 256;
};

// ----------------------------------------------------------------------------------------------- phase 1
//
// One item (chunk x value head) at a time per workgroup of 16 waves, one workgroup per CU (148,736 bytes of LDS
// at D = 128: the chunk's q, k (L2-normalised when asked) and v rows, A (then R), T, P and the per-token
// factors); a workgroup walks the items item, item + grid, .. and loads the next item's rows into registers
// while it computes. Bound by the fp32 matrix rate: 2,060 products of 32 cycles at D = 128 are 6.9 us an item on
// a CU's four SIMDs, so the item is split to keep all four busy and the serial inverse out of the way:
//   1  rows -> LDS (their norm on the way, 16 lanes a row), the per-token factors (wave 15)
//   2  the 10 tiles of A (diagonal ones stored transposed) and 6 of P's
//   3  waves 0-3 (one a SIMD) invert A's diagonal blocks in registers
//   4  wave d < 4 the rest of block column d of T, its blocks passed on in registers; waves 4-7 P's last 4 tiles
//   5  R (waves 0-3), Ub, Ub', Ob (NK waves, a value tile each) and W', K^T (the others)
//   6  Q' (all waves)
// and the item's stores (164 KB) and the next one's loads (98 KB) in different stretches of it. The 1,024 items of
// T = 4096 at 16 heads take 83 us, of which 52 us are what their 268 MB take at the rate of a large copy; the 16
// items of T = 256, 4 heads, D = 64, one a workgroup, 13.7 us. With four waves an item, no loads ahead and the
// inverse's four levels behind each other: 111-114 and 18 us.
template <int D>
struct Lds32 {
  static constexpr int RB = D * 4;
  static constexpr int K = 0, Q = 64 * RB, V = 2 * 64 * RB, A = 3 * 64 * RB, T = A + 16384, P = T + 16384;
  static constexpr int F = P + 16384;                                   // factors: 64 floats each
  static constexpr int FG = F, FB = F + 256, FEG = F + 512, FFK = F + 768, FBW = F + 1024;  // G, beta, e^G, Fk, beta e^G
  static constexpr int BYTES = F + 1280;
};

constexpr int P32_WAVES = 16;

// Lower-triangle tile t (0..9) of a 4 x 4 block grid -> (row block, column block), row-major order.
__device__ __forceinline__ void tri_tile(int t, int& rb, int& cb) {
  rb = t < 1 ? 0 : (t < 3 ? 1 : (t < 6 ? 2 : 3));
  cb = t - rb * (rb + 1) / 2;
}

// Four consecutive elements of a q / k / v row as loaded through a buffer resource (zeros past its range) or from a
// pointer (zeros where it is null), and as floats.
template <typename T>
struct Row4;
template <>
struct Row4<float> {
  f32x4 v;
  __device__ __forceinline__ void load(Rsrc r, uint32_t off) {
    v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  }
  __device__ __forceinline__ void load(const float* p) {
    v = p != nullptr ? *reinterpret_cast<const f32x4*>(p) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ f32x4 get() const { return v; }
};
template <>
struct Row4<bf16> {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  u32x2 v;
  __device__ __forceinline__ void load(Rsrc r, uint32_t off) {
    v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  }
  __device__ __forceinline__ void load(const bf16* p) {
    v = p != nullptr ? *reinterpret_cast<const u32x2*>(p) : u32x2{0u, 0u};
  }
  __device__ __forceinline__ f32x4 get() const {
    return f32x4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                 __uint_as_float(v.y & 0xffff0000u)};
  }
};

// acc += X[16 xr .., 16 xc ..] . Y for a 16 x 16 block of a 64 x 64 LDS matrix X and a block Y held as a D tile.
__device__ __forceinline__ f32x4 blk_mm_d(const uint8_t* lb, int m, int g, int xm, int xr, int xc, f32x4 y, f32x4 acc) {
  const f32x4 a = ld4(lb, xm + swz<256>(16 * xr + m, 16 * xc + 4 * g));
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = mma(a[i], y[i], acc);
  return acc;
}
// Stores a D tile as block (br, bc) of a 64 x 64 LDS matrix; blk_put_t stores its transpose (one 16-byte write).
__device__ __forceinline__ void blk_put(uint8_t* lb, int m, int g, int mat, int br, int bc, f32x4 d) {
#pragma unroll
  for (int i = 0; i < 4; ++i) st1(lb, mat + swz<256>(16 * br + 4 * g + i, 16 * bc + m), d[i]);
}
__device__ __forceinline__ void blk_put_t(uint8_t* lb, int m, int g, int mat, int br, int bc, f32x4 d) {
  st4(lb, mat + swz<256>(16 * br + m, 16 * bc + 4 * g), d);
}

// Workgroup barrier over LDS traffic only: global loads and stores stay in flight across it.
__device__ __forceinline__ void bar() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A gate input as loaded through a buffer resource, and as a float.
template <typename T>
struct GateReg;
template <>
struct GateReg<float> {
  float v;
  __device__ __forceinline__ void load(Rsrc r, uint32_t off) {
    v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  }
  __device__ __forceinline__ void load(const float* p) { v = p != nullptr ? *p : 0.f; }
  __device__ __forceinline__ float get() const { return v; }
};
template <>
struct GateReg<bf16> {
  uint16_t v;
  __device__ __forceinline__ void load(Rsrc r, uint32_t off) { v = __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0); }
  __device__ __forceinline__ void load(const bf16* p) { v = p != nullptr ? *reinterpret_cast<const uint16_t*>(p) : 0; }
  __device__ __forceinline__ float get() const { return bf16_to_f32(v); }
};

// An item's rows (four elements of D / 64 column groups of row tid / 16 of each of q, k, v) and gate inputs.
template <typename TIn, typename TG, int D>
struct Rows32 {
  Row4<TIn> q[D / 64], k[D / 64], v[D / 64];
  GateReg<TG> g, beta;
  // waits for the loads (an empty asm that takes their registers)
  __device__ __forceinline__ void arrive() {
#pragma unroll
    for (int j = 0; j < D / 64; ++j) asm volatile("" : "+v"(q[j].v), "+v"(k[j].v), "+v"(v[j].v));
    asm volatile("" : "+v"(g.v), "+v"(beta.v));
  }
};

// The chunks of a launch's items: item i is (chunk, head) = (at(i / Hv), i % Hv); all of them, or chunks lo .. lo + n -
// 1 of each of B sequences of nct chunks.
struct Items32 {
  int lo, n, nct;
  __device__ __forceinline__ int chunk(int cc) const { return cc < n ? lo + cc : cc / n * nct + lo + cc % n; }
};

template <typename TIn, typename TG, int D>
__device__ __forceinline__ void load_item(Rows32<TIn, TG, D>& x, int item, const Items32& at, const TIn* q, const TIn* k, const TIn* v,
                                          const TG* g, const TG* beta, const int32_t* cu, const int32_t* chunk_idx,
                                          int n_seqs, int T, int Hk, int Hv, const RowStrides& rs) {
  const int c = at.chunk(item / Hv), h = item % Hv, hk = h / (Hv / Hk);
  const ChunkRange cr = chunk_range(c, cu, chunk_idx, T, n_seqs);
  constexpr uint32_t E = sizeof(TIn);
  const uint32_t r = threadIdx.x >> 4, c0 = (threadIdx.x & 15) * 4 * E;
  auto rows = [&](const TIn* p, long ld, int col, Row4<TIn>* out) {
    const Rsrc w = raw_rsrc(p + (size_t)cr.t0 * ld + col, (uint32_t)cr.len * (uint32_t)ld * E);
#pragma unroll
    for (int j = 0; j < D / 64; ++j) out[j].load(w, r * (uint32_t)ld * E + c0 + 64 * E * j);
  };
  rows(q, rs.q, hk * D, x.q);
  rows(k, rs.k, hk * D, x.k);
  rows(v, rs.v, h * D, x.v);
  // the gate inputs of token `lane` (zeros past the chunk end)
  const uint32_t gbytes = (uint32_t)cr.len * (uint32_t)rs.gb * (uint32_t)sizeof(TG);
  const uint32_t goff = (threadIdx.x & 63) * (uint32_t)rs.gb * (uint32_t)sizeof(TG);
  const size_t t = (size_t)cr.t0 * rs.gb + h;
  x.g.load(raw_rsrc(g + t, gbytes), goff);
  x.beta.load(raw_rsrc(beta + t, gbytes), goff);
}

// load_item for rows so far apart (64 of them 4 GiB or more) that a buffer resource, whose range and offsets are 32
// bits, does not reach the chunk's last ones: from pointers.
template <typename TIn, typename TG, int D>
__device__ __forceinline__ void load_item_far(Rows32<TIn, TG, D>& x, int item, const Items32& at, const TIn* q, const TIn* k,
                                              const TIn* v, const TG* g, const TG* beta, const int32_t* cu,
                                              const int32_t* chunk_idx, int n_seqs, int T, int Hk, int Hv,
                                              const RowStrides& rs) {
  const int c = at.chunk(item / Hv), h = item % Hv, hk = h / (Hv / Hk);
  const ChunkRange cr = chunk_range(c, cu, chunk_idx, T, n_seqs);
  const int r = threadIdx.x >> 4, c0 = (threadIdx.x & 15) * 4, lane = threadIdx.x & 63;
  auto rows = [&](const TIn* p, long ld, int col, Row4<TIn>* out) {
#pragma unroll
    for (int j = 0; j < D / 64; ++j) out[j].load(r < cr.len ? p + (size_t)(cr.t0 + r) * ld + col + c0 + 64 * j : nullptr);
  };
  rows(q, rs.q, hk * D, x.q);
  rows(k, rs.k, hk * D, x.k);
  rows(v, rs.v, h * D, x.v);
  const size_t t = (size_t)(cr.t0 + lane) * rs.gb + h;
  x.g.load(lane < cr.len ? g + t : nullptr);
  x.beta.load(lane < cr.len ? beta + t : nullptr);
}

// The inputs of phase 1.
template <typename TIn, typename TG>
struct Prep32 {
  const TIn *q, *k, *v;
  const TG *g, *beta;
  const float *A_log, *dt_bias;
  const int32_t *cu, *chunk_idx;
  int n_seqs, n_items, T, Hk, Hv, qk_l2norm;
  float scale;
  RowStrides rs;
  uint8_t* ws;
  Items32 at;
};

// Items first, first + stride, .. by one workgroup.
template <typename TIn, typename TG, int D, bool GATE, bool FAR>
__device__ __forceinline__ void prep32(uint8_t* lb, const Prep32<TIn, TG>& p, int first, int stride) {
  using L = Lds32<D>;
  using WS = Ws32<D>;
  constexpr int RB = L::RB, NK = WS::NK;
  const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
  const int n_items = p.n_items, Hv = p.Hv;
  Rows32<TIn, TG, D> R;
  if (first >= n_items) return;
  auto load = [&](int item) {
    if constexpr (FAR)
      load_item_far<TIn, TG, D>(R, item, p.at, p.q, p.k, p.v, p.g, p.beta, p.cu, p.chunk_idx, p.n_seqs, p.T, p.Hk, Hv, p.rs);
    else
      load_item<TIn, TG, D>(R, item, p.at, p.q, p.k, p.v, p.g, p.beta, p.cu, p.chunk_idx, p.n_seqs, p.T, p.Hk, Hv, p.rs);
  };
  load(first);

  for (int item = first; item < n_items; item += stride) {
    // the lane's and wave's indexes pass through an empty asm per item: the addresses derived from them are then
    // formed inside the item instead of being hoisted out of the loop, where they would not fit the registers
    int tid = threadIdx.x, wave = wave_id();
    asm volatile("" : "+v"(tid));
    asm volatile("" : "+s"(wave));
    const int l = tid & 63, m = l & 15, gq = l >> 4;
    const int c = p.at.chunk(item / Hv), h = item % Hv;
    const int len = chunk_range(c, p.cu, p.chunk_idx, p.T, p.n_seqs).len;
    uint8_t* out = p.ws + ((size_t)c * Hv + h) * WS::ITEM;
    const float scale = p.scale;

    // ---- 1. rows of q, k (key head hk) and v (value head h) into LDS as fp32 (zeros past the chunk end), q and k
    // L2-normalised when asked: x * rsqrt(sum x^2 + 1e-6)
    {
      const int r = tid >> 4, c0 = (tid & 15) * 4;
      f32x4 xq[D / 64], xk[D / 64];
      float sq = 0.f, sk = 0.f;
#pragma unroll
      for (int j = 0; j < D / 64; ++j) {
        xq[j] = R.q[j].get();
        xk[j] = R.k[j].get();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sq = fmaf(xq[j][e], xq[j][e], sq);
          sk = fmaf(xk[j][e], xk[j][e], sk);
        }
      }
      float rq = 1.f, rk = 1.f;
      if (p.qk_l2norm) {
        rq = 1.f / sqrtf(group_sum<16>(sq) + 1e-6f);
        rk = 1.f / sqrtf(group_sum<16>(sk) + 1e-6f);
      }
#pragma unroll
      for (int j = 0; j < D / 64; ++j) {
        st4(lb, L::Q + swz<RB>(r, c0 + 64 * j), xq[j] * rq);
        st4(lb, L::K + swz<RB>(r, c0 + 64 * j), xk[j] * rk);
        st4(lb, L::V + swz<RB>(r, c0 + 64 * j), R.v[j].get());
      }
    }
    // per-token factors (wave 15, lane = token): g (the in-kernel gate when asked), beta, G = inclusive scan
    if (wave == P32_WAVES - 1) {
      float gt = 0.f, bt = 0.f;
      if (l < len) {
        const float gr = R.g.get(), br = R.beta.get();
        gt = GATE ? -expf(p.A_log[h]) * softplus_exact(gr + p.dt_bias[h]) : gr;
        bt = p.rs.beta_sigmoid ? 1.f / (1.f + expf(-br)) : br;
      }
      float G = gt;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const float o = __shfl_up(G, d, 64);
        if (l >= d) G += o;
      }
      const float GL = __shfl(G, 63, 64);
      const float eg = expf(G);
      st1(lb, L::FG + 4 * l, G);
      st1(lb, L::FB + 4 * l, bt);
      st1(lb, L::FEG + 4 * l, eg);
      st1(lb, L::FFK + 4 * l, expf(GL - G));
      st1(lb, L::FBW + 4 * l, bt * eg);
      if (l == 0) *reinterpret_cast<float*>(out + WS::G) = GL;
    }
    bar();

    // ---- A = strictly-lower(beta_i e^{G_i - G_j} k_i.k_j) (tiles u = 0 .. 9), P = s lower-incl(e^{G_i - G_j}
    // q_i.k_j) (u = 10 .. 19)
    auto ap_tile = [&](int u) {
      const bool isP = u >= 10;
      int I, J;
      tri_tile(isP ? u - 10 : u, I, J);
      f32x4 a0 = z4, a1 = z4;
#pragma unroll
      for (int n = 0; n < NK; n += 2) {
        const f32x4 xa = ld4(lb, (isP ? L::Q : L::K) + swz<RB>(16 * I + m, 16 * n + 4 * gq));
        const f32x4 xb = ld4(lb, L::K + swz<RB>(16 * J + m, 16 * n + 4 * gq));
        const f32x4 ya = ld4(lb, (isP ? L::Q : L::K) + swz<RB>(16 * I + m, 16 * n + 16 + 4 * gq));
        const f32x4 yb = ld4(lb, L::K + swz<RB>(16 * J + m, 16 * n + 16 + 4 * gq));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a0 = mma(xa[i], xb[i], a0);
          a1 = mma(ya[i], yb[i], a1);
        }
      }
      f32x4 acc = a0 + a1;
      const int cc = 16 * J + m, r0 = 16 * I + 4 * gq;
      const float Gc = ld1(lb, L::FG + 4 * cc);
      const f32x4 Gr = ld4(lb, L::FG + 4 * r0), br = ld4(lb, L::FB + 4 * r0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool keep = isP ? r0 + i >= cc : r0 + i > cc;
        acc[i] = keep ? (isP ? scale : br[i]) * expf(Gr[i] - Gc) * acc[i] : 0.f;
      }
      if (isP || I != J)
        blk_put(lb, m, gq, isP ? L::P : L::A, I, J, acc);
      else
        blk_put_t(lb, m, gq, L::A, I, I, acc);
    };
    // ---- 2. A and P's first 6 tiles
    ap_tile(wave);
    bar();
    // the next item's rows (the last item's again past it), in flight over steps 3 and 4: by now the stores of the
    // item before are through, behind which these loads would hold up the waves that issue them
    load(min(item + stride, n_items - 1));

    // ---- 3. T = (I + A)^-1, the diagonal blocks: wave d < 4 by right-looking substitution on block d held as a D
    // tile (lane: rows 4 gq + i of column m). Step j subtracts column j of the block (row j of its transpose,
    // read ahead) times row j of the result, which the lanes of group j / 4 hand to the others by lane swaps.
    f32x4 td[4];  // wave d < 4: column d of T as D tiles, td[i] = T_(d + i, d)
    if (wave < 4) {
      constexpr int AHEAD = 4;  // reads ahead (all 15 would not fit the registers beside the next item's rows)
      f32x4 a[AHEAD];
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) a[j] = ld4(lb, L::A + swz<256>(16 * wave + j, 16 * wave + 4 * gq));
      f32x4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = 4 * gq + i == m ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < 15; ++j) {
        const uint32_t own = __float_as_uint(x[j & 3]);
        auto p = __builtin_amdgcn_permlane32_swap(own, own, false, false);
        const uint32_t hw = p[j >> 3];  // groups (0, 1) or (2, 3) in both halves
        p = __builtin_amdgcn_permlane16_swap(hw, hw, false, false);
        const float t = __uint_as_float(p[(j >> 2) & 1]);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = fmaf(-a[j % AHEAD][i], t, x[i]);
        if (j + AHEAD < 15) a[j % AHEAD] = ld4(lb, L::A + swz<256>(16 * wave + j + AHEAD, 16 * wave + 4 * gq));
      }
      td[0] = x;
      blk_put(lb, m, gq, L::T, wave, wave, x);
    }
    bar();
    // ---- 4. wave d < 4: the rest of column d, T_id = -T_ii sum_{d <= m < i} A_im T_md, its blocks taken on as D
    // tiles (no other column's off-diagonal block enters); waves 4-7 form P's last 4 tiles
    if (wave < 4) {
#pragma unroll
      for (int i = 1; i < 4; ++i) {
        td[i] = z4;
        if (wave + i < 4) {  // (wave-uniform)
          f32x4 y = z4;
#pragma unroll
          for (int e = 0; e < i; ++e) y = blk_mm_d(lb, m, gq, L::A, wave + i, wave + e, td[e], y);
          td[i] = -blk_mm_d(lb, m, gq, L::T, wave + i, wave + i, y, z4);
          blk_put(lb, m, gq, L::T, wave + i, wave, td[i]);
        }
      }
    } else if (wave < 8) {
      ap_tile(12 + wave);
    }
    bar();

    // the next item's rows are waited for here, ahead of this item's stores: a wait behind them would cover the
    // stores too (one counter), i.e. every workgroup's burst of writes
    R.arrive();
    // ---- 5. beside each other (all of them need T and P alone):
    if (wave < 4) {
      // R = P T diag(beta e^G) into A's place: wave d column d, from its D tiles
      const float bw = ld1(lb, L::FBW + 4 * (16 * wave + m));
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (wave + i < 4) {
          f32x4 acc = z4;
#pragma unroll
          for (int e = 0; e <= i; ++e) acc = blk_mm_d(lb, m, gq, L::P, wave + i, wave + e, td[e], acc);
          blk_put(lb, m, gq, L::A, wave + i, wave, acc * bw);
          __builtin_amdgcn_sched_barrier(0);
        }
    } else if (wave < 4 + NK) {
      // Ub = T diag(beta) V and Ob = P Ub (value tile vb); Ub' = diag(Fk) Ub
      const int vb = wave - 4;
      f32x4 ub[4];
#pragma unroll
      for (int I = 0; I < 4; ++I) ub[I] = z4;
#pragma unroll
      for (int J = 0; J < 4; ++J) {
        const f32x4 b4 = ld4(lb, L::FB + 4 * (16 * J + 4 * gq));
        f32x4 vv;
#pragma unroll
        for (int i = 0; i < 4; ++i) vv[i] = b4[i] * ld1(lb, L::V + swz<RB>(16 * J + 4 * gq + i, 16 * vb + m));
#pragma unroll
        for (int I = J; I < 4; ++I) ub[I] = blk_mm_d(lb, m, gq, L::T, I, J, vv, ub[I]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int I = 0; I < 4; ++I) {
        f32x4 ob = z4;
#pragma unroll
        for (int J = 0; J <= I; ++J) ob = blk_mm_d(lb, m, gq, L::P, I, J, ub[J], ob);
        const f32x4 fk = ld4(lb, L::FFK + 4 * (16 * I + 4 * gq));
        st4(out, (int)(WS::U + ((size_t)(vb * 4 + I) * 64 + l) * 16), ub[I] * fk);
        st4(out, (int)(WS::O + ((size_t)(vb * 4 + I) * 64 + l) * 16), ob);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // W'^T = K^T (diag(Fk) T diag(beta e^G))^T, with K^T: each D tile is the phase-2 A operand block (tt = I, n)
      for (int n = wave - 4 - NK; n < NK; n += 12 - NK) {
        f32x4 aw[4];
#pragma unroll
        for (int I = 0; I < 4; ++I) aw[I] = z4;
#pragma unroll
        for (int J = 0; J < 4; ++J) {
          const f32x4 bw = ld4(lb, L::FBW + 4 * (16 * J + 4 * gq));
          f32x4 kv, kb;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            kv[i] = ld1(lb, L::K + swz<RB>(16 * J + 4 * gq + i, 16 * n + m));
            kb[i] = kv[i] * bw[i];
          }
          st4(out, (int)(WS::K + ((size_t)(n * 4 + J) * 64 + l) * 16), kv);
#pragma unroll
          for (int I = J; I < 4; ++I) {
            const f32x4 t4 = ld4(lb, L::T + swz<256>(16 * I + m, 16 * J + 4 * gq));
#pragma unroll
            for (int i = 0; i < 4; ++i) aw[I] = mma(kb[i], t4[i], aw[I]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int I = 0; I < 4; ++I)
          st4(out, (int)(WS::W + ((size_t)(I * NK + n) * 64 + l) * 16), aw[I] * ld1(lb, L::FFK + 4 * (16 * I + m)));
      }
    }
    bar();

    // ---- 6. Q'^T = s Q^T diag(e^G) - K^T R^T: (token tile, key tile) jobs, each wave one long and one short one
    // (D = 128: token tiles {3, 0} or {2, 1} of one key tile; D = 64: one job a wave)
#pragma unroll
    for (int half = 0; half < NK / 4; ++half) {
      const int n = wave % NK, u = wave / NK;
      const int I = NK == 8 ? (half == 0 ? 3 - u : u) : 3 - u;
      const int tr = 16 * I + m;
      f32x4 aq = ld4(lb, L::Q + swz<RB>(tr, 16 * n + 4 * gq)) * (scale * ld1(lb, L::FEG + 4 * tr));
      for (int J = 0; J <= I; ++J) {
        const f32x4 r4 = ld4(lb, L::A + swz<256>(tr, 16 * J + 4 * gq));
#pragma unroll
        for (int i = 0; i < 4; ++i) aq = mma(ld1(lb, L::K + swz<RB>(16 * J + 4 * gq + i, 16 * n + m)), -r4[i], aq);
      }
      st4(out, (int)(WS::Q + ((size_t)(I * NK + n) * 64 + l) * 16), aq);
    }
    bar();  // the next item's rows overwrite the LDS
  }
}

template <typename TIn, typename TG, int D, bool GATE, bool FAR>
__global__ __launch_bounds__(64 * P32_WAVES) void chunk32_prep_kernel(const Prep32<TIn, TG> p) {
  extern __shared__ f32x4 lds32[];
  prep32<TIn, TG, D, GATE, FAR>(reinterpret_cast<uint8_t*>(lds32), p, blockIdx.x, gridDim.x);
}

// ----------------------------------------------------------------------------------------------- phase 2
//
// One workgroup of 8 waves per (sequence, value head, 16 value rows vb). Wave n < NK holds key tile n of the
// state rows as a D tile of S^T (lane: S[16 vb + m][16 n + 4 g + i]), which is the B operand of W' S^T and Q' S^T
// as it stands. Per chunk: the tiles go to LDS; wave tt < 4 forms U' = Ub' - W' S^T of token tile tt over all keys
// and puts it in LDS, wave 4 + tt the outputs O = Ob + Q' S^T of token tile tt; then every wave n < NK takes all
// of U' into its tile, S^T <- e^{G_L} S^T + K^T U'. Each SIMD runs one wave of either kind, so its matrix unit
// (96 products of 32 cycles a chunk at D = 128, 1.28 us, the pass's bound) has a second wave to work for while
// one is at a barrier or in LDS; the next chunk's operands are loaded in three groups between the phases, as
// loads issued in one burst hold up the waves that issue them. T = 4096 at 16 heads, D = 128 (64 chunks): 129 us,
// 2.0 us a chunk; T = 256, 4 heads, D = 64: 5.5 us. With 4 waves, each doing all three products over its quarter
// of the keys (partial sums through LDS) and the loads in one burst: 190 and 9.6 us.
template <int D>
struct Ops32 {
  static constexpr int NK = D / 16;
  f32x4 A[NK];  // W' (waves 0-3) or Q' (4-7) of this wave's token tile
  f32x4 K[4];   // K^T of this wave's key tile
  f32x4 X;      // Ub' or Ob of this wave's token tile
  float GL;
};

// Stores a D tile of outputs (rows r0 .. r0 + 3 of column col of the chunk's rows, lanes l and l ^ 1 adjacent
// columns) through a buffer resource that ends with the chunk's last token: two rows a lane as column pairs.
template <typename TOut>
__device__ __forceinline__ void store_tile32(Rsrc w, uint32_t row_bytes, int r0, int col, f32x4 d) {
  const bool odd = (threadIdx.x & 1) != 0;
  const float x0 = dpp<DPP_QUAD_XOR1>(odd ? d[0] : d[2]), x1 = dpp<DPP_QUAD_XOR1>(odd ? d[1] : d[3]);
  const float a0 = odd ? x0 : d[0], b0 = odd ? d[2] : x0, a1 = odd ? x1 : d[1], b1 = odd ? d[3] : x1;
  const uint32_t off = (uint32_t)(r0 + (odd ? 2 : 0)) * row_bytes + (uint32_t)(col & ~1) * (uint32_t)sizeof(TOut);
  if constexpr (sizeof(TOut) == 2) {
    __builtin_amdgcn_raw_buffer_store_b32(pack_bf16x2(a0, b0), w, off, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b32(pack_bf16x2(a1, b1), w, off + row_bytes, 0, 0);
  } else {
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(a0), __float_as_uint(b0)}, w, off, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(a1), __float_as_uint(b1)}, w, off + row_bytes, 0, 0);
  }
}

template <int D>
struct StateShared32 {
  f32x4 S[D / 16][64];  // the state's D tiles
  f32x4 U[4][64];       // U' of the 4 token tiles
};

// The chunk loop of one wave (U: waves 0-3, else the output waves).
template <bool U, typename TOut, int D>
__device__ __forceinline__ void state_loop32(StateShared32<D>& sh, f32x4& st, const uint8_t* ws, TOut* o, int c0,
                                             int nc, int bos, int len, int Hv, int h, int vb, int wave) {
  using WS = Ws32<D>;
  constexpr int NK = WS::NK;
  const int l = threadIdx.x & 63, m = l & 15, gq = l >> 4;
  const int tt = wave & 3;
  const bool upd = wave < NK;  // this wave holds a state tile (all 8 at D = 128, the U waves at 64)
  const uint32_t offA = (uint32_t)((U ? WS::W : WS::Q) + (size_t)tt * NK * 1024) + 16u * l;
  const uint32_t offX = (uint32_t)((U ? WS::U : WS::O) + (size_t)(vb * 4 + tt) * 1024) + 16u * l;
  const uint32_t offK = (uint32_t)(WS::K + (size_t)(wave & (NK - 1)) * 4 * 1024) + 16u * l;
  auto chunk_ws = [&](int ci) { return raw_rsrc(ws + ((size_t)(c0 + ci) * Hv + h) * WS::ITEM, (uint32_t)WS::ITEM); };
  auto ld = [](Rsrc w, uint32_t off) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(w, off, 0, 0));
  };
  auto fetch1 = [&](Rsrc w, Ops32<D>& p) {
#pragma unroll
    for (int n = 0; n < NK / 2; ++n) p.A[n] = ld(w, offA + 1024u * n);
    p.GL = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(w, 0, (int)WS::G, 0));
  };
  auto fetch2 = [&](Rsrc w, Ops32<D>& p) {
#pragma unroll
    for (int n = NK / 2; n < NK; ++n) p.A[n] = ld(w, offA + 1024u * n);
    p.X = ld(w, offX);
  };
  auto fetch3 = [&](Rsrc w, Ops32<D>& p) {
#pragma unroll
    for (int t = 0; t < 4; ++t) p.K[t] = ld(w, offK + 1024u * t);
  };
  const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
  auto process = [&](int ci, const Ops32<D>& cur, int ni, Ops32<D>& nxt) {
    if (upd) sh.S[wave][l] = st;
    const Rsrc wn = chunk_ws(ni);
    fetch1(wn, nxt);
    bar();
    f32x4 x0 = z4, x1 = z4;
#pragma unroll
    for (int n = 0; n < NK; n += 2) {
      const f32x4 s0 = sh.S[n][l], s1 = sh.S[n + 1][l];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x0 = mma(cur.A[n][i], s0[i], x0);
        x1 = mma(cur.A[n + 1][i], s1[i], x1);
      }
    }
    f32x4 ov = z4;
    if constexpr (U)
      sh.U[tt][l] = cur.X - (x0 + x1);
    else
      ov = cur.X + (x0 + x1);
    fetch2(wn, nxt);
    bar();
    fetch3(wn, nxt);
    if (upd) {
      f32x4 s0 = st * expf(cur.GL), s1 = z4;
#pragma unroll
      for (int t = 0; t < 4; t += 2) {
        const f32x4 u0 = sh.U[t][l], u1 = sh.U[t + 1][l];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s0 = mma(cur.K[t][i], u0[i], s0);
          s1 = mma(cur.K[t + 1][i], u1[i], s1);
        }
      }
      st = s0 + s1;
    }
    if constexpr (!U) {
      const uint32_t row = (uint32_t)Hv * D * (uint32_t)sizeof(TOut);
      const int tl = min(CHUNK_LEN, len - ci * CHUNK_LEN);
      store_tile32<TOut>(raw_rsrc(o + ((size_t)(bos + ci * CHUNK_LEN) * Hv + h) * D + 16 * vb, (uint32_t)tl * row), row,
                         16 * tt + 4 * gq, m, ov);
    }
  };
  // two register buffers in turn, filled one chunk ahead (the last chunk is fetched again at the end, so that
  // every path issues the same loads)
  const int last = nc - 1;
  Ops32<D> b0, b1;
  {
    const Rsrc w0 = chunk_ws(0);
    fetch1(w0, b0);
    fetch2(w0, b0);
    fetch3(w0, b0);
  }
  process(0, b0, min(1, last), b1);
  int ci = 1;
  for (; ci + 1 < nc; ci += 2) {
    process(ci, b1, ci + 1, b0);
    process(ci + 1, b0, min(ci + 2, last), b1);
  }
  if (ci < nc) process(ci, b1, ci, b0);
}

// The inputs of the state pass: chunks lo .. lo + n - 1 of each sequence, from s_in (zeros without it) to s_out.
template <typename TOut>
struct State32 {
  const uint8_t* ws;
  const float* s_in;
  float* s_out;
  TOut* o;
  const int32_t* cu;
  int n_seqs, n_chunks, T, Hv, lo, n;
};

template <typename TOut, int D>
__device__ __forceinline__ void state32(StateShared32<D>& sh, const State32<TOut>& p, int id) {
  constexpr int NK = Ws32<D>::NK;
  // the NK workgroups of one (sequence, head) share an id % 8, so they run on one XCD and share its L2 copy of
  // the chunk workspace (the grid is padded to whole groups of 8 NK)
  const int pair = (id / (8 * NK)) * 8 + id % 8, vb = (id % (8 * NK)) / 8;
  if (pair >= p.n_seqs * p.Hv) return;
  const int seq = pair / p.Hv, h = pair % p.Hv;
  const int wave = wave_id(), l = threadIdx.x & 63, m = l & 15, gq = l >> 4;
  int c0, bos, len;
  seq_chunks(p.cu, seq, p.T, c0, bos, len);
  c0 += p.lo;
  bos += p.lo * CHUNK_LEN;
  len = max(0, len - p.lo * CHUNK_LEN);
  // chunks past the workspace (a chunk table shorter than the sequences need) are not read
  const int nc = max(0, min(min((len + CHUNK_LEN - 1) / CHUNK_LEN, p.n), p.n_chunks - c0));

  const size_t at = ((size_t)pair * D + 16 * vb + m) * D + 16 * (wave & (NK - 1)) + 4 * gq;  // this lane's entries
  f32x4 st = {0.f, 0.f, 0.f, 0.f};
  if (p.s_in != nullptr) st = *reinterpret_cast<const f32x4*>(p.s_in + at);
  if (nc > 0) {
    if (wave < 4)
      state_loop32<true, TOut, D>(sh, st, p.ws, p.o, c0, nc, bos, len, p.Hv, h, vb, wave);
    else
      state_loop32<false, TOut, D>(sh, st, p.ws, p.o, c0, nc, bos, len, p.Hv, h, vb, wave);
  }
  if (p.s_out != nullptr && wave < NK) *reinterpret_cast<f32x4*>(p.s_out + at) = st;
}

template <typename TOut, int D>
__global__ __launch_bounds__(512) void chunk32_state_kernel(const State32<TOut> p) {
  __shared__ StateShared32<D> sh;
  state32<TOut, D>(sh, p, blockIdx.x);
}

// Both phases side by side, on different chunks: the first n_state workgroups run the state pass over chunks that an
// earlier launch prepared, the others prepare the chunks after them (the launches' order is all the synchronisation).
// Each workgroup has a CU to itself (phase 1's LDS). For the batches whose state pass leaves CUs idle; see slices32.
template <typename TIn, typename TG, int D, bool GATE>
__global__ __launch_bounds__(64 * P32_WAVES) void chunk32_both_kernel(const Prep32<TIn, TG> p, const State32<TIn> st,
                                                                      int n_state) {
  extern __shared__ f32x4 lds32[];
  static_assert(sizeof(StateShared32<D>) <= Lds32<D>::BYTES, "the state pass's LDS");
  if ((int)blockIdx.x < n_state) {
    if (threadIdx.x >= 512) return;  // (whole waves; the barriers count the waves that are left)
    state32<TIn, D>(*reinterpret_cast<StateShared32<D>*>(lds32), st, blockIdx.x);
  } else {
    prep32<TIn, TG, D, GATE, false>(reinterpret_cast<uint8_t*>(lds32), p, blockIdx.x - n_state, gridDim.x - n_state);
  }
}

// Phase 1's dynamic LDS is above the default 64 KiB (148,736 bytes at D = 128, 99,584 at 64): raised once per device and kernel (the first
// call on that device); false when the device refuses.
constexpr int C32_MAX_DEVICES = 64;
template <typename K>
bool lds_ready(K kernel, int bytes, std::atomic<signed char>* state) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= C32_MAX_DEVICES) return false;
  const signed char s = state[dev].load(std::memory_order_acquire);
  if (s != 0) return s > 0;
  const bool ok = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) ==
                  hipSuccess;
  if (!ok) (void)hipGetLastError();
  state[dev].store(ok ? 1 : -1, std::memory_order_release);
  return ok;
}

// The state pass's workgroups: whole groups of 8 NK (8 chains, one on each XCD).
template <int D>
constexpr int state_grid(int chains) {
  return (chains + 7) / 8 * 8 * (D / 16);
}

// Slices of a call of N sequences of nct chunks (1: phase 1, then the state pass). A state pass of few chains leaves CUs
// idle, and phase 1 of the next slice of chunks runs on them beside it (chunk32_both_kernel). Times in us measured on
// MI355X: a round of phase-1 items (one a CU) and a chunk of the state pass 19 and 2.0 at D = 128, 9 and 1.0 at 64; a
// launch more costs about 2. Taken where the sum over the slices is the smallest, by 3 % or more. Measured, in two
// launches -> sliced: D = 128, 16 heads, 2048 tokens 102 -> 92 us (2 slices), 4096 200 -> 170 (4), 8192 453 -> 331 (8:
// a slice's workspace is read while it is still in the last-level cache); 8 heads, 4096 tokens 160 -> 147 (2); 4 heads,
// 9580 tokens 334 -> 306 (3); D = 64, 16 heads, 4096 tokens 109 -> 104 (4).
template <int D>
int slices32(int N, int nct, int Hv, int n_cu) {
  constexpr double item = D == 128 ? 19. : 9., chunk = D == 128 ? 2. : 1., launch = 2.;
  // CUs of the state pass, on the XCDs that have most of it, and left beside it (the items spread over all XCDs)
  const int ns = state_grid<D>(N * Hv), rest = n_cu - ns;
  if (ns > n_cu / 2) return 1;
  auto prep = [&](int n, int cus) { return item * ((N * n * Hv + cus - 1) / cus); };
  const double plain = prep(nct, n_cu) + chunk * nct;
  double best = 0.97 * plain;
  int slices = 1;
  for (int k = 2; k <= 8 && 4 * k <= nct; ++k) {
    const int n = (nct + k - 1) / k;  // (the last slice may be shorter)
    const double t = prep(n, n_cu) + (k - 1) * (std::max(chunk * n + launch, prep(n, rest)) + launch) + chunk * n;
    if (t < best) {
      best = t;
      slices = k;
    }
  }
  return slices;
}

// Whether a chunk of rows `ld` elements apart is past a buffer resource's 32-bit range.
inline bool far_rows(long ld, size_t elem) { return (unsigned long long)ld * CHUNK_LEN * elem > UINT32_MAX; }

template <typename TIn, typename TG, int D, bool GATE>
int launch32(const char* fn, Prep32<TIn, TG> p, State32<TIn> st, int N, int nct, hipStream_t s) {
  static std::atomic<signed char> prep_lds[2][C32_MAX_DEVICES], both_lds[C32_MAX_DEVICES];
  constexpr int bytes = Lds32<D>::BYTES;
  const bool far = far_rows(std::max({p.rs.q, p.rs.k, p.rs.v}), sizeof(TIn)) || far_rows(p.rs.gb, sizeof(TG));
  auto prep_kernel = far ? chunk32_prep_kernel<TIn, TG, D, GATE, true> : chunk32_prep_kernel<TIn, TG, D, GATE, false>;
  if (!lds_ready(prep_kernel, bytes, prep_lds[far]))
    return fail(ZGDN_EHIP, "%s: the device refused %d bytes of LDS for the fp32 chunk kernel", fn, bytes);
  const int n_cu = device_cus(), n_state = state_grid<D>(N * p.Hv);
  // the states between slices stay in s_out; packed sequences (of different lengths) are not sliced, nor are rows
  // far apart
  int k = p.cu == nullptr && st.s_out != nullptr && !far ? slices32<D>(N, nct, p.Hv, n_cu) : 1;
  if (k > 1 && !lds_ready(chunk32_both_kernel<TIn, TG, D, GATE>, bytes, both_lds)) k = 1;
  const int n = k > 1 ? (nct + k - 1) / k : p.at.n;
  auto prep_of = [&](int lo) {
    Prep32<TIn, TG> x = p;
    if (k > 1) {
      x.at = Items32{lo, std::min(n, nct - lo), nct};
      x.n_items = N * x.at.n * p.Hv;
    }
    return x;
  };
  if (p.n_items > 0) {
    const Prep32<TIn, TG> x = prep_of(0);
    hipLaunchKernelGGL(prep_kernel, dim3(std::min(x.n_items, n_cu)), dim3(64 * P32_WAVES), bytes, s, x);
  }
  if (k > 1) {
    st.n = n;
    for (; st.lo + n < nct; st.lo += n) {
      const Prep32<TIn, TG> x = prep_of(st.lo + n);
      const int rest = std::min(x.n_items, n_cu - n_state);
      hipLaunchKernelGGL((chunk32_both_kernel<TIn, TG, D, GATE>), dim3(n_state + rest), dim3(64 * P32_WAVES), bytes, s, x, st,
                         n_state);
      st.s_in = st.s_out;
    }
  }
  hipLaunchKernelGGL((chunk32_state_kernel<TIn, D>), dim3(n_state), dim3(512), 0, s, st);
  return check_launch(fn);
}

template <typename TIn, int D>
int run32(const char* fn, int n_chunks, const void* q, const void* k, const void* v, const void* g, int gb_dtype,
          const void* beta, const float* A_log, const float* dt_bias, const int32_t* cu, const int32_t* chunk_idx,
          int N, int T, int Hk, int Hv, float scale, int qk_l2norm, const RowStrides& rs, const float* s_in,
          float* s_out, void* o, uint8_t* ws, hipStream_t s) {
  const int nct = (T + CHUNK_LEN - 1) / CHUNK_LEN;
  const State32<TIn> st{ws, s_in, s_out, (TIn*)o, cu, N, n_chunks, T, Hv, 0, std::max(1, n_chunks)};
  auto go = [&](auto* tag, auto gate) {
    using TG = std::remove_pointer_t<decltype(tag)>;
    const Prep32<TIn, TG> p{(const TIn*)q, (const TIn*)k, (const TIn*)v, (const TG*)g, (const TG*)beta, A_log, dt_bias, cu,
                            chunk_idx, N, n_chunks * Hv, T, Hk, Hv, qk_l2norm, scale, rs, ws,
                            Items32{0, std::max(1, n_chunks), 0}};
    return launch32<TIn, TG, D, decltype(gate)::value>(fn, p, st, N, nct, s);
  };
  if (gb_dtype == ZGDN_F32)
    return A_log != nullptr ? go((float*)nullptr, std::true_type{}) : go((float*)nullptr, std::false_type{});
  return A_log != nullptr ? go((bf16*)nullptr, std::true_type{}) : go((bf16*)nullptr, std::false_type{});
}

}  // namespace

size_t chunk32_item_bytes(int D) { return D == 64 ? Ws32<64>::ITEM : Ws32<128>::ITEM; }

// The fp32-arithmetic chunked forward (arguments checked by the caller): q, k, v, o of element type qkv_dtype,
// K == V == D in {64, 128}; the workspace holds n_chunks * Hv items of chunk32_item_bytes(D).
int chunk32_fwd(const char* fn, const void* q, const void* k, const void* v, int qkv_dtype, const void* g,
                const void* beta, int gb_dtype, const float* A_log, const float* dt_bias, int qk_l2norm,
                const float* s_in, float* s_out, void* o, const int32_t* cu, const int32_t* chunk_idx, int N,
                int n_chunks, int T, int Hk, int Hv, int D, float scale, const RowStrides& rs, void* workspace,
                hipStream_t s) {
  uint8_t* ws = (uint8_t*)workspace;
#define ZGDN_RUN32(TIN, DD)                                                                                        \
  run32<TIN, DD>(fn, n_chunks, q, k, v, g, gb_dtype, beta, A_log, dt_bias, cu, chunk_idx, N, T, Hk, Hv, scale,    \
                 qk_l2norm, rs, s_in, s_out, o, ws, s)
  if (qkv_dtype == ZGDN_F32) return D == 64 ? ZGDN_RUN32(float, 64) : ZGDN_RUN32(float, 128);
  return D == 64 ? ZGDN_RUN32(bf16, 64) : ZGDN_RUN32(bf16, 128);
#undef ZGDN_RUN32
}

}  // namespace zgdn

// Slices that an unpacked call of B sequences with a final state takes on the current device (for tests).
extern "C" int zgdn_chunk32_slices(int D, int B, int T, int Hv) {
  using namespace zgdn;
  const int nct = (T + CHUNK_LEN - 1) / CHUNK_LEN;
  return D == 64 ? slices32<64>(B, nct, Hv, device_cus()) : slices32<128>(B, nct, Hv, device_cus());
}
