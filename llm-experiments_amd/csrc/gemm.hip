// Projections over many rows (the model's prompt prefill): a tiled GEMM with
// fp32 operands and fp32 accuracy on the bf16 matrix cores,
// y = act(LN(x) . w_t^T + bias) + residual, with the semantics of skv_linear
// (the reference's jnp.dot projections, simple-llm/src/jax_backend.py:110-129,
// 147, over every position of a window). skv_linear runs this kernel when a
// call has more than 64 rows; the decode step's few rows stay on k_linear
// (model_ops.hip), which is bound by reading the weights rather than by the
// products.
//
// Products: every fp32 operand is split into three bf16 parts and a product
// takes six partial products on v_mfma_f32_32x32x16_bf16 (split_bf16.h).
// Measured on MI355X against the fp32 MFMA form of the same kernel (128 x 128
// tiles, one LDS stage): 2048 x 50304 x 768 1390 -> 853 us (186 TFLOP/s),
// 2048 x 3072 x 768 with LayerNorm 137 -> 69 us, 2048 x 768 x 3072 220 -> 84
// us, 111 x 640 x 2560 192 -> 49 us; error against float64 (relative
// 2-norm) 5.0e-7 -> 4.2e-7 at K = 768 and 9.9e-7 -> 8.6e-7 at K = 3072.
// Outputs that are not finite (an infinity, or a value too large to split,
// among the operands) are computed again on v_mfma_f32_32x32x2_f32, which
// gives what fp32 products give.
//
// Design: a workgroup computes BM x BN outputs, its wavefronts 64 x 64 or 32
// x 32 each. K goes in steps of 32: quads of 4 consecutive k are read as fp32
// two steps ahead, split in registers and stored as three 8-byte pieces, one
// per plane, into the LDS stage the next step's products read (two stages, one
// barrier a step). The splitting, 6.5 vector instructions a value, is placed
// between the MFMAs, which run meanwhile. LDS planes are [rows][32] bf16 with
// the 16-byte chunks of a row at chunk ^ (row / 4 % 4): 16 rows of one chunk,
// the operand read, hit 16 distinct 16-byte bank groups. LayerNorm rows are
// normalised once into the workspace (k_layernorm_rows), or, without one, as
// they are split. Workgroups that share a weight tile are neighbours on one
// XCD, so its L2 serves all but the first of them. What bounds it: full tiles
// run the matrix cores at about 1.1 PFLOP/s of bf16 products (library bf16
// products reach 1.38 on this card); small calls, the chain of steps of one
// tile (0.5 us a step for 64 x 64).
#include <type_traits>

#include "split_bf16.h"

namespace skv {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kBK = 32;  // k per step
constexpr int kXCD = 8;  // XCDs of an MI355X

__device__ __forceinline__ float gelu_tanh_g(float v) {
  const float k0 = 0.7978845608028654f;  // sqrt(2 / pi)
  return 0.5f * v * (1.f + tanhf(k0 * (v + 0.044715f * v * v * v)));
}

struct GemmArgs {
  float* y;
  const float* x;
  const float* wt;
  const float* bias;
  const float* res;
  const float* ln_g;   // LayerNorm of the x rows (NULL: none)
  const float* ln_b;
  float ln_eps;
  int M, N, K;
  int act;    // 0 none, 1 GELU (tanh form)
  int split;  // > 0: column n goes to segment n / split of a [N/split][M][split] output
  int mt;     // row tiles (set at launch)
};

// Mean and 1/sqrt(var + eps) of a row of K values (population variance,
// jax_backend.py:78-82), by one wavefront: sums of the values shifted by the
// row's first element.
__device__ __forceinline__ float2 row_stats(const float* xr, int K, float eps, int lane) {
  const float c = xr[0];
  float s = 0.f, q = 0.f;
  for (int j = 4 * lane; j < K; j += 256) {  // K % 4 == 0
    const f32x4 v = *reinterpret_cast<const f32x4*>(xr + j);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float d = v[t] - c;
      s += d;
      q += d * d;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    s += __shfl_xor(s, o);
    q += __shfl_xor(q, o);
  }
  const float ms = s / K;
  return make_float2(c + ms, 1.f / sqrtf(fmaxf(q / K - ms * ms, 0.f) + eps));
}

// y = LayerNorm(x) of M rows, one wavefront per row (the second pass over a
// row reads it from the caches). Normalised once here, the rows cost the GEMM
// nothing; normalising them as each column tile splits them took 3 more
// vector instructions a value and the gamma and beta loads.
__global__ __launch_bounds__(256) void k_layernorm_rows(float* __restrict__ y,
                                                        const float* __restrict__ x,
                                                        const float* __restrict__ g,
                                                        const float* __restrict__ b, int M, int K,
                                                        float eps) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  const float* xr = x + (size_t)row * K;
  const float2 st = row_stats(xr, K, eps, lane);
  for (int j = 4 * lane; j < K; j += 256) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(xr + j);
    const f32x4 gj = *reinterpret_cast<const f32x4*>(g + j);
    const f32x4 bj = *reinterpret_cast<const f32x4*>(b + j);
    f32x4 o;
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] = (v[t] - st.x) * st.y * gj[t] + bj[t];
    *reinterpret_cast<f32x4*>(y + (size_t)row * K + j) = o;
  }
}

// 16-byte chunk `chunk` (8 k) of row `row` in an LDS plane (element offset).
__device__ __forceinline__ int plane_at(int row, int chunk) {
  return row * kBK + ((chunk ^ ((row >> 2) & 3)) * 8);
}

// 16 bytes at byte offset off of a buffer; zeros where off passes its end.
__device__ __forceinline__ f32x4 buf_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_of(const float* p, long floats) {
  // 32-bit sizes: callers pass at most a tile's rows
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)(uint32_t)(floats * 4),
                                           0x00020000 /* raw 32-bit data */);
}

// One workgroup: BM x BN outputs, (BM / WM) * (BN / WN) wavefronts of WM x
// WN. LN: LayerNorm of the x values as they are split (calls without the
// workspace for k_layernorm_rows). LONG: rows too long for 32-bit offsets into a
// tile, read through 64-bit addresses.
template <int BM, int BN, int WM, int WN, bool LN, bool LONG>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void k_gemm(GemmArgs a) {
  constexpr int NT = (BM / WM) * (BN / WN) * 64;
  constexpr int TI = WM / 32, TJ = WN / 32;          // 32 x 32 tiles of a wavefront
  constexpr int QA = BM * 8 / NT, QB = BN * 8 / NT;  // quads of x and of w per thread and step
  static_assert(QA * NT == BM * 8 && QB * NT == BN * 8, "staging shape");
  constexpr int PA = BM * kBK, PB = BN * kBK;  // elements of a plane
  // [stage][x planes h, m, l; w planes h, m, l]
  __shared__ __attribute__((aligned(16))) uint16_t lds[2 * 3 * (PA + PB)];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane & 31, hf = lane >> 5;
  const int wm = wave / (BN / WN), wn = wave % (BN / WN);
  const int xcd = blockIdx.x % kXCD, rest = blockIdx.x / kXCD;
  const int m0 = (rest % a.mt) * BM, n0 = ((rest / a.mt) * kXCD + xcd) * BN;
  if (n0 >= a.N) return;

  float mu[LN ? QA : 1], rs[LN ? QA : 1];
  if constexpr (LN) {
    // statistics of this tile's rows, one wavefront per row
    __shared__ float sstat[BM][2];
    for (int rr = wave; rr < BM; rr += NT / 64) {
      const float2 ms = row_stats(a.x + (size_t)min(m0 + rr, a.M - 1) * a.K, a.K, a.ln_eps, lane);
      if (lane == 0) {
        sstat[rr][0] = ms.x;
        sstat[rr][1] = ms.y;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < QA; ++u) {
      mu[u] = sstat[(tid + NT * u) >> 3][0];
      rs[u] = sstat[(tid + NT * u) >> 3][1];
    }
  }

  // Quad e = tid + NT u of a step is row e / 8, k 4 (e % 8) .. + 3 (a
  // wavefront's load covers 8 whole 128-byte rows), through buffer descriptors
  // over the tile's rows, so that rows past M or N and k past K read zeros and
  // no load sits behind a branch (K % 4 == 0: a quad lies wholly inside or
  // past K).
  const __amdgpu_buffer_rsrc_t bx =
      buf_of(a.x + (size_t)m0 * a.K, (long)min(BM, a.M - m0) * a.K);
  const __amdgpu_buffer_rsrc_t bw =
      buf_of(a.wt + (size_t)n0 * a.K, (long)min(BN, a.N - n0) * a.K);
  const __amdgpu_buffer_rsrc_t bg = buf_of(LN ? a.ln_g : a.x, LN ? a.K : 0);
  const __amdgpu_buffer_rsrc_t bb = buf_of(LN ? a.ln_b : a.x, LN ? a.K : 0);
  // (NT % 8 == 0: every quad of a thread has the same k)
  const int kq = 4 * (tid & 7);
  uint32_t offx[QA], offw[QB];
#pragma unroll
  for (int u = 0; u < QA; ++u) offx[u] = (uint32_t)((tid + NT * u) >> 3) * a.K * 4u;
#pragma unroll
  for (int u = 0; u < QB; ++u) offw[u] = (uint32_t)((tid + NT * u) >> 3) * a.K * 4u;
  struct Set {
    f32x4 q[QA + QB], g[1], b[1];
  } set[2];
  auto load_quad = [&](Set& r, int k0, int u) {  // quad u: of x, then of w
    const int kk = k0 + kq;
    if constexpr (LONG) {
      const int row = u < QA ? m0 + ((tid + NT * u) >> 3) : n0 + ((tid + NT * (u - QA)) >> 3);
      const bool in = kk < a.K && row < (u < QA ? a.M : a.N);
      const float* p = (u < QA ? a.x : a.wt) + (in ? (size_t)row * a.K + kk : 0);
      const f32x4 v = *reinterpret_cast<const f32x4*>(p);
      r.q[u] = in ? v : f32x4{0.f, 0.f, 0.f, 0.f};
      return;
    }
    const uint32_t past = kk < a.K ? 0u : 0xffffffffu;
    r.q[u] = u < QA ? buf_load(bx, (offx[u < QA ? u : 0] + kk * 4u) | past)
                    : buf_load(bw, (offw[u < QA ? 0 : u - QA] + kk * 4u) | past);
  };
  auto load_ln = [&](Set& r, int k0) {
    if constexpr (LN) {
      r.g[0] = buf_load(bg, (uint32_t)(k0 + kq) * 4u);
      r.b[0] = buf_load(bb, (uint32_t)(k0 + kq) * 4u);
    }
  };
  u32x2 ph, pm, pl;  // the parts of the quad being split
  // Pair i of a step: half i % 2 of quad i / 2; the second half stores the
  // quad and loads its successor.
  auto split_pair = [&](Set& r, int stage, int i, int k_next) {
    const int u = i >> 1, q = i & 1;
    float x = r.q[u][2 * q], y = r.q[u][2 * q + 1];
    if constexpr (LN) {
      if (u < QA) {
        const float mm = mu[u < QA ? u : 0], ss = rs[u < QA ? u : 0];
        x = (x - mm) * ss * r.g[0][2 * q] + r.b[0][2 * q];
        y = (y - mm) * ss * r.g[0][2 * q + 1] + r.b[0][2 * q + 1];
      }
    }
    uint32_t h, m, l;
    split2(x * kSplitScale, y * kSplitScale, h, m, l);
    ph[q] = h;
    pm[q] = m;
    pl[q] = l;
    if (q == 1) {
      const int e = tid + NT * (u < QA ? u : u - QA);
      uint16_t* p = lds + stage * 3 * (PA + PB) + (u < QA ? 0 : 3 * PA) +
                    plane_at(e >> 3, (e & 7) >> 1) + 4 * (e & 1);
      const int stride = u < QA ? PA : PB;
      *reinterpret_cast<u32x2*>(p) = ph;
      *reinterpret_cast<u32x2*>(p + stride) = pm;
      *reinterpret_cast<u32x2*>(p + 2 * stride) = pl;
      load_quad(r, k_next, u);
      if (u == QA - 1) load_ln(r, k_next);
    }
  };

  f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x16{};

  const int steps = (a.K + kBK - 1) / kBK;
  constexpr int NP = 2 * (QA + QB);  // pairs of a thread and step
  // step 0 goes to LDS at once; steps 1 and 2 wait in registers
#pragma unroll
  for (int f = 0; f < 2; ++f) {
#pragma unroll
    for (int u = 0; u < QA + QB; ++u) load_quad(set[f], f * kBK, u);
    load_ln(set[f], f * kBK);
    __builtin_amdgcn_sched_barrier(0);  // the sets' loads in the loop's order
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) split_pair(set[0], 0, i, 2 * kBK);
  __syncthreads();

  // Operands of one 16-k block: the two blocks of a step have a register set
  // each, so the second one's reads are issued before the products of the
  // first.
  struct Frag {
    bf16x8 x[TI][3], w[TJ][3];
  } fr[2];
  auto read_block = [&](int stage, int ks) {
    const uint16_t* base = lds + stage * 3 * (PA + PB);
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < TI; ++i)
        fr[ks].x[i][p] = *reinterpret_cast<const bf16x8*>(
            base + p * PA + plane_at(wm * WM + i * 32 + c, 2 * ks + hf));
#pragma unroll
      for (int j = 0; j < TJ; ++j)
        fr[ks].w[j][p] = *reinterpret_cast<const bf16x8*>(
            base + 3 * PA + p * PB + plane_at(wn * WN + j * 32 + c, 2 * ks + hf));
    }
  };

  // Step s (s % 2 == F): its products from LDS stage F, and between them the
  // split of step s + 1 into the other stage and the loads of step s + 3.
  auto step = [&](auto fc, int s) {
    constexpr int F = decltype(fc)::value, W = F ^ 1;
    constexpr int SLOTS = kBK / 16 * 6;
    read_block(F, 0);
#pragma unroll
    for (int ks = 0; ks < kBK / 16; ++ks) {
      if (ks == 0) read_block(F, 1);
      // the six partial products
#pragma unroll
      for (int t = 0; t < 6; ++t) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                fr[ks].x[i][kSplitA[t]], fr[ks].w[j][kSplitB[t]], acc[i][j], 0, 0, 0);
        const int slot = ks * 6 + t;
#pragma unroll
        for (int i = 0; i < NP; ++i)
          if (i * SLOTS / NP == slot) split_pair(set[W], W, i, (s + 3) * kBK);
      }
    }
    __syncthreads();  // stage F is read, stage W written
  };
  // steps in pairs without a branch between them (a step past K adds zeros)
  for (int s = 0; s < steps; s += 2) {
    step(std::integral_constant<int, 0>{}, s);
    step(std::integral_constant<int, 1>{}, s + 1);
  }

  // Output tile (i, j) of the wavefront with fp32 products, straight from
  // global memory: k 8 g + 4 hf + t in step (g, t).
  auto tile_f32 = [&](int i, int j) {
    const float* xr = a.x + (size_t)min(m0 + wm * WM + i * 32 + c, a.M - 1) * a.K;
    const float* wr = a.wt + (size_t)min(n0 + wn * WN + j * 32 + c, a.N - 1) * a.K;
    float mi = 0.f, ri = 0.f;
    if constexpr (LN) {  // one row per lane here, as row_stats
      float sm = 0.f, sq = 0.f;
      for (int k = 0; k < a.K; ++k) {
        const float v = xr[k] - xr[0];
        sm += v;
        sq += v * v;
      }
      const float ms = sm / a.K;
      mi = xr[0] + ms;
      ri = 1.f / sqrtf(fmaxf(sq / a.K - ms * ms, 0.f) + a.ln_eps);
    }
    f32x16 e = f32x16{};
    for (int k0 = 0; k0 < a.K; k0 += 8) {
      const bool in = k0 + 4 * hf < a.K;  // (K % 4 == 0)
      const int k = in ? k0 + 4 * hf : 0;
      f32x4 x = *reinterpret_cast<const f32x4*>(xr + k);
      f32x4 w = *reinterpret_cast<const f32x4*>(wr + k);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (LN) x[t] = (x[t] - mi) * ri * a.ln_g[k + t] + a.ln_b[k + t];
        e = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? x[t] : 0.f, in ? w[t] : 0.f, e, 0, 0, 0);
      }
    }
    return e;
  };
  // Outputs that are not finite (an infinity among the operands, a value too
  // large to scale, or a result that is none) take the value of the fp32
  // products; the others keep theirs, so a row's bits do not depend on the rows
  // and columns beside it.
  bool bad = false;
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) bad |= !finite(acc[i][j][r]);
  const bool redo = __ballot(bad) != 0ull;

  // acc[i][j][r]: row m0 + WM wm + 32 i + 8 (r/4) + 4 hf + r%4, column n0 + WN wn + 32 j + c
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int n = n0 + wn * WN + j * 32 + c;
    const float bv = a.bias && n < a.N ? a.bias[n] : 0.f;
    const int seg = a.split > 0 ? n / a.split : 0;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      f32x16 y;
#pragma unroll
      for (int r = 0; r < 16; ++r) y[r] = fmaf(acc[i][j][r], kSplitUnscale, bv);
      if (redo) {
        const f32x16 e = tile_f32(i, j);
#pragma unroll
        for (int r = 0; r < 16; ++r) y[r] = finite(acc[i][j][r]) ? y[r] : e[r] + bv;
      }
      if (n >= a.N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm * WM + i * 32 + 8 * (r >> 2) + 4 * hf + (r & 3);
        if (m >= a.M) continue;
        const size_t o = a.split > 0 ? ((size_t)seg * a.M + m) * a.split + (n - seg * a.split)
                                     : (size_t)m * a.N + n;
        float v = y[r];
        if (a.act == 1) v = gelu_tanh_g(v);
        if (a.res) v += a.res[o];
        a.y[o] = v;
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, bool LN = false, bool LONG = false>
int launch_gemm(GemmArgs a, hipStream_t s) {
  a.mt = (a.M + BM - 1) / BM;
  const long nt = ((a.N + BN - 1) / BN + kXCD - 1) / kXCD * kXCD;
  SKV_REQUIRE(nt * a.mt < (1L << 31), SKV_E_UNSUPPORTED, "skv_linear: M=%d too large", a.M);
  hipLaunchKernelGGL((k_gemm<BM, BN, WM, WN, LN, LONG>), dim3((unsigned)(nt * a.mt)),
                     dim3((BM / WM) * (BN / WN) * 64), 0, s, a);
  return check_launch("skv_linear");
}

}  // namespace

// skv_linear's path for calls of more than 64 rows (model_ops.hip). norm
// (may be NULL) holds M * K floats for the normalised rows of a LayerNorm
// call.
int gemm_linear(float* y, const float* x, const float* w_t, const float* bias,
                const float* residual, const float* ln_gamma, const float* ln_beta, float ln_eps,
                int M, int N, int K, int activation, int split_cols, float* norm,
                hipStream_t s) {
  GemmArgs a{y, x, w_t, bias, residual, ln_gamma, ln_beta, ln_eps, M, N, K, activation,
             split_cols, 0};
  const bool lng = (long)256 * K * 4 >= (1L << 32);  // 256 rows past a buffer's 32-bit range
  if (ln_gamma != nullptr) {
    if (norm == nullptr)
      return lng ? launch_gemm<64, 64, 32, 32, true, true>(a, s)
                 : launch_gemm<64, 64, 32, 32, true>(a, s);
    hipLaunchKernelGGL(k_layernorm_rows, dim3((M + 3) / 4), dim3(256), 0, s, norm, x, ln_gamma,
                       ln_beta, M, K, ln_eps);
    const int rc = check_launch("skv_linear");
    if (rc) return rc;
    a.x = norm;
    a.ln_g = a.ln_b = nullptr;
  }
  if (lng) return launch_gemm<64, 64, 32, 32, false, true>(a, s);
  // Tiles by how they fill the chip's 256 CUs (measured on MI355X, us, all of
  // them before the operands were scaled, which costs up to 6 %):
  //  - 256 x 128 where there are more than two rounds of them: the fewest
  //    values split per product (2048 x 50304 x 768: 853, 128 x 64 955, 64 x
  //    64 1128). With fewer, its long workgroups leave CUs idle (2048 x 2304 x
  //    768: 70 against 63; 2048 x 768 x 3072: 172 against 79).
  //  - 64 x 64 where 128 x 64 would not reach half the CUs (644 x 768 x 768:
  //    18.7 against 20.1; 111 x 640 x 2560: 48 against 53).
  //  - else 128 x 64 in 8 wavefronts of 32 x 32 (2048 x 768 x 768: 23.5,
  //    64 x 64 27.7, 256 x 128 53; 644 x 2304 x 768: 29, 64 x 64 34).
  const auto tiles = [&](long bm, long bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  if (tiles(256, 128) > 2 * 256) return launch_gemm<256, 128, 64, 64>(a, s);
  if (tiles(128, 64) < 128) return launch_gemm<64, 64, 32, 32>(a, s);
  return launch_gemm<128, 64, 32, 32>(a, s);
}

}  // namespace skv
