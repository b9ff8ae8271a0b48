// The fp32 flash forward and backward up to a head dim of 128 on the bf16
// matrix cores: every product as six partial products of operands split into three bf16
// parts (split_bf16.h), so results have fp32 accuracy.
//
// Reference: flash_attention (simple-llm/src/gpu/gpu_pass_forward.py:497-588,
// kernel create_flash_attention_kernel simple-llm/src/gpu/gpu_kernels.py:499-770),
// flash_attention_backward (gpu/gpu_pass_backward.py:445-580).
//
// What bounds these kernels: the matrix cores do a third of the fp32 MFMA
// kernels' cycles, and the vector instructions that split the operands (6.5 a
// value) and form the probabilities come to about as many; the forward at B=8,
// N=2048, H=16, D=64 is 56 % MFMA busy, at the 1.83 GHz that the card's power
// allows this mix (the fp32 form: 77 % at 2.4 GHz).
//
// Lane layout of v_mfma_f32_32x32x16_bf16 (lane l, c = l % 32, hf = l / 32):
//   A (32 x 16): A[c][8 hf + j]   B (16 x 32): B[8 hf + j][c], j < 8
//   C (32 x 32), register r: row 8 (r / 4) + 4 hf + r % 4, column c.
// A C tile is the operand of the next product as it stands: registers 8 kk ..
// 8 kk + 7 are the k-block kk of either half, the k order being the tile's
// rows 16 kk + 4 hf + (0..3, 8..11).
//
// The rows staged through LDS are split once per workgroup into three bf16
// planes [rows][DP] (DP: the head dim padded to a multiple of 32), whose
// 16-byte chunks sit at chunk ^ key(row), so that both reads hit distinct
// banks: the row operand (ds_read_b128, one chunk of 16 rows) and the
// transposed one (ds_read_b64_tr_b16, 4 chunks of 4 rows per 32 lanes).
#include <type_traits>

#include "flash_args.h"
#include "split_bf16.h"

namespace skv {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef flash_f32x4 f32x4;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kRows = 32 * kWaves;  // queries (or keys) of one workgroup

constexpr int pad32(int D) { return (D + 31) / 32 * 32; }

// Element offset of 16-byte chunk `chunk` of row `row` in a plane of DP-wide
// rows.
template <int DP>
__device__ __forceinline__ int swz(int row, int chunk) {
  int key;
  if constexpr (DP == 128) key = 4 * (row & 3) + ((row >> 2) & 3);
  else if constexpr (DP == 64) key = 4 * ((row >> 1) & 1) + ((row >> 2) & 3);
  else key = (row >> 2) & 3;  // 32 and 96: the low two bits of the chunk
  return row * DP + ((chunk ^ key) * 8);
}

__device__ __forceinline__ i16x4 lds_read_tr16(const uint16_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(p));
}

// R rows x D of one tensor: global -> registers (fp32) -> three LDS planes, a
// quad (4 elements of a row) at a time. Rows at or beyond n_rows repeat row
// n_rows - 1 (every product that involves them is masked by a select).
template <int D, int MODE, int R>
struct SplitStage {
  static constexpr int DP = pad32(D), PS = R * DP;  // plane size (elements)
  static constexpr int C4 = D / 4, NQ = R * C4;      // quads of a row, of the tile
  static constexpr int NV = (NQ + kThreads - 1) / kThreads;
  f32x4 r[NV];

  __device__ __forceinline__ static int quad(int u) {  // threads past NQ repeat the last quad
    const int e = threadIdx.x + kThreads * u;
    return NQ % kThreads == 0 ? e : min(e, NQ - 1);
  }
  __device__ __forceinline__ void load(int u, const float* t, int row0, int n_rows,
                                       uint32_t rs, int Dr) {
    const int e = quad(u);
    const int n = min(row0 + e / C4, n_rows - 1);
    r[u] = load4m<MODE>(t + (uint64_t)(uint32_t)n * rs, 4 * (e % C4), Dr);
  }
  __device__ __forceinline__ void store(int u, uint16_t* planes, float scale) const {
    const int e = quad(u), row = e / C4, q = e % C4;
    u32x2 h, m, l;
    uint32_t a, b, c;
    const f32x4 x = r[u] * scale;
    split2(x.x, x.y, a, b, c);
    h.x = a; m.x = b; l.x = c;
    split2(x.z, x.w, a, b, c);
    h.y = a; m.y = b; l.y = c;
    uint16_t* p = planes + swz<DP>(row, q >> 1) + 4 * (q & 1);
    *reinterpret_cast<u32x2*>(p) = h;
    *reinterpret_cast<u32x2*>(p + PS) = m;
    *reinterpret_cast<u32x2*>(p + 2 * PS) = l;
  }
};

// Row operand: row `row`, elements 16 kb + 8 hf .. + 7 of every plane.
template <int DP, int PS>
__device__ __forceinline__ void read_rows(const uint16_t* planes, int row, int kb, int hf,
                                          bf16x8 (&f)[3]) {
#pragma unroll
  for (int p = 0; p < 3; ++p)
    f[p] = *reinterpret_cast<const bf16x8*>(planes + p * PS + swz<DP>(row, 2 * kb + hf));
}

// Transposed operand: column db * 32 + c of rows r0 + 4 hf + (0..3, 8..11) of
// every plane. (ds_read_b64_tr_b16 gives lane i of a 16-lane group element
// i % 4 of the four 16-bit values addressed by lane 4 j + i / 4, as its slot j.)
template <int DP, int PS>
__device__ __forceinline__ void read_cols(const uint16_t* planes, int r0, int db, int lane,
                                          bf16x8 (&f)[3]) {
  const int g = lane >> 5, gr = lane >> 4, L = lane & 15;
  const int d = db * 32 + (gr & 1) * 16 + 4 * (L & 3);
  const int ra = r0 + 4 * g + (L >> 2);
  const int oa = swz<DP>(ra, d >> 3) + (d & 7), ob = swz<DP>(ra + 8, d >> 3) + (d & 7);
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    const i16x4 lo = lds_read_tr16(planes + p * PS + oa);
    const i16x4 hi = lds_read_tr16(planes + p * PS + ob);
    f[p] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
}

// 8 consecutive scaled values of a row, split.
__device__ __forceinline__ void split8(const f32x4& x, const f32x4& y, bf16x8 (&f)[3]) {
  u32x4 w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t h, m, l;
    if (i < 2) split2(x[2 * i], x[2 * i + 1], h, m, l);
    else split2(y[2 * i - 4], y[2 * i - 3], h, m, l);
    w[0][i] = h; w[1][i] = m; w[2][i] = l;
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) f[p] = __builtin_bit_cast(bf16x8, w[p]);
}

// k-block kk of a (scaled) C tile as an operand.
__device__ __forceinline__ void split_tile(const f32x16& t, int kk, bf16x8 (&f)[3]) {
  split8(f32x4{t[8 * kk], t[8 * kk + 1], t[8 * kk + 2], t[8 * kk + 3]},
         f32x4{t[8 * kk + 4], t[8 * kk + 5], t[8 * kk + 6], t[8 * kk + 7]}, f);
}

// The elements of DT tiles that are not finite, bit 16 dt + r.
template <int DT>
__device__ __forceinline__ uint64_t non_finite(const f32x16 (&t)[DT]) {
  uint64_t set = 0;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) set |= (uint64_t)(finite(t[dt][r]) ? 0 : 1) << (16 * dt + r);
  return set;
}

// Unrolling of the loops that take non-finite sums from fp32 products: they run
// rarely and must not cost the kernels registers.
template <int MODE>
constexpr int kAgain = MODE == 2 ? 1 : 2;

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// Forward. One workgroup per (128 queries, b, query head), rank-major: all (b,
// h) of one block rank before the next, ranks in order of decreasing causal
// work (the dispatcher's round robin then gives every XCD the same load). Each
// wave owns 32 queries (lane c, both halves): per 32-key piece S^T = K Q^T, an
// online softmax over the piece, then O^T += V^T P^T. The running max moves
// only when a piece's max exceeds it by more than 8 (log2 units), so O and l
// are rescaled on few pieces; the true maximum is kept beside it for M and the
// final L.
// K and V go through LDS 32 keys at a time in two stages: while the scores of
// a piece are multiplied, the next piece is split into the other stage and the
// one after it loaded into registers, and the second half of P is split while
// the first is multiplied, so most vector instructions run between MFMAs.
// Measured on MI355X against the fp32 MFMA form (B, N, H, D; us): 8, 2048, 16,
// 64: 570 -> 403; 2, 1024, 12, 64: 78 -> 51; 2, 2048, 16, 128: 330 -> 222; 5,
// 1605, 8, 96: 254 -> 139; 4, 333, 8, 48: 30.5 -> 19.9. Relative 2-norm error
// against float64 at N = 150, D = 64: 2.2e-7 -> 1.5e-7. With 64 keys a step in
// one LDS stage: 399 for the first, against 388 at the time; with 8 wavefronts
// a workgroup 374, but 66 for the second and 145 for the fourth.
// ---------------------------------------------------------------------------
constexpr float kQueryScale = 0x1p40f, kScoreUnscale = 0x1p-64f;
template <int D, int MODE>
__global__ __launch_bounds__(kThreads, D <= 96 ? 2 : 1) void k_flash_fwd_split(FfwdArgs a) {
  constexpr int KB = D / 16;             // k-blocks of Q K^T
  constexpr int DT = (D + 31) / 32;      // 32-row tiles of O^T
  typedef SplitStage<D, MODE, 32> St;
  constexpr int DP = St::DP, PS = St::PS;
  const int RS = MODE == 0 ? D : a.D;  // the real head dim
  __shared__ __attribute__((aligned(16))) uint16_t lds[2][6 * PS];  // [stage][K, V planes]

  const int Hq = a.Hq, C = a.C;
  const int bh = (int)(blockIdx.x % (unsigned)a.BH), rank = (int)(blockIdx.x / (unsigned)a.BH);
  const int b = bh / Hq, h = bh % Hq, hk = h / (Hq / a.Hkv);
  const int blk = a.n_blocks - 1 - rank;
  const int P = a.start ? min(max(a.start[b], 0), a.T_cap) : 0;
  const int n = max(0, min(a.n_new ? min(a.n_new[b], C) : C, a.T_cap - P));  // valid queries
  const int kv_end = P + n;  // keys [0, kv_end) exist
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 31, hf = lane >> 5;
  const int qi = blk * kRows + wave * 32 + c;  // this lane's query (row of the chunk)
  const bool qok = qi < n;
  const int qlim = qok ? P + qi : -1;          // keys <= qlim are unmasked
  const float* const qp = a.q + (((size_t)b * C + min(qi, max(n, 1) - 1)) * Hq + h) * RS;

  // keys this workgroup and this wave need
  const int blk_q = min(blk * kRows + kRows, n);  // valid queries of the block end here
  const int steps = blk * kRows < n ? (P + blk_q + 31) / 32 : 0;
  const int wq0 = blk * kRows + wave * 32;  // the wave's first query
  const bool wfull = wq0 + 31 < n;           // all 32 of its queries valid
  const int wq_last = wq0 < n ? P + min(wq0 + 31, n - 1) : -1;
  const uint32_t rs = (uint32_t)(a.Hkv * RS);
  const float* kh = a.k + ((size_t)b * a.T_cap * a.Hkv + hk) * RS;
  const float* vh = a.v + ((size_t)b * a.T_cap * a.Hkv + hk) * RS;

  // O^T, and (where the registers allow) its small partial products apart
  constexpr bool LO = D <= 64 || D > 96;
  f32x16 acc[DT], acl[LO ? DT : 1];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = acl[LO ? dt : 0] = f32x16{};
  float m_run = -INFINITY, m_true = -INFINITY, l = 0.f;

  // The online softmax of the piece at key0: s holds its scores in log2 units
  // (key key0 + 8 (r / 4) + 4 hf + r % 4 of this lane's query) times 2^64, and
  // gets the probabilities times 2^24.
  auto softmax = [&](f32x16& s, int key0) {
    // A piece wholly at or below the diagonal of a wave whose 32 queries are
    // all valid masks nothing (wave-uniform test).
    float tmax = -INFINITY;
    if (!(wfull && key0 + 31 <= P + wq0)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = key0 + 8 * (r / 4) + 4 * hf + (r % 4);
        s[r] = key <= qlim ? s[r] : -INFINITY;
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[r]);
    tmax = xor32_max(tmax) * kScoreUnscale;  // both halves hold the same query
    m_true = fmaxf(m_true, tmax);
    const bool upd = tmax > m_run + 8.f;  // also true on the first piece with a key
    if (__ballot(upd) != 0ull) {          // wave-uniform branch
      const float alpha = upd ? fast_exp2(m_run - tmax) : 1.f;  // m_run = -inf: 0
      if (upd) m_run = tmax;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        acc[dt] *= alpha;
        if (LO) acl[LO ? dt : 0] *= alpha;
      }
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;  // nothing unmasked yet
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(fmaf(s[r], kScoreUnscale, -m_use));
      l += s[r];
      s[r] *= kSplitScale;
    }
  };

  // the query, so that the scores come out in log2 units: rounded, so its
  // smallest values have more bits to keep than an operand's own
  bf16x8 qf[KB][3];
  const float qs = a.sl2 * kQueryScale;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
    split8(load4m<MODE>(qp, 16 * kb + 8 * hf, RS) * qs,
           load4m<MODE>(qp, 16 * kb + 8 * hf + 4, RS) * qs, qf[kb]);
  St st[2];  // K, V: the piece after the one in LDS
  constexpr int NV = St::NV;
  auto load_quad = [&](int i, int key0) {  // quad i of a piece: of K, then of V
    st[i / NV].load(i % NV, i < NV ? kh : vh, key0, kv_end, rs, RS);
  };
  if (steps > 0) {
#pragma unroll
    for (int i = 0; i < 2 * NV; ++i) load_quad(i, 0);
#pragma unroll
    for (int i = 0; i < 2 * NV; ++i) {
      st[i / NV].store(i % NV, lds[0] + (i / NV) * 3 * PS, kSplitScale);
      load_quad(i, 32);
    }
  }
  __syncthreads();
  // Piece j (j % 2 == F) from stage F.
  auto step = [&](auto fc, int j) {
    constexpr int F = decltype(fc)::value;
    const uint16_t* const sK = lds[F];
    const uint16_t* const sV = lds[F] + 3 * PS;
    const int key0 = j * 32;
    auto stage_quad = [&](int i) {  // of piece j + 1; its register then takes piece j + 2
      st[i / NV].store(i % NV, lds[F ^ 1] + (i / NV) * 3 * PS, kSplitScale);
      load_quad(i, key0 + 64);
    };
    if (key0 <= wq_last) {  // wave-uniform: else every key is masked for this wave
      f32x16 s = f32x16{};
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        bf16x8 ka[3];
        read_rows<DP, PS>(sK, c, kb, hf, ka);
        s = mfma_split(ka, qf[kb], s);
#pragma unroll
        for (int i = 0; i < 2 * NV; ++i)
          if (i * KB / (2 * NV) == kb) stage_quad(i);
      }
      softmax(s, key0);
      // O^T[d][query] += sum_key V[key][d] P^T[key][query]
      bf16x8 pf[2][3];
      split_tile(s, 0, pf[0]);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          bf16x8 va[3];
          read_cols<DP, PS>(sV, 16 * kk, dt, lane, va);
          if constexpr (LO) mfma_split(va, pf[kk], acc[dt], acl[dt]);
          else acc[dt] = mfma_split(va, pf[kk], acc[dt]);
          if (kk == 0 && dt == 0) split_tile(s, 1, pf[1]);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2 * NV; ++i) stage_quad(i);
    }
    __syncthreads();  // stage F is read, the other one written
  };
  for (int j = 0; j < steps; j += 2) {
    step(std::integral_constant<int, 0>{}, j);
    if (j + 1 < steps) step(std::integral_constant<int, 1>{}, j + 1);
  }
  float lt = xor32_sum(l);
  if constexpr (LO)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] += acl[dt];

  // Sums that are not all finite (an infinity, a NaN or a value too large to
  // scale among the operands), or a query whose scores all came out as -inf:
  // taken below from fp32 products.
  const bool row_bad = qok && !(lt > 0.f && finite(lt));
  bool bad = row_bad;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      bad |= qok && dt * 32 + 8 * (r / 4) + 4 * hf + (r % 4) < RS && !finite(acc[dt][r]);
  const bool again = __ballot(bad) != 0ull;
  // (out may be q: the queries wait in LDS, each lane's own quads)
  f32x4* const ql = reinterpret_cast<f32x4*>(lds) + (wave * 32 + c) * (D / 4);
  if (again)
    for (int g = hf; g < D / 4; g += 2) ql[g] = load4m<MODE>(qp, 4 * g, RS);

  const size_t orow = ((size_t)b * C + qi) * Hq + h;
  if (qi < C) {
    const float inv = qok ? 1.f / lt * kSplitUnscale : 0.f;  // a valid row saw its own key: lt >= 1
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int qq = 0; qq < 4; ++qq) {
        const int d0 = dt * 32 + 8 * qq + 4 * hf;
        f32x4 y = {acc[dt][4 * qq] * inv, acc[dt][4 * qq + 1] * inv, acc[dt][4 * qq + 2] * inv,
                   acc[dt][4 * qq + 3] * inv};
        if (!qok) y = f32x4{0.f, 0.f, 0.f, 0.f};
        store4m<MODE>(a.out + orow * RS, d0, RS, y);
      }
    }
    if (hf == 0 && qok) {
      if (a.L) a.L[orow] = lt * fast_exp2(m_run - m_true);  // relative to the true maximum
      if (a.M) a.M[orow] = m_true * (1.f / LOG2E);          // natural units, as the scores
    }
  }
  if (!again) return;

  // The elements that are not finite, and no others (a row's bits do not depend
  // on the rows beside it), from fp32 products straight from global memory.
  const uint64_t redo = !qok ? 0ull : row_bad ? ~0ull : non_finite(acc);
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{};
  float m = -INFINITY, lsum = 0.f;
#pragma unroll 1
  for (int key0 = 0; key0 <= wq_last; key0 += 32) {
    f32x16 s = f32x16{};
    const float* kr = kh + (size_t)min(key0 + c, kv_end - 1) * rs;
#pragma unroll kAgain<MODE>
    for (int g = 0; g < D / 8; ++g) {
      const f32x4 ka = load4m<MODE>(kr, 8 * g + 4 * hf, RS);
      const f32x4 qa = ql[2 * g + hf];
#pragma unroll
      for (int t = 0; t < 4; ++t) s = mfma_f32(ka[t], qa[t], s);
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = key0 + 8 * (r / 4) + 4 * hf + (r % 4) <= qlim ? s[r] * a.sl2 : -INFINITY;
      tmax = fmaxf(tmax, s[r]);
    }
    const float mn = fmaxf(m, xor32_max(tmax)), m_use = mn == -INFINITY ? 0.f : mn;
    const float alpha = fast_exp2(m - m_use);  // m = -inf: 0
    m = mn;
    lsum *= alpha;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r] - m_use);
      lsum += s[r];
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int d = dt * 32 + c;
      o[dt] *= alpha;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = min(key0 + 8 * (r / 4) + 4 * hf + (r % 4), kv_end - 1);
        const float vv = vh[(size_t)key * rs + (d < RS ? d : 0)];
        o[dt] = mfma_f32(d < RS ? vv : 0.f, s[r], o[dt]);
      }
    }
  }
  lsum = xor32_sum(lsum);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int d = dt * 32 + 8 * (r / 4) + 4 * hf + (r % 4);
      if (d < RS && ((redo >> (16 * dt + r)) & 1) != 0) a.out[orow * RS + d] = o[dt][r] / lsum;
    }
  if (row_bad && hf == 0) {
    if (a.L) a.L[orow] = lsum;
    if (a.M) a.M[orow] = m * (1.f / LOG2E);
  }
}

// ---------------------------------------------------------------------------
// Backward. Reference: simple-llm/src/gpu/gpu_kernels.py:2038-2455. Per (batch
// b, head h), with S = scale * Q K^T, masked to key <= query:
//   P  = exp(S - M) / L,  dP = dO V^T,  dS = P * (dP - Dl)
//   dQ = scale * dS K,  dK = scale * dS^T Q,  dV = P^T dO
// No atomics and every sum in a fixed order. dK and dV: one workgroup per (128
// keys, b, h), each wave 32 keys, their K in registers and V beside it in LDS
// (each lane's own operands); Q and dO go through LDS 32 rows at a time. dQ
// either repeats S and dP per (128 queries, b, h), or is formed from the dS
// that the dK/dV kernel wrote (the same bits: the partial products are taken
// in the same order).
// Measured on MI355X against the fp32 MFMA forms (B, N, H, D; us): 8, 2048, 16,
// 64: 1520 -> 1125; 2, 1024, 12, 64: 203 -> 140; 2, 2048, 16, 128: 1055 -> 709;
// 5, 1605, 8, 96: 707 -> 483; 4, 333, 8, 48: 81 -> 51. The largest relative
// 2-norm error against float64 of dQ, dK and dV at the first: 1.1e-6 -> 8.3e-7.
// Before P and dS were formed under the products, and with dQ's K 32 rows a
// step: 1160, 164 and 60 for the first, second and last, against 1110, 138 and 51.
// ---------------------------------------------------------------------------

// What the chain of products carries: 2^48 for S and dP, 2^16 for P (its
// smallest normal value keeps every bit), so 2^40 for dV, 2^64 for dS and 2^88
// for dK and dQ formed from it. Sums past the largest float, gradients from
// 2^40, take the fp32 form.
constexpr float kProdScale = kSplitScale * kSplitScale;
constexpr float kPScale = 0x1p16f, kDvUnscale = 0x1p-40f;
constexpr float kDsUnscale = 0x1p-64f, kGradUnscale = 0x1p-88f;

// c += A B as mfma_split(b, a, c) orders the partial products of its factors.
__device__ __forceinline__ f32x16 mfma_split_swapped(const bf16x8 (&a)[3], const bf16x8 (&b)[3],
                                                     f32x16 c) {
#pragma unroll
  for (int t = 0; t < 6; ++t)
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kSplitB[t]], b[kSplitA[t]], c, 0, 0, 0);
  return c;
}

// Element offset of row n of head h in batch b of a [B, N, H, D] tensor.
__device__ __forceinline__ size_t row_off(int b, int n, int N, int H, int h, int D) {
  return ((size_t)(b * N + n) * H + h) * D;
}

// dS of the five-product backward in 32 x 32 tiles: tile (query block qb, key
// block kb) of (b, h) holds 32 rows of 32 floats, row = query qb*32 + i, and
// within a row key kb*32 + 8 qq + 4 hf + t at position 16 hf + 4 qq + t: the
// order in which lane (query i, half hf) of k_fbwd_dq_ds_split takes the keys
// of a product, so that lane reads 64 contiguous bytes and a wavefront a whole
// 4 KB tile.
__device__ __forceinline__ float* ds_tile(const FbwdArgs& a, int bh, int qb, int kb) {
  const int nt = (a.N + 31) >> 5;
  return a.ds + (((size_t)bh * nt + qb) * nt + kb) * 1024;
}
__device__ __forceinline__ int ds_key_pos(int c) {  // key c of a block: 8 qq + 4 hf + t
  return 16 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3);
}

// dK and dV; rank 0 = key block 0 (the most queries). DSO: also write dS
// (a.ds).
template <int D, int MODE, bool DSO>
__global__ __launch_bounds__(kThreads, D <= 64 ? 2 : 1) void k_fbwd_dkv_split(FbwdArgs a) {
  constexpr int KB = D / 16, DT = (D + 31) / 32;
  typedef SplitStage<D, MODE, 32> St;
  constexpr int DP = St::DP, PS = St::PS, NV = St::NV;
  const int RS = MODE == 0 ? D : a.D;  // the real head dim
  struct alignas(16) Smem {
    uint16_t q[3 * PS], d[3 * PS];          // Q and dO of a piece
    bf16x8 v[kWaves][KB][3][64];             // each lane's V operands
    float m2[32], il[32], dl[32];            // the piece's row statistics
  };
  __shared__ Smem sm;

  const int H = a.H, N = a.N;
  const int bh = (int)(blockIdx.x % (unsigned)a.BH), rank = (int)(blockIdx.x / (unsigned)a.BH);
  const int b = bh / H, h = bh % H;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 31, hf = lane >> 5;
  const int wk0 = rank * kRows + wave * 32;  // the wave's first key
  const int krow = wk0 + c;  // a key past N is masked for every query (query < N <= krow)
  const size_t koff = row_off(b, min(krow, N - 1), N, H, h, RS);
  const uint32_t rs = (uint32_t)(H * RS);
  const float* qh = a.q + row_off(b, 0, N, H, h, RS);
  const float* dh = a.dout + row_off(b, 0, N, H, h, RS);

  bf16x8 kf[KB][3];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int d0 = 16 * kb + 8 * hf;
    split8(load4m<MODE>(a.k + koff, d0, RS) * kSplitScale,
           load4m<MODE>(a.k + koff, d0 + 4, RS) * kSplitScale, kf[kb]);
    bf16x8 vf[3];
    split8(load4m<MODE>(a.v + koff, d0, RS) * kSplitScale,
           load4m<MODE>(a.v + koff, d0 + 4, RS) * kSplitScale, vf);
#pragma unroll
    for (int p = 0; p < 3; ++p) sm.v[wave][kb][p][lane] = vf[p];
  }
  f32x16 dva[DT], dka[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dva[dt] = dka[dt] = f32x16{};
  // DSO: this lane's place in the dS tiles of its key block (query block 0;
  // the query block adds a whole row of tiles): key c, rows 4 hf + ...
  float* dsw = nullptr;
  if constexpr (DSO) dsw = ds_tile(a, bh, 0, wk0 >> 5) + ds_key_pos(c) + 128 * hf;
  auto store_ds = [&](auto interior, const f32x16& ds, int q0) {
    // for each slot the 32 lanes of a half write one query's 128-byte tile
    // row, past the caches (read once, later)
    if (decltype(interior)::value || krow < N) {
      float* tp = dsw + (size_t)(q0 >> 5) * ((N + 31) >> 5) * 1024;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (decltype(interior)::value || q0 + 8 * (r / 4) + 4 * hf + (r % 4) < N)
          __builtin_nontemporal_store(ds[r] * kDsUnscale, tp + (8 * (r / 4) + (r % 4)) * 32);
    }
  };

  const int pieces = (N + 31) / 32;
  const int j0 = rank * (kRows / 32);  // first piece holding a query >= the block's first key
  St st[2];  // Q, dO
  float m2 = 0.f, il = 0.f, dl = 0.f;
  auto load_piece = [&](int j) {
#pragma unroll
    for (int i = 0; i < 2 * NV; ++i)
      st[i / NV].load(i % NV, i < NV ? qh : dh, j * 32, N, rs, RS);
    if (threadIdx.x < 32) {  // statistics of query j * 32 + threadIdx.x, clamped
      const size_t sr = (size_t)(b * N + min(j * 32 + (int)threadIdx.x, N - 1)) * H + h;
      m2 = a.M[sr] * LOG2E;
      il = 1.f / a.L[sr] * kPScale;
      dl = a.delta[sr] * kProdScale;
    }
  };
  const float sl2 = a.sl2 * kSplitUnscale;
  // One piece. s[r], dp[r]: query q0 + 8(r/4) + 4hf + r%4, key krow. The
  // vector work stands between products that do not wait for it: P is formed
  // and split under dP = dO V^T, dS under dV += P^T dO.
  auto piece = [&](auto interior, int q0) {
    f32x16 s = f32x16{}, dp = f32x16{};
    bf16x8 pf[2][3], df[2][3];
    auto form_p = [&](int half) {
#pragma unroll
      for (int qq = 2 * half; qq < 2 * half + 2; ++qq) {
        const f32x4 m4 = *reinterpret_cast<const f32x4*>(sm.m2 + 8 * qq + 4 * hf);
        const f32x4 i4 = *reinterpret_cast<const f32x4*>(sm.il + 8 * qq + 4 * hf);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int r = 4 * qq + t, query = q0 + 8 * qq + 4 * hf + t;
          const float e = fast_exp2(fmaf(s[r], sl2, -m4[t])) * i4[t];
          s[r] = decltype(interior)::value || (krow <= query && query < N) ? e : 0.f;
        }
      }
    };
    auto form_ds = [&](int half) {
#pragma unroll
      for (int qq = 2 * half; qq < 2 * half + 2; ++qq) {
        const f32x4 d4 = *reinterpret_cast<const f32x4*>(sm.dl + 8 * qq + 4 * hf);
#pragma unroll
        for (int t = 0; t < 4; ++t) dp[4 * qq + t] = (dp[4 * qq + t] - d4[t]) * s[4 * qq + t];
      }
    };
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      bf16x8 qa[3];
      read_rows<DP, PS>(sm.q, c, kb, hf, qa);
      s = mfma_split(qa, kf[kb], s);
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      bf16x8 da[3], vf[3];
      read_rows<DP, PS>(sm.d, c, kb, hf, da);
#pragma unroll
      for (int p = 0; p < 3; ++p) vf[p] = sm.v[wave][kb][p][lane];
      dp = mfma_split(da, vf, dp);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i * KB / 4 == kb) {
          if (i < 2) form_p(i);
          else split_tile(s, i - 2, pf[i - 2]);
        }
    }
    // dV[key][d] += sum_query P^T[key][query] dO[query][d]; dK likewise with dS and Q
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        bf16x8 x[3];
        read_cols<DP, PS>(sm.d, 16 * kk, dt, lane, x);
        dva[dt] = mfma_split(pf[kk], x, dva[dt]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (i * 2 * DT / 4 == kk * DT + dt) {
            if (i < 2) form_ds(i);
            else split_tile(dp, i - 2, df[i - 2]);
          }
      }
    if constexpr (DSO) store_ds(interior, dp, q0);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        bf16x8 x[3];
        read_cols<DP, PS>(sm.q, 16 * kk, dt, lane, x);
        dka[dt] = mfma_split(df[kk], x, dka[dt]);
      }
  };
  if (j0 < pieces) load_piece(j0);
  for (int j = j0; j < pieces; ++j) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2 * NV; ++i) st[i / NV].store(i % NV, i < NV ? sm.q : sm.d, kSplitScale);
    if (threadIdx.x < 32) {
      sm.m2[threadIdx.x] = m2;
      sm.il[threadIdx.x] = il;
      sm.dl[threadIdx.x] = dl;
    }
    __syncthreads();
    if (j + 1 < pieces) load_piece(j + 1);
    const int q0 = j * 32;
    // wave-uniform: every query precedes the wave's keys, or the wave has no key
    if (q0 + 31 < wk0 || wk0 >= N) continue;
    // wave-uniform: every key of the wave precedes every query of the piece
    // and every query exists, so no slot is masked
    if (q0 >= wk0 + 31 && q0 + 32 <= N) piece(std::true_type{}, q0);
    else piece(std::false_type{}, q0);
  }

  // dva[dt][r], dka[dt][r]: key wk0 + 8(r/4) + 4hf + r%4, d = dt*32 + c
  bool bad = false;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const int d = dt * 32 + c;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = wk0 + 8 * (r / 4) + 4 * hf + (r % 4);
      if (key < N && d < RS) {
        const size_t off = row_off(b, key, N, H, h, RS) + d;
        a.dk[off] = dka[dt][r] * kGradUnscale * a.scale;
        a.dv[off] = dva[dt][r] * kDvUnscale;
        bad |= !(finite(dva[dt][r]) && finite(dka[dt][r]));
      }
    }
  }
  // Sums that are not all finite: those elements of the wave's keys (and of
  // dS), and no others, from fp32 products, straight from global memory.
  if (__ballot(bad) != 0ull) {
    const uint64_t redo_v = non_finite(dva), redo_k = non_finite(dka);
    f32x16 ev[DT], ek[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) ev[dt] = ek[dt] = f32x16{};
#pragma unroll 1
    for (int q0 = wk0; q0 < N; q0 += 32) {
      f32x16 s = f32x16{}, dp = f32x16{};
      const size_t qo = (size_t)min(q0 + c, N - 1) * rs;
#pragma unroll kAgain<MODE>
      for (int g = 0; g < D / 8; ++g) {
        const int d0 = 8 * g + 4 * hf;
        const f32x4 qa = load4m<MODE>(qh + qo, d0, RS), da = load4m<MODE>(dh + qo, d0, RS);
        const f32x4 ka = load4m<MODE>(a.k + koff, d0, RS), va = load4m<MODE>(a.v + koff, d0, RS);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          s = mfma_f32(qa[t], ka[t], s);
          dp = mfma_f32(da[t], va[t], dp);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int query = q0 + 8 * (r / 4) + 4 * hf + (r % 4);
        const size_t sr = (size_t)(b * N + min(query, N - 1)) * H + h;
        const float e = fast_exp2(fmaf(s[r], a.sl2, -(a.M[sr] * LOG2E))) * (1.f / a.L[sr]);
        s[r] = (krow <= query && query < N) ? e : 0.f;
        dp[r] = s[r] * (dp[r] - a.delta[sr]);
      }
      if (DSO && krow < N) {  // dS where it is not finite
        float* tp = dsw + (size_t)(q0 >> 5) * ((N + 31) >> 5) * 1024;
        uint32_t bad_ds = 0;
#pragma unroll
        for (int r = 0; r < 16; ++r)  // (a query past N: this tile's own memory, not used)
          bad_ds |= (uint32_t)(finite(tp[(8 * (r / 4) + (r % 4)) * 32]) ? 0 : 1) << r;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (((bad_ds >> r) & 1) != 0 && q0 + 8 * (r / 4) + 4 * hf + (r % 4) < N)
            tp[(8 * (r / 4) + (r % 4)) * 32] = dp[r];
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int d = dt * 32 + c;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const size_t o = (size_t)min(q0 + 8 * (r / 4) + 4 * hf + (r % 4), N - 1) * rs +
                           (d < RS ? d : 0);
          const float xo = dh[o], xq = qh[o];
          ev[dt] = mfma_f32(s[r], d < RS ? xo : 0.f, ev[dt]);
          ek[dt] = mfma_f32(dp[r], d < RS ? xq : 0.f, ek[dt]);
        }
      }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int d = dt * 32 + c;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = wk0 + 8 * (r / 4) + 4 * hf + (r % 4);
        if (key < N && d < RS) {
          const size_t off = row_off(b, key, N, H, h, RS) + d;
          if ((redo_k >> (16 * dt + r)) & 1) a.dk[off] = ek[dt][r] * a.scale;
          if ((redo_v >> (16 * dt + r)) & 1) a.dv[off] = ev[dt][r];
        }
      }
    }
  }
}

// dQ^T of 32 queries (lane c) to its rows.
template <int DT, int MODE>
__device__ __forceinline__ void store_dq(const FbwdArgs& a, const f32x16 (&acc)[DT], float unit,
                                         size_t qoff, int hf, int RS) {
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
      const f32x4 y = {acc[dt][4 * qq] * unit * a.scale, acc[dt][4 * qq + 1] * unit * a.scale,
                       acc[dt][4 * qq + 2] * unit * a.scale,
                       acc[dt][4 * qq + 3] * unit * a.scale};
      store4m<MODE>(a.dq + qoff, dt * 32 + 8 * qq + 4 * hf, RS, y);
    }
}

// dQ of a wave's queries, and where it is not finite, those elements and no
// others from fp32 products: form(key0) gives dS of the piece at key0.
template <int DT, int MODE, typename F>
__device__ __forceinline__ void finish_dq(const FbwdArgs& a, const f32x16 (&acc)[DT], float unit,
                                          size_t qoff, bool qok, int wq_last, const float* kh,
                                          uint32_t rs, int RS, int c, int hf, F form) {
  bool bad = false;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      bad |= qok && dt * 32 + 8 * (r / 4) + 4 * hf + (r % 4) < RS && !finite(acc[dt][r]);
  if (qok) store_dq<DT, MODE>(a, acc, unit, qoff, hf, RS);
  if (__ballot(bad) == 0ull) return;
  const uint64_t redo = qok ? non_finite(acc) : 0ull;
  f32x16 e[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) e[dt] = f32x16{};
#pragma unroll 1
  for (int key0 = 0; key0 <= wq_last; key0 += 32) {
    const f32x16 ds = form(key0);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int d = dt * 32 + c;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = min(key0 + 8 * (r / 4) + 4 * hf + (r % 4), a.N - 1);
        const float kv = kh[(size_t)key * rs + (d < RS ? d : 0)];
        e[dt] = mfma_f32(d < RS ? kv : 0.f, ds[r], e[dt]);
      }
    }
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int d = dt * 32 + 8 * (r / 4) + 4 * hf + (r % 4);
      if (d < RS && ((redo >> (16 * dt + r)) & 1) != 0) a.dq[qoff + d] = e[dt][r] * a.scale;
    }
}

// dQ and the row deltas; rank 0 = the last query block (the most keys).
template <int D, int MODE>
__global__ __launch_bounds__(kThreads, D <= 64 ? 2 : 1) void k_fbwd_dq_split(FbwdArgs a) {
  constexpr int KB = D / 16, DT = (D + 31) / 32;
  typedef SplitStage<D, MODE, 32> St;
  constexpr int DP = St::DP, PS = St::PS, NV = St::NV;
  const int RS = MODE == 0 ? D : a.D;
  __shared__ __attribute__((aligned(16))) uint16_t lds[6 * PS];
  uint16_t* const sK = lds;
  uint16_t* const sV = lds + 3 * PS;

  const int H = a.H, N = a.N;
  const int bh = (int)(blockIdx.x % (unsigned)a.BH), rank = (int)(blockIdx.x / (unsigned)a.BH);
  const int b = bh / H, h = bh % H;
  const int blk = a.n_blocks - 1 - rank;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 31, hf = lane >> 5;
  const int wq0 = blk * kRows + wave * 32;
  const int qrow = wq0 + c;
  const bool qok = qrow < N;
  const int qr = qok ? qrow : N - 1;
  const size_t qoff = row_off(b, qr, N, H, h, RS);
  const uint32_t rs = (uint32_t)(H * RS);
  const float* kh = a.k + row_off(b, 0, N, H, h, RS);
  const float* vh = a.v + row_off(b, 0, N, H, h, RS);

  // Dl of this lane's query, the sum taken as k_fbwd_delta takes it
  float dl = 0.f;
#pragma unroll
  for (int g = 0; g < D / 8; ++g) {
    const f32x4 x = load4m<MODE>(a.dout + qoff, 8 * g + 4 * hf, RS);
    const f32x4 y = load4m<MODE>(a.o + qoff, 8 * g + 4 * hf, RS);
    dl += x.x * y.x + x.y * y.y + x.z * y.z + x.w * y.w;
  }
  dl = xor32_sum(dl);
  const size_t srow = (size_t)(b * N + qr) * H + h;
  if (qok && hf == 0) a.delta[srow] = dl;
  const float m2 = a.M[srow] * LOG2E;
  const float il = 1.f / a.L[srow];
  const int qlim = qok ? qrow : -1;  // keys <= qlim are unmasked

  bf16x8 qf[KB][3], df[KB][3];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int d0 = 16 * kb + 8 * hf;
    split8(load4m<MODE>(a.q + qoff, d0, RS) * kSplitScale,
           load4m<MODE>(a.q + qoff, d0 + 4, RS) * kSplitScale, qf[kb]);
    split8(load4m<MODE>(a.dout + qoff, d0, RS) * kSplitScale,
           load4m<MODE>(a.dout + qoff, d0 + 4, RS) * kSplitScale, df[kb]);
  }
  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16{};
  const int pieces = (min(blk * kRows + kRows, N) + 31) / 32;
  const int wq_last = wq0 < N ? min(wq0 + 31, N - 1) : -1;  // -1: the wave has no query

  // dS of a piece from S and dP, which carry prod (1 / unit), P taking p_scale
  auto to_ds = [&](const f32x16& s, f32x16& dp, int key0, float unit, float prod, float p_scale) {
    const float sl2 = a.sl2 * unit, dlp = dl * prod, ilp = il * p_scale;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = key0 + 8 * (r / 4) + 4 * hf + (r % 4);
      const float e = fast_exp2(fmaf(s[r], sl2, -m2)) * ilp;
      const float p = key <= qlim ? e : 0.f;
      dp[r] = (dp[r] - dlp) * p;
    }
  };
  St st[2];  // K, V
  auto load_piece = [&](int j) {
#pragma unroll
    for (int i = 0; i < 2 * NV; ++i)
      st[i / NV].load(i % NV, i < NV ? kh : vh, j * 32, N, rs, RS);
  };
  load_piece(0);
  for (int j = 0; j < pieces; ++j) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2 * NV; ++i) st[i / NV].store(i % NV, i < NV ? sK : sV, kSplitScale);
    __syncthreads();
    if (j + 1 < pieces) load_piece(j + 1);
    const int key0 = j * 32;
    if (key0 > wq_last) continue;  // wave-uniform: every later key is masked for this wave
    f32x16 s = f32x16{}, dp = f32x16{};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      bf16x8 ka[3], va[3];
      read_rows<DP, PS>(sK, c, kb, hf, ka);
      read_rows<DP, PS>(sV, c, kb, hf, va);
      s = mfma_split_swapped(ka, qf[kb], s);
      dp = mfma_split_swapped(va, df[kb], dp);
    }
    to_ds(s, dp, key0, kSplitUnscale, kProdScale, kPScale);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 f[3];
      split_tile(dp, kk, f);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        bf16x8 kt[3];
        read_cols<DP, PS>(sK, 16 * kk, dt, lane, kt);
        acc[dt] = mfma_split(kt, f, acc[dt]);
      }
    }
  }
  finish_dq<DT, MODE>(a, acc, kGradUnscale, qoff, qok, wq_last, kh, rs, RS, c, hf, [&](int key0) {
    f32x16 s = f32x16{}, dp = f32x16{};
    const size_t ko = (size_t)min(key0 + c, N - 1) * rs;
#pragma unroll kAgain<MODE>
    for (int g = 0; g < D / 8; ++g) {
      const int d0 = 8 * g + 4 * hf;
      const f32x4 ka = load4m<MODE>(kh + ko, d0, RS), va = load4m<MODE>(vh + ko, d0, RS);
      const f32x4 qa = load4m<MODE>(a.q + qoff, d0, RS), da = load4m<MODE>(a.dout + qoff, d0, RS);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        s = mfma_f32(ka[t], qa[t], s);
        dp = mfma_f32(va[t], da[t], dp);
      }
    }
    to_ds(s, dp, key0, 1.f, 1.f, 1.f);
    return dp;
  });
}

// dQ from the stored dS: per 32-key piece the lane of query c loads its dS
// row's keys a step ahead, and K goes through LDS. dS of a key past the
// query (or past N) is masked by a select: k_fbwd_dkv_split wrote only the
// pieces it formed.
template <int D, int MODE>
__global__ __launch_bounds__(kThreads) void k_fbwd_dq_ds_split(FbwdArgs a) {
  constexpr int DT = (D + 31) / 32;
  typedef SplitStage<D, MODE, 64> St;
  constexpr int DP = St::DP, PS = St::PS, NV = St::NV;
  const int RS = MODE == 0 ? D : a.D;
  __shared__ __attribute__((aligned(16))) uint16_t sK[3 * PS];

  const int H = a.H, N = a.N;
  const int bh = (int)(blockIdx.x % (unsigned)a.BH), rank = (int)(blockIdx.x / (unsigned)a.BH);
  const int b = bh / H, h = bh % H;
  const int blk = a.n_blocks - 1 - rank;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 31, hf = lane >> 5;
  const int wq0 = blk * kRows + wave * 32;
  const int qrow = wq0 + c;
  const bool qok = qrow < N;
  const int qlim = qok ? qrow : -1;  // keys <= qlim are unmasked
  const uint32_t rs = (uint32_t)(H * RS);
  const float* kh = a.k + row_off(b, 0, N, H, h, RS);

  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16{};
  const int pieces = (min(blk * kRows + kRows, N) + 31) / 32;
  const int wq_last = wq0 < N ? min(wq0 + 31, N - 1) : -1;

  // masked only where it is used, so that the load is not waited for at once
  auto load_ds = [&](int key0, f32x4 (&x)[4]) {
    const float* tp = ds_tile(a, bh, wq0 >> 5, key0 >> 5) + c * 32 + 16 * hf;
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) x[qq] = *reinterpret_cast<const f32x4*>(tp + 4 * qq);
  };
  auto mask_ds = [&](int key0, f32x4 (&x)[4]) {
#pragma unroll
    for (int qq = 0; qq < 4; ++qq)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        x[qq][t] = key0 + 8 * qq + 4 * hf + t <= qlim ? x[qq][t] : 0.f;
  };
  // 64 keys a step: their dS (two pieces) and K are loaded a step ahead, the
  // dS into two register sets used in turn.
  f32x4 ds[2][2][4] = {};
  auto load_step = [&](int j, f32x4 (&x)[2][4]) {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
      if (j * 64 + sub * 32 <= wq_last) load_ds(j * 64 + sub * 32, x[sub]);
  };
  const int steps = (pieces + 1) / 2;
  load_step(0, ds[0]);
  St st;
#pragma unroll
  for (int i = 0; i < NV; ++i) st.load(i, kh, 0, N, rs, RS);
  auto step = [&](auto fc, int j) {
    constexpr int F = decltype(fc)::value;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; ++i) st.store(i, sK, kSplitScale);
    __syncthreads();
    if (j + 1 < steps) {
#pragma unroll
      for (int i = 0; i < NV; ++i) st.load(i, kh, (j + 1) * 64, N, rs, RS);
      load_step(j + 1, ds[F ^ 1]);
    }
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int key0 = j * 64 + sub * 32;
      if (key0 > wq_last) break;  // wave-uniform: every later key is masked for this wave
      f32x4 (&cur)[4] = ds[F][sub];
      mask_ds(key0, cur);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        bf16x8 f[3];
        split8(cur[2 * kk] * kSplitScale, cur[2 * kk + 1] * kSplitScale, f);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          bf16x8 kt[3];
          read_cols<DP, PS>(sK, sub * 32 + 16 * kk, dt, lane, kt);
          acc[dt] = mfma_split(kt, f, acc[dt]);
        }
      }
    }
  };
  for (int j = 0; j < steps; j += 2) {
    step(std::integral_constant<int, 0>{}, j);
    if (j + 1 < steps) step(std::integral_constant<int, 1>{}, j + 1);
  }
  finish_dq<DT, MODE>(a, acc, kSplitUnscale, row_off(b, qrow, N, H, h, RS), qok, wq_last, kh, rs, RS, c,
                      hf, [&](int key0) {
    f32x4 x[4];
    load_ds(key0, x);
    mask_ds(key0, x);
    f32x16 y;
#pragma unroll
    for (int r = 0; r < 16; ++r) y[r] = x[r >> 2][r & 3];
    return y;
  });
}

}  // namespace

int flash_fwd_split(const FfwdArgs& a, hipStream_t s, const char* fn) {
  const FlashShape fs = flash_shape(a.D);
  const dim3 grid((unsigned)(a.n_blocks * a.BH));
#define SKV_FF(DD, MM)             \
  if (fs.DP == DD && fs.mode == MM) \
    hipLaunchKernelGGL((k_flash_fwd_split<DD, MM>), grid, dim3(kThreads), 0, s, a);
  SKV_FLASH_SHAPES(SKV_FF)
#undef SKV_FF
  return check_launch(fn);
}

int flash_bwd_split(const FbwdArgs& a, hipStream_t s, const char* fn) {
  const FlashShape fs = flash_shape(a.D);
  const dim3 grid((unsigned)(a.n_blocks * a.BH));
  // seven products: dQ (and the deltas), then dK and dV
#define SKV_FB(DD, MM)                                                                         \
  if (fs.DP == DD && fs.mode == MM) {                                                          \
    hipLaunchKernelGGL((k_fbwd_dq_split<DD, MM>), grid, dim3(kThreads), 0, s, a);              \
    const int rc = check_launch(fn);                                                           \
    if (rc) return rc;                                                                         \
    hipLaunchKernelGGL((k_fbwd_dkv_split<DD, MM, false>), grid, dim3(kThreads), 0, s, a);      \
    return check_launch(fn);                                                                   \
  }
  // five products (a.ds set, the deltas written): dK, dV and dS, then dQ from dS
#define SKV_FB_DS(DD, MM)                                                                      \
  if (fs.DP == DD && fs.mode == MM) {                                                          \
    hipLaunchKernelGGL((k_fbwd_dkv_split<DD, MM, true>), grid, dim3(kThreads), 0, s, a);       \
    const int rc = check_launch(fn);                                                           \
    if (rc) return rc;                                                                         \
    hipLaunchKernelGGL((k_fbwd_dq_ds_split<DD, MM>), grid, dim3(kThreads), 0, s, a);           \
    return check_launch(fn);                                                                   \
  }
  if (a.ds != nullptr) {
    SKV_FB_DS(16, 0) SKV_FB_DS(16, 1) SKV_FB_DS(16, 2) SKV_FB_DS(32, 0) SKV_FB_DS(32, 1)
    SKV_FB_DS(32, 2) SKV_FB_DS(48, 0) SKV_FB_DS(48, 1) SKV_FB_DS(48, 2) SKV_FB_DS(64, 0)
    SKV_FB_DS(64, 1) SKV_FB_DS(64, 2)
  } else {
    SKV_FLASH_SHAPES(SKV_FB)
  }
#undef SKV_FB
#undef SKV_FB_DS
  return set_error(SKV_E_UNSUPPORTED, "%s: no kernel for head_dim %d", fn, a.D);
}

}  // namespace skv
