// Gated DeltaNet recurrence (gfx950, wave64): the decode step for S sessions and the chunked prefill.
//
// Per value head h (key head h % Hk), with decay = exp(g) and the state S[i][j] (i key, j value), a token does
// (reference ReferenceModel::LinearAttention, src/model/reference.cpp:329-364):
//   u = (decay S)^T k,  delta = (v - u) * beta,  S <- decay S + k delta^T,  o = S^T q / sqrt(d).
// State layout in HBM: fp32 [session][head][i][j], key-major (row i holds the 128 value columns contiguously),
// so that a lane's 16-byte load covers 4 value columns and a wave covers whole rows.
#include "common.h"

using halo::kWave;

namespace {
constexpr int kD = 128;       // head dim (d_k = d_v)
constexpr int kJBlock = 32;   // value columns per block
}  // namespace

// grid (S * Hv * 4), block 256. Block -> (session s, head h, value columns [32 jb, 32 jb + 32)); thread: 4 value
// columns (one float4) x 4 key rows. Columns are independent in the recurrence, so the four column blocks of a
// head run in parallel.
//   state [S][Hv][128][128] fp32 (in place), q, k [S][Hk][128], v [S][Hv][128], g, beta [S][Hv], o [S][Hv][128].
extern "C" __global__ void __launch_bounds__(256)
    halo_gdn_decode_d128(float* __restrict__ state, const float* __restrict__ q, const float* __restrict__ k,
                         const float* __restrict__ v, const float* __restrict__ g, const float* __restrict__ beta,
                         float* __restrict__ o, std::uint32_t S, std::uint32_t Hv, std::uint32_t Hk) {
  __shared__ float red[32][kJBlock + 1];
  __shared__ float dl[kJBlock];
  const std::uint32_t b = blockIdx.x, jb = b % 4, h = (b / 4) % Hv, s = b / (4 * Hv);
  if (s >= S) return;
  const std::uint32_t t = threadIdx.x, r8 = t % 8, ig = t / 8;
  const std::uint32_t j0 = jb * kJBlock + r8 * 4, i0 = ig * 4;
  const std::uint32_t kh = h % Hk;
  float* St = state + ((static_cast<std::size_t>(s) * Hv + h) * kD) * kD;
  const float* kk = k + (static_cast<std::size_t>(s) * Hk + kh) * kD;
  const float* qq = q + (static_cast<std::size_t>(s) * Hk + kh) * kD;
  const float decay = expf(g[s * Hv + h]);
  const float bt = beta[s * Hv + h];
  float4 row[4];
  float ki[4], qi[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    row[r] = *reinterpret_cast<const float4*>(St + static_cast<std::size_t>(i0 + r) * kD + j0);
    ki[r] = kk[i0 + r];
    qi[r] = qq[i0 + r];
  }
  float u[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    row[r].x *= decay;
    row[r].y *= decay;
    row[r].z *= decay;
    row[r].w *= decay;
    u[0] += row[r].x * ki[r];
    u[1] += row[r].y * ki[r];
    u[2] += row[r].z * ki[r];
    u[3] += row[r].w * ki[r];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) red[ig][r8 * 4 + c] = u[c];
  __syncthreads();
  if (t < kJBlock) {
    float acc = 0.0f;
    for (int i = 0; i < 32; ++i) acc += red[i][t];
    const float vj = v[(static_cast<std::size_t>(s) * Hv + h) * kD + jb * kJBlock + t];
    dl[t] = (vj - acc) * bt;
  }
  __syncthreads();
  const float d0 = dl[r8 * 4], d1 = dl[r8 * 4 + 1], d2 = dl[r8 * 4 + 2], d3 = dl[r8 * 4 + 3];
  float oo[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    row[r].x += ki[r] * d0;
    row[r].y += ki[r] * d1;
    row[r].z += ki[r] * d2;
    row[r].w += ki[r] * d3;
    oo[0] += row[r].x * qi[r];
    oo[1] += row[r].y * qi[r];
    oo[2] += row[r].z * qi[r];
    oo[3] += row[r].w * qi[r];
    *reinterpret_cast<float4*>(St + static_cast<std::size_t>(i0 + r) * kD + j0) = row[r];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) red[ig][r8 * 4 + c] = oo[c];
  __syncthreads();
  if (t < kJBlock) {
    float acc = 0.0f;
    for (int i = 0; i < 32; ++i) acc += red[i][t];
    o[(static_cast<std::size_t>(s) * Hv + h) * kD + jb * kJBlock + t] = acc * (1.0f / sqrtf(static_cast<float>(kD)));
  }
}

// ---- chunked prefill (C = 64) over a ragged batch of sequences, on fp32 MFMA -----------------------------------
// Within a chunk of C tokens with cumulative log-decay G_t (gamma_t = exp(G_t)) and initial state S0, the token
// recurrence above is exactly (reference math comment src/kernels/core.hip:6035-6048, there with C = 16):
//   (I + A) Delta = diag(beta) V - diag(beta gamma) K S0,   A[t][s] = beta_t exp(G_t - G_s) (k_t . k_s), s < t
//   O = (diag(gamma) Q S0 + P Delta) / sqrt(d),             P[t][s] = exp(G_t - G_s) (q_t . k_s),         s <= t
//   S_C = gamma_C S0 + K^T diag(exp(G_C - G_s)) Delta.
// With T = (I + A)^-1 this splits into what does not depend on the state (WY form, computed for every chunk in
// parallel by halo_gdn_wy_prep):
//   Uk = T diag(beta gamma) K,  Wv = T diag(beta) V,  Qe = diag(gamma) Q - P Uk,  Ov = P Wv      (64 x 128 each)
// and the chunk-serial part (halo_gdn_wy_scan), three products per chunk:
//   Delta = Wv - Uk S0,  O = (Qe S0 + Ov) / sqrt(d),  S_C = gamma_C S0 + K^T diag(exp(G_C - G_s)) Delta.
// Tokens past a partial chunk's end have k = 0, beta = 0, g = 0 in the preparation, so their rows of Uk and Wv are zero, and
// weight 0 in the state's update; their q and v repeat the last token's (v meets beta = 0, the rows of Qe are not used). Inputs q, k [tokens][Hk][128] and v [tokens][Hv][128] are bf16 (the C3 operator) or fp32 (the model's
// prefill, which matches its decode step); g, beta [tokens][Hv] fp32 (g = log decay, beta after its sigmoid); state
// fp32 [seq][Hv][128][128] key-major. chunks [n][3] = {first token, length, sequence}; seqs [n_seq][2] = {first
// chunk, chunk count}. Workspace per (chunk, head): Uk, Qe, Wv, Ov fp32 [64][128] and the weights [64].
namespace {
constexpr int kC = 64;
typedef float V4F __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float Bf(std::uint16_t h) { return __uint_as_float(static_cast<std::uint32_t>(h) << 16); }
__device__ __forceinline__ float Cv(std::uint16_t h) { return Bf(h); }
__device__ __forceinline__ float Cv(float x) { return x; }
// eight consecutive inputs (16 bytes of bf16, 32 of fp32)
template <typename In>
struct alignas(16) Pack8 {
  In v[8];
};
template <typename In>
__device__ __forceinline__ Pack8<In> Ld8(const In* p) {
  return *reinterpret_cast<const Pack8<In>*>(p);
}
}  // namespace

// grid (n_chunks, Hv), block 512 (8 waves). All products on v_mfma_f32_16x16x4f32 with instruction e of a 16-deep step taking
// k = 4 (lane / 16) + e: an A operand is then 16 bytes of a row, and a result (column lane % 16, rows 4 (lane / 16) + r) is in
// place the B operand of a product over its rows. A (then T = (I + A)^-1) and P are lower triangular: the ten 16 x 16
// tiles on and below the diagonal, tile i (i + 1) / 2 + j in LDS with rows of 20 floats (free of bank conflicts), and
// nothing above is computed.
//   1. K into LDS (fp32, 16-byte groups xor-swizzled by the row); the 20 tiles of K K^T and Q K^T over the waves (five per
//      SIMD), Q rows straight from memory; scaled into A and P.
//   2. T by 16 x 16 blocks: four waves invert the diagonal blocks by forward substitution (a column per lane), then each
//      forms one block column, T_ij = -T_ii sum_m A_im T_mj, its blocks passing from result to operand in registers.
//   3. wave w, columns 16 w .. + 16: Uk = (T diag(beta gamma)) K and Wv = (T diag(beta)) V, and from those registers
//      Qe = diag(gamma) Q - P Uk and Ov = P Wv.
// What bounds it: the fp32 matrix products (80 + 160 + 160 instructions of 32 cycles per SIMD pair of waves); 59 KB of LDS,
// so that two blocks per CU cover each other's barriers and the substitution. (With whole 64 x 64 products, K, Q and V
// in 137 KB of LDS and the substitution in one wave: 0.76 ms on the ragged batch {37, 512, 2048, 8191}; this 0.37 ms, of
// which the 709 MB it writes take about half.)
namespace {
constexpr int kTS = 20;          // floats per row of a 16 x 16 tile
constexpr int kTF = 16 * kTS;    // floats per tile
__device__ __forceinline__ constexpr int Tri(int i, int j) { return i * (i + 1) / 2 + j; }
__device__ __forceinline__ V4F Mfma16(const float4& a, const V4F& b, V4F c) {
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b[1], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b[2], c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b[3], c, 0, 0, 0);
}
__device__ __forceinline__ float4 Ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 Ld4(const std::uint16_t* p) {
  const ushort4 u = *reinterpret_cast<const ushort4*>(p);
  return make_float4(Bf(u.x), Bf(u.y), Bf(u.z), Bf(u.w));
}

template <typename In>
__device__ __forceinline__ void WyPrep(const In* __restrict__ q, const In* __restrict__ k, const In* __restrict__ v,
                                       const float* __restrict__ g, const float* __restrict__ beta,
                                       const std::uint32_t* __restrict__ chunks, float* __restrict__ wy,
                                       float* __restrict__ Wt, std::uint32_t Hv, std::uint32_t Hk) {
  __shared__ __attribute__((aligned(16))) float kl[kC * kD];
  __shared__ __attribute__((aligned(16))) float am[10 * kTF], pm[10 * kTF];
  __shared__ __attribute__((aligned(16))) float G[kC], Gl[kC], Bt[kC], Bg[kC], Gm[kC];  // G + Gl: the log-decays
  const std::uint32_t c = blockIdx.x, h = blockIdx.y, kh = h % Hk, tid = threadIdx.x;
  const std::uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave, fc = lane % 16, fq = lane / 16;
  const std::uint32_t start = chunks[c * 3], L = chunks[c * 3 + 1];
  const auto klat = [&](std::uint32_t t, std::uint32_t f4) { return &kl[t * kD + 4 * (f4 ^ (t & 7))]; };
  const In* kbase = k + (static_cast<std::size_t>(start) * Hk + kh) * kD;
  const In* qbase = q + (static_cast<std::size_t>(start) * Hk + kh) * kD;
  const In* vbase = v + (static_cast<std::size_t>(start) * Hv + h) * kD;
  // K: thread -> rows tid / 16 and + 32, 8 values at 8 (tid % 16)
  const std::uint32_t kt = tid / 16, kp = tid % 16;
  const Pack8<In> k0 = Ld8(kbase + static_cast<std::size_t>(min(kt, L - 1)) * Hk * kD + 8 * kp);
  const Pack8<In> k1 = Ld8(kbase + static_cast<std::size_t>(min(kt + 32, L - 1)) * Hk * kD + 8 * kp);
  float gv = 0.0f, bv = 0.0f;
  if (wave == 0) {
    const std::size_t at = static_cast<std::size_t>(start + min(lane, L - 1)) * Hv + h;
    gv = lane < L ? g[at] : 0.0f;
    bv = lane < L ? beta[at] : 0.0f;
  }
  const auto put = [&](std::uint32_t t, const Pack8<In>& x) {
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = t < L ? Cv(x.v[e]) : 0.0f;
    *reinterpret_cast<float4*>(klat(t, 2 * kp)) = make_float4(f[0], f[1], f[2], f[3]);
    *reinterpret_cast<float4*>(klat(t, 2 * kp + 1)) = make_float4(f[4], f[5], f[6], f[7]);
  };
  put(kt, k0);
  put(kt + 32, k1);
  if (wave == 0) {  // cumulative log-decays, in double: tokens apart by little are weighted by differences of large sums
    double sum = gv;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const double up = __shfl_up(sum, d);
      sum += lane >= static_cast<std::uint32_t>(d) ? up : 0.0;
    }
    const float hi = static_cast<float>(sum), lo = static_cast<float>(sum - hi);
    const float e = expf(hi), gm = __builtin_fmaf(e, lo, e);
    G[lane] = hi;
    Gl[lane] = lo;
    Bt[lane] = bv;
    Gm[lane] = gm;
    Bg[lane] = bv * gm;
  }
  __syncthreads();
  // tiles of K K^T (jobs 0-9) and Q K^T (10-19)
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    const std::uint32_t job = wave + 8 * n;
    if (job < 20) {
      const bool isp = job >= 10;
      const std::uint32_t tl = isp ? job - 10 : job, i = tl < 1 ? 0 : tl < 3 ? 1 : tl < 6 ? 2 : 3, j = tl - i * (i + 1) / 2;
      const std::uint32_t ra = 16 * i + fc, rb = 16 * j + fc;
      float4 a[8];
      if (isp) {
        const In* qr = qbase + static_cast<std::size_t>(min(ra, L - 1)) * Hk * kD + 4 * fq;
#pragma unroll
        for (int sb = 0; sb < 8; ++sb) a[sb] = Ld4(qr + 16 * sb);
      } else {
#pragma unroll
        for (int sb = 0; sb < 8; ++sb) a[sb] = *reinterpret_cast<const float4*>(klat(ra, 4 * sb + fq));
      }
      V4F acc[2] = {V4F{0.0f, 0.0f, 0.0f, 0.0f}, V4F{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
      for (int sb = 0; sb < 8; ++sb)
        acc[sb % 2] = Mfma16(a[sb], __builtin_bit_cast(V4F, *reinterpret_cast<const float4*>(klat(rb, 4 * sb + fq))), acc[sb % 2]);
      const float4 gt = *reinterpret_cast<const float4*>(&G[16 * i + 4 * fq]), bt = *reinterpret_cast<const float4*>(&Bt[16 * i + 4 * fq]);
      const float4 gl = *reinterpret_cast<const float4*>(&Gl[16 * i + 4 * fq]);
      const float gs = G[rb], gsl = Gl[rb], gta[4] = {gt.x, gt.y, gt.z, gt.w}, gla[4] = {gl.x, gl.y, gl.z, gl.w};
      const float bta[4] = {bt.x, bt.y, bt.z, bt.w};
      float* out = (isp ? pm : am) + tl * kTF + 4 * fq * kTS + fc;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const std::uint32_t t = 16 * i + 4 * fq + r;
        const float x = acc[0][r] + acc[1][r], dec = expf(rb <= t ? (gta[r] - gs) + (gla[r] - gsl) : 0.0f);
        out[r * kTS] = isp ? (rb <= t ? dec * x : 0.0f) : (rb < t ? bta[r] * dec * x : 0.0f);
      }
    }
  }
  // this wave's columns of V (B operand) and Q (result layout), in flight across the inversion
  const std::uint32_t col = 16 * wave + fc;
  V4F vb[4], qc[4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const std::size_t t = min(16u * m + 4 * fq + e, L - 1);
      vb[m][e] = Cv(vbase[t * Hv * kD + col]);
      qc[m][e] = Cv(qbase[t * Hk * kD + col]);
    }
  halo::LdsSync();
  if (wave < 4) {  // diagonal block `wave`
    float* d = am + Tri(wave, wave) * kTF;
    float T[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float s4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int x = 0; x < t; x += 4) {
        const float4 ar = *reinterpret_cast<const float4*>(d + t * kTS + x);
        const float av[4] = {ar.x, ar.y, ar.z, ar.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (x + e < t) s4[e] = __builtin_fmaf(av[e], T[x + e], s4[e]);
      }
      T[t] = (fc == static_cast<std::uint32_t>(t) ? 1.0f : 0.0f) - ((s4[0] + s4[1]) + (s4[2] + s4[3]));
    }
#pragma unroll
    for (int t = 0; t < 16; ++t) d[t * kTS + fc] = T[t];  // (the block's rows have all been read: program order)
  }
  halo::LdsSync();
  const auto atile = [&](const float* m, int tl) { return *reinterpret_cast<const float4*>(m + tl * kTF + fc * kTS + 4 * fq); };
  V4F tc[4];
  if (wave < 4) {  // block column `wave` of T
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (static_cast<std::uint32_t>(j) == wave) {
#pragma unroll
        for (int e = 0; e < 4; ++e) tc[j][e] = am[Tri(j, j) * kTF + (4 * fq + e) * kTS + fc];
#pragma unroll
        for (int i = j + 1; i < 4; ++i) {
          V4F acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int m = j; m < i; ++m) acc = Mfma16(atile(am, Tri(i, m)), tc[m], acc);
          const V4F z = {0.0f, 0.0f, 0.0f, 0.0f};
          tc[i] = -Mfma16(atile(am, Tri(i, i)), acc, z);
        }
      }
  }
  halo::LdsSync();  // A has been read
  if (wave < 4) {
#pragma unroll
    for (int j = 0; j < 3; ++j)
      if (static_cast<std::uint32_t>(j) == wave) {
#pragma unroll
        for (int i = j + 1; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) am[Tri(i, j) * kTF + (4 * fq + e) * kTS + fc] = tc[i][e];
      }
  }
  halo::LdsSync();
  V4F uk[4], wv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) uk[i] = wv[i] = V4F{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    V4F kb;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const std::uint32_t t = 16 * m + 4 * fq + e;
      kb[e] = klat(t, col / 4)[col % 4];
    }
    const float4 bg = *reinterpret_cast<const float4*>(&Bg[16 * m + 4 * fq]), bt = *reinterpret_cast<const float4*>(&Bt[16 * m + 4 * fq]);
#pragma unroll
    for (int i = m; i < 4; ++i) {
      const float4 t = atile(am, Tri(i, m));
      uk[i] = Mfma16(make_float4(t.x * bg.x, t.y * bg.y, t.z * bg.z, t.w * bg.w), kb, uk[i]);
      wv[i] = Mfma16(make_float4(t.x * bt.x, t.y * bt.y, t.z * bt.z, t.w * bt.w), vb[m], wv[i]);
    }
  }
  float* out = wy + (static_cast<std::size_t>(c) * Hv + h) * 4 * kC * kD;  // Uk, Qe, Wv, Ov
  const auto store = [&](int which, int i, const V4F& x) {
#pragma unroll
    for (int r = 0; r < 4; ++r) out[which * kC * kD + (16 * i + 4 * fq + r) * kD + col] = x[r];
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    store(0, i, uk[i]);
    store(2, i, wv[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 gm = *reinterpret_cast<const float4*>(&Gm[16 * i + 4 * fq]);
    V4F qe = {gm.x * qc[i][0], gm.y * qc[i][1], gm.z * qc[i][2], gm.w * qc[i][3]}, ov = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m <= i; ++m) {
      const float4 p = atile(pm, Tri(i, m));
      qe = Mfma16(make_float4(-p.x, -p.y, -p.z, -p.w), uk[m], qe);
      ov = Mfma16(p, wv[m], ov);
    }
    store(1, i, qe);
    store(3, i, ov);
  }
  // the scan's weights: exp(G_C - G_t) of token t, 0 past the end; the last word, whose weight is 1 in a whole chunk and
  // 0 in a shorter one, holds gamma_C instead
  if (tid < kC)
    Wt[(static_cast<std::size_t>(c) * Hv + h) * kC + tid] =
        tid == kC - 1 ? Gm[kC - 1] : tid < L ? expf((G[kC - 1] - G[tid]) + (Gl[kC - 1] - Gl[tid])) : 0.0f;
}

// grid (n_seq * Hv * 128 / kNC), block 512 (8 waves): block -> (sequence, kNC value columns, head); walks the sequence's
// chunks carrying its 128 x kNC slice of S. MFMA v_mfma_f32_16x16x4f32 (A lane l = A[l % 16][k], B lane l = B[k][l % 16],
// D lane l holds column l % 16 and rows 4 (l / 16) + r); instruction (sb, e) takes k = 16 sb + 4 (l / 16) + e, so every
// operand is 16 bytes of a row for four instructions.
// Per chunk: waves 0-3 form Delta rows 16 w .. + 16 (= Wv - Uk S0), waves 4-7 the output rows (Qe S0 + Ov); then wave w
// updates S rows (keys) 16 w .. + 16, which it keeps in its accumulators for the whole sequence.
// What bounds it: the chunk-serial path of one block (a long sequence has one block per CU), so everything off that path
// is off it: Uk, Qe, K, Wv, Ov and the weights are read once by exactly the lanes that multiply them, so they come
// from memory straight into operand registers, one chunk ahead (each register is reloaded as soon as its chunk has used
// it); LDS holds only what the waves exchange, S^T and Delta^T, with two barriers per chunk. The loads stand among
// the products: issued behind them, they take the vector memory pipe as long again as half the products. (Staging the
// operands in LDS: 515 us for 8000 tokens in slices of 16 columns, 720 us for the ragged batch in slices of 32; this 440
// and 590.)
// h varies fastest over the grid: a head's slices land on one XCD (Hv % 8 == 0), whose L2 they share (the time is the same in
// either order: memory is not what binds).
template <typename In, int kNC>
__device__ __forceinline__ void WyScan(const In* __restrict__ k, const float* __restrict__ wy,
                                       const float* __restrict__ Wt, const std::uint32_t* __restrict__ chunks,
                                       const std::uint32_t* __restrict__ seqs, float* __restrict__ state,
                                       float* __restrict__ o, std::uint32_t Hv, std::uint32_t Hk) {
  constexpr int kNB = kD / kNC, kNT = kNC / 16, kDL = kC + 4, kStL = kD + 4;
  __shared__ __attribute__((aligned(16))) float st[kNC][kStL];  // S^T slice: [column][key]
  __shared__ __attribute__((aligned(16))) float dt[kNC][kDL];   // Delta^T slice: [column][token]
  // Blocks are dispatched in id order, so the longest sequences take the lowest ids (rank by descending chunk count, ties
  // by index; up to 64 sequences, else in order): the chunk-serial critical path starts first.
  __shared__ std::uint32_t sq_s;
  const std::uint32_t b = blockIdx.x, h = b % Hv, cb = (b / Hv) % kNB, rank = b / (kNB * Hv);
  const std::uint32_t n_seq = gridDim.x / (kNB * Hv);
  if (threadIdx.x == 0) {
    std::uint32_t pick = rank;
    if (n_seq <= 64) {
      for (std::uint32_t j = 0; j < n_seq; ++j) {
        const std::uint32_t cj = seqs[j * 2 + 1];
        std::uint32_t r = 0;
        for (std::uint32_t i = 0; i < n_seq; ++i) {
          const std::uint32_t ci = seqs[i * 2 + 1];
          r += (ci > cj) || (ci == cj && i < j);
        }
        if (r == rank) pick = j;
      }
    }
    sq_s = pick;
  }
  __syncthreads();
  const std::uint32_t sq = __builtin_amdgcn_readfirstlane(sq_s), kh = h % Hk;
  const std::uint32_t tid = threadIdx.x, lane = tid % kWave, fc = lane % 16, fq = lane / 16;
  const std::uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const std::uint32_t j0 = cb * kNC, r0 = 16 * (wave % 4), s0 = 16 * wave;
  const bool delta = wave < 4;
  const std::uint32_t c0 = seqs[sq * 2], nc = seqs[sq * 2 + 1];
  if (nc == 0) return;
  // a sequence's chunks are consecutive 64-token runs: chunk ci starts at first + 64 ci and holds
  // min(64, len - 64 ci) tokens (no chunk-table read per chunk: those scalar loads sat on the serial path)
  const std::uint32_t first = chunks[c0 * 3];
  const std::uint32_t len = chunks[(c0 + nc - 1) * 3] + chunks[(c0 + nc - 1) * 3 + 1] - first;
  float* Sg = state + (static_cast<std::size_t>(sq) * Hv + h) * kD * kD;
  V4F S[kNT];  // S[s0 + 4 fq + i][j0 + 16 ct + fc]
#pragma unroll
  for (int ct = 0; ct < kNT; ++ct) {
#pragma unroll
    for (int i = 0; i < 4; ++i) S[ct][i] = Sg[static_cast<std::size_t>(s0 + 4 * fq + i) * kD + j0 + 16 * ct + fc];
    *reinterpret_cast<float4*>(&st[16 * ct + fc][s0 + 4 * fq]) = make_float4(S[ct][0], S[ct][1], S[ct][2], S[ct][3]);
  }
  // this lane's operands of the chunk to come: A rows of Uk or Qe, the Wv or Ov values its results join, K^T rows, weights
  float4 ra[8], rw[4];
  float rv[kNT][4], rk[16];
  const std::size_t tile = kC * kD, step = static_cast<std::size_t>(Hv) * 4 * tile;
  const float* pa = wy + (static_cast<std::size_t>(c0) * Hv + h) * 4 * tile;  // Uk, Qe, Wv, Ov of the chunk to load
  const float* pw = Wt + (static_cast<std::size_t>(c0) * Hv + h) * kC;
  const std::uint32_t aoff = (delta ? 0u : kC * kD) + (r0 + fc) * kD + 4 * fq;
  const std::uint32_t voff = (delta ? 2u : 3u) * kC * kD + (r0 + 4 * fq) * kD + j0 + fc;
  const auto load_a = [&](int sb) { ra[sb] = *reinterpret_cast<const float4*>(pa + aoff + 16 * sb); };
  const auto load_v = [&]() {
#pragma unroll
    for (int ct = 0; ct < kNT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) rv[ct][i] = pa[voff + i * kD + 16 * ct];
  };
  // K^T row s0 + fc, tokens 16 sb + 4 fq + e: a uniform row address plus the lane's offset; rows past a short chunk's end
  // reload its last one (their weights are zero)
  const std::uint32_t kstride = Hk * kD;
  const auto load_k = [&](std::uint32_t ci, int sb) {
    const std::uint32_t start = first + 64 * ci, L = min(64u, len - 64 * ci);
    const In* kc = k + (static_cast<std::size_t>(start) * Hk + kh) * kD;
#pragma unroll
    for (int e = 0; e < 4; ++e) rk[4 * sb + e] = Cv(kc[__umul24(min(16u * sb + 4 * fq + e, L - 1), kstride) + s0 + fc]);
    rw[sb] = *reinterpret_cast<const float4*>(pw + 16 * sb + 4 * fq);
  };
#pragma unroll
  for (int sb = 0; sb < 8; ++sb) load_a(sb);
  load_v();
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) load_k(0, sb);
  float gc = pw[kC - 1];
  const float inv_sqrt_d = 1.0f / sqrtf(static_cast<float>(kD));
  halo::LdsSync();
  for (std::uint32_t ci = 0; ci < nc; ++ci) {
    const std::uint32_t start = first + 64 * ci, L = min(64u, len - 64 * ci), cn = ci + 1 < nc ? ci + 1 : ci;
    if (cn != ci) pa += step, pw += static_cast<std::size_t>(Hv) * kC;  // the last chunk reloads itself
    V4F acc[kNT][2];
#pragma unroll
    for (int ct = 0; ct < kNT; ++ct) acc[ct][0] = acc[ct][1] = V4F{0.0f, 0.0f, 0.0f, 0.0f};
    // operand rows of S^T in groups of kG steps, each read ahead of the group before it
    constexpr int kG = 2;
    float4 bv[2][kG][kNT];
    const auto read_s = [&](int g) {
#pragma unroll
      for (int i = 0; i < kG; ++i)
#pragma unroll
        for (int ct = 0; ct < kNT; ++ct)
          bv[g % 2][i][ct] = *reinterpret_cast<const float4*>(&st[16 * ct + fc][16 * (kG * g + i) + 4 * fq]);
    };
    read_s(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 8 / kG; ++g) {
      if (g + 1 < 8 / kG) read_s(g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kG; ++i) {
        const int sb = kG * g + i;
        const float4 av = ra[sb];
#pragma unroll
        for (int ct = 0; ct < kNT; ++ct) {
          const float4 x = bv[g % 2][i][ct];
          V4F& a = acc[ct][sb % 2];  // two chains
          a = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, x.x, a, 0, 0, 0);
          a = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, x.y, a, 0, 0, 0);
          a = __builtin_amdgcn_mfma_f32_16x16x4f32(av.z, x.z, a, 0, 0, 0);
          a = __builtin_amdgcn_mfma_f32_16x16x4f32(av.w, x.w, a, 0, 0, 0);
        }
        load_a(sb);  // among the products: issued together after them, the loads took as long as half the products
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int ct = 0; ct < kNT; ++ct) {
      const V4F a = acc[ct][0] + acc[ct][1];
      if (delta) {
        *reinterpret_cast<float4*>(&dt[16 * ct + fc][r0 + 4 * fq]) =
            make_float4(rv[ct][0] - a[0], rv[ct][1] - a[1], rv[ct][2] - a[2], rv[ct][3] - a[3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const std::uint32_t t = r0 + 4 * fq + i;
          if (t < L) o[(static_cast<std::size_t>(start + t) * Hv + h) * kD + j0 + 16 * ct + fc] = (a[i] + rv[ct][i]) * inv_sqrt_d;
        }
      }
    }
    load_v();
    halo::LdsSync();  // Delta^T is whole, S^T has been read
    // S rows: gamma_C S + (K diag(W))^T Delta over 64 tokens
    V4F upd[kNT];
#pragma unroll
    for (int ct = 0; ct < kNT; ++ct) S[ct] *= gc, upd[ct] = V4F{0.0f, 0.0f, 0.0f, 0.0f};
    gc = pw[kC - 1];
    float4 dv[4][kNT];
#pragma unroll
    for (int sb = 0; sb < 4; ++sb)
#pragma unroll
      for (int ct = 0; ct < kNT; ++ct) dv[sb][ct] = *reinterpret_cast<const float4*>(&dt[16 * ct + fc][16 * sb + 4 * fq]);
    float ka[16];  // K^T diag(W): while Delta^T arrives
#pragma unroll
    for (int sb = 0; sb < 4; ++sb) {
      ka[4 * sb] = rk[4 * sb] * rw[sb].x, ka[4 * sb + 1] = rk[4 * sb + 1] * rw[sb].y;
      ka[4 * sb + 2] = rk[4 * sb + 2] * rw[sb].z;
      ka[4 * sb + 3] = rk[4 * sb + 3] * (sb == 3 && fq == 3 ? (L == 64 ? 1.0f : 0.0f) : rw[sb].w);  // W[63]: gamma_C
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int sb = 0; sb < 4; ++sb) {
      load_k(cn, sb);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ct = 0; ct < kNT; ++ct) {
        V4F& u = sb % 2 ? upd[ct] : S[ct];
        u = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[4 * sb], dv[sb][ct].x, u, 0, 0, 0);
        u = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[4 * sb + 1], dv[sb][ct].y, u, 0, 0, 0);
        u = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[4 * sb + 2], dv[sb][ct].z, u, 0, 0, 0);
        u = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[4 * sb + 3], dv[sb][ct].w, u, 0, 0, 0);
      }
    }
#pragma unroll
    for (int ct = 0; ct < kNT; ++ct) {
      S[ct] += upd[ct];
      *reinterpret_cast<float4*>(&st[16 * ct + fc][s0 + 4 * fq]) = make_float4(S[ct][0], S[ct][1], S[ct][2], S[ct][3]);
    }
    halo::LdsSync();
  }
#pragma unroll
  for (int ct = 0; ct < kNT; ++ct)
#pragma unroll
    for (int i = 0; i < 4; ++i) Sg[static_cast<std::size_t>(s0 + 4 * fq + i) * kD + j0 + 16 * ct + fc] = S[ct][i];
}
}  // namespace

extern "C" __global__ void __launch_bounds__(512, 4)
    halo_gdn_wy_prep(const std::uint16_t* __restrict__ q, const std::uint16_t* __restrict__ k,
                     const std::uint16_t* __restrict__ v, const float* __restrict__ g, const float* __restrict__ beta,
                     const std::uint32_t* __restrict__ chunks, float* __restrict__ wy, float* __restrict__ Gc,
                     std::uint32_t Hv, std::uint32_t Hk) {
  WyPrep(q, k, v, g, beta, chunks, wy, Gc, Hv, Hk);
}
extern "C" __global__ void __launch_bounds__(512, 4)
    halo_gdn_wy_prep_f32(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                         const float* __restrict__ g, const float* __restrict__ beta,
                         const std::uint32_t* __restrict__ chunks, float* __restrict__ wy, float* __restrict__ Gc,
                         std::uint32_t Hv, std::uint32_t Hk) {
  WyPrep(q, k, v, g, beta, chunks, wy, Gc, Hv, Hk);
}
extern "C" __global__ void __launch_bounds__(512)
    halo_gdn_wy_scan(const std::uint16_t* __restrict__ k, const float* __restrict__ wy, const float* __restrict__ Gc,
                     const std::uint32_t* __restrict__ chunks, const std::uint32_t* __restrict__ seqs,
                     float* __restrict__ state, float* __restrict__ o, std::uint32_t Hv, std::uint32_t Hk) {
  WyScan<std::uint16_t, 32>(k, wy, Gc, chunks, seqs, state, o, Hv, Hk);
}
extern "C" __global__ void __launch_bounds__(512)
    halo_gdn_wy_scan_f32(const float* __restrict__ k, const float* __restrict__ wy, const float* __restrict__ Gc,
                         const std::uint32_t* __restrict__ chunks, const std::uint32_t* __restrict__ seqs,
                         float* __restrict__ state, float* __restrict__ o, std::uint32_t Hv, std::uint32_t Hk) {
  WyScan<float, 32>(k, wy, Gc, chunks, seqs, state, o, Hv, Hk);
}
// 16 value columns per block (eight blocks per head): for batches with too few (sequence, head) pairs to fill the
// CUs at 32 columns, halving each block's matrix work on the chunk-serial path
extern "C" __global__ void __launch_bounds__(512)
    halo_gdn_wy_scan_n16(const std::uint16_t* __restrict__ k, const float* __restrict__ wy, const float* __restrict__ Gc,
                         const std::uint32_t* __restrict__ chunks, const std::uint32_t* __restrict__ seqs,
                         float* __restrict__ state, float* __restrict__ o, std::uint32_t Hv, std::uint32_t Hk) {
  WyScan<std::uint16_t, 16>(k, wy, Gc, chunks, seqs, state, o, Hv, Hk);
}
extern "C" __global__ void __launch_bounds__(512)
    halo_gdn_wy_scan_f32_n16(const float* __restrict__ k, const float* __restrict__ wy, const float* __restrict__ Gc,
                             const std::uint32_t* __restrict__ chunks, const std::uint32_t* __restrict__ seqs,
                             float* __restrict__ state, float* __restrict__ o, std::uint32_t Hv, std::uint32_t Hk) {
  WyScan<float, 16>(k, wy, Gc, chunks, seqs, state, o, Hv, Hk);
}

// ---- the whole DeltaNet token step of the decode graph, one block per (session, value head) -----------------
// Fuses the prologue (causal conv + SiLU, q / k L2 norms, decay and beta gates), the delta-rule recurrence and the
// output RMSNorm * w * sigmoid(z) with its Q8 quantization for the output projection (reference
// ReferenceModel::LinearAttention, src/model/reference.cpp:278-366). The conv history is a ring of K slots per
// channel: position p's projection lives in slot p % K, so step p reads slots (p + 1 + j) % K (j < K - 1) and writes
// slot p % K, which no block of the same step reads; q / k channels of key head kh are read by every value head with
// h % Hk == kh but written only by value head h = kh (h < Hk), v channels by their own head. Positions: nkv[s] - 1.
//   qkv [S][C] (C = 2 Hk d + Hv d), z [S][Hv d], ab [S][2 Hv] (alpha | beta logits), ring [S][K][C], conv_w [C][K],
//   a, dt [Hv], norm_w [d], state [S][Hv][d][d] key-major fp32 (in place) -> oq [S][Hv d] int8, os [S][Hv d / 32].
// grid (S * Hv), block 512: thread t owns state rows 8 (t / 32) .. + 8 and columns 4 (t % 32) .. + 4. d = 128.
// halo_gdn_step_q8 takes K <= 4 (the ring slots in registers, loaded before the state), _kn any K <= 8.
namespace {
template <bool kSmallK>
__device__ __forceinline__ void GdnStepQ8(
    const float* __restrict__ qkv, const float* __restrict__ z, const float* __restrict__ ab, float* __restrict__ ring,
    const float* __restrict__ conv_w, const float* __restrict__ a, const float* __restrict__ dt,
    const float* __restrict__ norm_w, float* __restrict__ state, const std::uint32_t* __restrict__ nkv,
    std::int8_t* __restrict__ oq, float* __restrict__ os, std::uint32_t Hk, std::uint32_t Hv, std::uint32_t K,
    float eps) {
  __shared__ float sq[kD], sk[kD], sv[kD], dl[kD];
  __shared__ float red[16][kD + 4];
  __shared__ float part[8];
  __shared__ float gates[2];
  const std::uint32_t s = blockIdx.x / Hv, h = blockIdx.x % Hv, kh = h % Hk;
  const std::uint32_t t = threadIdx.x, wave = t / kWave, lane = t % kWave;
  const std::uint32_t cg = t % 32, rg = t / 32, j0 = 4 * cg, i0 = 8 * rg;
  const std::uint32_t Dk = Hk * kD, Dv = Hv * kD, C = 2 * Dk + Dv;
  float* St = state + (static_cast<std::size_t>(s) * Hv + h) * kD * kD;
  HALO_PHASE(0, 0);
  // prologue: threads 0..383 take the q, k and v channels of this head (128 each: waves 0-1, 2-3, 4-5). With K <= 4
  // every ring slot is loaded before the position arrives, so the ring loads do not wait for nkv; the slots are
  // selected by position afterwards.
  const std::uint32_t seg = t / kD, i = t % kD;
  const std::uint32_t ch = seg == 0 ? kh * kD + i : seg == 1 ? Dk + kh * kD + i : 2 * Dk + h * kD + min(i, kD - 1);
  float* rs = ring + static_cast<std::size_t>(s) * K * C;
  const std::uint32_t pos = nkv[s] - 1;
  const float zg = z[static_cast<std::size_t>(s) * Dv + h * kD + min(t, static_cast<std::uint32_t>(kD - 1))];  // t < kD
  float y = 0.0f;
  // the prologue's loads are issued before the state's (64 KB per block, eight 16-byte loads per thread), so the conv
  // and norms below run while the state streams in
  // (unconditional loads from clamped addresses, selected afterwards: a load under a branch would wait at the join
  // for every load issued before it, the state's included)
  const float x = qkv[static_cast<std::size_t>(s) * C + ch];
  float slot[4], w[4];
#pragma unroll
  for (std::uint32_t j = 0; j < 4; ++j) {
    const std::uint32_t jj = min(j, K - 1);
    slot[j] = rs[static_cast<std::size_t>(jj) * C + ch];
    w[j] = conv_w[static_cast<std::size_t>(ch) * K + jj];
  }
  const float ga = a[h], gdt = dt[h], galpha = ab[static_cast<std::size_t>(s) * 2 * Hv + h],
              gbeta = ab[static_cast<std::size_t>(s) * 2 * Hv + Hv + h];
  __builtin_amdgcn_sched_barrier(0);  // keep the issue order
  // Measured: the state issued only once the prologue's inputs have landed streams in ~2 us and leaves the conv and
  // norms free to run; issued right behind them, the wave stalls on issuing it (until ~2.7 us) with the conv waiting.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  float4 row[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) row[r] = *reinterpret_cast<const float4*>(St + static_cast<std::size_t>(i0 + r) * kD + j0);
  __builtin_amdgcn_sched_barrier(0);
  // the conv in every thread (waves 6-7 on a clamped channel, discarded), so the loads above stay where they are
  float acc;
  if constexpr (kSmallK) {
    acc = w[K - 1] * x;
#pragma unroll
    for (std::uint32_t j = 0; j < 3; ++j)
      if (j + 1 < K) acc += w[j] * slot[(pos + 1 + j) % K];
  } else {
    acc = conv_w[static_cast<std::size_t>(ch) * K + K - 1] * x;
    for (std::uint32_t j = 0; j + 1 < K; ++j)
      acc += conv_w[static_cast<std::size_t>(ch) * K + j] * rs[static_cast<std::size_t>((pos + 1 + j) % K) * C + ch];
  }
  if (seg < 3) {
    if (seg == 2 || h < Hk) rs[static_cast<std::size_t>(pos % K) * C + ch] = x;
    y = halo::Silu(acc);
  }
  const float ss = halo::GroupSum(y * y);
  if (lane == 0) part[wave] = ss;
  const float g0 = ga * halo::Softplus(galpha + gdt), g1 = halo::Sigmoid(gbeta);
  if (t == 0) {
    gates[0] = g0;
    gates[1] = g1;
  }
  __syncthreads();
  HALO_PHASE(0, 1);
  if (seg < 2) {
    const float sc = 1.0f / sqrtf(part[2 * seg] + part[2 * seg + 1] + eps);
    (seg == 0 ? sq : sk)[i] = y * sc;
  } else if (seg == 2) {
    sv[i] = y;
  }
  __syncthreads();
  HALO_PHASE(0, 2);
  // recurrence: u = (decay S)^T k, delta = (v - u) beta, S <- decay S + k delta^T, o = S^T q / sqrt(d)
  const float decay = expf(gates[0]), bt = gates[1];
  float u[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const float ki = sk[i0 + r];
    row[r].x *= decay;
    row[r].y *= decay;
    row[r].z *= decay;
    row[r].w *= decay;
    u[0] += row[r].x * ki;
    u[1] += row[r].y * ki;
    u[2] += row[r].z * ki;
    u[3] += row[r].w * ki;
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) red[rg][j0 + c] = u[c];
  __syncthreads();
  HALO_PHASE(0, 3);
  if (t < kD) {
    float acc = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc += red[r][t];
    dl[t] = (sv[t] - acc) * bt;
  }
  __syncthreads();
  HALO_PHASE(0, 4);
  const float d0 = dl[j0], d1 = dl[j0 + 1], d2 = dl[j0 + 2], d3 = dl[j0 + 3];
  float oo[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const float ki = sk[i0 + r], qi = sq[i0 + r];
    row[r].x += ki * d0;
    row[r].y += ki * d1;
    row[r].z += ki * d2;
    row[r].w += ki * d3;
    oo[0] += row[r].x * qi;
    oo[1] += row[r].y * qi;
    oo[2] += row[r].z * qi;
    oo[3] += row[r].w * qi;
    *reinterpret_cast<float4*>(St + static_cast<std::size_t>(i0 + r) * kD + j0) = row[r];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) red[rg][j0 + c] = oo[c];
  __syncthreads();
  HALO_PHASE(0, 5);
  // output: RMSNorm over the head's 128 values * w * sigmoid(z), quantized per 32 (waves 0 and 1)
  float o = 0.0f;
  if (t < kD) {
#pragma unroll
    for (int r = 0; r < 16; ++r) o += red[r][t];
    o *= 1.0f / sqrtf(static_cast<float>(kD));
  }
  const float so = halo::GroupSum(o * o);
  if (lane == 0 && wave < 2) part[wave] = so;
  __syncthreads();
  HALO_PHASE(0, 6);
  if (t < kD) {
    const float sc = 1.0f / sqrtf((part[0] + part[1]) / static_cast<float>(kD) + eps);
    const std::size_t off = static_cast<std::size_t>(s) * Dv + h * kD + t;
    const float v = o * sc * norm_w[t] * halo::Sigmoid(zg);
    const float amax = halo::GroupMax<32>(fabsf(v));
    const float scale = amax / 127.0f;
    oq[off] = static_cast<std::int8_t>(scale > 0.0f ? static_cast<int>(rintf(v / scale)) : 0);
    if (t % 32 == 0) os[off / 32] = scale;
  }
  HALO_PHASE(0, 7);
}
}  // namespace

extern "C" __global__ void __launch_bounds__(512) halo_gdn_step_q8(
    const float* qkv, const float* z, const float* ab, float* ring, const float* conv_w, const float* a,
    const float* dt, const float* norm_w, float* state, const std::uint32_t* nkv, std::int8_t* oq, float* os,
    std::uint32_t Hk, std::uint32_t Hv, std::uint32_t K, float eps) {
  GdnStepQ8<true>(qkv, z, ab, ring, conv_w, a, dt, norm_w, state, nkv, oq, os, Hk, Hv, K, eps);
}
extern "C" __global__ void __launch_bounds__(512) halo_gdn_step_q8_kn(
    const float* qkv, const float* z, const float* ab, float* ring, const float* conv_w, const float* a,
    const float* dt, const float* norm_w, float* state, const std::uint32_t* nkv, std::int8_t* oq, float* os,
    std::uint32_t Hk, std::uint32_t Hv, std::uint32_t K, float eps) {
  GdnStepQ8<false>(qkv, z, ab, ring, conv_w, a, dt, norm_w, state, nkv, oq, os, Hk, Hv, K, eps);
}
