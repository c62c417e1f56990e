// GQA decode attention over a paged KV cache shared by a ragged batch of sessions (gfx950, wave64).
//
// Reference semantics: ReferenceModel::Attention dense branch (src/model/reference.cpp:368-416, 492-527) and the
// GPU halo_attention_decode / halo_attention_select_b (src/kernels/core.hip:514-544, 898): per query head h (kv
// head h / G), o = softmax(q . K^T / sqrt(d)) V, then o *= sigmoid(gate).
//
// KV layout in HBM: pages of 16 tokens; K and V pools [page][kv_head][16][d] fp32; each session has a page table
// [max_pages]. Sessions of one batch share their first `prefix` tokens (identical page-table entries): a prefix
// chunk is read once and scored against the queries of every session (S * G query vectors), a suffix chunk only
// against its own session's G queries. Each (kv head, 32-token chunk) is one block producing flash partials
// (running max, sum, weighted V); halo_attn_decode_combine merges them per (session, head) and applies the gate.
#include <type_traits>

#include "common.h"

using halo::kWave;

namespace {
constexpr int kHd = 256;      // head dim
constexpr int kPage = 16;     // tokens per page
constexpr int kChunk = 32;    // tokens per block
constexpr int kMaxQ = 32;     // query vectors per block (sessions * G)
}  // namespace

using halo::H4;
using halo::H8;
using halo::Mfma3;
using halo::SplitHalves;
using halo::V4F;
namespace {
// Operand scales of the split-fp16 paths (powers of two, undone on the results): q and k (RMS-normalized) and V by 2^8,
// so values down to 2^-11 keep the full 22-bit split; a group (query row, K or V chunk) with a magnitude of 255.875 or
// more takes a smaller power of two instead (halo::SplitScale), keeping it in the fp16 range. The probabilities (<= 1)
// by 2^14.
constexpr float kSqk = 256.0f, kSvv = 256.0f, kSpp = 16384.0f;
constexpr float kLog2e = 1.4426950408889634f;
}  // namespace

// grid (Hkv * (prefix_chunks + S * suffix_chunks)), block 256.
//   q [S][Hq][256]; kpool, vpool [pages][Hkv][16][256]; pages [S][max_pages]; nkv [S] visible positions;
//   partial m, l [items][S * G], acc [items][S * G][256] (item = blockIdx.x).
// Prefix chunks cover tokens [32 c, 32 c + 32) < prefix of every session; suffix chunk c of session s covers
// [prefix + 32 c, ...) up to nkv[s]; positions at or past nkv[s] are masked, empty chunks record m = -inf.
//
// Every K and V load of the chunk (64 KB) is issued before any arithmetic, so a block keeps its whole chunk in
// flight. Scores: 16-lane row r of the block owns tokens r and r + 16, lane `sub` of the row dims
// {4 (16 u + sub) .. +4 : u < 4} (each load instruction reads 256 contiguous bytes per row); the 16 partial dots
// are summed with row DPP. V arrives as 16-byte loads and is staged through LDS (over the queries, once the scores
// are done). Weighted V: thread = one of the 256 dims, all 32 tokens in registers.
namespace {
// The partial kernel's body. kFused: q arrives as the raw q | gate projection qg [S][Hq][2 * 256] and is RMSNormed
// (wq) and rotated here at each session's position nkv[s] - 1, and the block whose chunk holds a session's newest
// position (the last suffix chunk) forms that position's K (RMSNorm wk, rotation) and V from kin / vin [S][Hkv][256],
// appends them to the pools and uses them for that row: the prologue launch before the attention disappears. The
// arithmetic is halo_attn_prep_decode's (halo::NormRopeHead), so q, K and V carry the same bits.
template <bool kFused, int kQW = 1, bool kMma = false>
__device__ __forceinline__ void AttnDecodePartial(
    const float* __restrict__ q, const float* __restrict__ kin, const float* __restrict__ vin,
    const float* __restrict__ wq, const float* __restrict__ wk, float* __restrict__ kpool, float* __restrict__ vpool,
    const std::uint32_t* __restrict__ pages, const std::uint32_t* __restrict__ nkv, float* __restrict__ pm,
    float* __restrict__ pl, float* __restrict__ pacc, std::uint32_t S, std::uint32_t Hq, std::uint32_t Hkv,
    std::uint32_t prefix, std::uint32_t max_pages, std::uint32_t prefix_chunks, std::uint32_t suffix_chunks,
    std::uint32_t rot, float theta, float eps) {
  // 32.5 KB: the queries, then the K chunk as halves, then the V chunk as halves (39 KB in all: four blocks per CU);
  // query rows padded by 16 bytes so the 16 rows of a matrix-core operand read fall on different banks
  __shared__ __attribute__((aligned(16))) float qs[kMaxQ][kHd + 4];
  __shared__ __attribute__((aligned(16))) float sc[kMaxQ][kChunk + 4];  // rows 16-byte aligned: vector reads
  static_assert(kChunk == 32 && kPage == 16, "two pages per chunk, two tokens per 16-lane row");
  const std::uint32_t G = Hq / Hkv, x = blockIdx.x, kvh = x % Hkv, c = x / Hkv;
  HALO_PHASE(1, 0);
  const std::uint32_t t = threadIdx.x, wave = t / kWave, lane = t % kWave;
  const bool is_prefix = c < prefix_chunks;
  const std::uint32_t sess = is_prefix ? 0 : (c - prefix_chunks) / suffix_chunks;
  const std::uint32_t start = is_prefix ? c * kChunk : prefix + ((c - prefix_chunks) % suffix_chunks) * kChunk;
  const std::uint32_t nq = is_prefix ? S * G : G;
  const std::uint32_t limit = is_prefix ? prefix : nkv[sess];
  const std::uint32_t slots = S * G;
  float* m_out = pm + static_cast<std::size_t>(x) * slots;
  float* l_out = pl + static_cast<std::size_t>(x) * slots;
  float* a_out = pacc + static_cast<std::size_t>(x) * slots * kHd;
  if (start >= limit) {
    if (t < nq) {
      const std::uint32_t slot = is_prefix ? t : sess * G + t;
      m_out[slot] = -INFINITY;
      l_out[slot] = 0.0f;
    }
    return;
  }
  // the chunk's two pages (a position past the visible range reads the last visible one; it is masked)
  const std::uint32_t* pt = pages + static_cast<std::size_t>(sess) * max_pages;
  const std::uint32_t last = limit - 1;
  const std::uint32_t pg0 = pt[min(start, last) / kPage], pg1 = pt[min(start + kPage, last) / kPage];
  auto row_of = [&](const float* pool, std::uint32_t j) {  // token start + j, clamped to the visible range
    const std::uint32_t tok = min(start + j, last);
    const std::uint32_t pg = (tok - start) < kPage ? pg0 : pg1;
    return pool + ((static_cast<std::size_t>(pg) * Hkv + kvh) * kPage + tok % kPage) * kHd;
  };
  const std::uint32_t sub = t % 16, r = t / 16;
  // Fused prologue inputs, all issued before the chunk's K / V (a load issued after them could only be waited for
  // behind them): this wave's queries (kQW of them, slots past nq reload the last), their sessions' positions,
  // the norm weights and the newest position's k / v (loaded by every block, used by the one that holds it).
  static_assert(kQW >= 1 && kQW <= kMaxQ / 4, "queries per wave");
  float xq[kQW][4], wqv[4], wkv[4], xk[4], xv[4];
  std::uint32_t qpos[kQW];
  const bool owner = kFused && !is_prefix && last - start < static_cast<std::uint32_t>(kChunk);
  if constexpr (kFused) {
#pragma unroll
    for (int m = 0; m < kQW; ++m) {
      const std::uint32_t qi = min(wave + 4u * m, nq - 1);
      const std::uint32_t s = is_prefix ? qi / G : sess, g = is_prefix ? qi % G : qi;
      const float* src = q + (static_cast<std::size_t>(s) * Hq + kvh * G + g) * 2 * kHd;
#pragma unroll
      for (int i = 0; i < 4; ++i) xq[m][i] = src[lane + 64 * i];
      qpos[m] = nkv[s] - 1;
    }
    const std::size_t kv_src = (static_cast<std::size_t>(sess) * Hkv + kvh) * kHd;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      wqv[i] = wq[lane + 64 * i];
      wkv[i] = wk[lane + 64 * i];
      xk[i] = kin[kv_src + lane + 64 * i];
      xv[i] = vin[kv_src + lane + 64 * i];
    }
  }
  float4 kf[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float4* kr = reinterpret_cast<const float4*>(row_of(kpool, r + 16 * h));
#pragma unroll
    for (int u = 0; u < 4; ++u) kf[h][u] = kr[16 * u + sub];
  }
  // The V chunk (fused prologue: issued only after the query prologue; a wave's loads issue in order and stall while
  // the stream is queued, so V issued with K would hold that prologue back, and V is needed only after the scores)
  float4 vq[2][4];
  const std::uint32_t vdg = t % 64, vkg = t / 64;
  float4 vreg[8];
  auto issue_v = [&]() {
  if constexpr (!kMma) {
  // V as 16-byte loads of the two pages (each page's 16 rows are 16 KB contiguous; thread t takes float4 t of every
  // 4 KB part: row 4 part + t / 64, dims 4 (t % 64) ..): 4-byte loads of a column would take 32 instructions per
  // thread and run the chunk's V stream at half the rate. Staged through LDS below, so the weighted sum still reads
  // one dim of every row.
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float4* vp = reinterpret_cast<const float4*>(vpool + (static_cast<std::size_t>(h ? pg1 : pg0) * Hkv + kvh) *
                                                                   kPage * kHd);
#pragma unroll
    for (int u = 0; u < 4; ++u) vq[h][u] = vp[u * 256 + t];
  }
  } else {
  // V: thread t takes keys 8 (t / 64) + e (e < 8, one page) at dims 4 (t % 64) ..: each load instruction reads one
  // whole 1 KB row; staged transposed below (positions past the visible range are zeroed there)
  {
    const float* vp = vpool + ((static_cast<std::size_t>(vkg < 2 ? pg0 : pg1) * Hkv + kvh) * kPage) * kHd + 4 * vdg;
#pragma unroll
    for (int e = 0; e < 8; ++e) vreg[e] = *reinterpret_cast<const float4*>(vp + ((8 * vkg + e) % kPage) * kHd);
  }
  }
  };
  if constexpr (!kFused && !kMma) issue_v();
  // queries of this kv head: slot i = session * G + g (prefix) or g (suffix)
  __shared__ __attribute__((aligned(16))) float knew[kFused ? 2 : 1][kFused ? kHd : 4];
  if constexpr (kFused) {
    // wave w prepares queries w, w + 4, ... (the angles once per position). The precise powf / cosf / sinf of a position cost
    // more than the norms: two to four sessions' angles are formed by one wave each and shared through LDS (the scores'
    // space): 4 sessions at 8576 positions 31.5 -> 30.8 us per layer.
    std::uint32_t cur = 0xFFFFFFFFu;
    halo::RopeCS cs{};
    float out[4];
    float4* shared_cs = reinterpret_cast<float4*>(&sc[0][0]);
    const bool share = kMma && is_prefix && S > 1 && S <= 4;
    static_assert(sizeof(sc) >= 4 * kWave * sizeof(float4));
    if (share) {
      if (wave < S) {
        cs = halo::RopeAngles(nkv[wave] - 1, rot, theta);
        shared_cs[wave * kWave + lane] = make_float4(cs.c[0], cs.c[1], cs.s[0], cs.s[1]);
      }
      halo::LdsSync();
    }
#pragma unroll
    for (int m = 0; m < kQW; ++m) {
      const std::uint32_t qi = wave + 4u * m;
      if (qi >= nq) break;
      if (share) {
        const float4 v = shared_cs[qi / G * kWave + lane];
        cs.c[0] = v.x, cs.c[1] = v.y, cs.s[0] = v.z, cs.s[1] = v.w;
      } else if (qpos[m] != cur) {
        cur = qpos[m];
        cs = halo::RopeAngles(cur, rot, theta);
      }
      halo::NormRopeHead(xq[m], wqv, cs, rot, eps, out);
#pragma unroll
      for (int i = 0; i < 4; ++i) qs[qi][lane + 64 * i] = out[i];
    }
    if (owner && wave == 3) {
      // the newest position's K and V: to LDS for this block's scores and weighted sum, and to the pools (its page
      // is one of the chunk's two)
      if (cur != last) cs = halo::RopeAngles(last, rot, theta);
      halo::NormRopeHead(xk, wkv, cs, rot, eps, out);
      const std::size_t dst =
          ((static_cast<std::size_t>(last - start < kPage ? pg0 : pg1) * Hkv + kvh) * kPage + last % kPage) * kHd;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        knew[0][lane + 64 * i] = out[i];
        knew[1][lane + 64 * i] = xv[i];
        kpool[dst + lane + 64 * i] = out[i];
        vpool[dst + lane + 64 * i] = xv[i];
      }
    }
  } else {
    for (std::uint32_t i = t; i < nq * (kHd / 4); i += blockDim.x) {
      const std::uint32_t qi = i / (kHd / 4), d4 = i % (kHd / 4);
      const std::uint32_t s = is_prefix ? qi / G : sess, g = is_prefix ? qi % G : qi;
      const float4 v = reinterpret_cast<const float4*>(q + (static_cast<std::size_t>(s) * Hq + kvh * G + g) * kHd)[d4];
      reinterpret_cast<float4*>(&qs[qi][0])[d4] = v;
    }
  }
  if constexpr (kFused && !kMma) issue_v();
  if constexpr (!kMma) {
  __syncthreads();
  HALO_PHASE(1, 1);
  if (owner) {
    // the newest row's K from LDS in place of the pool's (not yet written when the loads were issued)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (start + r + 16 * h == last)
#pragma unroll
        for (int u = 0; u < 4; ++u) kf[h][u] = reinterpret_cast<const float4*>(&knew[0][0])[16 * u + sub];
  }
  const float scale = 1.0f / sqrtf(static_cast<float>(kHd));
  const bool live0 = start + r < limit, live1 = start + r + 16 < limit;
  // queries in groups of 8, the group's dot products and row reductions interleaved (independent chains; each
  // query's arithmetic is the same as one at a time)
  constexpr int kQG = 8;
  for (std::uint32_t i0 = 0; i0 < nq; i0 += kQG) {
    float s0[kQG], s1[kQG];
#pragma unroll
    for (int k = 0; k < kQG; ++k) {
      const float4* qv = reinterpret_cast<const float4*>(&qs[min(i0 + k, nq - 1)][0]);
      s0[k] = 0.0f;
      s1[k] = 0.0f;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4 b = qv[16 * u + sub];
        s0[k] += kf[0][u].x * b.x + kf[0][u].y * b.y + kf[0][u].z * b.z + kf[0][u].w * b.w;
        s1[k] += kf[1][u].x * b.x + kf[1][u].y * b.y + kf[1][u].z * b.z + kf[1][u].w * b.w;
      }
    }
#pragma unroll
    for (int k = 0; k < kQG; ++k) {
      s0[k] = halo::GroupSum<16>(s0[k]);
      s1[k] = halo::GroupSum<16>(s1[k]);
    }
    if (sub == 0)
#pragma unroll
      for (int k = 0; k < kQG; ++k)
        if (i0 + k < nq) {
          sc[i0 + k][r] = live0 ? s0[k] * scale : -INFINITY;
          sc[i0 + k][r + 16] = live1 ? s1[k] * scale : -INFINITY;
        }
  }
  __syncthreads();  // the scores are in sc and qs is free: the V rows go there (rows past the visible range as 0)
  HALO_PHASE(1, 2);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const std::uint32_t j = 16 * h + 4 * u + t / 64;
      float4 v = start + j < limit ? vq[h][u] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (owner && start + j == last) v = reinterpret_cast<const float4*>(&knew[1][0])[t % 64];
      reinterpret_cast<float4*>(&qs[j][0])[t % 64] = v;
    }
  // softmax over the chunk per query: wave w takes queries w, w + 4, ...; lanes 0..31 are the tokens
  for (std::uint32_t i = wave; i < nq; i += 4) {
    const float s = lane < kChunk ? sc[i][lane] : -INFINITY;
    const float m = halo::GroupMax(s);
    const float p = s == -INFINITY ? 0.0f : expf(s - m);
    const float l = halo::GroupSum(p);
    if (lane < kChunk) sc[i][lane] = p;
    if (lane == 0) {
      const std::uint32_t slot = is_prefix ? i : sess * G + i;
      m_out[slot] = m;
      l_out[slot] = l;
    }
  }
  __syncthreads();
  HALO_PHASE(1, 3);
  // weighted V, 8 queries' sums interleaved (each still adds its tokens in order j = 0 .. 31); V and the weights
  // are read from LDS four tokens at a time
  for (std::uint32_t i0 = 0; i0 < nq; i0 += kQG) {
    float acc[kQG];
#pragma unroll
    for (int k = 0; k < kQG; ++k) acc[k] = 0.0f;
#pragma unroll 2
    for (int j4 = 0; j4 < kChunk; j4 += 4) {
      const float v0 = qs[j4][t], v1 = qs[j4 + 1][t], v2 = qs[j4 + 2][t], v3 = qs[j4 + 3][t];
#pragma unroll
      for (int k = 0; k < kQG; ++k) {
        const float4 p4 = *reinterpret_cast<const float4*>(&sc[min(i0 + k, nq - 1)][j4]);
        acc[k] += p4.x * v0;
        acc[k] += p4.y * v1;
        acc[k] += p4.z * v2;
        acc[k] += p4.w * v3;
      }
    }
#pragma unroll
    for (int k = 0; k < kQG; ++k)
      if (i0 + k < nq) {
        const std::uint32_t slot = is_prefix ? i0 + k : sess * G + i0 + k;
        a_out[static_cast<std::size_t>(slot) * kHd + t] = acc[k];
      }
  }
  HALO_PHASE(1, 4);
  } else {
  __syncthreads();
  HALO_PHASE(1, 1);
  // Matrix-core tiles: nqt tiles of 16 query rows (rows past nq repeat the last query and are never stored); the
  // scores are tiles (query tile w / 2, key tile w % 2) of waves w < 2 nqt; each query row's products, softmax and
  // weighted sum depend only on that row, so a query gets the same bits whichever block and batch it is scored in.
  const std::uint32_t nqt = (nq + 15) / 16, kq = lane / 16, lr = lane % 16;
  const std::uint32_t qt = wave / 2, kt = wave % 2;
  const bool score_wave = qt < nqt;
  // Operand scales (powers of two): per query row, and per block for the K and the V chunk (halo::SplitScale:
  // kSqk / kSvv unless the group's largest magnitude would overflow the fp16 range)
  __shared__ float qsc[kMaxQ], kvmax[2][4];
  H8 qh[kHd / 32], ql[kHd / 32];
  if (score_wave) {
    // two passes over the query row in LDS (its magnitude, then the split), so the row is never held in registers
    // next to its halves (that took the kernel to 180 VGPRs: two blocks per CU instead of three)
    const float* qr = &qs[min(16 * qt + lr, nq - 1)][0];
    float amax = 0.0f;
#pragma unroll
    for (int c = 0; c < kHd / 32; ++c) {
      const float4 a0 = *reinterpret_cast<const float4*>(qr + 32 * c + 8 * kq);
      const float4 a1 = *reinterpret_cast<const float4*>(qr + 32 * c + 8 * kq + 4);
      amax = fmaxf(amax, fmaxf(fmaxf(fmaxf(fabsf(a0.x), fabsf(a0.y)), fmaxf(fabsf(a0.z), fabsf(a0.w))),
                               fmaxf(fmaxf(fabsf(a1.x), fabsf(a1.y)), fmaxf(fabsf(a1.z), fabsf(a1.w)))));
    }
    amax = fmaxf(amax, __shfl_xor(amax, 16));
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    const float sq = halo::SplitScale(amax, kSqk);
#pragma unroll
    for (int c = 0; c < kHd / 32; ++c) {
      const float4 a0 = *reinterpret_cast<const float4*>(qr + 32 * c + 8 * kq);
      const float4 a1 = *reinterpret_cast<const float4*>(qr + 32 * c + 8 * kq + 4);
      const float x[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
      SplitHalves(x, qh[c], ql[c], sq);
    }
    if (kq == 0) qsc[16 * qt + lr] = sq;
  }
  {  // the block's K and V magnitudes over the visible rows (rows past them repeat the pool's row `last`, which for
     // the owner block is not yet written: the newest row comes from LDS, and the masked rows' scores are dropped)
    float ka = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const std::uint32_t j = r + 16 * h;
      const bool fresh = owner && start + j == last;
      if (start + j < limit)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float4 kv = fresh ? *reinterpret_cast<const float4*>(&knew[0][64 * u + 4 * sub]) : kf[h][u];
          ka = fmaxf(ka, fmaxf(fmaxf(fabsf(kv.x), fabsf(kv.y)), fmaxf(fabsf(kv.z), fabsf(kv.w))));
        }
    }
    ka = halo::GroupMax(ka);
    if (lane == 0) kvmax[0][wave] = ka;
  }
  __syncthreads();  // qs is free: the K chunk goes there as halves
  const float sk = halo::SplitScale(fmaxf(fmaxf(kvmax[0][0], kvmax[0][1]), fmaxf(kvmax[0][2], kvmax[0][3])), kSqk);
  // K halves kh / kl [32 keys][256]: 16-byte chunk c of key row j at c ^ (j & 15) (the 16 lanes of an operand read
  // take 16 different bank groups); the newest row (owner) from LDS, not yet in the pool when it was loaded
  _Float16* kh = reinterpret_cast<_Float16*>(&qs[0][0]);
  _Float16* kl = kh + kChunk * kHd;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const std::uint32_t j = r + 16 * h;
    const bool fresh = owner && start + j == last;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const std::uint32_t dim = 64 * u + 4 * sub;
      const float4 kv = fresh ? *reinterpret_cast<const float4*>(&knew[0][dim]) : kf[h][u];
      const float x[4] = {kv.x, kv.y, kv.z, kv.w};
      const std::uint32_t off = j * kHd + 8 * ((dim / 8) ^ (j & 15)) + dim % 8;
      H4 hi, lo;
      halo::SplitHalves4(x, hi, lo, sk);
      *reinterpret_cast<H4*>(&kh[off]) = hi;
      *reinterpret_cast<H4*>(&kl[off]) = lo;
    }
  }
  __syncthreads();
  HALO_PHASE(1, 2);
  // the V chunk issued only now that the K fragments are in LDS (its 32 destination registers and the K fragments
  // are never live together: held together they spilled, and the spill's reloads waited for V before the K phase)
  issue_v();
  const float scale = 1.0f / sqrtf(static_cast<float>(kHd));
  if (score_wave) {
    V4F c4 = {0.0f, 0.0f, 0.0f, 0.0f};
    const std::uint32_t key = 16 * kt + lr;
#pragma unroll
    for (int c = 0; c < kHd / 32; ++c) {
      const std::uint32_t off = key * kHd + 8 * ((4 * c + kq) ^ (key & 15));
      c4 = Mfma3(qh[c], ql[c], *reinterpret_cast<const H8*>(&kh[off]), *reinterpret_cast<const H8*>(&kl[off]), c4);
    }
    // C tile: lane (key lr, kq) holds rows 16 qt + 4 kq + i
    const bool live = start + key < limit;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const std::uint32_t qi = 16 * qt + 4 * kq + i;
      if (qi < nq) sc[qi][key] = live ? c4[i] * (scale / (qsc[qi] * sk)) : -INFINITY;
    }
  }
  {  // the V chunk's magnitude over the visible rows (the newest row from LDS), only now that the scores are done
    float va = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const std::uint32_t j = 8 * vkg + e;
      float4 vv = vreg[e];
      if (owner && start + j == last) vv = *reinterpret_cast<const float4*>(&knew[kFused ? 1 : 0][4 * vdg]);
      if (start + j < limit)
        va = fmaxf(va, fmaxf(fmaxf(fabsf(vv.x), fabsf(vv.y)), fmaxf(fabsf(vv.z), fabsf(vv.w))));
    }
    va = halo::GroupMax(va);
    if (lane == 0) kvmax[1][wave] = va;
  }
  __syncthreads();
  HALO_PHASE(1, 3);
  const float sv = halo::SplitScale(fmaxf(fmaxf(kvmax[1][0], kvmax[1][1]), fmaxf(kvmax[1][2], kvmax[1][3])), kSvv);
  // the K chunk is done with: the V chunk goes to the same LDS as halves transposed, vh / vl [256 dims][32 keys]
  // (chunk c of 8 keys of a dim row at c ^ ((dim >> 2) & 3))
  _Float16* vh = kh;
  _Float16* vl = kh + kHd * kChunk;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const std::uint32_t dim = 4 * vdg + d;
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const std::uint32_t j = 8 * vkg + e;
      const float4 vv = vreg[e];
      float val = d == 0 ? vv.x : d == 1 ? vv.y : d == 2 ? vv.z : vv.w;
      if (owner && start + j == last) val = knew[kFused ? 1 : 0][dim];
      x[e] = start + j < limit ? val : 0.0f;
    }
    H8 hi, lo;
    SplitHalves(x, hi, lo, sv);
    const std::uint32_t off = dim * kChunk + 8 * (vkg ^ ((dim >> 2) & 3));
    *reinterpret_cast<H8*>(&vh[off]) = hi;
    *reinterpret_cast<H8*>(&vl[off]) = lo;
  }
  // softmax over the chunk per query: wave w takes queries w, w + 4, ...; lanes 0..31 are the tokens
  for (std::uint32_t i = wave; i < nq; i += 4) {
    const float s = lane < kChunk ? sc[i][lane] : -INFINITY;
    const float m = halo::GroupMax(s);
    const float p = s == -INFINITY ? 0.0f : expf(s - m);
    const float l = halo::GroupSum(p);
    if (lane < kChunk) sc[i][lane] = p;
    if (lane == 0) {
      const std::uint32_t slot = is_prefix ? i : sess * G + i;
      m_out[slot] = m;
      l_out[slot] = l;
    }
  }
  __syncthreads();
  HALO_PHASE(1, 5);
  // weighted V: output tiles (query tile, 16-dim tile); two query tiles: wave w takes tile w / 2, dim tiles
  // 8 (w % 2) ..; one: dim tiles 4 w .. + 3
  const std::uint32_t pqt = nqt == 2 ? wave / 2 : 0, ndt = nqt == 2 ? 8 : 4, dt0 = nqt == 2 ? 8 * (wave % 2) : 4 * wave;
  H8 pah, pal;
  {
    const float* pr = &sc[min(16 * pqt + lr, nq - 1)][8 * kq];
    const float4 a0 = *reinterpret_cast<const float4*>(pr), a1 = *reinterpret_cast<const float4*>(pr + 4);
    const float x[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
    SplitHalves(x, pah, pal, kSpp);
  }
#pragma unroll
  for (std::uint32_t dc = 0; dc < 8; ++dc) {
    if (dc >= ndt) break;
    const std::uint32_t dim = 16 * (dt0 + dc) + lr;
    const std::uint32_t off = dim * kChunk + 8 * (kq ^ ((dim >> 2) & 3));
    const V4F acc = Mfma3(pah, pal, *reinterpret_cast<const H8*>(&vh[off]), *reinterpret_cast<const H8*>(&vl[off]),
                          V4F{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const std::uint32_t qi = 16 * pqt + 4 * kq + i;
      if (qi < nq) {
        const std::uint32_t slot = is_prefix ? qi : sess * G + qi;
        a_out[static_cast<std::size_t>(slot) * kHd + dim] = acc[i] * (1.0f / (kSpp * sv));
      }
    }
  }
  HALO_PHASE(1, 4);
  }
}
}  // namespace

// (the matrix-core forms ask for 3 waves per SIMD, i.e. at most 168 VGPRs: three 4-wave blocks per CU; at 180 the
// 608 blocks of the 4-session C4 step ran in two rounds)
#define HALO_ATTN_PARTIAL(NAME, MMA)                                                                                   \
  extern "C" __global__ void __launch_bounds__(256, MMA ? 3 : 1) NAME(                                                \
      const float* __restrict__ q, const float* __restrict__ kpool, const float* __restrict__ vpool,                 \
      const std::uint32_t* __restrict__ pages, const std::uint32_t* __restrict__ nkv, float* __restrict__ pm,        \
      float* __restrict__ pl, float* __restrict__ pacc, std::uint32_t S, std::uint32_t Hq, std::uint32_t Hkv,      \
      std::uint32_t prefix, std::uint32_t max_pages, std::uint32_t prefix_chunks, std::uint32_t suffix_chunks) {    \
    AttnDecodePartial<false, 1, MMA>(q, nullptr, nullptr, nullptr, nullptr, const_cast<float*>(kpool),             \
                                     const_cast<float*>(vpool), pages, nkv, pm, pl, pacc, S, Hq, Hkv, prefix,      \
                                     max_pages, prefix_chunks, suffix_chunks, 0, 0.0f, 0.0f);                     \
  }
// fp32 VALU dot products (one session: eight queries per kv head, latency-bound) / split-fp16 matrix cores (several
// sessions: up to 32 queries per block score a shared-prefix chunk)
HALO_ATTN_PARTIAL(halo_attn_decode_partial, false)
HALO_ATTN_PARTIAL(halo_attn_decode_partial_mma, true)
#undef HALO_ATTN_PARTIAL

// The partial launch with the attention prologue folded in (see AttnDecodePartial<true>): qg [S][Hq][2 * 256],
// kin, vin [S][Hkv][256], wq, wk [256]; rot <= 128. Every session's newest position nkv[s] - 1 must lie past the
// shared prefix (it is in that session's last suffix chunk). Same grid and partial outputs as
// halo_attn_decode_partial; the gate for the combine is the second half of each qg head.
// _qk: up to 32 query vectors per block (S * Hq / Hkv <= 32), split-fp16 matrix cores; _qk2: up to 8 (two per
// wave), fp32 VALU.
#define HALO_ATTN_PARTIAL_QK(NAME, QW, MMA)                                                                           \
  extern "C" __global__ void __launch_bounds__(256, MMA ? 3 : 1) NAME(                                          \
      const float* __restrict__ qg, const float* __restrict__ kin, const float* __restrict__ vin,               \
      const float* __restrict__ wq, const float* __restrict__ wk, float* __restrict__ kpool,                    \
      float* __restrict__ vpool, const std::uint32_t* __restrict__ pages, const std::uint32_t* __restrict__ nkv, \
      float* __restrict__ pm, float* __restrict__ pl, float* __restrict__ pacc, std::uint32_t S, std::uint32_t Hq, \
      std::uint32_t Hkv, std::uint32_t prefix, std::uint32_t max_pages, std::uint32_t prefix_chunks,            \
      std::uint32_t suffix_chunks, std::uint32_t rot, float theta, float eps) {                                 \
    AttnDecodePartial<true, QW, MMA>(qg, kin, vin, wq, wk, kpool, vpool, pages, nkv, pm, pl, pacc, S, Hq, Hkv, prefix,  \
                                max_pages, prefix_chunks, suffix_chunks, rot, theta, eps);                       \
  }
HALO_ATTN_PARTIAL_QK(halo_attn_decode_partial_qk, 8, true)
HALO_ATTN_PARTIAL_QK(halo_attn_decode_partial_qk2, 2, false)
#undef HALO_ATTN_PARTIAL_QK


// grid (S * Hq * NS), block 256: block (s, h, slice) merges the partials of session s, head h over its prefix and
// suffix chunks (log-sum-exp) for the slice's 256 / NS dims: o = acc / l, then o *= sigmoid(gate) when gate is
// non-null. o, gate [S][Hq][256] (o may be null); with oq non-null also the Q8 quantization of o (oq [S][Hq * 256],
// os [S][Hq * 8]). At most 1024 items. Thread: float4 lane f of the slice, item group t / (lanes per slice), eight
// loads in flight. NS = 8 doubles the blocks of small batches (more loads in flight over the chip).
namespace {
template <int NS, int kGS = 1>
__device__ __forceinline__ void AttnDecodeCombine(
    const float* __restrict__ pm, const float* __restrict__ pl, const float* __restrict__ pacc,
    const float* __restrict__ gate, float* __restrict__ o, std::int8_t* __restrict__ oq, float* __restrict__ os,
    std::uint32_t S, std::uint32_t Hq, std::uint32_t Hkv, std::uint32_t prefix_chunks,
    std::uint32_t suffix_chunks) {
  constexpr std::uint32_t kW = kHd / NS, kF = kW / 4, kG = 256 / kF;  // slice dims, float4 lanes, item groups
  __shared__ float wts[1024];
  __shared__ float red[4], redl[4];
  __shared__ float4 part[kG][kF];
  const std::uint32_t quarter = blockIdx.x % NS, sh = blockIdx.x / NS;
  const std::uint32_t G = Hq / Hkv, s = sh / Hq, h = sh % Hq, kvh = h / G, g = h % G;
  const std::uint32_t slot = s * G + g, slots = S * G, t = threadIdx.x;
  const std::uint32_t n = min(prefix_chunks + suffix_chunks, 1024u);
  auto item = [&](std::uint32_t i) -> std::size_t {
    const std::uint32_t c = i < prefix_chunks ? i : prefix_chunks + s * suffix_chunks + (i - prefix_chunks);
    return static_cast<std::size_t>(c) * Hkv + kvh;
  };
  // The loads that do not depend on each other are issued together (unconditionally, from clamped items, then
  // selected): the items' m and l for n <= 512 (two each per thread), this thread's first group of kU partial sums
  // and its gate value; further items (n > 512, groups past the first) are loaded where they are used. The
  // arithmetic runs in the order it always had.
  const std::uint32_t f = t % kF, ig = t / kF;
  constexpr int kU = 8;
  float mv[2], lv[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const std::uint32_t i = min(t + 256u * j, n - 1);
    mv[j] = pm[item(i) * slots + slot];
    lv[j] = pl[item(i) * slots + slot];
  }
  float4 a0[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const std::uint32_t i = min(ig + kG * u, n - 1);
    a0[u] = reinterpret_cast<const float4*>(pacc + (item(i) * slots + slot) * kHd)[quarter * kF + f];
  }
  const float gv = *(gate != nullptr ? gate + (static_cast<std::size_t>(s) * Hq + h) * kGS * kHd + quarter * kW +
                                           min(t, kW - 1)
                                     : pl);  // (any valid address without a gate; unused then)
  const std::size_t off = (static_cast<std::size_t>(s) * Hq + h) * kHd + quarter * kW + min(t, kW - 1);
  float M = -INFINITY;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const std::uint32_t i = t + 256u * j;
    if (i < n) {
      wts[i] = mv[j];
      M = fmaxf(M, mv[j]);
    }
  }
  for (std::uint32_t i = t + 512; i < n; i += blockDim.x) {
    const float m = pm[item(i) * slots + slot];
    wts[i] = m;
    M = fmaxf(M, m);
  }
  M = halo::GroupMax(M);
  if (t % kWave == 0) red[t / kWave] = M;
  __syncthreads();
  M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float L = 0.0f;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const std::uint32_t i = t + 256u * j;
    if (i < n) {
      const float m = mv[j];
      const float w = m == -INFINITY ? 0.0f : expf(m - M);
      wts[i] = w;
      L += w * lv[j];
    }
  }
  for (std::uint32_t i = t + 512; i < n; i += blockDim.x) {
    const float m = wts[i];
    const float w = m == -INFINITY ? 0.0f : expf(m - M);
    wts[i] = w;
    L += w * pl[item(i) * slots + slot];
  }
  L = halo::GroupSum(L);
  if (t % kWave == 0) redl[t / kWave] = L;  // (its own array: red may still be read for M)
  __syncthreads();
  L = (redl[0] + redl[1]) + (redl[2] + redl[3]);
  float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (std::uint32_t i0 = ig, r = 0; i0 < n; i0 += kG * kU, ++r) {
    float4 b[kU];
    float w[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const std::uint32_t i = i0 + kG * u;
      const float wi = wts[min(i, n - 1)];
      w[u] = i < n ? wi : 0.0f;
      // past the preloaded group: load here (clamped item); an empty chunk's partial is never written
      const float4 av = r == 0 ? a0[u]
                               : reinterpret_cast<const float4*>(pacc + (item(min(i, n - 1)) * slots + slot) *
                                                                           kHd)[quarter * kF + f];
      b[u] = w[u] == 0.0f ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : av;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      acc.x += w[u] * b[u].x;
      acc.y += w[u] * b[u].y;
      acc.z += w[u] * b[u].z;
      acc.w += w[u] * b[u].w;
    }
  }
  part[ig][f] = acc;
  __syncthreads();
  if (t >= kW) return;
  // lane = dim of the slice
  float sum = 0.0f;
#pragma unroll
  for (std::uint32_t k = 0; k < kG; ++k) sum += reinterpret_cast<const float*>(&part[k][0])[t];
  float r = sum / L;
  if (gate != nullptr) r *= halo::Sigmoid(gv);
  if (o != nullptr) o[off] = r;
  if (oq != nullptr) {
    // the row's Q8 quantization for the output projection: 32-value blocks are half waves
    const float amax = halo::GroupMax<32>(fabsf(r));
    const float scale = amax / 127.0f;
    oq[off] = static_cast<std::int8_t>(scale > 0.0f ? static_cast<int>(rintf(r / scale)) : 0);
    if (t % 32 == 0) os[off / 32] = scale;
  }
}
}  // namespace

// _qg: gate rows with a head stride of 2 * 256 (the gate halves of the q | gate projection, gate = qg + 256).
#define HALO_ATTN_COMBINE(NAME, NS, GS)                                                                          \
  extern "C" __global__ void __launch_bounds__(256) NAME(                                                       \
      const float* __restrict__ pm, const float* __restrict__ pl, const float* __restrict__ pacc,               \
      const float* __restrict__ gate, float* __restrict__ o, std::int8_t* __restrict__ oq, float* __restrict__ os, \
      std::uint32_t S, std::uint32_t Hq, std::uint32_t Hkv, std::uint32_t prefix_chunks,                         \
      std::uint32_t suffix_chunks) {                                                                             \
    AttnDecodeCombine<NS, GS>(pm, pl, pacc, gate, o, oq, os, S, Hq, Hkv, prefix_chunks, suffix_chunks);         \
  }
HALO_ATTN_COMBINE(halo_attn_decode_combine, 4, 1)
HALO_ATTN_COMBINE(halo_attn_decode_combine8, 8, 1)
HALO_ATTN_COMBINE(halo_attn_decode_combine_qg, 4, 2)
HALO_ATTN_COMBINE(halo_attn_decode_combine8_qg, 8, 2)
#undef HALO_ATTN_COMBINE

// Appends one token's K and V per session at position nkv[s] - 1: k, v [S][Hkv][256] -> pools via page tables.
// grid (S * Hkv), block 64 (a float4 per lane).
extern "C" __global__ void __launch_bounds__(64)
    halo_kv_append(const float* __restrict__ k, const float* __restrict__ v, float* __restrict__ kpool,
                   float* __restrict__ vpool, const std::uint32_t* __restrict__ pages,
                   const std::uint32_t* __restrict__ nkv, std::uint32_t Hkv, std::uint32_t max_pages) {
  const std::uint32_t s = blockIdx.x / Hkv, kvh = blockIdx.x % Hkv, pos = nkv[s] - 1;
  const std::uint32_t pg = pages[static_cast<std::size_t>(s) * max_pages + pos / kPage];
  const std::size_t dst = ((static_cast<std::size_t>(pg) * Hkv + kvh) * kPage + pos % kPage) * kHd;
  const std::size_t src = (static_cast<std::size_t>(s) * Hkv + kvh) * kHd;
  reinterpret_cast<float4*>(kpool + dst)[threadIdx.x] = reinterpret_cast<const float4*>(k + src)[threadIdx.x];
  reinterpret_cast<float4*>(vpool + dst)[threadIdx.x] = reinterpret_cast<const float4*>(v + src)[threadIdx.x];
}

// ---- causal GQA attention for a ragged batch of prefill tokens (split-fp16 MFMA) -----------------------------------
// Reference semantics: ReferenceModel::Attention (src/model/reference.cpp:368-416, 492-527) for every token of a
// prompt: softmax(q . K[0..p]^T / sqrt(d)) V[0..p] * sigmoid(gate), K / V already appended at the tokens' positions.
// tiles [n][4] = {first token index in the batch, tokens (<= 16), session, position of the first token}; a tile's
// tokens are consecutive positions of one session. Output o (fp32, may be null) and its Q8 quantization oq / os (may
// be null), per token [Hq * 256], after o /= l and o *= sigmoid(gate). q, gate [T][Hq][256]. G = Hq / Hkv = 8.
//
// Every fp32 operand x enters as a pair of halves, hi = fp16(x) and lo = fp16(x - hi) (|x - hi - lo| <= 2^-22 |x|
// for normal values), and each product is formed as hi * hi + hi * lo + lo * hi on v_mfma_f32_32x32x16_f16
// (products of halves are exact in the fp32 accumulator; the dropped lo * lo term is below 2^-22 of the product).
// q, K and V are scaled by 2^8 and the probabilities by 2^14 before the split (kSqk, kSvv, kSpp); a query row, K chunk
// or V chunk whose magnitude would overflow fp16 at 2^8 takes a smaller power of two (halo::SplitScale), so any finite
// operand range is accepted; V keeps the smallest scale from there on.
//
// Block (tile, kv head): 128 queries = 16 tokens x 8 q heads; wave w the tokens 4 w .. 4 w + 3, query n = 8 (token -
// 4 w) + head. Both products run transposed, so that a query is a column and stays in one lane pair (n, n + 32)
// throughout: S^T = K Q^T (A = K chunk from LDS, B = the wave's queries, kept in registers) leaves each lane 16 of its
// query's 32 scores, the softmax needs one exchange between the pair, and the probabilities are, in place, the B
// operand of O^T += V^T P^T: its k order (lane half h, slot j -> key 16 s + 8 (j / 4) + 4 h + j % 4) is matched by the
// order in which V's keys are read (ds_read_b64_tr_b16: 4 keys of one dim per lane from a row-major V chunk).
//
// 32-key chunks, double-buffered in LDS as halves (K and V, hi and lo, [key][256]: 128 KB); one barrier per chunk: while
// chunk i's softmax and P V run, the scores of chunk i + 1 are formed, chunk i + 2 of K and i + 1 of V are converted
// into the buffers that became free, and the next raw chunks are on their way into registers. Overflow of the
// operand scale is flagged while converting; the flag is read after the barrier that publishes the chunk, and a flagged
// chunk (outliers) is staged again with its own scale by the whole block.
//
// What bounds it: the matrix products (96 instructions of 32 cycles per wave and chunk, one wave per SIMD) and the 80 KB
// of LDS reads and writes per wave beside them. 32 queries per wave, because every wave reads the whole staged chunk: at
// 16 queries the LDS reads alone outlast the products; 16 tokens per block halve the K and V read from the caches and
// the conversions per query. One wave per SIMD hides nothing by itself, hence the hand-placed slices of vector work after each
// matrix instruction. Registers: accumulators and most of Q in AGPRs (pinned; otherwise the compiler moves all 128
// accumulators through VGPRs each chunk), no scratch.
// One block per CU also means that nothing covers a block's ends: the query row and the first chunk are loaded in one
// round trip, the gate's values in another, and the last chunk forms no further scores (20 tokens 33 -> 28 us a call, 512
// tokens 70 -> 65, 400 prompts of 20 tokens 237 -> 168).
// One 8192-token prompt, 16 heads (550 GFLOP of fp32 products): 3.70 -> 1.75 ms = 314 TFLOP/s (943 of fp16 MFMA issue; a
// large library bf16 matrix product reaches 1380 on this card). The form before held 16 queries per wave, 8 tokens per
// block, with P through LDS.
// AttnPrefill<2> (halo_attn_prefill_d2): 8-token tiles, two waves share 32 queries and split the output dims: 0.75x the
// matrix work per wave and twice the blocks, for batches that 16-token tiles would spread unevenly over the CUs (256 tokens
// at position 8192: 694 us with 16-token tiles, 589 with these; 1160 in the form before).
namespace {
constexpr int kHalf = kChunk * kHd * 2;          // bytes of one staged matrix's hi (or lo) halves
constexpr int kBuf = 2 * kHalf;                  // bytes of one staged chunk of K or V
// The running max may lag by this (base 2) before a rescale: probabilities up to 2^1.9 stay below 65504 at 2^14 (kSpp), the
// scale that keeps 2^-39 of the row's largest. (2^10 with a lag of 5 saves the rescaling, 4% of an 8192-token prompt,
// but a probability 2^20 below the largest then has an error of up to 4e-5 of itself.)
constexpr float kLazy = 1.9f;
static_assert(kSpp == 16384.0f);
typedef float V16F __attribute__((ext_vector_type(16)));
typedef short S4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ V16F Mfma3x32(const H8& ah, const H8& al, const H8& bh, const H8& bl, V16F c) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, c, 0, 0, 0);
}
// 4 keys (rows) of one dim (column) per lane: within 16 lanes, lane i addresses 8 bytes of row i / 4 and receives column
// i of the four rows.
__device__ __forceinline__ H4 ReadTr(const char* p) {
  return __builtin_bit_cast(
      H4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) S4*)(const_cast<char*>(p))));
}
// 8 floats of 4 pieces of a K or V row: the largest magnitude, and the conversion of the pieces into a staged row
__device__ __forceinline__ float MaxAbs(const float4 (&r)[8]) {
  float a = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) a = fmaxf(a, fmaxf(fmaxf(fabsf(r[e].x), fabsf(r[e].y)), fmaxf(fabsf(r[e].z), fabsf(r[e].w))));
  return a;
}
__device__ __forceinline__ void StagePiece(const float4& u, const float4& v, char* at, float scale) {
  const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
  H8 hi, lo;
  SplitHalves(x, hi, lo, scale);
  *reinterpret_cast<H8*>(at) = hi;
  *reinterpret_cast<H8*>(at + kHalf) = lo;
}
// (piece part + 8 j at byte a0 ^ 128 (j & 1) + 256 (j / 2) of the hi half: the swizzle touches the low four piece bits)
__device__ __forceinline__ void StageRow(const float4 (&r)[8], char* lds, std::uint32_t a0, float scale) {
#pragma unroll
  for (int j = 0; j < 4; ++j) StagePiece(r[2 * j], r[2 * j + 1], lds + (a0 ^ (128u * (j & 1))) + 256 * (j / 2), scale);
}
}  // namespace

namespace {
template <int DS>
__device__ __forceinline__ void AttnPrefill(
    const float* __restrict__ q, const float* __restrict__ gate, const float* __restrict__ kpool,
    const float* __restrict__ vpool, const std::uint32_t* __restrict__ pages, const std::uint32_t* __restrict__ tiles,
    float* __restrict__ o, std::int8_t* __restrict__ oq, float* __restrict__ os, std::uint32_t Hq, std::uint32_t Hkv,
    std::uint32_t max_pages) {
  constexpr int NJ = 16 / DS;  // steps of the wave's P V: 8 / DS tiles of 32 dims x two steps of 16 keys
  // K rows: 16-byte piece c of key at c ^ (key & 15); V rows: at c ^ 2 (key & 7) (four keys of a 16-lane transposing read
  // in four different 32-byte bank groups)
  __shared__ __attribute__((aligned(1024))) char lds[4 * kBuf];  // K buffers 0, 1, V buffers 0, 1: hi then lo halves
  __shared__ float red[4];
  __shared__ __attribute__((aligned(16))) std::uint32_t flags[2][2][4];  // [buffer][K, V][wave]: the scale overflowed
  const std::uint32_t* tl = tiles + 4 * static_cast<std::size_t>(blockIdx.x / Hkv);
  const std::uint32_t first = tl[0], ntok = tl[1], sess = tl[2], p0 = tl[3];
  const std::uint32_t kvh = blockIdx.x % Hkv;
  const std::uint32_t t = threadIdx.x, wave = t / kWave, lane = t % kWave, n = lane % 32, h = lane / 32;
  const std::uint32_t tok0 = 4 * (wave / DS), d0 = wave % DS * (kHd / DS);  // the wave's first token and output dim
  const std::uint32_t last = p0 + ntok - 1, nchunks = last / kChunk + 1;
  const std::uint32_t* pt = pages + static_cast<std::size_t>(sess) * max_pages;
  // staging: thread t holds key t / 8 of a chunk, 32-byte pieces part + 8 j
  const std::uint32_t skey = t / 8, spart = t % 8;
  const std::uint32_t ksa = skey * 512 + 16 * (spart ^ (skey & 15));
  const std::uint32_t vsa = 2 * kBuf + skey * 512 + 16 * (spart ^ (2 * (skey & 7)));
  // reads: K step c (dims 16 c + 8 h ..) of key n at ka ^ 32 (c & 7) + 256 (c / 8); V's keys 4 h + lane % 16 / 4 (+ 8, + 16 per step),
  // dims 32 c + 16 (lane / 16 % 2) + 4 (lane % 4) at va ^ 64 (c & 3) + 256 (c / 4)
  const std::uint32_t ka = n * 512 + 16 * (h ^ (n & 15));
  const std::uint32_t vk = 4 * h + (lane % 16) / 4;
  const std::uint32_t va = 2 * kBuf + vk * 512 + 16 * ((2 * (lane / 16 % 2) + lane % 4 / 2) ^ (2 * vk)) + 8 * (lane % 2) + 2 * d0;
  float4 kraw[8], vraw[8];
  const auto position = [&](std::uint32_t c) { return min(c * kChunk + skey, last); };
  const auto row = [&](const float* pool, std::uint32_t page, std::uint32_t c) {
    return reinterpret_cast<const float4*>(
        pool + ((static_cast<std::size_t>(page) * Hkv + kvh) * kPage + position(c) % kPage) * kHd);
  };
  const auto load = [&](const float* pool, std::uint32_t page, std::uint32_t c, float4 (&r)[8]) {
    const float4* s = row(pool, page, c);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      r[2 * j] = s[2 * (spart + 8 * j)];
      r[2 * j + 1] = s[2 * (spart + 8 * j) + 1];
    }
  };
  std::uint32_t pg0 = pt[position(0) / kPage], pg1 = pt[position(1) / kPage], pg2 = pt[position(2) / kPage];
  __builtin_amdgcn_sched_barrier(0);
  // this lane's query: dims 16 c + 8 h .. + 7 of step c (the B operand). Its whole row and the first chunk are in flight
  // together (read in two passes, the second a few values at a time, the row took longer than a short prompt's products)
  const std::uint32_t tok = min(tok0 + n / 8, ntok - 1);
  const std::size_t qbase = ((static_cast<std::size_t>(first) + tok) * Hq + kvh * 8 + n % 8) * kHd;
  H8 qh[kHd / 16], ql[kHd / 16];
  float fq;
  {
    const float* qrow = q + qbase + 8 * h;
    float4 x4[kHd / 8];
    float amax = 0.0f;
#pragma unroll
    for (int c = 0; c < kHd / 8; ++c) x4[c] = *reinterpret_cast<const float4*>(qrow + 16 * (c / 2) + 4 * (c % 2));
    __builtin_amdgcn_sched_barrier(0);
    load(kpool, pg0, 0, kraw);
    load(vpool, pg0, 0, vraw);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kHd / 8; ++c)
      amax = fmaxf(amax, fmaxf(fmaxf(fabsf(x4[c].x), fabsf(x4[c].y)), fmaxf(fabsf(x4[c].z), fabsf(x4[c].w))));
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    const float sq = halo::SplitScale(amax, kSqk);
#pragma unroll
    for (int c = 0; c < kHd / 16; ++c) {
      const float4 a = x4[2 * c], b = x4[2 * c + 1];
      const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      SplitHalves(x, qh[c], ql[c], sq);
      __builtin_amdgcn_sched_barrier(0);
      asm("" : "+a"(qh[c]));
      if (c < 8) asm("" : "+a"(ql[c]));
    }
    // scores and the running max in base-2 units: each exponential is one v_exp_f32
    fq = (1.0f / sqrtf(static_cast<float>(kHd))) * kLog2e / sq;
  }
  const std::uint32_t qpos = p0 + tok0 + n / 8;
  float sva = kSvv;  // V's scale (uniform): the smallest of the chunks so far, at which acc stands and V is staged
  float l = 0.0f;
  V16F acc[NJ / 2];
#pragma unroll
  for (int c = 0; c < NJ / 2; ++c) {
    acc[c] = V16F{};
    asm("" : "+a"(acc[c]));
  }

  // a chunk of K or V from registers into buffer b at the default scale, flagged by the waves where that overflows (every
  // lane of a wave stores the same word: a store under a branch would cut the schedule); the prologue's chunks
  const auto stage = [&](int which, const float4 (&r)[8], std::uint32_t b) {
    flags[b ^ which][which][wave] = __any(MaxAbs(r) * 256.0f >= 65504.0f) ? 1u : 0u;
    StageRow(r, lds, (which ? vsa : ksa) + b * kBuf, 256.0f);
  };
  // at iteration i the block reads the pair (K of chunk i + 1, V of chunk i) in one row: K's buffer index and the
  // complement of V's
  const auto flagged = [&](std::uint32_t row_) {
    const uint4 k = *reinterpret_cast<const uint4*>(flags[row_][0]), v = *reinterpret_cast<const uint4*>(flags[row_][1]);
    const std::uint32_t w = k.x | k.y | k.z | k.w | (v.x | v.y | v.z | v.w) << 1;
    return __builtin_amdgcn_readfirstlane(w);
  };
  static_assert(kSqk == 256.0f && kSvv == 256.0f);
  // a flagged chunk again, by the whole block, at the scale of its largest magnitude; returns the scale, below the
  // one that overflowed (not above it either where the magnitude is infinite and has no scale: one infinite V then
  // spoils its own dim alone)
  const auto restage = [&](const float* pool, std::uint32_t c, bool is_v, std::uint32_t b, float base) {
    const float4* src = row(pool, pt[position(c) / kPage], c);
    float w = 0.0f;
#pragma unroll 1
    for (int j = 0; j < 8; ++j) {
      const float4 x = src[2 * (spart + 8 * (j / 2)) + j % 2];
      w = fmaxf(w, fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))));
    }
    w = halo::GroupMax(w);
    if (lane == 0) red[wave] = w;
    __syncthreads();
    const float s = __uint_as_float(__builtin_amdgcn_readfirstlane(
        __float_as_uint(fminf(base, halo::SplitScale(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])), base)))));
    const std::uint32_t a0 = (is_v ? vsa : ksa) + b * kBuf;
#pragma unroll 1
    for (int j = 0; j < 4; ++j) {
      const float4 u = src[2 * (spart + 8 * j)], v = src[2 * (spart + 8 * j) + 1];
      StagePiece(u, v, lds + (a0 ^ (128u * (j & 1))) + 256 * (j / 2), s);
    }
    __syncthreads();
    return s;
  };
  // operand fragments of K step c and of V step j = 2 c + st (dims 32 c .., keys 16 st ..)
  const auto kfrag = [&](std::uint32_t b, int c, H8& hi, H8& lo) {
    const char* at = lds + ((ka + b * kBuf) ^ (32u * (c & 7))) + 256 * (c / 8);
    hi = *reinterpret_cast<const H8*>(at);
    lo = *reinterpret_cast<const H8*>(at + kHalf);
  };
  const auto vfrag = [&](std::uint32_t b, int j, H8& hi, H8& lo) {
    const int c = j / 2, st = j % 2;
    const char* at = lds + ((va + b * kBuf) ^ (64u * (c & 3))) + 256 * (c / 4) + 8192 * st;
    const H4 h0 = ReadTr(at), h1 = ReadTr(at + 4096), l0 = ReadTr(at + kHalf), l1 = ReadTr(at + kHalf + 4096);
    hi = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
    lo = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  stage(0, kraw, 0);
  load(kpool, pg1, 1, kraw);
  stage(1, vraw, 0);
  load(vpool, pg1, 1, vraw);
  __syncthreads();
  float f = fq / kSqk;
  if (flagged(0) & 1u) f = fq / restage(kpool, 0, false, 0, kSqk);
  V16F s = {};
#pragma unroll
  for (int c = 0; c < kHd / 16; ++c) {
    H8 ah, al;
    kfrag(0, c, ah, al);
    s = Mfma3x32(ah, al, qh[c], ql[c], s);
  }
  // masked scores of a chunk (slot j: key 8 (j / 4) + 4 h + j % 4 of it; lim: the query's position in it, less 4 h) and
  // their largest over the lane pair
  const auto mask = [&](float x, int j, int lim) { return 8 * (j / 4) + j % 4 <= lim ? x : -INFINITY; };
  const auto pair_max = [](float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  };
  float cm = -INFINITY;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    s[j] = mask(s[j], j, static_cast<int>(qpos - 4 * h));
    cm = fmaxf(cm, s[j]);
  }
  cm = pair_max(cm) * f;
  float m = cm;
  stage(0, kraw, 1);
  load(kpool, pg2, 2, kraw);
  pg1 = pg2;  // at iteration i: pg1, pg2 the pages of chunks i + 2, i + 3
  pg2 = pt[position(3) / kPage];
  // chunk i; the last one has no scores to form and nothing to stage (a third of a one-chunk block's products)
  const auto step = [&](auto is_last, std::uint32_t i) __attribute__((always_inline)) {
    constexpr bool kLast = is_last;
    const std::uint32_t b = i & 1, nb = b ^ 1;
    halo::LdsSync();  // K of chunk i + 1 and V of chunk i are staged; the buffers of K i and V i - 1 are free
    float fn = fq / kSqk, vfac = 1.0f;  // score factor of chunk i + 1 (exact: the scales are powers of two)
    const std::uint32_t fl = flagged(nb);
    if (fl != 0u) {
      if (!kLast && (fl & 1u)) fn = fq / restage(kpool, i + 1, false, nb, kSqk);
      if (fl & 2u) {
        const float svc = restage(vpool, i, true, b, sva);
        vfac = svc / sva;
        sva = svc;
      }
    }
    // the running max (base-2 units) lags by up to kLazy, so few chunks rescale; a query's own scores decide when its max
    // moves, so its bits do not depend on the queries that share its wave
    const bool up = cm > m + kLazy;
    if (__any(up) || vfac != 1.0f) {
      const float alpha = up ? __builtin_amdgcn_exp2f(m - cm) : 1.0f;
      m = up ? cm : m;
      l *= alpha;
#pragma unroll
      for (int c = 0; c < NJ / 2; ++c) {
        // through vector registers 16 at a time: without the pins the accumulators live there from the loop's start on,
        // and every iteration copies all of them
        V16F a = acc[c];
        asm("" : "+v"(a));
        a *= alpha * vfac;
        asm("" : "+a"(a));
        acc[c] = a;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // P^T of chunk i (slots 8 st .. 8 st + 7 are the k order of step st) beside the scores of chunk i + 1,
    // then P V beside the conversions: after each matrix instruction a slice of the vector
    // work that it hides (the barriers keep that order), each step's fragments read one step ahead.
    H8 ah[2], al[2];
    V16F sn = {};
    float e[16], ls = 0.0f;
    std::uint32_t pw[16], sw[8];
    const auto softmax_slice = [&](int k) {  // k < 24: scores 2 p, 2 p + 1 in slices 3 p .. 3 p + 2
      const int p = k / 3;
      if (k >= 24) return;
      if (k % 3 == 0) {
        e[2 * p] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * p], f, -m));
        e[2 * p + 1] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * p + 1], f, -m));
      } else if (k % 3 == 1) {
        halo::SplitPair(e[2 * p], e[2 * p + 1], kSpp, pw[p], pw[8 + p]);
      } else {
        ls += e[2 * p] + e[2 * p + 1];
      }
    };
    // k < 24: as stage(which, buf), in four pieces: its splits, its two stores, and the same piece of the chunk after into
    // the registers that became free (in flight for a whole iteration). V at the smallest scale so far, so that P and acc
    // need no factor of their own: a small P has no bits to spare, V loses only what the outlier's fp32 sum would
    const auto stage_slice = [&](int k, int which, float4 (&r)[8], const float4* next, std::uint32_t buf, float& top) {
      const int j = k / 6, e = k % 6;
      const float scale = which ? sva : kSqk;
      if (e < 4) {
        const float4 x = r[2 * j + e / 2];
        halo::SplitPair(e % 2 ? x.z : x.x, e % 2 ? x.w : x.y, scale, sw[e], sw[4 + e]);
        if (e % 2 == 0) top = fmaxf(top, fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))));
      } else if (e == 4) {
        char* at = lds + (((which ? vsa : ksa) + buf * kBuf) ^ (128u * (j & 1))) + 256 * (j / 2);
        *reinterpret_cast<uint4*>(at) = make_uint4(sw[0], sw[1], sw[2], sw[3]);
        *reinterpret_cast<uint4*>(at + kHalf) = make_uint4(sw[4], sw[5], sw[6], sw[7]);
      } else {
        r[2 * j] = next[2 * (spart + 8 * j)];
        r[2 * j + 1] = next[2 * (spart + 8 * j) + 1];
        if (j == 3) flags[buf ^ which][which][wave] = __any(top * scale >= 65504.0f) ? 1u : 0u;
      }
    };
    // k < 24: the masked scores of chunk i + 1 and their max (from slice 4 on: the last score product has landed)
    const int lim = static_cast<int>(qpos - 4 * h) - static_cast<int>(i * kChunk + kChunk);
    const auto score_slice = [&](int k) {
      if (k >= 4 && k < 20) {
        s[k - 4] = mask(sn[k - 4], k - 4, lim);
        cm = fmaxf(cm, s[k - 4]);
      } else if (k == 20) {
        cm = pair_max(cm) * fn;
      }
    };
    const float4 *knext = nullptr, *vnext = nullptr;
    float top = 0.0f;
    if constexpr (!kLast) {
      kfrag(nb, 0, ah[0], al[0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 9; ++k) softmax_slice(k);  // while the first fragments arrive
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        if (c < 15)
          kfrag(nb, c + 1, ah[(c + 1) % 2], al[(c + 1) % 2]);
        else
          vfrag(b, 0, ah[0], al[0]);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          sn = __builtin_amdgcn_mfma_f32_32x32x16_f16(p == 0 ? al[c % 2] : ah[c % 2], p == 1 ? ql[c] : qh[c], sn, 0, 0, 0);
          if (c == 0 && p == 1) {
            knext = row(kpool, pg2, i + 3);
            vnext = row(vpool, pg1, i + 2);
            pg1 = pg2;
            pg2 = pt[position(i + 4) / kPage];  // ahead of this iteration's row loads: not waited for with them
          }
          if (c < 8)
            softmax_slice(3 * c + p + 9 < 24 ? 3 * c + p + 9 : 24);
          else
            stage_slice(3 * (c - 8) + p, 0, kraw, knext, b, top);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else {
      vfrag(b, 0, ah[0], al[0]);
#pragma unroll
      for (int k = 0; k < 24; ++k) softmax_slice(k);
    }
    l += ls;
    cm = -INFINITY;
    H8 ph[2], pl[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      ph[st] = __builtin_bit_cast(H8, make_uint4(pw[4 * st], pw[4 * st + 1], pw[4 * st + 2], pw[4 * st + 3]));
      pl[st] = __builtin_bit_cast(H8, make_uint4(pw[8 + 4 * st], pw[9 + 4 * st], pw[10 + 4 * st], pw[11 + 4 * st]));
    }
    top = 0.0f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if (j < NJ - 1) vfrag(b, j + 1, ah[(j + 1) % 2], al[(j + 1) % 2]);
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        acc[j / 2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(p == 0 ? al[j % 2] : ah[j % 2], p == 1 ? pl[j % 2] : ph[j % 2],
                                                             acc[j / 2], 0, 0, 0);
        if (!kLast && j < 8) score_slice(3 * j + p);
        if (!kLast && j >= NJ - 8) stage_slice(3 * (j - (NJ - 8)) + p, 1, vraw, vnext, nb, top);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    f = fn;
  };
  for (std::uint32_t i = 0; i + 1 < nchunks; ++i) step(std::false_type{}, i);
  step(std::true_type{}, nchunks - 1);
  // epilogue: this lane's query, dims d0 + 32 c + 8 g + 4 h + e (slot 4 g + e)
  float4 gt[NJ / 2][4];  // all in flight at once: between the branches below each would be waited for by itself
#pragma unroll
  for (int c = 0; c < NJ / 2; ++c)
#pragma unroll
    for (int g = 0; g < 4; ++g) gt[c][g] = *reinterpret_cast<const float4*>(gate + qbase + d0 + 32 * c + 8 * g + 4 * h);
  __builtin_amdgcn_sched_barrier(0);
  l += __shfl_xor(l, 32);
  const bool live = tok0 + n / 8 < ntok;
  const float inv = 1.0f / l * (1.0f / (kSpp * sva));
#pragma unroll
  for (int c = 0; c < NJ / 2; ++c) {
    float v[16], amax = 0.0f;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const std::size_t at = qbase + d0 + 32 * c + 8 * g + 4 * h;
      v[4 * g] = acc[c][4 * g] * inv * halo::Sigmoid(gt[c][g].x);
      v[4 * g + 1] = acc[c][4 * g + 1] * inv * halo::Sigmoid(gt[c][g].y);
      v[4 * g + 2] = acc[c][4 * g + 2] * inv * halo::Sigmoid(gt[c][g].z);
      v[4 * g + 3] = acc[c][4 * g + 3] * inv * halo::Sigmoid(gt[c][g].w);
      if (live && o != nullptr) *reinterpret_cast<float4*>(o + at) = make_float4(v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]);
#pragma unroll
      for (int e = 0; e < 4; ++e) amax = fmaxf(amax, fabsf(v[4 * g + e]));
    }
    if (oq != nullptr) {  // a Q8 block is this step's 32 dims: 16 in each lane of the pair
      const float qs = fmaxf(amax, __shfl_xor(amax, 32)) / 127.0f;
      const halo::CodeScale cs(qs);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        std::uint32_t word = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int code = cs.Code(v[4 * g + e]);
          word |= (static_cast<std::uint32_t>(code) & 0xFFu) << (8 * e);
        }
        if (live) *reinterpret_cast<std::uint32_t*>(oq + qbase + d0 + 32 * c + 8 * g + 4 * h) = word;
      }
      if (live && h == 0) os[(qbase + d0 + 32 * c) / 32] = qs;
    }
  }
}
}  // namespace

#define HALO_ATTN_PREFILL(NAME, DS)                                                                                   \
  extern "C" __global__ void __launch_bounds__(256, 1) NAME(                                                          \
      const float* q, const float* gate, const float* kpool, const float* vpool, const std::uint32_t* pages,          \
      const std::uint32_t* tiles, float* o, std::int8_t* oq, float* os, std::uint32_t Hq, std::uint32_t Hkv,          \
      std::uint32_t max_pages) {                                                                                      \
    AttnPrefill<DS>(q, gate, kpool, vpool, pages, tiles, o, oq, os, Hq, Hkv, max_pages);                              \
  }
HALO_ATTN_PREFILL(halo_attn_prefill, 1)
HALO_ATTN_PREFILL(halo_attn_prefill_d2, 2)
#undef HALO_ATTN_PREFILL
