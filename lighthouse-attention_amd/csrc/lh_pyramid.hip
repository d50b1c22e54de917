// Norm scorer + mean-pooled Q/K/V pyramid (forward) and the pyramid backward.
//
// Forward restates DialatedLighthouseNormScorer.forward
// (src/lighthouse_selection.py:589-616): base scores are the L2 norms of q and
// k rows, rounded to the row type (bf16 or fp16) like torch's `norm` of such
// rows; level j = 1..L-1 rows are
// the means of p^j consecutive base rows (fp32 sum, one rounding), and level-j
// scores are maxima of the base scores over the same span.  One pass streams
// xq/xk/xv once: 16 lanes (8 for D <= 64) own one (b, span, head) unit, 8 bf16 each, and walk
// the p^(L-1) base tokens of the span.  Base rows are never copied: pooled rows
// go to a separate [B, Sp, H, D] buffer.
//
// Backward restates the autograd of gather + cat + mean: each base row gets
// its own selected-space gradient plus, for every pooled level that contains
// it, that node's gradient / c_l.  Gather-formulated through the inverse map,
// so there are no atomics and the result is deterministic.
#include "lh_common.h"

#include <algorithm>

namespace {

struct PyrArgs {
  const bf16_t *xq, *xk, *xv;
  int64_t sb, ss, sh;
  bf16_t *pq, *pk, *pv;
  int64_t pb, ps, ph;
  float *sqk, *skq;
  const float* fs;   // rotary (cos, sin) table [>= S, D/2, 2] (ROPE)
  bf16_t *rq, *rk;   // rotated base rows out (ROPE)
  int64_t rb, rs, rh;
  bf16_t *cq, *ck, *cv;  // CAT: base rows out (strides pb, ps, ph)
  bf16_t *hq, *hk;       // CAT: all levels' scores in the row type, [B, H, S_tot]
  int B, S, H, D, L, shift, S_tot, nspan, cmax, units;
  int off[9], len[9];
};

__device__ __forceinline__ uint4 ld16(const bf16_t* p) { return *reinterpret_cast<const uint4*>(p); }

constexpr int PYR_CHUNK = 4;  // base tokens whose loads are issued together

// One base token t of (b, h): unpack the 16-byte slices of its q, k, v rows,
// rotate q and k (ROPE: rounded to bf16 and stored to rq / rk, the rounded
// values kept), and make its base scores: the bf16-rounded L2 norms of q and k
// (every lane of the row's group gets them), or the given ones (GIVEN: sq, sk
// on entry).
template <typename T, typename Ln, bool GIVEN, bool ROPE>
__device__ __forceinline__ void pyr_token(const PyrArgs& a, int b, int h, int l16, int t,
                                          const uint4 xq, const uint4 xk, const uint4 xv, float* fq, float* fk,
                                          float* fv, float& sq, float& sk) {
  unpack8_t<T>(xq, fq);
  unpack8_t<T>(xk, fk);
  unpack8_t<T>(xv, fv);
  if (ROPE) {
    float4 c01, c23;
    rope_freqs8(a.fs, t, LH_D, 8 * l16, c01, c23);
    rope_rotate8<true>(fq, c01, c23);
    rope_rotate8<true>(fk, c01, c23);
    const uint4 wq = pack8_t<T>(fq), wk = pack8_t<T>(fk);
    const int64_t ro = (int64_t)b * a.rb + (int64_t)t * a.rs + (int64_t)h * a.rh + 8 * l16;
    *reinterpret_cast<uint4*>(a.rq + ro) = wq;
    *reinterpret_cast<uint4*>(a.rk + ro) = wk;
    unpack8_t<T>(wq, fq);
    unpack8_t<T>(wk, fk);
  }
  if (!GIVEN) {
    float pq = 0.f, pk = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { pq = fmaf(fq[e], fq[e], pq); pk = fmaf(fk[e], fk[e], pk); }
#pragma unroll
    for (int m = 1; m < Ln::LPR; m <<= 1) { pq += __shfl_xor(pq, m, Ln::LPR); pk += __shfl_xor(pk, m, Ln::LPR); }
    sq = round_to<T>(sqrtf(pq));
    sk = round_to<T>(sqrtf(pk));
  }
}

// ROPE: xq / xk are the projection's unrotated rows; each is rotated by its
// position's angles, rounded to bf16 and written to rq / rk, and the norms and
// means below are taken of those rounded rows, exactly as if the rotated rows
// had been stored first and read back.
// CAT: the scorer modules' form, whose outputs are the concatenated pyramids: the
// base rows are written out as they stream by (in front of the pooled rows, as
// three separate copies they were read a second time: 71 us of a 285 us scorer
// call at 8 x 32768 rows) and every score also in the row type.
template <typename T, typename Ln, int NL, bool GIVEN, bool ROPE, bool CAT>
__global__ __launch_bounds__(256) void pyramid_fwd_kernel(const PyrArgs a) {
  const int tid = threadIdx.x;
  const int u = blockIdx.x * Ln::ROWS + tid / Ln::LPR;
  const int l16 = tid % Ln::LPR;
  const bool in = Ln::in(l16, a.D);
  if (u >= a.units) return;
  const int h = u % a.H;
  const int rest = u / a.H;
  const int span = rest % a.nspan;
  const int b = rest / a.nspan;
  const int t0 = span * a.cmax;
  const int t1 = min(a.S, t0 + a.cmax);
  const size_t srow = (size_t)(b * a.H + h) * a.S_tot;

  constexpr int NA = NL > 0 ? NL : 1;
  float accq[NA][8], acck[NA][8], accv[NA][8], mq[NA], mk[NA];
#pragma unroll
  for (int l = 0; l < NL; ++l) {
    mq[l] = -INFINITY; mk[l] = -INFINITY;
#pragma unroll
    for (int e = 0; e < 8; ++e) { accq[l][e] = 0.f; acck[l][e] = 0.f; accv[l][e] = 0.f; }
  }
  const int64_t xoff = (int64_t)b * a.sb + (int64_t)h * a.sh + 8 * l16;
  float bq = 0.f, bk = 0.f;  // this lane's pending base scores
  // one base token: rows (q, k, v) as loaded, base scores when GIVEN
  auto token = [&](int t, const uint4 xq, const uint4 xk, const uint4 xv, float sq, float sk)
      __attribute__((always_inline)) {
    float fq[8], fk[8], fv[8];
    pyr_token<T, Ln, GIVEN, ROPE>(a, b, h, l16, t, xq, xk, xv, fq, fk, fv, sq, sk);
    if (CAT && in) {
      const int64_t co = (int64_t)b * a.pb + (int64_t)t * a.ps + (int64_t)h * a.ph + 8 * l16;
      *reinterpret_cast<uint4*>(a.cq + co) = xq;
      *reinterpret_cast<uint4*>(a.ck + co) = xk;
      *reinterpret_cast<uint4*>(a.cv + co) = xv;
    }
    if (!GIVEN || CAT) {
      // base scores leave LPR tokens at a time: lane j keeps token t0 + LPR i + j,
      // and the group stores them as one contiguous run per tensor
      const int j = (t - t0) & (Ln::LPR - 1);
      if (l16 == j) { bq = sq; bk = sk; }
      if ((j == Ln::LPR - 1 || t == t1 - 1) && l16 <= j) {
        if (!GIVEN) {
          a.sqk[srow + t - j + l16] = bq;
          a.skq[srow + t - j + l16] = bk;
        }
        if (CAT) {
          a.hq[srow + t - j + l16] = (bf16_t)(T::pack2(bq, 0.f) & 0xffffu);
          a.hk[srow + t - j + l16] = (bf16_t)(T::pack2(bk, 0.f) & 0xffffu);
        }
      }
    }
#pragma unroll
    for (int l = 0; l < NL; ++l) {
#pragma unroll
      for (int e = 0; e < 8; ++e) { accq[l][e] += fq[e]; acck[l][e] += fk[e]; accv[l][e] += fv[e]; }
      mq[l] = fmaxf(mq[l], sq);
      mk[l] = fmaxf(mk[l], sk);
      const int cs = (l + 1) * a.shift;  // log2 of the span of level l+2
      if (((t + 1) & ((1 << cs) - 1)) == 0) {
        const int node = t >> cs;
        const int lvl = l + 2;
        const float inv_c = 1.0f / (float)(1 << cs);
        float mo[8];
        const int64_t prow = (int64_t)b * a.pb + (int64_t)(a.off[lvl] - a.S + node) * a.ps + (int64_t)h * a.ph + 8 * l16;
#pragma unroll
        for (int e = 0; e < 8; ++e) mo[e] = accq[l][e] * inv_c;
        if (in) *reinterpret_cast<uint4*>(a.pq + prow) = pack8_t<T>(mo);
#pragma unroll
        for (int e = 0; e < 8; ++e) mo[e] = acck[l][e] * inv_c;
        if (in) *reinterpret_cast<uint4*>(a.pk + prow) = pack8_t<T>(mo);
#pragma unroll
        for (int e = 0; e < 8; ++e) mo[e] = accv[l][e] * inv_c;
        if (in) *reinterpret_cast<uint4*>(a.pv + prow) = pack8_t<T>(mo);
        if (l16 == 0) {
          a.sqk[srow + a.off[lvl] + node] = mq[l];
          a.skq[srow + a.off[lvl] + node] = mk[l];
          if (CAT) {
            a.hq[srow + a.off[lvl] + node] = (bf16_t)(T::pack2(mq[l], 0.f) & 0xffffu);
            a.hk[srow + a.off[lvl] + node] = (bf16_t)(T::pack2(mk[l], 0.f) & 0xffffu);
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) { accq[l][e] = 0.f; acck[l][e] = 0.f; accv[l][e] = 0.f; }
        mq[l] = -INFINITY; mk[l] = -INFINITY;
      }
    }
  };
  // Tokens in chunks of PYR_CHUNK with every load of a chunk issued before the
  // first is used, so a wave keeps PYR_CHUNK rows per tensor in flight instead
  // of one; tokens are still summed in order.
  const uint4 zero = make_uint4(0, 0, 0, 0);
  int t = t0;
  for (; t + PYR_CHUNK <= t1; t += PYR_CHUNK) {
    uint4 cq[PYR_CHUNK], ck[PYR_CHUNK], cv[PYR_CHUNK];
    float gq[PYR_CHUNK], gk[PYR_CHUNK];
#pragma unroll
    for (int i = 0; i < PYR_CHUNK; ++i) {
      const int64_t o = xoff + (int64_t)(t + i) * a.ss;
      cq[i] = in ? ld16(a.xq + o) : zero;
      ck[i] = in ? ld16(a.xk + o) : zero;
      cv[i] = in ? ld16(a.xv + o) : zero;
      gq[i] = GIVEN ? a.sqk[srow + t + i] : 0.f;
      gk[i] = GIVEN ? a.skq[srow + t + i] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < PYR_CHUNK; ++i) token(t + i, cq[i], ck[i], cv[i], gq[i], gk[i]);
  }
  for (; t < t1; ++t) {
    const int64_t o = xoff + (int64_t)t * a.ss;
    token(t, in ? ld16(a.xq + o) : zero, in ? ld16(a.xk + o) : zero, in ? ld16(a.xv + o) : zero, GIVEN ? a.sqk[srow + t] : 0.f,
          GIVEN ? a.skq[srow + t] : 0.f);
  }
}

// The forward for few spans.  pyramid_fwd_kernel has one group walk the
// p^(L-1) tokens of a span, four loads in flight, so a short sequence leaves
// most of the chip idle and waits for memory several times in a row (8 heads of
// 2048 tokens: 64 blocks, 15 us).  Here a block takes a tile of tokens of one
// (b, h), whole spans, with one token per group at a time, keeps their rows in
// LDS, and then its groups share the pooled nodes, (level, node, tensor) each,
// summing a node's tokens in their order: the same bits as the walk.
constexpr int PYR_TILE = 64;  // most tokens of a tile: spans longer than that take the walk

template <typename T, typename Ln, bool ROPE>
__global__ __launch_bounds__(256) void pyramid_tile_kernel(const PyrArgs a, int tt) {
  __shared__ uint4 X[3][PYR_TILE * Ln::LPR];
  __shared__ float SC[2][PYR_TILE];
  const int tid = threadIdx.x, g = tid / Ln::LPR, l16 = tid % Ln::LPR;
  const bool in = Ln::in(l16, a.D);
  const int chunks = (a.S + tt - 1) / tt;
  const int bh = blockIdx.x / chunks, b = bh / a.H, h = bh - b * a.H;
  const int t0 = (blockIdx.x - bh * chunks) * tt;
  const size_t srow = (size_t)bh * a.S_tot;
  const int64_t xoff = (int64_t)b * a.sb + (int64_t)h * a.sh + 8 * l16;
  const uint4 zero = make_uint4(0, 0, 0, 0);
  for (int i = g; i < tt && t0 + i < a.S; i += Ln::ROWS) {
    const int t = t0 + i;
    const int64_t o = xoff + (int64_t)t * a.ss;
    const uint4 xq = in ? ld16(a.xq + o) : zero, xk = in ? ld16(a.xk + o) : zero, xv = in ? ld16(a.xv + o) : zero;
    float fq[8], fk[8], fv[8], sq, sk;
    pyr_token<T, Ln, false, ROPE>(a, b, h, l16, t, xq, xk, xv, fq, fk, fv, sq, sk);
    X[0][i * Ln::LPR + l16] = ROPE ? pack8_t<T>(fq) : xq;  // the rotated rows' own 16 bits
    X[1][i * Ln::LPR + l16] = ROPE ? pack8_t<T>(fk) : xk;
    X[2][i * Ln::LPR + l16] = xv;
    if (l16 == 0) {
      SC[0][i] = sq;
      SC[1][i] = sk;
    }
  }
  __syncthreads();
  if (tid < 2 * PYR_TILE) {
    const int i = tid & (PYR_TILE - 1);
    if (i < tt && t0 + i < a.S) (tid < PYR_TILE ? a.sqk : a.skq)[srow + t0 + i] = SC[tid / PYR_TILE][i];
  }
  int task = g;
  for (int lvl = 2; lvl <= a.L; ++lvl) {
    const int cs = (lvl - 1) * a.shift, c = 1 << cs, nodes = tt >> cs;
    for (; task < 3 * nodes; task += Ln::ROWS) {
      const int x = task / nodes, i = task - x * nodes, node = (t0 >> cs) + i;
      if (node >= a.len[lvl]) continue;
      float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0}, mx = -INFINITY;
      for (int j = i << cs; j < (i + 1) << cs; ++j) {
        float f[8];
        unpack8_t<T>(X[x][j * Ln::LPR + l16], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += f[e];
        if (x < 2) mx = fmaxf(mx, SC[x][j]);
      }
      const float inv_c = 1.0f / (float)c;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] *= inv_c;
      const int r = a.off[lvl] + node;
      bf16_t* pool = x == 0 ? a.pq : x == 1 ? a.pk : a.pv;
      if (in)
        *reinterpret_cast<uint4*>(pool + (int64_t)b * a.pb + (int64_t)(r - a.S) * a.ps + (int64_t)h * a.ph + 8 * l16) =
            pack8_t<T>(acc);
      if (x < 2 && l16 == 0) (x ? a.skq : a.sqk)[srow + r] = mx;
    }
    task -= 3 * nodes;
  }
}

struct PyrBwdArgs {
  const bf16_t *gq, *gk, *gv;
  int64_t gb, gh, gs;
  const int32_t* inv;
  bf16_t *dq, *dk, *dv;
  int64_t ob, os, oh;  // strides of the three outputs (element units)
  const float* fs;     // ROPE: (cos, sin) table; dq, dk are rotated back by -theta
  int B, S, H, D, L, shift, S_tot;
  int off[9], len[9];
  long long rows;
  int chunks;  // chunks of 16 (D <= 64: 32) tokens per (b, h)
};

// One 16-lane group per (b, t, h) row, 8 d each; a block covers 16 consecutive
// tokens of one (b, h) (D <= 64: 8 lanes, 32 tokens), so the rows of a pooled node spanning up to 16 tokens
// are read by one block (the wave or block coalesces the repeats instead of
// several blocks fetching the row through L2), and runs of 32 consecutive
// chunks of a head stay on one XCD (`xcd_run`; one whole head per XCD left the
// XCDs unevenly loaded, as the gathered rows per token differ by head).  All
// levels' inverse lookups
// are issued first, then all gradient-row loads, so a row costs two dependent
// memory round trips instead of two per level.  ROPE: the q and k sums are
// the gradients of rotated rows; they are rotated back (the adjoint of the
// forward rotation) in fp32 before the one rounding.
template <typename T, typename Ln, int NL, bool ROPE>
__global__ __launch_bounds__(256) void pyramid_bwd_kernel(const PyrBwdArgs a) {
  const int tid = threadIdx.x;
  const long long blk = xcd_run(blockIdx.x, gridDim.x, 32);
  const long long bh = blk / a.chunks;
  const int t = (int)(blk - bh * a.chunks) * Ln::ROWS + tid / Ln::LPR;
  const int l16 = tid % Ln::LPR;
  if (t >= a.S || !Ln::in(l16, a.D)) return;
  const int h = (int)(bh % a.H);
  const int b = (int)(bh / a.H);
  const size_t irow = (size_t)(b * a.H + h) * a.S_tot;
  const int64_t gbase = (int64_t)b * a.gb + (int64_t)h * a.gh + 8 * l16;
  int s[NL];
#pragma unroll
  for (int l = 0; l < NL; ++l) {
    const int node = t >> (l * a.shift);
    const int r = a.off[l + 1] + node;
    s[l] = node < a.len[l + 1] ? (a.inv ? a.inv[irow + r] : r) : -1;
  }
  const uint4 z = make_uint4(0, 0, 0, 0);
  uint4 gq[NL], gk[NL], gv[NL];
#pragma unroll
  for (int l = 0; l < NL; ++l) {
    const int64_t go = gbase + (int64_t)max(s[l], 0) * a.gs;
    gq[l] = (a.gq && s[l] >= 0) ? ld16(a.gq + go) : z;
    gk[l] = (a.gk && s[l] >= 0) ? ld16(a.gk + go) : z;
    gv[l] = (a.gv && s[l] >= 0) ? ld16(a.gv + go) : z;
  }
  float fq[8] = {0}, fk[8] = {0}, fv[8] = {0};
#pragma unroll
  for (int l = 0; l < NL; ++l) {
    const float w = 1.0f / (float)(1 << (l * a.shift));
    float g[8];
    unpack8_t<T>(gq[l], g);
#pragma unroll
    for (int e = 0; e < 8; ++e) fq[e] = fmaf(g[e], w, fq[e]);
    unpack8_t<T>(gk[l], g);
#pragma unroll
    for (int e = 0; e < 8; ++e) fk[e] = fmaf(g[e], w, fk[e]);
    unpack8_t<T>(gv[l], g);
#pragma unroll
    for (int e = 0; e < 8; ++e) fv[e] = fmaf(g[e], w, fv[e]);
  }
  if (ROPE) {
    float4 c01, c23;
    rope_freqs8(a.fs, t, LH_D, 8 * l16, c01, c23);
    rope_rotate8<false>(fq, c01, c23);
    rope_rotate8<false>(fk, c01, c23);
  }
  const int64_t o = (int64_t)b * a.ob + (int64_t)t * a.os + (int64_t)h * a.oh + 8 * l16;
  if (a.dq) store16_nt(a.dq + o, pack8_t<T>(fq));
  if (a.dk) store16_nt(a.dk + o, pack8_t<T>(fk));
  if (a.dv) store16_nt(a.dv + o, pack8_t<T>(fv));
}

// Tokens of a pyramid_tile_kernel block, 0 where the walk is taken: the tiles
// win while the walk has at most a wave per CU, with the rotation's extra loads
// up to four.  Cold caches, walk / tiles: 8 heads, L = 3, p = 4, 2048 tokens
// 25.4 / 20.8 us, 4096 26.7 / 26.9, 8192 33.0 / 39.0; with rotation 33.0 / 22.3,
// 8192 46.7 / 43.4, 32768 109 / 122; L = 4 (spans of 64) 8192 66.7 / 48.2.
int tile_tokens(const PyrArgs& a, bool given) {
  if (given || a.cq || a.cmax > PYR_TILE) return 0;
  const int rows = a.D <= 64 ? 32 : 16;
  const int waves = (a.units + rows / 4 - 1) / (rows / 4);
  return waves <= (a.fs ? 4 : 1) * lh_cu_count() ? std::max(rows, a.cmax) : 0;
}

template <typename T, int NL>
int launch_fwd(const PyrArgs& a, bool given, hipStream_t st) {
  if (const int tt = tile_tokens(a, given)) {
    const dim3 grid(a.B * a.H * ((a.S + tt - 1) / tt));
    if (a.fs) {
      using Ln = Lanes<16, true>;
      hipLaunchKernelGGL((pyramid_tile_kernel<BF16, Ln, true>), grid, dim3(256), 0, st, a, tt);
    } else {
      LH_DISPATCH_LANES(a.D, hipLaunchKernelGGL((pyramid_tile_kernel<T, Ln, false>), grid, dim3(256), 0, st, a, tt));
    }
    LH_CHECK_LAUNCH();
    return LH_OK;
  }
  if (a.fs) {  // D == LH_D
    using Ln = Lanes<16, true>;
    hipLaunchKernelGGL((pyramid_fwd_kernel<BF16, Ln, NL, false, true, false>), dim3((a.units + Ln::ROWS - 1) / Ln::ROWS),
                       dim3(256), 0, st, a);
  } else {
    LH_DISPATCH_LANES(a.D, {
      const dim3 grid((a.units + Ln::ROWS - 1) / Ln::ROWS);
      if (a.cq && given)
        hipLaunchKernelGGL((pyramid_fwd_kernel<T, Ln, NL, true, false, true>), grid, dim3(256), 0, st, a);
      else if (a.cq)
        hipLaunchKernelGGL((pyramid_fwd_kernel<T, Ln, NL, false, false, true>), grid, dim3(256), 0, st, a);
      else if (given)
        hipLaunchKernelGGL((pyramid_fwd_kernel<T, Ln, NL, true, false, false>), grid, dim3(256), 0, st, a);
      else
        hipLaunchKernelGGL((pyramid_fwd_kernel<T, Ln, NL, false, false, false>), grid, dim3(256), 0, st, a);
    });
  }
  LH_CHECK_LAUNCH();
  return LH_OK;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

namespace {

int pyramid_fwd_impl(const void* xq, const void* xk, const void* xv, int64_t sb, int64_t ss, int64_t sh,
                     const float* freqs, void* rq, void* rk, int64_t rb, int64_t rs, int64_t rh,
                     void* pq, void* pk, void* pv, int64_t pb, int64_t ps, int64_t ph,
                     float* scores_qk, float* scores_kq, int B, int S, int H, int D, int L, int p,
                     bool given, int dtype, void* stream, void* const* cat = nullptr) {
  if (!lanes_supported(D) || (freqs && D != LH_D)) return LH_ERR_UNSUPPORTED;
  if (!valid_dtype(dtype) || (freqs && dtype != LH_DTYPE_BF16)) return LH_ERR_INVALID_ARG;
  if (!xq || !xk || !xv || !scores_qk || !scores_kq || B <= 0 || H <= 0 || S <= 0) return LH_ERR_INVALID_ARG;
  const int shift = ilog2_exact(p);
  if (shift <= 0 || L < 1) return LH_ERR_INVALID_ARG;
  if (L > 6) return LH_ERR_UNSUPPORTED;
  if (L > 1 && (!pq || !pk || !pv)) return LH_ERR_INVALID_ARG;
  if ((sb | ss | sh) % 8 || (L > 1 && (pb | ps | ph) % 8)) return LH_ERR_INVALID_ARG;
  if (!aligned16(xq) || !aligned16(xk) || !aligned16(xv) || (L > 1 && (!aligned16(pq) || !aligned16(pk) || !aligned16(pv))))
    return LH_ERR_INVALID_ARG;
  if (freqs && (!rq || !rk || !aligned16(freqs) || !aligned16(rq) || !aligned16(rk) || (rb | rs | rh) % 8))
    return LH_ERR_INVALID_ARG;
  Pyramid g;
  if (!make_pyramid(S, L, p, &g)) return LH_ERR_INVALID_ARG;
  PyrArgs a{};
  a.xq = (const bf16_t*)xq; a.xk = (const bf16_t*)xk; a.xv = (const bf16_t*)xv;
  a.sb = sb; a.ss = ss; a.sh = sh;
  a.pq = (bf16_t*)pq; a.pk = (bf16_t*)pk; a.pv = (bf16_t*)pv;
  a.pb = pb; a.ps = ps; a.ph = ph;
  a.sqk = scores_qk; a.skq = scores_kq;
  a.fs = freqs; a.rq = (bf16_t*)rq; a.rk = (bf16_t*)rk;
  a.rb = rb; a.rs = rs; a.rh = rh;
  if (cat) {
    for (int i = 0; i < 5; ++i)
      if (!cat[i] || (i < 3 && !aligned16(cat[i]))) return LH_ERR_INVALID_ARG;
    if ((pb | ps | ph) % 8) return LH_ERR_INVALID_ARG;
    a.cq = (bf16_t*)cat[0]; a.ck = (bf16_t*)cat[1]; a.cv = (bf16_t*)cat[2];
    a.hq = (bf16_t*)cat[3]; a.hk = (bf16_t*)cat[4];
  }
  a.B = B; a.S = S; a.H = H; a.D = D; a.L = L; a.shift = shift; a.S_tot = g.total;
  a.cmax = ipow(p, L - 1);
  if (a.cmax > 4096) return LH_ERR_UNSUPPORTED;
  a.nspan = (S + a.cmax - 1) / a.cmax;
  const long long units = (long long)B * a.nspan * H;
  if (units > (1LL << 30)) return LH_ERR_UNSUPPORTED;
  a.units = (int)units;
  for (int l = 1; l <= L; ++l) { a.off[l] = g.off[l]; a.len[l] = g.len[l]; }
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  int rc = LH_OK;
  LH_DISPATCH_DTYPE(dtype, switch (L - 1) {
    case 0: rc = launch_fwd<T, 0>(a, given, st); break;
    case 1: rc = launch_fwd<T, 1>(a, given, st); break;
    case 2: rc = launch_fwd<T, 2>(a, given, st); break;
    case 3: rc = launch_fwd<T, 3>(a, given, st); break;
    case 4: rc = launch_fwd<T, 4>(a, given, st); break;
    default: rc = launch_fwd<T, 5>(a, given, st); break;
  });
  return rc;
}

template <typename T, typename Ln, bool ROPE>
void launch_bwd(const PyrBwdArgs& a, dim3 grid, hipStream_t st) {
  const dim3 blk(256);
  switch (a.L) {
    case 1: hipLaunchKernelGGL((pyramid_bwd_kernel<T, Ln, 1, ROPE>), grid, blk, 0, st, a); break;
    case 2: hipLaunchKernelGGL((pyramid_bwd_kernel<T, Ln, 2, ROPE>), grid, blk, 0, st, a); break;
    case 3: hipLaunchKernelGGL((pyramid_bwd_kernel<T, Ln, 3, ROPE>), grid, blk, 0, st, a); break;
    case 4: hipLaunchKernelGGL((pyramid_bwd_kernel<T, Ln, 4, ROPE>), grid, blk, 0, st, a); break;
    case 5: hipLaunchKernelGGL((pyramid_bwd_kernel<T, Ln, 5, ROPE>), grid, blk, 0, st, a); break;
    case 6: hipLaunchKernelGGL((pyramid_bwd_kernel<T, Ln, 6, ROPE>), grid, blk, 0, st, a); break;
    case 7: hipLaunchKernelGGL((pyramid_bwd_kernel<T, Ln, 7, ROPE>), grid, blk, 0, st, a); break;
    default: hipLaunchKernelGGL((pyramid_bwd_kernel<T, Ln, 8, ROPE>), grid, blk, 0, st, a); break;
  }
}

int pyramid_bwd_impl(const void* gq, const void* gk, const void* gv, int64_t gb, int64_t gh, int64_t gs,
                     const int32_t* inverse, const float* freqs, void* dxq, void* dxk, void* dxv, int64_t ob,
                     int64_t os, int64_t oh, int B, int S, int H, int D, int L, int p, int dtype, void* stream) {
  if (!lanes_supported(D) || (freqs && D != LH_D)) return LH_ERR_UNSUPPORTED;
  if (B <= 0 || H <= 0 || S <= 0 || L < 1 || L > 8) return LH_ERR_INVALID_ARG;
  if (!valid_dtype(dtype) || (freqs && dtype != LH_DTYPE_BF16)) return LH_ERR_INVALID_ARG;
  const int shift = ilog2_exact(p);
  if (shift <= 0) return LH_ERR_INVALID_ARG;
  if ((gq != nullptr) != (dxq != nullptr) || (gk != nullptr) != (dxk != nullptr) || (gv != nullptr) != (dxv != nullptr))
    return LH_ERR_INVALID_ARG;
  if ((gb | gh | gs) % 8 || (ob | os | oh) % 8) return LH_ERR_INVALID_ARG;
  for (const void* x : {gq, gk, gv, (const void*)dxq, (const void*)dxk, (const void*)dxv})
    if (x && !aligned16(x)) return LH_ERR_INVALID_ARG;
  if (freqs && !aligned16(freqs)) return LH_ERR_INVALID_ARG;
  Pyramid g;
  if (!make_pyramid(S, L, p, &g)) return LH_ERR_INVALID_ARG;
  PyrBwdArgs a{};
  a.gq = (const bf16_t*)gq; a.gk = (const bf16_t*)gk; a.gv = (const bf16_t*)gv;
  a.gb = gb; a.gh = gh; a.gs = gs; a.inv = inverse;
  a.dq = (bf16_t*)dxq; a.dk = (bf16_t*)dxk; a.dv = (bf16_t*)dxv;
  a.ob = ob; a.os = os; a.oh = oh; a.fs = freqs;
  a.B = B; a.S = S; a.H = H; a.D = D; a.L = L; a.shift = shift; a.S_tot = g.total;
  for (int l = 1; l <= L; ++l) { a.off[l] = g.off[l]; a.len[l] = g.len[l]; }
  a.rows = (long long)B * S * H;
  const int rows = D <= 64 ? 32 : 16;
  a.chunks = (S + rows - 1) / rows;
  const long long blocks = (long long)B * H * a.chunks;
  if (blocks > 2147483647LL) return LH_ERR_UNSUPPORTED;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (freqs)
    launch_bwd<BF16, Lanes<16, true>, true>(a, dim3((unsigned)blocks), st);
  else
    LH_DISPATCH_DTYPE(dtype, LH_DISPATCH_LANES(D, (launch_bwd<T, Ln, false>(a, dim3((unsigned)blocks), st))));
  LH_CHECK_LAUNCH();
  return LH_OK;
}

}  // namespace

extern "C" int lh_pyramid_fwd_nd(const void* xq, const void* xk, const void* xv, int64_t sb, int64_t ss, int64_t sh,
                                 void* pq, void* pk, void* pv, int64_t pb, int64_t ps, int64_t ph, float* scores_qk,
                                 float* scores_kq, int B, int S, int H, int D, int L, int p, int base_scores_given,
                                 int dtype, void* stream) {
  return pyramid_fwd_impl(xq, xk, xv, sb, ss, sh, nullptr, nullptr, nullptr, 0, 0, 0, pq, pk, pv, pb, ps, ph,
                          scores_qk, scores_kq, B, S, H, D, L, p, base_scores_given != 0, dtype, stream);
}

extern "C" int lh_pyramid_fwd(const void* xq, const void* xk, const void* xv, int64_t sb, int64_t ss, int64_t sh,
                              void* pq, void* pk, void* pv, int64_t pb, int64_t ps, int64_t ph, float* scores_qk,
                              float* scores_kq, int B, int S, int H, int D, int L, int p, int base_scores_given,
                              int dtype, void* stream) {
  if (D != LH_D) return LH_ERR_UNSUPPORTED;
  return lh_pyramid_fwd_nd(xq, xk, xv, sb, ss, sh, pq, pk, pv, pb, ps, ph, scores_qk, scores_kq, B, S, H, D, L, p,
                           base_scores_given, dtype, stream);
}

extern "C" int lh_pyramid_cat(const void* xq, const void* xk, const void* xv, int64_t sb, int64_t ss, int64_t sh,
                              void* cq, void* ck, void* cv, int64_t cb, int64_t cs, int64_t ch, float* scores_qk,
                              float* scores_kq, void* row_qk, void* row_kq, int B, int S, int H, int D, int L, int p,
                              int base_scores_given, int dtype, void* stream) {
  if (!cq || !ck || !cv || S <= 0) return LH_ERR_INVALID_ARG;
  void* const cat[5] = {cq, ck, cv, row_qk, row_kq};
  bf16_t* pool[3];
  for (int i = 0; i < 3; ++i) pool[i] = (bf16_t*)cat[i] + (int64_t)S * cs;  // the pooled rows follow the base rows
  return pyramid_fwd_impl(xq, xk, xv, sb, ss, sh, nullptr, nullptr, nullptr, 0, 0, 0, pool[0], pool[1], pool[2], cb, cs,
                          ch, scores_qk, scores_kq, B, S, H, D, L, p, base_scores_given != 0, dtype, stream, cat);
}

extern "C" int lh_rope_pyramid_fwd(const void* xq, const void* xk, const void* xv, int64_t sb, int64_t ss,
                                   int64_t sh, const float* freqs, void* rq, void* rk, int64_t rb, int64_t rs,
                                   int64_t rh, void* pq, void* pk, void* pv, int64_t pb, int64_t ps, int64_t ph,
                                   float* scores_qk, float* scores_kq, int B, int S, int H, int D, int L, int p,
                                   void* stream) {
  if (!freqs) return LH_ERR_INVALID_ARG;
  return pyramid_fwd_impl(xq, xk, xv, sb, ss, sh, freqs, rq, rk, rb, rs, rh, pq, pk, pv, pb, ps, ph, scores_qk,
                          scores_kq, B, S, H, D, L, p, false, LH_DTYPE_BF16, stream);
}

extern "C" int lh_pyramid_bwd_nd(const void* gq, const void* gk, const void* gv, int64_t gb, int64_t gh, int64_t gs,
                                 const int32_t* inverse, void* dxq, void* dxk, void* dxv, int B, int S, int H, int D,
                                 int L, int p, int dtype, void* stream) {
  const int64_t oh = D, os = (int64_t)H * D, ob = (int64_t)S * os;
  return pyramid_bwd_impl(gq, gk, gv, gb, gh, gs, inverse, nullptr, dxq, dxk, dxv, ob, os, oh, B, S, H, D, L, p,
                          dtype, stream);
}

extern "C" int lh_pyramid_bwd(const void* gq, const void* gk, const void* gv, int64_t gb, int64_t gh, int64_t gs,
                              const int32_t* inverse, void* dxq, void* dxk, void* dxv, int B, int S, int H, int D,
                              int L, int p, int dtype, void* stream) {
  if (D != LH_D) return LH_ERR_UNSUPPORTED;
  return lh_pyramid_bwd_nd(gq, gk, gv, gb, gh, gs, inverse, dxq, dxk, dxv, B, S, H, D, L, p, dtype, stream);
}

extern "C" int lh_pyramid_rope_bwd(const void* gq, const void* gk, const void* gv, int64_t gb, int64_t gh,
                                   int64_t gs, const int32_t* inverse, const float* freqs, void* dxq, void* dxk,
                                   void* dxv, int64_t ob, int64_t os, int64_t oh, int B, int S, int H, int D, int L,
                                   int p, void* stream) {
  if (!freqs) return LH_ERR_INVALID_ARG;
  return pyramid_bwd_impl(gq, gk, gv, gb, gh, gs, inverse, freqs, dxq, dxk, dxv, ob, os, oh, B, S, H, D, L, p,
                          LH_DTYPE_BF16, stream);
}
