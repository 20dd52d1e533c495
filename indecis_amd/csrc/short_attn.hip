// short_attn.hip — the QKV projection, Attn8.Prepare and the attention of
// one head in one workgroup, for batches whose sequences have at most 128
// tokens.
//
// Replaces qkv_attn.hip and attn_main_kernel (attention_i8.hip) for such
// batches, with the same arithmetic: the int8 GEMM of the sequence's rows by
// the head's 192 weight rows, the reference's dequantisation, RoPE on Q and
// K, Q quantised per row with 1/sqrt(D) folded into its scale
// (attention8.go:211-220), K centred on its mean — 64 float32 sums in key
// order — and quantised per key (:224-251), V quantised per dimension
// (:259-279), then Attend (:298-376): the row max of the valid scores, P =
// RNE(255 exp(s - max)), O = (P . V) / sum P with exact int32 sums.
//
// Why: with few tokens both kernels were latency: 9.5 us and 6.2 us a layer
// for a sequence of 24 tokens, one row block on one wave of eight, Q, K and V
// through HBM between them.
//
// 12 waves: Q, K and V take 4 each; RT is the row blocks of 32 of the longest
// sequence. RT 1: the 4 waves share the depth of the head's 64 columns; 2: 2
// a row block share it; 4: one a row block. Q and K are computed transposed
// (a lane holds a token), V not (a lane holds a dimension), so that every
// later step has what it reduces over in a lane's registers. The scores of a
// query block are dealt to NG waves by accumulator groups, each wave
// computing the block's S^T tiles itself.
#include <type_traits>

#include "ixh_device.h"
#include "ixh_internal.h"

namespace ixh {

namespace {

constexpr int D = 64, NXCD = 8;
constexpr int FLD = 68;  // floats a row of the float32 Q and K
constexpr int BLD = 80;  // bytes a row of the int8 Q and K

template <int RT>
struct Shape {
  static constexpr int KS = 4 / RT;            // waves sharing a row block's depth
  static constexpr int NG = RT == 4 ? 2 : 4;   // waves sharing a query block's scores
  static constexpr int R = 32 * RT;            // rows
  static constexpr int VLD = R + 16;           // bytes a dimension of V^T
  // LDS: partial sums, then over them the float32 Q and K
  static constexpr int PART = KS > 1 ? 12 * 2 * 4 * 64 * 16 : 0;
  static constexpr int SLABS = 2 * R * FLD * 4;
  static constexpr int QKV = PART + SLABS;
  static constexpr int SMEM = QKV + 2 * R * BLD + D * VLD + RT * RT * 64 * 16;
};

// The LayerNorm variant's LDS past Shape<1>'s: the int8 rows as MFMA operands
// (half a K step is 32 rows x 16 bytes, padded by a bank group's 16), gamma.
template <int KT>
struct LnShape {
  static constexpr int H = 32 * KT, LD = H + 8, HALF = 528, KB = 2 * HALF;
  static constexpr int SMEM = Shape<1>::SMEM + KT * KB + 4 * H;
  static_assert(4 * 32 * LD <= Shape<1>::QKV, "the float32 rows under the partial sums");
};

// LNV: -1, or (one row block) the lane width of the LayerNorm and quantisation
// of the sequence's rows done first by each head's workgroup, 32 threads a row,
// the weight loads in flight meanwhile. us a layer, the LayerNorm kernel and this
// one, then both in one: hidden 768, 24 rows 13.6 and 11.7; 384, 15 rows 12.7
// and 9.5; 256, 64 sequences of 15 12.4 and 9.8.
template <int KT, int RT, int LNV>
__global__ __launch_bounds__(768) void short_attn_kernel(GemmArgs g, AttnArgs a, ShortLn ln) {
  using S = Shape<RT>;
  constexpr bool LN = LNV >= 0;
  static_assert(!LN || RT == 1, "one row block");
  constexpr int KS = S::KS, GO = 4 / KS, KW = KT / KS, R = S::R, VLD = S::VLD, NG = S::NG;
  constexpr int PF = KW <= 6 ? KW : 4;  // K steps in flight
  static_assert(KT % KS == 0 && KW % PF == 0, "depth");
  extern __shared__ __attribute__((aligned(1024))) int8_t smem[];
  int4 *const part_s = (int4 *)smem;                   // [12 waves][2 tiles][4 groups][64]
  float *const qf = (float *)(smem + S::PART), *const kf = qf + R * FLD;
  int8_t *const qq = smem + S::QKV, *const kq = qq + R * BLD, *const vt = kq + R * BLD;
  int *const pb = (int *)(vt + D * VLD);               // P: [RT query blocks][RT key blocks][64 lanes][4]
  __shared__ __attribute__((aligned(16))) float mean_s[D], vs_s[D], sq_s[R], ks_s[R];
  __shared__ float vmax_s[4][D], mx_s[RT][NG][64], om_s[2][R];
  __shared__ int vsum_s[D], psum_s[R];
  __shared__ float lmean_s[LN ? 32 : 1], lrstd_s[LN ? 32 : 1], sa_s[LN ? 32 : 1];
  using SL = LnShape<KT>;
  float *const xs = (float *)smem, *const gamma_s = (float *)(smem + S::SMEM + KT * SL::KB);
  int8_t *const panel = smem + S::SMEM;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, fh = lane >> 5;
  // item = head * B + sequence; each XCD takes a contiguous run of items, so
  // that a head's weights are read by one L2
  const int per = (a.B * a.nh + NXCD - 1) / NXCD;
  const int item = (int)(blockIdx.x % NXCD) * per + (int)(blockIdx.x / NXCD);
  if ((int)(blockIdx.x / NXCD) >= per || item >= a.B * a.nh) return;
  const int h = item / a.B, b = item - h * a.B;
  const int base = a.offs[b], n = a.offs[b + 1] - base;
  if (n == 0) return;
  const int part = wave >> 2, sub = wave & 3;          // Q, K, V; the wave of its four
  const int rt = RT == 1 ? 0 : sub / KS, ks = RT == 4 ? 0 : sub % KS;
  if (tid < D) vsum_s[tid] = 0;
  if (tid < R) psum_s[tid] = 0;

  // ---- the products: rows 32 rt .. of the sequence by the head's 64 rows of
  // Q, K or V, K steps ks*KW .. ----
  const int tok = min(32 * rt + fr, n - 1);            // this lane's row (past n: row n-1)
  const int wrow = part * a.H + h * D;
  // weight rows: transposed (Q, K) so that accumulator r is channel 16 fh + r
  const int lw = part == 2 ? fr : 16 * ((fr >> 2) & 1) + 4 * (fr >> 3) + (fr & 3);
  // a lane's byte offsets in VGPRs, a K step's in SGPRs
  const auto wrs = buf_rsrc(g.Bk, (uint32_t)KT * g.Np * 32), xrs = buf_rsrc(g.Ak, (uint32_t)KT * g.ak_rows * 32);
  const uint32_t wvo = (uint32_t)(wrow + lw) * 32 + 16 * fh, xvo = (uint32_t)(base + tok) * 32 + 16 * fh;
  const uint32_t wst = (uint32_t)g.Np * 32, xst = (uint32_t)g.ak_rows * 32;
  if constexpr (LN) {  // the float32 rows, 24 at a time (as many as the threads hold)
    const int lr = tid >> 5, lc = 4 * (tid & 31);
    float4 v[SL::H / 128];
    for (int r = lr; r - lr < n; r += 24) {
      const float *xp = ln.x + (size_t)(base + min(r, n - 1)) * SL::H + lc;
#pragma unroll
      for (int u = 0; u < SL::H / 128; u++) v[u] = *(const float4 *)(xp + 128 * u);
      if (r < 32) {
#pragma unroll
        for (int u = 0; u < SL::H / 128; u++) *(float4 *)&xs[r * SL::LD + lc + 128 * u] = v[u];
      }
    }
    if (tid < SL::H / 4) *(float4 *)&gamma_s[4 * tid] = *(const float4 *)(ln.gamma + 4 * tid);
  }
  v4i w[PF][2], x[PF];
  auto load = [&](int k, int s) {
    const uint32_t kk = ks * KW + k;
    if constexpr (!LN) x[s] = __builtin_amdgcn_raw_buffer_load_b128(xrs, xvo, __builtin_amdgcn_readfirstlane(kk * xst), 0);
    w[s][0] = __builtin_amdgcn_raw_buffer_load_b128(wrs, wvo, __builtin_amdgcn_readfirstlane(kk * wst), 0);
    w[s][1] = __builtin_amdgcn_raw_buffer_load_b128(wrs, wvo + 1024, __builtin_amdgcn_readfirstlane(kk * wst), 0);
  };
#pragma unroll
  for (int k = 0; k < PF; k++) load(k, k);
  // what the dequantisation needs: with one row block loaded here, its
  // latency under the products'; with more, after them (registers)
  float4 pcos[GO], psin[GO], psb[2][GO];
  float psa[GO][4], vsb[2], vzc[2];
  int vc1[2];
  auto constants = [&] {
    if (part < 2) {
      if constexpr (!LN) psa[0][0] = g.sa[base + tok];
#pragma unroll
      for (int q = 0; q < GO; q++) {
        const int d0 = 16 * fh + 4 * (GO * ks + q);
        pcos[q] = *(const float4 *)(g.rope_cos + (size_t)tok * 32 + d0);
        psin[q] = *(const float4 *)(g.rope_sin + (size_t)tok * 32 + d0);
        psb[0][q] = *(const float4 *)(g.sb + wrow + d0);
        psb[1][q] = *(const float4 *)(g.sb + wrow + d0 + 32);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int ch = wrow + 32 * j + fr;
        vsb[j] = g.sb[ch];
        vzc[j] = g.zc[ch];
        vc1[j] = g.c128[ch];
      }
#pragma unroll
      for (int q = 0; q < GO; q++)
#pragma unroll
        for (int u = 0; u < 4; u++)  // rows past n: row n-1 again
          if constexpr (!LN) psa[q][u] = g.sa[base + min(32 * rt + 8 * (GO * ks + q) + 4 * fh + u, n - 1)];
    }
  };
  if constexpr (RT == 1) constants();
  if constexpr (LN) {
    static_assert(KW == PF, "every weight load in flight");
    lds_barrier();
    if (tid < ln_chain_threads<LNV>(n)) ln_chains<SL::H, LNV, true>(xs, SL::LD, tid, lane, n, ln.eps, lmean_s, lrstd_s);
    lds_barrier();
    const int lc = 4 * (tid & 31);
    for (int r = tid >> 5; r < n; r += 24) {
      const float mean = lmean_s[r], rstd = lrstd_s[r];
      float4 v[SL::H / 128];
      float mx = 0.f;
#pragma unroll
      for (int u = 0; u < SL::H / 128; u++) {
        const float4 t = *(const float4 *)&xs[r * SL::LD + lc + 128 * u], gm = *(const float4 *)&gamma_s[lc + 128 * u];
        v[u] = make_float4(((t.x - mean) * rstd) * gm.x, ((t.y - mean) * rstd) * gm.y, ((t.z - mean) * rstd) * gm.z,
                           ((t.w - mean) * rstd) * gm.w);
        mx = amax(amax(amax(amax(mx, v[u].x), v[u].y), v[u].z), v[u].w);
      }
#pragma unroll
      for (int o = 1; o < 32; o <<= 1) mx = __builtin_fmaxf(mx, __shfl_xor(mx, o));
      float sc = 0.f, inv = 0.f;
      if (mx != 0.f) {  // quantizeA: s = max/127, inv = 1/s (int8.go:175-183)
        sc = mx / 127.0f;
        inv = 1.0f / sc;
      }
      if (lc == 0) sa_s[r] = sc;
#pragma unroll
      for (int u = 0; u < SL::H / 128; u++) {
        const int col = lc + 128 * u;
        *(int *)(panel + (col >> 5) * SL::KB + ((col >> 4) & 1) * SL::HALF + r * 16 + (col & 15)) = pack4(v[u], inv);
      }
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < PF; k++) x[k] = *(const v4i *)(panel + (ks * KW + k) * SL::KB + fh * SL::HALF + 16 * tok);
    if (part < 2) {
      psa[0][0] = sa_s[tok];
    } else {
#pragma unroll
      for (int q = 0; q < GO; q++)
#pragma unroll
        for (int u = 0; u < 4; u++) psa[q][u] = sa_s[min(8 * (GO * ks + q) + 4 * fh + u, n - 1)];
    }
  }
  const bool small = g.small;
  v16i acc[2] = {};
  auto products = [&](auto vpart) {
    // (not unrolled further: the loads would be hoisted past the registers)
#pragma unroll 1
    for (int k0 = 0; k0 < KW; k0 += PF)
#pragma unroll
      for (int u = 0; u < PF; u++) {
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[j] = decltype(vpart)::value ? mfma32(x[u], w[u][j], acc[j]) : mfma32(w[u][j], x[u], acc[j]);
        if (KW > PF) load(min(k0 + PF + u, KW - 1), u);  // past the last step: it again, unused
      }
  };
  if (part == 2) products(std::true_type{});
  else products(std::false_type{});
  int4 sum[2][GO];
  if constexpr (KS > 1) {
    int4 *const ps = part_s + (size_t)(wave - ks) * (2 * 4 * 64);  // [KS][4][64] a tile
    put_sums<KS>(ps, ks, lane, acc[0]);
    put_sums<KS>(ps + KS * 256, ks, lane, acc[1]);
    __syncthreads();
    gather_sums<KS>(ps, ks, lane, acc[0], sum[0]);
    gather_sums<KS>(ps + KS * 256, ks, lane, acc[1], sum[1]);
  } else {
    __syncthreads();  // vsum_s, psum_s
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) sum[j][q] = int4{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
  }

  // ---- dequantisation; RoPE and the float32 Q and K; max |V| ----
  if constexpr (RT > 1) constants();
  float v[2][GO][4];  // V: rows 8 (GO ks + q) + 4 fh + u of the block, dimension 32 j + fr
  if (part < 2) {
    const float sa = psa[0][0];
    float *const dst = (part ? kf : qf) + (32 * rt + fr) * FLD;
#pragma unroll
    for (int q = 0; q < GO; q++) {
      const int d0 = 16 * fh + 4 * (GO * ks + q), ch = wrow + d0;
      const float4 c = pcos[q], s = psin[q];
      const float4 x1 = deq4(sum[0][q], small, g.c128 + ch, g.zc + ch, psb[0][q], sa);
      const float4 x2 = deq4(sum[1][q], small, g.c128 + ch + 32, g.zc + ch + 32, psb[1][q], sa);
      // linalg.Rope (vec_simd.go:408-425): x1' = x1*c - x2*s, x2' = x2*c + x1*s
      *(float4 *)(dst + d0) = make_float4(x1.x * c.x - x2.x * s.x, x1.y * c.y - x2.y * s.y, x1.z * c.z - x2.z * s.z, x1.w * c.w - x2.w * s.w);
      *(float4 *)(dst + 32 + d0) = make_float4(x2.x * c.x + x1.x * s.x, x2.y * c.y + x1.y * s.y, x2.z * c.z + x1.z * s.z, x2.w * c.w + x1.w * s.w);
    }
  } else {
    float vm[2] = {0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; j++) {
#pragma unroll
      for (int q = 0; q < GO; q++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
          // rows past n are row n-1 again: they leave the maximum as it is
          const int t = u == 0 ? sum[j][q].x : u == 1 ? sum[j][q].y : u == 2 ? sum[j][q].z : sum[j][q].w;
          v[j][q][u] = small ? ((float)t * vsb[j]) * psa[q][u] : deq(t + vc1[j], vzc[j], vsb[j], psa[q][u]);
          vm[j] = amax(vm[j], v[j][q][u]);
        }
      vm[j] = __builtin_fmaxf(vm[j], __shfl_xor(vm[j], 32));
      if (fh == 0) vmax_s[sub][32 * j + fr] = vm[j];
    }
  }
  __syncthreads();

  // int8 rows of the float32 rows src (n of them, 8 threads a row), centred
  // on mu when not null; the row scales times f
  auto quant_rows = [&](const float *src, const float *mu, int8_t *dst, float *sc_s, float f) {
    const int t = tid & 255;
#pragma unroll
    for (int r0 = 0; r0 < R; r0 += 32) {
      const int r = r0 + (t >> 3), c = 8 * (t & 7);
      float4 p0 = *(const float4 *)(src + r * FLD + c), p1 = *(const float4 *)(src + r * FLD + c + 4);
      if (mu) {
        const float4 m0 = *(const float4 *)(mu + c), m1 = *(const float4 *)(mu + c + 4);
        p0 = make_float4(p0.x - m0.x, p0.y - m0.y, p0.z - m0.z, p0.w - m0.w);
        p1 = make_float4(p1.x - m1.x, p1.y - m1.y, p1.z - m1.z, p1.w - m1.w);
      }
      float mx = amax(amax(amax(amax(amax(amax(amax(amax(0.f, p0.x), p0.y), p0.z), p0.w), p1.x), p1.y), p1.z), p1.w);
#pragma unroll
      for (int o = 1; o < 8; o <<= 1) mx = __builtin_fmaxf(mx, __shfl_xor(mx, o));
      float sc = 0.f, inv = 0.f;
      if (mx != 0.f) {
        sc = mx / 127.0f;
        inv = 1.0f / sc;
      }
      *(int2 *)(dst + r * BLD + c) = int2{pack4(p0, inv), pack4(p1, inv)};
      if ((t & 7) == 0) sc_s[r] = f == 0.f ? sc : sc * f;
    }
  };
  if (part == 0) {
    quant_rows(qf, nullptr, qq, sq_s, g.attn_scale);
  } else if (part == 1) {
    if (sub == 0) {  // the K mean: one lane a dimension, in key order
      float ksum = 0.f;
      const float *col = kf + lane;
      int r = 0;
      for (; r + 16 <= n; r += 16) {
        float t[16];
#pragma unroll
        for (int u = 0; u < 16; u++) t[u] = col[(r + u) * FLD];
#pragma unroll
        for (int u = 0; u < 16; u++) ksum = ksum + t[u];
      }
      float t[16];  // the rest: rows past n read (in LDS), not added
#pragma unroll
      for (int u = 0; u < 15; u++) t[u] = col[min(r + u, R - 1) * FLD];
#pragma unroll
      for (int u = 0; u < 15; u++)
        if (r + u < n) ksum = ksum + t[u];
      mean_s[lane] = ksum * (1.0f / (float)n);  // Scale(mean, 1/n)
    }
  } else {
    // V's scales (attention8.go:262-269), its int8 values transposed, their sums
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int d = 32 * j + fr;
      float vs = __builtin_fmaxf(__builtin_fmaxf(vmax_s[0][d], vmax_s[1][d]), __builtin_fmaxf(vmax_s[2][d], vmax_s[3][d]));
      float vi = 0.f;
      if (vs > 0.f) {
        vs = vs / 127.0f;
        vi = 1.0f / vs;
      }
      if (sub == 0 && fh == 0) vs_s[d] = vs;
      int total = 0;
#pragma unroll
      for (int q = 0; q < GO; q++) {
        const int gq = GO * ks + q, lim = n - (32 * rt + 8 * gq + 4 * fh);  // keys of the four in the sequence
        const unsigned keep = lim >= 4 ? 0xffffffffu : lim <= 0 ? 0u : (1u << (8 * lim)) - 1u;
        const int wv = (int)((unsigned)pack4(make_float4(v[j][q][0], v[j][q][1], v[j][q][2], v[j][q][3]), vi) & keep);
        // a key block's dwords in the order of the S^T accumulator rows
        *(int *)(vt + d * VLD + 32 * rt + 16 * fh + 4 * gq) = wv;
        total = __builtin_amdgcn_sdot4(wv, 0x01010101, total, false);
      }
      atomicAdd(&vsum_s[d], total);
    }
  }
  __syncthreads();
  if (part == 1) quant_rows(kf, mean_s, kq, ks_s, 0.f);
  __syncthreads();

  // ---- attention: query block wave / NG, accumulator groups of wave % NG ----
  constexpr int GW = 4 / NG;  // groups of 4 keys a wave takes of each key block
  const int qt = wave / NG, gs = wave % NG;
  const bool active = qt < RT && 32 * qt < n;
  const int W = a.window, V = a.lanes;
  const int qi = 32 * qt + fr;  // this lane's query
  const bool qact = qi < n;
  const int cs = W < 0 ? 0 : max(0, qi - W), ce = W < 0 ? n : min(n, qi + W + 1);
  const uint32_t span = qact ? (uint32_t)(ce - cs) : 0u;
  const int ts = V > 0 ? cs + ((ce - cs) / V) * V : cs;  // the exp32 tail (vec_simd.go:258-262)
  const int nkb = (n + 31) / 32;
  float sv[RT][GW][4];
  float m = -__builtin_huge_valf();
  if (active) {
    const v4i q0 = *(const v4i *)(qq + qi * BLD + 16 * fh), q1 = *(const v4i *)(qq + qi * BLD + 32 + 16 * fh);
#pragma unroll
    for (int kb = 0; kb < RT; kb++) {
      if (kb >= nkb) continue;
      const int8_t *kr = kq + (32 * kb + fr) * BLD + 16 * fh;
      v16i s = mfma32(*(const v4i *)kr, q0, v16i{});
      s = mfma32(*(const v4i *)(kr + 32), q1, s);
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (q / GW == gs) {  // wave-uniform
          const float4 k4 = *(const float4 *)(ks_s + 32 * kb + 8 * q + 4 * fh);
          const float kk[4] = {k4.x, k4.y, k4.z, k4.w};
#pragma unroll
          for (int u = 0; u < 4; u++) {
            sv[kb][q % GW][u] = (float)s[4 * q + u] * kk[u];
            if ((uint32_t)(32 * kb + 8 * q + 4 * fh + u - cs) < span) m = __builtin_fmaxf(m, sv[kb][q % GW][u]);
          }
        }
    }
    m = __builtin_fmaxf(m, __shfl_xor(m, 32));
    mx_s[qt][gs][lane] = m;
  }
  __syncthreads();
  if (active) {
    // max_j f32(x_j * sq) = f32(max_j x_j * sq): rounding is monotone, sq >= 0
#pragma unroll
    for (int q = 0; q < NG; q++) m = __builtin_fmaxf(m, mx_s[qt][q][lane]);
    const float sq = sq_s[qi];
    m = m * sq;
    unsigned ps = 0;
#pragma unroll
    for (int kb = 0; kb < RT; kb++) {
      if (kb >= nkb) continue;
#pragma unroll
      for (int q = 0; q < GW; q++) {
        const int g4 = GW * gs + q, j0 = 32 * kb + 8 * g4 + 4 * fh;
        unsigned pw = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
          // P = RNE(255 exp(s - max)): exp255_fast decides away from a
          // half-integer, else the reference formula (attention_i8.hip)
          const float d = sv[kb][q][u] * sq - m;
          const float y = exp255_fast(d);
          float p = rne(y);
          if (fabsf(y - p) > 0.5f - kExp255Tol) p = rne(((j0 + u >= ts) ? exp32_scalar(d) : exp32_simd(d)) * 255.0f);
          p = (uint32_t)(j0 + u - cs) < span ? p : 0.f;
          pw = __builtin_amdgcn_cvt_pk_u8_f32(p, u, pw);
        }
        ps = __builtin_amdgcn_udot4(pw, 0x01010101u, ps, false);
        pb[((qt * RT + kb) * 64 + lane) * 4 + g4] = (int)(pw ^ 0x80808080u);  // P - 128 as int8
      }
    }
    ps += __shfl_xor(ps, 32);
    if (fh == 0) atomicAdd(&psum_s[qi], (int)ps);
  }
  __syncthreads();
  // O^T = V^T . P^T: wave = (query block, half of the dimensions)
  const int ob = wave >> 1, dt = wave & 1;
  const bool owork = ob < RT && 32 * ob < n;
  const int oq = 32 * ob + fr;
  if (owork) {
    v16i o = {};
#pragma unroll
    for (int kb = 0; kb < RT; kb++) {
      if (kb >= nkb) continue;
      o = mfma32(*(const v4i *)(vt + (32 * dt + fr) * VLD + 32 * kb + 16 * fh), *(const v4i *)(pb + ((ob * RT + kb) * 64 + lane) * 4), o);
    }
    const bool act = oq < n;
    const float sp = act ? 1.0f / (float)psum_s[oq] : 0.f;
    float om = 0.f;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int d0 = 32 * dt + 8 * q + 4 * fh;
      const int4 c = *(const int4 *)(vsum_s + d0);  // 128 sum V: the keys' P were taken less 128
      const float4 vs = *(const float4 *)(vs_s + d0);
      const float4 r = make_float4(((float)(o[4 * q] + 128 * c.x) * vs.x) * sp, ((float)(o[4 * q + 1] + 128 * c.y) * vs.y) * sp,
                                   ((float)(o[4 * q + 2] + 128 * c.z) * vs.z) * sp, ((float)(o[4 * q + 3] + 128 * c.w) * vs.w) * sp);
      om = amax(amax(amax(amax(om, r.x), r.y), r.z), r.w);
      if (act) *(float4 *)(a.ctx + (size_t)(base + oq) * a.H + h * D + d0) = r;
    }
    om = __builtin_fmaxf(om, __shfl_xor(om, 32));
    if (fh == 0) om_s[dt][oq] = om;
  }
  if (a.rmax) {
    __syncthreads();
    if (tid < n) a.rmax[(size_t)(base + tid) * a.nh + h] = __builtin_fmaxf(om_s[0][tid], om_s[1][tid]);
  }
}

template <int KT, int RT, int LNV>
bool launch_one(const GemmArgs &g, const AttnArgs &a, const ShortLn &ln, hipStream_t s) {
  constexpr int shm = LNV < 0 ? Shape<RT>::SMEM : LnShape<KT>::SMEM;
  static PerDevice lds;
  const auto kern = short_attn_kernel<KT, RT, LNV>;
  if (!lds_granted(lds, (const void *)kern, shm)) return false;
  kern<<<NXCD * ((a.B * a.nh + NXCD - 1) / NXCD), 768, shm, s>>>(g, a, ln);
  return true;
}
template <int KT>
bool launch_kt(const GemmArgs &g, const AttnArgs &a, const ShortLn &ln, hipStream_t s) {
  if (ln.x) {
    switch (ln.lanes) {
    case 0: return launch_one<KT, 1, 0>(g, a, ln, s);
    case 4: return launch_one<KT, 1, 4>(g, a, ln, s);
    case 8: return launch_one<KT, 1, 8>(g, a, ln, s);
    default: return launch_one<KT, 1, 16>(g, a, ln, s);
    }
  }
  if (a.max_n <= 32) return launch_one<KT, 1, -1>(g, a, ln, s);
  if (a.max_n <= 64) return launch_one<KT, 2, -1>(g, a, ln, s);
  return launch_one<KT, 4, -1>(g, a, ln, s);
}

}  // namespace

// us a layer of the whole pass, on this kernel and on the two it replaces, by
// rounds of the CUs (a workgroup fills one). At most 32 tokens: hidden 768, 16
// tokens, 1 sequence 32.7 and 41.1, 64 (3 rounds) 59.7 and 65.2, 106 of 4-32
// (5) 88.5 and 91.2, 128 (6) 92.0 and 90.2, 512 (24) 230 and 185; 384, 200 (5)
// 84.7 and 84.3, 512 (12) 133 and 120; 256, 384 (6) 65.8 and 67.8, 512 (8) 77.6
// and 74.3. At most 64, 64 tokens: 768, 1 42.5 and 45.9, 21 (1) 63.4 and 71.9,
// 32 (1.5) 80.9 and 78.5, 42 of 33-64 (2) 81.6 and 85.9, 64 (3) 107 and 102;
// 384, 32 (0.75) 49.4 and 54.2, 85 (2) 80.6 and 81.4, 128 (3) 92.1 and 91.4 (200 121
// and 111); 256, 64 (1) 41.1 and 46.0, 128 (2) 52.1 and 52.5, 200 80.1 and
// 72.2. At most 128, 128 tokens: 768, 1 51.7 and 49.4, 8 (0.4) 63.1 and 61.2, 12
// (0.6) 73.4 and 75.3, 21 (1) 90.6 and 97.2, 32 112 and 102; 384, 1 41.7 and 39.6,
// 42 of 65-128 (1) 78.5 and 81.9; 256, 1 39.2 and 37.7, 64 (1) 53.4 and 55.8. This
// kernel over the two, a pass of 6 layers at 65, 96 and 128 tokens: 768, 0.3 rounds
// 0.99, 1.01 and 1.02, 0.4 0.99, 1.00 and 1.05, 0.5 0.92, 0.96 and 0.97; 384, 0.2
// 0.97, 1.02 and 1.01, 0.3 0.94, 0.98 and 1.00, 0.4 0.94, 0.96 and 0.98; 256, 0.1 0.98,
// 0.96 and 1.00, 0.2 0.97, 0.99 and 0.98, 0.5 0.93, 0.97 and 0.96.
// With another part's kernels beside this pass's, us a pass of 6 layers in two
// parts, on the two and on this kernel, by the rounds of a part: at most 32 tokens
// (16; 32), 256, 3 618 and 564; 653 and 619, 5 748 and 727; 870 and 854, 6 833 and
// 803; 965 and 977; 384, 2.5 (32) 732 and 728, 3 742 and 704; 749 and 770, 3.5 766 and
// 793; 807 and 830; 768, 3 (32) 814 and 840, 4 901 and 934. At most 64 (33; 64): 256,
// 1.5 557 and 530; 589 and 579, 1.75 589 and 561; 616 and 621; 384, 1.25 (64) 726 and
// 700, 1.5 738 and 719; 723 and 738; 768, 1.5 (64) 796 and 815. At most 128 (128): 256,
// 0.5 523 and 482, 1 641 and 644; 384, 0.5 689 and 653, 1 778 and 771, 1.25 838 and
// 900; 768, 0.75 783 and 730, 1 863 and 866, 1.25 886 and 921.
bool short_attn_picked(int Kp, int max_n, int workgroups, bool beside) {
  if (!short_attn_supported(Kp, max_n)) return false;
  const int wg = workgroups, cus = device_cus();
  if (max_n <= 32) {
    if (beside) return 2 * wg <= (Kp == 256 ? 10 : Kp == 384 && max_n <= 16 ? 6 : 5) * cus;
    return wg <= (Kp == 256 ? 6 : 5) * cus;
  }
  if (max_n <= 64) {
    if (beside) return 4 * wg <= (Kp == 256 ? 6 : 5) * cus;
    return wg <= cus || (wg <= 2 * cus && (Kp < 768 || 4 * wg > 7 * cus));
  }
  return wg <= cus && (beside || wg > (Kp == 768 ? 2 * cus / 5 : Kp == 384 ? cus / 4 : cus / 8));
}

bool short_attn_supported(int Kp, int max_n) { return (Kp == 768 || Kp == 384 || Kp == 256) && max_n <= 128; }

// a workgroup fills a CU (154 KB of LDS): one round of them
bool short_attn_ln_supported(int max_n, int workgroups) { return max_n <= 32 && workgroups <= device_cus(); }

bool launch_short_attn(const GemmArgs &g, const AttnArgs &a, const ShortLn &ln, hipStream_t s) {
  if (a.B <= 0) return true;
  if (!short_attn_supported(g.Kp, a.max_n) || !(g.Ak || ln.x)) return false;
  if (ln.x && !short_attn_ln_supported(a.max_n, a.B * a.nh)) return false;
  if (g.Kp == 768) return launch_kt<24>(g, a, ln, s);
  if (g.Kp == 384) return launch_kt<12>(g, a, ln, s);
  return launch_kt<8>(g, a, ln, s);
}

}  // namespace ixh
