// split_rows.hip — the encoder's Wo and MLP products for batches of few
// rows: every product cut into 32-channel tiles over many workgroups, its
// depth over the waves of a workgroup.
//
// Replaces, for such batches, the whole-row kernels of gemm_res.hip and
// mlp_block.hip (infer.go:401-424: MatMul8N of ctx into x, mlp_norm, Wi +
// GeluMul, MatMul8N of g into x, the next attn_norm), with the same
// arithmetic: quantizeA of the input rows (int8.go:160-191), q*w summed in
// int32 by v_mfma_i32_32x32x32_i8, the reference tile's dequantisation
// ((f32(tile) - zc) * sb) * sa, GELU in the FMA form.
//
// Why: a whole-row kernel gives 32 or 64 rows to one workgroup, which then
// streams every weight of the block through one CU; one row costs it as
// much as 64, and a batch of 24 rows ran on one CU of 256. Cut by output
// channel, a weight byte is read by one workgroup per 32 rows, and the
// chip's CUs read different weights.
//
//  res_split_kernel  x[:, tile] += quantizeA(A) . W^T tile: one workgroup
//      per (32 rows, CT tiles of 32 output channels), KS waves a tile, each
//      its part of the depth. A (ctx or g, float32) is quantised into an LDS
//      panel from the row maxima its producer wrote (attention per head,
//      wi_split per 32 columns), so no pass over the row comes before the
//      product.
//  wi_split_kernel   g tile = GeGLU(xn . Wi^T): one workgroup per (32 rows,
//      gated tile of 32 columns), 4 waves over the depth; also max |g| of
//      each row's 32 columns.
//
//  ln_wi_split_kernel  wi_split with mlp_norm before it in the same workgroup,
//      for the fewest rows.
//
// What bounds them: latency at few rows. At 24 rows of hidden 768 (36 and 24
// workgroups) a launch takes 4.9 us (Wi; 7.9 with its LayerNorm), 4.5 us (Wo)
// and 5.9 us (WoMLP), a LayerNorm of its own (ln_rows_kernel, rownorm.hip) 4.8:
// against 25 us (Wo + LayerNorm) and 50 us (the MLP block) on the whole-row
// kernels; a pass of 22 layers 2.07 -> 0.74 ms with short_attn.hip. A wave's
// global loads are all issued before its first MFMA. With more rows, the
// float32 rows read from L2 and the last-level cache by every tile's
// workgroup: at 4,096 rows WoMLP took 69 us, Wo 47, Wi 26 before
// the arrangement for many rows (kManyBlocks).
//
// The products are transposed as in mlp_block.hip (weights the A operand,
// rows the B operand): a lane holds one row and 16 consecutive channels,
// so results leave as float4.
#include <type_traits>

#include "ixh_device.h"
#include "ixh_internal.h"

namespace ixh {

namespace {

constexpr int NXCD = 8;

// the weight row that lane row i loads, so that accumulator r of a lane is
// channel 16*(lane/32) + r of the tile (mlp_block.hip)
__device__ __forceinline__ int perm32(int i) { return 16 * ((i >> 2) & 1) + 4 * (i >> 3) + (i & 3); }

// Row blocks from which the kernels are arranged for many rows (512 rows):
// measured with 4 waves a tile and the tiles dealt to the XCDs, then 2 waves
// a tile, 4 tiles a workgroup (res) and the row blocks dealt to the XCDs, us
// a launch at hidden 768: Wo 5.7 and 6.7 at 256 rows, 9.2 and 7.5 at 768, 47
// and 16 at 4,096 (26 with the dealing alone); WoMLP 6.9 and 7.9, 12.0 and
// 8.7, 69 and 22 (37); Wi 5.5 at 256 rows, 26 and 21 at 4,096 by the dealing.
constexpr int kManyBlocks = 16;

// Workgroup -> (tile, row block); workgroup L runs on XCD L % 8. With few
// row blocks the row blocks of one tile go to one XCD, so that one L2 reads
// the tile's weights; with many the tiles of one row block do, so that its
// float32 rows reach one L2 once (they are most of the traffic). False past
// the last tile or block.
__device__ __forceinline__ bool tile_of(int ntiles, int nblk, int *tile, int *blk) {
  const int i = blockIdx.x / NXCD, x = blockIdx.x % NXCD;
  if (nblk >= kManyBlocks) {
    *blk = x + NXCD * (i / ntiles);
    *tile = i % ntiles;
    return *blk < nblk;
  }
  *tile = x + NXCD * (i / nblk);
  *blk = i % nblk;
  return *tile < ntiles;
}
int tile_grid(int ntiles, int nblk) {
  return nblk >= kManyBlocks ? NXCD * ((nblk + NXCD - 1) / NXCD) * ntiles : NXCD * ((ntiles + NXCD - 1) / NXCD) * nblk;
}

template <int KT>
__global__ __launch_bounds__(256) void wi_split_kernel(SplitArgs a) {
  constexpr int KS = 4, KW = KT / KS;  // waves, K steps of a wave
  static_assert(KT % KS == 0, "depth over the waves");
  __shared__ int4 part[2][KS * 4 * 64];
  __shared__ float mx_s[KS][64];
  const int tid = threadIdx.x, lane = tid & 63, ks = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, fh = lane >> 5;
  int t, blk;
  if (!tile_of(a.n / 64, (a.M + 31) / 32, &t, &blk)) return;
  const int m0 = 32 * blk, row = min(m0 + fr, a.M - 1);  // rows past M: row M-1, never stored
  v4i w[KW][2], x[KW];
  const int8_t *wp = a.Bk + ((size_t)(ks * KW) * a.Np + 64 * t + perm32(fr)) * 32 + 16 * fh;
  const int8_t *xp = a.Ak + ((size_t)(ks * KW) * a.ak_rows + row) * 32 + 16 * fh;
#pragma unroll
  for (int k = 0; k < KW; k++) {
    x[k] = *(const v4i *)(xp + (size_t)k * a.ak_rows * 32);
    w[k][0] = *(const v4i *)(wp + (size_t)k * a.Np * 32);
    w[k][1] = *(const v4i *)(wp + (size_t)k * a.Np * 32 + 1024);
  }
  const float sa = a.sa[row];
  const int ch = 64 * t + 16 * fh + 4 * ks;  // this lane's GELU-input channels (the multiplier's: + 32)
  const float4 sba = *(const float4 *)(a.sb + ch), sbb = *(const float4 *)(a.sb + ch + 32);
  v16i acc[2] = {};
#pragma unroll
  for (int k = 0; k < KW; k++) {
    acc[0] = mfma32(w[k][0], x[k], acc[0]);
    acc[1] = mfma32(w[k][1], x[k], acc[1]);
  }
  put_sums<KS>(part[0], ks, lane, acc[0]);
  put_sums<KS>(part[1], ks, lane, acc[1]);
  __syncthreads();
  int4 ta, tb;
  gather_sums<KS>(part[0], ks, lane, acc[0], &ta);
  gather_sums<KS>(part[1], ks, lane, acc[1], &tb);
  const float4 za = deq4(ta, a.small, a.c128 + ch, a.zc + ch, sba, sa);
  const float4 zb = deq4(tb, a.small, a.c128 + ch + 32, a.zc + ch + 32, sbb, sa);
  const float4 g = make_float4(gelu_fma(za.x) * zb.x, gelu_fma(za.y) * zb.y, gelu_fma(za.z) * zb.z, gelu_fma(za.w) * zb.w);
  if (m0 + fr < a.M) *(float4 *)(a.C + (size_t)row * a.ldc + 32 * t + 16 * fh + 4 * ks) = g;
  mx_s[ks][lane] = amax(amax(amax(amax(0.f, g.x), g.y), g.z), g.w);
  __syncthreads();
  if (tid < 32 && m0 + tid < a.M) {
    float m = 0.f;
#pragma unroll
    for (int q = 0; q < KS; q++) m = __builtin_fmaxf(__builtin_fmaxf(m, mx_s[q][tid]), mx_s[q][32 + tid]);
    a.rmax[(size_t)(m0 + tid) * a.P + t] = m;
  }
}

// wi_split_kernel with the LayerNorm before it (mlp_norm and its quantizeA) in
// the same workgroup: each recomputes it for its 32 rows, 32 threads a row, so
// that no launch and no int8 row stand between x and the product. The weight
// loads of the 4 product waves are in flight during the chains of 4 others. Its
// time is the chains' latency; us of the two kernels and of this: hidden 768 9.9
// and 8.0 at 24 rows, 10.8 and 9.3 at 192; 384 9.5 and 6.6 at 15 rows; 256 9.5
// and 7.1 at 480.
template <int KT, int V>
__global__ __launch_bounds__(1024) void ln_wi_split_kernel(SplitArgs a) {
  constexpr int KS = 4, KW = KT / KS, H = 32 * KT, LD = H + 8, C4 = H / 128;
  constexpr int HALF = 528, KB = 2 * HALF;  // bytes of half a K step (32 rows x 16 and a bank group's 16), a K step
  static_assert(KT % KS == 0 && 2 * KS * 4 * 64 * 16 <= 32 * LD * 4, "depth over the waves, the sums over the rows");
  __shared__ __attribute__((aligned(16))) float xs[32 * LD];
  __shared__ __attribute__((aligned(16))) int8_t panel[KT * KB];
  __shared__ __attribute__((aligned(16))) float gamma_s[H];
  __shared__ float mean_s[32], rstd_s[32], sa_s[32], mx_s[KS][64];
  int4 *const part = (int4 *)xs;  // [2][KS * 4 * 64], once the rows are quantised
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int t, blk;
  if (!tile_of(a.n / 64, (a.M + 31) / 32, &t, &blk)) return;
  const int m0 = 32 * blk, r = tid >> 5, c = tid & 31;
  const float *xp = a.A + (size_t)min(m0 + r, a.M - 1) * a.lda + 4 * c;  // rows past M: row M-1, never stored
  float4 v[C4];
#pragma unroll
  for (int u = 0; u < C4; u++) v[u] = *(const float4 *)(xp + 128 * u);
  if (tid < H / 4) *(float4 *)&gamma_s[4 * tid] = *(const float4 *)(a.gamma + 4 * tid);
#pragma unroll
  for (int u = 0; u < C4; u++) *(float4 *)&xs[r * LD + 4 * (c + 32 * u)] = v[u];
  const int fr = lane & 31, fh = lane >> 5, ks = wave & (KS - 1);
  const int ch = 64 * t + 16 * fh + 4 * ks;  // this lane's GELU-input channels (the multiplier's: + 32)
  v4i w[KW][2];
  float4 sba, sbb;
  if (wave < KS) {
    const int8_t *wp = a.Bk + ((size_t)(ks * KW) * a.Np + 64 * t + perm32(fr)) * 32 + 16 * fh;
#pragma unroll
    for (int k = 0; k < KW; k++) {
      w[k][0] = *(const v4i *)(wp + (size_t)k * a.Np * 32);
      w[k][1] = *(const v4i *)(wp + (size_t)k * a.Np * 32 + 1024);
    }
    sba = *(const float4 *)(a.sb + ch);
    sbb = *(const float4 *)(a.sb + ch + 32);
  }
  lds_barrier();
  const int ct = tid - 64 * KS;
  if (ct >= 0 && ct < ln_chain_threads<V>(32)) ln_chains<H, V, true>(xs, LD, ct, lane, 32, a.eps, mean_s, rstd_s);
  lds_barrier();
  const float mean = mean_s[r], rstd = rstd_s[r];
  float mx = 0.f;
#pragma unroll
  for (int u = 0; u < C4; u++) {
    const float4 x = *(const float4 *)&xs[r * LD + 4 * (c + 32 * u)], g = *(const float4 *)&gamma_s[4 * (c + 32 * u)];
    v[u] = make_float4(((x.x - mean) * rstd) * g.x, ((x.y - mean) * rstd) * g.y, ((x.z - mean) * rstd) * g.z,
                       ((x.w - mean) * rstd) * g.w);
    mx = amax(amax(amax(amax(mx, v[u].x), v[u].y), v[u].z), v[u].w);
  }
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) mx = __builtin_fmaxf(mx, __shfl_xor(mx, o));
  float s = 0.f, inv = 0.f;
  if (mx != 0.f) {  // quantizeA: s = max/127, inv = 1/s (int8.go:175-183)
    s = mx / 127.0f;
    inv = 1.0f / s;
  }
  if (c == 0) sa_s[r] = s;
#pragma unroll
  for (int u = 0; u < C4; u++) {
    const int col = 4 * (c + 32 * u);
    *(int *)(panel + (col >> 5) * KB + ((col >> 4) & 1) * HALF + r * 16 + (col & 15)) = pack4(v[u], inv);
  }
  lds_barrier();
  v16i acc[2] = {};
  if (wave < KS) {
#pragma unroll
    for (int k = 0; k < KW; k++) {
      const v4i x = *(const v4i *)(panel + (ks * KW + k) * KB + fh * HALF + 16 * fr);
      acc[0] = mfma32(w[k][0], x, acc[0]);
      acc[1] = mfma32(w[k][1], x, acc[1]);
    }
    put_sums<KS>(part, ks, lane, acc[0]);
    put_sums<KS>(part + KS * 4 * 64, ks, lane, acc[1]);
  }
  lds_barrier();
  if (wave < KS) {
    int4 ta, tb;
    gather_sums<KS>(part, ks, lane, acc[0], &ta);
    gather_sums<KS>(part + KS * 4 * 64, ks, lane, acc[1], &tb);
    const float sa = sa_s[fr];
    const float4 za = deq4(ta, a.small, a.c128 + ch, a.zc + ch, sba, sa);
    const float4 zb = deq4(tb, a.small, a.c128 + ch + 32, a.zc + ch + 32, sbb, sa);
    const float4 g = make_float4(gelu_fma(za.x) * zb.x, gelu_fma(za.y) * zb.y, gelu_fma(za.z) * zb.z, gelu_fma(za.w) * zb.w);
    if (m0 + fr < a.M) *(float4 *)(a.C + (size_t)(m0 + fr) * a.ldc + 32 * t + 16 * fh + 4 * ks) = g;
    mx_s[ks][lane] = amax(amax(amax(amax(0.f, g.x), g.y), g.z), g.w);
  }
  lds_barrier();
  if (tid < 32 && m0 + tid < a.M) {
    float m = 0.f;
#pragma unroll
    for (int q = 0; q < KS; q++) m = __builtin_fmaxf(__builtin_fmaxf(m, mx_s[q][tid]), mx_s[q][32 + tid]);
    a.rmax[(size_t)(m0 + tid) * a.P + t] = m;
  }
}

template <int KT, int KS, int CT>
__global__ __launch_bounds__(64 * KS * CT) void res_split_kernel(SplitArgs a) {
  constexpr int KW = KT / KS, GO = 4 / KS;                 // K steps and accumulator groups of a wave
  constexpr int TPR = 2 * KS * CT, NV = 8 * KT / TPR;      // threads a row, float4s a thread
  static_assert(KT % KS == 0 && 4 % KS == 0 && 8 * KT % TPR == 0, "depth and groups over the waves");
  __shared__ __attribute__((aligned(16))) int8_t panel[KT * 1024];  // [KT][64 lanes][16]
  __shared__ int4 part[CT][KS * 4 * 64];
  __shared__ float sa_s[32];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, fh = lane >> 5, ks = wave % KS, ct = wave / KS;
  int t, blk;
  if (!tile_of(a.n / 32 / CT, (a.M + 31) / 32, &t, &blk)) return;
  t = t * CT + ct;
  const int m0 = 32 * blk;
  // the row's maxima and its values: TPR threads a row, a float4 each a step
  const int tr = tid / TPR, j = tid % TPR;
  const int arow = min(m0 + tr, a.M - 1);  // rows past M: row M-1, never stored
  float mx = 0.f;
  for (int p = j; p < a.P; p += TPR) mx = __builtin_fmaxf(mx, a.rmax[(size_t)arow * a.P + p]);
  float4 v[NV];
  const float *ap = a.A + (size_t)arow * a.lda + 4 * j;
#pragma unroll
  for (int u = 0; u < NV; u++) v[u] = *(const float4 *)(ap + 4 * TPR * u);
  v4i w[KW];
  const int8_t *wp = a.Bk + ((size_t)(ks * KW) * a.Np + 32 * t + perm32(fr)) * 32 + 16 * fh;
#pragma unroll
  for (int k = 0; k < KW; k++) w[k] = *(const v4i *)(wp + (size_t)k * a.Np * 32);
  const int ch = 32 * t + 16 * fh + 4 * GO * ks;  // this lane's channels
  float *const xp = a.C + (size_t)min(m0 + fr, a.M - 1) * a.ldc + ch;
  float4 sb[GO], x[GO];
#pragma unroll
  for (int q = 0; q < GO; q++) {
    sb[q] = *(const float4 *)(a.sb + ch + 4 * q);
    x[q] = *(const float4 *)(xp + 4 * q);
  }
#pragma unroll
  for (int o = 1; o < TPR; o <<= 1) mx = __builtin_fmaxf(mx, __shfl_xor(mx, o));
  float s = 0.f, inv = 0.f;
  if (mx != 0.f) {  // quantizeA: s = max/127, inv = 1/s (int8.go:175-183)
    s = mx / 127.0f;
    inv = 1.0f / s;
  }
  if (j == 0) sa_s[tr] = s;
#pragma unroll
  for (int u = 0; u < NV; u++) {
    const int col = 4 * (j + TPR * u);  // K step col / 32, half (col / 16) % 2, bytes col % 16 .. of row tr
    *(int *)(panel + (col >> 5) * 1024 + (tr + 32 * ((col >> 4) & 1)) * 16 + (col & 15)) = pack4(v[u], inv);
  }
  __syncthreads();
  v16i acc = {};
#pragma unroll
  for (int k = 0; k < KW; k++) acc = mfma32(w[k], *(const v4i *)(panel + (ks * KW + k) * 1024 + 16 * lane), acc);
  put_sums<KS>(part[ct], ks, lane, acc);
  __syncthreads();
  int4 sum[GO];
  gather_sums<KS>(part[ct], ks, lane, acc, sum);
  if (m0 + fr < a.M) {
#pragma unroll
    for (int q = 0; q < GO; q++) {
      const float4 d = deq4(sum[q], a.small, a.c128 + ch + 4 * q, a.zc + ch + 4 * q, sb[q], sa_s[fr]);
      *(float4 *)(xp + 4 * q) = make_float4(x[q].x + d.x, x[q].y + d.y, x[q].z + d.z, x[q].w + d.w);
    }
  }
}

}  // namespace

bool split_rows_supported(int H, int I, int KpH, int KpI) {
  if (KpH != H || KpI != I) return false;
  return (H == 768 && I == 1152) || (H == 384 && I == 1152) || (H == 256 && I == 512);
}

namespace {
template <int KT>
void wi_one(const SplitArgs &a, hipStream_t s) {
  wi_split_kernel<KT><<<tile_grid(a.n / 64, (a.M + 31) / 32), 256, 0, s>>>(a);
}
template <int KT>
void ln_wi_one(const SplitArgs &a, hipStream_t s) {
  const int grid = tile_grid(a.n / 64, (a.M + 31) / 32);
  switch (a.lanes) {
  case 0: ln_wi_split_kernel<KT, 0><<<grid, 1024, 0, s>>>(a); break;
  case 4: ln_wi_split_kernel<KT, 4><<<grid, 1024, 0, s>>>(a); break;
  case 8: ln_wi_split_kernel<KT, 8><<<grid, 1024, 0, s>>>(a); break;
  default: ln_wi_split_kernel<KT, 16><<<grid, 1024, 0, s>>>(a); break;
  }
}
template <int KT>
void res_one(const SplitArgs &a, hipStream_t s) {
  const int nblk = (a.M + 31) / 32;
  if (nblk < kManyBlocks) res_split_kernel<KT, 4, 1><<<tile_grid(a.n / 32, nblk), 256, 0, s>>>(a);
  else res_split_kernel<KT, 2, 4><<<tile_grid(a.n / 128, nblk), 512, 0, s>>>(a);
}
}  // namespace

void launch_wi_split(const SplitArgs &a, hipStream_t s) {
  if (a.M <= 0) return;
  if (a.K == 768) wi_one<24>(a, s);
  else if (a.K == 384) wi_one<12>(a, s);
  else wi_one<8>(a, s);
}

// one workgroup fills a CU: as long as no XCD has more than its CUs (hidden 768,
// 224 rows, 35 workgroups on an XCD of 32 CUs: 14.6 us, the two kernels 10.8)
bool ln_wi_split_supported(int I, int M, int cus) { return tile_grid(I / 32, (M + 31) / 32) <= cus; }

void launch_ln_wi_split(const SplitArgs &a, hipStream_t s) {
  if (a.M <= 0) return;
  if (a.K == 768) ln_wi_one<24>(a, s);
  else if (a.K == 384) ln_wi_one<12>(a, s);
  else ln_wi_one<8>(a, s);
}

void launch_res_split(const SplitArgs &a, hipStream_t s) {
  if (a.M <= 0) return;
  if (a.K == 1152) res_one<36>(a, s);
  else if (a.K == 768) res_one<24>(a, s);
  else if (a.K == 512) res_one<16>(a, s);
  else if (a.K == 384) res_one<12>(a, s);
  else res_one<8>(a, s);
}

}  // namespace ixh
