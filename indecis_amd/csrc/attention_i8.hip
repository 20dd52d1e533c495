// attention_i8.hip — int8 attention of indecis (linalg/attention8.go) on
// gfx950: QK^T and PV on i8 MFMA, the reference's full-row softmax in fp32,
// sliding-window (local) and global layers, sequences packed by offsets.
//
// Prologue, one workgroup per (sequence, head) — Attn8.Prepare
// (attention8.go:203-280): Q quantised per row with 1/sqrt(D) folded into
// its scale; K centred on its mean over the sequence (a sequential float32
// sum in key order, then times f32(1/n)) and quantised per key; V
// quantised per dimension. K is stored [head][slot][64], V transposed
// [head][d][slot]; each sequence's slots are padded with zeros to 64.
//
// Main, one workgroup per (sequence, block of 128 queries, head), 4 waves
// of 32 queries — Attn8.Attend (attention8.go:298-376). Each wave computes
// S^T = K.Q^T in 32x32 tiles (a lane holds one query, 16 keys), so the
// score tile is already the B operand of O^T = V^T.P^T. The softmax is
// the reference's two-pass one, exactly: pass 1 the row max of the valid
// scores, pass 2 e = exp(s - max) (the vector formula, or exp32 on the
// last len%V keys of a row as ExpShift does), P = RNE(255 e) as uint8,
// normalised by 1/f32(sum P). P (0..255) does not fit int8: the MFMA
// takes P - 128 and the accumulators get 128 * (sum of V over the keys of
// the tiles) added from per-chunk prefix sums, exactly. Scores need
// ((f32(tile) - kzc)*ks)*sq with the uint8 tile; tile - kzc is exactly the
// signed sum, so the kernel uses f32(sum q*k).
#include "ixh_device.h"
#include "ixh_internal.h"

namespace ixh {

namespace {

constexpr int D = 64;
constexpr int CHUNK = 256;       // keys staged in LDS at a time
constexpr int KS = 80;           // LDS row stride of K (bytes)
constexpr int VS = CHUNK + 16;   // LDS row stride of V^T (bytes)

__device__ __forceinline__ float absmax16(const float4 *v) {
  float m = 0.f;
#pragma unroll
  for (int c = 0; c < 16; c++)
    m = amax(amax(amax(amax(m, v[c].x), v[c].y), v[c].z), v[c].w);
  return m;
}

__device__ __forceinline__ int pack4(int a, int b, int c, int d) {
  return (a & 0xff) | ((b & 0xff) << 8) | ((c & 0xff) << 16) | (d << 24);
}

constexpr int kShortSeq = 512;   // keys one prologue workgroup holds in registers

// Statistics of a long sequence (more than kShortSeq keys) for
// Attn8.Prepare (attention8.go:224-230, 259-269), split 4 ways per
// (sequence, head): blockIdx.z 0 and 1 run the float32 chains of the K mean
// of 32 dimensions each, in key order (AddTo, then Scale by f32(1/n));
// blockIdx.z 2 and 3 take max |V| of 32 dimensions (MaxAbsTo). Writes the V
// scale to a.vs and, per (sequence, head), the K mean and 1/V scale to
// a.kstat.
//
// What bounds it: the chain of n dependent adds where few sequences run (one
// of 4,096 tokens: 48 us with the chain waiting on LDS every 4 keys and the
// slabs one ahead), the reading of K and V where many do. So K comes into an
// LDS ring by direct-to-LDS loads of waves 0-3, kStatRing - 1 slabs ahead,
// and wave 4, which has no load of its own to wait for, runs the chains, 32
// keys read from LDS ahead of their adds (about 9 cycles a key). With the
// prologue below, one sequence of 4,096 tokens 60 -> 31 us a layer, 8 of 1,024
// 34 -> 31, 8 of 8,192 199 -> 178 (hidden 768).
constexpr int kStatDims = 32;    // dimensions of a workgroup: a 128-byte line of a key's row
constexpr int kStatKeys = 128;   // keys of a slab: four loads of each loading wave
constexpr int kStatRing = 4;     // slabs in LDS
constexpr int kStatThreads = 320;
__global__ __launch_bounds__(kStatThreads) void attn_long_stats_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(1024))) float ring[kStatRing][kStatKeys * kStatDims];
  const int b = blockIdx.x, h = blockIdx.y, z = blockIdx.z, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dg = (z & 1) * kStatDims;
  const int base = a.offs[b], n = a.offs[b + 1] - base;
  const int ld = 3 * a.H;
  const float *src = a.qkv + (size_t)base * ld + (z < 2 ? a.H : 2 * a.H) + h * D + dg;
  float *stat = a.kstat + ((size_t)b * a.nh + h) * 2 * D;
  if (z < 2) {
    const int nslab = (n + kStatKeys - 1) / kStatKeys;
    if (wave < 4) {
      // slab s: key 32 wave + 8 u + lane / 8 of it, 16 bytes lane % 8 (keys
      // past n: key n-1, never added; past the last slab: the load count a
      // wave has in flight stays the same)
      auto issue = [&](int s) {
#pragma unroll
        for (int u = 0; u < kStatKeys / 32; u++) {
          const int key = min(s * kStatKeys + 32 * wave + 8 * u + (lane >> 3), n - 1);
          __builtin_amdgcn_global_load_lds((glb_ptr)(src + (size_t)key * ld + 4 * (lane & 7)),
                                           (lds_ptr)(&ring[s % kStatRing][(32 * wave + 8 * u) * kStatDims]), 16, 0, 0);
        }
      };
      if (nslab > 0)
        for (int s = 0; s < kStatRing - 1; s++) issue(s);
      for (int s = 0; s < nslab; s++) {
        wait_vmcnt<kStatKeys / 32 * (kStatRing - 2)>();  // slab s landed
        __builtin_amdgcn_s_barrier();       // every wave's; the chains are past slab s - 1
        issue(s + kStatRing - 1);
      }
      wait_vmcnt<0>();  // no load into LDS outlives the workgroup
    } else {
      float ksum = 0.f;
      for (int s = 0; s < nslab; s++) {
        lds_barrier();  // slab s is there; this wave's reads of slab s - 1 are done
        const float *col = &ring[s % kStatRing][lane & (kStatDims - 1)];
        const int cnt = n - s * kStatKeys;
        if (cnt >= kStatKeys) {
          constexpr int NB = 32;
          float v[2][NB];
#pragma unroll
          for (int r = 0; r < NB; r++) v[0][r] = col[r * kStatDims];
#pragma unroll
          for (int k = 0; k < kStatKeys / NB; k++) {
            if (k + 1 < kStatKeys / NB) {
#pragma unroll
              for (int r = 0; r < NB; r++) v[(k + 1) & 1][r] = col[(NB * (k + 1) + r) * kStatDims];
            }
            __builtin_amdgcn_sched_barrier(0);  // the next batch is read before this one is added
#pragma unroll
            for (int r = 0; r < NB; r++) ksum = ksum + v[k & 1][r];
          }
        } else {
          for (int r = 0; r < cnt; r++) ksum = ksum + col[r * kStatDims];
        }
      }
      if (lane < kStatDims) stat[dg + lane] = n > 0 ? ksum * (1.0f / (float)n) : 0.f;
    }
  } else {
    // 8 threads a key (a float4 each), 40 keys a load, 16 loads in flight
    constexpr int KR = kStatThreads / 8, NL = 16;
    const int q = tid & 7, r0 = tid >> 3;
    float4 vm = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int c0 = 0; c0 < n; c0 += KR * NL) {
      float4 v[NL];
#pragma unroll
      for (int u = 0; u < NL; u++) v[u] = *(const float4 *)(src + (size_t)min(c0 + r0 + KR * u, n - 1) * ld + 4 * q);
#pragma unroll
      for (int u = 0; u < NL; u++)
        vm = make_float4(amax(vm.x, v[u].x), amax(vm.y, v[u].y), amax(vm.z, v[u].z), amax(vm.w, v[u].w));
    }
    // threads with the same q hold the same 4 dimensions
    for (int t = 8; t < 64; t <<= 1) {
      vm.x = __builtin_fmaxf(vm.x, __shfl_xor(vm.x, t));
      vm.y = __builtin_fmaxf(vm.y, __shfl_xor(vm.y, t));
      vm.z = __builtin_fmaxf(vm.z, __shfl_xor(vm.z, t));
      vm.w = __builtin_fmaxf(vm.w, __shfl_xor(vm.w, t));
    }
    float *red = &ring[0][0];  // [wave][32]
    if (lane < 8) *(float4 *)(red + wave * kStatDims + 4 * q) = vm;
    __syncthreads();
    if (tid < kStatDims) {
      float vs = 0.f;
      for (int w = 0; w < kStatThreads / 64; w++) vs = __builtin_fmaxf(vs, red[w * kStatDims + tid]);
      float vi = 0.f;
      if (vs > 0.f) {  // attention8.go:262-269
        vs = vs / 127.0f;
        vi = 1.0f / vs;
      }
      a.vs[((size_t)b * a.nh + h) * D + dg + tid] = vs;
      stat[D + dg + tid] = vi;
    }
  }
}

// Single-read prologue: one workgroup of 512 threads per (sequence, head,
// K or V) holds up to kShortSeq keys of the 64-wide head slice in
// registers (16 float4 per thread), so K and V are read from HBM once.
// PART: a long sequence's keys in parts of kShortSeq (blockIdx.z = 2 part
// + K/V), with the K mean and 1/V scale from attn_long_stats_kernel;
// otherwise (all sequences at most kShortSeq) the statistics are computed
// here.
//  K (blockIdx.z even): row j = rg + 32u (rg = tid/16, u < 16). The 64
//    sequential float32 chains of the mean run in wave 0 over 32-row pieces
//    written to a double-buffered LDS slab (one barrier per piece); then
//    each row is centred and quantised from registers.
//  V (blockIdx.z odd): row j = 16 rg + u, so a thread holds 16 consecutive
//    keys of 4 dimensions: max |V| per dimension by a block reduction, then
//    each dimension's 16 quantised keys leave as one 16-byte store into
//    V^T.
template <bool PART>
__global__ __launch_bounds__(512, 4) void attn_prologue_rows_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) float kst[2][32 * D];
  __shared__ __attribute__((aligned(16))) float red[8][D];
  __shared__ __attribute__((aligned(16))) float mean[D];
  const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int sub = tid & 15, rg = tid >> 4, wave = tid >> 6, lane = tid & 63;
  const int j0 = PART ? (int)(blockIdx.z >> 1) * kShortSeq : 0;  // first key of the part
  const int nseq = a.offs[b + 1] - a.offs[b];
  const int npseq = (nseq + kKeyPad - 1) / kKeyPad * kKeyPad;
  if (PART && j0 >= npseq) return;  // j0 < npseq implies j0 < nseq
  const int base = a.offs[b] + j0, n = min(nseq - j0, kShortSeq);
  const int slot0 = a.padoff[b] + j0;
  const int npad = min(npseq - j0, kShortSeq);
  const int H = a.H, ld = 3 * H;
  const float *stat = a.kstat + ((size_t)b * a.nh + h) * 2 * D;
  // the sequence's rows of qkv; a row is 4*ld bytes
  const __amdgpu_buffer_rsrc_t rows = buf_rsrc(a.qkv + (size_t)base * ld, (uint32_t)n * ld * 4);
  const uint32_t col = 4u * (H + h * D + 4 * sub);  // byte offset of this thread's K float4
  const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);

  if ((blockIdx.z & 1) == 0) {
    float4 kr[16];
    const uint32_t voff = (uint32_t)rg * ld * 4 + col;
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int j = rg + 32 * u;
      kr[u] = j < n ? buf_load_f4<kStreamPolicy>(rows, voff, (uint32_t)(32 * u) * ld * 4) : zero4;
    }
    // sum of K in key order (AddTo, attention8.go:224-228)
    float ksum = 0.f;
#pragma unroll
    for (int u = 0; u < 16; u++) {
      if (!PART && 32 * u < n) {  // block-uniform
        *(float4 *)&kst[u & 1][rg * D + 4 * sub] = kr[u];
        __syncthreads();
        if (wave == 0) {
          const float *col = &kst[u & 1][lane];
          const int cnt = min(32, n - 32 * u);
          if (cnt == 32) {
#pragma unroll
            for (int rr = 0; rr < 32; rr++) ksum = ksum + col[rr * D];
          } else {
            for (int rr = 0; rr < cnt; rr++) ksum = ksum + col[rr * D];
          }
        }
      }
    }
    if (wave == 0) mean[lane] = PART ? stat[lane] : n > 0 ? ksum * (1.0f / (float)n) : 0.f;  // Scale(mean, 1/n)
    __syncthreads();
    // centred rows quantised per key (quantRowAVX2 without the flip,
    // attention8.go:240-251); padding slots [n, npad) get zeros
    int8_t *kp = a.kp + ((size_t)h * a.Npad + slot0) * D;
    float *ks = a.ks + (size_t)h * a.Npad + slot0;
    const float4 mu = *(const float4 *)&mean[4 * sub];
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int j = rg + 32 * u;
      if (j < npad) {  // uniform over the 16 lanes of a row
        int kq = 0;
        float sc = 0.f;
        if (j < n) {
          const float4 c = make_float4(kr[u].x - mu.x, kr[u].y - mu.y, kr[u].z - mu.z, kr[u].w - mu.w);
          float mx = amax(amax(amax(amax(0.f, c.x), c.y), c.z), c.w);
          for (int t = 1; t < 16; t <<= 1) mx = __builtin_fmaxf(mx, __shfl_xor(mx, t, 16));
          float inv = 0.f;
          if (mx != 0.f) {
            sc = mx / 127.0f;
            inv = 1.0f / sc;
          }
          kq = pack4(q8(c.x, inv), q8(c.y, inv), q8(c.z, inv), q8(c.w, inv));
        }
        *(int *)(kp + (size_t)j * D + 4 * sub) = kq;
        if (sub == 0) ks[j] = sc;
      }
    }
  } else {
    float4 vr[16];
    const uint32_t voff = (uint32_t)(16 * rg) * ld * 4 + col + 4 * H;
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int j = 16 * rg + u;
      vr[u] = j < n ? buf_load_f4<kStreamPolicy>(rows, voff, (uint32_t)u * ld * 4) : zero4;
    }
    if (PART) {
      if (tid < D) mean[tid] = stat[D + tid];
    } else {
      // max |V| per dimension (MaxAbsTo, attention8.go:259-261)
      float4 vm = zero4;
#pragma unroll
      for (int u = 0; u < 16; u++)
        vm = make_float4(amax(vm.x, vr[u].x), amax(vm.y, vr[u].y),
                         amax(vm.z, vr[u].z), amax(vm.w, vr[u].w));
      for (int t = 16; t < 64; t <<= 1) {
        vm.x = __builtin_fmaxf(vm.x, __shfl_xor(vm.x, t));
        vm.y = __builtin_fmaxf(vm.y, __shfl_xor(vm.y, t));
        vm.z = __builtin_fmaxf(vm.z, __shfl_xor(vm.z, t));
        vm.w = __builtin_fmaxf(vm.w, __shfl_xor(vm.w, t));
      }
      if (lane < 16) *(float4 *)&red[wave][4 * sub] = vm;
      __syncthreads();
      if (tid < D) {
        float vs = 0.f;
        for (int g = 0; g < 8; g++) vs = __builtin_fmaxf(vs, red[g][tid]);
        float vi = 0.f;
        if (vs > 0.f) {  // attention8.go:262-269
          vs = vs / 127.0f;
          vi = 1.0f / vs;
        }
        mean[tid] = vi;
        a.vs[((size_t)b * a.nh + h) * D + tid] = vs;
      }
    }
    __syncthreads();
    // quantCols (attention8.go:270-279), 16 keys of a dimension per store
    const float4 vi = *(const float4 *)&mean[4 * sub];
    if (16 * rg < npad) {
      int8_t *vt = a.vt + ((size_t)h * D + 4 * sub) * a.Npad + slot0 + 16 * rg;
      int w[4][4];
#pragma unroll
      for (int u = 0; u < 16; u += 4) {
        w[0][u / 4] = pack4(q8(vr[u].x, vi.x), q8(vr[u + 1].x, vi.x), q8(vr[u + 2].x, vi.x), q8(vr[u + 3].x, vi.x));
        w[1][u / 4] = pack4(q8(vr[u].y, vi.y), q8(vr[u + 1].y, vi.y), q8(vr[u + 2].y, vi.y), q8(vr[u + 3].y, vi.y));
        w[2][u / 4] = pack4(q8(vr[u].z, vi.z), q8(vr[u + 1].z, vi.z), q8(vr[u + 2].z, vi.z), q8(vr[u + 3].z, vi.z));
        w[3][u / 4] = pack4(q8(vr[u].w, vi.w), q8(vr[u + 1].w, vi.w), q8(vr[u + 2].w, vi.w), q8(vr[u + 3].w, vi.w));
      }
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const v4i o = {w[c][0], w[c][1], w[c][2], w[c][3]};
        *(v4i *)(vt + (size_t)c * a.Npad) = o;
      }
    }
  }
}

// Q per (row, head) for Attend8 callers whose queries did not come out of
// the QKV GEMM epilogue: 16 threads per row, as the prologue's K pass.
__global__ __launch_bounds__(256) void attn_quant_q_kernel(AttnArgs a) {
  const int g = blockIdx.x * 16 + (threadIdx.x >> 4), sub = threadIdx.x & 15;
  if (g >= a.N * a.nh) return;  // whole 16-lane groups leave together
  const int row = g / a.nh, h = g % a.nh;
  const float4 v = *(const float4 *)(a.qkv + (size_t)row * 3 * a.H + h * D + 4 * sub);
  float mx = amax(amax(amax(amax(0.f, v.x), v.y), v.z), v.w);
  for (int t = 1; t < 16; t <<= 1) mx = __builtin_fmaxf(mx, __shfl_xor(mx, t, 16));
  float s = 0.f, inv = 0.f;
  if (mx != 0.f) {
    s = mx / 127.0f;
    inv = 1.0f / s;
  }
  *(int *)(a.qq + (size_t)row * a.H + h * D + 4 * sub) =
      pack4(q8(v.x, inv), q8(v.y, inv), q8(v.z, inv), q8(v.w, inv));
  if (sub == 0) a.sq[(size_t)row * a.nh + h] = s * a.scale;
}

// Four waves a SIMD (at most 128 VGPRs) for both layer kinds: local layers
// 116-118 us a launch on cfg4 against 129-131 at three waves a SIMD.
// KSPL: waves that share 32 queries, each taking a part of every chunk's key
// tiles; their maxima, sums of P and (exact int32) products meet in LDS. 1:
// 256 threads; 2 and 4 for launches too small to fill the chip.
template <bool GLOBAL, int KSPL>
__global__ __launch_bounds__(256 * KSPL, KSPL == 1 ? 4 : 2) void attn_main_kernel(AttnArgs a) {
  constexpr int T = 256 * KSPL;
  __shared__ __attribute__((aligned(16))) int8_t Ks[CHUNK * KS];
  __shared__ __attribute__((aligned(16))) int8_t Vs[D * VS];
  __shared__ __attribute__((aligned(16))) float kss[CHUNK];
  // per 32-key group g of the staged chunk: vpre[g][d] = 128 times the sum
  // of V over the keys of groups 0..g (int, exact: at most 128 * 256 * 127);
  // 40 KB of LDS in all, 4 workgroups per CU
  __shared__ __attribute__((aligned(16))) int vpre[CHUNK / 32][D];

  // the wave index as a scalar: the tile loops and the full-tile tests
  // that derive from it are then scalar branches, not lane masks
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wid & 3, kh = wid >> 2;  // the wave's queries, its share of the keys
  // work item j = head * nblocks + entry (a sequence's query blocks are
  // consecutive entries). Workgroup L runs on XCD L % 8; each XCD takes a
  // contiguous run of items, so the query blocks of one (sequence, head)
  // run on one XCD and share its K and V in that XCD's L2.
  const int per = (a.nblocks * a.nh + 7) / 8;
  const int j = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (j >= a.nblocks * a.nh) return;  // the whole workgroup
  const int h = j / a.nblocks, ent = j - h * a.nblocks;
  const int b = a.blocks[2 * ent], Q0 = a.blocks[2 * ent + 1];
  const int base = a.offs[b], n = a.offs[b + 1] - base;
  const int slot0 = a.padoff[b];
  const int npad = (n + kKeyPad - 1) / kKeyPad * kKeyPad;
  const int H = a.H, W = a.window;
  constexpr bool global = GLOBAL;

  // this lane's query
  const int q0 = Q0 + 32 * wave;
  const int qi = q0 + (lane & 31);
  const bool qact = qi < n;
  v4i qb[2];
  {
    const v4i z = {0, 0, 0, 0};
    const int8_t *qsrc = a.qq + (size_t)(base + (qact ? qi : 0)) * H + h * D + 16 * (lane >> 5);
    qb[0] = qact ? *(const v4i *)(qsrc) : z;
    qb[1] = qact ? *(const v4i *)(qsrc + 32) : z;
  }
  const float sqv = qact ? a.sq[(size_t)(base + qi) * a.nh + h] : 0.f;
  // valid keys [cs, ce) of the query and the start of the exp32 tail
  // (ExpShift's scalar loop over the last len%V values, vec_simd.go:258-262)
  const int cs = global ? 0 : max(0, qi - W);
  const int ce = global ? n : min(n, qi + W + 1);
  const uint32_t span = (uint32_t)(ce - cs);  // > 0 for an active query
  const int V = a.lanes;
  const int ts = V > 0 ? cs + ((ce - cs) / V) * V : cs;
  // wave-wide bounds over the active queries: a tile [k0, k0+32) with
  // k0 >= cs_hi and k0+32 <= ce_lo is valid for every query
  int cs_hi = qact ? cs : 0, ce_lo = qact ? ce : 1 << 30;
  for (int t = 1; t < 64; t <<= 1) {
    cs_hi = max(cs_hi, __shfl_xor(cs_hi, t));
    ce_lo = min(ce_lo, __shfl_xor(ce_lo, t));
  }
  cs_hi = __builtin_amdgcn_readfirstlane(cs_hi);  // every lane holds the same value
  ce_lo = __builtin_amdgcn_readfirstlane(ce_lo);

  // key tiles (32 keys) of this wave and of the block
  int wt0, wt1, bk0, bk1;
  if (global) {
    wt0 = 0;
    wt1 = (n + 31) / 32;
    bk0 = 0;
    bk1 = n;
  } else {
    wt0 = max(0, q0 - W) / 32;
    wt1 = (min(n, q0 + 31 + W + 1) + 31) / 32;
    bk0 = max(0, Q0 - W) / 32 * 32;
    bk1 = min(n, Q0 + kAttnQBlock - 1 + W + 1);
  }
  if (q0 >= n) wt1 = wt0;  // idle wave (still takes part in the barriers)
  const bool one_chunk = bk1 - bk0 <= CHUNK;

  const int8_t *kglob = a.kp + ((size_t)h * a.Npad + slot0) * D;
  const float *ksglob = a.ks + (size_t)h * a.Npad + slot0;
  const int8_t *vglob = a.vt + (size_t)h * D * a.Npad + slot0;

  // Stage the chunk of keys c0 .. c0+CHUNK-1: K rows and their scales,
  // and with with_v V^T with the 8 dwords of each 32-key group permuted so
  // that lane half hf reads the keys 8*(b/4) + 4*hf + b%4 (the S^T
  // accumulator rows) as 16 contiguous bytes, plus each group's sum of V
  // per dimension. Every global load of the thread is issued before the
  // first LDS write, so the staging waits on memory once. Buffer loads:
  // keys past the sequence's slots read 0 (V^T rows continue into the next
  // sequence's slots, so those loads get an offset past the range).
  static_assert(CHUNK == 256, "one key scale a thread (the first 256)");
  constexpr int NKP = CHUNK * 4 / T;                              // 16-byte K pieces a thread
  constexpr int NVG = D * (CHUNK / 32) / T > 0 ? D * (CHUNK / 32) / T : 1;  // V (dimension, group) items a thread
  constexpr bool VALL = D * (CHUNK / 32) >= T;                    // (KSPL 4: of the first 512)
  const auto krs = buf_rsrc(kglob, (uint32_t)npad * D);
  const auto ksrs = buf_rsrc(ksglob, (uint32_t)npad * 4);
  const auto vrs = buf_rsrc(vglob, (uint32_t)((D - 1) * a.Npad + npad));
  auto stage = [&](int c0, bool with_v) {
    // local layers: the thread's offsets are recomputed at each call from
    // an opaque copy of its index, instead of being kept in VGPRs across
    // the score loops between calls (held to 128 VGPRs, the kernel spilled
    // 8 of them: 8 KB a workgroup written to scratch)
    int tid = threadIdx.x;
    if constexpr (!GLOBAL) asm volatile("" : "+v"(tid));
    v4i kw[NKP], vlo[NVG], vhi[NVG];
#pragma unroll
    for (int i = 0; i < NKP; i++)
      kw[i] = __builtin_amdgcn_raw_buffer_load_b128(krs, (uint32_t)((c0 + (tid >> 2) + T / 4 * i) * D + 16 * (tid & 3)), 0, 0);
    const float kv = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ksrs, (uint32_t)(c0 + tid) * 4, 0, 0));
    if (with_v) {
#pragma unroll
      for (int i = 0; i < NVG; i++) {
        const int e = (tid + T * i) % (D * (CHUNK / 32)), d = e / (CHUNK / 32), g = e % (CHUNK / 32);
        const uint32_t off = c0 + 32 * g < npad ? (uint32_t)(d * a.Npad + c0 + 32 * g) : 0x7fffffe0u;
        vlo[i] = __builtin_amdgcn_raw_buffer_load_b128(vrs, off, 0, 0);
        vhi[i] = __builtin_amdgcn_raw_buffer_load_b128(vrs, off + 16, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < NKP; i++) *(v4i *)&Ks[((tid >> 2) + T / 4 * i) * KS + 16 * (tid & 3)] = kw[i];
    if (T == 256 || tid < CHUNK) kss[tid] = kv;
    if (with_v && (VALL || tid < D * (CHUNK / 32))) {
#pragma unroll
      for (int i = 0; i < NVG; i++) {
        const int e = tid + T * i, d = e / (CHUNK / 32), g = e % (CHUNK / 32);
        const int w[8] = {vlo[i][0], vlo[i][1], vlo[i][2], vlo[i][3], vhi[i][0], vhi[i][1], vhi[i][2], vhi[i][3]};
        const v4i o0 = {w[0], w[2], w[4], w[6]}, o1 = {w[1], w[3], w[5], w[7]};
        *(v4i *)&Vs[d * VS + 32 * g] = o0;
        *(v4i *)&Vs[d * VS + 32 * g + 16] = o1;
        int sum = 0;
#pragma unroll
        for (int u = 0; u < 8; u++) sum = __builtin_amdgcn_sdot4(w[u], 0x01010101, sum, false);
        vpre[g][d] = sum;
      }
    }
  };
  // after the barrier that follows stage_v: group sums -> prefix sums (the
  // group sums read together, then written: one wait on LDS, not one a
  // group)
  // global layers: thread d < 64 keeps 128 times the sum of V over the
  // chunks so far
  int vtot = 0;
  auto prefix_v = [&] {
    if (tid < D) {
      int gsum[CHUNK / 32];
#pragma unroll
      for (int g = 0; g < CHUNK / 32; g++) gsum[g] = vpre[g][tid];
#pragma unroll
      for (int g = 1; g < CHUNK / 32; g++) gsum[g] += gsum[g - 1];
      if constexpr (GLOBAL) {
        vtot += 128 * gsum[CHUNK / 32 - 1];  // the chunk's sum (each chunk once)
      } else {
#pragma unroll
        for (int g = 0; g < CHUNK / 32; g++) vpre[g][tid] = 128 * gsum[g];
      }
    }
    __syncthreads();
  };
  // Scores of tile t without the query scale: f32(sum q*k) * ks, in the S^T
  // layout (rows = keys 8*(r/4) + 4*(lane/32) + r%4 of the tile, column =
  // this query). The score is that times sq.
  // The integer tile of tile t (two MFMAs), then its scaled scores.
  // (Issuing tile t+1's MFMAs before tile t's VALU work was tried: no gain.)
  auto score_acc = [&](int t, int c0) {
    v16i acc = {};
    const int8_t *kr = &Ks[(t * 32 - c0 + (lane & 31)) * KS + 16 * (lane >> 5)];
    acc = mfma32(*(const v4i *)kr, qb[0], acc);
    acc = mfma32(*(const v4i *)(kr + 32), qb[1], acc);
    return acc;
  };
  auto score_scale = [&](int t, int c0, const v16i &acc, float *sv) {
    const float *kt = &kss[t * 32 - c0 + 4 * (lane >> 5)];
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const float4 k4 = *(const float4 *)(kt + 8 * g);
      sv[4 * g] = (float)acc[4 * g] * k4.x;
      sv[4 * g + 1] = (float)acc[4 * g + 1] * k4.y;
      sv[4 * g + 2] = (float)acc[4 * g + 2] * k4.z;
      sv[4 * g + 3] = (float)acc[4 * g + 3] * k4.w;
    }
  };

  // of the chunk's tiles t0 .. t1 - 1 of these queries, this wave's
  auto my_tiles = [&](int &t0, int &t1) {
    if constexpr (KSPL > 1) {
      const int cnt = max(t1 - t0, 0), b0 = t0;
      t0 = b0 + cnt * kh / KSPL;
      t1 = b0 + cnt * (kh + 1) / KSPL;
    }
  };

  // ---- pass 1: row max of the valid scores ----
  // max_j f32(x_j * sq) = f32(max_j x_j * sq): rounding is monotone and
  // sq >= 0, so the query scale is applied once, to the max.
  float m = -__builtin_huge_valf();
  for (int c0 = bk0; c0 < bk1; c0 += CHUNK) {
    __syncthreads();
    stage(c0, one_chunk);
    __syncthreads();
    if (one_chunk) prefix_v();
    int t0 = max(wt0, c0 / 32), t1 = min(wt1, (c0 + CHUNK) / 32);
    my_tiles(t0, t1);
    for (int t = t0; t < t1; t++) {
      float sv[16];
      score_scale(t, c0, score_acc(t, c0), sv);
      const int k0 = t * 32;
      if (k0 >= cs_hi && k0 + 32 <= ce_lo) {  // every key valid for every query
#pragma unroll
        for (int r = 0; r < 16; r++) m = __builtin_fmaxf(m, sv[r]);  // no NaN: v_max
      } else {
        // key j valid: cs <= j < ce, as one unsigned compare of j - cs
        const int jb = k0 - cs + 4 * (lane >> 5);
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const bool in = (uint32_t)(jb + 8 * (r >> 2) + (r & 3)) < span;
          m = __builtin_fmaxf(m, in ? sv[r] : -__builtin_huge_valf());
        }
      }
    }
  }
  m = __builtin_fmaxf(m, __shfl_xor(m, 32));
  if constexpr (KSPL > 1) {
    __shared__ float mx_s[4 * KSPL][32];
    if (lane < 32) mx_s[wid][lane] = m;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < KSPL; q++) m = __builtin_fmaxf(m, mx_s[4 * q + wave][lane & 31]);
  }
  m = m * sqv;

  // ---- pass 2: P = RNE(255 exp(s - m)), O^T += V^T . P^T ----
  // P (0..255) enters the MFMA as P - 128 (an int8: the byte P ^ 0x80);
  // the missing 128 * sum_j v[j][d] over every key of the tiles a wave
  // processes is the same for all its queries and is added to the
  // accumulators per chunk from the prefix sums: O stays exact.
  // With x = f32(q.k) * ks, y = 2^(x (sq log2 e) + (log2 255 - m log2 e)) is
  // 255 exp(s - max) up to a relative error the score bounds: P is its
  // rounding where y less that error and y plus it round alike. Where they do
  // not (about 1 group of 4 scores in 100), s - max is formed as the reference
  // forms it and rounded from exp255_fast, unless that lands within
  // kExp255Tol of a half-integer; there the reference formula decides: exp32
  // on the tail keys j >= ts (all keys when lanes = 0), ExpShift's vector
  // formula elsewhere.
  //
  // The error, with u = 2^-24 and the scores that matter (P > 0: s - m >
  // -6.3, so |s| <= |m| + 6.3). In the exponent, against the one that
  // exp255_fast forms of the reference's s - m: the reference's roundings of s
  // and of s - m log2 e (|s| + |s - m|) u, that of es log2 e |s| u, the two of
  // eb (the fma, then kap's subtraction) 2 (log2 e |m| + 8) u, that of either
  // exponent 8 u; the constants are the same in both. Together (59.3 + 4 log2 e
  // |m|) u, times ln 2 in y: (41.1 + 4 |m|) u. exp255_fast against the reference
  // formulas 10 u (kExp255Rel), the hardware exponential twice and the scaling
  // by hi 6 u. The sum, (57.1 + 4 |m|) u, is taken as kap = (64 + 4.25 |m|) u;
  // kap <= 0.0084, so its squares stay inside the 0.125 kap that hi has over
  // (1 + kap) / (1 - kap). A lower score (s - m < -6.3, 255 exp below 0.469) stays
  // under a half: per unit of |s| past |m| + 6.3 its error gains 3 u while its
  // logarithm falls by 1. Past |m| = 2^15 every
  // group takes the other way. 11 VALU slots a score instead of 13 (the
  // exponential takes 4) and fewer scores formed twice: global layers of
  // 8,192 tokens 2,900 -> 2,650 us a launch, of 4,096 162 -> 146, of 256 64.5
  // -> 60.3; local layers 97 -> 93.5 and 50.2 -> 49.
  float es = sqv * 1.44269504088896341f;
  const float kap = (64.0f + 4.25f * fabsf(m)) * 0x1p-24f;
  float eb = __builtin_fmaf(-m, 1.44269504088896341f, 7.99435343685885793f) - 1.4427f * kap;
  float hi = 1.0f + 2.125f * kap;  // (1 - kap) hi >= 1 + kap
  // (also a query scale whose product with log2 e overflows: such a scale
  // times the scores can still be finite). y = 1, its upper bound 300
  if (qact && !(fabsf(m) <= 32768.0f && es < __builtin_huge_valf())) {
    es = 0.0f;
    eb = 0.0f;
    hi = 300.0f;
  }
  v16i o[2];
#pragma unroll
  for (int dt = 0; dt < 2; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[dt][r] = 0;
  unsigned psum = 0;
  for (int c0 = bk0; c0 < bk1; c0 += CHUNK) {
    if (!one_chunk) {
      __syncthreads();
      stage(c0, true);
      __syncthreads();
      prefix_v();
    }
    int t0 = max(wt0, c0 / 32), t1 = min(wt1, (c0 + CHUNK) / 32);
    my_tiles(t0, t1);
    if (!GLOBAL && t1 > t0) {
      // rows of this lane: dims dt*32 + 8g + 4*(lane/32) + 0..3
#pragma unroll
      for (int dt = 0; dt < 2; dt++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int d0 = dt * 32 + 8 * g + 4 * (lane >> 5);
          const int4 hi = *(const int4 *)&vpre[t1 - 1 - c0 / 32][d0];
          const int4 lo = t0 > c0 / 32 ? *(const int4 *)&vpre[t0 - 1 - c0 / 32][d0] : int4{0, 0, 0, 0};
          o[dt][4 * g] += hi.x - lo.x;
          o[dt][4 * g + 1] += hi.y - lo.y;
          o[dt][4 * g + 2] += hi.z - lo.z;
          o[dt][4 * g + 3] += hi.w - lo.w;
        }
    }
    for (int t = t0; t < t1; t++) {
      float sv[16];
      score_scale(t, c0, score_acc(t, c0), sv);
      const int k0 = t * 32;
      const bool full = k0 >= cs_hi && k0 + 32 <= ce_lo;  // every key valid for every query
      unsigned pw[4];
#pragma unroll
      for (int g = 0; g < 4; g++) {
        unsigned lo = 0, up = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const float y = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[4 * g + u], es, eb));
          lo = __builtin_amdgcn_cvt_pk_u8_f32(y, u, lo);
          up = __builtin_amdgcn_cvt_pk_u8_f32(y * hi, u, up);
        }
        if (lo != up) {
          // a bound either side of a half-integer: the score as the
          // reference forms it, its exponential checked float by float
          lo = 0;
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const float d = sv[4 * g + u] * sqv - m;
            const float y = exp255_fast(d);
            float p = rne(y);
            if (fabsf(y - p) > 0.5f - kExp255Tol) {
              const int j = k0 + 8 * g + 4 * (lane >> 5) + u;
              const float e = (j >= ts) ? exp32_scalar(d) : exp32_simd(d);
              // QuantizeRowU8 (vec_simd.go:64-91): RNE(e*255) in [0, 255]
              p = rne(e * 255.0f);
            }
            lo = __builtin_amdgcn_cvt_pk_u8_f32(p, u, lo);
          }
        }
        pw[g] = lo;
      }
      if (!full) {
        // the tile's valid keys as bits, a group's 4 bits as byte masks
        const int first = min(max(cs - k0, 0), 32), last = min(max(ce - k0, 0), 32);
        const unsigned ok = ((unsigned)((1ull << last) - 1) & (unsigned)(~0ull << first)) >> (4 * (lane >> 5));
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const unsigned one = (((ok >> (8 * g)) & 0xfu) * 0x204081u) & 0x01010101u;
          pw[g] &= (one << 8) - one;
        }
      }
#pragma unroll
      for (int g = 0; g < 4; g++) psum = __builtin_amdgcn_udot4(pw[g], 0x01010101u, psum, false);
      // P - 128 as int8
      const v4i bp = {(int)(pw[0] ^ 0x80808080u), (int)(pw[1] ^ 0x80808080u),
                      (int)(pw[2] ^ 0x80808080u), (int)(pw[3] ^ 0x80808080u)};
#pragma unroll
      for (int dt = 0; dt < 2; dt++) {
        const v4i fv = *(const v4i *)&Vs[(dt * 32 + (lane & 31)) * VS + (t * 32 - c0) + 16 * (lane >> 5)];
        o[dt] = mfma32(fv, bp, o[dt]);
      }
    }
  }
  if constexpr (GLOBAL) {
    // a wave with queries takes every tile of the sequence, so its
    // correction is 128 times the sequence's sum of V (keys past it are
    // zero), added once
    // (vpre is free: its last reader, the last prefix, passed its barrier)
    if (tid < D) vpre[0][tid] = vtot;
    __syncthreads();
    if (wt1 > wt0 && kh == 0) {
#pragma unroll
      for (int dt = 0; dt < 2; dt++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int4 tv = *(const int4 *)&vpre[0][dt * 32 + 8 * g + 4 * (lane >> 5)];
          o[dt][4 * g] += tv.x;
          o[dt][4 * g + 1] += tv.y;
          o[dt][4 * g + 2] += tv.z;
          o[dt][4 * g + 3] += tv.w;
        }
    }
  }
  psum += __shfl_xor(psum, 32);
  if constexpr (KSPL > 1) {
    // the other waves' products and sums of P, a wave's 32 registers a time
    // through the free K and V staging areas (16 KB each: [4 waves][16][64])
    __shared__ unsigned ps_s[4][32];
    static_assert(4 * 16 * 64 * 4 <= CHUNK * KS && 4 * 16 * 64 * 4 <= D * VS, "partial products");
    int4 *const pk = (int4 *)Ks + wave * (4 * 64) + lane, *const pv = (int4 *)Vs + wave * (4 * 64) + lane;
#pragma unroll
    for (int q = 1; q < KSPL; q++) {
      __syncthreads();  // Ks and Vs are free (pass 2, or the part before)
      if (kh == q) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
          pk[64 * g] = int4{o[0][4 * g], o[0][4 * g + 1], o[0][4 * g + 2], o[0][4 * g + 3]};
          pv[64 * g] = int4{o[1][4 * g], o[1][4 * g + 1], o[1][4 * g + 2], o[1][4 * g + 3]};
        }
        if (lane < 32) ps_s[wave][lane] = psum;
      }
      __syncthreads();
      if (kh == 0) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int4 x = pk[64 * g], y = pv[64 * g];
          o[0][4 * g] += x.x; o[0][4 * g + 1] += x.y; o[0][4 * g + 2] += x.z; o[0][4 * g + 3] += x.w;
          o[1][4 * g] += y.x; o[1][4 * g + 1] += y.y; o[1][4 * g + 2] += y.z; o[1][4 * g + 3] += y.w;
        }
        psum += ps_s[wave][lane & 31];
      }
    }
  }
  // The context rows leave through LDS: each wave stages its 32 queries x
  // 64 dimensions in the free K or V staging area, then stores whole
  // 256-byte row pieces (16 lanes a query), non-temporal (the Wo kernel
  // reads them once).
  constexpr int OLD = D + 4;  // floats a staged row (conflict-free writes)
  static_assert(2 * 32 * OLD * 4 <= CHUNK * KS && 2 * 32 * OLD * 4 <= D * VS, "context staging");
  __syncthreads();  // every wave is past pass 2: Ks and Vs are free
  if (KSPL > 1 && kh > 0) return;
  float *stg = (float *)(wave < 2 ? Ks : Vs) + (wave & 1) * (32 * OLD);
  const float sp = qact ? 1.0f / (float)(int)psum : 0.f;
  const float *vsd = a.vs + ((size_t)b * a.nh + h) * D;
  float mx = 0.f;  // max |ctx| of this (row, head), for the fused Wo GEMM
  // the V scales of this lane's 32 dimensions, every load issued before
  // the first store (the compiler cannot tell vs from ctx)
  float4 vsv[2][4];
#pragma unroll
  for (int dt = 0; dt < 2; dt++)
#pragma unroll
    for (int g = 0; g < 4; g++) vsv[dt][g] = *(const float4 *)&vsd[dt * 32 + acc_row(4 * g, lane)];
#pragma unroll
  for (int dt = 0; dt < 2; dt++) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int d0 = dt * 32 + acc_row(4 * g, lane);
      const float4 v4 = vsv[dt][g];
      const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
      float ov[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int r = 4 * g + u;
        const int tile = o[dt][r];
        ov[u] = (((float)tile - 0.0f) * vv[u]) * sp;
        mx = __builtin_fmaxf(mx, fabsf(ov[u]));
      }
      *(float4 *)(stg + (lane & 31) * OLD + d0) = make_float4(ov[0], ov[1], ov[2], ov[3]);
    }
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt 0: this wave's staging writes are done
  __builtin_amdgcn_wave_barrier();
  // query 4u + lane/16 of the wave, dimensions 4 (lane % 16) .. + 3
#pragma unroll
  for (int u = 0; u < 8; u++) {
    const int ql = 4 * u + (lane >> 4), qg = q0 + ql;
    const float4 v = *(const float4 *)(stg + ql * OLD + 4 * (lane & 15));
    if (qg < n)
      store_stream_16(a.ctx + (size_t)(base + qg) * H + h * D + 4 * (lane & 15),
                      v4i{__float_as_int(v.x), __float_as_int(v.y), __float_as_int(v.z), __float_as_int(v.w)});
  }
  if (a.rmax && qact) {
    mx = __builtin_fmaxf(mx, __shfl_xor(mx, 32));  // the other 32 dimensions
    if (lane < 32) a.rmax[(size_t)(base + qi) * a.nh + h] = mx;
  }
}

// Every float v = bits -> float over [lo, hi) (v <= 0 expected): counts
// the v where exp255_fast decides the rounding (away from a half-integer by
// more than kExp255Tol) and RNE differs from the reference's
// RNE(f32(255*exp(v))), and the v >= -6.4 where exp255_fast is further than
// kExp255Rel from f32(255*exp(v)), for exp32_simd (res[0]) and exp32_scalar (res[1]);
// res[2], res[3]: largest |exp255_fast - 255*exp| of each formula, as
// float bits; res[4]: number of undecided v.
__global__ __launch_bounds__(256) void check_exp255_kernel(uint32_t lo, uint32_t hi,
                                                           unsigned long long *res) {
  unsigned long long bad_v = 0, bad_s = 0, amb = 0;
  float err_v = 0.f, err_s = 0.f;
  const uint32_t stride = gridDim.x * 256u;
  for (uint32_t u = lo + blockIdx.x * 256u + threadIdx.x; u < hi && u >= lo; u += stride) {
    const float v = __uint_as_float(u);
    const float y = exp255_fast(v);
    const float p = rne(y);
    const bool decided = fabsf(y - p) <= 0.5f - kExp255Tol;
    const float yv = exp32_simd(v) * 255.0f, ys = exp32_scalar(v) * 255.0f;
    err_v = amax(err_v, y - yv);
    err_s = amax(err_s, y - ys);
    if (v >= -6.4f) {  // where P > 0: the relative distance too
      bad_v += fabsf(y - yv) > kExp255Rel * yv;
      bad_s += fabsf(y - ys) > kExp255Rel * ys;
    }
    if (decided) {
      bad_v += rne(yv) != p;
      bad_s += rne(ys) != p;
    } else {
      amb++;
    }
  }
  for (int t = 1; t < 64; t <<= 1) {
    bad_v += __shfl_xor(bad_v, t);
    bad_s += __shfl_xor(bad_s, t);
    amb += __shfl_xor(amb, t);
    err_v = __builtin_fmaxf(err_v, __shfl_xor(err_v, t));
    err_s = __builtin_fmaxf(err_s, __shfl_xor(err_s, t));
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&res[0], bad_v);
    atomicAdd(&res[1], bad_s);
    atomicMax(&res[2], (unsigned long long)__float_as_uint(err_v));
    atomicMax(&res[3], (unsigned long long)__float_as_uint(err_s));
    atomicAdd(&res[4], amb);
  }
}

}  // namespace

void launch_check_exp255(uint32_t lo, uint32_t hi, unsigned long long *res, hipStream_t s) {
  if (hi <= lo) return;
  check_exp255_kernel<<<4096, 256, 0, s>>>(lo, hi, res);
}

void launch_attn_quant_q(const AttnArgs &a, hipStream_t s) {
  const long groups = (long)a.N * a.nh;
  if (groups <= 0) return;
  attn_quant_q_kernel<<<(unsigned)((groups + 15) / 16), 256, 0, s>>>(a);
}

void launch_attn_prologue(const AttnArgs &a, hipStream_t s) {
  if (a.B <= 0) return;
  if (a.max_n <= kShortSeq) {
    attn_prologue_rows_kernel<false><<<dim3(a.B, a.nh, 2), 512, 0, s>>>(a);
  } else {
    attn_long_stats_kernel<<<dim3(a.B, a.nh, 4), kStatThreads, 0, s>>>(a);
    const int parts = (a.max_n + kShortSeq - 1) / kShortSeq;
    attn_prologue_rows_kernel<true><<<dim3(a.B, a.nh, 2 * parts), 512, 0, s>>>(a);
  }
}

void launch_attn_main(const AttnArgs &a, hipStream_t s) {
  if (a.nblocks <= 0) return;
  // 8 runs of (nblocks * nh + 7) / 8 items, one an XCD (see the kernel)
  const int items = a.nblocks * a.nh, cus = device_cus();
  const dim3 grid(8 * ((items + 7) / 8));
  // Waves that share a query block's keys: 2 up to two workgroups a CU (up to
  // one in local layers), 4 up to one over more than 512 keys. us a layer of the
  // whole pass with 1, 2 and 4. Global, hidden 768: 96 workgroups of 512 keys 82.4,
  // 78.9, 79.1; 192 of 2,048 169, 153, 149; 384 of 256 105.7, 105.2, 110.5, of
  // 4,096 280, 259, 292; 504 of 384 122.3, 120.8, 129; 612 139, 144, 155; 576 of
  // 6,144 432, 439, 493; 768 of 8,192 603, 605, 680; hidden 256: 248 of 256 59.4,
  // 57.7, 58.0; 512 of 1,024 147, 141, 152, of 8,192 501, 450, 508; 768 648, 654,
  // 733. Local: 96 of 512 75.0, 72.9; 240 of 256 91.7, 89.7; 288 104, 108. With
  // one, a grid of less than three workgroups a CU leaves SIMDs with one wave, or
  // with none; from two on their shared work costs more than that.
  if (a.window < 0) {
    if (items <= cus && a.max_n > 512) attn_main_kernel<true, 4><<<grid, 1024, 0, s>>>(a);
    else if (items <= 2 * cus) attn_main_kernel<true, 2><<<grid, 512, 0, s>>>(a);
    else attn_main_kernel<true, 1><<<grid, 256, 0, s>>>(a);
  } else {
    if (items <= cus) attn_main_kernel<false, 2><<<grid, 512, 0, s>>>(a);
    else attn_main_kernel<false, 1><<<grid, 256, 0, s>>>(a);
  }
}

}  // namespace ixh
