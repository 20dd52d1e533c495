// host_sched.cpp — the host-only scheduling of the C ABI (options, pass
// planning, the serving batcher's queue); no HIP calls, so the sanitizer
// builds of tests/sanitize run it on the CPU.
#include "host_sched.h"

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>

#include "../../include/indecis_hip.h"

namespace ixh {
namespace {

int fail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  return set_error(code, buf);
}

}  // namespace

int set_tuning(Tuning &t, int option, int64_t v, bool model_opts) {
  auto bad = [&]() { return fail(IXH_EINVAL, "indecis: option %d: value %lld out of range", option, (long long)v); };
  switch (option) {
  case IXH_OPT_GEMM:
    if (v < 0 || v > 2) return bad();
    t.gemm = (int)v;
    return IXH_OK;
  case IXH_OPT_GEMM_TILE:
    if (v < 0 || v > 2) return bad();
    t.gemm_tile = (int)v;
    return IXH_OK;
  default: break;
  }
  if (!model_opts) return fail(IXH_EINVAL, "linalg: option %d does not apply to a PackedB8", option);
  switch (option) {
  case IXH_OPT_PARTS:
    if (v < 0 || v > 4) return bad();
    t.parts = (int)v;
    return IXH_OK;
  case IXH_OPT_PASS_TOKENS:
    if (v < 1 || v > kMaxPassTokensOpt) return bad();
    t.pass_tokens = (int)v;
    return IXH_OK;
  case IXH_OPT_QKV_FUSED:
    if (v != 0 && v != 1) return bad();
    t.qkv_fused = (int)v;
    return IXH_OK;
  case IXH_OPT_QKV_HEADS:
    if (v != 1 && v != 2) return bad();
    t.qkv_heads = (int)v;
    return IXH_OK;
  case IXH_OPT_LN_SEG:
    if (v != 0 && v != 1) return bad();
    t.ln_seg = (int)v;
    return IXH_OK;
  case IXH_OPT_FUSE_RES:
    if (v < 0 || v > 4) return bad();
    t.fuse_res = (int)v;
    return IXH_OK;
  case IXH_OPT_FUSE_MLP:
    if (v < 0 || v > 2) return bad();
    t.fuse_mlp = (int)v;
    return IXH_OK;
  case IXH_OPT_QKV_KBLOCK:
    if (v != 0 && v != 1) return bad();
    t.qkv_kblock = (int)v;
    return IXH_OK;
  case IXH_OPT_FEW_ROWS:
    if (v != 0 && v != 1) return bad();
    t.few_rows = (int)v;
    return IXH_OK;
  default: return fail(IXH_EINVAL, "indecis: unknown option %d", option);
  }
}

int get_tuning(const Tuning &t, int option, int64_t *v) {
  switch (option) {
  case IXH_OPT_PARTS: *v = t.parts; return IXH_OK;
  case IXH_OPT_PASS_TOKENS: *v = t.pass_tokens; return IXH_OK;
  case IXH_OPT_QKV_FUSED: *v = t.qkv_fused; return IXH_OK;
  case IXH_OPT_QKV_HEADS: *v = t.qkv_heads; return IXH_OK;
  case IXH_OPT_GEMM: *v = t.gemm; return IXH_OK;
  case IXH_OPT_GEMM_TILE: *v = t.gemm_tile; return IXH_OK;
  case IXH_OPT_LN_SEG: *v = t.ln_seg; return IXH_OK;
  case IXH_OPT_FUSE_RES: *v = t.fuse_res; return IXH_OK;
  case IXH_OPT_FUSE_MLP: *v = t.fuse_mlp; return IXH_OK;
  case IXH_OPT_QKV_KBLOCK: *v = t.qkv_kblock; return IXH_OK;
  case IXH_OPT_FEW_ROWS: *v = t.few_rows; return IXH_OK;
  default: return fail(IXH_EINVAL, "indecis: unknown option %d", option);
  }
}

int pass_token_cap(int H, int I) {
  const int64_t per_token = 4 * (int64_t)std::max({3 * (int64_t)H, (int64_t)I, (int64_t)1});
  const int64_t cap = (((int64_t)1 << 31) - 1) / per_token;  // N * per_token < 2^31
  return (int)std::max<int64_t>(1, std::min<int64_t>(kMaxPassTokensOpt, cap));
}

int check_offs(const int32_t *offs, int B) {
  if (B < 0 || (B > 0 && !offs)) return fail(IXH_EINVAL, "modernbert: inconsistent batch");
  if (B == 0) return IXH_OK;
  if (offs[0] != 0) return fail(IXH_EINVAL, "modernbert: inconsistent batch");
  for (int b = 0; b < B; b++)
    if (offs[b + 1] < offs[b]) return fail(IXH_EINVAL, "modernbert: inconsistent batch");
  return IXH_OK;
}

void qkv_groups(const int32_t *offs, const int32_t *padoff, const std::vector<int32_t> &order, int slots,
                bool share, std::vector<int32_t> &groups) {
  constexpr int kSlots = 16, kSeqs = 8;
  groups.clear();
  std::vector<int> open[kSlots], count;  // groups with w free slots; their sequences
  for (int32_t b : order) {
    const int n = offs[b + 1] - offs[b];
    const int nb = std::max(2, (n + 63) / 64 * 2);
    int w = nb;
    while (w < slots && open[w].empty()) w++;  // the fullest group it fits into
    int g;
    if (w < slots) {
      g = open[w].back();
      open[w].pop_back();
    } else {
      w = slots;
      g = (int)count.size();
      groups.insert(groups.end(), kQkvGroup, 0);
      for (int s = 0; s < kSlots; s++) groups[(size_t)kQkvGroup * g + 4 * s] = -1;
      for (int s = 0; s < kSeqs; s++) groups[(size_t)kQkvGroup * g + 64 + s] = -1;
      count.push_back(0);
    }
    int32_t *e = &groups[(size_t)kQkvGroup * g];
    const int first = slots - w;
    for (int k = 0; k < nb; k++) {
      int32_t *s = e + 4 * (first + k);
      s[0] = 16 * b + k;
      s[1] = offs[b];
      s[2] = n;
      s[3] = padoff[b];
    }
    e[64 + count[g]++] = 16 * n + first;
    if (share && w - nb > 0 && count[g] < kSeqs) open[w - nb].push_back(g);
  }
}

// Alone, the tiles' workgroups read the rows too many times over past some
// rows. Sequences of 128 tokens, a pass with the 64-row MLP kernel (the 32-row
// one at hidden 768 and 256) over one on these: hidden 768 1.75 (1.49) at 1,024
// rows, 1.40 (1.20) at 2,048, 1.17 (1.00) at 3,072, 1.10 (0.94) at 4,096; 384
// 1.37 at 2,048, 1.08 at 4,096, 0.91 at 6,144; 256 1.20 (1.06) at 2,048, 1.10
// (0.98) at 2,560.
// In parts, whose workgroups fill the idle CUs too, it loses from the smallest
// batch that is split (4,096 rows) on, but at 384: us a pass of 8 layers (6 at
// 256) in two parts of sequences of 512, on these, with the 32- and with the 64-row
// kernel: 768 1,147, 1,059 and 1,196 at 4,096 rows, 1,389, 1,110 and 1,237 at
// 6,144; 256 606, 548 and 585 at 4,096; 384 883 and (64) 916 at 4,096, 904 and 921
// at 4,608, 931 and 924 at 5,120, 1,085 and 938 at 8,192 (three parts 1,058 and
// 1,066 at 4,608, four 1,217 and 1,198). One sequence a part, 840 of 4,200 rows in
// the second: 768 1,235 and 1,166, 256 843 and 806, 384 965 and 992 (of 5,000 1,031
// and 1,034). At 384 the smaller of two parts runs on these past that, beside the
// larger's whole-row kernels, other resources bound: both, the smaller alone and
// none of two near halves of sequences of 512, 735, 679 and 745 at 5,120 rows, 860,
// 732 and 749 at 8,192, (-) 890 and 800 at 10,240; with 0.4 of the rows in it
// (-) 1,235 and 1,282 at 8,000, with 0.3 1,355 and 1,328 (three sequences, 0.29 of
// 7,172: 22 layers, 3,510 and 3,800). At 768 the same up to 2,304 rows in it: 130
// ragged batches of 4,131-6,453 rows, the smaller part alone over none 0.92-1.06,
// 0.98 in the mean up to there and 1.03 past it; at 256 it loses always.
// Beside the passes of other threads: us a call of 6 layers on these and with
// the better whole-row kernel, sequences of 256. 768, two threads of 1,536 rows
// 291 and 324, of 2,048 335 and 330; four of 768 158 and 176, of 1,024 177 and 182,
// of 1,536 219 and 186; eight (four run at a time) of 512 137 and 169, of 1,024 178
// and 181, of 1,536 220 and 183. 384, two of 2,048 243 and 283, of 3,072 319 and
// 319; four of 1,536 142 and 152, of 2,048 162 and 155; eight 147 and 156, 166 and
// 153. 256, two of 1,536 193 and 198, of 2,048 199 and 191; four of 512 99 and 99,
// of 768 104 and 104, of 1,024 106 and 102; eight of 512 93 and 93, of 1,024 99 and 96.
bool split_rows_picked(int H, int N, int64_t batch, bool parts) {
  if (N > (H == 768 ? 3072 : H == 384 ? 4096 : 2048)) return false;
  if (batch <= N) return true;
  if (parts) {
    const bool smaller = 2 * (int64_t)N < batch && 4 * (int64_t)N > batch;
    return H == 384 ? batch <= 5000 || (batch <= 8192 && smaller) : H == 768 && N <= 2304 && smaller;
  }
  return N <= (H == 768 ? 1024 : H == 384 ? 1536 : 512) || batch <= (H == 768 ? 4095 : H == 384 ? 6144 : 3072);
}

// Alone, up to one round of the 256 CUs, where 64 rows a workgroup leave half of
// them idle. Hidden 768: 2.51 against 2.89 ms a pass at 6,144 rows, 2.90 against
// 3.18 at 8,192 (38 against 52 us a launch); past one round a 32-row block costs
// as much as a 64-row one. 256: a launch 12.9 against 19.1 us at 2,560 rows, 13.5
// and 19.3 at 4,096, 15.0 and 19.7 at 8,192. Beside others the CUs are shared: us
// a pass in two parts as above with the 32- and the 64-row kernel, sequences of
// 160 and of 512, 768 1,381 and 1,401, 1,474 and 1,469 at 10,240 rows, 1,581 and
// 1,542, 1,594 and 1,581 at 12,288, 1,977 and 1,887, 1,865 and 1,744 at 16,384; 256
// 631 and 656, 638 and 661 at 14,336, 671 and 683, 662 and 678 (1,024: 939 and 915)
// at 16,384. Ragged batches (20-512 to 500-3,000 tokens), the 32-row over the 64-row
// kernel: 768 0.95-1.03 at 9,000-10,000 rows, 0.99-1.06 at 11,000-12,700; 256 0.95-0.98
// at 15,000, 0.99-1.05 at 17,500. Threads, as above: 768, eight of 1,536 rows 183 and 201, of 2,048 199
// and 207, of 3,072 271 and 261; 256, eight of 3,072 126 and 131.
bool mlp32_picked(int H, int N, int64_t batch) {
  return N <= (H == 768 ? 2048 : 3072) || (N <= 8192 && (batch <= N || batch <= (H == 768 ? 10240 : 16384)));
}

// Rows do not depend on their batch (TestMatMul8RowsIndependent), so the
// results of several passes are those of one.
int plan_passes(const Tuning &t, int H, int I, const int32_t *offs, int B, std::vector<int> &cut) {
  const int cap = pass_token_cap(H, I);
  const int64_t limit = std::min(t.pass_tokens, cap);
  cut.assign(1, 0);
  for (int b = 0; b < B; b++) {
    const int n = offs[b + 1] - offs[b];
    if (n > cap)
      return fail(IXH_EINVAL, "modernbert: hip: sequence of %d tokens over the %d-token limit of a pass", n, cap);
    if (b > cut.back() && (int64_t)offs[b + 1] - offs[cut.back()] > limit) cut.push_back(b);
  }
  cut.push_back(B);
  return IXH_OK;
}

void split_points(const int32_t *offs, int B, int P, std::vector<int> &cut) {
  const int64_t N = B > 0 ? offs[B] : 0;
  cut.assign(P + 1, B);
  cut[0] = 0;
  for (int p = 1; p < P; p++) {
    int b = cut[p - 1];
    while (b < B && (int64_t)P * offs[b] < (int64_t)p * N) b++;
    cut[p] = b;
  }
}

BatchQueue::BatchQueue(int width, int workers, int max_rows, Encode encode)
    : width_(width), max_rows_(max_rows), encode_(std::move(encode)) {
  for (int i = 0; i < workers; i++) workers_.emplace_back(&BatchQueue::work, this);
}

BatchQueue::~BatchQueue() {
  close();
  for (std::thread &t : workers_) t.join();
}

void BatchQueue::close() {
  {
    std::lock_guard<std::mutex> lk(mu_);
    stop_ = true;
  }
  work_cv_.notify_all();
}

void BatchQueue::counts(int64_t *batches, int64_t *requests) {
  std::lock_guard<std::mutex> lk(mu_);
  *batches = batches_;
  *requests = requests_;
}

int BatchQueue::submit(const int32_t *ids, const int32_t *offs, int B, float *out, std::string &err) {
  Req r{ids, offs, B, offs[B], out};
  {
    std::unique_lock<std::mutex> lk(mu_);
    if (stop_) {
      err = "modernbert: batcher closed";
      return IXH_EINVAL;
    }
    queue_.push_back(&r);
    work_cv_.notify_one();
    done_cv_.wait(lk, [&] { return r.done; });
  }
  if (r.rc) err = r.err;
  return r.rc;
}

// batcher.work (batch.go:51-82)
void BatchQueue::work() {
  std::vector<Req *> batch;
  std::vector<int32_t> ids, offs;
  std::vector<float> pooled;
  std::string err;
  for (;;) {
    batch.clear();
    {
      std::unique_lock<std::mutex> lk(mu_);
      work_cv_.wait(lk, [&] { return stop_ || !queue_.empty(); });
      if (queue_.empty()) return;  // closed and drained
      batch.push_back(queue_.front());
      queue_.pop_front();
      int rows = batch[0]->rows;
      while (rows < max_rows_ && !queue_.empty()) {
        batch.push_back(queue_.front());
        rows += queue_.front()->rows;
        queue_.pop_front();
      }
    }
    int B = 0;
    for (Req *r : batch) B += r->B;
    offs.assign(B + 1, 0);
    ids.clear();
    int k = 0;
    for (Req *r : batch) {
      ids.insert(ids.end(), r->ids, r->ids + r->offs[r->B]);
      for (int s = 0; s < r->B; s++, k++) offs[k + 1] = offs[k] + (r->offs[s + 1] - r->offs[s]);
    }
    pooled.resize((size_t)B * width_);
    err.clear();
    const int rc = encode_(ids.data(), offs.data(), B, pooled.data(), err);
    size_t off = 0;
    for (Req *r : batch) {
      if (rc) {
        r->rc = rc;
        r->err = err;
      } else {
        memcpy(r->out, pooled.data() + off, sizeof(float) * (size_t)r->B * width_);
      }
      off += (size_t)r->B * width_;
    }
    {
      std::lock_guard<std::mutex> lk(mu_);
      for (Req *r : batch) r->done = true;
      batches_++;
      requests_ += (int64_t)batch.size();
    }
    done_cv_.notify_all();
  }
}

}  // namespace ixh
