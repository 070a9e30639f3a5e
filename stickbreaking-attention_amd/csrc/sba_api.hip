// C ABI of libsba.so (declarations and the upstream functions each entry point replaces are
// in include/sba.h).  Host code only validates, sizes and launches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>

#include "sba.h"
#include "sba_kernels.hpp"

namespace {

using namespace sba;

// Process-wide on purpose: PyTorch runs the backward on its own autograd thread.
std::atomic<int> g_timing{0};
std::atomic<int> g_dkdv_workgroups{0};   // sba_set_dkdv_workgroups
std::atomic<int> g_backward_form{0};     // sba_set_backward_form
int backward_form() { return g_backward_form.load() & 0xff; }
std::atomic<float> g_ms[3];

inline int cdiv_i(long long a, long long b) { return (int)((a + b - 1) / b); }

struct Sizes {
  int n_docs;        // documents the scheduler sees (fixed: batch)
  long long rows;    // batch * tokens
  int n_q_max, n_kv_max;
};

int check_problem(const sba_problem* p, bool fixed, Sizes* sz) {
  if (p == nullptr) return SBA_E_NULL;
  if (p->dtype != SBA_BF16 && p->dtype != SBA_F16) return SBA_E_DTYPE;
  if (p->head_dim <= 0 || p->head_dim > 256 || p->head_dim % 8) return SBA_E_HEAD_DIM;
  if (p->heads <= 0 || p->tokens < 0 || p->batch <= 0 || p->max_doc_len < 0) return SBA_E_SHAPE;
  if (fixed != ((p->flags & SBA_FIXED_LENGTH) != 0)) return SBA_E_SHAPE;
  if (fixed) {
    if (p->max_doc_len != p->tokens) return SBA_E_SHAPE;
  } else {
    if (p->batch != 1 || p->n_docs < 0) return SBA_E_SHAPE;
    if (p->n_docs > 0 && p->cu_seqlens == nullptr) return SBA_E_NULL;
  }
  sz->n_docs = fixed ? p->batch : p->n_docs;
  sz->rows = (long long)p->batch * p->tokens;
  sz->n_q_max = (int)(sz->rows / BM) + sz->n_docs + 1;
  sz->n_kv_max = (int)(sz->rows / BKV) + sz->n_docs + 1;
  return 0;
}

// Carry-table entries per head.  Fixed-length: exact.  Packed documents: the most any split of
// `tokens` tokens into n_docs documents of at most max_doc_len tokens can need.  A document
// occupies what its length rounded up to a multiple of 32 needs, and that need is convex in
// the length, so the worst split is as many longest documents as fit plus the rest, with every
// document's rounding (at most 31 tokens each) added to the token count.
long long table_entries_bound(const sba_problem* p, bool fixed) {
  if (fixed) return (long long)p->batch * tab_doc_entries(p->tokens);
  const long long tokens = (long long)p->tokens + 31ll * p->n_docs;
  long long lmax = (p->max_doc_len > 0 && p->max_doc_len < p->tokens) ? p->max_doc_len : p->tokens;
  lmax = (lmax + 31) & ~31ll;
  if (lmax <= 0) return 0;
  return (tokens / lmax) * tab_doc_entries((int)lmax) + tab_doc_entries((int)(tokens % lmax));
}

// Grid bounds of the dk/dv pass.  The second group of the key-tile list holds at most TAIL_TILES
// tiles of every document.  The first group holds ceil(L / BKV) - 1 tiles of a document of more
// than TAIL_TILES * BKV tokens and none of a shorter one: at most rows / BKV in all and, with the
// declared longest document, at most that many per document.  The declaration is checked on the
// device: a longer document makes every backward kernel return and the outputs NaN.
int declared_max_doc_len(const sba_problem* p, bool fixed) {
  return (fixed || p->max_doc_len <= 0 || p->max_doc_len > p->tokens) ? p->tokens : p->max_doc_len;
}
struct BwdBounds { int n_long_max, n_tail_max; };
BwdBounds backward_bounds(const sba_problem* p, bool fixed, const Sizes& sz) {
  const int max_doc_len = declared_max_doc_len(p, fixed);
  const long long per_doc = (max_doc_len + BKV - 1) / BKV - kv_tail_tiles(max_doc_len);
  BwdBounds b;
  b.n_long_max = (int)std::min<long long>(sz.rows / BKV, per_doc * sz.n_docs);
  b.n_tail_max = (int)std::min<long long>(sz.n_kv_max, (long long)TAIL_TILES * sz.n_docs);
  return b;
}

size_t schedule_bytes(const Sizes& sz) {
  size_t words = SCHED_HDR + TILE_WORDS * ((size_t)sz.n_q_max + sz.n_kv_max) + 6 * (size_t)sz.n_docs + 2;
  return (words * sizeof(int) + 255) & ~(size_t)255;
}

int check_view(const sba_view* v, bool need_ptr) {
  if (v == nullptr) return SBA_E_NULL;
  if (need_ptr && v->ptr == nullptr) return SBA_E_NULL;
  return 0;
}

// 16-byte vector loads/stores need every row start aligned: strides multiple of 8 elements.
// Tile loads address a (document, head) slice with 32-bit byte offsets: the token stride must
// keep every row of the slice (plus one tile of slack) below 2 GiB.
int check_mat(const sba_view* v, const sba_problem* p, bool out = false) {
  int e = check_view(v, true);
  if (e) return e;
  if ((v->stride_b % 8) || (v->stride_h % 8) || (v->stride_t % 8) || ((uintptr_t)v->ptr % 16)) return SBA_E_STRIDE;
  if (v->stride_t < p->head_dim) return SBA_E_STRIDE;
  if (((long long)p->tokens + 8 * BM) * v->stride_t * (out && (p->flags & SBA_F32_OUT) ? 4 : 2) >= (1ll << 31)) return SBA_E_SHAPE;
  return 0;
}

View to_view(const sba_view* v) {
  View r;
  r.ptr = v ? (char*)v->ptr : nullptr;
  r.sb = v ? v->stride_b : 0;
  r.sh = v ? v->stride_h : 0;
  r.st = v ? v->stride_t : 0;
  return r;
}
// An output's view.  The kernels address every tensor in 16-bit words, so float32 strides count double.
View to_view_out(const sba_view* v, const sba_problem* p) {
  View r = to_view(v);
  if (p->flags & SBA_F32_OUT) { r.sb *= 2; r.sh *= 2; r.st *= 2; }
  return r;
}

// The counter words at the end of a table workspace of `table_bytes` bytes.
unsigned* work_words(float* table, size_t table_bytes) {
  return reinterpret_cast<unsigned*>(table) + (table_bytes / sizeof(unsigned) - WORK_WORDS);
}

// Compute units of the current device (0 if it cannot be asked: launches then take one workgroup per item).
int device_cus() {
  static std::atomic<int> cached[64];   // by device ordinal; 0 = not asked yet
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if ((n = cached[dev].load(std::memory_order_relaxed)) > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
  cached[dev].store(n, std::memory_order_relaxed);
  return n;
}

int check_arch() {
  static int cached = -1;   // immutable once set
  if (cached >= 0) return cached ? 0 : SBA_E_ARCH;
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return SBA_E_ARCH;
  cached = std::strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 0;
  return cached ? 0 : SBA_E_ARCH;
}

// Brackets one compute launch with HIP events on the caller's stream.  Nothing waits here: the
// pair is parked and resolved when sba_last_kernel_ms asks for it, so that timed kernels follow
// one another on the device exactly as untimed ones do.
struct EventPair {
  hipEvent_t e0 = nullptr, e1 = nullptr;
};
std::mutex g_ev_mutex;
EventPair g_ev[3];

struct Timer {
  EventPair ev;
  hipStream_t s;
  int which;
  bool on;
  Timer(int which_, hipStream_t s_, bool allowed = true) : s(s_), which(which_), on(allowed && g_timing.load() != 0) {
    if (on) {
      on = hipEventCreate(&ev.e0) == hipSuccess && hipEventCreate(&ev.e1) == hipSuccess;
      if (on) (void)hipEventRecord(ev.e0, s);
    }
  }
  ~Timer() {
    EventPair done = ev;   // (timing off, or creation failed half-way: nothing to park)
    if (on) {
      (void)hipEventRecord(ev.e1, s);
      std::lock_guard<std::mutex> lock(g_ev_mutex);
      done = g_ev[which];
      g_ev[which] = ev;
    }
    if (done.e0) (void)hipEventDestroy(done.e0);
    if (done.e1) (void)hipEventDestroy(done.e1);
  }
};

// Entries per head that a table workspace holds: its last WORK_WORDS words are the work counters of the call's
// persistent launches.
int64_t table_stride(const sba_problem* p, size_t table_bytes) {
  if (table_bytes < WORK_WORDS * sizeof(unsigned)) return 0;
  return (int64_t)((table_bytes - WORK_WORDS * sizeof(unsigned)) / sizeof(float) / (size_t)p->heads) & ~(int64_t)31;   // heads start on 128-byte lines
}

// `table_bytes`: size of EACH carry table handed in (ignored when none is).
int fill_common(const sba_problem* p, bool fixed, const Sizes& sz, const void* schedule, size_t sched_bytes,
                bool with_table, size_t table_bytes, KArgs* a) {
  if (schedule == nullptr) return SBA_E_NULL;
  if (reinterpret_cast<uintptr_t>(schedule) & 15) return SBA_E_STRIDE;   // kernels read the header as one 16-byte word
  if (sched_bytes < schedule_bytes(sz)) return SBA_E_WORKSPACE;
  a->tab_stride = -1;
  if (with_table) {
    if (table_bytes < WORK_WORDS * sizeof(unsigned)) return SBA_E_WORKSPACE;
    a->tab_stride = table_stride(p, table_bytes);
    // fixed-length needs are known here; packed documents are checked on the device against
    // what the scheduler found (kernels refuse to run, outputs are filled with NaN)
    if (fixed && a->tab_stride < table_entries_bound(p, true)) return SBA_E_WORKSPACE;
    if (a->tab_stride <= 0) return SBA_E_WORKSPACE;
  }
  a->sched = reinterpret_cast<const int*>(schedule);
  a->kv_list_off = SCHED_HDR + TILE_WORDS * sz.n_q_max;
  a->n_kv_alloc = sz.n_kv_max;
  a->docs_off = a->kv_list_off + TILE_WORDS * sz.n_kv_max + chain_docs_offset(sz.n_docs);
  a->n_docs = sz.n_docs;
  a->heads = p->heads;
  a->head_dim = p->head_dim;
  a->tokens = p->tokens;
  a->fuse = (p->flags & SBA_FUSE_REMAINDER) ? 1 : 0;
  a->out_f32 = (p->flags & SBA_F32_OUT) ? 1 : 0;
  a->inv_temp = p->inv_temp;
  a->c = p->inv_temp * 1.4426950408889634f;
  return 0;
}

// Where the kernels for problems that leave most of the chip idle (sba_small.hip) are the faster ones: both times
// estimated, in us, from what 90 problems of 4 to 32 heads, 128 to 4096 tokens and 1 to 16 documents took at head_dim
// 32, 64, 128 and 256.
//   The general kernels take at least `base` and `step` for every 32 tokens of the longest document (more, once
//   workgroups share a compute unit); the small ones their own `small_base` and the longer of what the longest
//   document's rounds of 128 take one after the other (`round` each) and of what `at_once` workgroups at a time need:
//   `group` each and `per_round` for every round, of which a workgroup has half its document's and half a one for the
//   remainder.  (By tokens, documents are about halfway between the mean and the longest.  A last group that is not
//   full counts half as if it were: 11 heads of 3 x 686 tokens at head_dim 80, 1.4 groups, took 23.5 us for 21.2.  A
//   group of workgroups for rows behind their document's end takes 2 us: 3 heads of 2212 tokens in 17 documents at
//   head_dim 256 took 23.6 us for 21.6.)
// `gain` must be gained, and 2 us, with which four times as many workgroups pay at the dispatcher (the forward of 13
// prompts of up to 172 tokens: 9.9 us alone with either, 10.6 for 11.3 in a row).
struct SmallCost { double base, step, small_base, round, group, per_round; int at_once; };
bool small_wins(const SmallCost* costs, double gain, const sba_problem* p, bool fixed, const Sizes& sz) {
  if (!(p->flags & SBA_PRODUCT_SPACE) || sz.n_docs <= 0) return false;
  const SmallCost& c = costs[p->head_dim <= 32 ? 0 : (p->head_dim <= 64 ? 1 : (p->head_dim <= 128 ? 2 : 3))];
  const double longest = declared_max_doc_len(p, fixed), typical = 0.5 * (longest + std::min(longest, (double)sz.rows / sz.n_docs));
  const double round = 32 * SMALL_WAVES, blocks = fixed ? (double)p->batch * ((p->tokens + 31) / 32) : sz.rows / 32.0 + 0.5 * sz.n_docs;
  double groups = blocks * p->heads / c.at_once;
  if (groups > 1.0) groups = 0.5 * (groups + std::ceil(groups));
  const double spare = ((double)sz.n_q_max * (BM / 32) - blocks) * p->heads / c.at_once;    // groups of workgroups that find nothing to do
  const double small = c.small_base + 2.0 * spare + std::max(c.round * longest / round, groups * (c.group + c.per_round * (0.5 * typical / round + 0.5)));
  return std::max(gain * small, small + 2.0) < c.base + c.step * longest / 32;
}
// Of 164 problems (general / few tiles, us) none of the 44 taken loses and they gain 1.41 by the geometric mean
// (head_dim 64: 4 heads x 512 14.4 / 9.7, 16 x 4096 80 / 68, 32 x 1024 23.5 / 17.2; head_dim 256, whose line serves 129
// on: 4 x 512 28 / 17, 16 x 1024 48 / 34).  Of the 120 left to fwd_kernel eight would gain more than a tenth, up to
// 1.24 (12 heads x 3001 tokens in 17 documents 20.8 / 17.7, 13 heads of 2 x 1360 30.2 / 24.5): `base` and `step` are
// those of a document alone.  Most lose (head_dim 64: 16 heads of 4 x 1024 24.8 / 26.9; head_dim 128: 32 x 2048 57 /
// 73; head_dim 256: 16 x 2048 88 / 95) or gain less than 4 x the workgroups may cost (32 x 2048 at 64 42 / 39).
bool forward_small(const sba_problem* p, bool fixed, const Sizes& sz) {
  if (p->flags & SBA_GENERAL_FORWARD) return false;
  if (p->flags & SBA_FEW_TILES_FORWARD) return (p->flags & SBA_PRODUCT_SPACE) && sz.n_docs > 0;
  static constexpr SmallCost COSTS[4] = {{5.2, 0.46, 5.5, 0.75, 2.7, 1.33, 1024}, {5.8, 0.55, 6.2, 0.90, 3.4, 1.66, 1024},
                                         {6.5, 0.73, 7.0, 1.19, 4.0, 1.60, 512}, {8.7, 1.22, 10.0, 1.93, 5.0, 2.0, 256}};
  return small_wins(COSTS, 1.1, p, fixed, sz);
}
// The backward, both passes, against the one-pass form (head_dim 64: 4 heads x 512 36.2 / 23.5, 16 x 1024 55 / 38, 16 x
// 2048 91 / 80, left out 16 x 4096 229 / 219, 32 x 4 x 256 28 / 34; head_dim 128: 4 heads x 512 42 / 32, 16 x 512 43 /
// 33.5, left out 16 x 1024 66 / 66).  Documents of one or two blocks are with the general two passes (head_dim 64: 64
// tokens 16.0 / 16.8; 2 heads of 68 documents of 38 tokens on average and 95 at most 18.5 / 23.9).
bool backward_small(const sba_problem* p, bool fixed, const Sizes& sz) {
  if (backward_form() != 0 || p->head_dim > 128 || declared_max_doc_len(p, fixed) <= 64 || sz.rows <= 64ll * sz.n_docs) return false;
  static constexpr SmallCost COSTS[3] = {{16.0, 1.04, 12.5, 1.9, 3.7, 2.35, 512}, {17.0, 1.15, 14.0, 2.34, 6.0, 2.75, 512}, {19.0, 1.42, 18.5, 3.6, 9.5, 3.6, 256}};
  return small_wins(COSTS, 1.05, p, fixed, sz);
}

// Workgroups per head: documents of more than 128 tokens one each, the others two or four (each class rounded up).
int short_parts(const sba_problem* p, bool fixed, const Sizes& sz) {
  const int longest = declared_max_doc_len(p, fixed);
  if (longest <= 64) return (sz.n_docs + 3) / 4;
  const long long alone = longest <= 128 ? 0 : std::min<long long>(sz.n_docs, sz.rows / 129);
  return (int)(alone + (sz.n_docs - alone + 1) / 2 + 1);
}
// Where bwd_short_kernel (sba_small.hip) is the faster one: short documents, and enough of them for a wave on two of
// five SIMDs (a wave has 64 tokens; dq and dk/dv passes / one-pass form before, us, at head_dim 64: 32 heads of 8 x 256
// tokens 44.5 / 31.6, of 32 x 128 49.6 / 35.3, of 128 x 33 75 / 44.3, of 128 x 256 390 / 320, 8 heads of 5000 tokens in
// documents of 1 .. 256 33.6 / 30.3).  With 24 K to 40 K rows (tokens x heads), gain over the kernels for few tiles and
// the one-pass form by kinds of lengths: head_dim 32 1.07 .. 1.66, 64 0.98 .. 1.60, documents of up to 64 tokens at 96
// and 128 1.05 .. 1.99; with 16 K 0.87 .. 1.23.  Above head_dim 64 a compute unit has room for one workgroup, and of
// longer documents only what the one-pass form does not take well gains:
// - most documents far shorter than the longest, each of which is a key tile, nearly empty, to the one-pass form: 172
//   problems of 4 to 32 heads and 2 K to 32 K tokens at head_dim 96 and 128 whose mean is up to 0.45 of the longest
//   1.40 times as fast by the geometric mean (0.98 .. 2.04; 32 heads x 16 K tokens in documents of 16 .. 256 438 /
//   406), with the longest up to 128 also up to 0.55 (1.08 .. 1.31);
// - what one round of workgroups does, and 256 key tiles would not: 201 problems of 40 K to 64 K rows at head_dim 72,
//   96 and 128 1.21 (0.99 .. 1.36).
// Beyond it loses (head_dim 128: 16 heads of 128 x 128 153 / 164, of 100 x 96 106 / 115, of 64 x 256 191 / 204; 16
// heads of 16 x 128 20 % slower).
bool backward_short(const sba_problem* p, bool fixed, const Sizes& sz) {
  if (backward_form() != 0) return false;
  const long long longest = declared_max_doc_len(p, fixed);
  if (!(p->flags & SBA_PRODUCT_SPACE) || p->head_dim > 128 || sz.n_docs <= 0 || sz.n_docs > RANK_LIMIT || longest > 32 * SHORT_BLOCKS) return false;
  if (p->head_dim <= 64 || longest <= 64) return sz.rows * p->heads >= 24000;
  return sz.rows * p->heads >= 40000 &&
         (20ll * sz.rows <= (longest <= 128 ? 11 : 9) * longest * sz.n_docs || (short_parts(p, fixed, sz) - 1) * (long long)p->heads <= device_cus());
}

// Whether the query tiles of documents of like length are listed tile-major (see sched_kernel): in launches of up to
// four rounds of the chip, and of more the fewer heads there are.  What is gained is the launch's end, where
// document-major the last document's most expensive tile starts late: the less the more rounds there are.  What it
// costs is that the tiles of a (document, head) that are under way at a time share its K/V rows in the caches with
// fewer others, the more heads (and documents) there are.  The line is that of 456 shapes of equal documents (two
// rounds and more, 1 to 32 heads, 512 to 32768 tokens, head_dim 64, 128 and 256, forward and dq pass): 1.067 times as
// fast as document-major by the geometric mean, tile-major always 1.050.  Forward, us, document-major / tile-major,
// head_dim 128: 12 heads of 4 x 4096 (2 rounds) 249 / 200, 8 of 8 x 4096 (2.7) 305 / 256, 12 of 8 x 4096 (4) 440 / 377,
// 2 of 16 x 8192 (2.7) 616 / 484; left out 16 heads of 4 x 8192 (5.3) 985 / 1020, 32 of 8 x 2048 (5.3) 291 / 341, 32 of
// 8 x 4096 (10.7) 1069 / 1410.
bool list_in_classes(const sba_problem* p, const Sizes& sz) {
  const int cus = device_cus();
  const long long items = sz.rows / BM * p->heads, round = (long long)fwd_per_cu(p->head_dim) * (cus > 0 ? cus : 256);
  return items <= 4 * round || items * p->heads <= 48 * round;
}

int forward(const sba_problem* p, bool fixed, const void* schedule, size_t sched_bytes, const sba_view* q,
            const sba_view* k, const sba_view* v, const sba_view* o, const sba_view* rem, float* stick,
            size_t table_bytes, float* weights, size_t weights_bytes, void* stream, bool timed = true) {
  Sizes sz;
  int e = check_problem(p, fixed, &sz);
  if (e) return e;
  const bool table_only = (p->flags & SBA_TABLE_ONLY) != 0;   // nothing but the carry table is written; v, o, rem are not looked at
  if (table_only && (stick == nullptr || weights != nullptr)) return SBA_E_NULL;
  if ((e = check_mat(q, p)) || (e = check_mat(k, p))) return e;
  if (!table_only && ((e = check_mat(v, p)) || (e = check_mat(o, p, true)) || (e = check_view(rem, true)))) return e;
  if (weights != nullptr &&
      weights_bytes / sizeof(float) < (size_t)p->batch * p->heads * (size_t)p->tokens * (size_t)p->tokens)
    return SBA_E_WORKSPACE;
  KArgs a;
  std::memset(&a, 0, sizeof(a));
  if ((e = fill_common(p, fixed, sz, schedule, sched_bytes, stick != nullptr, table_bytes, &a))) return e;
  if ((e = check_arch())) return e;
  if (sz.rows == 0) return 0;
  a.q = to_view(q); a.k = to_view(k);
  if (table_only) a.v = a.o = a.rem = to_view(k);   // (placeholders: the kernel touches none of them)
  else { a.v = to_view(v); a.o = to_view_out(o, p); a.rem = to_view_out(rem, p); }
  a.stick = stick;
  a.weights = weights;
  // (the grid may hold a few slots more than there are items)
  const long long cus = device_cus(), items = (fixed ? (long long)p->batch * ((p->tokens + BM - 1) / BM) : sz.rows / BM) * p->heads;
  a.lg_deal = items > cus && items <= fwd_per_cu(p->head_dim) * cus && (cus & (cus - 1)) == 0 ? __builtin_ctzll(cus) : NO_DEAL;
  a.heads_inv = 0xffffffffu / (unsigned)p->heads;
  a.n_items = (int)std::min<long long>(0x7fffffff, (long long)sz.n_q_max * p->heads);
  a.clear_spare = fixed ? 0 : 1;
  a.nan_pair = p->dtype == SBA_F16 && !a.out_f32 ? 0x7e007e00u : 0x7fc07fc0u;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  hipError_t he = hipSuccess;
  {   // (packed input without a single document still launches: the spare workgroups clear the outputs)
    Timer tm(0, s, timed);
    if (weights == nullptr && !table_only && forward_small(p, fixed, sz))
      he = (p->dtype == SBA_F16 ? f16::launch_fwd_small : bf16::launch_fwd_small)(a, (p->flags & SBA_ATTEND_CURRENT) != 0, sz.n_q_max, s);
    else he = (p->dtype == SBA_F16 ? f16::launch_fwd : bf16::launch_fwd)(a, p->head_dim, (p->flags & SBA_ATTEND_CURRENT) != 0,
                    (p->flags & SBA_PRODUCT_SPACE) != 0, weights != nullptr ? 1 : (table_only ? 2 : 0), sz.n_q_max, s);
  }
  return (int)he;
}

int backward(const sba_problem* p, bool fixed, const void* schedule, size_t sched_bytes, const sba_view* q,
             const sba_view* k, const sba_view* v, const sba_view* go, const sba_view* grem, const float* stick,
             float* gtab, size_t table_bytes, const sba_view* dq, const sba_view* dk, const sba_view* dv,
             void* stream) {
  Sizes sz;
  int e = check_problem(p, fixed, &sz);
  if (e) return e;
  if ((e = check_mat(q, p)) || (e = check_mat(k, p)) || (e = check_mat(v, p)) || (e = check_mat(go, p)) ||
      (e = check_mat(dq, p, true)) || (e = check_mat(dk, p, true)) || (e = check_mat(dv, p, true)))
    return e;
  if (stick == nullptr || gtab == nullptr) return SBA_E_NULL;
  KArgs a;
  std::memset(&a, 0, sizeof(a));
  if ((e = fill_common(p, fixed, sz, schedule, sched_bytes, true, table_bytes, &a))) return e;
  if ((e = check_arch())) return e;
  if (sz.rows == 0) return 0;
  a.q = to_view(q); a.k = to_view(k); a.v = to_view(v); a.go = to_view(go);
  a.grem = to_view(grem);
  a.dq = to_view_out(dq, p); a.dk = to_view_out(dk, p); a.dv = to_view_out(dv, p);
  a.stick = const_cast<float*>(stick);
  a.gtab = gtab;
  // The main kernel of the dk/dv pass fills a compute unit with one workgroup.  With many more key tiles than
  // compute units it is launched once per compute unit and walks the tiles itself (see work_next in
  // sba_device.hpp); with few it pays more for the hand-over between tiles than the hardware does for a
  // fresh workgroup (measured: 960 tiles on 256 compute units, 124 against 118 us).
  const int forced = g_dkdv_workgroups.load();
  a.work = work_words(gtab, table_bytes);
  a.resident = forced > 0 ? std::max(8, forced & ~7) : (forced < 0 ? 0 : device_cus());
  a.min_items_each = forced > 0 ? 1 : 8;
  a.max_doc_len = declared_max_doc_len(p, fixed);
  const BwdBounds bb = backward_bounds(p, fixed, sz);
  const int n_long_max = bb.n_long_max, n_tail_max = bb.n_tail_max;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool ac = (p->flags & SBA_ATTEND_CURRENT) != 0, prod = (p->flags & SBA_PRODUCT_SPACE) != 0;
  a.clear_spare = fixed ? 0 : 1;
  a.nan_pair = p->dtype == SBA_F16 && !a.out_f32 ? 0x7e007e00u : 0x7fc07fc0u;
  hipError_t he = hipSuccess;
  if (backward_short(p, fixed, sz)) {
    Timer tm(2, s);
    return (int)(p->dtype == SBA_F16 ? f16::launch_bwd_short : bf16::launch_bwd_short)(a, ac, short_parts(p, fixed, sz), s);
  }
  if (backward_small(p, fixed, sz)) {
    {
      Timer tm(1, s);
      he = (p->dtype == SBA_F16 ? f16::launch_bwd_dq_small : bf16::launch_bwd_dq_small)(a, ac, sz.n_q_max, s);
    }
    if (he == hipSuccess) {
      Timer tm(2, s);
      he = (p->dtype == SBA_F16 ? f16::launch_bwd_dkdv_small : bf16::launch_bwd_dkdv_small)(a, ac, sz.n_q_max, s);
    }
    return (int)he;
  }
  {
    Timer tm(1, s);
    he = (p->dtype == SBA_F16 ? f16::launch_bwd_dq : bf16::launch_bwd_dq)(a, p->head_dim, ac, prod, sz.n_q_max, s);
  }
  if (he == hipSuccess && sz.n_docs > 0) {
    Timer tm(2, s);
    he = (p->dtype == SBA_F16 ? f16::launch_bwd_dkdv : bf16::launch_bwd_dkdv)(a, p->head_dim, ac, prod, n_long_max, n_tail_max, s);
  }
  return (int)he;
}

// ---- the one-pass backward (sba_chain.hip) ------------------------------------------------------------
int chain_width(int head_dim) { return head_dim <= 64 ? 64 : 128; }   // columns of its rows
struct ChainScratch { size_t partial, carry, flags, queues, homes, total; };   // byte offsets
ChainScratch chain_scratch(const sba_problem* p, const Sizes& sz) {
  const size_t tiles = (size_t)p->heads * (size_t)sz.n_kv_max;
  auto line = [](size_t n) { return (n + 255) & ~(size_t)255; };
  ChainScratch c;
  c.partial = 0;
  c.carry = line(tiles * BM * chain_width(p->head_dim) * sizeof(float));
  c.flags = c.carry + line(2 * tiles * BM * sizeof(float));
  c.queues = c.flags + line(tiles * sizeof(int));
  c.homes = c.queues + line(CHAIN_QUEUES * CHAIN_QUEUE_STRIDE * sizeof(unsigned));
  c.total = c.homes + line(CHAIN_HOMES * sizeof(int));
  return c;
}

// What a problem's chains look like from the host: one document of the longest declared length, the others alike.
struct Chains { long long number, longest, other, squares, per_xcd, long_per_xcd, most; };   // squares: of a chain's length, over all of them; most: over those of one XCD
Chains chains_of(const sba_problem* p, bool fixed, const Sizes& sz) {
  Chains c;
  c.number = (long long)sz.n_docs * p->heads;
  c.longest = std::min<long long>(declared_max_doc_len(p, fixed), sz.rows);
  c.other = sz.n_docs > 1 ? (sz.rows - c.longest) / (sz.n_docs - 1) : 0;
  c.squares = p->heads * (c.longest * c.longest + (sz.n_docs - 1) * c.other * c.other);
  c.per_xcd = (c.number + CHAIN_QUEUES - 1) / CHAIN_QUEUES;          // (dealt out longest first)
  c.long_per_xcd = (p->heads + CHAIN_QUEUES - 1) / CHAIN_QUEUES;
  c.most = c.long_per_xcd * c.longest * c.longest + (c.per_xcd - c.long_per_xcd) * c.other * c.other;
  return c;
}

// ---- the two passes of head_dim 129 .. 256 with p and dz handed on (sba_wide.hip) -----------------------
// The dq pass stores p and dz, 4 bytes per causal pair, and the dk/dv pass multiplies them instead of forming both
// again.  It is the faster form of 99 problems of 2 to 16 heads and 256 to 8192 tokens in 1 to 60 documents at head_dim
// 136, 160 and 256 (1.12 by the geometric mean, 0.98 ..  1.39) and of the larger ones (16 heads x 16 K tokens in eight
// documents at 256: 1515 -> 1180 us, 12 x 4 x 4096 1520 -> 1203).  Heads are independent: where the room (32 times a
// carry table, 32 bytes more for every query and 32 keys) does not hold them all, equal groups of them are taken one
// after the other in the same place (head_dim 256, us, scores formed twice / in groups: 16 heads of 2 x 8192 3826 /
// 2960, 32 of 16 x 2048 4527 / 3690, 16 of 8 x 4096 3948 / 3342, 5 of 2 x 16384 4823 / 3741).  A group has to fill the
// chip by itself, its launches ending with the most expensive of its tiles: the line is at three quarters as many of
// its blocks per compute unit as that tile has (3 heads of 20000, 0.92 of them, 4241 / 3236; 2 of 24576, 0.75, 4035 /
// 3604; 1 of 32768, 0.5, 7045 / 8998).  How many blocks there are is what the carry table holds, if it was sized by the
// documents' lengths.  A table of the most that the declared sizes allow says nothing about them: the room goes by
// that, the line by the least they allow (16 heads of one document of 16384 and 96 of 512 9280 us with scores formed
// twice, 7276 in groups of six by the lengths; the most leaves room for one head at a time, 17740).
struct Given { int group; long long entries; size_t bytes; };   // heads at a time (0: not in this form), table entries of each, room for all
Given given(const sba_problem* p, bool fixed, const Sizes& sz, size_t table_bytes) {
  const long long most = table_entries_bound(p, fixed), held = table_bytes ? (long long)table_stride(p, table_bytes) : most;
  Given g = {0, std::min(most, held), 0};
  if (!(p->flags & SBA_PRODUCT_SPACE) || p->head_dim <= 128 || sz.n_docs <= 0) return g;
  const size_t each = (size_t)g.entries * (2 * PZ_WORDS);
  const long long room = (long long)(GIVEN_SCRATCH_MAX / std::max<size_t>(each, 1));
  if (room >= p->heads) {
    g.group = p->heads;
  } else if (room > 0) {
    const int groups = (int)((p->heads + room - 1) / room), heads = (p->heads + groups - 1) / groups;
    const long long cus = device_cus() > 0 ? device_cus() : 256;
    const long long blocks = held < most ? g.entries : std::min(g.entries, chains_of(p, fixed, sz).squares / p->heads / 64);
    if (heads * blocks >= 3 * cus * declared_max_doc_len(p, fixed)) g.group = heads;
  }
  g.bytes = (size_t)g.group * each;
  return g;
}

int backward_given(const sba_problem* p, bool fixed, const Sizes& sz, KArgs& a, void* scratch, const Given& g, hipStream_t s) {
  const int group = g.group;
  a.pz = static_cast<unsigned short*>(scratch);
  a.pz_entries = g.entries;
  const BwdBounds bb = backward_bounds(p, fixed, sz);
  const DkdvGrid grid = dkdv_grid(false, bb.n_long_max, bb.n_tail_max, sz.n_kv_max);
  const bool ac = (p->flags & SBA_ATTEND_CURRENT) != 0, f16 = p->dtype == SBA_F16, whole = group == p->heads;
  hipError_t he = hipSuccess;
  Timer all(2, s, !whole);                    // (several groups: one figure for everything, like the one-pass form)
  for (int head = 0; head < p->heads && he == hipSuccess; head += group) {
    a.heads = std::min(group, p->heads - head);
    {
      Timer tm(1, s, whole);
      he = (f16 ? f16::launch_bwd_dq_wide : bf16::launch_bwd_dq_wide)(a, ac, true, sz.n_q_max, s);
    }
    if (he == hipSuccess) {
      Timer tm(2, s, whole);
      he = (f16 ? f16::launch_bwd_dkdv_given : bf16::launch_bwd_dkdv_given)(a, grid.main_tiles, s);
    }
    for (View* v : {&a.q, &a.k, &a.v, &a.go, &a.grem, &a.dq, &a.dk, &a.dv})
      if (v->ptr != nullptr) v->ptr += 2 * (int64_t)group * v->sh;   // (strides count 16-bit words)
    a.stick += (int64_t)group * a.tab_stride;
  }
  return (int)he;
}

// Whether the kernels can take the problem at all: a device of eight XCDs with 32 compute units each, ranked documents,
// room for the queue's groups in LDS and 32-bit offsets into a document's partial dq.
bool chain_possible(const sba_problem* p, bool fixed, const Sizes& sz) {
  const long long chains = (long long)sz.n_docs * p->heads;
  return (p->flags & SBA_PRODUCT_SPACE) && p->head_dim <= 128 && sz.n_docs > 0 && sz.n_docs <= RANK_LIMIT &&
         chains <= (long long)CHAIN_QUEUES * CHAIN_GROUP * CHAIN_MAX_GROUPS &&
         ((long long)declared_max_doc_len(p, fixed) + BM) * chain_width(p->head_dim) * 4 < (1ll << 31) && device_cus() == 256;
}
// Steps of 64 queries instead of 32 (head_dim <= 64).  They do more per step and CU (4 x 16 x 2048 at head_dim 64: 159
// us for 187) but a key tile lags its predecessor by three steps of either size, so as long as that lag is what a
// problem takes (8 heads of 8192 keys: 430 us for 372) the small ones are the better ones.  The line: the work of a CU
// in steps, squares / (2 x 64 x 128 x 256 CUs), against the steps of the longest document and a twentieth more (32
// heads of 7 K tokens in six documents of up to 3000 264 us for 298, 12 x 3 x 2500 161 for 175, 4 x 2 x 8192 428 for
// 371).  Up to 4096 keys, where the XCDs need not come out even (see chain_wanted), it is the work of a CU of the
// busiest one (20 heads of 3000 at head_dim 32 142 us for 152, 26 of 2200 114 for 120).
bool chain_wide(const sba_problem* p, bool fixed, const Sizes& sz) {
  const int form = backward_form();
  if (form == 2 || form == 3) return form == 3;
  const Chains c = chains_of(p, fixed, sz);
  return 20 * (c.longest <= 32 * BKV ? CHAIN_QUEUES * c.most : c.squares) >= 21 * c.longest * 65536;
}
// Whether Q and dO rows stream past an XCD's L2 (4 MiB) instead of staying in it, where they compete with the partial
// dq on its way from key tile to key tile.  They are better kept until the rows an XCD has to do, whatever their
// documents, are several times what it holds: time streamed over kept, on 420 problems of 8 to 32 heads in documents of
// 128 to 8192 tokens, at head_dim 128 (512 bytes a row) 1.03 .. 1.08 up to 16 K rows and 0.96 .. 1.0 from 24 K on, at
// 96 1.03 .. 1.08 up to 16 K rows, and of documents of up to 1024 1.0 at 24 K and 0.97 .. 1.0 at 32 K, of longer ones
// 1.0 .. 1.08 everywhere, at 64 1.0 .. 1.08 up to 32 K.  A document of one tile hands nothing on (0.93 .. 1.0).
bool chain_streams(const sba_problem* p, bool fixed, const Sizes& sz) {
  const int width = used_width(p->head_dim);
  const long long longest = declared_max_doc_len(p, fixed), rows = sz.rows * p->heads / CHAIN_QUEUES;
  if (width < 96) return false;
  return longest <= BKV || (width == 128 ? rows > 20 * 1024 : rows > 28 * 1024 && longest + sz.rows / sz.n_docs <= 2048);
}
// Where the one-pass form is the faster one (gain over the two passes; measured on 1220 problems of 1 to 32 heads and
// 512 to 200 K tokens in 1 to 128 documents, declared lengths exact).  On 1600 others, drawn with more spread among a
// problem's lengths, the choice of form and step costs 0.6 % against the best at head_dim 80 to 128, 3.1 % at 64 and
// 4.0 % at 32 by the geometric mean, 1.4 to 1.5 times at the worst.
bool chain_wanted(const sba_problem* p, bool fixed, const Sizes& sz) {
  const int form = backward_form();
  if (form == 1 || !chain_possible(p, fixed, sz)) return false;
  if (form == 2 || form == 3) return true;
  if (backward_short(p, fixed, sz) || backward_small(p, fixed, sz)) return false;
  const Chains c = chains_of(p, fixed, sz);
  const long long items = (long long)sz.n_kv_max * p->heads, mean = sz.rows / sz.n_docs, longest = declared_max_doc_len(p, fixed);
  // a document of one or two steps: nothing to hand on, and one launch more (0.85 .. 1.01)
  if (longest <= 64) return false;
  // Every chain stays on one XCD.  While an XCD holds nearly all its tiles at once (32 CUs, 4096 keys; twice that for
  // its few last chains) how the chains fall on the XCDs does not matter (1.1 .. 1.4, one chain alone included; 3 heads
  // of 2 documents of 2500 at head_dim 128 1.21).  Beyond, the XCDs have to come out even, the more the longer the
  // chains are: one that has half as much again to do as their mean is made up for by chains of up to 4096 keys (12
  // heads of 4096 1.05), a third more is too much for longer ones (12 heads of 16384 0.91; two heads of 20000 next to
  // short documents 0.55) and at head_dim 32 (18 heads of 3000 0.95, of 4096 1.01).  Even ones gain at any length (8
  // heads of 8192 1.12, of 16384 and 8192 1.3, of 8192, 4096 and 2048 1.23 .. 1.38).  Of many chains the estimate takes
  // all but the longest for alike, and puts the longest with as many others as any: they do come out even by their
  // number, with a tenth of the last round idle at most and, beyond 4096 keys, none longer than its share of the whole
  // (2 heads of 2796 and 118 x 322 at head_dim 96 1.28; 9 of 4881 and twelve shorter ones 1.23; seven such problems of
  // 1600 drawn ones 1.10 .. 1.28).
  if (std::max(c.long_per_xcd * c.longest, c.per_xcd * mean) > 64 * BKV) {
    const bool even = 10 * c.number >= 9 * CHAIN_QUEUES * c.per_xcd && (longest <= 32 * BKV || c.number * mean * mean >= (CHAIN_QUEUES + 4) * longest * longest);
    if (!even && 10 * CHAIN_QUEUES * c.most > (longest <= 32 * BKV && p->head_dim > 32 ? 15 : 13) * c.squares) return false;
  }
  // Wide heads gain from there on (1.03 .. 1.38; 0.96 where every document ends in a nearly empty tile).  For narrow
  // ones what an item costs before its first step weighs more: with several items per CU only documents of some length
  // gain (head_dim 64: 320 long 0.94 .. 1.02, 512 1.04 .. 1.25, 2048 1.3; head_dim 32: 512 long 0.92 .. 1.06, 768 1.01
  // .. 1.07, 2048 1.3 .. 1.5), with about one per CU also shorter ones (head_dim 64: 1.03 .. 1.5; head_dim 32: 200 long
  // 1.0, 384 1.2).
  if (chain_width(p->head_dim) == 128) return true;
  const bool narrow = p->head_dim <= 32;
  return mean >= (narrow ? 5 * BKV : 7 * BKV / 2) || (items <= 512 && longest >= (narrow ? 3 * BKV : BKV)) ||
         (items <= 1024 && mean >= (narrow ? 3 * BKV : 15 * BKV / 8));
}

int backward_chained(const sba_problem* p, bool fixed, const void* schedule, size_t sched_bytes, const sba_view* q,
                     const sba_view* k, const sba_view* v, const sba_view* go, const sba_view* grem, const float* stick,
                     size_t table_bytes, void* scratch, size_t scratch_bytes, const sba_view* dq, const sba_view* dk,
                     const sba_view* dv, void* stream) {
  Sizes sz;
  int e = check_problem(p, fixed, &sz);
  if (e) return e;
  if ((e = check_mat(q, p)) || (e = check_mat(k, p)) || (e = check_mat(v, p)) || (e = check_mat(go, p)) ||
      (e = check_mat(dq, p, true)) || (e = check_mat(dk, p, true)) || (e = check_mat(dv, p, true)))
    return e;
  if (stick == nullptr || scratch == nullptr) return SBA_E_NULL;
  KArgs c;
  std::memset(&c, 0, sizeof(c));
  if ((e = fill_common(p, fixed, sz, schedule, sched_bytes, true, table_bytes, &c))) return e;
  if (p->head_dim > 128) {
    Given g = given(p, fixed, sz, table_bytes);
    const Given most = given(p, fixed, sz, 0);                 // (what sba_chain_scratch_bytes goes by)
    if (sz.rows > 0 && g.group == 0 && most.group == 0) return SBA_E_SHAPE;
    if (g.group == 0 || (scratch_bytes < g.bytes && most.group > 0)) g = most;
    if (scratch_bytes < g.bytes || (reinterpret_cast<uintptr_t>(scratch) & 15)) return SBA_E_WORKSPACE;
    if ((e = check_arch())) return e;
    if (sz.rows == 0) return 0;
    c.q = to_view(q); c.k = to_view(k); c.v = to_view(v); c.go = to_view(go); c.grem = to_view(grem);
    c.dq = to_view_out(dq, p); c.dk = to_view_out(dk, p); c.dv = to_view_out(dv, p);
    c.stick = const_cast<float*>(stick);
    c.max_doc_len = declared_max_doc_len(p, fixed);
    c.clear_spare = fixed ? 0 : 1;
    c.nan_pair = p->dtype == SBA_F16 && !c.out_f32 ? 0x7e007e00u : 0x7fc07fc0u;
    return backward_given(p, fixed, sz, c, scratch, g, reinterpret_cast<hipStream_t>(stream));
  }
  const ChainScratch at = chain_scratch(p, sz);
  if (scratch_bytes < at.total || (reinterpret_cast<uintptr_t>(scratch) & 15)) return SBA_E_WORKSPACE;
  if ((e = check_arch())) return e;
  if (sz.rows == 0) return 0;
  if (!chain_possible(p, fixed, sz)) return SBA_E_SHAPE;
  ChainArgs a;
  std::memset(&a, 0, sizeof(a));
  a.q = to_view(q); a.k = to_view(k); a.v = to_view(v); a.go = to_view(go); a.grem = to_view(grem);
  a.dq = to_view_out(dq, p); a.dk = to_view_out(dk, p); a.dv = to_view_out(dv, p);
  a.sched = c.sched;
  a.stick = stick;
  char* const base = static_cast<char*>(scratch);
  a.partial = reinterpret_cast<float*>(base + at.partial);
  a.carry = reinterpret_cast<float*>(base + at.carry);
  a.flags = reinterpret_cast<int*>(base + at.flags);
  a.queues = reinterpret_cast<unsigned*>(base + at.queues);
  a.homes = reinterpret_cast<int*>(base + at.homes);
  a.tab_stride = c.tab_stride;
  a.docs_off = c.docs_off;
  a.n_docs = sz.n_docs;
  a.heads = p->heads;
  a.head_dim = p->head_dim;
  a.tokens = p->tokens;
  a.tiles = sz.n_kv_max;
  a.fixed = fixed ? 1 : 0;
  a.fuse = c.fuse;
  a.out_f32 = c.out_f32;
  a.clear_spare = fixed ? 0 : 1;
  a.nan_pair = p->dtype == SBA_F16 && !a.out_f32 ? 0x7e007e00u : 0x7fc07fc0u;
  a.max_doc_len = declared_max_doc_len(p, fixed);
  const int form = g_backward_form.load();
  a.spin_limit = form & SBA_FORM_SHORT_WAITS ? 0 : CHAIN_SPIN_LIMIT;
  a.idle_xcds = ((form >> 16) & 0xff) == 0xff ? 0 : (form >> 16) & 0xff;
  a.n_homes = (int)std::min<long long>(CHAIN_HOMES, (long long)sz.n_q_max * p->heads);
  a.c = c.c;
  a.inv_temp = c.inv_temp;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  Timer tm(2, s);
  return (int)(p->dtype == SBA_F16 ? f16::launch_bwd_chain : bf16::launch_bwd_chain)(a, (p->flags & SBA_ATTEND_CURRENT) != 0, chain_wide(p, fixed, sz),
                                                                                    chain_streams(p, fixed, sz), sz.n_q_max, device_cus(), s);
}

// Schedule workspace of sba_varlen_fwd_static: one array per GPU, inside the code object, so the
// entry point needs no allocation.  In host code the name `scratch` is only a handle for
// hipGetSymbolAddress; kernels get the device address looked up once per device.
static __device__ __align__(256) unsigned char scratch[SBA_STATIC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::atomic<void*> g_scratch_ptr[MAX_DEVICES];

// Device address of `scratch` on the current device (looked up on the first call per device).
int static_scratch(void** out) {
  int dev = 0;
  hipError_t he = hipGetDevice(&dev);
  if (he != hipSuccess) return (int)he;
  if (dev < 0 || dev >= MAX_DEVICES) return SBA_E_ARCH;
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (ptr == nullptr) {
    he = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (he != hipSuccess) return (int)he;
    if (ptr == nullptr) return SBA_E_NULL;
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);   // every thread computes the same address
  }
  *out = ptr;
  return 0;
}

}  // namespace

extern "C" {

int sba_version(void) { return SBA_VERSION; }

const char* sba_error_string(int code) {
  switch (code) {
    case 0: return "ok";
    case SBA_E_NULL: return "a required pointer is NULL";
    case SBA_E_HEAD_DIM: return "head_dim must be a multiple of 8, at most 256";
    case SBA_E_DTYPE: return "unsupported element type (SBA_BF16 or SBA_F16)";
    case SBA_E_SHAPE: return "negative or inconsistent sizes";
    case SBA_E_STRIDE: return "pointer or stride breaks 16-byte row alignment";
    case SBA_E_WORKSPACE: return "workspace too small";
    case SBA_E_ARCH: return "current device is not gfx950 (MI355X)";
    default: return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown error";
  }
}

size_t sba_schedule_bytes(const sba_problem* p) {
  Sizes sz;
  const bool fixed = p != nullptr && (p->flags & SBA_FIXED_LENGTH) != 0;
  if (check_problem(p, fixed, &sz)) return 0;
  return schedule_bytes(sz);
}

size_t sba_table_bytes(const sba_problem* p) {
  Sizes sz;
  const bool fixed = p != nullptr && (p->flags & SBA_FIXED_LENGTH) != 0;
  if (check_problem(p, fixed, &sz)) return 0;
  return (size_t)p->heads * (size_t)table_entries_bound(p, fixed) * sizeof(float) + WORK_WORDS * sizeof(unsigned);
}

size_t sba_table_bytes_for_lengths(const sba_problem* p, const int64_t* doc_lengths, int n_lengths) {
  Sizes sz;
  const bool fixed = p != nullptr && (p->flags & SBA_FIXED_LENGTH) != 0;
  if (check_problem(p, fixed, &sz) || (n_lengths > 0 && doc_lengths == nullptr)) return 0;
  if (fixed) return sba_table_bytes(p);
  long long entries = 0;
  for (int i = 0; i < n_lengths; ++i) {
    if (doc_lengths[i] < 0 || doc_lengths[i] > p->tokens) return 0;
    entries += tab_doc_entries((int)doc_lengths[i]);
  }
  if (entries > 0x7fffffffll) return 0;   // a document's base must fit the scheduler's int32 field
  return (size_t)p->heads * (size_t)(entries > 0 ? entries : 32) * sizeof(float)   // never empty: one 128-byte line per head
         + WORK_WORDS * sizeof(unsigned);
}

int sba_build_schedule(const sba_problem* p, void* schedule, size_t schedule_size, void* stream) {
  Sizes sz;
  const bool fixed = p != nullptr && (p->flags & SBA_FIXED_LENGTH) != 0;
  int e = check_problem(p, fixed, &sz);
  if (e) return e;
  if (schedule == nullptr) return SBA_E_NULL;
  if (schedule_size < schedule_bytes(sz)) return SBA_E_WORKSPACE;
  if ((e = check_arch())) return e;
  SchedArgs a;
  a.cu = fixed ? nullptr : p->cu_seqlens;
  a.cu_is64 = (p->flags & SBA_CU_INT64) ? 1 : 0;
  a.n_docs = sz.n_docs;
  a.tokens = p->tokens;
  a.n_q_max = sz.n_q_max;
  a.n_kv_max = sz.n_kv_max;
  a.classes = !fixed && list_in_classes(p, sz);
  a.out = reinterpret_cast<int*>(schedule);
  return (int)launch_schedule(a, reinterpret_cast<hipStream_t>(stream));
}

int sba_varlen_fwd(const sba_problem* p, const void* schedule, size_t schedule_size, const sba_view* q,
                   const sba_view* k, const sba_view* v, const sba_view* o, const sba_view* rem,
                   float* stick_table, size_t table_size, void* stream) {
  return forward(p, false, schedule, schedule_size, q, k, v, o, rem, stick_table, table_size, nullptr, 0, stream);
}

int sba_attn_fwd(const sba_problem* p, const void* schedule, size_t schedule_size, const sba_view* q,
                 const sba_view* k, const sba_view* v, const sba_view* o, const sba_view* rem,
                 float* stick_table, size_t table_size, void* stream) {
  return forward(p, true, schedule, schedule_size, q, k, v, o, rem, stick_table, table_size, nullptr, 0, stream);
}

int sba_varlen_fwd_weights(const sba_problem* p, const void* schedule, size_t schedule_size, const sba_view* q,
                           const sba_view* k, const sba_view* v, const sba_view* o, const sba_view* rem,
                           float* stick_table, size_t table_size, float* weights, size_t weights_size,
                           void* stream) {
  if (weights == nullptr) return SBA_E_NULL;
  return forward(p, false, schedule, schedule_size, q, k, v, o, rem, stick_table, table_size, weights, weights_size,
                 stream);
}

int sba_attn_fwd_weights(const sba_problem* p, const void* schedule, size_t schedule_size, const sba_view* q,
                         const sba_view* k, const sba_view* v, const sba_view* o, const sba_view* rem,
                         float* stick_table, size_t table_size, float* weights, size_t weights_size,
                         void* stream) {
  if (weights == nullptr) return SBA_E_NULL;
  return forward(p, true, schedule, schedule_size, q, k, v, o, rem, stick_table, table_size, weights, weights_size,
                 stream);
}

int sba_varlen_bwd(const sba_problem* p, const void* schedule, size_t schedule_size, const sba_view* q,
                   const sba_view* k, const sba_view* v, const sba_view* grad_o, const sba_view* grad_rem,
                   const float* stick_table, float* grad_table, size_t table_size, const sba_view* dq,
                   const sba_view* dk, const sba_view* dv, void* stream) {
  return backward(p, false, schedule, schedule_size, q, k, v, grad_o, grad_rem, stick_table, grad_table, table_size,
                  dq, dk, dv, stream);
}

int sba_attn_bwd(const sba_problem* p, const void* schedule, size_t schedule_size, const sba_view* q,
                 const sba_view* k, const sba_view* v, const sba_view* grad_o, const sba_view* grad_rem,
                 const float* stick_table, float* grad_table, size_t table_size, const sba_view* dq,
                 const sba_view* dk, const sba_view* dv, void* stream) {
  return backward(p, true, schedule, schedule_size, q, k, v, grad_o, grad_rem, stick_table, grad_table, table_size,
                  dq, dk, dv, stream);
}

size_t sba_bwd_scratch_bytes(const sba_problem* p, size_t table_bytes) {
  Sizes sz;
  const bool fixed = p != nullptr && (p->flags & SBA_FIXED_LENGTH) != 0;
  if (check_problem(p, fixed, &sz)) return 0;
  if (p->head_dim > 128) return backward_form() == 1 ? 0 : given(p, fixed, sz, table_bytes).bytes;
  return chain_wanted(p, fixed, sz) ? chain_scratch(p, sz).total : 0;
}
size_t sba_chain_scratch_bytes(const sba_problem* p) { return sba_bwd_scratch_bytes(p, 0); }

int sba_varlen_bwd_chained(const sba_problem* p, const void* schedule, size_t schedule_size, const sba_view* q,
                           const sba_view* k, const sba_view* v, const sba_view* grad_o, const sba_view* grad_rem,
                           const float* stick_table, size_t table_size, void* scratch, size_t scratch_size,
                           const sba_view* dq, const sba_view* dk, const sba_view* dv, void* stream) {
  return backward_chained(p, false, schedule, schedule_size, q, k, v, grad_o, grad_rem, stick_table, table_size, scratch, scratch_size,
                          dq, dk, dv, stream);
}

int sba_attn_bwd_chained(const sba_problem* p, const void* schedule, size_t schedule_size, const sba_view* q,
                         const sba_view* k, const sba_view* v, const sba_view* grad_o, const sba_view* grad_rem,
                         const float* stick_table, size_t table_size, void* scratch, size_t scratch_size,
                         const sba_view* dq, const sba_view* dk, const sba_view* dv, void* stream) {
  return backward_chained(p, true, schedule, schedule_size, q, k, v, grad_o, grad_rem, stick_table, table_size, scratch, scratch_size,
                          dq, dk, dv, stream);
}

int sba_varlen_fwd_static(const sba_problem* p, const sba_view* q, const sba_view* k, const sba_view* v,
                          const sba_view* o, const sba_view* rem, void* stream) {
  Sizes sz;
  int e = check_problem(p, false, &sz);
  if (e) return e;
  if (schedule_bytes(sz) > (size_t)SBA_STATIC_SCRATCH_BYTES) return SBA_E_WORKSPACE;
  if ((e = check_arch())) return e;
  void* sched = nullptr;
  if ((e = static_scratch(&sched))) return e;
  // The scheduler rewrites the header and every list entry the kernels will use; nothing of
  // the previous call's contents is read, so nothing needs clearing.
  if ((e = sba_build_schedule(p, sched, SBA_STATIC_SCRATCH_BYTES, stream))) return e;
  return forward(p, false, sched, SBA_STATIC_SCRATCH_BYTES, q, k, v, o, rem, nullptr, 0, nullptr, 0, stream,
                 /*timed=*/false);   // (timing creates events)
}

int sba_round_floats(int dtype, int n, const void* const* src, void* const* dst, const int64_t* counts, void* stream) {
  if (dtype != SBA_BF16 && dtype != SBA_F16) return SBA_E_DTYPE;
  if (n < 1 || n > 3) return SBA_E_SHAPE;
  if (src == nullptr || dst == nullptr || counts == nullptr) return SBA_E_NULL;
  RoundArgs a;
  std::memset(&a, 0, sizeof(a));
  int64_t groups = 0;
  for (int i = 0; i < 3; ++i) {
    if (i < n) {
      if (counts[i] < 0 || counts[i] % 8) return SBA_E_SHAPE;
      if (counts[i] > 0 && (src[i] == nullptr || dst[i] == nullptr)) return SBA_E_NULL;
      if ((reinterpret_cast<uintptr_t>(src[i]) | reinterpret_cast<uintptr_t>(dst[i])) & 15) return SBA_E_STRIDE;
      a.src[i] = static_cast<const float*>(src[i]);
      a.dst[i] = static_cast<unsigned short*>(dst[i]);
      groups += counts[i] / 8;
    }
    a.upto[i] = groups;
  }
  int e;
  if ((e = check_arch())) return e;
  return groups == 0 ? 0 : (int)launch_round_f32(a, dtype == SBA_F16, reinterpret_cast<hipStream_t>(stream));
}

int sba_launch_geometry(const sba_problem* p, sba_geometry* out) {
  Sizes sz;
  const bool fixed = p != nullptr && (p->flags & SBA_FIXED_LENGTH) != 0;
  int e = check_problem(p, fixed, &sz);
  if (e) return e;
  if (out == nullptr) return SBA_E_NULL;
  const BwdBounds bb = backward_bounds(p, fixed, sz);
  const DkdvGrid g = dkdv_grid(has_dkdv_tail_kernel(p->head_dim), bb.n_long_max, bb.n_tail_max, sz.n_kv_max);
  out->query_list_tiles = sz.n_q_max;
  out->key_list_tiles = sz.n_kv_max;
  out->query_list_word = SCHED_HDR;
  out->key_list_word = SCHED_HDR + TILE_WORDS * sz.n_q_max;
  out->tile_words = TILE_WORDS;
  out->schedule_words = (long long)(schedule_bytes(sz) / sizeof(int));
  out->fwd_tiles = sz.n_q_max;     // forward and dq pass: one workgroup per slot of the query-tile list and head
  out->dq_tiles = sz.n_q_max;
  out->long_tiles_bound = bb.n_long_max;
  out->tail_tiles_bound = bb.n_tail_max;
  out->dkdv_main_tiles = g.main_tiles;
  out->dkdv_tail_tiles = g.tail_tiles;
  out->dkdv_main_workgroups = dkdv_main_workgroups(p->head_dim, g.main_tiles);
  const bool is_short = backward_short(p, fixed, sz);
  out->fwd_small_workgroups = forward_small(p, fixed, sz) ? small_workgroups(sz.n_q_max) : 0;
  out->bwd_small_workgroups = !is_short && backward_small(p, fixed, sz) ? small_workgroups(sz.n_q_max) : 0;
  out->bwd_short_workgroups = is_short ? short_parts(p, fixed, sz) : 0;
  out->docs_word = SCHED_HDR + TILE_WORDS * (sz.n_q_max + sz.n_kv_max) + chain_docs_offset(sz.n_docs);
  out->bwd_rows_streamed = sz.n_docs > 0 && p->head_dim <= 128 && chain_streams(p, fixed, sz) ? 1 : 0;
  return 0;
}

void sba_set_timing(int on) {
  if (on) {   // what was timed before is forgotten: a kernel that is not launched from here on reads 0
    std::lock_guard<std::mutex> lock(g_ev_mutex);
    for (int i = 0; i < 3; ++i) {
      if (g_ev[i].e0) (void)hipEventDestroy(g_ev[i].e0);
      if (g_ev[i].e1) (void)hipEventDestroy(g_ev[i].e1);
      g_ev[i] = EventPair();
      g_ms[i].store(0.0f);
    }
  }
  g_timing.store(on);
}
void sba_set_dkdv_workgroups(int n) { g_dkdv_workgroups.store(n); }
void sba_set_backward_form(int form) { g_backward_form.store(form); }
float sba_last_kernel_ms(int which) {
  if (which < 0 || which >= 3) return 0.f;
  std::lock_guard<std::mutex> lock(g_ev_mutex);
  const EventPair& ev = g_ev[which];
  float ms = 0.f;
  if (ev.e0 != nullptr && ev.e1 != nullptr && hipEventSynchronize(ev.e1) == hipSuccess &&
      hipEventElapsedTime(&ms, ev.e0, ev.e1) == hipSuccess)
    g_ms[which].store(ms);
  return g_ms[which].load();
}

}  // extern "C"
