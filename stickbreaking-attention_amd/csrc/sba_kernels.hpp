// Kernel argument block and launch prototypes shared by the translation units of libsba.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "sba_device.hpp"

namespace sba {

struct KArgs {
  View q, k, v, o, rem;        // forward tensors (rem has no head_dim axis)
  View go, grem, dq, dk, dv;   // backward tensors (grem.ptr may be null)
  const int* sched;            // schedule workspace
  int kv_list_off;             // int32 offset of the KV tile list inside `sched`
  int n_kv_alloc;              // tiles that list has room for (no launch may index it beyond)
  int docs_off, n_docs;        // the ranked documents in the schedule, if there are at most RANK_LIMIT
  float* stick;                // carry table written by the forward (may be null in fwd): per (row, 32-key block) the
                               // stick left on entering the block; per-row plane: rem in fp32
  float* gtab;                 // gradient prefix table (backward scratch); per-row plane: the full d(rem)
  float* weights;              // forward, debug variant only: dense attention weights
                               // [batch][heads][tokens][tokens] (row = query token, column = key token)
  int heads;
  unsigned heads_inv;          // forward: (2^32 - 1) / heads
  int head_dim;                // a multiple of 8, at most the width D of the kernel (see make_rows)
  int tokens;                  // tokens per batch entry
  int fuse;                    // the output is o + rem * v (and grad_o is the gradient of that)
  int clear_spare;             // packed input: spare workgroups clear the rows that belong to no document (or fill
                               // everything with NaN when the launch is refused)
  unsigned nan_pair;           // two NaNs of the 16-bit element type (one of float32 outputs)
  int out_f32;                 // outputs are float32; their strides still count 16-bit words (see to_view_out)
  int64_t tab_stride;          // carry-table entries per head the caller's tables hold
  int max_doc_len;             // backward: the longest document the caller declared (its grids are sized with it;
                               // the kernels refuse to run when the scheduler found a longer one)
  float c;                     // inv_temp * log2(e)
  float inv_temp;
  unsigned* work;              // work counters of the backward's persistent launch (WORK_WORDS words at the end of the
                               // gradient table; the dq pass clears them), or null: one workgroup per work item
  int n_items;                 // work items of this launch (what the grid is with one workgroup per item)
  int resident;                // backward, host side: workgroups of a persistent launch (0: never persistent)
  int min_items_each;          // host side: a launch is persistent when it has this many items per workgroup
  unsigned short* pz;          // backward at head_dim 129 .. 256: p and dz of every 32 x 32 block, left by the dq pass for the dk/dv pass
  int64_t pz_entries;          // carry-table entries per head it has room for: 128 bytes each
  int lg_deal;                 // forward: the logarithm of the device's compute units if it holds the launch at once (see deal_item), or NO_DEAL
};

constexpr size_t GIVEN_SCRATCH_MAX = 0xf0000000u;   // bytes of p and dz that are handed on at a time: 32-bit offsets reach them
static_assert(pz_offset((int)(GIVEN_SCRATCH_MAX / (2 * PZ_WORDS)) - 32) == GIVEN_SCRATCH_MAX - 32 * 2 * PZ_WORDS, "the last block's place");

constexpr int NO_DEAL = 31;    // (no launch has a second round of 2^31 workgroups)
// Workgroups of the forward that a compute unit holds.
inline int fwd_per_cu(int head_dim) { return head_dim <= 32 ? 6 : (head_dim <= 64 ? 4 : (head_dim <= 128 ? 3 : 2)); }

// Arguments of the one-pass backward (sba_chain.hip).
constexpr int CHAIN_QUEUES = 8;            // one per XCD
constexpr int CHAIN_QUEUE_STRIDE = 32;     // words between the queues' counters: a 128-byte line each
constexpr int CHAIN_HOMES = 64;            // workgroups of the prep kernel that note their XCD: dealt out in turn, 8 of them meet all
constexpr int CHAIN_GROUP = 8;             // chains of a queue whose items are interleaved
constexpr int CHAIN_MAX_GROUPS = 256;
constexpr int CHAIN_SPIN_LIMIT = 1 << 20;  // polls of a wait (about a second) before it gives up and the results turn to NaN
struct ChainArgs {
  View q, k, v, go, grem, dq, dk, dv;
  const int* sched;
  const float* stick;          // carry table written by the forward
  float* partial;              // [heads][tiles][BM x D] fp32: dq of a query over the key tiles so far
  float* carry;                // [2][heads][tiles][BM] fp32: the running sum along the keys, by parity of the key tile that reads it
  int* flags;                  // [heads][tiles]: steps a key tile has published
  unsigned* queues;            // CHAIN_QUEUES counters
  int* homes;                  // [n_homes] XCD of the prep kernel's first workgroups
  int64_t tab_stride;
  int docs_off;                // int32 offset of the ranked documents inside `sched`
  int n_docs, heads, head_dim, tokens, tiles;
  int fixed, fuse, clear_spare, out_f32;
  unsigned nan_pair;
  int max_doc_len;
  int spin_limit;              // CHAIN_SPIN_LIMIT, or what a test asks for
  int n_homes;
  int idle_xcds;               // test: XCDs (a bit each) taken for ones this launch cannot run on
  float c, inv_temp;
};

// Pointers rebuilt from integer words are generic pointers to the compiler (64-bit flat addresses in
// vector registers for every access); say again what it knows of pointers in a kernel's argument
// list: they point into global memory.
template <class T>
__device__ __forceinline__ void as_global(T*& p) {
  typedef __attribute__((address_space(1))) char* GlobalBytes;
  p = reinterpret_cast<T*>((char*)(GlobalBytes)(unsigned long long)p);
}
__device__ __forceinline__ void globals_of(KArgs& a) {
  as_global(a.q.ptr); as_global(a.k.ptr); as_global(a.v.ptr); as_global(a.o.ptr); as_global(a.rem.ptr);
  as_global(a.go.ptr); as_global(a.grem.ptr); as_global(a.dq.ptr); as_global(a.dk.ptr); as_global(a.dv.ptr);
  as_global(a.sched); as_global(a.stick); as_global(a.gtab); as_global(a.weights); as_global(a.work); as_global(a.pz);
}
__device__ __forceinline__ void globals_of(ChainArgs& a) {
  as_global(a.q.ptr); as_global(a.k.ptr); as_global(a.v.ptr); as_global(a.go.ptr); as_global(a.grem.ptr);
  as_global(a.dq.ptr); as_global(a.dk.ptr); as_global(a.dv.ptr);
  as_global(a.sched); as_global(a.stick); as_global(a.partial); as_global(a.carry); as_global(a.flags); as_global(a.queues); as_global(a.homes);
}

// The argument block read afresh from the kernel-argument segment.  A persistent kernel calls this at
// the top of every work item with a pointer the compiler cannot see through: argument words it
// needs would otherwise be loaded once, ahead of the item loop, and stay in scalar registers across
// the whole loop (the block is 380 bytes; the loop bodies have no such room, and spilled scalar
// registers end up as vector registers spilled to scratch memory).
template <class Args = KArgs>
__device__ __forceinline__ Args fresh_args() {
  typedef const __attribute__((address_space(4))) unsigned long long* Words;
  Words w = (Words)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(w));
  static_assert(sizeof(Args) % 8 == 0, "copied in 8-byte words");
  union { Args a; unsigned long long u[sizeof(Args) / 8]; } out;
#pragma unroll
  for (unsigned i = 0; i < sizeof(Args) / 8; ++i) out.u[i] = w[i];
  globals_of(out.a);
  return out.a;
}

// Grid of a launch over n_items work items: one workgroup per item, or -- when the caller has work counters and
// there are enough items for every workgroup of a persistent launch -- a.resident workgroups (a multiple of 8).
inline unsigned launch_grid(const KArgs& a, long long n_items) {
  const long long resident = a.resident & ~7;
  const bool persistent = a.work != nullptr && resident >= 8 && n_items > resident &&
                          n_items >= resident * (long long)a.min_items_each;
  return (unsigned)(persistent ? resident : n_items);
}

// Arrays of sba_round_floats: 8-element groups, `upto` counted over the arrays so far.
struct RoundArgs {
  const float* src[3];
  unsigned short* dst[3];
  int64_t upto[3];
};

struct SchedArgs {
  const void* cu;   // null for fixed-length
  int cu_is64;
  int n_docs;       // documents (fixed: batch)
  int tokens;       // T per batch entry
  int n_q_max, n_kv_max;
  int classes;      // query tiles of documents of like length are listed tile-major
  int* out;
};

hipError_t launch_schedule(const SchedArgs& a, hipStream_t s);
hipError_t launch_round_f32(const RoundArgs& a, bool f16, hipStream_t s);

// Key-tile slots the two kernels of the dk/dv pass are launched over (one workgroup per slot and
// head).  Every workgroup of the main kernel reads the tile descriptor of its slot BEFORE it knows
// how many tiles the list really holds, so the main grid must never exceed the room of the list
// (n_kv_alloc); the tail kernel compares its slot with the true length first.  Head dimensions
// without a tail kernel give both groups of the list to the main kernel.
struct DkdvGrid { int main_tiles, tail_tiles; };
inline DkdvGrid dkdv_grid(bool has_tail_kernel, int n_long_max, int n_last_max, int n_kv_alloc) {
  DkdvGrid g;
  g.main_tiles = has_tail_kernel ? (n_long_max < n_kv_alloc ? n_long_max : n_kv_alloc)
                                 : (n_long_max + n_last_max < n_kv_alloc ? n_long_max + n_last_max : n_kv_alloc);
  g.tail_tiles = has_tail_kernel ? n_last_max : 0;
  return g;
}
// Width of the kernels a head_dim runs on.
inline int kernel_width(int head_dim) { return head_dim <= 32 ? 32 : head_dim <= 64 ? 64 : head_dim <= 128 ? 128 : 256; }
// Columns the product-space kernels multiply.  A head_dim in the lower half of a width's range would leave up to half of
// the matrix instructions multiplying zeros, so the two wide kernels exist with three quarters of theirs as
// well (same tiles in LDS, fewer contraction steps and output columns); below 64 a call is not bound by them.
inline int used_width(int head_dim) {
  if (head_dim > 64 && head_dim <= 96) return 96;
  if (head_dim > 128 && head_dim <= 192) return 192;
  return kernel_width(head_dim);
}
inline bool has_dkdv_tail_kernel(int head_dim) { return head_dim <= 64; }
// Workgroups per head: of the kernels of sba_small.hip that own 32 rows of a query tile, and of the dk/dv main kernel, which
// above head_dim 128 owns half a key tile.
inline int small_workgroups(int n_q_max) { return n_q_max * (BM / 32); }
constexpr int WIDE_KEYS = 64;
inline int dkdv_main_workgroups(int head_dim, int main_tiles) { return main_tiles * (kernel_width(head_dim) > 128 ? BKV / WIDE_KEYS : 1); }

// One set of compute launchers per element type (sba_fwd.hip and sba_bwd.hip are compiled once
// for each, see SBA_ELEM_NS).
#ifdef SBA_ELEM_F16
#define SBA_INLINE_bf16
#define SBA_INLINE_f16 inline
#else
#define SBA_INLINE_bf16 inline
#define SBA_INLINE_f16
#endif
#define SBA_DECLARE_LAUNCHERS(NS)                                                                                \
  SBA_INLINE_##NS namespace NS {                                                                                 \
  hipError_t launch_fwd(const KArgs& a, int head_dim, bool attend_current, bool product, int mode,               \
                        int n_q_max, hipStream_t s);                                                             \
  hipError_t launch_bwd_dq(const KArgs& a, int head_dim, bool attend_current, bool product, int n_q_max,         \
                           hipStream_t s);                                                                       \
  hipError_t launch_bwd_dkdv(const KArgs& a, int head_dim, bool attend_current, bool product, int n_long_max,    \
                             int n_last_max, hipStream_t s);                                                     \
  hipError_t launch_bwd_dq_wide(const KArgs& a, bool attend_current, bool product, int n_q_max, hipStream_t s);   \
  hipError_t launch_bwd_dkdv_given(const KArgs& a, int tiles, hipStream_t s);                                    \
  hipError_t launch_bwd_dkdv_wide(const KArgs& a, bool attend_current, bool product, int tiles, hipStream_t s);   \
  hipError_t launch_fwd_small(const KArgs& a, bool attend_current, int n_q_max, hipStream_t s);                  \
  hipError_t launch_bwd_short(const KArgs& a, bool attend_current, int parts, hipStream_t s);                  \
  hipError_t launch_bwd_dq_small(const KArgs& a, bool attend_current, int n_q_max, hipStream_t s);                  \
  hipError_t launch_bwd_dkdv_small(const KArgs& a, bool attend_current, int n_q_max, hipStream_t s);                  \
  hipError_t launch_bwd_chain(const ChainArgs& a, bool attend_current, bool wide, bool stream, int n_q_max,      \
                              int workgroups, hipStream_t s);                                                                    \
  }
SBA_DECLARE_LAUNCHERS(bf16)
SBA_DECLARE_LAUNCHERS(f16)
#undef SBA_DECLARE_LAUNCHERS

}  // namespace sba
