// Backward in one pass: dq, dk and dv of long documents by workgroups that hand their queries' partial
// results from key tile to key tile.
//
// The two-pass backward (sba_bwd.hip) forms every score twice, once for dq and once for dk / dv, because
// dq is summed over keys and dk, dv over queries: 56 matrix instructions per 32 x 32 block at head_dim 128
// and the vector work of the weights and of dz twice.  One pass needs 40 and does the vector work once, but
// one of the two sums then crosses workgroups.  fp32 atomics are out (1.36 TB/s of payload on
// this part, see sba_bwd.hip).  Here a workgroup owns 128 keys of one (document, head) -- dk and dv stay in
// registers -- and dq of 32 queries at a time is handed on: the workgroup of key tile c takes the partial
// sum that tile c - 1 left in scratch memory, adds its own keys on the matrix cores and leaves it for tile
// c + 1; the tile that holds the queries' own keys writes dq.  The running sum along the keys that
// dz needs travels the same way, so the gradient table of the two-pass form and the pass that fills it are gone.
//
// What makes this affordable is the XCD's L2: 16 KiB in and out per 32 queries is 8 TB/s over the chip, which the
// L2s deliver (11 TB/s each way measured with plain stores and one chain per XCD; 1.9 TB/s with
// stores that write through to memory, as a hand-over between XCDs would need).  So all key tiles of a
// (document, head) -- a chain -- run on one XCD: a workgroup reads which XCD it is on (XCC_ID) and draws its
// items from that XCD's queue.  Every CU of an XCD shares that XCD's L2 and L1 is write-through, so a
// store is visible to the XCD's other CUs when vmcnt says it has been acknowledged; consumers read with sc1,
// which L1 does not answer.
//
// Order and progress.  Queries are walked from the document's end down to the tile's own keys, so that the tiles of a
// chain start together and end one after the other; the items of a queue are ordered by key tile, so the item an item
// waits for was drawn before it by a workgroup that is running: waits end.  `flags` holds a number per item: at the
// start of step t a tile publishes t - 2, which stands for the carried sums of its blocks up to t - 2 (formed two steps
// ago) and the partial dq of those up to t - 3 (formed by the product waves a step after the sums); both have been
// acknowledged by then.  Step s asks for the carried sum of block s + 1 and the partial dq of block s, so it needs s +
// 1: a tile runs three steps behind the one before (it was four while a sum was published no earlier than its block's
// dq).  What the tile before has published is copied to LDS in the background, a step old when it is looked at; only
// where that is not enough does a score wave -- the one all others wait for -- stop to ask.
//
// Measured (kernel time of the backward with its prep kernel, before and after the shorter lag, the poll in the
// background and leaner product waves, alternating on one MI355X): 32 heads x 16 K tokens in eight documents, head_dim
// 128, 1311 -> 1292 us; 12 x 4 x 4096 694 -> 683; 16 x 7 K in six documents, head_dim 96, 240 -> 226; 12 heads of 1500,
// 900 and 601 tokens, head_dim 64, 80.0 -> 69.8 and 128, 95.8 -> 88.  (Documents of one or two
// tiles above head_dim 64, where an item's beginning and end are the time, are up to 3 % slower: 32 heads of 64 x 256 at
// 128 346 -> 354, 19 of 235 x 118 310 -> 317.  Each role's change costs half of it, and each makes long documents 1 to
// 2 % faster; of the changes one by one only the poll's absence gives back 1 %, and takes 1 % from long documents.)
// At head_dim 128 it waits: 44 % of the wave cycles on 32 heads x 16 K tokens (22 .. 25 % in the two passes;
// profiles/c3_sq_counters_pmc.txt), with the matrix pipe busy for 36 %.  Such a launch fetches 4.5 GB from behind the
// L2s and writes 3.1 GB there, 5.8 TB/s where a plain copy reaches 4.9: of the 2.8 GB of partial dq each way, all that
// is written leaves L2 (eight chains of 2 MiB share 4 MiB).
//
// What does not help: waves that are all alike.  Eight of them with 256 registers (steps of 64 queries, two barriers)
// took 1510 us at head_dim 96 where this takes 1130, four with 512 registers and every matrix instruction placed by
// hand 1235: a wave alone on its SIMD issues for 56 % of its cycles and has nothing to cover the rest.
//
// Carried sum: with C[j] the sum of G over the keys up to j and ex the stick on entering a key, D = C + drem ex
// obeys D[j] = D[j-1] + p_j (do.v_j) and dz_j = r_j D[j] - D[j-1] (see grad_dz in sba_bwd.hip); the gradient of
// rem enters only through the value in front of the row's oldest key, D = drem * rem (chain_prep_kernel).
#include <type_traits>

#include "sba_kernels.hpp"

namespace sba {
inline namespace SBA_ELEM_NS {

__device__ __forceinline__ int this_xcd() { return __builtin_amdgcn_s_getreg(20 | (3 << 11)) & (CHAIN_QUEUES - 1); }   // HW_REG_XCC_ID, bits 3:0

// Ahead of the main kernel: clears the flags and the queues, notes which XCDs its workgroups run on (the main kernel's
// will run on the same), forms D in front of the oldest key of every row, and writes the rows that belong to no
// document (or NaN everywhere when the launch is refused).  One workgroup per query tile and head.
template <int D>
__global__ void __launch_bounds__(NT) chain_prep_kernel(const ChainArgs a) {
  const int* sched = a.sched;
  const int slot = blockIdx.x / a.heads;
  const int head = blockIdx.x - slot * a.heads;
  const int4 hdr = *reinterpret_cast<const int4*>(sched);   // status, query tiles, key tiles, table entries needed
  const Tile t = reinterpret_cast<const Tile*>(sched + SCHED_HDR)[slot];
  asm volatile("" ::"s"(t.tok_start), "s"(t.doc_len), "s"(t.idx), "s"(t.batch), "s"(t.tab_base));
  const bool refused = hdr.x != 0 || hdr.w > a.tab_stride || sched[SCHED_MAXLEN] > a.max_doc_len;
  const int tid = threadIdx.x;
  if (blockIdx.x == 0 && tid < CHAIN_QUEUES * CHAIN_QUEUE_STRIDE) a.queues[tid] = 0u;
  if (blockIdx.x < CHAIN_HOMES && tid == 0) {
    const int xcd = this_xcd();
    a.homes[blockIdx.x] = (a.idle_xcds >> xcd) & 1 ? -1 : xcd;
  }
  if (tid == 0) a.flags[head * a.tiles + slot] = 0;
  if (refused || slot >= hdr.y) {
    if (a.clear_spare) {
      int row0, row1;
      unsigned pair;
      spare_rows(refused, slot, hdr.y, sched[SCHED_TOTAL], a.tokens, a.nan_pair, row0, row1, pair);
      fill_rows16(a.dq, head, row0, row1, a.head_dim << a.out_f32, pair, tid, NT);
      fill_rows16(a.dk, head, row0, row1, a.head_dim << a.out_f32, pair, tid, NT);
      fill_rows16(a.dv, head, row0, row1, a.head_dim << a.out_f32, pair, tid, NT);
    }
    return;
  }
  __shared__ float dots[BM];
  const int row0 = t.idx * BM;
  const int n_rows = min(BM, t.doc_len - row0);
  const int64_t tok0 = t.tok_start + row0;
  if (a.fuse) {   // d(rem) = do . v_row as well (see bwd_dq_kernel): 16-byte chunks, the lanes of a row next to one another
    constexpr int LPR = D / 8 < 16 ? D / 8 : 16;    // lanes per row
    const elem_t* gb = reinterpret_cast<const elem_t*>(a.go.ptr) + t.batch * a.go.sb + head * a.go.sh + tok0 * a.go.st;
    const elem_t* vb = reinterpret_cast<const elem_t*>(a.v.ptr) + t.batch * a.v.sb + head * a.v.sh + tok0 * a.v.st;
    const int sub = tid % LPR;
    for (int r = tid / LPR; r < BM; r += NT / LPR) {
      float dot = 0.0f;
      if (r < n_rows && 8 * sub < a.head_dim) {
        const el8 g = *reinterpret_cast<const el8*>(gb + r * a.go.st + 8 * sub);
        const el8 v = *reinterpret_cast<const el8*>(vb + r * a.v.st + 8 * sub);
#pragma unroll
        for (int e = 0; e < 8; ++e) dot = fmaf((float)g[e], (float)v[e], dot);
      }
#pragma unroll
      for (int m = LPR / 2; m > 0; m >>= 1) dot += __shfl_xor(dot, m, 64);
      if (sub == 0) dots[r] = dot;
    }
    __syncthreads();
  }
  if (tid < n_rows) {
    float dr = a.fuse ? dots[tid] : 0.0f;
    if (a.grem.ptr != nullptr)
      dr += (float)(reinterpret_cast<const elem_t*>(a.grem.ptr) + t.batch * a.grem.sb + head * a.grem.sh + tok0 * a.grem.st)[(int64_t)tid * a.grem.st];
    const float rem = a.stick[(int64_t)head * a.tab_stride + t.tab_base + tab_rowplane32(t.doc_len) + row0 + tid];
    a.carry[((int64_t)head * a.tiles + t.tile_base) * BM + row0 + tid] = dr * rem;
  }
}

// One dword, the same for every lane, to LDS at dst + 4 * lane.  Counted by vmcnt like async_copy16.
__device__ __forceinline__ void async_word(const int* from, const int* dst) {
  const unsigned lds_addr = __builtin_amdgcn_readfirstlane((unsigned)(size_t)dst);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2 sc1" ::"s"(lds_addr), "v"(0), "s"(from) : "memory", "m0");
}

// NSQ: 32-query blocks per step.  4 * NSQ score waves (one per 32-key block and query block) and 4 product waves.  At
// head_dim 128 registers leave room for one score wave per SIMD, whose vector work (180 instructions, 32 of them
// transcendental, per block) is the step; at 64 and below two fit (168 registers): 16 heads x 4 documents of 2048 at
// head_dim 64 in steps of 64 queries 159 us for 187 in steps of 32, at head_dim 32 135 for 164 (two passes: 225, 173).
// STREAM: Q and dO rows, which every key tile of the chain reads again, stream past the L2 (see chain_streams).
template <int D, int U, bool AC, int NSQ, bool STREAM>
__global__ void __launch_bounds__((4 * NSQ + 4) * 64, 1) bwd_chain_kernel(const ChainArgs a) {
  constexpr int KS = U / 16, DB = U / 32;
  constexpr int TQ = 32 * NSQ;      // queries per step
  constexpr bool DEEP = NSQ == 1;   // score waves form block w + 2's products in step w, else block w + 1's
  constexpr int RING = DEEP ? 6 : 5;     // Q / dO slots: tiles w-1 (dk) .. w+2 or w+1 (scores) of step w and two in flight
  constexpr int AHEAD = RING - 2;
  constexpr int PBUF = DEEP ? 3 : 2;     // staged p: with the weights, one step ahead of dz, or with dz
  constexpr int QTILE = TQ * D, PTILE = TQ * BKV;
  constexpr int DIAG = BKV / TQ;    // steps of an item whose queries may not see all of its keys: its last ones
  __shared__ __attribute__((aligned(16))) unsigned short Qs[RING * QTILE];
  __shared__ __attribute__((aligned(16))) unsigned short Gs[RING * QTILE];
  __shared__ __attribute__((aligned(16))) unsigned short PZ[(PBUF + 2) * PTILE];   // p: PBUF buffers, dz: two buffers, [query][key]
  __shared__ float tot[2][NSQ][4][32];       // by step parity: every key block's sum of p (do.v) per query
  __shared__ float given_up;                 // 0, or NaN once a wait of this workgroup has run out (see await)
  __shared__ int prefix[CHAIN_MAX_GROUPS];   // key tiles of the longest chains, up to and including each group's
  __shared__ int place;                      // this XCD's number among those that serve a queue, their count (bits 8 ..)
  __shared__ int mbox[2][8];
  __shared__ int fbox[64];                   // what the tile before this one had published a step ago
  __shared__ __attribute__((aligned(16))) unsigned short spare[4][512];   // where a product wave's copies of nothing go
  unsigned short* const Ps = PZ;
  unsigned short* const Zs = PZ + PBUF * PTILE;
  static_assert((PBUF + 2) * PTILE >= (DEEP ? 1 : 2) * BKV * D, "the key tile (and the value tile) is staged in the p / dz buffers between items");

  const int* sched = a.sched;
  const int4 hdr = *reinterpret_cast<const int4*>(sched);
  if (hdr.x != 0 || hdr.w > a.tab_stride || sched[SCHED_MAXLEN] > a.max_doc_len) return;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, blk = (lane >> 4) & 1;
  const bool scorer = w < 4 * NSQ;

  struct Item { int kt, head, tok_start, doc_len, tab_base, tile_base, batch; };
  const int2* const docs = reinterpret_cast<const int2*>(sched + a.docs_off);   // per rank: {token start, length}, {table base, tile base}
  const int n_chains = a.n_docs * a.heads;
  const int head_dim = a.head_dim;
  auto rows_of = [head_dim](const View& v, const Item& it) {
    return make_rows(reinterpret_cast<const elem_t*>(v.ptr) + it.batch * v.sb + it.head * v.sh + (int64_t)it.tok_start * v.st,
                     v.st, it.doc_len, head_dim);
  };
  auto read_box = [&](int parity, Item& it) {
    it.kt = __builtin_amdgcn_readfirstlane(mbox[parity][0]);
    it.head = __builtin_amdgcn_readfirstlane(mbox[parity][1]);
    it.tok_start = __builtin_amdgcn_readfirstlane(mbox[parity][2]);
    it.doc_len = __builtin_amdgcn_readfirstlane(mbox[parity][3]);
    it.tab_base = __builtin_amdgcn_readfirstlane(mbox[parity][4]);
    it.tile_base = __builtin_amdgcn_readfirstlane(mbox[parity][5]);
    it.batch = __builtin_amdgcn_readfirstlane(mbox[parity][6]);
    return it.kt >= 0;
  };
  using Copy = TileCopy<D, TQ, 256, false, STREAM>;
  constexpr int LOADS_PER_TILE = 2 * Copy::NCH;

  // ---- the queue of this XCD ---------------------------------------------------------------------
  // Chains (document rank, head), longest documents first, are dealt to the XCDs in turn, CHAIN_GROUP to each from every
  // group of eight times as many.  The key tiles of an XCD's chains of a group are interleaved (tile 0 of each, tile 1 of
  // each, ...), so that the tiles that start together at the beginning of a launch have few predecessors to wait for.
  // Ticket numbers run over the groups' items; a group has room for its longest chain, the tickets behind a
  // shorter one's end name no item and are drawn past.
  // An XCD that the launch cannot run on (a CU mask) is dealt none: the XCDs counted are those that the prep kernel met.
  // With n of them each takes every n-th chain of a group, in room for the next power of two.
  const int xcd = this_xcd();
  unsigned* const ctr = a.queues + xcd * CHAIN_QUEUE_STRIDE;
  const int n_groups = (n_chains + CHAIN_QUEUES * CHAIN_GROUP - 1) / (CHAIN_QUEUES * CHAIN_GROUP);
  auto group_tiles = [&](int g) {   // of group g's longest chain: the first one belongs to its longest document
    if (g >= n_groups) return 0;
    const int len = docs[2 * (CHAIN_QUEUES * CHAIN_GROUP * g / a.heads)].y;
    return (len + BKV - 1) / BKV;
  };
  // first score wave: the item of a ticket, or the items of further tickets, as `mbox` words of the lanes 0 .. 7
  auto resolve = [&](unsigned ticket) -> int {
    const int first = prefix[lane], here = __builtin_amdgcn_readfirstlane(place), n_xcds = here >> 8;
    const int lg = 3 + __builtin_clz(n_xcds) - __builtin_clz(CHAIN_QUEUES);    // room for 2^lg chains per group
    static_assert(CHAIN_GROUP == 8 && CHAIN_MAX_GROUPS % 64 == 0, "lg; 64 prefixes at a time");
    for (;;) {
      const int tk = __builtin_amdgcn_readfirstlane((int)ticket);
      int group = -1, before = 0;
      for (int g0 = 0; g0 < n_groups; g0 += 64) {
        const int upto = g0 == 0 ? first : prefix[g0 + lane];       // (past the last group: anything)
        const unsigned long long m = __builtin_amdgcn_ballot_w64((tk >> lg) < upto && g0 + lane < n_groups);
        if (m != 0) {
          const int at = __builtin_ctzll(m);
          group = g0 + at;
          before = at > 0 ? __builtin_amdgcn_readlane(upto, at - 1) : g0 > 0 ? __builtin_amdgcn_readfirstlane(prefix[g0 - 1]) : 0;
          break;
        }
      }
      if (group < 0) return -1;
      const int kt = (tk >> lg) - before, in_group = (tk & ((1 << lg) - 1)) * n_xcds + (here & 0xff);
      const int chain = CHAIN_QUEUES * CHAIN_GROUP * group + in_group;
      if (in_group < CHAIN_QUEUES * CHAIN_GROUP && chain < n_chains) {
        const int rank = chain / a.heads;
        const int2 d0 = docs[2 * rank], d1 = docs[2 * rank + 1];
        if (kt * BKV < d0.y) {
          int v = kt;
          v = lane == 1 ? chain - rank * a.heads : v;
          v = lane == 2 ? d0.x : v;
          v = lane == 3 ? d0.y : v;
          v = lane == 4 ? d1.x : v;
          v = lane == 5 ? d1.y : v;
          v = lane == 6 ? (a.fixed ? rank : 0) : v;
          return v;
        }
      }
      unsigned next = 0;
      if (lane == 0) next = atomicAdd(ctr, 1u);
      ticket = next;
    }
  };
  if (w == 0) {
    unsigned ticket = 0;
    if (lane == 0) {
      ticket = atomicAdd(ctr, 1u);
      given_up = 0.0f;
    }
    const int home = lane < a.n_homes ? a.homes[lane] : -1;
    int base = 0;
    for (int g0 = 0; g0 < n_groups; g0 += 64) {
      int v = group_tiles(g0 + lane);
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
      }
      if (g0 + lane < n_groups) prefix[g0 + lane] = base + v;
      base += __shfl(v, 63, 64);
    }
    int met = 0;
#pragma unroll
    for (int x = 0; x < CHAIN_QUEUES; ++x) met |= __builtin_amdgcn_ballot_w64(home == x) != 0 ? 1 << x : 0;
    if (lane == 0) place = __builtin_popcount(met) << 8 | __builtin_popcount(met & ((1 << xcd) - 1));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int word = (met >> xcd) & 1 ? resolve(ticket) : -1;
    if (lane < 8) mbox[1][lane] = word;
  }
  lds_barrier();
  Item cur;
  if (!read_box(1, cur)) return;

  using Yes = std::true_type;
  using No = std::false_type;
  if (scorer) {
    __builtin_amdgcn_s_setprio(3);
    const int kb = w & 3, sq = w >> 2;            // 32-key block and 32-query block of this wave
    el8 kf[KS], vf[KS];                           // MFMA row n holds key k0 + kperm(n)
    int k0, nsteps, doc_len, t_last, n_wait;
    float rem_own;
    int row4, last4;
    __amdgpu_buffer_rsrc_t stick_rs, in_rs, out_rs;
    float se0, se1, se2;                          // stick on entering the block, requested ahead, three steps in turn
    float d_next;                                 // carried sum of the next step's query, requested one step ahead
    const int* pred = nullptr;                    // steps the chain's tile before this one has published
    int* mine = nullptr;
    int seen = 0;
    int roff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) roff[ks] = swz_off<D>(32 * sq + n, 2 * ks + h);

    auto row_off = [&](int step) { return min(row4 - step * (4 * TQ), last4); };   // (below zero: outside the resource)
    auto request_e = [&](int step, float& e) { e = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(stick_rs, row_off(step), 0, 0)); };
    auto request_d = [&](int step) { d_next = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(in_rs, row_off(step), 0, 16 /* sc1 */)); };
    auto open_item = [&](const ChainArgs& a, const Item& it) {
      int n = lane & 31, h = lane >> 5;           // (opaque here: nothing per-lane of an item's prologue is to live through its steps)
      asm volatile("" : "+v"(n), "+v"(h));
      doc_len = it.doc_len;
      k0 = it.kt * BKV + 32 * kb;
      t_last = (doc_len - 1) / TQ;
      nsteps = t_last - it.kt * DIAG + 1;
      const int tblock = min((BKV / 32) * it.kt + kb, (doc_len - 1) / 32);   // (a block behind the document's end reads the last one's rows, unused)
      const int64_t tab = (int64_t)it.head * a.tab_stride + it.tab_base;
      rem_own = 0.0f;
      if (a.fuse && k0 + n < doc_len) rem_own = a.stick[tab + tab_rowplane32(doc_len) + k0 + n];
      const unsigned run_bytes = (unsigned)doc_len * 4u;
      stick_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.stick) + tab + tab_seg32(doc_len, tblock), 0, run_bytes, 0x00020000);
      const int64_t plane = (int64_t)a.heads * a.tiles * BM, at = ((int64_t)it.head * a.tiles + it.tile_base) * BM;
      in_rs = __builtin_amdgcn_make_buffer_rsrc(a.carry + (it.kt & 1) * plane + at, 0, run_bytes, 0x00020000);
      out_rs = __builtin_amdgcn_make_buffer_rsrc(a.carry + ((it.kt + 1) & 1) * plane + at, 0, run_bytes, 0x00020000);
      row4 = 4 * (t_last * TQ + 32 * sq + n);
      last4 = 4 * (doc_len - 1);
      int* fl = a.flags + (int64_t)it.head * a.tiles + it.tile_base + it.kt;
      pred = fl - 1;
      mine = fl;
      n_wait = it.kt > 0 ? nsteps : 0;
      seen = 0;
      request_e(0, se0);
      request_e(1, se1);
      if constexpr (DEEP) request_e(2, se2);
    };
    // the first AHEAD tiles of an item (first query block's score waves copy)
    auto open_tiles = [&](const ChainArgs& a, const Item& it) {
      if (sq != 0) return;
      int l = lane;
      asm volatile("" : "+v"(l));
      const Rows qrows = rows_of(a.q, it), grows = rows_of(a.go, it);
      Copy qcopy, gcopy;
      qcopy.init(64 * kb + l, qrows.row_bytes, qrows.used_bytes);
      gcopy.init(64 * kb + l, grows.row_bytes, grows.used_bytes);
#pragma unroll
      for (int s = 0; s < AHEAD; ++s)
        if (s < nsteps) {
          qcopy.issue(qrows, (t_last - s) * TQ, Qs + s * QTILE);
          gcopy.issue(grows, (t_last - s) * TQ, Gs + s * QTILE);
        }
    };
    // K and V fragments of this wave's keys from the tiles the product waves have staged
    auto take_fragments = [&]() {
      int n = lane & 31, h = lane >> 5;
      asm volatile("" : "+v"(n), "+v"(h));
      const int r = 32 * kb + kperm(n);
      const unsigned short* Vt = DEEP ? (kb < 2 ? Qs : Gs) + AHEAD * QTILE : PZ + BKV * D;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        kf[ks] = lds_row8(PZ + swz_off<D>(r, 2 * ks + h));
        vf[ks] = lds_row8(Vt + swz_off<D>(DEEP ? r & 63 : r, 2 * ks + h));
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    // First score wave: the tile before this one has published `steps` steps (all of them: nothing to wait for any
    // more).  A wait that runs out -- it cannot while workgroups make progress -- must end in NaN and not in plausible
    // numbers, in every wave: what it stood for is requested by all of them behind the barrier that follows, the
    // partial dq of the block whose dz is formed there and the carried sum of the next one.  The waves of the oldest
    // key block add `given_up` to that dz, which makes all of the block's dq NaN, and to the stick of the next block,
    // whose weights they form in the same step: its p and dz are NaN, so is the sum every newer key block takes from
    // `tot` for its D, and with dz of all of the tile's keys dk, dq and what is handed on.
    auto await = [&](int steps) {
      const int need = min(steps, n_wait);
      auto published = [&]() {
        seen = __builtin_amdgcn_readfirstlane(__hip_atomic_load(pred, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        return seen >= need;
      };
      if (seen >= need || published()) return;
      const int limit = fresh_args<ChainArgs>().spin_limit;
      for (int tries = 0; tries < limit; ++tries) {
        __builtin_amdgcn_s_sleep(2);
        if (published()) return;
      }
      if (lane == 0) given_up = __builtin_nanf("");
      n_wait = 0;
    };
    auto chains = [&](int slot, f32x16& x, f32x16& da) {
      const unsigned short* Qt = Qs + slot * QTILE;
      const unsigned short* Gt = Gs + slot * QTILE;
#pragma unroll
      for (int j = 0; j < 16; ++j) { x[j] = 0.0f; da[j] = 0.0f; }
      el8 qfr[KS], gfr[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) { qfr[ks] = lds_row8(Qt + roff[ks]); gfr[ks] = lds_row8(Gt + roff[ks]); }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        x = mfma32(kf[ks], qfr[ks], x);
        da = mfma32(vf[ks], gfr[ks], da);
      }
    };

    // A block none of whose keys the queries from qw0 on may see: zeros in the place of its dz, staged before.  (By a
    // second store: with a choice between the two values in the step itself the values alive across it do not fit the
    // registers, and a mask costs every step.)
    auto hide = [&](int qw0, int par) {
      if (!sub_skip<AC>(k0, qw0)) return;
#pragma unroll
      for (int c = 0; c < 2; ++c) *reinterpret_cast<el8*>(Zs + par * PTILE + swz_off<BKV>(32 * sq + n, 4 * kb + 2 * h + c)) = zero8();
    };
    // What a step keeps of a block between forming its weights and forming its dz, one step later.
    struct Weights { float p[16], r[16], lo; };
    // Step w: dz of block w (weights and do.v in `wc`, `dc`, formed a step ago), weights of block w + 1 (scores `xn`,
    // do.v `dn`) into `wn`, and the two MFMA chains of block w + 2 into `xf`, `df`, interleaved with the vector work in
    // eight chunks (see bulk in sba_bwd.hip).  The sum over the key blocks before this wave's goes through `tot`:
    // written with the weights, read a step later.  FIRST: there is no block w yet.  BAND: block w or w + 1 may hold
    // keys its queries must not see.  A block that hides all of them stages zeros and nothing computed: where a key has
    // a value that is not finite, or a query a running sum that is not, 0 times it is not zero.  SLOT >= 0: ring slot
    // of tile w + 2, else taken from w.
    auto step = [&](auto first_tag, auto band_tag, auto slot_tag, const int w, Weights& wc, f32x16& dc, f32x16& xn, f32x16& dn,
                    Weights& wn, f32x16& xf, f32x16& df, float& se) __attribute__((always_inline)) {
      constexpr bool FIRST = decltype(first_tag)::value, BAND = decltype(band_tag)::value;
      constexpr int SLOT = decltype(slot_tag)::value;
      constexpr int NCHUNK = 8, PER = 2 * (D / 16) / NCHUNK, LEAD = 2;
      const int slot = SLOT >= 0 ? SLOT : (w + 2) % RING;
      const int par = SLOT >= 0 ? (SLOT & 1) : (w & 1);
      const int p_buf = SLOT >= 0 ? (SLOT + 2) % 3 : (w + 1) % 3;    // of block w + 1
      float d_in = 0.0f, t0 = 0.0f, t1 = 0.0f, t2 = 0.0f;
      if constexpr (!FIRST) {
        d_in = d_next;
        if (kb > 0) t0 = tot[par][sq][0][n];
        if (kb > 1) t1 = tot[par][sq][1][n];
        if (kb > 2) t2 = tot[par][sq][2][n];
      }
      request_d(w + 1);
      float e_in = se, doubt = 0.0f;
      if (kb == 0) doubt = given_up;
      e_in += doubt;
      request_e(w + 4, se);
      const unsigned short* Qt = Qs + slot * QTILE;
      const unsigned short* Gt = Gs + slot * QTILE;
#pragma unroll
      for (int j = 0; j < 16; ++j) { xf[j] = 0.0f; df[j] = 0.0f; }
      el8 fr[LEAD + 1][PER];
      auto pre = [&](int c) {
        if (c >= NCHUNK) return;
#pragma unroll
        for (int m = 0; m < PER; ++m) {
          const int k = c * PER + m;
          if (k >= 2 * KS) continue;
          fr[c % (LEAD + 1)][m] = lds_row8(((k & 1) ? Gt : Qt) + roff[k >> 1]);
        }
      };
      auto post = [&](int c) {
#pragma unroll
        for (int m = 0; m < PER; ++m) {
          const int k = c * PER + m;
          if (k >= 2 * KS) continue;
          if (k & 1) df = mfma32(vf[k >> 1], fr[c % (LEAD + 1)][m], df);
          else xf = mfma32(kf[k >> 1], fr[c % (LEAD + 1)][m], xf);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      const int qw0 = (t_last - (w + 1)) * TQ + 32 * sq;
      const int lim = qw0 + n - k0 - 16 * h + (AC ? 1 : 0);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        wn.r[j] = fast_rcp(1.0f + fast_exp2(a.c * xn[j]));
        if (BAND && !(j < lim)) wn.r[j] = 1.0f;
      }
      __builtin_amdgcn_sched_barrier(0);
      pre(0);
      pre(1);
#pragma unroll
      for (int j = 8; j < 16; ++j) {
        wn.r[j] = fast_rcp(1.0f + fast_exp2(a.c * xn[j]));
        if (BAND && !(j < lim)) wn.r[j] = 1.0f;
      }
      __builtin_amdgcn_sched_barrier(0);
      pre(2);
      const int row = n;
      if constexpr (!FIRST) {
        const float before = (d_in + doubt) + ((t0 + t1) + t2);
        float dprev = h == 1 ? before + wc.lo : before;
        float dz[16];
#pragma unroll
        for (int j = 0; j < 8; ++j) { const float dj = fmaf(wc.p[j], dc[j], dprev); dz[j] = fmaf(wc.r[j], dj, -dprev); dprev = dj; }
        post(0);
        pre(3);
#pragma unroll
        for (int j = 8; j < 16; ++j) { const float dj = fmaf(wc.p[j], dc[j], dprev); dz[j] = fmaf(wc.r[j], dj, -dprev); dprev = dj; }
        unsigned short* Zt = Zs + par * PTILE;
        *reinterpret_cast<el8*>(Zt + swz_off<BKV>(32 * sq + row, 4 * kb + 2 * h)) = pack8(dz);
        *reinterpret_cast<el8*>(Zt + swz_off<BKV>(32 * sq + row, 4 * kb + 2 * h + 1)) = pack8(dz + 8);
        // what the next key tile starts from (the half-wave with the newer keys ends with the sum over all)
        if (kb == 3 && h == 1) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, dprev), out_rs, row4 - w * (4 * TQ), 0, 0);
        post(1);
      } else {
        post(0);
        pre(3);
        post(1);
      }
      pre(4);
      post(2);
      // block w + 1: stick left after the newer keys, weights
      pre(5);
      float ex[16];
      // (a block none of whose keys the queries may see: the table holds no value for it)
      if (BAND) e_in = sub_skip<AC>(k0, qw0) ? 0.0f : e_in;
      (void)suffix_prod32_excl(wn.r, ex, h, e_in);
      post(3);
      pre(6);
      wn.p[0] = ex[0] - ex[0] * wn.r[0];
#pragma unroll
      for (int j = 1; j < 16; ++j) wn.p[j] = ex[j] - ex[j - 1];
      unsigned short* Pt = Ps + p_buf * PTILE;
      if (BAND && a.fuse && qw0 == k0) {      // o + rem v: rem_j do_j reaches dv_j through the diagonal of p (see sba_bwd.hip)
        float pd[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) pd[j] = wn.p[j] + (16 * h + j == n ? rem_own : 0.0f);
        *reinterpret_cast<el8*>(Pt + swz_off<BKV>(32 * sq + row, 4 * kb + 2 * h)) = pack8(pd);
        *reinterpret_cast<el8*>(Pt + swz_off<BKV>(32 * sq + row, 4 * kb + 2 * h + 1)) = pack8(pd + 8);
      } else {
        *reinterpret_cast<el8*>(Pt + swz_off<BKV>(32 * sq + row, 4 * kb + 2 * h)) = pack8(wn.p);
        *reinterpret_cast<el8*>(Pt + swz_off<BKV>(32 * sq + row, 4 * kb + 2 * h + 1)) = pack8(wn.p + 8);
      }
      post(4);
      pre(7);
      float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
      for (int j = 0; j < 16; j += 2) { s0 = fmaf(wn.p[j], dn[j], s0); s1 = fmaf(wn.p[j + 1], dn[j + 1], s1); }
      float lo, hi;
      both_halves(s0 + s1, lo, hi);
      wn.lo = lo;
      if (h == 0) tot[par ^ 1][sq][kb][n] = lo + hi;
      post(5);
      post(6);
      post(7);
      if constexpr (BAND && !FIRST) hide(qw0 + TQ, par);
    };
    // The same with one step less between a block's products and its weights, for three waves per SIMD (168 registers), which
    // hide what the pipeline above hides: step w forms the products of block w + 1 next to dz of block w, stages p and
    // dz of block w and then forms the weights of block w + 1 in their place.  `dc`, `dn`: do.v of the two blocks.
    auto shallow = [&](auto first_tag, auto band_tag, const int w, const int slot, Weights& wc, f32x16& dc, f32x16& dn, float& se) __attribute__((always_inline)) {
      constexpr bool FIRST = decltype(first_tag)::value, BAND = decltype(band_tag)::value;
      const int par = w & 1;
      float d_in = 0.0f, t0 = 0.0f, t1 = 0.0f, t2 = 0.0f;
      if constexpr (!FIRST) {
        d_in = d_next;
        if (kb > 0) t0 = tot[par][sq][0][n];
        if (kb > 1) t1 = tot[par][sq][1][n];
        if (kb > 2) t2 = tot[par][sq][2][n];
      }
      request_d(w + 1);
      float e_in = se, doubt = 0.0f;
      if (kb == 0) doubt = given_up;
      e_in += doubt;
      request_e(w + 3, se);
      const unsigned short* Qt = Qs + slot * QTILE;
      const unsigned short* Gt = Gs + slot * QTILE;
      f32x16 x;
#pragma unroll
      for (int j = 0; j < 16; ++j) { x[j] = 0.0f; dn[j] = 0.0f; }
      el8 fq[2], fg[2];
      auto pre = [&](int c) {
        if (c >= KS) return;
        fq[c & 1] = lds_row8(Qt + roff[c]);
        fg[c & 1] = lds_row8(Gt + roff[c]);
      };
      auto post = [&](int c) {
        if (c >= KS) return;
        x = mfma32(kf[c], fq[c & 1], x);
        dn = mfma32(vf[c], fg[c & 1], dn);
        pre(c + 2);
        __builtin_amdgcn_sched_barrier(0);
      };
      const int qw1 = (t_last - (w + 1)) * TQ + 32 * sq, qw0 = qw1 + TQ;
      pre(0);
      pre(1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!FIRST) {
        const float before = (d_in + doubt) + ((t0 + t1) + t2);
        float dprev = h == 1 ? before + wc.lo : before;
        float dz[16];
#pragma unroll
        for (int j = 0; j < 8; ++j) { const float dj = fmaf(wc.p[j], dc[j], dprev); dz[j] = fmaf(wc.r[j], dj, -dprev); dprev = dj; }
        post(0);
        unsigned short* Zt = Zs + par * PTILE;
        unsigned short* Pt = Ps + par * PTILE;
        *reinterpret_cast<el8*>(Zt + swz_off<BKV>(32 * sq + n, 4 * kb + 2 * h)) = pack8(dz);
#pragma unroll
        for (int j = 8; j < 16; ++j) { const float dj = fmaf(wc.p[j], dc[j], dprev); dz[j] = fmaf(wc.r[j], dj, -dprev); dprev = dj; }
        post(1);
        *reinterpret_cast<el8*>(Zt + swz_off<BKV>(32 * sq + n, 4 * kb + 2 * h + 1)) = pack8(dz + 8);
        if (kb == 3 && h == 1) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, dprev), out_rs, row4 - w * (4 * TQ), 0, 0);
        if (BAND && a.fuse && qw0 == k0) {
#pragma unroll
          for (int j = 0; j < 16; ++j) wc.p[j] += 16 * h + j == n ? rem_own : 0.0f;
        }
        *reinterpret_cast<el8*>(Pt + swz_off<BKV>(32 * sq + n, 4 * kb + 2 * h)) = pack8(wc.p);
        *reinterpret_cast<el8*>(Pt + swz_off<BKV>(32 * sq + n, 4 * kb + 2 * h + 1)) = pack8(wc.p + 8);
        post(2);
        post(3);
      } else {
#pragma unroll
        for (int c = 0; c < KS; ++c) post(c);
      }
      const int lim = qw1 + n - k0 - 16 * h + (AC ? 1 : 0);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        wc.r[j] = fast_rcp(1.0f + fast_exp2(a.c * x[j]));
        if (BAND && !(j < lim)) wc.r[j] = 1.0f;
      }
      float ex[16];
      if (BAND) e_in = sub_skip<AC>(k0, qw1) ? 0.0f : e_in;
      (void)suffix_prod32_excl(wc.r, ex, h, e_in);
      wc.p[0] = ex[0] - ex[0] * wc.r[0];
#pragma unroll
      for (int j = 1; j < 16; ++j) wc.p[j] = ex[j] - ex[j - 1];
      float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
      for (int j = 0; j < 16; j += 2) { s0 = fmaf(wc.p[j], dn[j], s0); s1 = fmaf(wc.p[j + 1], dn[j + 1], s1); }
      float lo, hi;
      both_halves(s0 + s1, lo, hi);
      wc.lo = lo;
      if (h == 0) tot[par ^ 1][sq][kb][n] = lo + hi;
      if constexpr (BAND && !FIRST) hide(qw0, par);
    };
    // ends a step: the first score wave makes sure that what the others request behind the barrier is there, the second
    // publishes what this tile has finished and, before a step, asks in the background how far the tile before is
    auto finish = [&](int w) {
      // (what a step issues: two requests and this store)
      if (kb == 3) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");     // the carried sum stored a step ago is acknowledged
      if (sq == 0 && kb == 0 && n_wait > 0) {
        if (seen < min(w + 2, n_wait)) seen = max(seen, __builtin_amdgcn_readfirstlane(fbox[0]));
        await(w + 2);
      }
      lds_barrier();
    };
    auto publish = [&](int w) {
      if (sq == 0 && kb == 0 && seen < min(w + 2, n_wait)) async_word(pred, fbox);
      if (sq == 0 && kb == 1 && w >= 3 && lane == 0) __hip_atomic_store(mine, w - 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const bool keeper = w == 0;
    unsigned ticket = 0;
    int word = -1;
    auto queue = [&](int w, int parity) {
      if (!keeper) return;
      if (w == max(nsteps - 6, 0) && lane == 0) ticket = atomicAdd(ctr, 1u);
      if (w == max(nsteps - 2, 0)) word = resolve(ticket);
      if (w == nsteps - 1 && lane < 8) mbox[parity][lane] = word;
    };

    using std::integral_constant;
    using RT = integral_constant<int, -1>;
    open_item(a, cur);
    open_tiles(a, cur);
#pragma unroll 1
    for (int m = 0;; ++m) {
      if (keeper) await(1);
      wait_loads<0>();
      lds_barrier();                 // tiles 0 .. AHEAD-1 and the K and V tiles have landed
      take_fragments();
      if (keeper) fbox[lane] = 0;
      lds_barrier();                 // every wave has its share of K and V in registers: their places are free
      if constexpr (DEEP) {
        f32x16 x0, x1, da0, da1, da2;
        Weights wa, wb;
        chains(0, x0, da0);
        // weights of block 0 (as step -1), chains of block 1
        step(Yes{}, Yes{}, RT{}, -1, wb, da2, x0, da0, wa, x1, da1, se0);
        if (keeper) await(1);
        lds_barrier();
        int i = 0;
        // Everything repeats with period six (ring slots, staging buffers, weights, scores, do.v sums, carries): step i
        // = 6 m has block i's weights in wa, its do.v in da0, block i+1's scores in x1 and do.v in da1.
#pragma unroll 1
        for (; i + 6 < nsteps - DIAG - 2; i += 6) {
          publish(i);     step(No{}, No{}, integral_constant<int, 2>{}, i, wa, da0, x1, da1, wb, x0, da2, se1);     finish(i);
          publish(i + 1); step(No{}, No{}, integral_constant<int, 3>{}, i + 1, wb, da1, x0, da2, wa, x1, da0, se2); finish(i + 1);
          publish(i + 2); step(No{}, No{}, integral_constant<int, 4>{}, i + 2, wa, da2, x1, da0, wb, x0, da1, se0); finish(i + 2);
          publish(i + 3); step(No{}, No{}, integral_constant<int, 5>{}, i + 3, wb, da0, x0, da1, wa, x1, da2, se1); finish(i + 3);
          publish(i + 4); step(No{}, No{}, integral_constant<int, 0>{}, i + 4, wa, da1, x1, da2, wb, x0, da0, se2); finish(i + 4);
          publish(i + 5); step(No{}, No{}, integral_constant<int, 1>{}, i + 5, wb, da2, x0, da0, wa, x1, da1, se0); finish(i + 5);
        }
#pragma unroll 1
        for (;; i += 6) {
          if (i >= nsteps) break;
          queue(i, m & 1);     publish(i);     step(No{}, Yes{}, RT{}, i, wa, da0, x1, da1, wb, x0, da2, se1);     finish(i);
          if (i + 1 >= nsteps) break;
          queue(i + 1, m & 1); publish(i + 1); step(No{}, Yes{}, RT{}, i + 1, wb, da1, x0, da2, wa, x1, da0, se2); finish(i + 1);
          if (i + 2 >= nsteps) break;
          queue(i + 2, m & 1); publish(i + 2); step(No{}, Yes{}, RT{}, i + 2, wa, da2, x1, da0, wb, x0, da1, se0); finish(i + 2);
          if (i + 3 >= nsteps) break;
          queue(i + 3, m & 1); publish(i + 3); step(No{}, Yes{}, RT{}, i + 3, wb, da0, x0, da1, wa, x1, da2, se1); finish(i + 3);
          if (i + 4 >= nsteps) break;
          queue(i + 4, m & 1); publish(i + 4); step(No{}, Yes{}, RT{}, i + 4, wa, da1, x1, da2, wb, x0, da0, se2); finish(i + 4);
          if (i + 5 >= nsteps) break;
          queue(i + 5, m & 1); publish(i + 5); step(No{}, Yes{}, RT{}, i + 5, wb, da2, x0, da0, wa, x1, da1, se0); finish(i + 5);
        }
      } else {
        f32x16 da0, da1;
        Weights wa;
        shallow(Yes{}, Yes{}, -1, 0, wa, da1, da0, se0);
        if (keeper) await(1);
        lds_barrier();
        int i = 0, slot = 1;
        auto advance = [&]() { slot = slot + 1 == RING ? 0 : slot + 1; };
#pragma unroll 1
        for (; i + 1 < nsteps - 6; i += 2) {
          publish(i);     shallow(No{}, No{}, i, slot, wa, da0, da1, se1);     advance(); finish(i);
          publish(i + 1); shallow(No{}, No{}, i + 1, slot, wa, da1, da0, se0); advance(); finish(i + 1);
        }
#pragma unroll 1
        for (; i < nsteps; i += 2) {
          queue(i, m & 1);     publish(i);     shallow(No{}, Yes{}, i, slot, wa, da0, da1, se1);     advance(); finish(i);
          if (i + 1 >= nsteps) break;
          queue(i + 1, m & 1); publish(i + 1); shallow(No{}, Yes{}, i + 1, slot, wa, da1, da0, se0); advance(); finish(i + 1);
        }
      }
      publish(nsteps);
      const bool more = read_box(m & 1, cur);
      if (more) open_item(fresh_args<ChainArgs>(), cur);
      lds_barrier();                 // the product waves are done with the last Q tile
      if (!more) break;
      open_tiles(fresh_args<ChainArgs>(), cur);
    }
  } else {
    __builtin_amdgcn_s_setprio(0);
    const int pw = w - 4 * NSQ;
    const int ptid = pw * 64 + lane;
    const int lane16 = lane * 16;
    const int mat = pw >> 1, half = pw & 1;       // (dv | dk) x 64 keys; all columns
    const bool has_dq = pw < NSQ * DB;            // 32 x 32 block of dq: query block pw / DB, columns 32 (pw % DB)
    const int dsq = has_dq ? pw / DB : 0, dcol = pw % DB;
    f32x16 acc[2][DB];
#pragma unroll
    for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
      for (int j = 0; j < DB; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[kb2][j][i] = 0.0f;
    // Offsets (bytes) of this lane's reads.  The swizzle is an XOR of the chunk number, so the offset of a further
    // chunk is the first one's with a constant XORed in: one register per row instead of one per read -- there is none
    // to spare, and a spilled one would be reloaded through the counter that the waits below count on.  In bytes, and
    // added to the tile's place as an integer: XOR and addition are then one instruction.
    int xb[2], yb[2];      // transpose reads of rows 8 h + 4 u + i16 / 4: staged block (chunk of key 64 half), tile (chunk of column 0)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = 8 * h + 4 * u + (i16 >> 2), c = 16 * blk + 4 * (i16 & 3);
      xb[u] = 2 * (swz_off<BKV>(r, (64 * half + c) >> 3) + (c & 7));
      yb[u] = 2 * (swz_off<D>(r, c >> 3) + (c & 7));
    }
    int zb = 2 * swz_off<BKV>(32 * dsq + n, h);      // row reads of staged dz: chunk 2 ks + h of row n
    auto place_of = [](const unsigned short* p) { return (int)(unsigned)(size_t)p; };     // LDS address
    auto tr8 = [](int at0, int at1) { return lds_tr8_at(at0, at1); };
    Copy qcopy, gcopy;
    qcopy.init(ptid, (unsigned)a.q.st * 2u, 2 * a.head_dim);
    gcopy.init(ptid, (unsigned)a.go.st * 2u, 2 * a.head_dim);
    el8 kt_f[BKV / 16];                            // this wave's 32 columns of the key tile, as the B operand of dq = dz K
    Rows qrows, grows;
    __amdgpu_buffer_rsrc_t part_rs;
    int t_last, nsteps, doc_len, kt;
    auto open_item = [&](const ChainArgs& a, const Item& it) {
      qrows = rows_of(a.q, it);
      grows = rows_of(a.go, it);
      doc_len = it.doc_len;
      kt = it.kt;
      t_last = (doc_len - 1) / TQ;
      nsteps = t_last - kt * DIAG + 1;
      // partial dq: per 32 rows and 32 columns 1024 floats as the accumulators lie
      float* part = a.partial + ((int64_t)it.head * a.tiles + it.tile_base) * (BM * D) + dcol * 1024;
      part_rs = __builtin_amdgcn_make_buffer_rsrc(part, 0, (unsigned)((doc_len + BM - 1) / BM) * (BM * D * 4u) - (unsigned)dcol * 4096u, 0x00020000);
      // The K tile into the staging buffers and the V tile into the two ring slots the item's first tiles leave free, in
      // natural order.  (Fragments straight from global memory -- 32 rows of 32 bytes per instruction -- took
      // 6400 cycles of an item's beginning to issue, these copies 1000.)
      static_assert(!DEEP || (AHEAD + 2 <= RING && 2 * QTILE >= 64 * D), "half of the V tile per ring");
      int l = lane16;
      asm volatile("" : "+v"(l));
      l = pw * 64 + (l >> 4);
      const Rows krows = rows_of(a.k, it), vrows = rows_of(a.v, it);
      TileCopy<D, BKV, 256, false, true> kcopy;
      kcopy.init(l, krows.row_bytes, krows.used_bytes);
      kcopy.issue(krows, kt * BKV, PZ);
      if constexpr (DEEP) {
        TileCopy<D, 64, 256, false, true> vcopy;
        vcopy.init(l, vrows.row_bytes, vrows.used_bytes);
        vcopy.issue(vrows, kt * BKV, Qs + AHEAD * QTILE);
        vcopy.issue(vrows, kt * BKV + 64, Gs + AHEAD * QTILE);
      } else {
        TileCopy<D, BKV, 256, false, true> vcopy;
        vcopy.init(l, vrows.row_bytes, vrows.used_bytes);
        vcopy.issue(vrows, kt * BKV, PZ + BKV * D);
      }
    };
    auto take_key_tile = [&]() {
      if (has_dq) {
#pragma unroll
        for (int ks = 0; ks < BKV / 16; ++ks)
          kt_f[ks] = tr8((yb[0] ^ (dcol << 6)) + place_of(PZ) + 32 * ks * D, (yb[1] ^ (dcol << 6)) + place_of(PZ) + 32 * ks * D);
      } else {
#pragma unroll
        for (int ks = 0; ks < BKV / 16; ++ks) kt_f[ks] = zero8();
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    Item nxt;
    open_item(a, cur);
#pragma unroll 1
    for (int m = 0;; ++m) {
      // the K and V tiles have landed (the stores of the item before may still be on their way)
      if (m == 0) wait_loads<0>();
      else wait_loads<4 * DB>();
      lds_barrier();
      take_key_tile();
      lds_barrier();
      lds_barrier();                 // weights of block 0 are staged
      // Iteration w: dq, and dv or dk, of block w - 1; a tile is copied and the next partial dq requested.
      // A product wave is bound by what it can issue next to a score wave: the eight dependent products of dq are
      // spread between those of dk / dv, and the memory instructions -- the partial dq stored, the next one requested, a
      // tile copied -- go out one behind each further product (in one go, 4 + 4 + 4 of every wave queue up in front of the
      // CU's address unit: 500 cycles of an iteration of 2800).  Every iteration issues the same ones in the
      // same order, with an offset outside the resource where there is nothing to store, request or copy, so that
      // the waits count constants and no value on its way has to be moved where two paths join.
      f32x4 l0, l1, l2, l3;           // partial dq on its way in
      constexpr int KQ = TQ / 16, KZ = BKV / 16, ZH = DEEP ? KZ / 2 : 2;
      constexpr int QB = 2 * QTILE, PB = 2 * PTILE;      // bytes of a tile, of a staged block
      constexpr bool ALL_DQ = NSQ * DB >= 4;             // every product wave has a block of dq
      constexpr int FETCH_OPS = 4 + 2 * Copy::NCH;
      constexpr int N_PRODUCTS = KQ * 2 * DB, REST = N_PRODUCTS - KZ / 2, OPS = 4 + FETCH_OPS;
      // What a block needs besides its products: 45 vector and 41 scalar instructions an iteration (108 and about 100
      // with the places computed from the block's number and selects for what only an item's last iterations need).
      // Places that move on with the blocks: staged blocks, tile read by dk / dv, ring slot that is copied to, and in
      // memory the partial dq of the block that is stored and the rows that are copied.
      const int y0 = place_of(mat ? Qs : Gs), x0 = place_of(mat ? Zs : Ps), x_end = x0 + (mat ? 2 : PBUF) * PB;
      int y_at = y0, x_at = x0, z_at = place_of(Zs), c_at = AHEAD * QB;
      int part_at = (t_last * NSQ + dsq) * (D * 128);                  // bytes of partial dq ahead of the next request's 32 rows
      int q_row = (t_last - AHEAD) * TQ * (int)qrows.row_bytes, g_row = (t_last - AHEAD) * TQ * (int)grows.row_bytes;
      const bool takes = has_dq && kt > 0;
      auto store_part = [&](const int i, const f32x16& dq, const bool store) __attribute__((always_inline)) {
        const f32x4 part = {dq[4 * i], dq[4 * i + 1], dq[4 * i + 2], dq[4 * i + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, part), part_rs, (store ? lane16 : OUTSIDE) + 1024 * i, part_at + NSQ * D * 128, 0);
        // The registers must not be written right behind the store.  The compiler leaves the wait state for that out
        // where the store's offset is in a scalar register; an address computed into one by the next instruction was
        // stored in its place in lanes 12 .. 15, now and then.  (The registers are an operand so that nothing else is
        // put in between.)
        asm volatile("s_nop 0" ::"v"(part) : "memory");
      };
      // operation i of those that request: partial dq of the block whose rows part_at names, then the tile AHEAD of it
      auto fetch = [&](const int i, const bool more, const bool fetched) __attribute__((always_inline)) {
        const int l_off = takes && more ? lane16 : OUTSIDE;
        if (i == 0) asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen sc1" : "=&v"(l0) : "v"(l_off), "s"(part_rs), "s"(part_at) : "memory");
        if (i == 1) asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen offset:1024 sc1" : "=&v"(l1) : "v"(l_off), "s"(part_rs), "s"(part_at) : "memory");
        if (i == 2) asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen offset:2048 sc1" : "=&v"(l2) : "v"(l_off), "s"(part_rs), "s"(part_at) : "memory");
        if (i == 3) asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen offset:3072 sc1" : "=&v"(l3) : "v"(l_off), "s"(part_rs), "s"(part_at) : "memory");
        if (i >= 4 && i < 4 + Copy::NCH) qcopy.issue_at(qrows, q_row, Qs, c_at, i - 4, fetched, spare[pw]);
        if (i >= 4 + Copy::NCH && i < FETCH_OPS) gcopy.issue_at(grows, g_row, Gs, c_at, i - 4 - Copy::NCH, fetched, spare[pw]);
      };
      // (the partial dq of queries older than the tile's own keys is never asked for: the row may not exist)
      auto advance = [&]() {
        part_at = max(part_at - NSQ * D * 128, 0);
        c_at = c_at == (RING - 1) * QB ? 0 : c_at + QB;
        q_row -= TQ * (int)qrows.row_bytes;
        g_row -= TQ * (int)grows.row_bytes;
      };
      auto read_y = [&](const int at, const int j) { return tr8((yb[0] ^ (j << 6)) + at, (yb[1] ^ (j << 6)) + at); };
      el8 bf[DB];       // columns of the tile for the next contraction step, the next block's first one included
      // iteration 0 has no block yet
#pragma unroll
      for (int i = 0; i < FETCH_OPS; ++i) fetch(i, true, AHEAD < nsteps);
      advance();
#pragma unroll
      for (int j = 0; j < DB; ++j) bf[j] = read_y(y_at, j);
      lds_barrier();
      // TAIL: the item's last iterations, which have nothing left to copy, dq to finish, nothing to request in the end.
      auto iteration = [&](auto tail_tag, const int w) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tail_tag)::value;
        asm volatile("" : "+v"(xb[0]), "+v"(xb[1]), "+v"(yb[0]), "+v"(yb[1]), "+v"(zb));   // (the XORs stay in the loop)
        const int b = w - 1;
        const bool finished = TAIL && b >= nsteps - DIAG;       // the queries of this tile's own keys: nothing is missing any more
        if (finished) {    // key blocks behind these queries stay out of their dq, finite or not (later steps have older queries)
          const int newest = (t_last - b) * NSQ + dsq - (BKV / 32) * kt;
#pragma unroll
          for (int kb = 1; kb < BKV / 32; ++kb)
            if (kb > newest) kt_f[2 * kb] = kt_f[2 * kb + 1] = zero8();
        }
        const int y_next = y_at == y0 + (RING - 1) * QB ? y0 : y_at + QB;
        el8 zf[ZH], af[2];
        auto read_x = [&](int ks, int kb2) { return tr8((xb[0] ^ (kb2 << 6)) + x_at + 32 * ks * BKV, (xb[1] ^ (kb2 << 6)) + x_at + 32 * ks * BKV); };
        auto read_z = [&](int ks) { return lds_row8_at((zb ^ (ks << 5)) + z_at); };
        af[0] = read_x(0, 0);
        af[1] = read_x(0, 1);
#pragma unroll
        for (int ks = 0; ks < ZH; ++ks) zf[ks] = read_z(ks);
        // product number i of dk / dv: contraction step i / (2 DB), column block, 32-key block; the fragment a column block
        // is done with gives way to the next step's (the columns of the next block's tile have landed long ago)
        auto product = [&](const int i) __attribute__((always_inline)) {
          const int ks = i / (2 * DB), j = (i / 2) % DB, kb2 = i & 1;
          acc[kb2][j] = mfma32(bf[j], af[kb2], acc[kb2][j]);
          if (kb2 == 1) bf[j] = ks + 1 < KQ ? read_y(y_at + 32 * (ks + 1) * D, j) : read_y(y_next, j);
          if (j == DB - 1 && ks + 1 < KQ) af[kb2] = read_x(ks + 1, kb2);
          __builtin_amdgcn_sched_barrier(0);
        };
        // the partial dq requested an iteration ago has arrived (and everything requested or stored before it is done)
        asm volatile("s_waitcnt vmcnt(%4)" : "+v"(l0), "+v"(l1), "+v"(l2), "+v"(l3) : "n"(LOADS_PER_TILE) : "memory");
        f32x16 dq = {l0[0], l0[1], l0[2], l0[3], l1[0], l1[1], l1[2], l1[3], l2[0], l2[1], l2[2], l2[3], l3[0], l3[1], l3[2], l3[3]};
#pragma unroll
        for (int ks = 0; ks < KZ; ++ks) {
          dq = mfma32(kt_f[ks], zf[ks % ZH], dq);
          if (ks + ZH < KZ) zf[ks % ZH] = read_z(ks + ZH);
          if (ks & 1) product(ks >> 1);
        }
        if (finished) {
          int at = lane16;      // (opaque: its offsets are not to be kept through the steps before)
          asm volatile("" : "+v"(at));
          const int n = (at >> 4) & 31, h = at >> 9;
          const int row = (t_last - b) * TQ + 32 * dsq + n;
          const Rows out = rows_of(a.dq, cur);
#pragma unroll
          for (int j = 0; j < 16; ++j) dq[j] *= a.inv_temp;      // (in place: it is not needed unscaled, and there is no register to spare)
          store_block32_rows(dq, 1.0f, out, row * (int)out.row_bytes, row < doc_len && has_dq, 32 * dcol, h, a.out_f32);
        }
#pragma unroll
        for (int i = 0; i < (REST > OPS ? REST : OPS); ++i) {
          if (i < 4) store_part(i, dq, (ALL_DQ || has_dq) && !finished);
          else if (i < OPS) fetch(i - 4, !TAIL || w < nsteps, !TAIL || w + AHEAD < nsteps);
          if (i < REST) product(KZ / 2 + i);
        }
        advance();
        y_at = y_next;
        x_at = x_at + PB == x_end ? x0 : x_at + PB;
        z_at = 2 * place_of(Zs) + PB - z_at;
        // The tile copied an iteration ago (read behind this barrier) has landed, what came after it may be in flight.
        // An item's last request, of nothing, has to come back all the same before its registers are used for something
        // else.
        if (!TAIL || w < nsteps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + LOADS_PER_TILE) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS_PER_TILE) : "memory");
        // (no wait for LDS: what was read of the staged blocks has been multiplied, the columns on their way stay where
        // they are)
        asm volatile("s_barrier" ::: "memory");
      };
      int w = 1;
      const int plain = nsteps - (AHEAD > DIAG ? AHEAD : DIAG);
#pragma unroll 1
      for (; w < plain; ++w) iteration(No{}, w);
#pragma unroll 1
      for (; w <= nsteps; ++w) iteration(Yes{}, w);
      // (behind the barrier of the last iteration every product wave is done with the staged blocks and the last tiles)
      const bool more = read_box(m & 1, nxt);
      const Item done = cur;
      const ChainArgs a = fresh_args<ChainArgs>();
      if (more) {
        cur = nxt;
        open_item(a, cur);
      }
      const Rows out = rows_of(mat ? a.dk : a.dv, done);
      int at = lane16;
      asm volatile("" : "+v"(at));
      const int n = (at >> 4) & 31, h = at >> 9;
#pragma unroll
      for (int kb2 = 0; kb2 < 2; ++kb2) {
        const int row = done.kt * BKV + 64 * half + 32 * kb2 + n;
#pragma unroll
        for (int j = 0; j < DB; ++j) {
          store_block32_rows(acc[kb2][j], mat ? a.inv_temp : 1.0f, out, row * (int)out.row_bytes, row < done.doc_len, 32 * j, h, a.out_f32);
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[kb2][j][e] = 0.0f;
        }
      }
      if (!more) break;
    }
  }
}

template __global__ void bwd_chain_kernel<128, 128, false, 1, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<128, 128, true, 1, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<128, 128, false, 1, true>(const ChainArgs);
template __global__ void bwd_chain_kernel<128, 128, true, 1, true>(const ChainArgs);
template __global__ void bwd_chain_kernel<128, 96, false, 1, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<128, 96, true, 1, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<128, 96, false, 1, true>(const ChainArgs);
template __global__ void bwd_chain_kernel<128, 96, true, 1, true>(const ChainArgs);

template __global__ void bwd_chain_kernel<64, 64, false, 1, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<64, 64, true, 1, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<64, 64, false, 2, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<64, 64, true, 2, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<64, 32, false, 1, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<64, 32, true, 1, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<64, 32, false, 2, false>(const ChainArgs);
template __global__ void bwd_chain_kernel<64, 32, true, 2, false>(const ChainArgs);

template <int D, int U, int NSQ, bool STREAM = false>
static hipError_t launch_chain_d(const ChainArgs& a, bool ac, int n_q_max, int workgroups, hipStream_t s) {
  hipLaunchKernelGGL((chain_prep_kernel<D>), dim3((unsigned)n_q_max * (unsigned)a.heads), dim3(NT), 0, s, a);
  const dim3 grid(workgroups), block((4 * NSQ + 4) * 64);
  if (ac) hipLaunchKernelGGL((bwd_chain_kernel<D, U, true, NSQ, STREAM>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((bwd_chain_kernel<D, U, false, NSQ, STREAM>), grid, block, 0, s, a);
  return hipGetLastError();
}

hipError_t launch_bwd_chain(const ChainArgs& a, bool ac, bool wide, bool stream, int n_q_max, int workgroups, hipStream_t s) {
  if (a.head_dim <= 32) return wide ? launch_chain_d<64, 32, 2>(a, ac, n_q_max, workgroups, s) : launch_chain_d<64, 32, 1>(a, ac, n_q_max, workgroups, s);
  if (a.head_dim <= 64) return wide ? launch_chain_d<64, 64, 2>(a, ac, n_q_max, workgroups, s) : launch_chain_d<64, 64, 1>(a, ac, n_q_max, workgroups, s);
  if (used_width(a.head_dim) == 96) return stream ? launch_chain_d<128, 96, 1, true>(a, ac, n_q_max, workgroups, s) : launch_chain_d<128, 96, 1>(a, ac, n_q_max, workgroups, s);
  return stream ? launch_chain_d<128, 128, 1, true>(a, ac, n_q_max, workgroups, s) : launch_chain_d<128, 128, 1>(a, ac, n_q_max, workgroups, s);
}

}  // inline namespace SBA_ELEM_NS
}  // namespace sba
