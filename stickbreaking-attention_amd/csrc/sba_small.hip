// Kernels for problems that leave most of the chip idle.
//
// With few tiles a launch takes as long as one workgroup's walk along the other axis, a block of 32 at a time: 47 steps
// of 0.65 us for the forward of 1500 tokens, whatever the chip could do beside them.  Here a workgroup owns 32 rows
// instead of 128, and its four waves take four consecutive blocks of the other axis at a time.  (Eight waves: a single
// head of 4096 keys 30 us for 35, but a full chip is served worse, since the last round of every walk is the emptier:
// 16 x 2048 29 us for 26, 16 x 4 x 1024 38 for 28.)
#include <type_traits>

#include "sba_kernels.hpp"

namespace sba {
inline namespace SBA_ELEM_NS {

// One wave's copy of a 32 x D block into its own unpadded, swizzled tile; KEYS: rows permuted as by TileCopy<.., KEYS =
// true>.
template <int D, bool KEYS>
struct WaveCopy {
  static constexpr int C8 = D / 8, RPI = 64 / C8, NCH = 32 / RPI;
  static constexpr int KINDS = 16 / RPI;              // instructions apart by this many have their rows' swizzle in common
  int voff[KINDS];
  __device__ __forceinline__ void init(int lane, unsigned row_bytes, int used_bytes) {
#pragma unroll
    for (int k = 0; k < KINDS; ++k) {
      const int m = k * RPI + lane / C8, logical = (lane % C8) ^ swz<D>(m);
      voff[k] = 16 * logical < used_bytes ? ((KEYS ? kperm(m) : m) - row_delta(k)) * (int)row_bytes + 16 * logical : OUTSIDE;
    }
  }
  // source row of instruction j's first row
  static constexpr int row_delta(int j) {
    const int m = j * RPI;
    return KEYS ? ((m & 4) << 2) | ((m >> 3) << 2) | (m & 3) : m;    // (kperm)
  }
  __device__ __forceinline__ void issue(const Rows& r, int row0, unsigned short* tile) const {
#pragma unroll
    for (int j = 0; j < NCH; ++j)
      async_copy16(r.rsrc, tile + j * RPI * D, voff[j % KINDS], __builtin_amdgcn_readfirstlane((row0 + row_delta(j)) * (int)r.row_bytes));
  }
};

// One word for each lane, from byte offset voff of the buffer to LDS at dst + 4 * lane (see async_copy16).
__device__ __forceinline__ void async_words(__amdgpu_buffer_rsrc_t rsrc, const float* dst, int voff) {
  const unsigned lds_addr = __builtin_amdgcn_readfirstlane((unsigned)(size_t)dst);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds_addr), "v"(voff), "s"(rsrc) : "memory", "m0");
}

// Four consecutive columns of a lane's output row, from `col` on (see store_rows_axpy for the sum).
__device__ __forceinline__ void store_quad(f32x4 v, const Rows& out, const Rows& addend, int row, bool ok, int col, bool fuse, float factor, bool f32) {
  typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
  typedef __attribute__((ext_vector_type(4))) elem_t el4;
  if (fuse) {
    const u32x2 raw = __builtin_amdgcn_raw_buffer_load_b64(addend.rsrc, 2 * col < addend.used_bytes ? row * (int)addend.row_bytes + 2 * col : OUTSIDE, 0, 0);
    const el4 other = __builtin_bit_cast(el4, raw);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = fmaf(factor, (float)other[e], (float)(elem_t)v[e]);
  }
  ok = ok && 2 * col < out.used_bytes;
  const el2 a = cvt2(v[0], v[1]), b = cvt2(v[2], v[3]);
  if (f32) {
    const f32x4 r = {(float)a[0], (float)a[1], (float)b[0], (float)b[1]};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, r), out.rsrc, ok ? row * (int)out.row_bytes + 4 * col : OUTSIDE, 0, 0);
  } else {
    const u32x2 r = {__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b)};
    __builtin_amdgcn_raw_buffer_store_b64(r, out.rsrc, ok ? row * (int)out.row_bytes + 2 * col : OUTSIDE, 0, 0);
  }
}

// The waves' accumulators of one output, a quad of every lane at a time, into LDS; behind a barrier wave w adds up and
// stores quads w, w + W ..
template <int DB, int W>
__device__ __forceinline__ void add_waves(float* sums, const f32x16 (&acc)[DB], int w, int lane) {
#pragma unroll
  for (int q = 0; q < 4 * DB; ++q) {
    const f32x4 v = {acc[q >> 2][4 * (q & 3)], acc[q >> 2][4 * (q & 3) + 1], acc[q >> 2][4 * (q & 3) + 2], acc[q >> 2][4 * (q & 3) + 3]};
    *reinterpret_cast<f32x4*>(sums + ((q * W + w) * 64 + lane) * 4) = v;
  }
}
template <int W>
__device__ __forceinline__ f32x4 sum_quad(const float* sums, int q, int lane) {
  f32x4 v = *reinterpret_cast<const f32x4*>(sums + (q * W * 64 + lane) * 4);
#pragma unroll
  for (int k = 1; k < W; ++k) v += *reinterpret_cast<const f32x4*>(sums + ((q * W + k) * 64 + lane) * 4);
  return v;
}

template <int DB, int W>
__device__ __forceinline__ void store_sum(const float* sums, int w, int lane, float scale, const Rows& out, int row, bool ok, int h, bool f32) {
  for (int q = w; q < 4 * DB; q += W) store_quad(sum_quad<W>(sums, q, lane) * scale, out, out, row, ok, 32 * (q >> 2) + 8 * (q & 3) + 4 * h, false, 0.0f, f32);
}

// Forward.  32 query rows of one (document, head); in a round wave w has the w-th newest key block that is left.  What
// a block leaves of the stick (its product of 1 - beta) is known before its weights are, so the waves form odds and
// products side by side, exchange the products through LDS (one barrier a round) and go on to weights and p V each on
// its own.  The output is the sum over the waves.  K and V rows come to every wave's own piece of LDS, the next round's
// as soon as this one's are read.  What bounds it: the round's serial chain (products, odds, barrier, weights) while
// the chip is empty, 0.9 us a round of 128 keys against 0.54 us a step of 32 in fwd_kernel; then the additive time of
// matrix and vector instructions, with 16 waves per compute unit at head_dim 64, 8 at 128 and 4 at 256.  Measured (us,
// fwd_kernel first): head_dim 64, 4 heads of 512 tokens 14.4 / 9.7, of 2048 40 / 20; 16 heads of 1024 23.7 / 15.2;
// head_dim 128, 4 heads of 512 18.0 / 11.7, 16 heads of 2048 54 / 43; head_dim 256, 4 heads of 512 28 / 18, of 2048 87
// / 41.
template <int D, bool AC, int U>
__global__ void __launch_bounds__(SMALL_WAVES * 64, D <= 64 ? 4 : (D <= 128 ? 2 : 1)) fwd_small_kernel(const KArgs a) {
  constexpr int W = SMALL_WAVES, KS = U / 16, DB = U / 32, TILE = 32 * D;
  __shared__ __attribute__((aligned(16))) unsigned short smem[2 * W * TILE];   // per wave: K block, V block; then the waves' outputs
  __shared__ float left[2][W][32];              // by round parity: what a wave's block leaves of a query's stick
  static_assert(2 * W * TILE * 2 >= W * 64 * DB * 16 * 4, "the waves' accumulators fit the tiles' place");

  const int* sched = a.sched;
  const int part = blockIdx.x / a.heads;
  const int head = blockIdx.x - part * a.heads;
  const int slot = part / (BM / 32), sub = part % (BM / 32);
  const int4 hdr = *reinterpret_cast<const int4*>(sched);   // status, query tiles, key tiles, table entries needed
  const Tile t = reinterpret_cast<const Tile*>(sched + SCHED_HDR)[slot];
  asm volatile("" ::"s"(t.tok_start), "s"(t.doc_len), "s"(t.idx), "s"(t.batch));   // keep the tile read above the branch
  const int tid = threadIdx.x;
  const bool refused = hdr.x != 0 || (a.stick != nullptr && hdr.w > a.tab_stride);
  if (refused || slot >= hdr.y) {
    if (a.clear_spare && sub == 0) {
      int row0, row1;
      unsigned pair;
      spare_rows(refused, slot, hdr.y, sched[SCHED_TOTAL], a.tokens, a.nan_pair, row0, row1, pair);
      fill_rows16(a.o, head, row0, row1, a.head_dim << a.out_f32, pair, tid, W * 64);
      fill_rows16(a.rem, head, row0, row1, 1 << a.out_f32, pair, tid, W * 64);
    }
    return;
  }
  const int L = t.doc_len, qw0 = t.idx * BM + 32 * sub;
  if (qw0 >= L) return;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, blk = (lane >> 4) & 1;
  const int qrow = qw0 + n;
  const bool qvalid = qrow < L;
  const int64_t tok0 = t.tok_start;
  auto rows_of = [&](const View& v) {
    return make_rows(reinterpret_cast<const elem_t*>(v.ptr) + t.batch * v.sb + head * v.sh + tok0 * v.st, v.st, L, a.head_dim);
  };
  const Rows qrows = rows_of(a.q), krows = rows_of(a.k), vrows = rows_of(a.v);
  unsigned short* const Kt = smem + 2 * w * TILE;
  unsigned short* const Vt = Kt + TILE;
  WaveCopy<D, true> kcopy, vcopy;
  kcopy.init(lane, krows.row_bytes, krows.used_bytes);
  vcopy.init(lane, vrows.row_bytes, vrows.used_bytes);
  constexpr int LOADS = WaveCopy<D, true>::NCH;
  const int n_blocks = qw0 / 32 + 1, n_rounds = (n_blocks + W - 1) / W;
  auto block_of = [&](int r) { return n_blocks - 1 - (r * W + w); };   // (below zero: none left for this wave)
  // (a wave without a block copies rows outside the document: zeros, nothing is fetched)
  auto row_of = [&](int r) { const int b = block_of(r); return b >= 0 ? 32 * b : L; };
  kcopy.issue(krows, row_of(0), Kt);
  vcopy.issue(vrows, row_of(0), Vt);
  el8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = load_frag(qrows, qrow, 32 * ks + 16 * h);
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.0f;
  const int kbase = swz_off<D>(n, h);
  int vbase[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = 16 * blk + 4 * (i16 & 3);
    vbase[u] = swz_off<D>(8 * u + 4 * h + (i16 >> 2), c >> 3) + (c & 7);
  }
  // the document's table area: every round's store is issued, outside the area where there is nothing to write
  const bool table = a.stick != nullptr;
  float* const stick = table ? a.stick + (int64_t)head * a.tab_stride + t.tab_base : nullptr;
  const __amdgpu_buffer_rsrc_t stick_rs = __builtin_amdgcn_make_buffer_rsrc(stick, 0, table ? (unsigned)min((int64_t)0x7fffffff, 4 * (int64_t)tab_doc_entries(L)) : 0u, 0x00020000);
  float run = 1.0f;                             // stick left in front of this round's newest block
  wait_loads<0>();
#pragma unroll 1
  for (int r = 0; r < n_rounds; ++r) {
    const int b = block_of(r), k0 = 32 * b;
    // K of this round has landed; behind it only the table's store and V may be on their way
    wait_loads<LOADS + 1>();
    f32x16 x;
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = 0.0f;
    {
      el8 kfr[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kfr[ks] = lds_row8(Kt + (kbase ^ ((ks & 7) << 4)) + 128 * (ks >> 3));   // (the swizzle leaves the upper half of 512-byte rows where it is)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) x = mfma32(kfr[ks], qf[ks], x);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    kcopy.issue(krows, r + 1 < n_rounds ? row_of(r + 1) : L, Kt);
    const int lim = b >= 0 ? qrow - k0 - 16 * h + (AC ? 1 : 0) : 0;     // visible keys of this lane: i < lim (all of them but in the newest block)
    float e[16], inv[4];
    float total = stick_odds<true, false>(x, a.c, lim, e, inv);
    if (__builtin_amdgcn_ballot_w64(!(total > 0.0f)) != 0) total = stick_odds<true, true>(x, a.c, lim, e, inv);   // (see stick_weights_fwd)
    float lo, hi;
    both_halves(total, lo, hi);
    if (h == 0) left[r & 1][w][n] = lo * hi;
    lds_barrier();
    float carry = run;
#pragma unroll
    for (int k = 0; k < W; ++k) {
      if (k == w) carry = run;
      run *= left[r & 1][k][n];
    }
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, carry), stick_rs, b >= 0 && qvalid && h == 0 ? 4 * (tab_seg32(L, b) + qrow) : OUTSIDE, 0, 0);
    float s = h == 0 ? carry * hi : carry, p[16];      // (keys of the h = 1 lane are the newer ones)
#pragma unroll
    for (int g = 3; g >= 0; --g) {
      s *= inv[g];
      float left_of = s;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        p[4 * g + j] = left_of * e[4 * g + j];
        if (j < 3) left_of += p[4 * g + j];
      }
    }
    wait_loads<LOADS + 1>();                    // V of this round
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const el8 pf = pack8(p + 8 * tt);
      const unsigned short* const vrow = Vt + 16 * tt * D;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const unsigned short* const vcol = vrow + 128 * (db >> 2);
        o[db] = mfma32(lds_tr8(vcol + (vbase[0] ^ ((db & 3) << 5)), vcol + (vbase[1] ^ ((db & 3) << 5))), pf, o[db]);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    vcopy.issue(vrows, r + 1 < n_rounds ? row_of(r + 1) : L, Vt);
  }
  if (w == 0 && h == 0 && qvalid) {
    elem_t* const at = reinterpret_cast<elem_t*>(a.rem.ptr) + t.batch * a.rem.sb + head * a.rem.sh + (tok0 + qrow) * a.rem.st;
    if (a.out_f32) *reinterpret_cast<float*>(at) = (float)(elem_t)run;
    else *at = (elem_t)run;
    if (table) stick[(unsigned)(tab_rowplane32(L) + qrow)] = run;
  }
  wait_loads<0>();                              // (copies of nothing into the place that is written now)
  lds_barrier();
  float* const sums = reinterpret_cast<float*>(smem);
  add_waves<DB, W>(sums, o, w, lane);
  lds_barrier();
  const Rows orows = rows_of(a.o);
  for (int q = w; q < 4 * DB; q += W)
    store_quad(sum_quad<W>(sums, q, lane), orows, vrows, qrow, qvalid, 32 * (q >> 2) + 8 * (q & 3) + 4 * h, a.fuse, run, a.out_f32);
}

// -------------------------------------------------------------------------------------------
// Backward, in two passes of the same kind.  The first owns 32 queries, four waves walk the keys from the oldest on, a
// block each at a time; they exchange every block's sum of p (do.v) and with it each knows the running sum D in front
// of its block (see sba_chain.hip), which goes into the gradient table.  With the table the second, which owns 32 keys,
// needs no order at all: its waves take the query blocks that can see them in turn.  Sums over the waves at the end.
// What bounds them: up to 8 waves per compute unit (head_dim 64; 4 at 128) each a round's chain of its own: two
// products, odds and weights, the barrier, the gradient of the logits, one or two products more: 1.1 us a round.  That
// is no shorter than a step of bwd_chain_kernel, but a round is 128 keys, and nothing is handed from one workgroup to
// the next.  Measured (us, one-pass form first): head_dim 64, 4 heads of 512 tokens 36.2 / 11.3 + 12.2, of 2048 89 / 25
// + 26; 16 heads of 1024 55 / 17 + 21; 2 x 8 of 1500 78 / 23 + 33; head_dim 128, 4 heads of 512 42 / 15 + 16.  Eight
// waves a workgroup gain where 4 heads are all there is (2048 tokens: 51 to 43) and lose from 16 heads on (1024 tokens:
// 37 to 45); two lose everywhere else (2 x 8 of 1500: 57 to 75).
// -------------------------------------------------------------------------------------------
template <int D, bool AC, int U>
__global__ void __launch_bounds__(SMALL_WAVES * 64, D <= 64 ? 2 : 1) bwd_dq_small_kernel(const KArgs a) {
  constexpr int W = SMALL_WAVES, KS = U / 16, DB = U / 32, TILE = 32 * D;
  __shared__ __attribute__((aligned(16))) unsigned short smem[3 * W * TILE];   // per wave: two K blocks, a V block; then the waves' dq
  __shared__ float tot[2][W][32];               // by round parity: a block's sum of p (do.v) per query
  static_assert(3 * W * TILE * 2 >= W * 64 * DB * 16 * 4, "the waves' accumulators fit the tiles' place");

  const int* sched = a.sched;
  const int part = blockIdx.x / a.heads;
  const int head = blockIdx.x - part * a.heads;
  const int slot = part / (BM / 32), sub = part % (BM / 32);
  const int4 hdr = *reinterpret_cast<const int4*>(sched);   // status, query tiles, key tiles, table entries needed
  const int longest = sched[SCHED_MAXLEN];
  const Tile t = reinterpret_cast<const Tile*>(sched + SCHED_HDR)[slot];
  asm volatile("" ::"s"(t.tok_start), "s"(t.doc_len), "s"(t.idx), "s"(t.batch), "s"(t.tab_base));   // keep the tile read above the branch
  const int tid = threadIdx.x;
  const bool refused = hdr.x != 0 || hdr.w > a.tab_stride || longest > a.max_doc_len;
  if (refused || slot >= hdr.y) {
    if (a.clear_spare && sub == 0) {            // for the second pass as well, which has no slots to spare
      int row0, row1;
      unsigned pair;
      spare_rows(refused, slot, hdr.y, sched[SCHED_TOTAL], a.tokens, a.nan_pair, row0, row1, pair);
      fill_rows16(a.dq, head, row0, row1, a.head_dim << a.out_f32, pair, tid, W * 64);
      fill_rows16(a.dk, head, row0, row1, a.head_dim << a.out_f32, pair, tid, W * 64);
      fill_rows16(a.dv, head, row0, row1, a.head_dim << a.out_f32, pair, tid, W * 64);
    }
    return;
  }
  const int L = t.doc_len, qw0 = t.idx * BM + 32 * sub;
  if (qw0 >= L) return;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, blk = (lane >> 4) & 1;
  const int qrow = qw0 + n;
  const bool qvalid = qrow < L;
  const int64_t tok0 = t.tok_start;
  auto rows_of = [&](const View& v) {
    return make_rows(reinterpret_cast<const elem_t*>(v.ptr) + t.batch * v.sb + head * v.sh + tok0 * v.st, v.st, L, a.head_dim);
  };
  const Rows qrows = rows_of(a.q), grows = rows_of(a.go), krows = rows_of(a.k), vrows = rows_of(a.v);
  unsigned short* const Kt = smem + 3 * w * TILE;       // (two of them)
  unsigned short* const Vt = Kt + 2 * TILE;
  WaveCopy<D, true> kcopy, vcopy;
  kcopy.init(lane, krows.row_bytes, krows.used_bytes);
  vcopy.init(lane, vrows.row_bytes, vrows.used_bytes);
  const int n_blocks = qw0 / 32 + 1, n_rounds = (n_blocks + W - 1) / W;
  auto block_of = [&](int r) { return r * W + w; };
  auto row_of = [&](int r) { return block_of(r) < n_blocks ? 32 * block_of(r) : L; };   // (outside the document: zeros, nothing is fetched)
  kcopy.issue(krows, row_of(0), Kt);
  vcopy.issue(vrows, row_of(0), Vt);
  el8 qf[KS], gf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qf[ks] = load_frag(qrows, qrow, 32 * ks + 16 * h);
    gf[ks] = load_frag(grows, qrow, 32 * ks + 16 * h);
  }
  float* const stick = a.stick + (int64_t)head * a.tab_stride + t.tab_base;
  float* const gtab = a.gtab + (int64_t)head * a.tab_stride + t.tab_base;
  const unsigned area = 4u * (unsigned)tab_doc_entries(L);
  const __amdgpu_buffer_rsrc_t stick_rs = __builtin_amdgcn_make_buffer_rsrc(stick, 0, area, 0x00020000);
  const __amdgpu_buffer_rsrc_t gtab_rs = __builtin_amdgcn_make_buffer_rsrc(gtab, 0, area, 0x00020000);
  auto entry = [&](int r) { const int b = block_of(r); return b < n_blocks && qvalid ? 4 * (tab_seg32(L, b) + qrow) : OUTSIDE; };
  float e_next = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(stick_rs, entry(0), 0, 0));
  // D in front of the oldest key: the complete gradient of rem, times rem
  float run;
  {
    float dr = 0.0f;
    if (a.grem.ptr != nullptr && qvalid)
      dr = (float)(reinterpret_cast<const elem_t*>(a.grem.ptr) + t.batch * a.grem.sb + head * a.grem.sh + tok0 * a.grem.st)[(int64_t)qrow * a.grem.st];
    if (a.fuse) {                               // d(rem) = do . v_row as well (see bwd_dq_kernel)
      float dot = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const el8 vown = load_frag(vrows, qrow, 32 * ks + 16 * h);
#pragma unroll
        for (int e = 0; e < 8; ++e) dot = fmaf((float)gf[ks][e], (float)vown[e], dot);
      }
      float lo, hi;
      both_halves(dot, lo, hi);
      dr += lo + hi;
    }
    run = qvalid ? dr * stick[(unsigned)(tab_rowplane32(L) + qrow)] : 0.0f;
  }
  f32x16 dq[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[db][i] = 0.0f;
  const int kbase = swz_off<D>(n, h);
  int tbase[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = 16 * blk + 4 * (i16 & 3);
    tbase[u] = swz_off<D>(8 * u + 4 * h + (i16 >> 2), c >> 3) + (c & 7);
  }
  wait_loads<0>();
#pragma unroll 1
  for (int r = 0; r < n_rounds; ++r) {
    const int b = block_of(r), k0 = 32 * b;
    wait_loads<1>();                            // K, V and the stick of this round; the table's store may be on its way
    const float e_in = b < n_blocks && qvalid ? e_next : 1.0f;
    const unsigned short* const Kr = Kt + (r & 1) * TILE;
    e_next = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(stick_rs, r + 1 < n_rounds ? entry(r + 1) : OUTSIDE, 0, 0));
    kcopy.issue(krows, r + 1 < n_rounds ? row_of(r + 1) : L, Kt + ((r + 1) & 1) * TILE);
    f32x16 x, da;
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = da[i] = 0.0f;
    {
      el8 kfr[KS], vfr[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) { kfr[ks] = lds_row8(Kr + (kbase ^ (ks << 4))); vfr[ks] = lds_row8(Vt + (kbase ^ (ks << 4))); }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) { x = mfma32(kfr[ks], qf[ks], x); da = mfma32(vfr[ks], gf[ks], da); }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    vcopy.issue(vrows, r + 1 < n_rounds ? row_of(r + 1) : L, Vt);
    float p[16], m[16], ends[2], c = e_in;      // m: 1 - beta
    stick_weights<AC, true, true, true>(x, a.c, b < n_blocks ? k0 : L + 32, qrow, h, c, p, m, ends);   // (no block: all keys masked)
    float t0 = 0.0f, t1 = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; j += 2) { t0 = fmaf(p[j], da[j], t0); t1 = fmaf(p[j + 1], da[j + 1], t1); }
    float lo, hi;
    both_halves(t0 + t1, lo, hi);
    if (h == 0) tot[r & 1][w][n] = lo + hi;
    lds_barrier();
    float before = run;
#pragma unroll
    for (int k = 0; k < W; ++k) {
      if (k == w) before = run;
      run += tot[r & 1][k][n];
    }
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, before), gtab_rs, h == 0 ? entry(r) : OUTSIDE, 0, 0);
    float dprev = h == 1 ? before + lo : before, dz[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) { const float dj = fmaf(p[j], da[j], dprev); dz[j] = fmaf(m[j], dj, -dprev); dprev = dj; }
    if (b < n_blocks) {
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const el8 zf = pack8(dz + 8 * tt);
        const unsigned short* const krow = Kr + 16 * tt * D;
#pragma unroll
        for (int db = 0; db < DB; ++db) dq[db] = mfma32(lds_tr8(krow + (tbase[0] ^ (db << 5)), krow + (tbase[1] ^ (db << 5))), zf, dq[db]);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  wait_loads<0>();                              // (copies of nothing into the place that is written now)
  lds_barrier();
  add_waves<DB, W>(reinterpret_cast<float*>(smem), dq, w, lane);
  lds_barrier();
  store_sum<DB, W>(reinterpret_cast<const float*>(smem), w, lane, a.inv_temp, rows_of(a.dq), qrow, qvalid, h, a.out_f32);
}

template <int D, bool AC, int U>
__global__ void __launch_bounds__(SMALL_WAVES * 64, D <= 64 ? 2 : 1) bwd_dkdv_small_kernel(const KArgs a) {
  constexpr int W = SMALL_WAVES, KS = U / 16, DB = U / 32, TILE = 32 * D, OWN = 4 * TILE + 32 * 32;
  __shared__ __attribute__((aligned(16))) unsigned short smem[W * OWN];   // per wave: two Q and two dO blocks, p or dz; then the waves' dk and dv
  static_assert(W * OWN * 2 >= 2 * W * 64 * DB * 16 * 4, "the waves' accumulators fit the tiles' place");

  const int* sched = a.sched;
  const int part = blockIdx.x / a.heads;
  const int head = blockIdx.x - part * a.heads;
  const int slot = part / (BM / 32), sub = part % (BM / 32);
  const int4 hdr = *reinterpret_cast<const int4*>(sched);   // status, query tiles, key tiles, table entries needed
  const int longest = sched[SCHED_MAXLEN];
  const Tile t = reinterpret_cast<const Tile*>(sched + SCHED_HDR)[slot];     // (the key blocks of a query tile's own rows)
  asm volatile("" ::"s"(t.tok_start), "s"(t.doc_len), "s"(t.idx), "s"(t.batch), "s"(t.tab_base));   // keep the tile read above the branch
  if (hdr.x != 0 || hdr.w > a.tab_stride || longest > a.max_doc_len || slot >= hdr.y) return;
  const int L = t.doc_len, k0 = t.idx * BM + 32 * sub, kb = k0 / 32;
  if (k0 >= L) return;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, blk = (lane >> 4) & 1;
  const int64_t tok0 = t.tok_start;
  auto rows_of = [&](const View& v) {
    return make_rows(reinterpret_cast<const elem_t*>(v.ptr) + t.batch * v.sb + head * v.sh + tok0 * v.st, v.st, L, a.head_dim);
  };
  const Rows qrows = rows_of(a.q), grows = rows_of(a.go), krows = rows_of(a.k), vrows = rows_of(a.v);
  unsigned short* const Qt = smem + w * OWN;            // (two of them)
  unsigned short* const Gt = Qt + 2 * TILE;
  unsigned short* const Bt = Gt + 2 * TILE;
  WaveCopy<D, false> qcopy, gcopy;
  qcopy.init(lane, qrows.row_bytes, qrows.used_bytes);
  gcopy.init(lane, grows.row_bytes, grows.used_bytes);
  const int n_blocks = (L + 31) / 32 - kb;              // query blocks that see these keys
  auto row_of = [&](int i) { return i < n_blocks ? k0 + 32 * i : L; };   // (outside the document: zeros, nothing is fetched)
  const unsigned area = 4u * (unsigned)tab_doc_entries(L);
  float* const stick = a.stick + (int64_t)head * a.tab_stride + t.tab_base;
  const __amdgpu_buffer_rsrc_t stick_rs = __builtin_amdgcn_make_buffer_rsrc(stick, 0, area, 0x00020000);
  const __amdgpu_buffer_rsrc_t gtab_rs = __builtin_amdgcn_make_buffer_rsrc(a.gtab + (int64_t)head * a.tab_stride + t.tab_base, 0, area, 0x00020000);
  auto entry = [&](int i) { const int row = k0 + 32 * i + n; return i < n_blocks && row < L ? 4 * (tab_seg32(L, kb) + row) : OUTSIDE; };
  float e_next = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(stick_rs, entry(w), 0, 0));
  float d_next = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(gtab_rs, entry(w), 0, 0));
  qcopy.issue(qrows, row_of(w), Qt);
  gcopy.issue(grows, row_of(w), Gt);
  el8 kf[KS], vf[KS];                           // MFMA row n holds key k0 + kperm(n)
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    kf[ks] = load_frag(krows, k0 + kperm(n), 32 * ks + 16 * h);
    vf[ks] = load_frag(vrows, k0 + kperm(n), 32 * ks + 16 * h);
  }
  float rem_own = 0.0f;                         // fused output: rem_j * do_j reaches dv_j through the diagonal of p (see bwd_dkdv_kernel)
  if (a.fuse && k0 + n < L) rem_own = stick[(unsigned)(tab_rowplane32(L) + k0 + n)];
  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[db][i] = dv[db][i] = 0.0f;
  const int qbase = swz_off<D>(n, h);
  // the private block has rows of 64 bytes, its chunks rotated with row / 4 (see bwd_dkdv_tail_kernel)
  auto blk_off = [](int row, int chunk) { return row * 32 + ((chunk ^ ((row >> 2) & 3)) << 3); };
  int xoff[2], ybase[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int row = 8 * h + 4 * u + (i16 >> 2), c = 16 * blk + 4 * (i16 & 3);
    xoff[u] = blk_off(row, c >> 3) + (c & 7);
    ybase[u] = swz_off<D>(row, c >> 3) + (c & 7);
  }
  wait_loads<0>();
#pragma unroll 1
  for (int i = w, buf = 0; i < n_blocks; i += W, buf ^= 1) {
    wait_loads<0>();
    const int qw0 = k0 + 32 * i, qrow = qw0 + n;
    const bool ok = qrow < L;
    float e_in = ok ? e_next : 1.0f;
    const float before = ok ? d_next : 0.0f;
    e_next = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(stick_rs, entry(i + W), 0, 0));
    d_next = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(gtab_rs, entry(i + W), 0, 0));
    qcopy.issue(qrows, row_of(i + W), Qt + (buf ^ 1) * TILE);
    gcopy.issue(grows, row_of(i + W), Gt + (buf ^ 1) * TILE);
    const unsigned short* const Qr = Qt + buf * TILE;
    const unsigned short* const Gr = Gt + buf * TILE;
    f32x16 x, da;
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = da[j] = 0.0f;
    {
      el8 qfr[KS], gfr[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) { qfr[ks] = lds_row8(Qr + (qbase ^ (ks << 4))); gfr[ks] = lds_row8(Gr + (qbase ^ (ks << 4))); }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) { x = mfma32(kf[ks], qfr[ks], x); da = mfma32(vf[ks], gfr[ks], da); }
    }
    float p[16], m[16], ends[2];
    if (i > 0) stick_weights<AC, true, false, true>(x, a.c, k0, qrow, h, e_in, p, m, ends);
    else stick_weights<AC, true, true, true>(x, a.c, k0, qrow, h, e_in, p, m, ends);
    float t0 = 0.0f, t1 = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; j += 2) { t0 = fmaf(p[j], da[j], t0); t1 = fmaf(p[j + 1], da[j + 1], t1); }
    float lo, hi;
    both_halves(t0 + t1, lo, hi);
    float dprev = h == 1 ? before + lo : before, dz[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) { const float dj = fmaf(p[j], da[j], dprev); dz[j] = fmaf(m[j], dj, -dprev); dprev = dj; }
    if (a.fuse && i == 0) {
#pragma unroll
      for (int j = 0; j < 16; ++j) p[j] += 16 * h + j == n ? rem_own : 0.0f;
    }
    // turn the blocks around, p first: [query][key] rows in, key-major operands out
    auto turn = [&](const float (&v)[16], el8 (&f)[2]) {
#pragma unroll
      for (int c = 0; c < 2; ++c) *reinterpret_cast<el8*>(Bt + blk_off(n, 2 * h + c)) = pack8(v + 8 * c);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) f[ks] = lds_tr8(Bt + xoff[0] + 16 * ks * 32, Bt + xoff[1] + 16 * ks * 32);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    el8 pf[2], zf[2];
    turn(p, pf);
    turn(dz, zf);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        dv[db] = mfma32(lds_tr8(Gr + (ybase[0] ^ (db << 5)) + 16 * ks * D, Gr + (ybase[1] ^ (db << 5)) + 16 * ks * D), pf[ks], dv[db]);
        dk[db] = mfma32(lds_tr8(Qr + (ybase[0] ^ (db << 5)) + 16 * ks * D, Qr + (ybase[1] ^ (db << 5)) + 16 * ks * D), zf[ks], dk[db]);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  wait_loads<0>();                              // (copies of nothing into the place that is written now)
  lds_barrier();
  float* const sums = reinterpret_cast<float*>(smem);
  constexpr int HALF = W * 64 * DB * 16;
  add_waves<DB, W>(sums, dk, w, lane);
  add_waves<DB, W>(sums + HALF, dv, w, lane);
  lds_barrier();
  store_sum<DB, W>(sums, w, lane, a.inv_temp, rows_of(a.dk), k0 + n, k0 + n < L, h, a.out_f32);
  store_sum<DB, W>(sums + HALF, w, lane, 1.0f, rows_of(a.dv), k0 + n, k0 + n < L, h, a.out_f32);
}

// -------------------------------------------------------------------------------------------
// Backward of documents of at most 32 x SHORT_BLOCKS tokens, both passes in one: a team of waves takes one (document,
// head), half as many waves as it has blocks of 32 tokens, and a workgroup has one team of four, two of two or four of
// one.  K and V go to LDS; every wave walks the keys of its own queries, oldest first, for dq, and leaves the running
// sum D of every block of 32 x 32 in LDS.  Then Q and dO, which the waves hold as their own operands, take the place of
// K and V, and the waves own keys.  Query block i takes i + 1 steps, key block i of n takes n - i: with blocks w and n
// - 1 - w a wave has n + 1 in either half.  What bounds it: the two passes it stands in for ran at the rate of a copy,
// four operands read by each and the sums D written and read between them; here operands come in once (32 heads x 16 K
// tokens in documents of 16 .. 256: 228 us for 161, of which 94 are its traffic).  What is left is that a workgroup
// loads, computes and stores one after the other, two of them (8 waves of 239 registers, 80 KB of LDS) per compute
// unit, one above head_dim 64: loads and stores alone take 115 us, and neither workgroups that start late nor an order
// that mixes long and short documents overlaps them better.  So nothing is read from memory behind the first barrier: a
// load there is waited for behind the stores of dq, in order, and the sticks one step ahead were later than a step.
// Sticks come to LDS with K and V, K and V rows of both key blocks are kept from there; the document's place is made
// scalar, which takes a loop over lanes away from every access, and operands are read four steps ahead of their
// multiplication.  On one GPU, us: these documents at head_dim 64 175 -> 164, at 32 104 -> 95; 32 heads of 128 x 256
// tokens 342 -> 320, of 128 x 33 46.3 -> 44.3; at head_dim 128 16 heads of 128 x 64 76 -> 68.  Streaming stores (nt)
// cost a third: they leave in quarters of a line.  One document to a workgroup whatever its length: 204 us, most waves
// idle; four slots of the tile list to a workgroup, long documents one after the other: 166 us, and 104 for 31 us where
// there are few of them.
// -------------------------------------------------------------------------------------------
template <int D, bool AC, int U>
__global__ void __launch_bounds__(SMALL_WAVES * 64, D <= 64 ? 2 : 1) bwd_short_kernel(const KArgs a) {
  constexpr int W = SMALL_WAVES, KS = U / 16, DB = U / 32, TILE = 32 * D, NB = SHORT_BLOCKS, AHEAD = KS < 4 ? KS : 4;
  static_assert(NB == 2 * W && W == 4, "two blocks for each wave");
  __shared__ __attribute__((aligned(16))) unsigned short smem[2 * NB * TILE + W * 32 * 32];   // K, V blocks, Q, dO blocks in their place; p or dz of a wave
  __shared__ float sums[NB * (NB + 1) / 2 * 32];                  // D in front of key block b, from its own queries on
  __shared__ float newer[W * (NB - 1) * 32];                      // per wave: stick left in front of its key blocks, for the queries of later blocks

  const int* sched = a.sched;
  const int part = blockIdx.x / a.heads;
  const int head = blockIdx.x - part * a.heads;
  const int4 hdr = *reinterpret_cast<const int4*>(sched);   // status, query tiles, key tiles, table entries needed
  const int total = sched[SCHED_TOTAL], longest = sched[SCHED_MAXLEN], over_64 = sched[SCHED_OVER_64], over_128 = sched[SCHED_OVER_128];
  const int tid = threadIdx.x;
  const bool refused = hdr.x != 0 || hdr.w > a.tab_stride || longest > a.max_doc_len;
  if (a.clear_spare && (refused || total < a.tokens)) {     // every workgroup clears its share
    const int from = refused ? 0 : total, share = (a.tokens - from + (int)gridDim.x / a.heads - 1) / ((int)gridDim.x / a.heads);
    const int row0 = min(from + part * share, a.tokens), row1 = min(row0 + share, a.tokens);
    const unsigned pair = refused ? a.nan_pair : 0u;
    fill_rows16(a.dq, head, row0, row1, a.head_dim << a.out_f32, pair, tid, W * 64);
    fill_rows16(a.dk, head, row0, row1, a.head_dim << a.out_f32, pair, tid, W * 64);
    fill_rows16(a.dv, head, row0, row1, a.head_dim << a.out_f32, pair, tid, W * 64);
  }
  if (refused) return;                          // (beyond here no document has more than NB blocks: see launch_bwd_short)
  // The documents are ranked, longest first: one for a workgroup, then two, then four.
  const int pairs = (over_64 - over_128 + 1) / 2;
  const int team_waves = part < over_128 ? W : (part - over_128 < pairs ? W / 2 : W / 4), teams = W / team_waves;
  const int doc0 = part < over_128 ? part : (part - over_128 < pairs ? over_128 + 2 * (part - over_128) : over_64 + 4 * (part - over_128 - pairs));
  const int doc_end = min(doc0 + teams, part < over_128 ? over_128 : (part - over_128 < pairs ? over_64 : a.n_docs));
  if (doc0 >= doc_end) return;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int team = w / team_waves, tw = w - team * team_waves;
  const int lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, blk = (lane >> 4) & 1;
  unsigned short* const At = smem + 2 * team * team_waves * TILE;
  unsigned short* const Bt = At + NB * TILE;
  unsigned short* const own = smem + 2 * NB * TILE + w * 32 * 32;
  float* const own_left = reinterpret_cast<float*>(own);          // during dq: stick left in front of the key blocks, for the wave's queries (turn 1 from 4 * 32 on)
  float* const newer_left = newer + w * (NB - 1) * 32;
  float* const team_sums = sums + team * (NB * (NB + 1) / 2 * 32) / teams;
  auto sum_at = [&](int b, int q) { return 64 * team_waves * b - 16 * b * (b + 1) + q; };   // (a block's row begins at its own queries)
  const int rowbase = swz_off<D>(n, h);
  int xoff[2], ybase[2], tbase[2];
  auto blk_off = [](int row, int chunk) { return row * 32 + ((chunk ^ ((row >> 2) & 3)) << 3); };   // (see bwd_dkdv_tail_kernel)
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = 16 * blk + 4 * (i16 & 3), row = 8 * h + 4 * u + (i16 >> 2);
    tbase[u] = swz_off<D>(8 * u + 4 * h + (i16 >> 2), c >> 3) + (c & 7);
    xoff[u] = blk_off(row, c >> 3) + (c & 7);
    ybase[u] = swz_off<D>(row, c >> 3) + (c & 7);
  }

  const int doc = min(doc0 + team, doc_end - 1);
  int4 about = reinterpret_cast<const int4*>(sched + a.docs_off)[doc];   // first token, length, first table entry
  about.x = __builtin_amdgcn_readfirstlane(about.x);
  about.y = __builtin_amdgcn_readfirstlane(about.y);
  about.z = __builtin_amdgcn_readfirstlane(about.z);
  const int L = doc0 + team < doc_end ? about.y : 0, n_blocks = (L + 31) / 32, batch = a.clear_spare ? 0 : doc;   // (fixed length: by batch entry)
  const int64_t tok0 = about.x;
  auto rows_of = [&](const View& v) {
    return make_rows(reinterpret_cast<const elem_t*>(v.ptr) + batch * v.sb + head * v.sh + tok0 * v.st, v.st, L, a.head_dim);
  };
  const Rows krows = rows_of(a.k), vrows = rows_of(a.v);
  // a wave's blocks (none: -1)
  const int block_of[2] = {tw < n_blocks ? tw : -1, n_blocks - 1 - tw >= team_waves ? n_blocks - 1 - tw : -1};
  {
    WaveCopy<D, true> kcopy, vcopy;
    kcopy.init(lane, krows.row_bytes, krows.used_bytes);
    vcopy.init(lane, vrows.row_bytes, vrows.used_bytes);
#pragma unroll
    for (int turn = 0; turn < 2; ++turn) {
      const int b = block_of[turn];
      if (b < 0) break;
      kcopy.issue(krows, 32 * b, At + b * TILE);
      vcopy.issue(vrows, 32 * b, Bt + b * TILE);
    }
  }
  el8 qf[2][KS], gf[2][KS];
  {
    const Rows qrows = rows_of(a.q), grows = rows_of(a.go);
#pragma unroll
    for (int turn = 0; turn < 2; ++turn)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int row = block_of[turn] >= 0 ? 32 * block_of[turn] + n : L;   // (outside the document: zeros)
        qf[turn][ks] = load_frag(qrows, row, 32 * ks + 16 * h);
        gf[turn][ks] = load_frag(grows, row, 32 * ks + 16 * h);
      }
  }
  // Everything else that is read from memory is asked for here as well: a load further down would be waited for behind
  // the stores of dq.
  const float* const stick = a.stick + (int64_t)head * a.tab_stride + about.z;
  const __amdgpu_buffer_rsrc_t stick_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(stick), 0, 4u * (unsigned)tab_doc_entries(L), 0x00020000);
  // byte offset of the stick left in front of key block b for row `row`
  auto stick_off = [&](int b, int row, bool ok) { return ok && row < L ? 4 * (tab_seg32(L, b) + row) : OUTSIDE; };
#pragma unroll
  for (int turn = 0; turn < 2; ++turn)
#pragma unroll
    for (int i = 0; i < W * (turn + 1); i += 2)         // two key blocks an instruction
      if (i <= block_of[turn]) async_words(stick_rs, own_left + 32 * (W * turn + i), stick_off(i + h, 32 * block_of[turn] + n, i + h <= block_of[turn]));
  const int later[2] = {block_of[0] >= 0 ? n_blocks - 1 - block_of[0] : 0, block_of[1] >= 0 ? n_blocks - 1 - block_of[1] : 0};   // (at most NB - 1 together)
#pragma unroll
  for (int i = 0; i < NB - 1; i += 2)
    if (i < later[0] + later[1] && (i < NB - 2 || h == 0)) {
      const int at = i + h, turn = at < later[0] ? 0 : 1;
      const int kb = turn == 0 ? block_of[0] : block_of[1], b = kb + 1 + (turn == 0 ? at : at - later[0]);
      async_words(stick_rs, newer_left + 32 * i, stick_off(kb, 32 * b + n, at < later[0] + later[1]));
    }
  float newest_left[2], rem[2], run0[2];      // stick left in front of the wave's own blocks on the diagonal; of its rows, at last; D in front of the oldest key (see bwd_dq_small_kernel)
#pragma unroll
  for (int turn = 0; turn < 2; ++turn) {
    const int qrow = block_of[turn] >= 0 ? 32 * block_of[turn] + n : L;
    const auto word = [&](int off) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(stick_rs, off, 0, 0)); };
    newest_left[turn] = word(stick_off(block_of[turn], qrow, true));
    rem[turn] = word(qrow < L ? 4 * (tab_rowplane32(L) + qrow) : OUTSIDE);
    run0[turn] = 0.0f;
    if (a.grem.ptr != nullptr && qrow < L)
      run0[turn] = (float)(reinterpret_cast<const elem_t*>(a.grem.ptr) + batch * a.grem.sb + head * a.grem.sh + tok0 * a.grem.st)[(int64_t)qrow * a.grem.st];
  }
  if (a.fuse) {
#pragma unroll
    for (int turn = 0; turn < 2; ++turn) {
      float dot = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const el8 vown = load_frag(vrows, block_of[turn] >= 0 ? 32 * block_of[turn] + n : L, 32 * ks + 16 * h);
#pragma unroll
        for (int e = 0; e < 8; ++e) dot = fmaf((float)gf[turn][ks][e], (float)vown[e], dot);
      }
      float lo, hi;
      both_halves(dot, lo, hi);
      run0[turn] += lo + hi;
    }
  }
#pragma unroll
  for (int turn = 0; turn < 2; ++turn) run0[turn] *= rem[turn];
  wait_loads<0>();
  lds_barrier();

  // ---- dq ----
#pragma unroll
  for (int turn = 0; turn < 2; ++turn) {
    const int qb = block_of[turn];
    if (qb >= 0) {
      const int qrow = 32 * qb + n;
      const bool qvalid = qrow < L;
      float run = run0[turn];
      f32x16 dq[DB];
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) dq[db][i] = 0.0f;
#pragma unroll 1
      for (int b = 0; b <= qb; ++b) {
        const unsigned short* const Kr = At + b * TILE;
        const unsigned short* const Vr = Bt + b * TILE;
        float c = own_left[32 * (W * turn + b) + n];
        if (!qvalid) c = 1.0f;
        if (h == 0) team_sums[sum_at(b, qrow)] = run;
        f32x16 x, da;
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = da[i] = 0.0f;
        el8 kr[AHEAD], vr[AHEAD];
#pragma unroll
        for (int ks = 0; ks < AHEAD; ++ks) { kr[ks] = lds_row8(Kr + (rowbase ^ (ks << 4))); vr[ks] = lds_row8(Vr + (rowbase ^ (ks << 4))); }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          x = mfma32(kr[ks % AHEAD], qf[turn][ks], x);
          da = mfma32(vr[ks % AHEAD], gf[turn][ks], da);
          if (ks + AHEAD < KS) { kr[ks % AHEAD] = lds_row8(Kr + (rowbase ^ ((ks + AHEAD) << 4))); vr[ks % AHEAD] = lds_row8(Vr + (rowbase ^ ((ks + AHEAD) << 4))); }
          __builtin_amdgcn_sched_barrier(0);
        }
        float p[16], m[16], ends[2];
        grad_weights<AC, true>(x, a.c, 32 * b, 32 * qb, qrow, h, c, p, m, ends);
        el8 zf[2];
        grad_dz<true>(p, m, da, ends, h, run, 0.0f, zf);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int db = 0; db < DB; ++db)
            dq[db] = mfma32(lds_tr8(Kr + 16 * tt * D + (tbase[0] ^ (db << 5)), Kr + 16 * tt * D + (tbase[1] ^ (db << 5))), zf[tt], dq[db]);
      }
      store_rows(dq, a.inv_temp, rows_of(a.dq), qrow, L, h, a.out_f32);
    }
  }

  // ---- dk, dv ----
  el8 kf[KS], vf[KS], kf1[KS], vf1[KS];       // MFMA row n holds key 32 b + kperm(n)
  {
    const int at = max(block_of[0], 0) * TILE, at1 = max(block_of[1], 0) * TILE;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kf[ks] = lds_row8(At + at + (rowbase ^ (ks << 4)));
      vf[ks] = lds_row8(Bt + at + (rowbase ^ (ks << 4)));
      kf1[ks] = lds_row8(At + at1 + (rowbase ^ (ks << 4)));
      vf1[ks] = lds_row8(Bt + at1 + (rowbase ^ (ks << 4)));
    }
  }
  lds_barrier();                              // K and V have been read
#pragma unroll
  for (int turn = 0; turn < 2; ++turn)
    if (block_of[turn] >= 0) {
      const int at = block_of[turn] * TILE;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        *reinterpret_cast<el8*>(At + at + (rowbase ^ (ks << 4))) = qf[turn][ks];
        *reinterpret_cast<el8*>(Bt + at + (rowbase ^ (ks << 4))) = gf[turn][ks];
      }
    }
  lds_barrier();
#pragma unroll 1
  for (int turn = 0; turn < 2; ++turn) {
    const int kb = turn == 0 ? block_of[0] : block_of[1];
    if (kb < 0) break;
    const int k0 = 32 * kb;
    const float rem_own = turn == 0 ? rem[0] : rem[1];   // fused output: rem_j * do_j reaches dv_j through the diagonal of p (see bwd_dkdv_kernel)
    const float newest = turn == 0 ? newest_left[0] : newest_left[1];
    const float* const left = newer_left + (turn == 0 ? 0 : 32 * later[0]) + n;
    f32x16 dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) dk[db][i] = dv[db][i] = 0.0f;
#pragma unroll 1
    for (int b = kb; b < n_blocks; ++b) {
      const int qrow = 32 * b + n;
      const bool ok = qrow < L;
      const float c = !ok ? 1.0f : b == kb ? newest : left[32 * max(b - kb - 1, 0)];
      float before = ok ? team_sums[sum_at(kb, qrow)] : 0.0f;
      const unsigned short* const Qr = At + b * TILE;
      const unsigned short* const Gr = Bt + b * TILE;
      f32x16 x, da;
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = da[i] = 0.0f;
      el8 qr[AHEAD], gr[AHEAD];
#pragma unroll
      for (int ks = 0; ks < AHEAD; ++ks) { qr[ks] = lds_row8(Qr + (rowbase ^ (ks << 4))); gr[ks] = lds_row8(Gr + (rowbase ^ (ks << 4))); }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        x = mfma32(kf[ks], qr[ks % AHEAD], x);
        da = mfma32(vf[ks], gr[ks % AHEAD], da);
        if (ks + AHEAD < KS) { qr[ks % AHEAD] = lds_row8(Qr + (rowbase ^ ((ks + AHEAD) << 4))); gr[ks % AHEAD] = lds_row8(Gr + (rowbase ^ ((ks + AHEAD) << 4))); }
        __builtin_amdgcn_sched_barrier(0);
      }
      float p[16], m[16], ends[2], carry = c;
      grad_weights<AC, true>(x, a.c, k0, 32 * b, qrow, h, carry, p, m, ends);
      el8 pz[2], f[2];
      grad_dz<true>(p, m, da, ends, h, before, 0.0f, pz);
      // turn the blocks around, dz first: [query][key] rows in, key-major operands out
      auto turned = [&] {
#pragma unroll
        for (int k = 0; k < 2; ++k) *reinterpret_cast<el8*>(own + blk_off(n, 2 * h + k)) = pz[k];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) f[ks] = lds_tr8(own + xoff[0] + 16 * ks * 32, own + xoff[1] + 16 * ks * 32);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      };
      turned();
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int db = 0; db < DB; ++db)
          dk[db] = mfma32(lds_tr8(Qr + (ybase[0] ^ (db << 5)) + 16 * ks * D, Qr + (ybase[1] ^ (db << 5)) + 16 * ks * D), f[ks], dk[db]);
      if (a.fuse && b == kb) {
#pragma unroll
        for (int j = 0; j < 16; ++j) p[j] += 16 * h + j == n ? rem_own : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) pz[k] = pack8(p + 8 * k);
      turned();
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int db = 0; db < DB; ++db)
          dv[db] = mfma32(lds_tr8(Gr + (ybase[0] ^ (db << 5)) + 16 * ks * D, Gr + (ybase[1] ^ (db << 5)) + 16 * ks * D), f[ks], dv[db]);
    }
    if (turn == 0 && block_of[1] >= 0) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) { kf[ks] = kf1[ks]; vf[ks] = vf1[ks]; }
    }
    store_rows(dk, a.inv_temp, rows_of(a.dk), k0 + n, L, h, a.out_f32);
    store_rows(dv, 1.0f, rows_of(a.dv), k0 + n, L, h, a.out_f32);
  }
}

#define SBA_SMALL(D, U)                                                   \
  template __global__ void fwd_small_kernel<D, false, U>(const KArgs);    \
  template __global__ void fwd_small_kernel<D, true, U>(const KArgs);     \
  template __global__ void bwd_dq_small_kernel<D, false, U>(const KArgs);    \
  template __global__ void bwd_dq_small_kernel<D, true, U>(const KArgs);     \
  template __global__ void bwd_dkdv_small_kernel<D, false, U>(const KArgs);  \
  template __global__ void bwd_dkdv_small_kernel<D, true, U>(const KArgs);   \
  template __global__ void bwd_short_kernel<D, false, U>(const KArgs);       \
  template __global__ void bwd_short_kernel<D, true, U>(const KArgs);
SBA_SMALL(64, 32)
SBA_SMALL(64, 64)
SBA_SMALL(128, 96)
SBA_SMALL(128, 128)
#undef SBA_SMALL
template __global__ void fwd_small_kernel<256, false, 192>(const KArgs);
template __global__ void fwd_small_kernel<256, true, 192>(const KArgs);
template __global__ void fwd_small_kernel<256, false, 256>(const KArgs);
template __global__ void fwd_small_kernel<256, true, 256>(const KArgs);

enum class SmallPass { FWD, DQ, DKDV };
template <SmallPass PASS, int D, int U>
static void launch_small_d(const KArgs& a, bool ac, int n_q_max, hipStream_t s) {
  const dim3 grid((unsigned)small_workgroups(n_q_max) * (unsigned)a.heads), block(SMALL_WAVES * 64);
  auto launch = [&](void (*plain)(KArgs), void (*current)(KArgs)) { hipLaunchKernelGGL(ac ? current : plain, grid, block, 0, s, a); };
  if constexpr (PASS == SmallPass::FWD) launch(fwd_small_kernel<D, false, U>, fwd_small_kernel<D, true, U>);
  else if constexpr (PASS == SmallPass::DQ) launch(bwd_dq_small_kernel<D, false, U>, bwd_dq_small_kernel<D, true, U>);
  else launch(bwd_dkdv_small_kernel<D, false, U>, bwd_dkdv_small_kernel<D, true, U>);
}
template <SmallPass PASS>
static hipError_t launch_small(const KArgs& a, bool ac, int n_q_max, hipStream_t s) {
  if (a.head_dim <= 32) launch_small_d<PASS, 64, 32>(a, ac, n_q_max, s);
  else if (a.head_dim <= 64) launch_small_d<PASS, 64, 64>(a, ac, n_q_max, s);
  else if (used_width(a.head_dim) == 96) launch_small_d<PASS, 128, 96>(a, ac, n_q_max, s);
  else if (a.head_dim <= 128) launch_small_d<PASS, 128, 128>(a, ac, n_q_max, s);
  else if constexpr (PASS == SmallPass::FWD) {
    if (used_width(a.head_dim) == 192) launch_small_d<PASS, 256, 192>(a, ac, n_q_max, s);
    else launch_small_d<PASS, 256, 256>(a, ac, n_q_max, s);
  } else return hipErrorInvalidValue;             // (the backward's two have no kernel of that width)
  return hipGetLastError();
}
hipError_t launch_fwd_small(const KArgs& a, bool ac, int n_q_max, hipStream_t s) { return launch_small<SmallPass::FWD>(a, ac, n_q_max, s); }
hipError_t launch_bwd_dq_small(const KArgs& a, bool ac, int n_q_max, hipStream_t s) { return launch_small<SmallPass::DQ>(a, ac, n_q_max, s); }
hipError_t launch_bwd_dkdv_small(const KArgs& a, bool ac, int n_q_max, hipStream_t s) { return launch_small<SmallPass::DKDV>(a, ac, n_q_max, s); }

hipError_t launch_bwd_short(const KArgs& a, bool ac, int parts, hipStream_t s) {
  if (a.head_dim > 128 || a.max_doc_len > 32 * SHORT_BLOCKS) return hipErrorInvalidValue;   // (longer ones than declared are refused on the device)
  const dim3 grid((unsigned)parts * (unsigned)a.heads), block(SMALL_WAVES * 64);
  auto launch = [&](void (*plain)(KArgs), void (*current)(KArgs)) { hipLaunchKernelGGL(ac ? current : plain, grid, block, 0, s, a); };
  if (a.head_dim <= 32) launch(bwd_short_kernel<64, false, 32>, bwd_short_kernel<64, true, 32>);
  else if (a.head_dim <= 64) launch(bwd_short_kernel<64, false, 64>, bwd_short_kernel<64, true, 64>);
  else if (used_width(a.head_dim) == 96) launch(bwd_short_kernel<128, false, 96>, bwd_short_kernel<128, true, 96>);
  else launch(bwd_short_kernel<128, false, 128>, bwd_short_kernel<128, true, 128>);
  return hipGetLastError();
}

}  // inline namespace SBA_ELEM_NS
}  // namespace sba
