// The two passes of the backward at head_dim 129 .. 256 (see sba_bwd.hip for the two-pass backward and its other
// kernels): the dk / dv pass, described here, and the dq pass, further down.
//
// At twice the width of the eight-wave kernel of sba_bwd.hip a wave's K and V fragments are 128 registers and the
// accumulators of 64 keys of one output 256: neither role fits two waves per SIMD.  So the work is cut smaller.  A
// workgroup owns 64 keys of one (document, head) and walks the queries that can see them, 32 per step:
//
//   waves 0, 1   "weights", one 32-key block each, K fragments in registers: scores, p, dz
//   waves 2, 3   "do.v" of the same blocks, V fragments in registers; handed to the weights wave through LDS in fp32
//   waves 4 .. 7 "products": dv = p^T dO and dk = dz^T Q, 64 keys x half of the columns of one output each (128 registers);
//                they also copy the Q / dO tiles
//
// A step has two phases with a barrier behind each.  In the first the weights waves have vector work only (p of block i) and
// the product waves, which share SIMDs 0 and 1 with them, multiply block i - 1; in the second the weights waves form the
// scores of block i + 1 between the vector instructions of dz, the do.v waves theirs, and the product waves read the Q / dO
// fragments of block i.  A tile is requested two steps before it is read (four slots of 32 KiB).
//
// Bound by the vector work of the two weights waves, alone with it on their SIMDs (of 2400 cycles of a step, stamped,
// they wait 350, the product waves 650, the do.v waves 1300), and by what a work item costs beside its steps (8000
// cycles, 45 steps on average); the matrix pipes are busy for a third of the time.  16 heads x 16 K tokens in eight
// documents, head_dim 256: 1525 -> 890 us against four independent waves of 32 keys each, which formed the scores
// twice, once for dv and once for dk, because both outputs' accumulators (256 registers) left the chains nowhere to go.
// Tried: a quarter or half of a block's products in the second phase (942, 970 for 922), the next tile requested ahead
// of the products (950).
#include <type_traits>

#include "sba_kernels.hpp"

namespace sba {
inline namespace SBA_ELEM_NS {

template <bool AC, bool PROD, int U>
__global__ void __launch_bounds__(512, 1) bwd_dkdv_wide_kernel(const KArgs a) {
  constexpr int D = 256, KS = U / 16, DBH = U / 64;     // U: columns multiplied; DBH: 32-wide column blocks of a product wave
  constexpr int TQ = 32, SLOTS = 4, QTILE = TQ * D, PTILE = TQ * WIDE_KEYS;
  __shared__ __attribute__((aligned(16))) unsigned short Qs[SLOTS * QTILE];
  __shared__ __attribute__((aligned(16))) unsigned short Gs[SLOTS * QTILE];
  __shared__ __attribute__((aligned(16))) unsigned short Ps[2 * PTILE];   // p and dz, [query][key]
  __shared__ __attribute__((aligned(16))) unsigned short Zs[2 * PTILE];
  __shared__ __attribute__((aligned(16))) float hand[WIDE_KEYS / 32][16 * 64];   // do.v of a block as the accumulators lie, a quad of every lane at a time

  // (the grid never exceeds the room of the list: its tile is read along with the header)
  const int* sched = a.sched;
  const int which = blockIdx.x / a.heads;
  const int head = blockIdx.x - which * a.heads;
  const int4 hdr = *reinterpret_cast<const int4*>(sched);   // status, query tiles, key tiles, table entries needed
  const int longest = sched[SCHED_MAXLEN];
  const Tile t = reinterpret_cast<const Tile*>(sched + a.kv_list_off)[which >> 1];
  asm volatile("" ::"s"(t.tok_start), "s"(t.doc_len), "s"(t.idx), "s"(t.batch), "s"(t.tab_base));   // keep the tile read above the branch
  if (hdr.x != 0 || hdr.w > a.tab_stride || longest > a.max_doc_len || (which >> 1) >= hdr.z) return;
  const int L = t.doc_len;
  const int q_first = t.idx * BKV + (which & 1) * WIDE_KEYS;       // first key, and first query that can see one
  if (q_first >= L) return;
  const int nsteps = (L - q_first + TQ - 1) / TQ;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, blk = (lane >> 4) & 1;
  const int64_t tok0 = t.tok_start;
  auto rows_of = [&](const View& v) {
    return make_rows(reinterpret_cast<const elem_t*>(v.ptr) + t.batch * v.sb + head * v.sh + tok0 * v.st, v.st, L, a.head_dim);
  };

  if (w < 4) {
    __builtin_amdgcn_s_setprio(3);
    const int kb = w & 1;
    const bool weights = w < 2;
    const int k0 = q_first + 32 * kb;
    float* const mine = &hand[kb][4 * lane];
    int roff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) roff[ks] = swz_off<D>(n, 2 * ks + h);
    el8 fr[KS];                               // K or V; MFMA row n holds key k0 + kperm(n)
    auto take_fragments = [&]() {
      const unsigned short* const T = (weights ? Qs : Gs) + 2 * QTILE;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) fr[ks] = lds_row8(T + swz_off<D>(32 * kb + kperm(n), 2 * ks + h));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    // one chain of a 32 x 32 block: rows of the tile in slot `T` against this wave's keys, operand reads LEAD ahead
    constexpr int LEAD = 4;
    el8 op[LEAD];
    auto chain_begin = [&](const unsigned short* T) {
#pragma unroll
      for (int k = 0; k < LEAD; ++k) op[k] = lds_row8(T + roff[k]);
    };
    auto chain_step = [&](const unsigned short* T, f32x16& x, int k) {
      x = mfma32(fr[k], op[k % LEAD], x);
      if (k + LEAD < KS) op[k % LEAD] = lds_row8(T + roff[k + LEAD]);
    };
    auto clear = [](f32x16& x) {
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = 0.0f;
    };
    lds_barrier();                            // the K and V rows and tiles 0 and 1 have landed
    take_fragments();
    lds_barrier();                            // their places are free
    using std::integral_constant;
    if (weights) {
      // a block that starts past the document's end is never visible; its table reads stay inside the document's area
      const int tblock = min(k0, L - 1) / 32;
      const int64_t tab_row0 = (int64_t)head * a.tab_stride + t.tab_base;
      const int64_t tab = tab_row0 + tab_seg32(L, tblock), tab_rowval = tab_row0 + tab_rowplane32(L);
      // fused output: rem_j * do_j reaches dv_j through the diagonal of p (see bwd_dkdv_kernel)
      float rem_own = 0.0f;
      if (a.fuse && k0 + n < L) rem_own = a.stick[tab_rowval + k0 + n];
      // carries of a step, requested three steps ahead; rows past the document's end take its last row's (see
      // bwd_dkdv_kernel)
      const unsigned run_bytes = (unsigned)L * 4u;
      const __amdgpu_buffer_rsrc_t stick_rs = __builtin_amdgcn_make_buffer_rsrc(a.stick + tab, 0, run_bytes, 0x00020000);
      const __amdgpu_buffer_rsrc_t gtab_rs = __builtin_amdgcn_make_buffer_rsrc(a.gtab + tab, 0, run_bytes, 0x00020000);
      const __amdgpu_buffer_rsrc_t drem_rs = __builtin_amdgcn_make_buffer_rsrc(a.gtab + tab_rowval, 0, run_bytes, 0x00020000);
      const int row4 = 4 * (q_first + n), last4 = 4 * (L - 1);
      struct Raw { float e, g, d; };
      Raw r0, r1, r2, r3;
      auto request = [&](int step, Raw& r) {
        const int off = min(row4 + step * (4 * TQ), last4);
        r.e = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(stick_rs, off, 0, 0));
        r.g = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(gtab_rs, off, 0, 0));
        r.d = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(drem_rs, off, 0, 0));
      };
      request(0, r0);
      request(1, r1);
      request(2, r2);
      f32x16 x;
      clear(x);
      chain_begin(Qs);
#pragma unroll
      for (int k = 0; k < KS; ++k) chain_step(Qs, x, k);
      // Step i.  SLOT: i mod 4, the tile's slot.  BAND: one of the first two steps, whose queries may not see all keys.
      auto step = [&](auto band_tag, auto slot_tag, const int i, Raw& set, Raw& ahead) __attribute__((always_inline)) {
        constexpr bool BAND = decltype(band_tag)::value;
        constexpr int SLOT = decltype(slot_tag)::value;
        unsigned short* const Pt = Ps + (SLOT & 1) * PTILE;
        unsigned short* const Zt = Zs + (SLOT & 1) * PTILE;
        const unsigned short* const Tn = Qs + ((SLOT + 1) % SLOTS) * QTILE;
        const float carry_e = set.e, carry_c = set.g, dr = set.d;
        request(i + 3, ahead);
        const int qw0 = q_first + i * TQ, qrow = qw0 + n;
        const bool hidden = BAND && sub_skip<AC>(k0, qw0);     // (the table holds nothing for such a block)
        float p[16], r[16], ends[2] = {0.0f, 0.0f};
        {
          float e = carry_e;
          stick_weights<AC, PROD, BAND, true>(x, a.c, k0, qrow, h, e, p, r, ends);
        }
        auto put = [&](unsigned short* T, const float* v, int c) {
          *reinterpret_cast<el8*>(T + swz_off<WIDE_KEYS>(n, 4 * kb + 2 * h + c)) = hidden ? zero8() : pack8(v + 8 * c);
        };
        if (BAND && a.fuse && qw0 == k0) {
          float pd[16];
#pragma unroll
          for (int j = 0; j < 16; ++j) pd[j] = p[j] + (16 * h + j == n ? rem_own : 0.0f);
          put(Pt, pd, 0);
          put(Pt, pd, 1);
        } else {
          put(Pt, p, 0);
          put(Pt, p, 1);
        }
        lds_barrier();
        f32x16 da;
        {
          f32x4 q4[4];
#pragma unroll
          for (int g = 0; g < 4; ++g) q4[g] = *reinterpret_cast<const f32x4*>(mine + 256 * g);
#pragma unroll
          for (int j = 0; j < 16; ++j) da[j] = q4[j >> 2][j & 3];
        }
        chain_begin(Tn);
        __builtin_amdgcn_sched_barrier(0);
        clear(x);
        float dz[16];
        if constexpr (PROD) {                 // grad_dz with the next block's chain between its instructions
          constexpr int A0 = KS / 4;
#pragma unroll
          for (int k = 0; k < A0; ++k) chain_step(Tn, x, k);
          __builtin_amdgcn_sched_barrier(0);
          float t0 = 0.0f, t1 = 0.0f;
#pragma unroll
          for (int j = 0; j < 16; j += 2) { t0 = fmaf(p[j], da[j], t0); t1 = fmaf(p[j + 1], da[j + 1], t1); }
          float lo, hi;
          both_halves(fmaf(-dr, ends[0] - ends[1], t0 + t1), lo, hi);
          float dprev = fmaf(dr, ends[1], h == 1 ? carry_c + lo : carry_c);
          __builtin_amdgcn_sched_barrier(0);
          constexpr int REST = KS - A0;
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const float dj = fmaf(p[j], da[j], dprev);
            dz[j] = fmaf(r[j], dj, -dprev);
            dprev = dj;
#pragma unroll
            for (int k = j * REST / 16; k < (j + 1) * REST / 16; ++k) chain_step(Tn, x, A0 + k);
            __builtin_amdgcn_sched_barrier(0);
          }
          put(Zt, dz, 0);
          put(Zt, dz, 1);
        } else {
#pragma unroll
          for (int k = 0; k < KS; ++k) chain_step(Tn, x, k);
          el8 zf[2];
          float c = carry_c;
          grad_dz<PROD>(p, r, da, ends, h, c, dr, zf);
#pragma unroll
          for (int c2 = 0; c2 < 2; ++c2)
            *reinterpret_cast<el8*>(Zt + swz_off<WIDE_KEYS>(n, 4 * kb + 2 * h + c2)) = hidden ? zero8() : zf[c2];
        }
        lds_barrier();
      };
      using Yes = std::true_type;
      using No = std::false_type;
      step(Yes{}, integral_constant<int, 0>{}, 0, r0, r3);
      if (nsteps > 1) step(Yes{}, integral_constant<int, 1>{}, 1, r1, r0);
#pragma unroll 1
      for (int i = 2;; i += 4) {
        if (i >= nsteps) break;
        step(No{}, integral_constant<int, 2>{}, i, r2, r1);
        if (i + 1 >= nsteps) break;
        step(No{}, integral_constant<int, 3>{}, i + 1, r3, r2);
        if (i + 2 >= nsteps) break;
        step(No{}, integral_constant<int, 0>{}, i + 2, r0, r3);
        if (i + 3 >= nsteps) break;
        step(No{}, integral_constant<int, 1>{}, i + 3, r1, r0);
      }
    } else {
      f32x16 da;
      clear(da);
      chain_begin(Gs);
#pragma unroll
      for (int k = 0; k < KS; ++k) chain_step(Gs, da, k);
      auto step = [&](auto slot_tag) __attribute__((always_inline)) {
        const unsigned short* const Tn = Gs + ((decltype(slot_tag)::value + 1) % SLOTS) * QTILE;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 q4 = {da[4 * g], da[4 * g + 1], da[4 * g + 2], da[4 * g + 3]};
          *reinterpret_cast<f32x4*>(mine + 256 * g) = q4;
        }
        lds_barrier();
        clear(da);
        chain_begin(Tn);
#pragma unroll
        for (int k = 0; k < KS; ++k) chain_step(Tn, da, k);
        lds_barrier();
      };
#pragma unroll 1
      for (int i = 0;; i += 4) {
        step(integral_constant<int, 0>{});
        if (i + 1 >= nsteps) break;
        step(integral_constant<int, 1>{});
        if (i + 2 >= nsteps) break;
        step(integral_constant<int, 2>{});
        if (i + 3 >= nsteps) break;
        step(integral_constant<int, 3>{});
        if (i + 4 >= nsteps) break;
      }
    }
  } else {
    __builtin_amdgcn_s_setprio(0);
    const int pw = w - 4, ptid = pw * 64 + lane;
    const int mat = pw >> 1, half = pw & 1;       // (dv | dk), half of the columns
    const Rows qrows = rows_of(a.q), grows = rows_of(a.go);
    using Copy = TileCopy<D, TQ, 256, false>;
    constexpr int LOADS_PER_TILE = 2 * Copy::NCH;
    Copy qcopy, gcopy;
    qcopy.init(ptid, qrows.row_bytes, qrows.used_bytes);
    gcopy.init(ptid, grows.row_bytes, grows.used_bytes);
    auto fetch = [&](int step) {
      qcopy.issue(qrows, q_first + step * TQ, Qs + (step % SLOTS) * QTILE);
      gcopy.issue(grows, q_first + step * TQ, Gs + (step % SLOTS) * QTILE);
    };
    fetch(0);
    {   // the 64 K and V rows wait in the places of tiles 2 and 3
      const Rows krows = rows_of(a.k), vrows = rows_of(a.v);
      TileCopy<D, WIDE_KEYS, 256, false> kcopy, vcopy;
      kcopy.init(ptid, krows.row_bytes, krows.used_bytes);
      vcopy.init(ptid, vrows.row_bytes, vrows.used_bytes);
      kcopy.issue(krows, q_first, Qs + 2 * QTILE);
      vcopy.issue(vrows, q_first, Gs + 2 * QTILE);
    }
    if (nsteps > 1) fetch(1);
    f32x16 acc[2][DBH];
#pragma unroll
    for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
      for (int j = 0; j < DBH; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[kb2][j][e] = 0.0f;
    // transpose reads of rows 8 h + 4 u + i16 / 4 (+ 16 ks): staged block, tile
    int xoff[2][2], yoff[2][DBH];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = 8 * h + 4 * u + (i16 >> 2);
#pragma unroll
      for (int kb2 = 0; kb2 < 2; ++kb2) {
        const int xc = 32 * kb2 + 16 * blk + 4 * (i16 & 3);
        xoff[u][kb2] = swz_off<WIDE_KEYS>(r, xc >> 3) + (xc & 7);
      }
#pragma unroll
      for (int j = 0; j < DBH; ++j) {
        const int yc = 32 * (half * DBH + j) + 16 * blk + 4 * (i16 & 3);
        yoff[u][j] = swz_off<D>(r, yc >> 3) + (yc & 7);
      }
    }
    el8 bf[2][DBH];
    auto read_y = [&](int b) {
      const unsigned short* Yt = (mat ? Qs : Gs) + (b % SLOTS) * QTILE;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int j = 0; j < DBH; ++j) bf[ks][j] = lds_tr8(Yt + yoff[0][j] + 16 * ks * D, Yt + yoff[1][j] + 16 * ks * D);
    };
    // (the queries of block 0 see none of the newer 32 keys: those rows stay out of its products, finite or not)
    auto products = [&](int b) __attribute__((always_inline)) {
      const unsigned short* Xt = (mat ? Zs : Ps) + (b & 1) * PTILE;
      el8 af[2][2];
#pragma unroll
      for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) af[kb2][ks] = lds_tr8(Xt + xoff[0][kb2] + 16 * ks * WIDE_KEYS, Xt + xoff[1][kb2] + 16 * ks * WIDE_KEYS);
      auto half_of = [&](int kb2) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int j = 0; j < DBH; ++j) acc[kb2][j] = mfma32(bf[ks][j], af[kb2][ks], acc[kb2][j]);
      };
      half_of(0);
      if (b > 0) half_of(1);
    };
    // Behind the products of step i - 1: tile i + 1, which the others read behind the barrier, has landed; the
    // fragments of tile i; tile i + 3 is requested (into the slot of tile i - 1; here and not ahead of the products,
    // which the weights waves wait for).
    auto turn = [&](int i) __attribute__((always_inline)) {
      if (i + 2 < nsteps) wait_loads<LOADS_PER_TILE>();
      else wait_loads<0>();
      lds_barrier();
      read_y(i);
      if (i + 3 < nsteps) fetch(i + 3);
      lds_barrier();
    };
    wait_loads<0>();
    lds_barrier();
    lds_barrier();
    if (2 < nsteps) fetch(2);
    turn(0);
#pragma unroll 1
    for (int i = 1; i < nsteps; ++i) {
      products(i - 1);
      turn(i);
    }
    products(nsteps - 1);
    const Rows out = rows_of(mat ? a.dk : a.dv);
#pragma unroll
    for (int kb2 = 0; kb2 < 2; ++kb2) {
      const int row = q_first + 32 * kb2 + n;
#pragma unroll
      for (int j = 0; j < DBH; ++j)
        store_block32_rows(acc[kb2][j], mat ? a.inv_temp : 1.0f, out, row * (int)out.row_bytes, row < L, 32 * (half * DBH + j), h, a.out_f32);
    }
  }
}

// -------------------------------------------------------------------------------------------
// dq pass of the same head dims: 128 queries of one (document, head) per workgroup, the keys walked from the oldest to
// the diagonal, 32 per step.  Q and dO fragments of 32 queries and their dq are 256 registers, so two waves of a SIMD
// share a block of 32 queries:
//
//   waves 0 .. 3  "scores": Q fragments; p, dz, the running sum and the gradient table waves 4 .. 7  "sums": dO
//   fragments and dq; do.v of a block, handed to the scores wave through LDS in fp32, and dq += dz K of the
//                 block before, whose dz comes back the same way; they also copy the K / V tiles
//
// A step has two phases with a barrier behind each: weights of block i next to the products of block i - 1, then dz of
// block i between the scores of block i + 1 next to its do.v.  A tile is requested two steps before it is read (four
// slots of 32 KiB).  Bound by the two phases, 3300 cycles of a step: vector work of one wave, then 32 matrix
// instructions of two.  16 heads x 16 K tokens in eight documents, head_dim 256: 795 -> 620 us against one wave per
// SIMD with 512 registers for everything.  Reading operands six or eight instead of four products ahead changes
// nothing.
// -------------------------------------------------------------------------------------------
template <bool AC, bool PROD, int U, bool GIVE>
__global__ void __launch_bounds__(512, 1) bwd_dq_wide_kernel(const KArgs a) {
  constexpr int D = 256, KS = U / 16, DB = U / 32;
  constexpr int BF = 32, SLOTS = 4, TILE = BF * D;
  static_assert(SLOTS * BF == BM, "the query rows wait in the ring first");
  __shared__ __attribute__((aligned(16))) unsigned short Ks[SLOTS * TILE];
  __shared__ __attribute__((aligned(16))) unsigned short Vs[SLOTS * TILE];
  // per block of queries: do.v of a key block as the accumulators lie, a quad of every lane at a time, and dz as
  // operand fragments
  constexpr int HAND_Z = 16 * 64, HAND = HAND_Z + 2 * 64 * 4;
  __shared__ __attribute__((aligned(16))) float hand[4 * HAND];
  __shared__ float drs[4][32];                                               // do . v_row of the fused output

  const int* sched = a.sched;
  const int slot = blockIdx.x / a.heads;
  const int head = blockIdx.x - slot * a.heads;
  const int4 hdr = *reinterpret_cast<const int4*>(sched);   // status, query tiles, key tiles, table entries needed
  const int longest = sched[SCHED_MAXLEN];
  const Tile t = reinterpret_cast<const Tile*>(sched + SCHED_HDR)[slot];
  asm volatile("" ::"s"(t.tok_start), "s"(t.doc_len), "s"(t.idx), "s"(t.batch), "s"(t.tab_base));   // keep the tile read above the branch
  const int tid = threadIdx.x;
  const bool refused = hdr.x != 0 || hdr.w > a.tab_stride || longest > a.max_doc_len || (GIVE && hdr.w > a.pz_entries);
  if (refused || slot >= hdr.y) {
    if (a.clear_spare) {     // for the dk/dv pass as well, which has no slots to spare
      int row0, row1;
      unsigned pair;
      spare_rows(refused, slot, hdr.y, sched[SCHED_TOTAL], a.tokens, a.nan_pair, row0, row1, pair);
      fill_rows16(a.dq, head, row0, row1, a.head_dim << a.out_f32, pair, tid, 512);
      fill_rows16(a.dk, head, row0, row1, a.head_dim << a.out_f32, pair, tid, 512);
      fill_rows16(a.dv, head, row0, row1, a.head_dim << a.out_f32, pair, tid, 512);
    }
    return;
  }
  const int L = t.doc_len;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int rb = w & 3;                                  // 32-query block of this wave
  const int m0 = t.idx * BM, qw0 = m0 + 32 * rb, qrow = qw0 + n;
  const bool qvalid = qrow < L;
  const int nblk = min(m0 + BM - 1, L - 1) / BF + 1;     // key blocks any query of the tile sees
  const int own = qw0 / BF;                              // the block's own keys: the last one it sees
  const int64_t tok0 = t.tok_start;
  auto rows_of = [&](const View& v) {
    return make_rows(reinterpret_cast<const elem_t*>(v.ptr) + t.batch * v.sb + head * v.sh + tok0 * v.st, v.st, L, a.head_dim);
  };
  // Row reads of chunk 2 ks + h: the swizzle is an XOR of the chunk number's low four bits, so the offset of a further
  // chunk is the first one's with a constant XORed in, and of the upper half's 256 bytes on: one register instead of
  // sixteen.
  int rbase = swz_off<D>(n, h);
  el8 fr[KS];                                            // Q or dO: operand column n is query qw0 + n
  constexpr int LEAD = 4;
  el8 op[LEAD];
  auto read_op = [&](const unsigned short* T, int k) { return lds_row8(T + (rbase ^ ((k % 8) << 4)) + 128 * (k / 8)); };
  auto chain_begin = [&](const unsigned short* T) {
#pragma unroll
    for (int k = 0; k < LEAD; ++k) op[k] = read_op(T, k);
  };
  auto chain_step = [&](const unsigned short* T, f32x16& x, int k) {
    x = mfma32(op[k % LEAD], fr[k], x);
    if (k + LEAD < KS) op[k % LEAD] = read_op(T, k + LEAD);
  };
  auto clear = [](f32x16& x) {
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = 0.0f;
  };
  // the tile's Q and dO rows by way of LDS (Q by the scores waves, dO by the others)
  {
    const Rows rows = rows_of(w < 4 ? a.q : a.go);
    TileCopy<D, BM, 256, false> copy;
    copy.init(tid & 255, rows.row_bytes, rows.used_bytes);
    copy.issue(rows, m0, w < 4 ? Ks : Vs);
  }
  wait_loads<0>();
  lds_barrier();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) fr[ks] = read_op((w < 4 ? Ks : Vs) + 32 * rb * D, ks);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lds_barrier();                              // the places are free
  float* const mine = hand + HAND * rb + 4 * lane;
  // GIVE: p and dz of a block as the lanes hold them, eight keys of a query in 16 bytes: lane's first eight keys, then
  // the lanes' other eight.  A block's place goes by the carry table's.
  const bool gives = GIVE && qw0 < L;         // (a block of queries behind the document's end has no place)
  __amdgpu_buffer_rsrc_t give_rs;
  if constexpr (GIVE)
    give_rs = __builtin_amdgcn_make_buffer_rsrc(a.pz + ((int64_t)head * a.pz_entries + t.tab_base) * PZ_WORDS, 0, pz_offset(tab_doc_entries(L)), 0x00020000);
  auto give = [&](const el8 (&v)[2], int block, int part) __attribute__((always_inline)) {
    const unsigned at = pz_offset(tab_seg32(L, block) + qw0) + 2048u * part;
    int give_at = 16 * lane;
    asm volatile("" : "+v"(give_at));         // (no register for it through the steps)
#pragma unroll
    for (int c = 0; c < 2; ++c) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v[c]), give_rs, give_at + 1024 * c, (int)at, 2 /* nt */);
    asm volatile("s_nop 0" ::"v"(v[0]), "v"(v[1]) : "memory");      // (the registers stay as they are behind the stores: see bwd_chain_kernel)
  };

  using std::integral_constant;
  if (w < 4) {
    __builtin_amdgcn_s_setprio(3);
    float dr = 0.0f;                          // d(rem) of this lane's row (see bwd_dq_kernel)
    if (a.grem.ptr != nullptr && qvalid) {
      const elem_t* grb = reinterpret_cast<const elem_t*>(a.grem.ptr) + t.batch * a.grem.sb + head * a.grem.sh + tok0 * a.grem.st;
      dr = (float)grb[(int64_t)qrow * a.grem.st];
    }
    // the document's area of the two tables (uniform); a lane adds its row and a block's 32-bit offset
    const int64_t tab0 = (int64_t)head * a.tab_stride + t.tab_base;
    const float* stick = a.stick + tab0;
    float* gtab = a.gtab + tab0;
    auto carry_of = [&](int i) {
      float e = PROD ? 1.0f : 0.0f;
      if (qvalid && i <= own) e = stick[(unsigned)(tab_seg32(L, i) + qrow)];
      return e;
    };
    float e0 = carry_of(0), e1 = carry_of(1), e2 = carry_of(2), e3;     // requested three steps ahead
    float carry_c = 0.0f;
    lds_barrier();                            // tile 0 has landed, do . v_row is there
    if (a.fuse) dr += drs[rb][n];
    if (!GIVE && qvalid && h == 0) gtab[(unsigned)(tab_rowplane32(L) + qrow)] = dr;
    f32x16 x;
    clear(x);
    chain_begin(Ks);
#pragma unroll
    for (int k = 0; k < KS; ++k) chain_step(Ks, x, k);
    auto step = [&](auto slot_tag, const int i, const float e, float& ahead) __attribute__((always_inline)) {
      constexpr int SLOT = decltype(slot_tag)::value;
      const unsigned short* const Tn = Ks + ((SLOT + 1) % SLOTS) * TILE;
      ahead = carry_of(i + 3);
      const bool visible = i <= own;
      float p[16], r[16], ends[2] = {0.0f, 0.0f};
      if (visible) {
        if (!GIVE && qvalid && h == 0) gtab[(unsigned)(tab_seg32(L, i) + qrow)] = carry_c;
        float c = e;
        if (i < own) stick_weights<AC, PROD, false, true>(x, a.c, i * BF, qrow, h, c, p, r, ends);
        else stick_weights<AC, PROD, true, true>(x, a.c, i * BF, qrow, h, c, p, r, ends);
        if (gives) {
          el8 pf[2] = {pack8(p), pack8(p + 8)};
          if (i == own && a.fuse) {           // fused output: rem_j * do_j reaches dv_j through the diagonal of p (see bwd_dkdv_kernel)
            float pd[16], rem_own = 0.0f;
            if (qvalid) rem_own = stick[(unsigned)(tab_rowplane32(L) + qrow)];
#pragma unroll
            for (int j = 0; j < 16; ++j) pd[j] = p[j] + (16 * h + j == n ? rem_own : 0.0f);
            pf[0] = pack8(pd);
            pf[1] = pack8(pd + 8);
          }
          if (qw0 + 32 > L && !qvalid) pf[0] = pf[1] = zero8();     // (rows behind the document's end leave nothing to be multiplied, finite or not)
          give(pf, i, 0);
        }
      }
      lds_barrier();
      if (visible) {
        f32x16 da;
        {
          f32x4 q4[4];
#pragma unroll
          for (int g = 0; g < 4; ++g) q4[g] = *reinterpret_cast<const f32x4*>(mine + 256 * g);
#pragma unroll
          for (int j = 0; j < 16; ++j) da[j] = q4[j >> 2][j & 3];
        }
        chain_begin(Tn);                      // (behind the last visible block: a tile that may not be there, unused)
        __builtin_amdgcn_sched_barrier(0);
        clear(x);
        el8 zf[2];
        if constexpr (PROD) {                 // grad_dz with the next block's chain between its instructions
          constexpr int A0 = KS / 4, REST = KS - A0;
#pragma unroll
          for (int k = 0; k < A0; ++k) chain_step(Tn, x, k);
          __builtin_amdgcn_sched_barrier(0);
          float t0 = 0.0f, t1 = 0.0f;
#pragma unroll
          for (int j = 0; j < 16; j += 2) { t0 = fmaf(p[j], da[j], t0); t1 = fmaf(p[j + 1], da[j + 1], t1); }
          float lo, hi;
          both_halves(fmaf(-dr, ends[0] - ends[1], t0 + t1), lo, hi);
          float dprev = fmaf(dr, ends[1], h == 1 ? carry_c + lo : carry_c);
          carry_c += lo + hi;
          __builtin_amdgcn_sched_barrier(0);
          float dz[16];
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const float dj = fmaf(p[j], da[j], dprev);
            dz[j] = fmaf(r[j], dj, -dprev);
            dprev = dj;
#pragma unroll
            for (int k = j * REST / 16; k < (j + 1) * REST / 16; ++k) chain_step(Tn, x, A0 + k);
            __builtin_amdgcn_sched_barrier(0);
          }
          zf[0] = pack8(dz);
          zf[1] = pack8(dz + 8);
        } else {
#pragma unroll
          for (int k = 0; k < KS; ++k) chain_step(Tn, x, k);
          grad_dz<PROD>(p, r, da, ends, h, carry_c, dr, zf);
        }
        if (GIVE && qw0 + 32 > L && !qvalid) zf[0] = zf[1] = zero8();
        *reinterpret_cast<el8*>(mine + HAND_Z) = zf[0];
        *reinterpret_cast<el8*>(mine + HAND_Z + 256) = zf[1];
      }
      lds_barrier();
    };
#pragma unroll 1
    for (int i = 0;; i += 4) {
      step(integral_constant<int, 0>{}, i, e0, e3);
      if (i + 1 >= nblk) break;
      step(integral_constant<int, 1>{}, i + 1, e1, e0);
      if (i + 2 >= nblk) break;
      step(integral_constant<int, 2>{}, i + 2, e2, e1);
      if (i + 3 >= nblk) break;
      step(integral_constant<int, 3>{}, i + 3, e3, e2);
      if (i + 4 >= nblk) break;
    }
  } else {
    __builtin_amdgcn_s_setprio(0);
    const int i16 = lane & 15, blk = (lane >> 4) & 1;
    const Rows krows = rows_of(a.k), vrows = rows_of(a.v);
    using Copy = TileCopy<D, BF, 256, true>;
    constexpr int LOADS_PER_TILE = 2 * Copy::NCH;
    Copy kcopy, vcopy;
    kcopy.init(tid & 255, krows.row_bytes, krows.used_bytes);
    vcopy.init(tid & 255, vrows.row_bytes, vrows.used_bytes);
    auto fetch = [&](int i) {
      kcopy.issue(krows, i * BF, Ks + (i % SLOTS) * TILE);
      vcopy.issue(vrows, i * BF, Vs + (i % SLOTS) * TILE);
    };
    if (a.fuse) {
      float dot = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const el8 vown = load_frag(vrows, qrow, 32 * ks + 16 * h);
#pragma unroll
        for (int e = 0; e < 8; ++e) dot = fmaf((float)fr[ks][e], (float)vown[e], dot);
      }
      float lo, hi;
      both_halves(dot, lo, hi);
      if (h == 0) drs[rb][n] = lo + hi;
    }
    wait_loads<0>();
    fetch(0);
    if (1 < nblk) fetch(1);
    if (2 < nblk) fetch(2);
    f32x16 dq[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int j = 0; j < 16; ++j) dq[db][j] = 0.0f;
    int tbase[2];                             // transpose reads of rows 8 u + 4 h + i16 / 4 (+ 16 tt), columns of block 0
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int col = 16 * blk + 4 * (i16 & 3);
      tbase[u] = swz_off<D>(8 * u + 4 * h + (i16 >> 2), col >> 3) + (col & 7);
    }
    if (nblk > 2) wait_loads<2 * LOADS_PER_TILE>();
    else if (nblk > 1) wait_loads<LOADS_PER_TILE>();
    else wait_loads<0>();
    lds_barrier();
    f32x16 da;
    clear(da);
    chain_begin(Vs);
#pragma unroll
    for (int k = 0; k < KS; ++k) chain_step(Vs, da, k);
    // dq += dz K of a block, whose tile is at Kt
    auto product = [&](const unsigned short* Kt, int block) __attribute__((always_inline)) {
      const el8 zf[2] = {*reinterpret_cast<const el8*>(mine + HAND_Z), *reinterpret_cast<const el8*>(mine + HAND_Z + 256)};
      if (gives) give(zf, block, 1);
      constexpr int N = 2 * DB, AHEAD = 4;    // operand reads run AHEAD products ahead
      el8 kt[AHEAD];
      auto read_k = [&](int m) {
        const int tt = m / DB, db = m % DB;
        const unsigned short* const krow = Kt + 16 * tt * D + 128 * (db / 4);
        return lds_tr8(krow + (tbase[0] ^ ((db % 4) << 5)), krow + (tbase[1] ^ ((db % 4) << 5)));
      };
#pragma unroll
      for (int m = 0; m < AHEAD; ++m) kt[m] = read_k(m);
#pragma unroll
      for (int m = 0; m < N; ++m) {
        dq[m % DB] = mfma32(kt[m % AHEAD], zf[m / DB], dq[m % DB]);   // (dq^T: see store_block32_rows)
        if (m + AHEAD < N) kt[m % AHEAD] = read_k(m + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto step = [&](auto slot_tag, const int i) __attribute__((always_inline)) {
      constexpr int SLOT = decltype(slot_tag)::value;
      const unsigned short* const Tn = Vs + ((SLOT + 1) % SLOTS) * TILE;
      asm volatile("" : "+v"(rbase), "+v"(tbase[0]), "+v"(tbase[1]));     // (the XORs stay here: there are no registers for their results)
      if (i <= own) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 q4 = {da[4 * g], da[4 * g + 1], da[4 * g + 2], da[4 * g + 3]};
          *reinterpret_cast<f32x4*>(mine + 256 * g) = q4;
        }
      }
      const bool multiplied = i > 0 && i - 1 <= own;
      if (multiplied) product(Ks + ((SLOT + SLOTS - 1) % SLOTS) * TILE, i - 1);
      // tile i + 1, which everyone reads behind this barrier, has landed (what the products stored came after tile i + 2)
      if (gives && multiplied && i + 2 < nblk) wait_loads<LOADS_PER_TILE + 2>();
      else if (i + 2 < nblk) wait_loads<LOADS_PER_TILE>();
      else wait_loads<0>();
      lds_barrier();
      if (i + 3 < nblk) fetch(i + 3);
      clear(da);        // (always: it must not live through the products)
      if (i + 1 <= own) {
        chain_begin(Tn);
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          chain_step(Tn, da, k);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      lds_barrier();
    };
#pragma unroll 1
    for (int i = 0;; i += 4) {
      step(integral_constant<int, 0>{}, i);
      if (i + 1 >= nblk) break;
      step(integral_constant<int, 1>{}, i + 1);
      if (i + 2 >= nblk) break;
      step(integral_constant<int, 2>{}, i + 2);
      if (i + 3 >= nblk) break;
      step(integral_constant<int, 3>{}, i + 3);
      if (i + 4 >= nblk) break;
    }
    if (nblk - 1 <= own) product(Ks + ((nblk - 1) % SLOTS) * TILE, nblk - 1);
    store_rows(dq, a.inv_temp, rows_of(a.dq), qrow, L, h, a.out_f32);
  }
}

// -------------------------------------------------------------------------------------------
// dk / dv pass of the same head dims where the dq pass has left p and dz of every block in memory (GIVE, above): 128
// keys of one (document, head) per workgroup, dv = p^T dO and dk = dz^T Q over the queries that can see them, 32 per
// step.  All eight waves are alike: 64 keys x half of the columns of one output each (128 registers), and a share of
// the copies.  A tile is 48 KiB (Q, dO, p, dz), three of them in a ring; one barrier per step, operands read a step
// ahead.
//
// Bound by what it reads: 16 heads x 16 K tokens in eight documents at head_dim 256, 456 us for 1.45 GB of p and dz,
// which are read once, and Q and dO, of which every key tile takes its own (398 without the former, 367 without the
// latter, both timing only); the matrix pipes are busy for 40 %.  So the queries are walked from the document's end:
// the key tiles of a (document, head) that start together then read the same rows at the same time (from the tile's own
// keys on 816 us for 678, 12 heads of 4 x 4096), and p and dz stream past the L2s that Q and dO are kept in (as do the
// dq pass's stores of them: 568 -> 456).  The pass that forms p and dz itself: 890.  Handing them on costs the dq pass
// 100 of 724 us, a third of it the packing.
// -------------------------------------------------------------------------------------------
template <int U>
__global__ void __launch_bounds__(512, 1) bwd_dkdv_given_kernel(const KArgs a) {
  constexpr int D = 256, DBH = U / 64;       // DBH: 32-wide column blocks of a wave
  constexpr int TQ = 32, SLOTS = 3, QTILE = TQ * D, PTILE = TQ * BKV, SLOT = 2 * QTILE + 2 * PTILE;
  __shared__ __attribute__((aligned(1024))) unsigned short tiles[SLOTS * SLOT];     // Q, dO, p, dz

  // (the grid never exceeds the room of the list: its tile is read along with the header)
  const int* sched = a.sched;
  const int which = blockIdx.x / a.heads;
  const int head = blockIdx.x - which * a.heads;
  const int4 hdr = *reinterpret_cast<const int4*>(sched);   // status, query tiles, key tiles, table entries needed
  const int longest = sched[SCHED_MAXLEN];
  const Tile t = reinterpret_cast<const Tile*>(sched + a.kv_list_off)[which];
  asm volatile("" ::"s"(t.tok_start), "s"(t.doc_len), "s"(t.idx), "s"(t.batch), "s"(t.tab_base));   // keep the tile read above the branch
  if (hdr.x != 0 || hdr.w > a.tab_stride || hdr.w > a.pz_entries || longest > a.max_doc_len || which >= hdr.z) return;
  const int L = t.doc_len, q_first = t.idx * BKV;
  const int nsteps = (L - q_first + TQ - 1) / TQ;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, blk = (lane >> 4) & 1;
  const int mat = w >> 2, khalf = (w >> 1) & 1, chalf = w & 1;       // (dv | dk), 64 keys, half of the columns
  const int64_t tok0 = t.tok_start;
  auto rows_of = [&](const View& v) {
    return make_rows(reinterpret_cast<const elem_t*>(v.ptr) + t.batch * v.sb + head * v.sh + tok0 * v.st, v.st, L, a.head_dim);
  };
  const Rows qrows = rows_of(a.q), grows = rows_of(a.go);
  using Copy = TileCopy<D, TQ, 512, false>;
  Copy qcopy, gcopy;
  qcopy.init(tid, qrows.row_bytes, qrows.used_bytes);
  gcopy.init(tid, grows.row_bytes, grows.used_bytes);
  // Staged p or dz: four blocks one behind the other, each as it lies in memory: eight keys of a query in 16 bytes, the
  // first eight keys of a half-wave's sixteen, then the other eight.  A wave copies one of those halves of a block.
  // The queries are XORed with four times the number of the eight keys, so that the transpose reads of all of them take
  // different banks.  (Of the first three blocks of queries the newer key blocks do not exist: what is copied in their
  // place is not multiplied.)
  const int from = 1024 * (w & 1) + 16 * (lane ^ (4 * ((lane >> 5) + 2 * (w & 1))));
  const int place = tab_seg32(L, min((BKV / 32) * t.idx + (w >> 1), (L - 1) / 32)) + q_first;
  const __amdgpu_buffer_rsrc_t pz_rs = __builtin_amdgcn_make_buffer_rsrc(a.pz + ((int64_t)head * a.pz_entries + t.tab_base) * PZ_WORDS, 0,
                                                                       pz_offset(tab_doc_entries(L)), 0x00020000);
  constexpr int LOADS_PER_TILE = 2 * Copy::NCH + 2;
  auto fetch = [&](int turn, int slot) {
    const int step = nsteps - 1 - turn;
    unsigned short* const T = tiles + slot * SLOT;
    qcopy.issue(qrows, q_first + step * TQ, T);
    gcopy.issue(grows, q_first + step * TQ, T + QTILE);
    const unsigned soff = __builtin_amdgcn_readfirstlane(pz_offset(place + step * TQ));
    async_copy16<true>(pz_rs, T + 2 * QTILE + 512 * w, from, (int)soff);
    async_copy16<true>(pz_rs, T + 2 * QTILE + PTILE + 512 * w, from, (int)(soff + 2048));
  };
  fetch(0, 0);
  if (nsteps > 1) fetch(1, 1);
  if (nsteps > 2) fetch(2, 2);
  f32x16 acc[2][DBH];
#pragma unroll
  for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
    for (int j = 0; j < DBH; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[kb2][j][e] = 0.0f;
  // transpose reads of rows 8 h + 4 u + i16 / 4 (+ 16 ks): staged block, tile (bytes)
  const int base = (int)(unsigned)(size_t)tiles;
  int xoff[2][2], yoff[2][DBH];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = 8 * h + 4 * u + (i16 >> 2), c = 16 * blk + 4 * (i16 & 3);
#pragma unroll
    for (int kb2 = 0; kb2 < 2; ++kb2)
      xoff[u][kb2] = base + 2 * (2 * QTILE + mat * PTILE) + 2048 * (2 * khalf + kb2) + 1024 * ((c >> 3) & 1) +
                     16 * (32 * blk + (r ^ (4 * (blk + 2 * ((c >> 3) & 1))))) + 2 * (c & 7);
#pragma unroll
    for (int j = 0; j < DBH; ++j)
      yoff[u][j] = base + 2 * ((mat ? 0 : QTILE) + swz_off<D>(r, (32 * (chalf * DBH + j) + c) >> 3) + (c & 7));
  }
  // Turn i multiplies what was read of tile i during turn i - 1, and a fragment that is done with gives way to tile i + 1's.
  el8 af[2][2], bf[2][DBH];
  auto read_x = [&](int at, int kb2, int ks) { af[kb2][ks] = lds_tr8_at(xoff[0][kb2] + at + 256 * ks, xoff[1][kb2] + at + 256 * ks); };
  auto read_y = [&](int at, int j, int ks) { bf[ks][j] = lds_tr8_at(yoff[0][j] + at + 32 * ks * D, yoff[1][j] + at + 32 * ks * D); };
  int slot = 0;                               // of tile i
  // LAST: the last three, whose queries may not see all key blocks: those stay out, finite or not.
  auto turn = [&](auto last_tag, const int i) __attribute__((always_inline)) {
    constexpr bool LAST = decltype(last_tag)::value;
    if (i + 2 < nsteps) wait_loads<LOADS_PER_TILE>();
    else wait_loads<0>();
    lds_barrier();                            // tile i + 1 has landed, everyone has read tile i
    if (i + 3 < nsteps) fetch(i + 3, slot);
    slot = slot == SLOTS - 1 ? 0 : slot + 1;
    const int at = slot * (2 * SLOT);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int j = 0; j < DBH; ++j) {
#pragma unroll
        for (int kb2 = 0; kb2 < 2; ++kb2)
          if (!LAST || 2 * khalf + kb2 <= nsteps - 1 - i) acc[kb2][j] = mfma32(bf[ks][j], af[kb2][ks], acc[kb2][j]);
        read_y(at, j, ks);
        __builtin_amdgcn_sched_barrier(0);
      }
      read_x(at, 0, ks);
      read_x(at, 1, ks);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (nsteps > 2) wait_loads<2 * LOADS_PER_TILE>();
  else if (nsteps > 1) wait_loads<LOADS_PER_TILE>();
  else wait_loads<0>();
  lds_barrier();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
    for (int j = 0; j < DBH; ++j) read_y(0, j, ks);
    read_x(0, 0, ks);
    read_x(0, 1, ks);
  }
  int i = 0;
#pragma unroll 1
  for (; i + 3 < nsteps; ++i) turn(std::false_type{}, i);
#pragma unroll 1
  for (; i < nsteps; ++i) turn(std::true_type{}, i);
  const Rows out = rows_of(mat ? a.dk : a.dv);
#pragma unroll
  for (int kb2 = 0; kb2 < 2; ++kb2) {
    const int row = q_first + 64 * khalf + 32 * kb2 + n;
#pragma unroll
    for (int j = 0; j < DBH; ++j)
      store_block32_rows(acc[kb2][j], mat ? a.inv_temp : 1.0f, out, row * (int)out.row_bytes, row < L, 32 * (chalf * DBH + j), h, a.out_f32);
  }
}

template __global__ void bwd_dkdv_wide_kernel<false, false, 256>(const KArgs);
template __global__ void bwd_dkdv_wide_kernel<true, false, 256>(const KArgs);
template __global__ void bwd_dkdv_wide_kernel<false, true, 256>(const KArgs);
template __global__ void bwd_dkdv_wide_kernel<true, true, 256>(const KArgs);
template __global__ void bwd_dkdv_wide_kernel<false, true, 192>(const KArgs);
template __global__ void bwd_dkdv_wide_kernel<true, true, 192>(const KArgs);

template __global__ void bwd_dq_wide_kernel<false, false, 256, false>(const KArgs);
template __global__ void bwd_dq_wide_kernel<true, false, 256, false>(const KArgs);
template __global__ void bwd_dq_wide_kernel<false, true, 256, false>(const KArgs);
template __global__ void bwd_dq_wide_kernel<true, true, 256, false>(const KArgs);
template __global__ void bwd_dq_wide_kernel<false, true, 192, false>(const KArgs);
template __global__ void bwd_dq_wide_kernel<true, true, 192, false>(const KArgs);
template __global__ void bwd_dq_wide_kernel<false, true, 256, true>(const KArgs);
template __global__ void bwd_dq_wide_kernel<true, true, 256, true>(const KArgs);
template __global__ void bwd_dq_wide_kernel<false, true, 192, true>(const KArgs);
template __global__ void bwd_dq_wide_kernel<true, true, 192, true>(const KArgs);

template __global__ void bwd_dkdv_given_kernel<256>(const KArgs);
template __global__ void bwd_dkdv_given_kernel<192>(const KArgs);

template <int U, bool GIVE>
static void launch_dq_product(const KArgs& a, bool ac, int n_q_max, hipStream_t s) {
  const dim3 grid((unsigned)n_q_max * (unsigned)a.heads), block(512);
  if (ac) hipLaunchKernelGGL((bwd_dq_wide_kernel<true, true, U, GIVE>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((bwd_dq_wide_kernel<false, true, U, GIVE>), grid, block, 0, s, a);
}
hipError_t launch_bwd_dq_wide(const KArgs& a, bool ac, bool prod, int n_q_max, hipStream_t s) {
  const dim3 grid((unsigned)n_q_max * (unsigned)a.heads), block(512);
  const bool narrow = used_width(a.head_dim) == 192;
  if (prod && a.pz != nullptr) narrow ? launch_dq_product<192, true>(a, ac, n_q_max, s) : launch_dq_product<256, true>(a, ac, n_q_max, s);
  else if (prod) narrow ? launch_dq_product<192, false>(a, ac, n_q_max, s) : launch_dq_product<256, false>(a, ac, n_q_max, s);
  else if (ac) hipLaunchKernelGGL((bwd_dq_wide_kernel<true, false, 256, false>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((bwd_dq_wide_kernel<false, false, 256, false>), grid, block, 0, s, a);
  return hipGetLastError();
}

// tiles: see launch_bwd_dkdv_wide
hipError_t launch_bwd_dkdv_given(const KArgs& a, int tiles, hipStream_t s) {
  const dim3 grid((unsigned)tiles * (unsigned)a.heads), block(512);
  if (used_width(a.head_dim) == 192) hipLaunchKernelGGL((bwd_dkdv_given_kernel<192>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((bwd_dkdv_given_kernel<256>), grid, block, 0, s, a);
  return hipGetLastError();
}

// tiles: upper bound on the tiles of the key-tile list, no more than it has room for
hipError_t launch_bwd_dkdv_wide(const KArgs& a, bool ac, bool prod, int tiles, hipStream_t s) {
  const dim3 grid((unsigned)dkdv_main_workgroups(a.head_dim, tiles) * (unsigned)a.heads), block(512);
  if (prod && used_width(a.head_dim) == 192) {
    if (ac) hipLaunchKernelGGL((bwd_dkdv_wide_kernel<true, true, 192>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((bwd_dkdv_wide_kernel<false, true, 192>), grid, block, 0, s, a);
  } else if (ac) {
    if (prod) hipLaunchKernelGGL((bwd_dkdv_wide_kernel<true, true, 256>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((bwd_dkdv_wide_kernel<true, false, 256>), grid, block, 0, s, a);
  } else {
    if (prod) hipLaunchKernelGGL((bwd_dkdv_wide_kernel<false, true, 256>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((bwd_dkdv_wide_kernel<false, false, 256>), grid, block, 0, s, a);
  }
  return hipGetLastError();
}

}  // inline namespace SBA_ELEM_NS
}  // namespace sba
