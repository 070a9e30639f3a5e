// Forward kernel: one 128-row query tile of one (document, head) per workgroup, KV tiles of
// 32 keys walked from the causal diagonal back to the start of the document.
//
// Replaces upstream `_forward` / `_forward_one_row`
// (stickbreaking_attention/sb_varlen/sb_varlen_fwd.py:81-215, :231-410) and the fixed-length
// wrapper (stickbreaking_attention/sb_attn/sb_fwd.py:15-136).
#include "sba_kernels.hpp"

#include <type_traits>

namespace sba {
inline namespace SBA_ELEM_NS {

// The item of this workgroup (items: tiles of every head, most expensive first).  Workgroup b starts on the same CU as
// b + n_cus, b + 2 n_cus ...; while the chip holds the whole launch at once, whoever comes first gets the most
// expensive tile of every round (tiles 15, 11, 7 and 3 for one CU against 12, 8, 4 and 0 for another).  Such a launch
// deals every second round backwards, eight workgroups at a time, which leaves an item's head on its XCD.  A larger
// launch fills in behind its expensive tiles by itself (lg_cus: NO_DEAL).  4 x 16 x 2048: 58.0 -> 55.7 us at head_dim
// 64 (with the carry table), 43.9 -> 41.9 at 32.  (Shifts, no branch, the grid's size as an argument, and the division
// by the heads a multiplication: every workgroup waits for this before its first load.  With divisions and a branch 31
// heads of 1003 tokens at head_dim 128 took 32.2 us for 31.6, 20 heads x 25 K tokens in 1682 documents at head_dim 32
// 94 for 84.)
__device__ __forceinline__ unsigned deal_item(int lg_cus, unsigned n) {
  const unsigned b = blockIdx.x, round = b >> lg_cus, first = round << lg_cus, eights = min(1u << lg_cus, n - first) >> 3, at = (b - first) >> 3;
  return (round & 1) && at < eights ? first + 8 * (eights - 1 - at) + (b & 7) : b;
}

// MODE 1 (WOUT): also write the attention weights (fp32, before their bf16 rounding) into a dense [tokens x tokens]
// matrix per (batch, head) -- upstream's `return_attention` debug output (sb_varlen_fwd.py:195-202).  MODE 2 (TAB):
// write the carry table and nothing else -- no V tiles, no P.V products, no o, no rem -- for a backward whose forward
// kept no table.  Separate instantiations, so the production kernel (MODE 0) carries none of it.  head_dim 256: two
// workgroups per CU, so that a wave's waits are another's time: a ring of two slots (64 KiB) and 256 registers, 64 of
// them Q fragments and 128 accumulators, the tile offsets of columns 128 .. 255 as immediates.  (One workgroup per CU,
// one wave per SIMD with 512 registers and three slots: 554 us on 16 heads x 16 K tokens in eight documents, this 415.)
// U: columns that are multiplied (see used_width); tile rows in LDS keep the width D.
template <int D, bool AC, bool PROD, int MODE, int U = D>
__global__ void __launch_bounds__(NT, D > 128 ? 2 : 3) fwd_kernel(const KArgs a) {
  constexpr bool WOUT = MODE == 1, TAB = MODE == 2;
  constexpr int KS = U / 16;     // contraction steps of K.Q^T
  constexpr int DB = U / 32;     // 32-wide output column blocks of P.V
  constexpr int BF = 32;         // keys per staged tile: one MFMA sub-block
  constexpr int TILE = BF * D;   // elements of one K or V tile (unpadded, swizzled)
  // K and V tiles of 32 keys in a ring of three slots (two at head_dim 256) filled by asynchronous global -> LDS copies:
  // 48 KiB per workgroup at head_dim 128, so three workgroups share a CU.
  constexpr int RING = D > 128 ? 2 : 3;
  __shared__ __attribute__((aligned(16))) unsigned short smem[2 * RING * TILE];
  unsigned short* const Ks = smem;
  unsigned short* const Vs = smem + RING * TILE;

  // Header words and this workgroup's tile are fetched together (the grid never exceeds the
  // allocated list, so the tile read is safe before the count is known): one round trip.
  const int* sched = a.sched;
  const unsigned item = deal_item(a.lg_deal, a.n_items), below = __umulhi(item, a.heads_inv);   // (the quotient or one less)
  const int over = (int)(item - below * a.heads) >= a.heads ? 1 : 0, slot = below + over, head = item - slot * a.heads;
  const int4 hdr = *reinterpret_cast<const int4*>(sched);   // status, query tiles, key tiles, table entries needed
  const Tile t = reinterpret_cast<const Tile*>(sched + SCHED_HDR)[slot];
  asm volatile("" ::"s"(t.tok_start), "s"(t.doc_len), "s"(t.idx), "s"(t.batch));   // keep the tile read above the branch
  const bool refused = hdr.x != 0 || (a.stick != nullptr && hdr.w > a.tab_stride);
  if (refused || slot >= hdr.y) {
    if (a.clear_spare && !TAB) {
      int row0, row1;
      unsigned pair;
      spare_rows(refused, slot, hdr.y, sched[SCHED_TOTAL], a.tokens, a.nan_pair, row0, row1, pair);
      fill_rows16(a.o, head, row0, row1, a.head_dim << a.out_f32, pair, threadIdx.x, NT);
      fill_rows16(a.rem, head, row0, row1, 1 << a.out_f32, pair, threadIdx.x, NT);
    }
    return;
  }

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int m0 = t.idx * BM;
  const int qw0 = m0 + 32 * w;
  const int qrow = qw0 + n;
  const bool qvalid = qrow < t.doc_len;

  const int64_t tok0 = t.tok_start;
  const elem_t* qb = reinterpret_cast<const elem_t*>(a.q.ptr) + t.batch * a.q.sb + head * a.q.sh + tok0 * a.q.st;
  const elem_t* kb = reinterpret_cast<const elem_t*>(a.k.ptr) + t.batch * a.k.sb + head * a.k.sh + tok0 * a.k.st;
  const elem_t* vb = reinterpret_cast<const elem_t*>(a.v.ptr) + t.batch * a.v.sb + head * a.v.sh + tok0 * a.v.st;
  elem_t* ob = reinterpret_cast<elem_t*>(a.o.ptr) + t.batch * a.o.sb + head * a.o.sh + tok0 * a.o.st;
  elem_t* rb = reinterpret_cast<elem_t*>(a.rem.ptr) + t.batch * a.rem.sb + head * a.rem.sh + tok0 * a.rem.st;
  const Rows qrows = make_rows(qb, a.q.st, t.doc_len, a.head_dim);
  const Rows krows = make_rows(kb, a.k.st, t.doc_len, a.head_dim);
  const Rows vrows = make_rows(vb, a.v.st, t.doc_len, a.head_dim);

  const int last_key = min(m0 + BM - 1, t.doc_len - 1);
  const int kt_last = last_key / BF;

  // Q^T operand fragments: lane (n, h) holds Q[qrow][16*ks + 8*h .. +7] (zeros past the document).
  el8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = load_frag(qrows, qrow, 32 * ks + 16 * h);

  // RING - 1 tiles are in flight while one is consumed.
  // (a 32 x 32 tile is one instruction each for two waves: the other two request nothing, wait for
  // nothing and meet the copies at the barrier)
  constexpr int CT = D == 32 ? NT / 2 : NT;   // threads that copy tiles
  const bool copier = tid < CT;               // (uniform per wave)
  TileCopy<D, BF, CT, true> kcopy, vcopy;
  kcopy.init(tid, krows.row_bytes, krows.used_bytes);
  vcopy.init(tid, vrows.row_bytes, vrows.used_bytes);
  constexpr int LOADS_PER_TILE = (TAB ? 1 : 2) * TileCopy<D, BF, CT, true>::NCH;
  if (copier) {
    kcopy.issue(krows, kt_last * BF, Ks);
    if (!TAB) vcopy.issue(vrows, kt_last * BF, Vs);
    if (RING == 3 && kt_last >= 1) {
      kcopy.issue(krows, (kt_last - 1) * BF, Ks + TILE);
      if (!TAB) vcopy.issue(vrows, (kt_last - 1) * BF, Vs + TILE);
    }
  }

  f32x16 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[db][i] = 0.0f;
  float carry = PROD ? 1.0f : 0.0f;

  // Offsets (elements) inside a tile.  K: row read of chunk 2*ks + h of LDS row n (= MFMA row n).
  // V: transpose reads of rows 8*u + 4*h + i/4 (+ 16*tt), columns 32*db + 16*blk + 4*(i%4).
  // (Rows of 512 bytes: the swizzle leaves the upper half of the columns where it is, 256 bytes on.)
  const int i16 = lane & 15, blk = (lane >> 4) & 1;
  constexpr int KO = KS < 8 ? KS : 8, DO = DB < 4 ? DB : 4;
  int koff[KO], voff[2][DO];
#pragma unroll
  for (int ks = 0; ks < KO; ++ks) koff[ks] = swz_off<D>(n, 2 * ks + h);
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = 8 * u + 4 * h + (i16 >> 2);
#pragma unroll
    for (int db = 0; db < DO; ++db) {
      const int col = 32 * db + 16 * blk + 4 * (i16 & 3);
      voff[u][db] = swz_off<D>(r, col >> 3) + (col & 7);
    }
  }
  // the document's triangular table area; a lane adds its row and a block's 32-bit offset
  float* stick = a.stick == nullptr ? nullptr : a.stick + (int64_t)head * a.tab_stride + t.tab_base;   // (uniform)

  // One tile step; the ring slot is a compile-time constant so every LDS address is a fixed
  // register plus an immediate.
  auto tile = [&](auto slot_c, const int kt) {
    constexpr int SLOT = decltype(slot_c)::value;
    constexpr int REFILL = (SLOT + RING - 1) % RING;   // slot of tile kt + 1, free once every wave is past it
    // Tile kt has landed when only the loads of tile kt - 1 (with three slots issued after it, returning in
    // order) can still be in flight; stores in between only make the wait stricter.
    if (RING == 3 && kt >= 1) wait_loads<LOADS_PER_TILE>(); else wait_loads<0>();
    lds_barrier();
    if (kt >= RING - 1 && copier) {
      kcopy.issue(krows, (kt - RING + 1) * BF, Ks + REFILL * TILE);
      if (!TAB) vcopy.issue(vrows, (kt - RING + 1) * BF, Vs + REFILL * TILE);
    }
    const unsigned short* Kt = Ks + SLOT * TILE;
    const unsigned short* Vt = Vs + SLOT * TILE;
    const int k0 = kt * BF;
    if (sub_skip<AC>(k0, qw0)) return;
    // stick left on entering this block: what both backward kernels start it from
    if (stick != nullptr && h == 0 && qvalid) stick[(unsigned)(tab_seg32(t.doc_len, kt) + qrow)] = carry;
    f32x16 x;
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = 0.0f;
    {
      // Beyond head_dim 64 K fragments are read four ahead of their multiplication, in an order that is pinned: left to
      // itself the compiler reads one or two ahead and waits for each.  32 heads of 64 K tokens, longest document 32 K,
      // at head_dim 128 10.98 -> 10.81 ms (sustained, at a lower clock than the 9.47 -> 9.41 of a few launches), 12
      // heads of 4 x 4096 218 -> 211 us, 16 heads x 16 K in eight documents at 256 430 -> 415, at 192 322 -> 315.
      // (Four or two fragments pinned at 64 and 32: 0.8 % slower to 0.  Half of V's fragments read before the weights
      // are formed: nothing at 64 and 96, spills from 128 on.)
      constexpr bool PIN = KS > 4;
      constexpr int AHEAD = KS < 4 ? KS : 4;
      el8 kfr[AHEAD];
#pragma unroll
      for (int ks = 0; ks < AHEAD; ++ks) kfr[ks] = lds_row8(Kt + koff[ks % KO] + 128 * (ks / KO));
      if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        x = mfma32(kfr[ks % AHEAD], qf[ks], x);
        if (ks + AHEAD < KS) kfr[ks % AHEAD] = lds_row8(Kt + koff[(ks + AHEAD) % KO] + 128 * ((ks + AHEAD) / KO));
        if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
      }
    }
    float p[16];
    if constexpr (PROD) {
      if (sub_full<AC>(k0, qw0)) stick_weights_fwd<AC, false>(x, a.c, k0, qrow, h, carry, p);
      else stick_weights_fwd<AC, true>(x, a.c, k0, qrow, h, carry, p);
    } else {
      float unused[16];
      if (sub_full<AC>(k0, qw0)) stick_weights<AC, PROD, false, false>(x, a.c, k0, qrow, h, carry, p, unused);
      else stick_weights<AC, PROD, true, false>(x, a.c, k0, qrow, h, carry, p, unused);
    }
    if constexpr (WOUT) {
      // this lane: query qrow, keys k0 + 16*h + i; masked positions already hold 0
      if (qvalid) {
        float* wrow = a.weights + (((int64_t)t.batch * a.heads + head) * a.tokens + tok0 + qrow) * a.tokens + tok0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = k0 + 16 * h + i;
          if (key < t.doc_len) wrow[key] = p[i];
        }
      }
    }
    if constexpr (TAB) return;
    // P as the B operand of O^T = V^T.P^T: slot s of step tt is key 16*h + 8*tt + s, which the
    // permuted tile keeps in LDS row 16*tt + 8*(s/4) + 4*h + s%4.
    el8 vfr[2][DB];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const unsigned short* vrow = Vt + 16 * tt * D;
#pragma unroll
      for (int db = 0; db < DB; ++db)
        vfr[tt][db] = lds_tr8(vrow + voff[0][db % DO] + 128 * (db / DO), vrow + voff[1][db % DO] + 128 * (db / DO));
    }
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const el8 pf = pack8(p + 8 * tt);
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[db] = mfma32(vfr[tt][db], pf, oacc[db]);   // (o^T: see store_block32_rows)
    }
  };

  // The Q fragments and both tiles have landed.  (A full wait, so that the compiler's bookkeeping
  // holds no load of its own when the loop begins: a wait it placed inside the loop for the Q
  // fragments would, from the second step on, wait for the tile copies issued in between.)
  wait_loads<0>();
  for (int kt = kt_last;;) {
    tile(std::integral_constant<int, 0>{}, kt);
    if (--kt < 0) break;
    tile(std::integral_constant<int, 1>{}, kt);
    if (--kt < 0) break;
    if constexpr (RING == 3) {
      tile(std::integral_constant<int, 2>{}, kt);
      if (--kt < 0) break;
    }
  }

  // epilogue: rem = what is left of the stick; o rows in the accumulator layout
  const float r = PROD ? carry : fast_exp2(carry);
  if (h == 0 && qvalid) {
    if (!TAB) {
      elem_t* const at = rb + (int64_t)qrow * a.rem.st;
      if (a.out_f32) *reinterpret_cast<float*>(at) = (float)(elem_t)r;
      else *at = (elem_t)r;
    }
    // rem in full precision for the backward of the fused output (last plane of the table)
    if (stick != nullptr) stick[(unsigned)(tab_rowplane32(t.doc_len) + qrow)] = r;
  }
  if constexpr (TAB) return;
  const Rows orows = make_rows(ob, a.o.st, t.doc_len, a.head_dim);
  // what every caller computes next (upstream tests/test_varlen.py:101): o + rem * v
  if (a.fuse) store_rows_axpy(oacc, orows, qrow, t.doc_len, h, a.out_f32, vrows, r);
  else store_rows(oacc, 1.0f, orows, qrow, t.doc_len, h, a.out_f32);
}

// Explicit instantiations: every (head_dim, attend_current, carry space) variant the launchers use.
template __global__ void fwd_kernel<32, false, false, 0>(const KArgs);
template __global__ void fwd_kernel<32, false, false, 1>(const KArgs);
template __global__ void fwd_kernel<32, false, true, 0>(const KArgs);
template __global__ void fwd_kernel<32, false, true, 1>(const KArgs);
template __global__ void fwd_kernel<32, true, false, 0>(const KArgs);
template __global__ void fwd_kernel<32, true, false, 1>(const KArgs);
template __global__ void fwd_kernel<32, true, true, 0>(const KArgs);
template __global__ void fwd_kernel<32, true, true, 1>(const KArgs);
template __global__ void fwd_kernel<64, false, false, 0>(const KArgs);
template __global__ void fwd_kernel<64, false, false, 1>(const KArgs);
template __global__ void fwd_kernel<64, false, true, 0>(const KArgs);
template __global__ void fwd_kernel<64, false, true, 1>(const KArgs);
template __global__ void fwd_kernel<64, true, false, 0>(const KArgs);
template __global__ void fwd_kernel<64, true, false, 1>(const KArgs);
template __global__ void fwd_kernel<64, true, true, 0>(const KArgs);
template __global__ void fwd_kernel<64, true, true, 1>(const KArgs);
template __global__ void fwd_kernel<128, false, false, 0>(const KArgs);
template __global__ void fwd_kernel<128, false, false, 1>(const KArgs);
template __global__ void fwd_kernel<128, false, true, 0>(const KArgs);
template __global__ void fwd_kernel<128, false, true, 1>(const KArgs);
template __global__ void fwd_kernel<128, true, false, 0>(const KArgs);
template __global__ void fwd_kernel<128, true, false, 1>(const KArgs);
template __global__ void fwd_kernel<128, true, true, 0>(const KArgs);
template __global__ void fwd_kernel<128, true, true, 1>(const KArgs);

template __global__ void fwd_kernel<32, false, false, 2>(const KArgs);
template __global__ void fwd_kernel<32, false, true, 2>(const KArgs);
template __global__ void fwd_kernel<32, true, false, 2>(const KArgs);
template __global__ void fwd_kernel<32, true, true, 2>(const KArgs);
template __global__ void fwd_kernel<64, false, false, 2>(const KArgs);
template __global__ void fwd_kernel<64, false, true, 2>(const KArgs);
template __global__ void fwd_kernel<64, true, false, 2>(const KArgs);
template __global__ void fwd_kernel<64, true, true, 2>(const KArgs);
template __global__ void fwd_kernel<128, false, false, 2>(const KArgs);
template __global__ void fwd_kernel<128, false, true, 2>(const KArgs);
template __global__ void fwd_kernel<128, true, false, 2>(const KArgs);
template __global__ void fwd_kernel<128, true, true, 2>(const KArgs);
template __global__ void fwd_kernel<256, false, false, 0>(const KArgs);
template __global__ void fwd_kernel<256, false, false, 1>(const KArgs);
template __global__ void fwd_kernel<256, false, true, 0>(const KArgs);
template __global__ void fwd_kernel<256, false, true, 1>(const KArgs);
template __global__ void fwd_kernel<256, true, false, 0>(const KArgs);
template __global__ void fwd_kernel<256, true, false, 1>(const KArgs);
template __global__ void fwd_kernel<256, true, true, 0>(const KArgs);
template __global__ void fwd_kernel<256, true, true, 1>(const KArgs);
template __global__ void fwd_kernel<256, false, false, 2>(const KArgs);
template __global__ void fwd_kernel<256, false, true, 2>(const KArgs);
template __global__ void fwd_kernel<256, true, false, 2>(const KArgs);
template __global__ void fwd_kernel<256, true, true, 2>(const KArgs);

template __global__ void fwd_kernel<128, false, true, 0, 96>(const KArgs);
template __global__ void fwd_kernel<128, true, true, 0, 96>(const KArgs);
template __global__ void fwd_kernel<256, false, true, 0, 192>(const KArgs);
template __global__ void fwd_kernel<256, true, true, 0, 192>(const KArgs);

template <int D, int U>
static hipError_t launch_fwd_narrow(const KArgs& a, bool ac, int n_q_max, hipStream_t s) {
  const dim3 grid((unsigned)n_q_max * (unsigned)a.heads), block(NT);
  if (ac) hipLaunchKernelGGL((fwd_kernel<D, true, true, 0, U>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((fwd_kernel<D, false, true, 0, U>), grid, block, 0, s, a);
  return hipGetLastError();
}

template <int D, int MODE>
static hipError_t launch_fwd_d(const KArgs& a, bool ac, bool prod, int n_q_max, hipStream_t s) {
  const dim3 grid((unsigned)n_q_max * (unsigned)a.heads), block(NT);
  if (ac) {
    if (prod) hipLaunchKernelGGL((fwd_kernel<D, true, true, MODE>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((fwd_kernel<D, true, false, MODE>), grid, block, 0, s, a);
  } else {
    if (prod) hipLaunchKernelGGL((fwd_kernel<D, false, true, MODE>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((fwd_kernel<D, false, false, MODE>), grid, block, 0, s, a);
  }
  return hipGetLastError();
}

// mode: 0 = o and rem (and the table when one is given), 1 = the attention weights as well, 2 = the table alone
hipError_t launch_fwd(const KArgs& a, int head_dim, bool ac, bool prod, int mode, int n_q_max, hipStream_t s) {
  if (mode == 0 && prod) {
    const int u = used_width(head_dim);
    if (u == 96) return launch_fwd_narrow<128, 96>(a, ac, n_q_max, s);
    if (u == 192) return launch_fwd_narrow<256, 192>(a, ac, n_q_max, s);
  }
  head_dim = kernel_width(head_dim);
  if (mode == 1) {
    if (head_dim == 256) return launch_fwd_d<256, 1>(a, ac, prod, n_q_max, s);
    if (head_dim == 128) return launch_fwd_d<128, 1>(a, ac, prod, n_q_max, s);
    if (head_dim == 64) return launch_fwd_d<64, 1>(a, ac, prod, n_q_max, s);
    return launch_fwd_d<32, 1>(a, ac, prod, n_q_max, s);
  }
  if (mode == 2) {
    if (head_dim == 256) return launch_fwd_d<256, 2>(a, ac, prod, n_q_max, s);
    if (head_dim == 128) return launch_fwd_d<128, 2>(a, ac, prod, n_q_max, s);
    if (head_dim == 64) return launch_fwd_d<64, 2>(a, ac, prod, n_q_max, s);
    return launch_fwd_d<32, 2>(a, ac, prod, n_q_max, s);
  }
  if (head_dim == 256) return launch_fwd_d<256, 0>(a, ac, prod, n_q_max, s);
  if (head_dim == 128) return launch_fwd_d<128, 0>(a, ac, prod, n_q_max, s);
  if (head_dim == 64) return launch_fwd_d<64, 0>(a, ac, prod, n_q_max, s);
  return launch_fwd_d<32, 0>(a, ac, prod, n_q_max, s);
}

}  // inline namespace SBA_ELEM_NS
}  // namespace sba
