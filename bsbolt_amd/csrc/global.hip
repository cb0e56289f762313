// Bit-exact batched ksw_global2 (bsbolt/External/BWA/ksw.c:504-606) for gfx950.
//
// A group of L lanes owns one task and holds the band of the current row: lane
// g keeps positions r = j - beg in [g*C, g*C+C) of H(i-1,j-1) and E(i,j) in
// VGPRs, so the group's width follows n_col = min(qlen, 2w+1), not qlen; rows
// are processed in order.  The band is fixed (beg = max(i-w,0),
// end = min(i+w+1,qlen), ksw.c:530-531).  F along a row is
//   F(j) = max_{beg<=k<j}(M_k - oe_ins + k*e_ins) - (j-1)*e_ins   (j > beg),
//   F(beg) = -inf,
// which equals the reference's sequential recurrence whenever every in-band M
// is finite -- guaranteed by the precondition |tlen - qlen| <= w together with
// the length limits checked per task.
//
// The direction byte of every in-band cell (bits 0-1: source of H, bit 2: E
// extended, bit 5: F extended; ksw.c:551-564) is written to the group's slot in
// a scratch buffer, row-major with n_col = min(qlen, 2w+1) bytes per row, and
// the group walks it back (ksw.c:588-602), writing the CIGAR into the task's
// caller-sized slot.  The walk reads the slot through an LDS window of whole
// rows: the group loads the next rows with all its lanes at once (one HBM
// latency per window, not one per step) and every step then reads LDS.
#include <algorithm>
#include <type_traits>

#include "bsx_internal.h"

namespace bsx {

constexpr int kNegInf = -0x40000000;  // MINUS_INF, ksw.c:490
// dwords of a group's LDS window on its direction bytes (16 KB per block)
template <int L>
constexpr int zwin_dw() { return L < 16 ? 128 : 256; }

// Group scans and reductions on DPP (L = 8, 16, 32 or 64 lanes; values may be
// negative, so lanes without a source keep the identity instead of 0).
template <int L>
__device__ __forceinline__ int g_incl_max(int x, int ident) {
  if (L == 8) {  // quad steps take the lane itself where there is no source (max is idempotent)
    x = max(x, __builtin_amdgcn_update_dpp(ident, x, 0x90, 0xf, 0xf, false));  // quad_perm [0,0,1,2]
    x = max(x, __builtin_amdgcn_update_dpp(ident, x, 0x40, 0xf, 0xf, false));  // quad_perm [0,0,0,1]
    const int q = __builtin_amdgcn_update_dpp(ident, x, 0xFF, 0xf, 0xf, false);  // quad_perm [3,3,3,3]
    // row_shr:4 into banks 1 and 3 only (lanes 4-7 of each 8-lane group)
    return max(x, __builtin_amdgcn_update_dpp(ident, q, 0x114, 0xf, 0xa, false));
  }
  x = max(x, __builtin_amdgcn_update_dpp(ident, x, 0x111, 0xf, 0xf, false));  // row_shr:1
  x = max(x, __builtin_amdgcn_update_dpp(ident, x, 0x112, 0xf, 0xf, false));  // row_shr:2
  x = max(x, __builtin_amdgcn_update_dpp(ident, x, 0x114, 0xf, 0xf, false));  // row_shr:4
  x = max(x, __builtin_amdgcn_update_dpp(ident, x, 0x118, 0xf, 0xf, false));  // row_shr:8
  if (L >= 32) x = max(x, __builtin_amdgcn_update_dpp(ident, x, 0x142, 0xa, 0xf, false));  // row_bcast:15
  if (L >= 64) x = max(x, __builtin_amdgcn_update_dpp(ident, x, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return x;
}

// exclusive prefix max over the group (ident for its first lane)
template <int L>
__device__ __forceinline__ int g_excl_max(int x, int lig, int ident) {
  const int incl = g_incl_max<L>(x, ident);
  const int e = L <= 16 ? __builtin_amdgcn_update_dpp(ident, incl, 0x111, 0xf, 0xf, false)   // row_shr:1
                        : __builtin_amdgcn_update_dpp(ident, incl, 0x138, 0xf, 0xf, false);  // wave_shr:1
  return lig == 0 ? ident : e;
}

// every lane of the group receives the maximum
template <int L>
__device__ __forceinline__ int g_max(int x) {
  if (L <= 16) {
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, true));   // quad_perm [1,0,3,2]
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, true));   // quad_perm [2,3,0,1]
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true));  // row_half_mirror
    if (L == 8) return x;
    return max(x, __builtin_amdgcn_update_dpp(0, x, 0x140, 0xf, 0xf, true));  // row_mirror
  }
  x = g_incl_max<L>(x, INT32_MIN);
  if (L == 64) return __builtin_amdgcn_readlane(x, 63);
  const int a = __builtin_amdgcn_readlane(x, 31), b = __builtin_amdgcn_readlane(x, 63);
  return (int)(threadIdx.x & 63) < 32 ? a : b;
}

// value of the previous lane of the group (lane 0: unused by the callers)
template <int L>
__device__ __forceinline__ int g_prev(int x) {
  return L <= 16 ? __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true)   // row_shr:1
                 : __builtin_amdgcn_update_dpp(0, x, 0x138, 0xf, 0xf, true);  // wave_shr:1
}

// value of the next lane of the group (lane L-1: unused by the callers)
template <int L>
__device__ __forceinline__ int g_next(int x) {
  return L <= 16 ? __builtin_amdgcn_update_dpp(0, x, 0x101, 0xf, 0xf, true)   // row_shl:1
                 : __builtin_amdgcn_update_dpp(0, x, 0x130, 0xf, 0xf, true);  // wave_shl:1
}

// Direction-byte slots per CU, one slot a group.  Launches that run one after
// another share kGlbSlotsOne of them; launches beside each other divide kGlbSlots
// (glb_part).
constexpr int kGlbSlotsOne = 128, kGlbSlots = 192;
// A batch without pair kernels takes the latency of its rows, 115-145 us a bin
// whatever its share of the tasks, so the bins that are seldom empty run beside each
// other, each as a part of its own, and the wide ones follow one another as another
// part.  With all of them on one stream but (16,4) the call took longer (us, so /
// now): 100 bp reads 32,000 tasks 581 / 280, 64,000 685 / 432; 150 bp 32,000 941 / 404,
// 64,000 1143 / 640; 250 bp 32,000 1848 / 874, 64,000 2156 / 1262.
constexpr int kGlbPart[kGlbBins] = {1, 0, 4, 2, 3, 3, 3, 3, 3};
constexpr int kGlbParts = 5;
constexpr int kGlbPartSlots[kGlbParts] = {56, 56, 32, 32, 16};  // slots a part has in any case
// slots per CU that a bin's launch can use
constexpr int glb_most_slots(int b) {
  const int s = 7 * (256 / kGlbShape[b].lanes);
  return s < kGlbSlots ? s : kGlbSlots;
}
constexpr int glb_part_slots() {
  int n = 0;
  for (int k = 0; k < kGlbParts; ++k) n += kGlbPartSlots[k];
  return n;
}
static_assert(glb_part_slots() == kGlbSlots, "slot parts");

// The slots of part k, for launches beside each other: what its largest list can use
// of its own share, and of what the other parts leave of theirs.  Every launch finds
// the same division from the counts.  With fixed shares a batch of one kind ran on a
// third of the slots (131,000 tasks of 150 bp reads, all of half band 7 / 11: 1043 /
// 1217 us, so 721 / 843).
struct GlbSlots { int64_t first, count; };
__device__ __forceinline__ GlbSlots glb_part(const uint32_t* __restrict__ counts, int k, int num_cu) {
  int64_t use[kGlbParts] = {}, part[kGlbParts];
#pragma unroll
  for (int b = 0; b < kGlbBins; ++b) {  // in steps of 32: whole blocks of any bin
    const int64_t n = ((int64_t)counts[b] + 31) / 32 * 32, most = (int64_t)glb_most_slots(b) * num_cu / 32 * 32;
    use[kGlbPart[b]] = max(use[kGlbPart[b]], min(n, most));
  }
  int64_t left = (int64_t)kGlbSlots * num_cu / 32 * 32;
#pragma unroll
  for (int s = 0; s < kGlbParts; ++s) {
    part[s] = min(use[s], (int64_t)kGlbPartSlots[s] * num_cu / 32 * 32);
    left -= part[s];
  }
  GlbSlots p{0, 0};
#pragma unroll
  for (int s = 0; s < kGlbParts; ++s) {
    const int64_t more = min(use[s] - part[s], left);
    left -= more;
    part[s] += more;
    p.first += s < k ? part[s] : 0;
    p.count = s == k ? part[s] : p.count;
  }
  return p;
}

constexpr int kGlbWinDwords = 4096;  // LDS windows of a block

// Block `block` of `blocks` on a bin's list.  first: of the list, or -1 (it follows
// the lists before it); slot0: the blocks' first direction slot.
template <int L, int C>
__device__ __forceinline__ void glb_run(const GlbArgs& A, const GlbWork& W, int bin, uint32_t block, uint32_t blocks,
                                        int64_t slot0, int64_t first, uint32_t* __restrict__ zwin_all,
                                        uint2* __restrict__ s_prof) {
  if (block >= blocks) return;  // uniform over the block
  const int lane = threadIdx.x & 63;
  const int lig = lane & (L - 1);
  const int base = lig * C;
  const int group = (int)block * (256 / L) + threadIdx.x / L;
  int64_t lbase = first;
  if (first < 0) {
    lbase = 0;
    for (int b = 0; b < bin; ++b) lbase += W.counts[b];
  }
  const int32_t* __restrict__ list = W.list + lbase;
  const uint32_t nlist = W.counts[bin];
  uint8_t* __restrict__ z = W.z + (slot0 + group) * W.zslot;
  constexpr int ZW = zwin_dw<L>();
  static_assert(256 / L * ZW <= kGlbWinDwords, "LDS windows");
  uint32_t* __restrict__ zwin = zwin_all + threadIdx.x / L * ZW;
  const int oe_del = A.o_del + A.e_del, oe_ins = A.o_ins + A.e_ins;
  const int e_del = A.e_del, e_ins = A.e_ins;

  // profile words by query code (code 4 for N and positions past the query),
  // for the position entering the band on each row
  if (threadIdx.x < 5) s_prof[threadIdx.x] = make_uint2(A.prof_lo[threadIdx.x], (uint32_t)A.prof_hi[threadIdx.x]);
  __syncthreads();
  // Every group's first task is its own number; only when the list is longer
  // than the grid do groups fetch more (each wave's fetch is a device atomic on
  // one address, ~10 ns apiece serialised, so an empty or short list has none).
  const uint32_t groups = blocks * (256 / L);
  uint32_t idx = (uint32_t)group;
  while (idx < nlist) {
    const int task = list[idx];
    const int qlen = A.qlen[task], tlen = A.tlen[task];
    // a band wider than both sequences is the same band (beg = 0, end = qlen
    // on every row): clamping keeps i + w + 1 and the like in int range
    const int w = min(A.w[task], max(qlen, tlen));
    const uint64_t qoff = A.q_off[task], toff = A.t_off[task];
    const int ncol = qlen < 2 * w + 1 ? qlen : 2 * w + 1;
    const bool want_cigar = A.cigar != nullptr;

    // Lanes hold band positions r = j - beg (lane g: r in [g*C, g*C+C)), so a
    // group needs L*C >= n_col columns whatever qlen is.  Row i works on
    // positions [0, end-beg).  While beg stays 0 (i < w) the state moves one
    // position right each row (H(i,j-1) becomes the next row's H(i-1,j-1));
    // once beg advances with i, position r of row i+1 is column beg+1+r, so
    // H stays in place and E and the query profile move one position left, the
    // top position taking query[beg+1+L*C-1].
    constexpr int LC = L * C;
    int G[C], E[C];
    uint32_t plo[C];
    int phi[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int j = base + c;  // row 0: beg = 0
      const int qc = j < qlen ? (int)A.query[qoff + j] : 4;
      uint32_t lo = A.prof_lo[4];
      int hi = A.prof_hi[4];
      if (qc == 0) { lo = A.prof_lo[0]; hi = A.prof_hi[0]; }
      if (qc == 1) { lo = A.prof_lo[1]; hi = A.prof_hi[1]; }
      if (qc == 2) { lo = A.prof_lo[2]; hi = A.prof_hi[2]; }
      if (qc == 3) { lo = A.prof_lo[3]; hi = A.prof_hi[3]; }
      plo[c] = lo;
      phi[c] = hi;
      // row -1 (ksw.c:522-525)
      G[c] = j == 0 ? 0 : (j <= w ? -(A.o_ins + e_ins * j) : kNegInf);
      E[c] = kNegInf;
    }
    int hq = qlen <= w ? -(A.o_ins + e_ins * qlen) : kNegInf;  // eh[qlen].h

    // Per-row codes, two rows per lane and 2L rows per chunk: byte 0 the
    // target base of row rho, byte 1 the query base entering the top position
    // after row rho (column rho + L*C - w; 4 outside the query).  The raw bytes
    // of the next chunk are loaded one chunk ahead from clamped (in-bounds)
    // addresses, unconditionally, so nothing waits for them before the next
    // refill combines them.
    uint32_t raw[4];
    auto load_raw = [&](int cb) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int rho = cb + 2 * lig + k;
        const int jq = rho + LC - w;
        raw[2 * k] = A.target[toff + (rho < tlen ? rho : tlen - 1)];
        raw[2 * k + 1] = A.query[qoff + (jq < 0 ? 0 : (jq < qlen ? jq : qlen - 1))];
      }
    };
    auto combine = [&](int cb) -> uint32_t {
      uint32_t v = 0;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int rho = cb + 2 * lig + k;
        const int jq = rho + LC - w;
        const uint32_t tb = rho < tlen ? raw[2 * k] : 0u;
        const uint32_t qb = (jq >= 0 && jq < qlen) ? raw[2 * k + 1] : 4u;
        v |= (tb | qb << 8) << (16 * k);
      }
      return v;
    };
    load_raw(0);
    uint32_t ch = combine(0);
    load_raw(2 * L);
    int cb = 0;
    for (int i = 0; i < tlen; ++i) {
      int tr = i - cb;
      if (tr >= 2 * L) {
        cb = i;
        tr = 0;
        ch = combine(i);
        load_raw(i + 2 * L);
      }
      const uint32_t wd = (uint32_t)__shfl((int)ch, tr >> 1, L) >> (16 * (tr & 1));
      const int t = (int)(wd & 0xffu), qn = (int)((wd >> 8) & 0xffu);
      const int beg = i > w ? i - w : 0;
      const int end = i + w + 1 < qlen ? i + w + 1 : qlen;
      const int nb = end - beg;  // in-band positions [0, nb)
      const int h1p = beg == 0 ? -(A.o_del + e_del * (i + 1)) : kNegInf;

      int M[C], ex[C];
      int run = INT32_MIN;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int r = base + c;
        const bool inb = r < nb;
        const int s = t < 4 ? __builtin_amdgcn_sbfe((int)plo[c], 8 * (t & 3), 8) : phi[c];  // signed byte t
        const int mm = G[c] + s;
        M[c] = mm;
        const int key = inb ? mm - oe_ins + r * e_ins : INT32_MIN;
        ex[c] = run;
        run = max(run, key);
      }
      const int lex = g_excl_max<L>(run, lig, INT32_MIN);
      int h[C];
      int h1c = INT32_MIN;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int r = base + c;
        const bool inb = r < nb;
        const int x = max(ex[c], lex);
        // positions without an in-band predecessor get -inf (this also keeps
        // the subtraction away from INT32_MIN on out-of-band positions)
        const int f = (r == 0 || x == INT32_MIN) ? kNegInf : x - (r - 1) * e_ins;
        const int mm = M[c], e = E[c];
        int d = mm >= e ? 0 : 1;
        int hh = mm >= e ? mm : e;
        if (!(hh >= f)) { d = 2; hh = f; }
        h[c] = hh;
        const int od = mm - oe_del, ee = e - e_del;
        if (ee > od) d |= 1 << 2;
        const int ne = ee > od ? ee : od;
        const int oi = mm - oe_ins, ff = f - e_ins;
        if (ff > oi) d |= 2 << 4;
        // out-of-band positions hold E = -inf: the position end (eh[end].e,
        // ksw.c:575) and every position that enters the band later
        E[c] = inb ? ne : kNegInf;
        if (want_cigar && inb) z[(int64_t)i * ncol + r] = (uint8_t)d;
        if (r == nb - 1) h1c = hh;
      }
      if (i >= w) {  // beg(i+1) = beg(i) + 1
#pragma unroll
        for (int c = 0; c < C; ++c) G[c] = h[c];
        const int e0 = g_next<L>(E[0]);
        const uint32_t p0 = (uint32_t)g_next<L>((int)plo[0]);
        const int q0 = g_next<L>(phi[0]);
#pragma unroll
        for (int c = 0; c + 1 < C; ++c) {
          E[c] = E[c + 1];
          plo[c] = plo[c + 1];
          phi[c] = phi[c + 1];
        }
        const uint2 pq = s_prof[qn < 4 ? qn : 4];
        const bool top = lig == L - 1;
        E[C - 1] = top ? kNegInf : e0;
        plo[C - 1] = top ? pq.x : p0;
        phi[C - 1] = top ? (int)pq.y : q0;
      } else {  // beg stays 0: H(i,j-1) moves to position j, eh[0].h = h1p
        const int hprev = g_prev<L>(h[C - 1]);
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const int r = base + c;
          const int left = c == 0 ? hprev : h[c - 1];
          G[c] = r == 0 ? h1p : left;
        }
      }
      h1c = g_max<L>(h1c);
      if (end == qlen) hq = h1c;  // eh[end] = {h1, -inf} with end == qlen
    }
    if (lig == 0) {
      if (A.score) A.score[task] = hq;
    }
    if (want_cigar) {
      // The slot was written by every lane of this group; the walk below reads
      // it back.  All lanes of the group run the walk (the loop is uniform over
      // the group; lanes outside this task's group are not involved), so no
      // lane-divergent loop is left in front of the next fetch broadcast; only
      // lane 0 stores.  Runs of equal ops are merged in registers, which gives
      // the CIGAR push_cigar builds (ksw.c:492-502).
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
      uint32_t* cg = A.cigar + (int64_t)task * A.cigar_slot;
      const int64_t cap = A.cigar_slot;
      int n = 0, state = 0, run_op = -1, run_len = 0;
      bool over = false;
      auto emit = [&]() {
        if (run_op < 0) return;
        if (n < cap) {
          if (lig == 0) cg[n] = (uint32_t)run_len << 4 | (uint32_t)run_op;
          ++n;
        } else {
          over = true;
        }
      };
      auto push = [&](int op, int len) {
        if (op == run_op) {
          run_len += len;
        } else {
          emit();
          run_op = op;
          run_len = len;
        }
      };
      int i = tlen - 1;
      int k = (i + w + 1 < qlen ? i + w + 1 : qlen) - 1;
      // LDS window: rows [wlo, whi] of the slot, from byte wbase (a dword
      // boundary) on; rows per window so that they fit with the alignment slack
      const int wrows = (4 * ZW - 3) / ncol;
      const uint32_t* __restrict__ zw = (const uint32_t*)z;
      int wlo = 1, whi = 0;
      uint32_t wbase = 0;
      // Offsets in the slot fit 32 bits: n_col <= 2048 and tlen <= 65536 are
      // checked per task.  Every lane computes the same (i, k, state), so the
      // step needs no cross-lane operation.
      while (i >= 0 && k >= 0) {
        const int kc = k - (i > w ? i - w : 0);
        if ((unsigned)kc >= (unsigned)ncol) {  // cannot happen under the preconditions; never read outside the slot
          over = true;
          break;
        }
        const uint32_t zi = (uint32_t)i * (uint32_t)ncol + (uint32_t)kc;
        int zb;
        if (wrows >= 1) {
          // refill: rows [i - wrows + 1, i], every lane loading; all groups of the
          // wave at once when one needs it, as the whole wave waits for each round
          // trip to memory (8 groups on their own and a dword at a time: 200 us
          // instead of 116 for the 8x2 bin of 9,319 tasks of 150 bp reads)
          if (__any(i < wlo || i > whi)) {
            const int r0 = i - wrows + 1 > 0 ? i - wrows + 1 : 0;
            const uint32_t d0 = ((uint32_t)r0 * (uint32_t)ncol) >> 2;
            const uint32_t d1 = ((uint32_t)(i + 1) * (uint32_t)ncol - 1u) >> 2;
            __builtin_amdgcn_wave_barrier();
            uint32_t v[ZW / L];  // every load in flight before the first is stored
#pragma unroll
            for (int u = 0; u < ZW / L; ++u) v[u] = zw[min(d0 + lig + u * L, d1)];
#pragma unroll
            for (int u = 0; u < ZW / L; ++u) zwin[lig + u * L] = v[u];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            wlo = r0; whi = i; wbase = d0 << 2;
          }
          const uint32_t q = zi - wbase;  // every lane reads the same byte
          zb = (int)__builtin_amdgcn_ubfe(zwin[q >> 2], 8 * (q & 3), 8);
        } else {
          zb = z[zi];  // every lane loads the same byte
        }
        state = zb >> (state << 1) & 3;
        // 0: M, i-1 and k-1; 1: D, i-1; otherwise I, k-1 (ksw.c:596-598)
        const int op = state == 0 ? 0 : (state == 1 ? 2 : 1);
        i -= state <= 1 ? 1 : 0;
        k -= state != 1 ? 1 : 0;
        if (op != run_op) {  // the run of run_op ends (there is none before the first step)
          emit();
          run_op = op;
          run_len = 1;
        } else {
          ++run_len;
        }
      }
      if (i >= 0) push(2, i + 1);
      if (k >= 0) push(1, k + 1);
      emit();
      if (over) {
        if (lig == 0) {
          A.n_cigar[task] = -1;
          atomicAdd(&W.err[2], 1);
        }
      } else {
        // reverse in place (the walk produced the ops from the end); uniform loop
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        for (int a = 0, b = n - 1; a < b; ++a, --b) {
          const uint32_t ta = cg[a], tb = cg[b];
          if (lig == 0) { cg[a] = tb; cg[b] = ta; }
        }
        if (lig == 0) A.n_cigar[task] = n;
      }
    } else if (A.n_cigar && lig == 0) {
      A.n_cigar[task] = 0;
    }
    if (groups >= nlist) break;  // uniform over the grid
    // Branch-free fetch: every lane issues the atomic (only lane 0 of the group
    // adds 1; the compiler folds it into one atomic per wave).  No lane-divergent
    // region may precede the broadcast: with `if (lig == 0)` around the atomic
    // the compiler can give the other lanes a loop of their own that reaches
    // the broadcast without lane 0's new value, and they never leave it.
    const uint32_t mine = atomicAdd(W.fetch + bin, lig == 0 ? 1u : 0u);
    idx = groups + __shfl(mine, 0, L);
  }
}

// part: the launch's among those beside each other, or -1 (it has kGlbSlotsOne
// slots per CU)
template <int B>
__global__ void __launch_bounds__(256) glb_kernel(GlbArgs A, GlbWork W, int part, int num_cu, int64_t first) {
  constexpr int L = kGlbShape[B].lanes, C = kGlbShape[B].cols;
  __shared__ uint32_t zwin[kGlbWinDwords];
  __shared__ uint2 s_prof[5];
  const GlbSlots p = part < 0 ? GlbSlots{0, (int64_t)kGlbSlotsOne * num_cu} : glb_part(W.counts, part, num_cu);
  glb_run<L, C>(A, W, B, blockIdx.x, min((uint32_t)(p.count / (256 / L)), gridDim.x), p.first, first, zwin, s_prof);
}

// Two bins in one launch, beside each other: bands of 25-32 are few in a read set's
// batch, and a launch of their own in front of another adds its latency to the call
// (32,000 tasks of 100 bp reads: 312 us on the stream of (8,3), 280 so).
template <int B1, int B2>
__global__ void __launch_bounds__(256) glb_two_kernel(GlbArgs A, GlbWork W, int num_cu) {
  constexpr int L1 = kGlbShape[B1].lanes, C1 = kGlbShape[B1].cols, L2 = kGlbShape[B2].lanes, C2 = kGlbShape[B2].cols;
  __shared__ uint32_t zwin[kGlbWinDwords];
  __shared__ uint2 s_prof[5];
  const GlbSlots p = glb_part(W.counts, kGlbPart[B1], num_cu), q = glb_part(W.counts, kGlbPart[B2], num_cu);
  const uint32_t np = min((uint32_t)(p.count / (256 / L1)), gridDim.x);
  const uint32_t nq = min((uint32_t)(q.count / (256 / L2)), gridDim.x - np);
  if (blockIdx.x < np) glb_run<L1, C1>(A, W, B1, blockIdx.x, np, p.first, -1, zwin, s_prof);
  else glb_run<L2, C2>(A, W, B2, blockIdx.x - np, nq, q.first, -1, zwin, s_prof);
}

// Bin of the two-tasks-per-lane kernel for a valid task, or -1: the whole band
// (not clipped to the query) fits, and every score fits its 16 bits.
__device__ __forceinline__ int glb_pair_bin_of(const GlbArgs& A, int ql, int tl, int w) {
  if (!A.pair || tl > kGlbPairTlen) return -1;
  const int width = 2 * min(w, max(ql, tl)) + 1;
  const int64_t range = (int64_t)(ql + tl) * (A.pen_max + max(A.e_del, A.e_ins) + A.mat_max) + A.o_del + A.o_ins;
  if (range > kGlbPairRange) return -1;
#pragma unroll
  for (int b = 0; b < kGlbPairBins; ++b)
    if (width <= kGlbPairCols[b]) return kGlbBins + b;
  return -1;
}

__global__ void __launch_bounds__(256)
glb_bin_count_kernel(GlbArgs A, GlbWork W) {
  __shared__ uint32_t hist[kGlbAllBins], khist[kGlbKeys];
  if (threadIdx.x < kGlbAllBins) hist[threadIdx.x] = 0;
  for (int k = threadIdx.x; k < kGlbKeys; k += blockDim.x) khist[k] = 0;
  __syncthreads();
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < A.n;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int ql = A.qlen[t], tl = A.tlen[t], w = A.w[t];
    int b;
    const bool ok = glb_task_ok(A, W, t);
    if (!ok) {
      b = 0xff;
      atomicAdd(&W.err[0], 1);
      atomicMin(&W.err[1], (int)t);
    } else {
      const int pb = glb_pair_bin_of(A, ql, tl, w);
      b = pb >= 0 ? pb : glb_bin_of((int)min((int64_t)ql, 2 * (int64_t)w + 1));  // a group holds n_col positions
      atomicAdd(&hist[b], 1u);
      atomicAdd(&khist[glb_key(b, tl)], 1u);
    }
    W.bin_of[t] = (uint8_t)b;
  }
  __syncthreads();
  if (threadIdx.x < kGlbAllBins && hist[threadIdx.x]) atomicAdd(&W.counts[threadIdx.x], hist[threadIdx.x]);
  for (int k = threadIdx.x; k < kGlbKeys; k += blockDim.x)
    if (khist[k]) atomicAdd(&W.kcount[k], khist[k]);
}

// One block: the start of every bucket's run in the lists.
__global__ void __launch_bounds__(1024) glb_bin_offset_kernel(GlbWork W) {
  __shared__ uint32_t part[1024];
  constexpr int PER = (kGlbKeys + 1023) / 1024;
  const int k0 = threadIdx.x * PER;
  uint32_t s = 0;
  for (int k = k0; k < k0 + PER && k < kGlbKeys; ++k) s += W.kcount[k];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {
    const uint32_t x = (int)threadIdx.x >= d ? part[threadIdx.x - d] : 0u;
    __syncthreads();
    part[threadIdx.x] += x;
    __syncthreads();
  }
  uint32_t at = part[threadIdx.x] - s;
  for (int k = k0; k < k0 + PER && k < kGlbKeys; ++k) {
    W.kcursor[k] = at;
    at += W.kcount[k];
  }
}

// Each block counts its contiguous range of tasks per bin and bucket in LDS and
// reserves each run with one device atomic (a same-address device atomic per
// task serialises the whole batch on a few addresses).
__global__ void __launch_bounds__(256)
glb_bin_scatter_kernel(GlbArgs A, GlbWork W, int64_t per_block) {
  __shared__ uint32_t cur[kGlbKeys];
  const int64_t t0 = (int64_t)blockIdx.x * per_block, t1 = min(A.n, t0 + per_block);
  for (int k = threadIdx.x; k < kGlbKeys; k += blockDim.x) cur[k] = 0;
  __syncthreads();
  for (int64_t t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
    const int b = W.bin_of[t];
    if (b != 0xff) atomicAdd(&cur[glb_key(b, A.tlen[t])], 1u);
  }
  __syncthreads();
  for (int x = threadIdx.x; x < kGlbKeys; x += blockDim.x)
    if (cur[x]) cur[x] = atomicAdd(&W.kcursor[x], cur[x]);
  __syncthreads();
  for (int64_t t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
    const int b = W.bin_of[t];
    if (b != 0xff) W.list[atomicAdd(&cur[glb_key(b, A.tlen[t])], 1u)] = (int32_t)t;
  }
}

static_assert(kGlbAllBins <= kCountSlots && kGlbAllBins <= 64, "CIGAR bin counters");
__global__ void __launch_bounds__(1024) glb_reset_kernel(GlbWork W) {
  for (int k = threadIdx.x; k < kGlbCounterWords; k += blockDim.x) W.counts[k] = 0;
  __syncthreads();
  if (threadIdx.x == 0) W.err[1] = 0x7fffffff;
}

__global__ void glb_clear_kernel(uint32_t* used) { *used = 0; }

// A task per lane; a wave reserves the words of its tasks with one atomic.  CIGARs
// of more than kGatherOps words stay in their slots, so the sum fits 32 bits.
constexpr int kGatherOps = 4096;
__global__ void __launch_bounds__(256)
glb_gather_kernel(const int32_t* __restrict__ score, const int32_t* __restrict__ n_cigar,
                  const uint32_t* __restrict__ cigar, const uint8_t* __restrict__ bin_of, int n, int64_t slot,
                  int32_t* __restrict__ rec, uint32_t* __restrict__ words, uint32_t room, uint32_t* __restrict__ used) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63;
  const bool ok = k < n && bin_of[k] != 0xff;
  const int nc = ok && n_cigar ? n_cigar[k] : 0;
  const int have = cigar && nc > 0 && nc <= kGatherOps ? nc : 0;
  int sum = have;  // inclusive sum over the wave
  for (int d = 1; d < 64; d <<= 1) {
    const int x = __shfl_up(sum, d);
    sum += lane >= d ? x : 0;
  }
  uint32_t first = 0;
  if (lane == 63 && sum > 0) first = atomicAdd(used, (uint32_t)sum);
  first = (uint32_t)__shfl((int)first, 63) + (uint32_t)(sum - have);
  const bool fits = have > 0 && first <= room && (uint32_t)have <= room - first;
  if (k < n) *(int4*)(rec + 4 * (int64_t)k) = make_int4(ok ? score[k] : 0, nc, fits ? (int)first : -1, ok ? 1 : 0);
  if (fits)
    for (int x = 0; x < have; ++x) words[first + x] = cigar[(int64_t)k * slot + x];
}

hipError_t launch_glb_gather(const int32_t* score, const int32_t* n_cigar, const uint32_t* cigar, const uint8_t* bin_of,
                             int n, int64_t slot, int32_t* rec, uint32_t* words, uint32_t room, uint32_t* used,
                             bool clear, hipStream_t st) {
  if (clear) hipLaunchKernelGGL(glb_clear_kernel, dim3(1), dim3(1), 0, st, used);
  hipLaunchKernelGGL(glb_gather_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, score, n_cigar, cigar,
                     bin_of, n, slot, rec, words, room, used);
  return hipGetLastError();
}

int64_t glb_groups(int num_cu, bool side) { return (int64_t)num_cu * (side ? kGlbSlots : kGlbSlotsOne); }

template <int B>
static int64_t glb_blocks(const GlbArgs& a, int num_cu, int most) {
  constexpr int L = kGlbShape[B].lanes;
  return std::min<int64_t>((int64_t)std::min(glb_most_slots(B), most) * num_cu / (256 / L), (a.n * L + 255) / 256);
}

template <int B>
static void glb_launch_bin(const GlbArgs& a, const GlbWork& w, int num_cu, hipStream_t st, int part = -1,
                           int64_t first = -1) {
  const int64_t blocks = glb_blocks<B>(a, num_cu, part < 0 ? kGlbSlotsOne : kGlbSlots);
  hipLaunchKernelGGL(glb_kernel<B>, dim3((unsigned)blocks), dim3(256), 0, st, a, w, part, num_cu, first);
}

hipError_t launch_global_impl(GlbArgs a, GlbWork w, int num_cu, hipStream_t st) {
  w.pair_bytes = glb_pair_bytes(num_cu);
  a.pair = a.n >= kGlbPairMinTasks && (!a.cigar || w.zpair);
  hipLaunchKernelGGL(glb_reset_kernel, dim3(1), dim3(1024), 0, st, w);
  if (a.n <= 0) return hipGetLastError();
  if (a.n <= std::min<int64_t>(kGlbDirectMaxTasks, (int64_t)num_cu * kGlbSlotsOne)) {
    launch_glb_direct(a, w, st);
    static_assert(kGlbRest == 3, "rest bins");
    glb_launch_bin<kGlbRestBin[0]>(a, w, num_cu, st, -1, 0);
    glb_launch_bin<kGlbRestBin[1]>(a, w, num_cu, st, -1, a.n);
    glb_launch_bin<kGlbRestBin[2]>(a, w, num_cu, st, -1, 2 * a.n);
    return hipGetLastError();
  }
  // each block ends with a global atomic per non-empty bucket
  const int64_t blocks = std::min<int64_t>((a.n + 255) / 256, (int64_t)num_cu * 4);
  hipLaunchKernelGGL(glb_bin_count_kernel, dim3((unsigned)blocks), dim3(256), 0, st, a, w);
  hipLaunchKernelGGL(glb_bin_offset_kernel, dim3(1), dim3(1024), 0, st, w);
  hipLaunchKernelGGL(glb_bin_scatter_kernel, dim3((unsigned)blocks), dim3(256), 0, st, a, w, (a.n + blocks - 1) / blocks);
  if (a.pair) {
    // Only bin 4 (bands of 65-128) is likely to hold tasks beside the pair
    // bins.  The others go ahead of everything, 5 us each while the chip is
    // empty: behind a pair kernel, or beside one, even an empty launch waits
    // until there is room for its blocks (0.5-1.3 ms measured).
    glb_launch_bin<8>(a, w, num_cu, st);
    glb_launch_bin<7>(a, w, num_cu, st);
    glb_launch_bin<6>(a, w, num_cu, st);
    glb_launch_bin<5>(a, w, num_cu, st);
    glb_launch_bin<3>(a, w, num_cu, st);
    glb_launch_bin<2>(a, w, num_cu, st);
    glb_launch_bin<1>(a, w, num_cu, st);
    glb_launch_bin<0>(a, w, num_cu, st);
    ss_fork(w.ss, st);
    glb_launch_bin<4>(a, w, num_cu, pick_stream(w.ss, st, 3));
    launch_glb_pair(a, w, num_cu, st);
  } else if (w.ss) {
    ss_fork(w.ss, st);  // side streams start after the scatter
    glb_launch_bin<1>(a, w, num_cu, st, kGlbPart[1]);
    hipLaunchKernelGGL((glb_two_kernel<2, 3>),
                       dim3((unsigned)(glb_blocks<2>(a, num_cu, kGlbSlots) + glb_blocks<3>(a, num_cu, kGlbSlots))),
                       dim3(256), 0, pick_stream(w.ss, st, 2), a, w, num_cu);
    glb_launch_bin<0>(a, w, num_cu, pick_stream(w.ss, st, 1), kGlbPart[0]);
    const hipStream_t s3 = pick_stream(w.ss, st, 3);
    glb_launch_bin<4>(a, w, num_cu, s3, kGlbPart[4]);
    glb_launch_bin<8>(a, w, num_cu, s3, kGlbPart[8]);
    glb_launch_bin<7>(a, w, num_cu, s3, kGlbPart[7]);
    glb_launch_bin<6>(a, w, num_cu, s3, kGlbPart[6]);
    glb_launch_bin<5>(a, w, num_cu, s3, kGlbPart[5]);
  } else {
    glb_launch_bin<1>(a, w, num_cu, st);
    glb_launch_bin<2>(a, w, num_cu, st);
    glb_launch_bin<3>(a, w, num_cu, st);
    glb_launch_bin<0>(a, w, num_cu, st);
    glb_launch_bin<4>(a, w, num_cu, st);
    glb_launch_bin<8>(a, w, num_cu, st);
    glb_launch_bin<7>(a, w, num_cu, st);
    glb_launch_bin<6>(a, w, num_cu, st);
    glb_launch_bin<5>(a, w, num_cu, st);
  }
  ss_join(w.ss, st);  // the call's stream waits for the side streams
  return hipGetLastError();
}

}  // namespace bsx
