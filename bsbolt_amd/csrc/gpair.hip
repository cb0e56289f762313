// Two-tasks-per-lane form of the bit-exact ksw_global2
// (bsbolt/External/BWA/ksw.c:504-606) for narrow bands (2w+1 <= 63).
//
// Each lane of a wave owns two whole tasks, one in each 16-bit half of its
// registers, and runs the reference's row loop inside the lane.  Position r of
// a task is column j = i - w + r of row i, r in [0, 2w].  H(i,j) stays at its
// position for the next row (it is the diagonal predecessor there), E and the
// query move one position left; E lands there by the choice of the register it
// is written to, and the query's codes shift one byte a row.
//
// Every row works on all positions with no masks:
//  - columns before 0: -inf, except column -1, whose E starts at
//    -(o_del + e_del) and runs down by e_del a row, which makes its H the
//    reference's first-column values (ksw.c:532); F is made from M only, so
//    nothing else of it reaches column 0 (ksw.c:546-565).
//  - columns past the query: nothing flows back from them.
//  - positions past 2w: F and H flow into them but only E flows out, and the E
//    that enters position 2w is set to -inf, as ksw.c:575 leaves it.
// Values are kept minus a per column (a = max(mat)): the diagonal step then
// subtracts the cell's penalty a - s >= 0 and the insertion costs gain a, so
// all of them are <= 0 and -inf is a floor that saturating subtraction cannot
// leave.  (qlen + tlen) * (largest penalty + largest gap extension + a) + the
// gap openings bounds their size and is checked per task against 16 bits.
//
// Directions.  The four decisions of a cell (ksw.c:548-563) are the signs of
// M - E, max(M,E) - F, and of the open minus the extended value of E and F;
// they are stored as a nibble, 8 cells to a dword, one row of a task after the
// other, the 64 lanes' rows side by side.  The walk (ksw.c:588-602) then takes
// the rows from the last to the first, all lanes one row per step and the next
// rows' loads in flight; an insertion step stays in its row.
//
// 24 packed instructions per cell of two tasks (11 of them the recurrences, 12
// the directions) against ~250 per row of 16-24 cells for 8 tasks in the group
// kernels.  596,416 tasks of 150 bp reads: 511M wave instructions, 0.9 ms of issue,
// of the call's 2.00 ms (4.81 with the group kernels); in order the five kernels
// take 3.1 ms, each mostly the latency of a wave or two per SIMD.  Register budgets
// are set so that no vector register spills (a spilled load in the row loop waits
// for the stores before it); uniform values of the walk do, 39 (NC = 15) to 231 (63),
// into vector registers.
#include <algorithm>

#include "bsx_internal.h"
#include "ext_common.h"
#include "packed.h"

namespace bsx {

constexpr uint32_t kFloor = 0x8ad0;  // -30000: -inf

// waves per SIMD the register budget leaves room for
constexpr int gpair_min_waves(int NC) { return NC <= 23 ? 3 : NC <= 47 ? 2 : 1; }

template <int NC>
__global__ void __launch_bounds__(64, gpair_min_waves(NC))
glb_pair_kernel(GlbArgs A, GlbWork W, int bin) {
  constexpr int NW = (NC + 7) / 8;      // direction dwords of a row
  constexpr int NQ = (NC + 3) / 4;      // query-code dwords of a row
  constexpr int TOP0 = glb_pair_top(NC);  // lowest top position (2w) of the bin
  __shared__ uint2 trow[8];  // penalties of a target code: query codes 0..3, and N
  const int lane = threadIdx.x;
  uint32_t lbase = 0;
  for (int b = 0; b < bin; ++b) lbase += W.counts[b];
  const uint32_t nlist = W.counts[bin];
  if (nlist == 0) return;  // uniform over the grid
  if (lane < 8) {
    const int t = lane < 5 ? lane : 4;
    uint32_t lo = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int s = t < 4 ? sbyte(A.prof_lo[q], t) : A.prof_hi[q];
      lo |= (uint32_t)((A.mat_max - s) & 0xff) << (8 * q);
    }
    const int sn = t < 4 ? sbyte(A.prof_lo[4], t) : A.prof_hi[4];
    trow[lane] = make_uint2(lo, (uint32_t)((A.mat_max - sn) & 0xff) * 0x01010101u);
  }
  __syncthreads();
  const bool want_cigar = A.cigar != nullptr;
  // this wave's part of the scratch: room for 128 tasks of the list's first
  // (longest) target; the waves past the last part leave
  uint32_t* __restrict__ zreg = nullptr;
  if (want_cigar) {
    const int64_t region = glb_pair_region(NC, glb_pair_rows(A.tlen[W.list[lbase]]));
    const int64_t at = (int64_t)blockIdx.x * region;
    if (at + region > W.pair_bytes && blockIdx.x > 0) return;
    zreg = (uint32_t*)(W.zpair + at);
  }
  const u16x2 oe_del = splat((uint32_t)(A.o_del + A.e_del)), e_del = splat((uint32_t)A.e_del);
  const u16x2 oe_ins = splat((uint32_t)(A.o_ins + A.e_ins + A.mat_max)), e_ins = splat((uint32_t)(A.e_ins + A.mat_max));
  const u16x2 kNone = splat(kFloor);

  for (;;) {
    // Branch-free fetch of the next 128 tasks: every lane issues the atomic and
    // only lane 0 adds; the value is read from lane 0 by all.
    const uint32_t mine = atomicAdd(W.fetch + bin, lane == 0 ? 1u : 0u);
    const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)mine) * 128u;
    if (first >= nlist) break;

    int task[2], qlen[2], tlen[2], w[2];
    bool have[2];
    DwordSeq ts[2], qs[2];
    int qd[2], qb[2];
    uint32_t qw[2][NQ + 1];  // query codes of the positions, and the dword moving in
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t p = first + 2u * lane + k;
      have[k] = p < nlist;
      task[k] = W.list[lbase + (have[k] ? p : first)];
      qlen[k] = A.qlen[task[k]];
      tlen[k] = A.tlen[task[k]];
      w[k] = min(A.w[task[k]], max(qlen[k], tlen[k]));
      ts[k].set(A.target + A.t_off[task[k]], tlen[k]);
      qs[k].set(A.query + A.q_off[task[k]], qlen[k]);
      const int sh = qs[k].sh - w[k];  // byte of position 0 relative to the first dword
      qd[k] = sh >> 2;
      qb[k] = sh & 3;
      uint32_t a0 = qs[k].at(qd[k]);
#pragma unroll
      for (int m = 0; m <= NQ; ++m) {
        const uint32_t a1 = qs[k].at(qd[k] + m + 1);
        qw[k][m] = __builtin_amdgcn_alignbyte(a1, a0, (uint32_t)qb[k]);
        a0 = a1;
      }
      if (!have[k]) tlen[k] = 0;
    }
    // the dwords after the window, one refill (4 rows) ahead
    uint32_t qn0[2], qn1[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) { qn0[k] = qs[k].at(qd[k] + NQ + 1); qn1[k] = qs[k].at(qd[k] + NQ + 2); }
    uint32_t tw0[2], tw1[2], tw2[2], t4[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) { tw0[k] = ts[k].at(0); tw1[k] = ts[k].at(1); tw2[k] = ts[k].at(2); t4[k] = 0; }

    // row -1 (ksw.c:522-525): column j at position w + j
    u16x2 G[NC], E[NC];
    {
      const u16x2 wv = pk2(w[0], w[1]);
      u16x2 ramp = splat(0u) - splat((uint32_t)(A.o_ins));
#pragma unroll
      for (int r = 0; r < NC; ++r) {
        const u16x2 d = splat((uint32_t)r) - wv;  // column of the position
        const uint32_t neg = negmask(d), zero = negmask(d - splat(1u)) & ~neg;
        const uint32_t minus1 = negmask(d) & ~negmask(d + splat(1u));
        ramp = ssat(ramp, pk(pku(e_ins) & ~(neg | zero)));
        G[r] = pk((pku(ramp) & ~(neg | zero)) | (pku(kNone) & neg));
        E[r] = sel(minus1, splat(0u) - oe_del, kNone);
      }
    }
    // E entering a task's top position 2w is -inf; the bin's tops are the even
    // positions from TOP0 on
    u16x2 cap[(NC - 1 - TOP0) / 2];
#pragma unroll
    for (int m = 0; m < (NC - 1 - TOP0) / 2; ++m)
      cap[m] = pk2(2 * w[0] == TOP0 + 2 * m ? (int)kFloor : 0x7fff, 2 * w[1] == TOP0 + 2 * m ? (int)kFloor : 0x7fff);
    int tmax = max(tlen[0], tlen[1]);
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) tmax = max(tmax, __shfl_xor(tmax, m));
    tmax = __builtin_amdgcn_readfirstlane(tmax);
    const u16x2 rf = pk2(qlen[0] - tlen[0] + w[0], qlen[1] - tlen[1] + w[1]);  // position of the last cell
    u16x2 fin = splat(0u);

    // Four rows a turn, with every store unconditional (rows past a task's end
    // stay inside the region): the count of memory operations between a load
    // and its use is then fixed, and no load waits for the stores behind it.
    for (int i0 = 0; i0 < tmax; i0 += 4) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        t4[k] = __builtin_amdgcn_alignbyte(tw1[k], tw0[k], (uint32_t)ts[k].sh);
        tw0[k] = tw1[k];
        tw1[k] = tw2[k];
        tw2[k] = ts[k].at((i0 >> 2) + 3);
        if (i0 > 0) {
          qw[k][NQ] = __builtin_amdgcn_alignbyte(qn1[k], qn0[k], (uint32_t)qb[k]);
          qn0[k] = qn1[k];
        }
        qn1[k] = qs[k].at(qd[k] + NQ + 2 + (i0 >> 2));
      }
      uint2 na = trow[min(t4[0] & 0xffu, 7u)], nb = trow[min(t4[1] & 0xffu, 7u)];
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int i = i0 + rr;
        const uint2 sa = na, sb = nb;
        t4[0] >>= 8;
        t4[1] >>= 8;
        if (rr < 3) {  // the next row's penalties
          na = trow[min(t4[0] & 0xffu, 7u)];
          nb = trow[min(t4[1] & 0xffu, 7u)];
        }
        u16x2 F = kNone;
        uint32_t acc[2 * NW];
#pragma unroll
        for (int m = 0; m < 2 * NW; ++m) acc[m] = 0;
        u16x2 n4p = splat(0u);
#pragma unroll
        for (int m = 0; m < NQ; ++m) {
          const uint32_t pa = __builtin_amdgcn_perm(sa.y, sa.x, qw[0][m]);
          const uint32_t pb = __builtin_amdgcn_perm(sb.y, sb.x, qw[1][m]);
          u16x2 n4 = splat(0u);
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int r = 4 * m + c;
            if (r >= NC) {
              n4 = n4 >> (uint16_t)4;
              continue;
            }
            const u16x2 M = ssat(G[r], pk(__builtin_amdgcn_perm(pb, pa, 0x0c040c00u + 0x00010001u * c)));
            const u16x2 e = E[r];
            const u16x2 hm = smax(M, e);
            const u16x2 od = ssat(M, oe_del), ee = ssat(e, e_del);
            const u16x2 oi = ssat(M, oe_ins), fe = ssat(F, e_ins);
            // sign bits: E taken over M; F taken over both; E extended; F extended
            const u16x2 x = ssat(M, e), y = ssat(hm, F), z = ssat(od, ee), v = ssat(oi, fe);
            const uint32_t xy = (pku(x) & 0x80008000u) | pku(y >> (uint16_t)1);
            const uint32_t zv = (pku(z) & 0x80008000u) | pku(v >> (uint16_t)1);
            const uint32_t nib = (xy & 0xc000c000u) | pku(pk(zv) >> (uint16_t)2);
            n4 = pk((nib & 0xf000f000u) | pku(n4 >> (uint16_t)4));
            G[r] = smax(hm, F);
            F = smax(oi, fe);
            if (r > 0) {
              u16x2 ne = smax(od, ee);
              if (r - 1 >= TOP0 && (r - 1 - TOP0) % 2 == 0) ne = smin(ne, cap[(r - 1 - TOP0) / 2]);
              E[r - 1] = ne;
            }
            // Keep the cells in order and their results materialised: left alone
            // the compiler defers the state updates and the packing of the
            // directions of a whole row and spills.  (The cell before this one:
            // an operand written by the instruction before costs a wait state.)
            if (r >= 2) asm volatile("" ::"v"(G[r - 1]), "v"(E[r - 2]), "v"(n4p));
            n4p = n4;
            if (c & 1) __builtin_amdgcn_sched_barrier(0);
          }
          acc[m] = pku(n4);
        }
        E[NC - 1] = kNone;
        // the query moves one position left
#pragma unroll
        for (int k = 0; k < 2; ++k) {
#pragma unroll
          for (int m = 0; m < NQ; ++m) qw[k][m] = __builtin_amdgcn_alignbyte(qw[k][m + 1], qw[k][m], 1u);
          qw[k][NQ] >>= 8;
        }
        if (want_cigar) {
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            uint32_t* __restrict__ zr = zreg + ((i * 2 + k) * 64 + lane) * NW;
#pragma unroll
            for (int m = 0; m < NW; ++m)
              zr[m] = __builtin_amdgcn_perm(acc[2 * m + 1], acc[2 * m], k ? 0x07060302u : 0x05040100u);
          }
        }
        const uint32_t last = (i == tlen[0] - 1 ? 0xffffu : 0u) | (i == tlen[1] - 1 ? 0xffff0000u : 0u);
        if (__any(last != 0)) {  // a task's last row: H(tlen-1, qlen-1)
          u16x2 g = splat(0u);
#pragma unroll
          for (int r = 0; r < NC; ++r) {
            const u16x2 d = rf - splat((uint32_t)r);
            const uint32_t eq = ~(negmask(d) | negmask(splat(0u) - d));
            g = g | (G[r] & pk(eq));
          }
          fin = sel(last, g, fin);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int hq = (k ? (int)((int32_t)pku(fin) >> 16) : (int)(int16_t)(pku(fin) & 0xffffu)) + A.mat_max * qlen[k];
      if (have[k] && A.score) A.score[task[k]] = hq;
      if (have[k] && !want_cigar && A.n_cigar) A.n_cigar[task[k]] = 0;
    }
    if (!want_cigar) continue;

    // ---- walk back (ksw.c:588-602) ----
    int r[2], i[2], state[2], run_op[2], run_len[2], n[2];
    bool over[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      i[k] = tlen[k] - 1;
      r[k] = qlen[k] - tlen[k] + w[k];
      state[k] = 0; run_op[k] = -1; run_len[k] = 0; n[k] = 0; over[k] = false;
    }
    auto emit = [&](int k) {
      if (run_op[k] < 0) return;
      if (n[k] < A.cigar_slot) {
        A.cigar[(int64_t)task[k] * A.cigar_slot + n[k]] = (uint32_t)run_len[k] << 4 | (uint32_t)run_op[k];
        ++n[k];
      } else {
        over[k] = true;
      }
    };
    auto push = [&](int k, int op, int len) {
      if (op == run_op[k]) {
        run_len[k] += len;
      } else {
        emit(k);
        run_op[k] = op;
        run_len[k] = len;
      }
    };
    constexpr int D = NC <= 31 ? 8 : 4;  // rows loaded ahead
    uint32_t cur[2][D][NW], nxt[2][D][NW];
    auto load = [&](int k, int row, uint32_t* dst) {
      const uint32_t* __restrict__ zr = zreg + ((max(row, 0) * 2 + k) * 64 + lane) * NW;
#pragma unroll
      for (int m = 0; m < NW; ++m) dst[m] = zr[m];
    };
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int d = 0; d < D; ++d) load(k, i[k] - d, cur[k][d]);
    // column of (i, r) is i - w + r; a task walks while its row and column are
    // >= 0.  left = min(row, column).  The words and shift of position r are
    // kept as masks, renewed when r changes.
    int left[2], sh[2];
    uint32_t wm[2][NW];
    bool odd[2];  // the last step was no M (or there was none)
    auto place = [&](int k) {
      over[k] = over[k] || (unsigned)r[k] >= (unsigned)NC;  // cannot happen under the preconditions
      left[k] = over[k] ? -1 : min(i[k], i[k] - w[k] + r[k]);
      sh[k] = 4 * (r[k] & 7);
#pragma unroll
      for (int m = 0; m < NW; ++m) wm[k][m] = (r[k] >> 3) == m ? ~0u : 0u;
    };
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      place(k);
      odd[k] = true;
    }
    while (__any((left[0] & left[1]) >= 0)) {
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int d = 0; d < D; ++d) load(k, i[k] - D - d, nxt[k][d]);
#pragma unroll
      for (int d = 0; d < D; ++d) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          auto nibble = [&]() -> uint32_t {  // bit 3: x, 2: y, 1: z, 0: v
            uint32_t zw = cur[k][d][0] & wm[k][0];
#pragma unroll
            for (int m = 1; m < NW; ++m) zw |= cur[k][d][m] & wm[k][m];
            return zw >> sh[k];
          };
          // Nearly every step is one more M of a run; a step that is not, of any
          // lane, takes the wave through the general form once.
          const bool on = left[k] >= 0;
          const bool plain = !on || !(odd[k] || (nibble() & 0xcu));
          const int step = on && plain ? 1 : 0;
          i[k] -= step;
          left[k] -= step;
          run_len[k] += step;
          if (__any(!plain)) {
            bool row = !plain;
            while (__any(row)) {
              if (row) {
                const uint32_t nib = nibble();
                const int s0 = (nib & 4u) ? 2 : (int)(nib >> 3 & 1u);
                const int s1 = (int)(nib >> 1 & 1u), s2 = (int)(nib << 1 & 2u);
                const int s = state[k] == 0 ? s0 : state[k] == 1 ? s1 : s2;
                state[k] = s;
                push(k, s == 0 ? 0 : 3 - s, 1);  // M; state 1: D, state 2: I
                odd[k] = s != 0;
                // M: row and column go down, the position stays; D: one row down,
                // one position right; I: one position left in the same row
                i[k] -= s != 2 ? 1 : 0;
                r[k] += s == 0 ? 0 : 3 - 2 * s;
                place(k);
                row = s == 2 && left[k] >= 0;
              }
            }
          }
        }
      }
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int d = 0; d < D; ++d)
#pragma unroll
          for (int m = 0; m < NW; ++m) cur[k][d][m] = nxt[k][d][m];
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (!have[k]) continue;
      const int col = i[k] - w[k] + r[k];
      if (i[k] >= 0) push(k, 2, i[k] + 1);
      if (col >= 0) push(k, 1, col + 1);
      emit(k);
      uint32_t* cg = A.cigar + (int64_t)task[k] * A.cigar_slot;
      if (over[k]) {
        A.n_cigar[task[k]] = -1;
        atomicAdd(&W.err[2], 1);
      } else {
        for (int a = 0, b = n[k] - 1; a < b; ++a, --b) {
          const uint32_t ta = cg[a], tb = cg[b];
          cg[a] = tb;
          cg[b] = ta;
        }
        A.n_cigar[task[k]] = n[k];
      }
    }
  }
}

// Streams: the bins are independent and each is mostly the latency of a wave or
// two (150 rows and a walk back), so they run side by side.  The widest, whose
// waves need a SIMD to themselves, starts first, on the call's own stream.
constexpr int kGlbPairStream[kGlbPairBins] = {3, 2, 0, 1, 0};

void launch_glb_pair(const GlbArgs& a, const GlbWork& w, int num_cu, hipStream_t st) {
  auto one = [&](auto kernel, int b) {
    GlbWork k = w;
    int64_t at = 0;
    for (int x = 0; x < b; ++x) at += kGlbPairShare[x];
    k.pair_bytes = w.pair_bytes / 64 * kGlbPairShare[b];
    if (w.zpair) k.zpair = w.zpair + w.pair_bytes / 64 * at;
    const int64_t blocks =
        std::min<int64_t>((a.n + 127) / 128, (int64_t)num_cu * 4 * gpair_min_waves(kGlbPairCols[b]));
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(64), 0, pick_stream(w.ss, st, kGlbPairStream[b]), a, k,
                       kGlbBins + b);
  };
  static_assert(kGlbPairBins == 5, "CIGAR pair kernels");
  one(glb_pair_kernel<kGlbPairCols[4]>, 4);
  one(glb_pair_kernel<kGlbPairCols[3]>, 3);
  one(glb_pair_kernel<kGlbPairCols[1]>, 1);
  one(glb_pair_kernel<kGlbPairCols[0]>, 0);
  one(glb_pair_kernel<kGlbPairCols[2]>, 2);
}
constexpr int glb_pair_shares() {
  int s = 0;
  for (int b = 0; b < kGlbPairBins; ++b) s += kGlbPairShare[b];
  return s;
}
static_assert(glb_pair_shares() <= 64 && kGlbPairScratch / 64 % 16 == 0, "scratch shares");
static_assert(kGlbPairScratch * 4 / 64 * kGlbPairShare[4] >= glb_pair_region(63, glb_pair_rows(kGlbPairTlen)) &&
                  kGlbPairScratch * 4 / 64 * kGlbPairShare[2] >= glb_pair_region(31, glb_pair_rows(kGlbPairTlen)),
              "one wave has room on four CUs");

}  // namespace bsx
