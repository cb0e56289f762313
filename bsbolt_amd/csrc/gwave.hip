// One wave per task: bit-exact ksw_global2 (bsbolt/External/BWA/ksw.c:504-606)
// for small batches, without a binning pass.
//
// The row is the group kernel's (global.hip) with 64 lanes of C columns: F comes
// from a prefix maximum, and the band is a frame of 64*C columns from column f0
// on, f0 = max(0, i - w) rounded down to a multiple of C, that moves by a lane at a
// time (a query of at most 64*C bases in a wider band stays in place).  A wave has one task, so the
// band, the row's target base and the whole walk back are uniform.
//
// The four comparisons that make a row's direction byte (ksw.c:551-564) are
// ballots.  They are kept with lane = row, 64 rows in 8*C registers, and only whole
// blocks of 64 rows go to the direction slot and come back.  The walk reads them
// with v_readlane; while it runs diagonally, all rows of a block look up their own
// cell at once, and a ballot gives the length of the run.
//
// Bound by instruction issue (13.5 ns a task of 150 bp reads; scalar instructions
// took as much of it as vector ones before the windows held shifts and profile
// words instead of bytes: 20 ns) and, in a batch that leaves SIMDs idle, by the
// latency of its longest task's rows.
#include <algorithm>

#include "bsx_internal.h"
#include "ext_common.h"

// v with `value` (uniform) in lane `at` (uniform)
extern "C" __device__ int bsx_writelane(int value, int at, int v) __asm("llvm.amdgcn.writelane.i32");

namespace bsx {

constexpr int kGNegInf = -0x40000000;  // MINUS_INF, ksw.c:490
__device__ __forceinline__ int guni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Keys of the prefix maximum are raised by kGRaise, so that those of finite values
// (glb_direct_kernel checks the range) are positive and 0 stands for none.
constexpr int kGRaise = 1 << 30, kGRange = 1 << 28;

// A CIGAR under construction, from its end: the last 64 words in a register.
struct Ops {
  uint32_t* cg;
  int64_t cap;
  uint32_t reg = 0;
  int n = 0, op = -1, len = 0;
  __device__ __forceinline__ void spill(int count) {  // words [n - count, n), not reversed
    const int at = n - count + (int)(threadIdx.x & 63);
    if ((int)(threadIdx.x & 63) < count && at < cap) cg[at] = reg;
  }
  __device__ __forceinline__ void emit() {
    if (op < 0) return;
    reg = (uint32_t)bsx_writelane(len << 4 | op, n & 63, (int)reg);
    ++n;
    if ((n & 63) == 0) spill(64);
  }
  __device__ __forceinline__ void push(int o, int l) {
    if (o == op) {
      len += l;
    } else {
      emit();
      op = o;
      len = l;
    }
  }
};

// All arguments are uniform; slot holds the blocks of directions but the last
// (2 KB * C each).  Returns the score; with a CIGAR wanted, *ncig its words or -1.
template <int C>
__device__ __forceinline__ int glb_wave_task(const GlbArgs& A, const uint8_t* __restrict__ query,
                                             const uint8_t* __restrict__ target, int qlen, int tlen, int w,
                                             uint32_t* __restrict__ slot, uint32_t* cg, int* ncig) {
  constexpr int WF = 64 * C;
  const int lane = threadIdx.x & 63, base = lane * C;
  const int e_del = A.e_del, e_ins = A.e_ins;
  const int oe_del = A.o_del + e_del, oe_ins = A.o_ins + e_ins;
  const bool want = cg != nullptr;
  const bool moves = 2 * w + C <= WF;                    // the frame follows the band; else it holds the query
  const bool wide = C > 1 || min(qlen, 2 * w + 1) > 32;  // the masks need their high words
  auto prof = [&](uint32_t qc) -> uint32_t {
    uint32_t lo = A.prof_lo[4];
    lo = qc == 0 ? A.prof_lo[0] : lo;
    lo = qc == 1 ? A.prof_lo[1] : lo;
    lo = qc == 2 ? A.prof_lo[2] : lo;
    lo = qc == 3 ? A.prof_lo[3] : lo;
    return lo;
  };
  int G[C], E[C];
  uint32_t plo[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int j = base + c;
    const uint32_t qb = query[min(j, qlen - 1)];
    const uint32_t qc = j < qlen ? min(qb, 4u) : 4u;
    plo[c] = prof(qc);
    G[c] = j == 0 ? 0 : (j <= w ? -(A.o_ins + e_ins * j) : kGNegInf);  // row -1 (ksw.c:522-525)
    E[c] = kGNegInf;
  }
  // The next 64 rows' bases by lane, as shifts into a profile word (32: not a base),
  // and the profile words of the next 64 columns to enter the frame; the bytes of
  // the 64 after them are already loading.
  auto shift_of = [&](uint32_t b) -> uint32_t { return 8 * min(b, 4u); };
  auto prof_at = [&](uint32_t b, int j) -> uint32_t { return prof(j < qlen ? min(b, 4u) : 4u); };
  auto t_at = [&](int i) -> uint32_t { return target[min(i + lane, tlen - 1)]; };
  auto q_at = [&](int j) -> uint32_t { return query[min(j + lane, qlen - 1)]; };
  uint32_t tch = shift_of(t_at(0)), tnx = t_at(64);
  uint32_t qch = prof_at(q_at(WF), WF + lane), qnx = q_at(WF + 64);

  uint32_t Z[8 * C];  // rows of the block by lane: per column, the masks of from M, not from F,
                      // E extends, F extends
#pragma unroll
  for (int q = 0; q < 8 * C; ++q) Z[q] = 0;
  const int key0 = kGRaise - oe_ins + base * e_ins, back0 = kGRaise + (base - 1) * e_ins;
  int f0 = 0, hq = 0;
  for (int i = 0; i < tlen; ++i) {
    const int zr = i & 63;
    if (i && zr == 0) {
      tch = shift_of(tnx);
      tnx = t_at(i + 64);
    }
    const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)tch, zr);
    const int beg = max(i - w, 0), end = min(i + w + 1, qlen);
    const int pb = beg - f0, pe = end - f0;
    int M[C], ex[C];
    if (__builtin_expect(t == 32, 0)) {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int j = f0 + base + c;
        const uint32_t qb = query[min(j, qlen - 1)], qc = j < qlen ? qb : 4u;
        int s = A.prof_hi[4];
        s = qc == 0 ? A.prof_hi[0] : s;
        s = qc == 1 ? A.prof_hi[1] : s;
        s = qc == 2 ? A.prof_hi[2] : s;
        s = qc == 3 ? A.prof_hi[3] : s;
        M[c] = s;
      }
    } else {
#pragma unroll
      for (int c = 0; c < C; ++c) M[c] = __builtin_amdgcn_sbfe((int)plo[c], t, 8u);
    }
    bool inb[C];
    int run = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      inb[c] = (uint32_t)(base + c - pb) < (uint32_t)(pe - pb);
      M[c] += G[c];
      ex[c] = run;
      run = max(run, inb[c] ? M[c] + (key0 + c * e_ins) : 0);
    }
    const int lex = __builtin_amdgcn_update_dpp(0, grp_incl_max<64>(run), 0x138, 0xf, 0xf, true);  // wave_shr:1
    int h[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int x = max(ex[c], lex);
      const int f = x == 0 ? kGNegInf : x - (back0 + c * e_ins);  // -inf in the band's first column
      const int mm = M[c], e = E[c], me = max(mm, e);
      const int od = mm - oe_del, ee = e - e_del;
      h[c] = max(me, f);
      E[c] = inb[c] ? max(ee, od) : kGNegInf;
      if (want) {
        const uint64_t fromM = __ballot(mm >= e), notF = __ballot(me >= f);
        const uint64_t eext = __ballot(ee > od), fext = __ballot(f - e_ins > mm - oe_ins);
        const uint64_t m[4] = {fromM, notF, eext, fext};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          Z[8 * c + q] = (uint32_t)bsx_writelane((int)(uint32_t)m[q], zr, (int)Z[8 * c + q]);
          if (wide)
            Z[8 * c + 4 + q] = (uint32_t)bsx_writelane((int)(uint32_t)(m[q] >> 32), zr, (int)Z[8 * c + 4 + q]);
        }
      }
    }
    if (end == qlen) {
      int he = h[0];
#pragma unroll
      for (int c = 1; c < C; ++c) he = ((pe - 1) & (C - 1)) == c ? h[c] : he;
      hq = __builtin_amdgcn_readlane(he, (pe - 1) / C);
    }
    if (moves && i + 1 - w - f0 >= C) {
      // the frame moves one lane: column j - 1 of the next row's G is C - 1 positions on
      const int jo = f0 & 63;  // column f0 + WF enters
      if (f0 > 0 && jo == 0) {
        qch = prof_at(qnx, f0 + WF + lane);
        qnx = q_at(f0 + WF + 64);
      }
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int in = __builtin_amdgcn_readlane((int)qch, jo + c);
        E[c] = __builtin_amdgcn_update_dpp(kGNegInf, E[c], 0x130, 0xf, 0xf, false);  // wave_shl:1
        plo[c] = (uint32_t)__builtin_amdgcn_update_dpp(in, (int)plo[c], 0x130, 0xf, 0xf, false);
        G[c] = c == 0 ? h[C - 1] : __builtin_amdgcn_update_dpp(kGNegInf, h[c - 1], 0x130, 0xf, 0xf, false);
      }
      f0 += C;
    } else {
      const int h1p = beg == 0 ? -(A.o_del + e_del * (i + 1)) : kGNegInf;  // eh[0].h
      const int left = __builtin_amdgcn_update_dpp(h1p, h[C - 1], 0x138, 0xf, 0xf, false);  // wave_shr:1
#pragma unroll
      for (int c = 0; c < C; ++c) G[c] = c == 0 ? left : h[c - 1];
    }
    if (want && zr == 63 && i + 1 < tlen) {
#pragma unroll
      for (int q = 0; q < 8 * C; ++q) slot[((i >> 6) * 8 * C + q) * 64 + lane] = Z[q];
    }
  }
  *ncig = 0;
  if (!want) return hq;

  // the walk back (ksw.c:588-602)
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  Ops O{cg, A.cigar_slot};
  auto frame_of = [&](int row) { return moves ? max(row - w, 0) / C * C : 0; };
  int i = tlen - 1, k = min(i + w + 1, qlen) - 1, state = 0, cur = i >> 6;
  while (i >= 0 && k >= 0) {
    if ((i >> 6) != cur) {
      cur = i >> 6;
#pragma unroll
      for (int q = 0; q < 8 * C; ++q) Z[q] = slot[(cur * 8 * C + q) * 64 + lane];
    }
    if (state == 0) {
      // every row's own cell of this diagonal
      const int row = (cur << 6) + lane, kr = k - (i - row);
      const int kc = kr - frame_of(row), bit = kc / C;
      uint32_t lo = Z[0] & Z[1], hi = Z[4] & Z[5];
#pragma unroll
      for (int c = 1; c < C; ++c) {
        lo = (kc & (C - 1)) == c ? Z[8 * c] & Z[8 * c + 1] : lo;
        hi = (kc & (C - 1)) == c ? Z[8 * c + 4] & Z[8 * c + 5] : hi;
      }
      const bool turn = !((bit & 32 ? hi : lo) >> (bit & 31) & 1u) && row <= i && kr >= 0;
      const uint64_t turns = __ballot(turn);
      const int r = turns ? (cur << 6) + 63 - __builtin_clzll(turns) : max((cur << 6) - 1, i - k - 1);
      if (i > r) O.push(0, i - r);
      k -= i - r;
      i = r;
      if (!turns) continue;
    }
    // one cell: state 0 turns to D or I here; D and I go on or end in a diagonal step
    const int kc = k - frame_of(i), bit = kc / C, zr = i & 63;
    const int q = state == 0 ? 1 : state + 1;  // state 0: a turn that is not from F is to D
    uint32_t word = 0;
#pragma unroll
    for (int x = 0; x < 8 * C; ++x)
      if (x == 8 * (kc & (C - 1)) + (bit & 32 ? 4 : 0) + q) word = (uint32_t)__builtin_amdgcn_readlane((int)Z[x], zr);
    const bool set = word >> (bit & 31) & 1u;
    state = state == 0 ? (set ? 1 : 2) : (set ? state : 0);
    O.push(state == 0 ? 0 : state == 1 ? 2 : 1, 1);
    i -= state != 2;
    k -= state != 1;
  }
  if (i >= 0) O.push(2, i + 1);
  if (k >= 0) O.push(1, k + 1);
  O.emit();
  const int n = O.n;
  if (n > A.cigar_slot) {
    *ncig = -1;
  } else if (n <= 63) {
    if (lane < n) cg[n - 1 - lane] = O.reg;
    *ncig = n;
  } else {
    O.spill(n & 63);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    for (int a = lane; a < n / 2; a += 64) {
      const uint32_t ta = cg[a], tb = cg[n - 1 - a];
      cg[a] = tb;
      cg[n - 1 - a] = ta;
    }
    *ncig = n;
  }
  return hq;
}

// Block t runs task t.  A task whose band is wider than 256 columns, whose scores
// may be large, or whose blocks of directions do not fit its slot, goes to the list of a group bin.
__global__ void __launch_bounds__(64, 4) glb_direct_kernel(GlbArgs A, GlbWork W) {
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x;
  const int ql = A.qlen[t], tl = A.tlen[t];
  const bool ok = glb_task_ok(A, W, t);
  if (lane == 0) {
    W.bin_of[t] = ok ? 0 : 0xff;
    if (!ok) {
      atomicAdd(&W.err[0], 1);
      atomicMin(&W.err[1], (int)t);
    }
  }
  if (!ok) return;
  const int w = min(A.w[t], max(ql, tl));
  const bool want = A.cigar != nullptr;
  const int64_t range = (int64_t)(ql + tl) * (A.pen_max + max(A.e_del, A.e_ins) + A.mat_max) + A.o_del + A.o_ins;
  const auto fits = [&](int C) {
    return range < kGRange && (ql <= 64 * C || 2 * w + C <= 64 * C) &&
           (!want || (int64_t)((tl - 1) >> 6) * 2048 * C <= W.zslot);
  };
  const int C = fits(1) ? 1 : fits(2) ? 2 : fits(4) ? 4 : 0;
  if (C == 0) {
    if (lane == 0) {
      const int r = glb_rest_of(min(ql, 2 * w + 1));
      W.list[(int64_t)r * A.n + atomicAdd(&W.counts[kGlbRestBin[r]], 1u)] = (int32_t)t;
    }
    return;
  }
  const uint8_t *q = A.query + A.q_off[t], *tg = A.target + A.t_off[t];
  uint32_t* slot = (uint32_t*)(W.z + t * W.zslot);
  uint32_t* cg = want ? A.cigar + t * A.cigar_slot : nullptr;
  int nc = 0, score;
  if (C == 1) score = glb_wave_task<1>(A, q, tg, ql, tl, w, slot, cg, &nc);
  else if (C == 2) score = glb_wave_task<2>(A, q, tg, ql, tl, w, slot, cg, &nc);
  else score = glb_wave_task<4>(A, q, tg, ql, tl, w, slot, cg, &nc);
  if (lane == 0) {
    if (A.score) A.score[t] = score;
    if (A.n_cigar) A.n_cigar[t] = nc;
    if (nc < 0) atomicAdd(&W.err[2], 1);
  }
}

void launch_glb_direct(const GlbArgs& a, const GlbWork& w, hipStream_t st) {
  hipLaunchKernelGGL(glb_direct_kernel, dim3((unsigned)a.n), dim3(64), 0, st, a, w);
}

}  // namespace bsx
