// One wave per task: bit-exact ksw_extend2 (bsbolt/External/BWA/ksw.c:380-479)
// for wide tasks, and for whole small batches without a binning pass.
//
// The row is the group kernels' row (extend.hip): lane g holds C consecutive
// columns of G = H(i-1, j-1) and E in VGPRs, F comes from a prefix maximum, and
// columns left of beg stay at G = E = 0.  Two things differ.
//
// A wave has one task, so everything about the row that is not a column is
// uniform: the band, the row's target base, the best score and the end tests
// live in SGPRs and branch, the value at the band's end is one v_readlane, and
// the first and last live columns come from a ballot and two v_readlanes.  Only
// F and the row maximum are reduced across lanes.
//
// The columns are a frame of 64*C from column f0 on, which follows the band cap:
//   f0 = max(0, i - w) rounded down to a multiple of C.
// Row i reads and writes columns beg..end only, with i - w <= beg and end <=
// i + w + 1 (ksw.c:413-416), so a frame of at least 2w + 1 + C columns holds every
// column that a row touches: nothing left of it is read again, and a column that
// enters from the right was never written and still holds its first-row value
// (ksw.c:395-397).  A task so needs min(qlen, 2w + 1 + C) columns: with the usual
// band of 100 a query of any length runs 256.
//
// The row is bound by instruction issue (about 130 vector and 60 scalar
// instructions for C = 4); a lone wave takes 0.6 us a row, as each waits for the one
// before.  4,001 flanks of 2 kb reads, most of band 100: 2.06 ms, where rows of all
// 2,048 columns took 8.1.  C = 32 spills 34 of its 256 registers where a whole bin
// is its own (140 bytes of scratch a lane).
#include <algorithm>

#include "bsx_internal.h"
#include "ext_common.h"

namespace bsx {

struct WaveRes {
  int best, qle, tle, gtle, gscore, moff;
  uint32_t ncell;
  bool fail;  // a frame run would have stopped (wave_task's `fw`)
};

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// A: the scoring fields (ExtArgs or ExtKArgs).  Every argument is uniform over
// the wave; query and target hold qlen >= 1 and tlen >= 0 bases.
// fw (CERT): also tells whether the band-following run in a frame of fw columns
// (narrow.hip) would have reached past it, by that run's own test on the same
// values: the two are equal up to the row where it stops.
template <int C, bool CERT, class Args>
__device__ __forceinline__ WaveRes wave_task(const Args& A, const uint8_t* __restrict__ query,
                                             const uint8_t* __restrict__ target, int qlen, int tlen, int h0, int w,
                                             int fw = 0) {
  constexpr int WF = 64 * C;
  const int lane = threadIdx.x & 63;
  const int base = lane * C;
  const int e_del = A.e_del, e_ins = A.e_ins;
  const int oe_del = A.o_del + e_del, oe_ins = A.o_ins + e_ins;
  WaveRes R{h0, 0, 0, 0, -1, 0, 0u, false};
  if (tlen <= 0) return R;  // ksw.c:473-478 with no row

  auto ramp = [&](int j) { const int g = j == 0 ? h0 : h0 - oe_ins - (j - 1) * e_ins; return g > 0 ? g : 0; };
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
  {
    uint32_t qb[C];
#pragma unroll
    for (int c = 0; c < C; ++c) qb[c] = query[min(base + c, qlen - 1)];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int j = base + c;
      const uint32_t qc = j < qlen ? min(qb[c], 4u) : 4u;
      plo[c] = prof(qc);
      G[c] = ramp(j);
      E[c] = 0;
    }
  }
  // The next 64 rows' bases by lane, as shifts into a profile word (32: not a base),
  // and the profile words of the next 64 columns to enter the frame; the bytes of
  // the 64 after them are already loading.  (Scalar instructions bound the row as
  // much as vector ones: 80,000 flanks of 150 bp reads 595 us with bytes in the
  // windows, 557 so.)
  auto shift_of = [&](uint32_t b) -> uint32_t { return 8 * min(b, 4u); };
  auto prof_at = [&](uint32_t b, int j) -> uint32_t { return prof(j < qlen ? min(b, 4u) : 4u); };
  auto t_at = [&](int i) -> uint32_t { return target[min(i + lane, tlen - 1)]; };
  auto q_at = [&](int j) -> uint32_t { return query[min(j + lane, qlen - 1)]; };
  uint32_t tch = shift_of(t_at(0)), tnx = t_at(64);
  uint32_t qch = 0, qnx = 0;
  if (qlen > WF) {
    qch = prof_at(q_at(WF), WF + lane);
    qnx = q_at(WF + 64);
  }

  int beg = 0, end = qlen, f0 = 0, ff = 0;  // ff: first column of the narrow frame
  int best = h0, best_i = -1, best_j = -1, gbest = -1, gbest_i = -1, moff = 0;
  uint32_t ncell = 0;
  const int kE0 = base * e_ins;  // frame position k contributes k*e_ins

  for (int i = 0; i < tlen; ++i) {
    if (i && (i & 63) == 0) {
      tch = shift_of(tnx);
      tnx = t_at(i + 64);
    }
    const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)tch, i & 63);

    const int cap_beg = i - w;
    if (cap_beg - f0 >= C && f0 + WF < qlen) {
      // the frame moves one lane: lane 63 takes the next C columns
      const int jn = f0 + WF, jo = f0 & 63;
      if (f0 > 0 && jo == 0) {
        qch = prof_at(qnx, jn + lane);
        qnx = q_at(jn + 64);
      }
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int in = __builtin_amdgcn_readlane((int)qch, jo + c);
        G[c] = __builtin_amdgcn_update_dpp(ramp(jn + c), G[c], 0x130, 0xf, 0xf, false);  // wave_shl:1
        E[c] = __builtin_amdgcn_update_dpp(0, E[c], 0x130, 0xf, 0xf, false);
        plo[c] = (uint32_t)__builtin_amdgcn_update_dpp(in, (int)plo[c], 0x130, 0xf, 0xf, false);
      }
      f0 += C;
    }
    if (beg < cap_beg) {  // the band cap moves beg: keep the dead-column invariant
      beg = cap_beg;
#pragma unroll
      for (int c = 0; c < C; ++c)
        if (f0 + base + c < beg) { G[c] = 0; E[c] = 0; }
    }
    end = min(min(end, i + w + 1), qlen);
    int h1p = 0;
    if (beg == 0) h1p = max(h0 - (A.o_del + e_del * (i + 1)), 0);

    const int d = end - f0 - base;  // live columns of this lane: c < d
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
    int run = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int mm = G[c] ? G[c] + M[c] : 0;
      M[c] = mm;
      const int kb = kE0 + (c + 1) * e_ins;
      ex[c] = run;
      run = max(run, max(mm + (kb - oe_ins), kb));
    }
    const int lex = grp_excl_from_incl<64>(grp_incl_max<64>(run), lane);
    int h[C];
    int mk = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int f = max(ex[c], lex) - (kE0 + c * e_ins);
      const int hh = max(max(M[c], E[c]), f);
      h[c] = hh;
      const int ne = max(max(E[c] - e_del, M[c] - oe_del), 0);
      const bool lt = c < d;
      mk = lt ? max(mk, (hh << 11) | (base + c)) : mk;
      E[c] = lt ? ne : (c == d ? 0 : E[c]);  // eh[end].e = 0
    }
    const int ke = end - 1 - f0;  // frame position of the band's last column
    int h1 = h1p;
    if (end > beg) {
      int he = h[0];
#pragma unroll
      for (int c = 1; c < C; ++c) he = (ke & (C - 1)) == c ? h[c] : he;
      h1 = __builtin_amdgcn_readlane(he, ke / C);
    }
    if (CERT && fw && end > ff + fw - 1) {  // the band reaches past the frame: its cells there must be 0
      const int eF = ff + fw - 1, ce = eF - f0;
      int he = h[0];
#pragma unroll
      for (int c = 1; c < C; ++c) he = (ce & (C - 1)) == c ? h[c] : he;
      const int hF = ce >= 0 ? __builtin_amdgcn_readlane(he, ce / C) : 0;  // left of the wave's frame all is 0
      R.fail = R.fail || hF != 0 || ramp(eF + 1) > 0;
    }
    // G(j) = H(i, j-1) for j <= end; column 0 receives the first-column value
    const int hsh = __builtin_amdgcn_update_dpp(h1p, h[C - 1], 0x138, 0xf, 0xf, false);  // wave_shr:1
    uint32_t nzb = 0;  // bit c: column c holds a non-zero G or E after the row
#pragma unroll
    for (int c = 0; c < C; ++c) {
      G[c] = c <= d ? (c == 0 ? hsh : h[c - 1]) : G[c];
      nzb |= (uint32_t)min((uint32_t)(G[c] | E[c]), 1u) << c;
    }
    nzb &= d >= C ? 0xffffffffu : d > 0 ? (1u << d) - 1u : 0u;  // columns < end
    const uint64_t lanes = __ballot(nzb != 0);
    mk = __builtin_amdgcn_readlane(grp_incl_max<64>(mk), 63);

    const int jafter = max(end, beg);
    if (jafter == qlen) {  // ksw.c:450-453
      if (!(gbest > h1)) gbest_i = i;
      gbest = max(gbest, h1);
    }
    ncell += (uint32_t)(jafter - beg);
    const int m = end > beg ? mk >> 11 : 0;
    if (m == 0) break;
    const int mj = (mk & 2047) + f0;
    if (m > best) {
      best = m; best_i = i; best_j = mj;
      moff = max(moff, mj > i ? mj - i : i - mj);
    } else if (A.zdrop > 0) {
      const int di = i - best_i, dj = mj - best_j;
      const int drop = di > dj ? best - m - (di - dj) * e_del : best - m - (dj - di) * e_ins;
      if (drop > A.zdrop) break;
    }
    // ksw.c:466-469
    int nb = end, hz = -1;
    if (lanes) {
      const int lf = __builtin_ctzll(lanes), ll = 63 - __builtin_clzll(lanes);
      nb = f0 + lf * C + __builtin_ctz((uint32_t)__builtin_amdgcn_readlane((int)nzb, lf));
      hz = f0 + ll * C + 31 - __builtin_clz((uint32_t)__builtin_amdgcn_readlane((int)nzb, ll));
    }
    if (h1 != 0) hz = end;
    beg = nb;
    end = min(hz >= 0 ? hz + 2 : nb + 1, qlen);
    if (CERT) ff += min(beg - ff, 2);
  }
  R.best = best; R.qle = best_j + 1; R.tle = best_i + 1; R.gtle = gbest_i + 1; R.gscore = gbest;
  R.moff = moff; R.ncell = ncell;
  return R;
}

// waves per SIMD the register budget must allow
constexpr int wave_min_waves(int C) { return C <= 4 ? 5 : C <= 8 ? 3 : 2; }

// A bin's list: block k takes descriptors k, k + gridDim.x, ...
template <int C>
__global__ void __launch_bounds__(64, wave_min_waves(C))
ext_wave_kernel(ExtKArgs A, const ExtDesc* __restrict__ desc_all, const uint32_t* __restrict__ counts, int bin) {
  uint32_t lbase = 0;
  for (int b = 0; b < bin; ++b) lbase += counts[b];
  const uint32_t nlist = counts[bin];
  for (uint32_t x = blockIdx.x; x < nlist; x += gridDim.x) {
    const int4* d = (const int4*)(desc_all + lbase + x);
    const int4 a = d[0], b = d[1], c = d[2];
    const int task = uni(a.x);
    const uint64_t qoff = (uint64_t)(uint32_t)uni(b.z) | (uint64_t)(uint32_t)uni(b.w) << 32;
    const uint64_t toff = (uint64_t)(uint32_t)uni(c.x) | (uint64_t)(uint32_t)uni(c.y) << 32;
    const WaveRes R = wave_task<C, false>(A, A.query + qoff, A.target + toff, uni(a.y), uni(a.z), uni(a.w), uni(b.x));
    write_rec<64>(A.rec, task, threadIdx.x, R.best, R.qle, R.tle, R.gtle, R.gscore, R.moff, R.ncell);
  }
}

template <int C>
void launch_wave_bin(const ExtKArgs& k, const ExtWork& wk, int bin, int64_t n, int num_cu, hipStream_t st) {
  // as many as are resident: surplus blocks of an empty bin cost 9 us a launch
  const int64_t blocks = std::min<int64_t>(n, (int64_t)num_cu * 4 * wave_min_waves(C));
  if (blocks < 1) return;
  time_begin(wk, time_of_bin(bin), st);
  hipLaunchKernelGGL(ext_wave_kernel<C>, dim3((unsigned)blocks), dim3(64), 0, st, k, (const ExtDesc*)wk.desc,
                     (const uint32_t*)wk.counts, bin);
  time_end(wk, time_of_bin(bin), st);
}
template void launch_wave_bin<4>(const ExtKArgs&, const ExtWork&, int, int64_t, int, hipStream_t);
template void launch_wave_bin<8>(const ExtKArgs&, const ExtWork&, int, int64_t, int, hipStream_t);
template void launch_wave_bin<16>(const ExtKArgs&, const ExtWork&, int, int64_t, int, hipStream_t);
template void launch_wave_bin<32>(const ExtKArgs&, const ExtWork&, int, int64_t, int, hipStream_t);


// A batch without binning: block t runs task t, checked here, and writes its
// results where the caller wants them, or as one record into pinned memory.  Tasks of
// more than 256 columns need waves of more registers: PART 0 takes the others, PART 1 these, PART 2 all.
// CERT: a batch that was checked and routed (nbin_of); also marks the tasks whose
// frame run fails (need_plain), and leaves every result in ExtWork::rec.
template <int PART, bool CERT>
__global__ void __launch_bounds__(64, wave_min_waves(PART == 0 ? 4 : 32))
ext_direct_kernel(ExtArgs A, ExtWork W) {
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x;
  const bool ok = CERT ? W.bin_of[t] != 0xff : ext_task_ok(A, t);
  if (!CERT && PART != 1) {
    if (A.rec_out) {
      if (!ok && lane < 8) A.rec_out[8 * t + lane] = 0;
    } else if (lane == 0) {
      W.bin_of[t] = ok ? 0 : 0xff;
      if (!ok) {
        atomicAdd(&W.err[0], 1);
        atomicMin(&W.err[1], (int)t);
      }
    }
  }
  if (!ok) return;
  const int ql = A.qlen[t], tl = A.tlen[t], h0 = A.h0[t];
  const int w = uni(ext_clamped_w(A, t));
  const auto fits = [&](int C) { return ql <= 64 * C || 2 * (int64_t)w + 1 + C <= 64 * C; };
  if (PART != 2 && fits(4) != (PART == 0)) return;
  const uint8_t *q = A.query + A.q_off[t], *tg = A.target + A.t_off[t];
  int fw = 0;
  if (CERT) {
    const int nb = W.nbin_of[t];
    fw = nb == 0 ? kFrameWidth[0] : nb == 1 ? kFrameWidth[1] : nb == 2 ? kFrameWidth[2] : nb == 3 ? kFrameWidth[3] : 0;
  }
  WaveRes R{};
  if (PART != 1 && fits(1)) R = wave_task<1, CERT>(A, q, tg, ql, tl, h0, w, fw);
  else if (PART != 1 && fits(2)) R = wave_task<2, CERT>(A, q, tg, ql, tl, h0, w, fw);
  else if (PART != 1 && fits(4)) R = wave_task<4, CERT>(A, q, tg, ql, tl, h0, w, fw);
  else if (PART != 0 && fits(8)) R = wave_task<8, CERT>(A, q, tg, ql, tl, h0, w, fw);
  else if (PART != 0 && fits(16)) R = wave_task<16, CERT>(A, q, tg, ql, tl, h0, w, fw);
  else if (PART != 0) R = wave_task<32, CERT>(A, q, tg, ql, tl, h0, w, fw);
  if (CERT && R.fail && lane == 0) W.need_plain[t] = 1;
  int32_t* rec = CERT ? W.rec : A.rec_out;
  if (rec) {
    write_rec<64>(rec, t, lane, R.best, R.qle, R.tle, R.gtle, R.gscore, R.moff, R.ncell, CERT ? 0 : 1);
  } else if (lane == 0) {
    if (A.score) A.score[t] = R.best;
    if (A.qle) A.qle[t] = R.qle;
    if (A.tle) A.tle[t] = R.tle;
    if (A.gtle) A.gtle[t] = R.gtle;
    if (A.gscore) A.gscore[t] = R.gscore;
    if (A.max_off) A.max_off[t] = R.moff;
    if (A.cells) A.cells[t] = (int64_t)R.ncell;
  }
}

// One launch with the registers of the widest task while the batch has at most
// as many tasks as the chip holds such waves.  Beyond, the wide tasks run beside
// the others: a long one takes milliseconds (4,000 flanks of 2 kb reads: 3.68 ms
// after them, 2.26 beside), though the fork costs every other batch some 9 us
// (2,000 flanks of 100 bp reads: 69 without, 78 with; 97 with a fork of all
// three side streams).
template <bool CERT>
static void direct(const ExtArgs& a, const ExtWork& wk, int num_cu, hipStream_t st) {
  const dim3 grid((unsigned)a.n), block(64);
  if (a.qmax <= 256) {
    hipLaunchKernelGGL((ext_direct_kernel<0, CERT>), grid, block, 0, st, a, wk);
  } else if (a.n <= (int64_t)num_cu * 4 * wave_min_waves(32)) {
    hipLaunchKernelGGL((ext_direct_kernel<2, CERT>), grid, block, 0, st, a, wk);
  } else {
    ss_fork(wk.ss, st, 1);
    hipLaunchKernelGGL((ext_direct_kernel<0, CERT>), grid, block, 0, st, a, wk);
    hipLaunchKernelGGL((ext_direct_kernel<1, CERT>), grid, block, 0, pick_stream(wk.ss, st, 1), a, wk);
    ss_join(wk.ss, st, 1);
  }
}

void launch_direct(const ExtArgs& a, const ExtWork& wk, int num_cu, hipStream_t st, bool cert) {
  if (cert) direct<true>(a, wk, num_cu, st);
  else direct<false>(a, wk, num_cu, st);
}

}  // namespace bsx
