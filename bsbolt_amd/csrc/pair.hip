// Two-tasks-per-lane form of the bit-exact ksw_extend2
// (bsbolt/External/BWA/ksw.c:380-479) for queries of up to 224 bases.
//
// Each lane of a wave owns two whole tasks, one in each 16-bit half of its
// registers, so one packed instruction advances two DP cells.  Per query
// column a lane keeps G1 = eh[j].h (plus the match score a where non-zero) and
// E = eh[j].e.  A row is the reference's column loop run inside the lane.
// Every value is an integer in [0, pair_score_max]: h0 + qlen * max(mat) bounds
// all scores of a run and is checked per task, so unsigned 16-bit arithmetic
// with subtraction saturating at 0 gives exactly the reference's values (its
// own recurrences clamp at 0 wherever a value could go below).
//
// Recurrences, with p = a - s >= 0 the penalty of a cell (s its substitution
// score, a = max(mat)) and "-" saturating:
//   M  = G1 - p                     (ksw.c:433-434: G ? G + s : 0)
//   H  = max(M, E, F)
//   E' = max(M - oe_del, E - e_del),  F' = max(M - oe_ins, F - e_ins)
//   G1'(j+1) = H ? H + a : 0
//
// Band.  A column outside [beg, end) holds G = E = 0, which makes its H, E and
// G successors 0 as well, so no per-column mask is needed except one: F is set
// to 0 at column `end` (the reference stops there).  That holds because beg
// never decreases, the columns the cap i-w cuts off are zeroed here, the
// reference's own end scan leaves only zero columns past `end`, and a column
// that no row has reached yet is given its first-row value (ksw.c:395-397) only
// when the band first includes it: the band grows by at most two columns a row,
// the first of them overwritten by the row before, so that is the one column
// past the largest `end` so far.
//
// Position p of a task is its column j + off, off = -qlen mod 8, so that the
// query ends on a multiple of 8: H(i, qlen-1) is then the value carried out of
// an eight-column block.  The first-column value enters at position off.
//
// Blocks of eight columns run only if one of the wave's 128 tasks has a live
// column there (one wave-uniform bit per block).  All tasks of a wave start
// together and the list is ordered longest run first, so the bands of a wave
// drift through the columns together and most blocks of a row are skipped.
//
// VALU-bound: 20 packed instructions per column (162 per block) and ~175 per
// row, for 128 tasks at once; the kernels it replaced took 31 per column for 64
// tasks (lane per task) and ~300 per row for 2-4 tasks (16-64 lanes per task).
// Widths 32 and 64 hold the state in the 256 VGPRs of two (three) waves per SIMD
// and issue VALU on 87-90% of the cycles.  Width 96 fills them and spills 28 (100
// bytes of scratch a lane, most of the 194 MB that a launch over 3.9M flanks
// writes): 79%.  Widths 128 and 224 take all 512 registers of a SIMD for one wave:
// the compiler keeps the columns past ~96 in accumulation registers, two to four
// moves per eight columns, 224 spills 44 (180 bytes), and a lone wave issues on
// half the cycles; that still is 3 (128) to 6 (224) times the group kernels' rate.  Kernel alone, queries of <= 32 / 33-64 / 65-96 / 97-128 /
// 129-224 bases: 3.9M flanks of 2x150 bp reads 0.42 / 1.42 / 1.47 / 0.85 / 0.14
// ms (was 1.16 / 3.5 / 5.0 / 2.5 / 0.33); 351,491 flanks of 250 bp reads 0.18 /
// 0.49 / 0.86 / 1.19 / 2.39 ms (97 and longer: was 2.3 / 9.2).  Whole calls: 4.2
// ms (was 11.9) and 2.9 ms (was 10.2).
#include "bsx_internal.h"
#include "ext_common.h"
#include "packed.h"

namespace bsx {

// x * e, at most 0xffff (x a column number below 2^14, e below 2^16)
__device__ __forceinline__ u16x2 emul(u16x2 x, u16x2 e) {
  const uint32_t lo = (pku(x) & 0xffffu) * (pku(e) & 0xffffu), hi = (pku(x) >> 16) * (pku(e) >> 16);
  return pk(min(lo, 0xffffu) | min(hi, 0xffffu) << 16);
}

// bitwise OR over the wave, as a scalar
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
  int x = (int)v;
  x |= __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
  x |= __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
  x |= __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
  x |= __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
  x |= __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x |= __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return (uint32_t)__builtin_amdgcn_readlane(x, 63);
}

// waves per SIMD the register budget leaves room for
constexpr int pair_min_waves(int Q) { return Q <= 32 ? 3 : Q <= 96 ? 2 : 1; }

template <int Q, bool SAME>
__global__ void __launch_bounds__(64, pair_min_waves(Q))
ext_pair_kernel(ExtKArgs A, const ExtDesc* __restrict__ desc_all, const uint32_t* __restrict__ counts, int bin) {
  constexpr int NB = Q / 8;
  static_assert(Q % 8 == 0 && NB < 31, "pair kernel width");
  constexpr int KB = Q <= 128 ? 7 : 8;                   // position bits of a (score, position) key
  constexpr uint32_t kStep = pair_score_max(Q);          // F cap per column left before `end`: no score above it
  constexpr uint32_t kEndStep = Q <= 120 ? 4096 : 2048;  // query-end test, per block left: above any score
  static_assert(kStep * Q <= 65535 && (kStep << KB) + Q <= 65536 && kEndStep * NB <= 65535, "16-bit ranges");
  __shared__ uint2 trow[8];         // penalties of a target code: query codes 0..3, and N
  __shared__ uint4 s_q[NB][64];     // query codes of a block: task 0 (.x .z), task 1 (.y .w)
  const int lane = threadIdx.x;
  uint32_t lbase = 0;
  for (int b = 0; b < bin; ++b) lbase += counts[b];
  const uint32_t nlist = counts[bin];
  const uint32_t first = blockIdx.x * 128u;
  if (first >= nlist) return;  // uniform over the block
  if (lane < 8) {
    const int t = lane < 5 ? lane : 4;
    uint32_t lo = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) lo |= (uint32_t)((A.mat_max - sbyte(A.trow_lo[t], q)) & 0xff) << (8 * q);
    trow[lane] = make_uint2(lo, (uint32_t)((A.mat_max - sbyte(A.trow_hi[t], 0)) & 0xff) * 0x01010101u);
  }
  const ExtDesc* __restrict__ desc = desc_all + lbase;

  const u16x2 one = hidden(1), step = hidden(kStep), skey = hidden(1u << KB);
  const u16x2 bit[8] = {one, hidden(2), hidden(4), hidden(8), hidden(16), hidden(32), hidden(64), hidden(128)};
  auto one_if = [&](u16x2 x) { return pkmin(x, one); };  // 1 in every non-zero half
  const u16x2 a_ = splat((uint32_t)A.mat_max);
  const u16x2 oe_del = splat((uint32_t)min(A.o_del + A.e_del, 0xffff));
  const u16x2 oe_ins = splat((uint32_t)min(A.o_ins + A.e_ins, 0xffff));
  const u16x2 e_del = splat((uint32_t)A.e_del), e_ins = splat((uint32_t)A.e_ins);

  // ---- the lane's two tasks ----
  int task[2];
  int qlen[2], tlen[2], h0[2], w[2];
  DwordSeq ts[2];
  bool have[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t p = first + 2u * lane + k;
    have[k] = p < nlist;
    const int4* d = (const int4*)(desc + (have[k] ? p : first));
    const int4 x = d[0], y = d[1], z = d[2];
    task[k] = x.x; qlen[k] = x.y; tlen[k] = x.z; h0[k] = x.w; w[k] = min(y.x, 0x3fff);
    const uint64_t qoff = (uint64_t)(uint32_t)y.z | (uint64_t)(uint32_t)y.w << 32;
    const uint64_t toff = (uint64_t)(uint32_t)z.x | (uint64_t)(uint32_t)z.y << 32;
    ts[k].set(tlen[k] > 0 ? A.target + toff : A.query + qoff, tlen[k]);
    DwordSeq qs;
    qs.set(A.query + qoff, qlen[k]);
    const int sh = qs.sh - ((8 - qlen[k]) & 7);  // byte of position 0 relative to the first dword
    const int d0 = sh >> 2, bs = sh & 3;
    uint32_t w0 = qs.at(d0);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint32_t w1 = qs.at(d0 + 2 * b + 1), w2 = qs.at(d0 + 2 * b + 2);
      const uint32_t lo = __builtin_amdgcn_alignbyte(w1, w0, (uint32_t)bs);
      const uint32_t hi = __builtin_amdgcn_alignbyte(w2, w1, (uint32_t)bs);
      uint32_t* s = (uint32_t*)&s_q[b][lane];
      s[k] = lo;
      s[2 + k] = hi;
      w0 = w2;
    }
  }
  __syncthreads();
  const u16x2 ql = pk2(qlen[0], qlen[1]), tl = pk2(have[0] ? tlen[0] : 0, have[1] ? tlen[1] : 0);
  const u16x2 off = pk2((8 - qlen[0]) & 7, (8 - qlen[1]) & 7), qpos = ql + off;
  const u16x2 offbit = pk2(1 << ((8 - qlen[0]) & 7), 1 << ((8 - qlen[1]) & 7));
  const u16x2 wv = pk2(w[0], w[1]);
  const u16x2 qcap = qpos * splat(kEndStep / 8);  // kEndStep per block of the query

  const u16x2 hh0 = pk2(h0[0], h0[1]);

  // ---- state ----
  u16x2 G[Q], E[Q];
  {  // first row (ksw.c:395-397): eh[0].h = h0, eh[j].h = max(h0 - oe_ins - (j-1)*e_ins, 0)
    const u16x2 hh = hh0;
    u16x2 ramp = pksat(hh, oe_ins), cap = smin(qpos, wv + off + splat(1u)) * splat(kStep);  // nothing past the first row's band
#pragma unroll
    for (int p = 0; p < Q; ++p) {
      u16x2 g;
      if (p < 8) {  // position off holds column 0; nothing before it
        const u16x2 at = (offbit >> (uint16_t)p) & splat(1u);  // column 0 here
        const u16x2 before = one_if(offbit >> (uint16_t)(p + 1));
        const u16x2 after = splat(1u) - at - before;
        g = at * hh + after * ramp;
        ramp = pksat(ramp, after * e_ins);
      } else {
        g = ramp;
        ramp = pksat(ramp, e_ins);
      }
      g = pkmin(g, cap);
      cap = pksat(cap, splat(kStep));
      G[p] = one_if(g) * a_ + g;
      E[p] = splat(0u);
    }
  }
  u16x2 beg = splat(0u), end = ql;  // columns, not positions
  u16x2 emax = smin(ql, wv + splat(1u));  // largest end so far
  // first-row values past the first row's band, of any task of the wave
  const bool ramped = __any(pku(pksat(pksat(hh0, oe_ins), emul(emax - splat(1u), e_ins)) &
                                pk(negmask(emax - ql))) != 0);
  u16x2 fcol = pksat(hh0, splat((uint32_t)min(A.o_del, 0xffff)));  // first-column value before row 0
  u16x2 best = hh0, best_i = splat(0xffffu), best_j = splat(0xffffu);
  u16x2 gbest = splat(0xffffu), gbest_i = splat(0xffffu), moff = splat(0u);
  uint32_t ncell[2] = {0, 0};
  uint32_t act = ~negmask(tl - splat(1u));  // halves whose task runs
  const u16x2 zd = splat((uint32_t)(A.zdrop > 0 && A.zdrop < 1023 ? A.zdrop : 1023));
  beg = beg & pk(act);
  end = end & pk(act);

  // target bases: dwords k, k+1 of the running 4-row window and the one after
  uint32_t tw0[2], tw1[2], tw2[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) { tw0[k] = ts[k].at(0); tw1[k] = ts[k].at(1); tw2[k] = ts[k].at(2); }
  uint32_t t4[2] = {0, 0};

  for (int i = 0; __any(act != 0); ++i) {
    if ((i & 3) == 0) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        t4[k] = __builtin_amdgcn_alignbyte(tw1[k], tw0[k], (uint32_t)ts[k].sh);
        tw0[k] = tw1[k];
        tw1[k] = tw2[k];
        tw2[k] = ts[k].at((i >> 2) + 3);
      }
    }
    const uint2 sa = trow[min(t4[0] & 0xffu, 7u)], sb = trow[min(t4[1] & 0xffu, 7u)];
    t4[0] >>= 8;
    t4[1] >>= 8;
    const u16x2 iv = splat((uint32_t)i);
    // band of the row (ksw.c:413-416)
    // The cap i-w moves beg by one column at most (the row before had i-1-w);
    // the live test below still counts the old one, whose block then zeroes it.
    const u16x2 beg0 = beg;
    const u16x2 cut = smax(iv - wv, splat(0u)) & pk(act);
    beg = smax(beg, cut);
    const bool capped = __any(pku(beg) != pku(beg0));
    end = smin(smin(end, iv + wv + splat(1u)), ql) & pk(act);
    fcol = pksat(fcol, e_del);
    fcol = fcol & pk(negmask(beg - splat(1u)));  // only while beg == 0
    const u16x2 fc1 = fcol + one_if(fcol) * a_;
    const u16x2 endp = end + off;
    // blocks with a column in [beg, end] of a running task
    u16x2 newcol = splat(0u), newg = splat(0u);
    bool grown = false;
    if (ramped) {
      const u16x2 nc = emax + splat(1u);
      const u16x2 r = pksat(pksat(hh0, oe_ins), emul(emax, e_ins)) & pk(negmask(nc - end));
      newg = r + one_if(r) * a_;
      newcol = nc + off;
      grown = __any(pku(newg) != 0);
      emax = smax(emax, end);
    }
    uint32_t live;
    {
      const uint32_t ep = pku(smin(endp, qpos - splat(1u))), bp = pku(beg0 + off);
      const uint32_t e0 = ep & 0xffffu, e1 = ep >> 16, b0 = bp & 0xffffu, b1 = bp >> 16;
      uint32_t v0 = (2u << (e0 >> 3)) - (1u << (b0 >> 3)), v1 = (2u << (e1 >> 3)) - (1u << (b1 >> 3));
      v0 = (act & 0xffffu) ? v0 : 0u;
      v1 = (act >> 16) ? v1 : 0u;
      live = wave_or(v0 | v1);
    }
    const u16x2 x0 = endp * splat(kStep);

    u16x2 F = splat(0u), carry = splat(0u), mk = splat(0u), hk = splat(0u), lk = splat(0u), hl = splat(0u);
    auto block = [&](auto bb) {
      constexpr int b = decltype(bb)::value;
      if (live >> b & 1u) {
        const uint4 q = s_q[b][lane];
        u16x2 X = pksat(x0, splat(kStep * 8u * b));
        u16x2 kb = splat(0u), hb = splat(0u), eb = splat(0u);
        if (capped) {  // columns the cap cut off
          u16x2 d = splat(8u * b) - (beg + off);
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const uint32_t keep = ~negmask(d);
            G[8 * b + c] = G[8 * b + c] & pk(keep);
            E[8 * b + c] = E[8 * b + c] & pk(keep);
            d = d + splat(1u);
          }
        }
        if (grown) {  // a column the band reaches for the first time
          u16x2 d = newcol - splat(8u * b);
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            G[8 * b + c] = G[8 * b + c] | (newg & pk(negmask(one_if(d) - splat(1u))));
            d = d - splat(1u);
          }
        }
        u16x2 M[8];
#pragma unroll
        for (int c = 0; c < 8; c += 4) {
          const uint32_t pa = __builtin_amdgcn_perm(sa.y, sa.x, c < 4 ? q.x : q.z);
          const uint32_t pb = __builtin_amdgcn_perm(sb.y, sb.x, c < 4 ? q.y : q.w);
#pragma unroll
          for (int d = 0; d < 4; ++d)
            M[c + d] = pksat(G[8 * b + c + d], pk(__builtin_amdgcn_perm(pb, pa, 0x0c040c00u + 0x00010001u * d)));
        }
        auto column = [&](auto cc) {
          constexpr int c = decltype(cc)::value;
          const int p = 8 * b + c;
          const u16x2 h = pkmax(pkmax(M[c], E[p]), F);
          if (b == 0) G[p] = ((offbit >> (uint16_t)c) & splat(1u)) * fc1 + carry;  // carry is 0 up to column 0
          else G[p] = carry;
          const u16x2 t = one_if(h);
          carry = t * a_ + h;
          const u16x2 open = pksat(M[c], oe_del);
          E[p] = pkmax(pksat(E[p], e_del), open);
          X = pksat(X, step);
          F = pkmin(pkmax(SAME ? open : pksat(M[c], oe_ins), pksat(F, e_ins)), X);
          kb = pkmax(kb, h * skey + splat((uint32_t)c));
          hb = t * bit[c] + hb;
          eb = one_if(E[p]) * bit[c] + eb;
        };
        for_each_index(column, std::make_integer_sequence<int, 8>{});
        mk = pkmax(mk, kb + splat(8u * b));
        // last block with a non-zero H: its bits below its number
        hk = pkmax(hk, one_if(hb) * splat(256u * b) + hb);
        // first block with a non-zero E(j) or G(j): bits of E | H shifted to G's column
        const u16x2 cb = pk(pku(hb) << 1 | pku(eb));
        lk = pkmax(lk, one_if(cb) * splat(512u * (31u - b)) + cb);
        // the value carried out of the block that ends the query is H(i, qlen-1);
        // nothing is carried past it
        const u16x2 z = pksat(qcap, splat(kEndStep * (b + 1)));
        hl = pkmax(hl, pksat(carry, z));
        carry = pkmin(carry, z);
      } else {
        carry = splat(0u);
        F = splat(0u);
      }
    };
    for_each_index(block, std::make_integer_sequence<int, NB>{});

    // ---- end of row (ksw.c:449-470) ----
    const uint32_t some = negmask(beg - end);  // end > beg
    const u16x2 h1 = pksat(hl, one_if(hl) * a_);
    {
      const u16x2 ja = smax(end, beg);
      const uint32_t ge = ~negmask(ja - ql) & act;  // ja == qlen (ja <= qlen always)
      const uint32_t up = ge & ~negmask(pk(pku(h1)) - gbest);  // h1 >= gbest
      gbest_i = sel(up, iv, gbest_i);
      gbest = sel(up, h1, gbest);
    }
    {
      const uint32_t w2 = pku(end - beg) & some & act;
      ncell[0] += w2 & 0xffffu;
      ncell[1] += w2 >> 16;
    }
    const u16x2 m = mk >> (uint16_t)KB;
    const u16x2 mj = (mk & splat((1u << KB) - 1)) - off;
    const uint32_t better = negmask(best - m) & act;
    const u16x2 di = iv - best_i, dj = mj - best_j;
    const u16x2 dd = di - dj;
    const u16x2 gap = smax(dd * e_del, (splat(0u) - dd) * e_ins);
    uint32_t fin = negmask(m - splat(1u)) | (negmask(zd + gap - (best - m)) & ~better);
    const u16x2 mo = smax(mj - iv, iv - mj);
    moff = sel(better, smax(moff, mo), moff);
    best = sel(better, m, best);
    best_i = sel(better, iv, best_i);
    best_j = sel(better, mj, best_j);
    fin |= negmask(tl - iv - splat(2u));  // i + 1 >= tlen
    act &= ~fin;
    {
      int nb[2], ne[2];
      const uint32_t hk32 = pku(hk), lk32 = pku(lk);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const uint32_t hv = k ? hk32 >> 16 : hk32 & 0xffffu, lv = k ? lk32 >> 16 : lk32 & 0xffffu;
        ne[k] = (int)((hv >> 8) * 8) + 31 - (int)__builtin_clz((hv & 255u) | 1u);
        nb[k] = (int)((31u - (lv >> 9)) * 8) + (int)__builtin_ctz(lv | 0x10000u);
      }
      const u16x2 npos = pk2(ne[0], ne[1]) - off + splat(3u);
      end = smin(npos, ql) & pk(act);
      const u16x2 fz = one_if(fcol);  // eh[0].h > 0 keeps beg at 0
      beg = ((pk2(nb[0], nb[1]) - off) & pk(~negmask(splat(0u) - fz))) & pk(act);
    }
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (!have[k]) continue;
    auto h16 = [&](u16x2 v) { return k ? (int)((int32_t)pku(v) >> 16) : (int)(int16_t)(pku(v) & 0xffffu); };
    int4* rp = (int4*)(A.rec + (int64_t)task[k] * 8);
    rp[0] = make_int4(h16(best), h16(best_j) + 1, h16(best_i) + 1, h16(gbest_i) + 1);
    rp[1] = make_int4(h16(gbest), h16(moff), (int)ncell[k], 0);
  }
}

template <int Q>
void launch_pair_bin(const ExtKArgs& k, const ExtWork& wk, int bin, int64_t n, hipStream_t st) {
  const int64_t blocks = (n + 127) / 128;  // surplus blocks exit at once
  if (blocks < 1) return;
  time_begin(wk, time_of_bin(bin), st);
  const bool same = k.o_del + k.e_del == k.o_ins + k.e_ins;  // one gap-open value serves E and F
  hipLaunchKernelGGL((same ? ext_pair_kernel<Q, true> : ext_pair_kernel<Q, false>), dim3((unsigned)blocks), dim3(64),
                     0, st, k, (const ExtDesc*)wk.desc, (const uint32_t*)wk.counts, bin);
  time_end(wk, time_of_bin(bin), st);
}
template void launch_pair_bin<32>(const ExtKArgs&, const ExtWork&, int, int64_t, hipStream_t);
template void launch_pair_bin<64>(const ExtKArgs&, const ExtWork&, int, int64_t, hipStream_t);
template void launch_pair_bin<96>(const ExtKArgs&, const ExtWork&, int, int64_t, hipStream_t);
template void launch_pair_bin<128>(const ExtKArgs&, const ExtWork&, int, int64_t, hipStream_t);
template void launch_pair_bin<224>(const ExtKArgs&, const ExtWork&, int, int64_t, hipStream_t);

}  // namespace bsx
