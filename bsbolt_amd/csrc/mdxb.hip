// NM, MD:Z and XB:Z of a CIGAR: the tail of bwa_gen_cigar2
// (bsbolt/External/BWA/bwa.c:250-343) with getMethylationContext (bwa.c:180-197).
//
// One lane per task, 32 bases of an M op at a time: the window bases (2-bit) and
// the read's bytes become bit planes, one bit a base, so that a few logic
// operations give the word's methylation calls, their contexts and the MD
// mismatches, and the counts are population counts.  Only the calls and the
// mismatches are then visited one by one, to write their strings.  A task
// whose walk could leave its window or overflow its slots, or a read of fewer
// than 32 bases, is walked base by base instead.
//
// A walk of every base by every lane was bound by instructions: some lane of the
// wave always had a call or a mismatch, so each of 150 steps ran the whole body.
// 400,009 regions of 150 bp reads: 871 us then, 158 now, of which the vector
// instructions (5,400 a wave) take 59; the rest is the addresses of 139 loads and
// stores a wave, each of whose lanes touches lines of its own.
#include "bsx_internal.h"

namespace bsx {

__device__ __forceinline__ int pac_at(const uint8_t* __restrict__ pac, int64_t p) {
  return (pac[p >> 2] >> ((~p & 3) << 1)) & 3;
}

// A lane's output string: characters gather in a register and leave as one
// dword store per four (the slot is dword-aligned), or byte by byte otherwise.
struct StrOut {
  char* __restrict__ p;
  int len, cap;
  uint32_t acc;
  bool words;
  __device__ __forceinline__ bool put(int c) {
    if (len >= cap) return false;
    acc |= (uint32_t)(c & 0xff) << (8 * (len & 3));
    ++len;
    if ((len & 3) == 0) {
      if (words) {
        *(uint32_t*)(p + len - 4) = acc;
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) p[len - 4 + k] = (char)(acc >> (8 * k));
      }
      acc = 0;
    }
    return true;
  }
  __device__ __forceinline__ void flush() {
    for (int k = 0; k < (len & 3); ++k) p[(len & ~3) + k] = (char)(acc >> (8 * k));
  }
  // appends the decimal digits of v >= 0 (kputw, kstring.h:62-76); false on
  // overflow.  The digits gather in nibbles of one register, most significant
  // in the low nibble, so no array is indexed at run time.
  __device__ __forceinline__ bool put_int(int v) {
    uint64_t dg = 0;
    int n = 0;
    do {
      dg = (dg << 4) | (uint64_t)(v % 10);
      v /= 10;
      ++n;
    } while (v > 0);
    if (len + n > cap) return false;
    for (int k = 0; k < n; ++k) put('0' + (int)((dg >> (4 * k)) & 15));
    return true;
  }
};

struct MdRes {
  int st, nm, md_len, xb_len, cgm, cgu, chm, chu;
};

// What a task's walks share.
struct MdTask {
  int64_t k0, clen;  // window base k is forward position k0 + k, of clen bases
  const uint8_t* oq;
  const uint32_t* cig;
  char *md, *xb;
  int l_query, nc;
  bool fwd, is_crick;
  int o1, o2, o3;  // window offsets of the three context bases (bwa.c:290-293)
};

// The walk base by base.  On the reverse strand the reversed
// reverse-complement window is 3 - opac, and the read runs backwards.
__device__ __forceinline__ MdRes md_walk(const MdArgs& a, const MdTask& T, bool md_words, bool xb_words) {
  MdRes R{};
  bool oob = false;
  auto cs = [&](int64_t k) -> int {
    if (k < 0 || k >= T.clen) { oob = true; return 4; }
    const int b = pac_at(a.opac, T.k0 + k);
    return T.fwd ? b : 3 - b;
  };
  const int ref_base = T.is_crick ? 2 : 1, methyl_base = T.is_crick ? 0 : 3;
  const char* i2b = T.fwd ? "ACGTN" : "TGCAN";
  StrOut md{T.md, 0, (int)a.md_slot, 0u, md_words};
  StrOut xb{T.xb, 0, (int)a.xb_slot, 0u, xb_words};
  int x = 0, y = 0, u = 0, n_mm = 0, n_gap = 0, meth_pos = 0;
  for (int k = 0; k < T.nc && R.st == 0; ++k) {
    const int op = (int)(T.cig[k] & 0xfu), len = (int)(T.cig[k] >> 4);
    if (op == 0) {
      for (int pos = 0; pos < len && R.st == 0; ++pos) {
        const int c = cs(y + pos + 2);
        const int o = T.oq[T.fwd ? x + pos : T.l_query - 1 - x - pos];
        const bool isref = c == ref_base;
        const bool ev = isref && (o == ref_base || o == methyl_base);  // methylation call
        const bool mm = isref ? !ev : o != c;                           // MD mismatch
        if (isref) {
          const int b1 = cs(y + pos + T.o1), b2 = cs(y + pos + T.o2), b3 = cs(y + pos + T.o3);
          if (ev) {
            const bool meth = o == ref_base;
            const bool cg = b1 == 1 && b2 == 2, chg = !cg && b1 == 1 && b3 == 2;
            const char m = (char)((cg ? 'X' : chg ? 'Y' : 'Z') + (meth ? 0 : 32));
            R.cgm += meth && cg; R.chm += meth && !cg; R.cgu += !meth && cg; R.chu += !meth && !cg;
            if ((meth_pos > 0 && !xb.put_int(meth_pos)) || !xb.put(m)) R.st = -1;
          }
        }
        if (mm && (!md.put_int(u) || !md.put(i2b[c]))) R.st = -1;
        n_mm += mm;
        u = mm ? 0 : u + 1;
        meth_pos = ev ? 0 : meth_pos + 1;
        if (oob) R.st = -2;
      }
      x += len; y += len;
    } else if (op == 2) {
      if (k > 0 && k < T.nc - 1) {  // not for a leading or trailing D
        if (!md.put_int(u) || !md.put('^')) R.st = -1;
        for (int i = 0; i < len && R.st == 0; ++i)
          if (!md.put(i2b[cs(y + i + 2)])) R.st = -1;
        if (R.st == 0 && oob) R.st = -2;
        u = 0; n_gap += len;
      }
      y += len;
    } else if (op == 1) {
      x += len; n_gap += len; meth_pos += len;
    }
  }
  if (R.st == 0 && !md.put_int(u)) R.st = -1;
  if (R.st == 0 && meth_pos > 0 && !xb.put_int(meth_pos)) R.st = -1;
  if (R.st == 0) {
    md.flush();
    xb.flush();
  }
  R.nm = n_mm + n_gap; R.md_len = md.len; R.xb_len = xb.len;
  return R;
}

// even bits of x to its low half, odd bits to its high half
__device__ __forceinline__ uint32_t unshuffle(uint32_t x) {
  uint32_t t = (x ^ (x >> 1)) & 0x22222222u;
  x ^= t ^ (t << 1);
  t = (x ^ (x >> 2)) & 0x0c0c0c0cu;
  x ^= t ^ (t << 2);
  t = (x ^ (x >> 4)) & 0x00f000f0u;
  x ^= t ^ (t << 4);
  t = (x ^ (x >> 8)) & 0x0000ff00u;
  return x ^ t ^ (t << 8);
}

// A string as its length in bits and the characters of its last, unfinished dword.
struct BitStr {
  char* __restrict__ p;
  uint32_t bits, acc;
};

// Appends the low n bits (8 to 32) of s, whose upper bits are 0; false if they
// do not fit.
__device__ __forceinline__ bool append(BitStr& o, uint32_t s, uint32_t n, uint32_t cap_bits, bool words) {
  const uint32_t to = o.bits + n;
  if (to > cap_bits) return false;
  const uint64_t v = (uint64_t)s << (o.bits & 31);
  const uint32_t lo = o.acc | (uint32_t)v;
  const bool full = (to ^ o.bits) >> 5;
  if (full) {
    char* d = o.p + (o.bits >> 5 << 2);
    if (words) {
      *(uint32_t*)d = lo;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) d[k] = (char)(lo >> (8 * k));
    }
  }
  o.acc = full ? (uint32_t)(v >> 32) : lo;
  o.bits = to;
  return true;
}

__device__ __forceinline__ void finish(const BitStr& o) {
  for (uint32_t k = 0; k < (o.bits >> 3 & 3); ++k) o.p[(o.bits >> 5 << 2) + k] = (char)(o.acc >> (8 * k));
}

constexpr int kMdBlock = 128;
constexpr int kMdNums = 1000;  // numbers written from a table of their digits

// Bit j of a plane from byte j of 32 (v[0..7]): weights 1, 2, 4, ... over the
// bytes' bit `mask`; scaled by that bit's value.
__device__ __forceinline__ uint32_t plane_of(const uint32_t (&v)[8], uint32_t mask, int shift) {
  uint32_t r = 0;
#pragma unroll
  for (int k = 0; k < 8; k += 2) {
    const uint32_t b = __builtin_amdgcn_udot4(
        v[k + 1] & mask, 0x80402010u, __builtin_amdgcn_udot4(v[k] & mask, 0x08040201u, 0u, false), false);
    r |= (b >> shift) << (4 * k);
  }
  return r;
}

// bases between the start of the reference's first dword and its first byte
__device__ __forceinline__ int md_lead(const MdArgs& a) { return 4 * (int)((uintptr_t)a.opac & 3); }

// The walk by words; st is 1 where only md_walk can tell (a slot overflows or a
// number has four digits).  The caller has checked that the walk stays in its
// window, that three dwords past the window's last lie in the reference, and
// that the read has 32 bases.
__device__ __forceinline__ MdRes md_words_walk(const MdArgs& a, const MdTask& T, const uint32_t* __restrict__ num,
                                               bool md_words, bool xb_words) {
  MdRes R{};
  // the reference from its first byte's dword on
  const uint32_t* __restrict__ opac32 = (const uint32_t*)((uintptr_t)a.opac & ~(uintptr_t)3);
  const int lead = md_lead(a);
  const uint32_t flip = T.fwd ? 0u : ~0u;
  const uint32_t i2b = T.fwd ? 0x54474341u : 0x41434754u;  // "ACGT", "TGCA"
  const uint32_t md_cap = (uint32_t)(a.md_slot < (1 << 28) ? a.md_slot : 1 << 28) * 8;
  const uint32_t xb_cap = (uint32_t)(a.xb_slot < (1 << 28) ? a.xb_slot : 1 << 28) * 8;
  BitStr md{T.md, 0u, 0u}, xb{T.xb, 0u, 0u};
  // bases of M ops walked (mpos), and the ones up to which the two strings have
  // counted (u0, m0; m0 goes back by the bases of an I)
  int x = 0, y = 0, mpos = 0, u0 = 0, m0 = 0, n_mm = 0, n_gap = 0;
  bool bad = false;
  auto number = [&](BitStr& o, int v, uint32_t ch, uint32_t chbits, bool zero, uint32_t cap, bool words) {
    if ((uint32_t)v >= (uint32_t)kMdNums) { bad = true; return; }
    uint32_t e = num[v];  // digits, and their bits in the top byte
    e = v == 0 && !zero ? 0u : e;
    const uint32_t sh = e >> 24;
    if (!append(o, (e & 0xffffffu) | ch << (sh & 31), sh + chbits, cap, words)) bad = true;
  };
  int k = 0, rem = 0;
  while (!bad && (rem > 0 || k < T.nc)) {
    if (rem == 0) {
      const uint32_t cw = T.cig[k++];
      const int op = (int)(cw & 0xfu), len = (int)(cw >> 4);
      if (op == 0) {
        rem = len;
      } else if (op == 1) {
        x += len; n_gap += len; m0 -= len;
      } else {
        if (k > 1 && k < T.nc) {  // not for a leading or trailing D
          number(md, mpos - u0, '^', 8, true, md_cap, md_words);
          for (int i = 0; i < len && !bad; ++i) {
            const int b = pac_at(a.opac, T.k0 + y + i + 2) ^ (int)(flip & 3);
            if (!append(md, i2b >> (8 * b) & 0xffu, 8, md_cap, md_words)) bad = true;
          }
          u0 = mpos; n_gap += len;
        }
        y += len;
      }
      if (op != 0 || len == 0) continue;
    }
    const int nb = min(rem, 32);
    // ---- window bases [y, y + 36) as planes (H: high bits of the codes, L: low) ----
    const int64_t p = T.k0 + y + lead;
    uint32_t d[4];
    __builtin_memcpy(d, opac32 + (p >> 4), 16);
    // base i of a dword's 16: bits 2i (high) and 2i + 1 (low)
#pragma unroll
    for (int q = 0; q < 4; ++q) d[q] = __builtin_bitreverse32(__builtin_bswap32(d[q]));
    const uint32_t sh = 2u * (uint32_t)(p & 15);
    const uint32_t s0 = unshuffle(__builtin_amdgcn_alignbit(d[1], d[0], sh) ^ flip);
    const uint32_t s1 = unshuffle(__builtin_amdgcn_alignbit(d[2], d[1], sh) ^ flip);
    const uint32_t s2 = unshuffle((__builtin_amdgcn_alignbit(d[3], d[2], sh) ^ flip) & 0xffu);
    const uint32_t H = (s0 & 0xffffu) | s1 << 16, L = s0 >> 16 | (s1 & 0xffff0000u);
    const uint32_t h2 = s2 & 0xffffu, l2 = s2 >> 16;
    const uint32_t Cl = ~H & L, Ch = ~h2 & l2, Gl = H & ~L, Gh = h2 & ~l2;
    const uint32_t cH = __builtin_amdgcn_alignbit(h2, H, 2), cL = __builtin_amdgcn_alignbit(l2, L, 2);
    const uint32_t ref = __builtin_amdgcn_alignbit(T.is_crick ? Gh : Ch, T.is_crick ? Gl : Cl, 2);
    const uint32_t b1 = __builtin_amdgcn_alignbit(Ch, Cl, (uint32_t)T.o1);
    const uint32_t CG = b1 & __builtin_amdgcn_alignbit(Gh, Gl, (uint32_t)T.o2);
    const uint32_t CHG = b1 & __builtin_amdgcn_alignbit(Gh, Gl, (uint32_t)T.o3);
    // ---- read bases [x, x + 32), from the 32 bases of the read that hold those of them that it has ----
    const int sb = min(x, T.l_query - 32);
    const uintptr_t at = (uintptr_t)T.oq + (uint32_t)(T.fwd ? sb : T.l_query - 32 - sb);
    const uint32_t* __restrict__ rp = (const uint32_t*)(at & ~(uintptr_t)3);
    const uint32_t bs = (uint32_t)(at & 3);
    uint32_t r[8];
    __builtin_memcpy(r, rp, 32);
    const uint32_t r8 = rp[bs ? 8 : 7];
#pragma unroll
    for (int q = 0; q < 8; ++q) r[q] = __builtin_amdgcn_alignbyte(q < 7 ? r[q + 1] : r8, r[q], bs);
    uint32_t rH = plane_of(r, 0x02020202u, 1), rL = plane_of(r, 0x01010101u, 0), rN = 0;
    uint32_t any = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) any |= r[q];
    if (any & 0xfcfcfcfcu) {  // codes past 3
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const uint32_t v = r[q] & 0xfcfcfcfcu;
        r[q] = (((v & 0x7f7f7f7fu) + 0x7f7f7f7fu) | v) >> 7;
      }
      rN = plane_of(r, 0x01010101u, 0);
    }
    if (!T.fwd) {
      rH = __builtin_bitreverse32(rH);
      rL = __builtin_bitreverse32(rL);
      rN = __builtin_bitreverse32(rN);
    }
    const int skip = x - sb;
    rH >>= skip; rL >>= skip; rN >>= skip;
    // ---- calls and mismatches ----
    const uint32_t in = nb == 32 ? ~0u : (1u << nb) - 1u;
    const uint32_t refo = ~rN & (T.is_crick ? rH & ~rL : ~rH & rL);   // the read has the reference's base
    const uint32_t conv = ~rN & (T.is_crick ? ~(rH | rL) : rH & rL);  // ... the converted one
    uint32_t ev = ref & (refo | conv) & in;
    uint32_t mm = ((ref & ~ev) | (~ref & (rN | (rH ^ cH) | (rL ^ cL)))) & in;
    R.cgm += __builtin_popcount(ev & refo & CG);
    R.chm += __builtin_popcount(ev & refo & ~CG);
    R.cgu += __builtin_popcount(ev & ~refo & CG);
    R.chu += __builtin_popcount(ev & ~refo & ~CG);
    n_mm += __builtin_popcount(mm);
    while (ev != 0 && !bad) {
      const int j = __builtin_ctz(ev);
      ev &= ev - 1;
      const uint32_t cg = CG >> j & 1u, chg = CHG >> j & 1u & ~cg;
      const uint32_t ch = (uint32_t)'Z' - 2 * cg - chg + 32u * (~refo >> j & 1u);
      number(xb, mpos + j - m0, ch, 8, false, xb_cap, xb_words);
      m0 = mpos + j + 1;
    }
    while (mm != 0 && !bad) {
      const int j = __builtin_ctz(mm);
      mm &= mm - 1;
      const uint32_t c = (cH >> j & 1u) * 2 + (cL >> j & 1u);
      number(md, mpos + j - u0, i2b >> (8 * c) & 0xffu, 8, true, md_cap, md_words);
      u0 = mpos + j + 1;
    }
    mpos += nb; x += nb; y += nb; rem -= nb;
  }
  if (!bad) number(md, mpos - u0, 0, 0, true, md_cap, md_words);
  if (!bad && mpos - m0 > 0) number(xb, mpos - m0, 0, 0, false, xb_cap, xb_words);
  if (!bad) {
    finish(md);
    finish(xb);
  }
  R.st = bad ? 1 : 0;
  R.nm = n_mm + n_gap; R.md_len = (int)(md.bits >> 3); R.xb_len = (int)(xb.bits >> 3);
  return R;
}

__global__ void __launch_bounds__(kMdBlock) md_kernel(MdArgs a) {
  __shared__ uint32_t num[kMdNums];
  for (int v = threadIdx.x; v < kMdNums; v += kMdBlock) {
    const uint32_t h = v / 100, t = v / 10 % 10, o = v % 10, d = v >= 100 ? 3 : v >= 10 ? 2 : 1;
    num[v] = ((('0' + h) | ('0' + t) << 8 | ('0' + o) << 16) >> (8 * (3 - d))) | (8 * d) << 24;
  }
  __syncthreads();
  // dword stores for the strings when every slot starts on a dword
  const bool md_words = ((uintptr_t)a.md & 3) == 0 && (a.md_slot & 3) == 0;
  const bool xb_words = ((uintptr_t)a.xb & 3) == 0 && (a.xb_slot & 3) == 0;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < a.n; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t rb = a.rb[t], re = a.re[t], l_pac = a.l_pac;
    MdTask T;
    T.l_query = a.l_query[t];
    T.nc = a.n_cigar[t];
    T.cig = a.cigar + t * a.cigar_slot;
    T.md = a.md + t * a.md_slot;
    T.xb = a.xb + t * a.xb_slot;
    MdRes R{};
    int64_t ysum = 0;
    {  // a region bwa_gen_cigar2 makes a CIGAR for, whose CIGAR fits its slot
       // and consumes at most the read
      bool bad = rb < 0 || rb >= re || re > 2 * l_pac || T.nc < 0 || (int64_t)T.nc > a.cigar_slot;
      int64_t qsum = 0;
      for (int k = 0; k < T.nc && !bad; ++k) {
        const uint32_t op = T.cig[k] & 0xfu, len = T.cig[k] >> 4;
        if (op > 2) bad = true;
        qsum += op == 2 ? 0 : len;
        ysum += op == 1 ? 0 : len;
      }
      if (bad || qsum > T.l_query) R.st = -3;
    }
    // window opac[rb-2, re+2) as bns_get_seq clamps it (rb < re, so no swap)
    const int64_t beg = max(rb - 2, (int64_t)0), end = min(re + 2, 2 * l_pac);
    // bridges the strands: the reference stops (bwa.c:262)
    if (R.st == 0 && !(beg >= l_pac || end <= l_pac)) R.st = 1;
    if (R.st == 0) {
      T.clen = end - beg;
      T.fwd = rb < l_pac;  // rb >= l_pac: window and read reversed (bwa.c:264-271)
      // base k of the window in the order the walk reads it: forward positions
      // beg + k; on the reverse strand the reversed reverse-complement window,
      // which is 3 - opac[2*l_pac - end + k]
      T.k0 = T.fwd ? beg : 2 * l_pac - end;
      T.oq = a.oquery + a.oq_off[t];
      const bool reverse = rb > l_pac;  // bwa.c:212 (strictly greater)
      T.is_crick = (rb >= a.crick_l && rb < l_pac) || rb >= a.crick_l + l_pac;
      // after the base on the forward Watson copy, around it on the others
      T.o1 = !reverse ? (!T.is_crick ? 2 : 1) : (!T.is_crick ? 2 : 3);
      T.o2 = !reverse ? (!T.is_crick ? 3 : 2) : (!T.is_crick ? 1 : 2);
      T.o3 = !reverse ? (!T.is_crick ? 4 : 3) : (!T.is_crick ? 0 : 1);
      const int lead = md_lead(a);
      const bool words = ysum + 4 <= T.clen && T.l_query >= 32 &&
                         ((T.k0 + T.clen + lead) >> 4) + 3 <= (l_pac - 1 + lead) >> 4;
      R.st = 1;
      if (words) R = md_words_walk(a, T, num, md_words, xb_words);
      if (R.st != 0) R = md_walk(a, T, md_words, xb_words);
    }
    const bool ok = R.st == 0;
    a.status[t] = R.st;
    a.nm[t] = ok ? R.nm : -1;
    a.md_len[t] = ok ? R.md_len : 0;
    a.xb_len[t] = ok ? R.xb_len : 0;
    int32_t* meth = a.meth + 4 * t;
    meth[0] = ok ? R.cgm : 0;
    meth[1] = ok ? R.cgu : 0;
    meth[2] = ok ? R.chm : 0;
    meth[3] = ok ? R.chu : 0;
  }
}

hipError_t launch_md(const MdArgs& a, int num_cu, hipStream_t st) {
  if (a.n <= 0) return hipSuccess;
  int64_t blocks = (a.n + kMdBlock - 1) / kMdBlock;
  if (blocks > (int64_t)num_cu * 64) blocks = (int64_t)num_cu * 64;
  hipLaunchKernelGGL(md_kernel, dim3((unsigned)blocks), dim3(kMdBlock), 0, st, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The tail of mem_reg2aln (bwamem.c:1237-1263): the SAM CIGAR of a region from
// the CIGAR bwa_gen_cigar2 made for it.  The position is bns_depos of rb (or
// of re - 1 on the reverse strand); a leading deletion is squeezed out and
// moves the position, or else (only if the first op is not one) a trailing
// deletion is dropped; then the unaligned read ends become clip ops
// (len << 4 | 3), 5' first, swapped on the reverse strand.  One lane per task:
// a handful of words each.
__global__ void __launch_bounds__(256)
reg2aln_cigar_kernel(Reg2alnArgs a) {
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < a.n;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t rb = a.rb[t], re = a.re[t];
    const int qb = a.qb[t], qe = a.qe[t], lq = a.l_seq[t], nc = a.n_cigar[t];
    const uint32_t* __restrict__ c = a.cigar + t * a.cigar_slot;
    if (nc < 0 || nc > a.cigar_slot || rb < 0 || re <= rb || re > 2 * a.l_pac || qb < 0 || qe < qb || qe > lq) {
      a.out_n[t] = -1;
      a.pos[t] = -1;
      a.is_rev[t] = 0;
      continue;
    }
    const int64_t p0 = rb < a.l_pac ? rb : re - 1;  // bns_depos (bntseq.h)
    const bool rev = p0 >= a.l_pac;
    int64_t pos = rev ? 2 * a.l_pac - 1 - p0 : p0;
    int first = 0, last = nc;
    if (nc > 0) {
      if ((c[0] & 0xf) == 2) {
        pos += c[0] >> 4;
        first = 1;
      } else if ((c[nc - 1] & 0xf) == 2) {
        last = nc - 1;
      }
    }
    int clip5 = 0, clip3 = 0;
    if (qb != 0 || qe != lq) {
      clip5 = rev ? lq - qe : qb;
      clip3 = rev ? qb : lq - qe;
    }
    const int n_out = (clip5 ? 1 : 0) + (last - first) + (clip3 ? 1 : 0);
    a.pos[t] = pos;
    a.is_rev[t] = rev ? 1 : 0;
    if (n_out > a.out_slot) {
      a.out_n[t] = -2;
      continue;
    }
    uint32_t* __restrict__ o = a.out + t * a.out_slot;
    int k = 0;
    if (clip5) o[k++] = (uint32_t)clip5 << 4 | 3u;
    for (int j = first; j < last; ++j) o[k++] = c[j];
    if (clip3) o[k++] = (uint32_t)clip3 << 4 | 3u;
    a.out_n[t] = k;
  }
}

hipError_t launch_reg2aln_cigar(const Reg2alnArgs& a, int num_cu, hipStream_t st) {
  if (a.n <= 0) return hipSuccess;
  int64_t blocks = (a.n + 255) / 256;
  if (blocks > (int64_t)num_cu * 16) blocks = (int64_t)num_cu * 16;
  hipLaunchKernelGGL(reg2aln_cigar_kernel, dim3((unsigned)blocks), dim3(256), 0, st, a);
  return hipGetLastError();
}

}  // namespace bsx
