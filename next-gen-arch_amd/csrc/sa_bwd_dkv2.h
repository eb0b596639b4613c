// dk2 / dv2 pass of the matrix-core backward: both gradients of a long key
// from one score tile (archlab/architectures/simplicial_kernels.py:75-101).
//
// A workgroup of 4 waves owns 128 SETS consecutive long keys of one KV head;
// wave w holds the K2 / V2 rows of SETS blocks of 32 of them (keys k0 + 128 c +
// 32 w ..) as MFMA fragments and both gradients' accumulators.  It walks the
// units (t, h, r) that reach its keys: query t, head h of the group, 32-row
// group r of t's short keys.  A step takes one unit -- or, with short windows
// of at most 16 (8) keys, PK = 2 (4) units of 16 (8) rows each, so that no
// MFMA row is spent on keys outside the window -- whose A rows bf16(q_th ⊙
// k1_j) and B rows bf16(dout_th ⊙ v1_j) the four waves form in LDS for the
// next step while this one's products run (double-buffered, one barrier per
// step).  Then, per set (BwdCore, rows j x keys):
//     S = A_t · K2^T,  dP = B_t · V2^T,  dV2^T += B_t^T · P,  dK2^T += A_t^T · dS
//
// The q, dout, k1_t and v1_t rows of a unit are staged by the last wave with
// full-wave DMAs two steps ahead; k1 / v1 rows of earlier queries come from a
// ring (row j at slot j % ring) into which wave 0 copies the staged rows.
//
// Measured, forward + backward (this pass in place of one launch per gradient,
// which formed the rows and the scores twice): adapter shape (2 x 8192 tokens,
// 8 / 2 heads, width 128, windows 32 x 512) bf16 8.39 -> 7.66 ms, fp32 18.96 ->
// 17.01 ms; width 256, windows 64 x 256, 8192 tokens 12.03 -> 9.69 ms; 16 short
// keys (2 x 4099 tokens, 16 / 4 heads, 16 x 512) 8.62 -> 7.06 ms.  What bounds
// it now (counters, adapter shape in bf16): one wave per SIMD, whose chain nothing
// hides.  It issues in half of its cycles (a step is 535 vector, 64 matrix, 76 LDS
// and 123 scalar instructions), waits in 38 % -- on the step's barrier and on reloads
// of spilled values (60 bytes a lane), which in the staging wave wait for the DMA
// that it has just issued too -- and the matrix cores are busy in 31 %.  fp32 (no
// spills): 45, 39 and 38 %.
//
// Score width 512 (determinant form of 256-wide heads): the accumulators of
// 512 + 256 columns do not fit; one launch takes dV2 and 128 columns of dK2, a
// second one the other 384, with the scores formed in both.
//
// Walks are cut into pieces when the (key block, KV head) workgroups alone
// leave CUs idle in the last wave of workgroups: each piece writes fp32 sums
// that bwd_dkv2_sum_kernel adds in piece order (no atomics).
#pragma once

#include "sa_bwd_core.h"
#include "sa_bwd_walk.h"
#include "sa_launch.h"
#include "sa_backward.h"

#include <algorithm>

namespace sa {

namespace {

struct Dkv2Geo {
  int nblocks;  // workgroups
  int kblocks;  // key blocks
  int splits;   // pieces per walk
  int nr;       // 32-row groups of short keys (1 with PK > 1)
  int ring;     // k1 / v1 ring rows (a power of two)
};

// LDS of a workgroup: two tile pairs, the ring, two stage slots, per-wave scalars
template <int DK, int DV, int PK, bool F32>
struct Dkv2Lds {
  static constexpr int EW = F32 ? 2 : 1;                            // bf16 units per element
  static constexpr int RBK = 2 * EW * DK, RBV = 2 * EW * DV;        // q / k1 and dout / v1 row bytes
  static constexpr int RKV = RBK + RBV;
  static constexpr int SS = (2 * RKV + 1023) / 1024 * 1024;         // stage bytes of one unit
  static constexpr int SI = SS / 1024;                              // ... and its DMA instructions
  static constexpr int TAB = 32 * RKV;                              // one A + B tile pair
  static constexpr int NW = 4;
  static constexpr size_t bytes(int ring) { return 2 * TAB + (size_t)ring * RKV + 2 * PK * SS + NW * 64 * 16; }
};

template <int DK, int DV, int SETS, int PK, bool F32, int KB0, int KBN, int VBN>
__global__ __launch_bounds__(256, 1) void bwd_dkv2_kernel(BwdParams p, Dkv2Geo geo) {
  using L = Dkv2Lds<DK, DV, PK, F32>;
  using C = BwdCore<DK, DV, SETS, F32, KB0, KBN, VBN>;
  constexpr int NW = 4, KB = 128 * SETS, R = 32 / PK, EW = L::EW;
  constexpr int RBK = L::RBK, RKV = L::RKV, SS = L::SS, SI = L::SI, TAB = L::TAB;
  static_assert(!F32 || DK == DV, "fp32 inputs: equal widths");
  extern __shared__ __attribute__((aligned(256))) char lds[];
  char* const ring = lds + 2 * TAB;               // [geo.ring][k1 row, v1 row]
  char* const stage = ring + geo.ring * RKV;      // [2][PK][q, dout, k1_t, v1_t rows]

  const int tid = tid_x(), lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, n = lane & 31;
  floatx4* const scal = (floatx4*)(stage + 2 * PK * SS) + 64 * wid;  // this wave's scalars of 64 units

  const int lb = xcd_remap(bid_x(), geo.nblocks);
  const int kb = lb % geo.kblocks;
  const int g = lb / geo.kblocks % p.hk, split = lb / geo.kblocks / p.hk;
  const int k0 = kb * KB, last = p.tokens - 1;
  const int G = p.group, nr = geo.nr;
  const int64_t kvg_k = (int64_t)g * p.k_sh, kvg_v = (int64_t)g * p.v_sh;

  // Walk: the queries that reach the block's keys, t = k0 .. the last key's
  // window end, no further than the last key's sequence; piece `split` of it.
  const int kl = min(last, k0 + KB - 1);
  auto seq_end = [&](int t) {  // one past the last token of token t's sequence (t < p.tokens)
    int e;
    if (p.cu == nullptr) {
      e = (t / p.seqlen + 1) * p.seqlen;
    } else {
      int lo = 0, hi = p.num_seqs - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (p.cu[mid] <= t) lo = mid;
        else hi = mid - 1;
      }
      e = p.cu[lo + 1];
    }
    return __builtin_amdgcn_readfirstlane(max(min(e, p.tokens), t + 1));
  };
  const int send = seq_end(kl);
  const int walk = min(send - 1, k0 + KB - 1 + p.wl - 1) - k0 + 1;
  const int tfirst = k0 + (int)((int64_t)walk * split / geo.splits);
  const int tlast = k0 + (int)((int64_t)walk * (split + 1) / geo.splits) - 1;
  const int nunits = (tlast - tfirst + 1) * G * nr;
  const int nsteps = (nunits + PK - 1) / PK;

  C core;
  core.clear();
  // acc[db] register e holds d = 32 db + acc_row(e, half) of key k0 + 128 c + 32 wid + n
  auto write_out = [&]() {
    acc_settle();
    const int lf = fresh_lane();
    const int nf = lf & 31, hf = lf >> 5;
#pragma unroll
    for (int c = 0; c < SETS; ++c) {
      const int kw = k0 + 128 * c + 32 * wid + nf;
      if (kw >= p.tokens) continue;
      if (geo.splits > 1) {
        float* part = p.dkv2s + (((int64_t)split * p.tokens + kw) * p.hk + g) * (DK + DV);
#pragma unroll
        for (int i = 0; i < 4 * (KBN + VBN); ++i) {
          const int db = i >> 2, q4 = i & 3;
          floatx4 x;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            x[e] = db < KBN ? acc_get(core.ak[c][db < KBN ? db : 0], 4 * q4 + e)
                            : acc_get(core.av[c][db < KBN ? 0 : db - KBN], 4 * q4 + e);
          *(floatx4*)(part + (db < KBN ? 32 * (KB0 + db) : DK + 32 * (db - KBN)) + 8 * q4 + 4 * hf) = x;
        }
        continue;
      }
      const int64_t ok = (int64_t)kw * p.dk_st + (int64_t)g * p.dk_sh, ov = (int64_t)kw * p.dv_st + (int64_t)g * p.dv_sh;
#pragma unroll
      for (int db = 0; db < KBN; ++db) {
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int d = 32 * (KB0 + db) + 8 * q4 + 4 * hf;
          if constexpr (F32) {
            floatx4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = acc_get(core.ak[c][db], 4 * q4 + e);
            *(floatx4*)((float*)p.dk2 + ok + d) = x;
          } else {
            bf16x4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = (bf16)acc_get(core.ak[c][db], 4 * q4 + e);
            *(bf16x4*)((bf16*)p.dk2 + ok + d) = x;
          }
        }
      }
#pragma unroll
      for (int db = 0; db < VBN; ++db) {
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int d = 32 * db + 8 * q4 + 4 * hf;
          if constexpr (F32) {
            floatx4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = acc_get(core.av[c][db], 4 * q4 + e);
            *(floatx4*)((float*)p.dv2 + ov + d) = x;
          } else {
            bf16x4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = (bf16)acc_get(core.av[c][db], 4 * q4 + e);
            *(bf16x4*)((bf16*)p.dv2 + ov + d) = x;
          }
        }
      }
    }
  };
  if (nsteps <= 0) {  // an empty piece (uniform, before any barrier): zero sums
    write_out();
    return;
  }

  // Unit state, carried from step to step (no divisions in the step loop).
  using Unit = WalkUnit;
  auto advance = [&](Unit u) { return walk_next(u, G, nr); };
  auto after = [&](Unit u) {  // the first unit of the next step
#pragma unroll
    for (int s = 0; s < PK; ++s) u = advance(u);
    return u;
  };

  // Stage slot st % 2: per unit its q, dout, k1_t and v1_t rows end to end
  // (lanes past them re-fetch the first segment into the unused tail); units
  // past the walk stage its last unit's rows again (walk_moves: nothing past
  // them is read, and their zero probabilities multiply rows that the walk
  // multiplies anyway).  A lane's tensor
  // is fixed by its byte offset: its row pointer is carried from unit to unit
  // (next head: + one head stride; next query: + the rest of a token stride),
  // in place of four row addresses and a selection per step.
  constexpr int kDmaWave = NW - 1;
  const char* dptr[SI];
  int dhead[SI], dtok[SI];  // pointer steps, 16-byte units (16-byte rows: strides are multiples)
#pragma unroll
  for (int k = 0; k < SI; ++k) {
    int b = 1024 * k + 16 * lane;
    if (b >= 2 * RKV) b = 0;
    const bool isq = b < RBK, isg = b < RKV, isk = b < RKV + RBK;
    const bf16* base = (const bf16*)(isq ? p.q : isg ? p.dout : isk ? p.k1 : p.v1);
    const int64_t st_t = EW * (isq ? p.q_st : isg ? p.do_st : isk ? p.k_st : p.v_st);
    const int64_t st_h = EW * (isq ? p.q_sh : isg ? p.do_sh : isk ? p.k_sh : p.v_sh);
    const int inrow = b - (isq ? 0 : isg ? RBK : isk ? RKV : RKV + RBK);
    dptr[k] = (const char*)(base + (int64_t)tfirst * st_t + (int64_t)(isg ? g * G : g) * st_h) + inrow;
    dhead[k] = isg ? (int)(st_h / 8) : 0;
    dtok[k] = (int)walk_query_step(st_t / 8, st_h / 8, isg ? G : 1);
  }
  Unit dunit{tfirst, 0, 0};
  auto dma_step = [&](int st) {  // called for st = 0, 1, 2, ..
    if (wid != kDmaWave || st >= nsteps) return;
#pragma unroll
    for (int s = 0; s < PK; ++s) {
#pragma unroll
      for (int k = 0; k < SI; ++k) dma16(dptr[k], stage + ((st & 1) * PK + s) * SS + 1024 * k);
      const Unit y = advance(dunit);
      if (walk_moves(dunit, y, st * PK + s, nunits, PK)) {
#pragma unroll
        for (int k = 0; k < SI; ++k) dptr[k] += (int64_t)(y.t == dunit.t ? dhead[k] : dtok[k]) * 16;
      }
      dunit = y;
    }
  };
  // wave 0 copies the staged k1_t / v1_t rows of step st into ring slot t % ring
  const int rmask = geo.ring - 1;
  auto to_ring = [&](int st, Unit u) {
    if (wid != 0 || st >= nsteps) return;
#pragma unroll
    for (int s = 0; s < PK; ++s, u = advance(u)) {
      char* const dst = ring + (min(u.t, tlast) & rmask) * RKV;
      const char* const src = stage + ((st & 1) * PK + s) * SS + RKV;
#pragma unroll
      for (int o = 0; o < RKV; o += 1024)
        if (o + 16 * lane < RKV) *(uint4*)(dst + o + 16 * lane) = *(const uint4*)(src + o + 16 * lane);
    }
  };

  Unit cur{tfirst, 0, 0}, nx1 = after(cur);
  dma_step(0);
  dma_step(1);

  // K2 / V2 rows of the wave's keys as MFMA operands (lane (n, half): d = 16 t + 8 half .. +7)
#pragma unroll
  for (int c = 0; c < SETS; ++c) {
    const int kwc = min(k0 + 128 * c + 32 * wid + n, last);
    const bf16* k2r = F32 ? p.k2s + ((int64_t)kwc * p.hk + g) * 2 * DK : (const bf16*)p.k2 + (int64_t)kwc * p.k_st + kvg_k;
    const bf16* v2r = F32 ? p.v2s + ((int64_t)kwc * p.hk + g) * 2 * DV : (const bf16*)p.v2 + (int64_t)kwc * p.v_st + kvg_v;
#pragma unroll
    for (int t = 0; t < DK / 16; ++t) {
      core.kx[c][t] = *(const bf16x8*)(k2r + 16 * t + 8 * half);
      if constexpr (F32) core.kxl[c][t] = *(const bf16x8*)(k2r + DK + 16 * t + 8 * half);
    }
#pragma unroll
    for (int t = 0; t < DV / 16; ++t) {
      core.vx[c][t] = *(const bf16x8*)(v2r + 16 * t + 8 * half);
      if constexpr (F32) core.vxl[c][t] = *(const bf16x8*)(v2r + DV + 16 * t + 8 * half);
    }
  }
  {  // the k1 / v1 rows before the first query into the ring
    const int rows = (PK == 1 ? 32 * nr : R) - 1;
    for (int idx = tid; idx < rows * (RKV / 16); idx += 64 * NW) {
      const int jj = idx / (RKV / 16), w = idx % (RKV / 16);  // w: 16-byte segment of the ring row
      const int j = tfirst - rows + jj;
      if (j >= 0) {
        const bf16* src = w < RBK / 16 ? (const bf16*)p.k1 + EW * ((int64_t)j * p.k_st + kvg_k) + 8 * w
                                       : (const bf16*)p.v1 + EW * ((int64_t)j * p.v_st + kvg_v) + 8 * (w - RBK / 16);
        *(uint4*)(ring + (j & rmask) * RKV + 16 * w) = *(const uint4*)src;
      }
    }
  }
  wait_vmcnt<0>();
  block_barrier();

  // Forming the A / B rows of a step: wave w builds rows 8 w .. 8 w + 7, all of
  // one unit, 16 source bytes of one row per lane and block.  A lane's segment
  // is the same in every block, so its q and dout values are read once.
  constexpr int SK = RBK / 16, SV = L::RBV / 16;   // 16-byte source segments per row
  constexpr int UA = 8 * SK / 64, UB = 8 * SV / 64;  // blocks of A and of B rows
  static_assert(UA >= 1 && UB >= 1 && SK <= 64 && SV <= 64, "whole lanes per formed block");
  // (lane-derived values from a fresh lane id per step: held through the loop
  // they cost the registers of the fragments)
  struct Form {
    u32x4 q, gr, src[UA + UB];
    uint32_t lane;
  } fm;
  auto form_row = [&](uint32_t block, uint32_t segs) { return 8u * (uint32_t)wid + (block * 64u + fm.lane) / segs; };
  const int fsub = PK == 1 ? 0 : 8 * wid / R;  // the unit of this wave's rows (uniform)
  // (rows before the unit's short window, which the scores mask, take its first
  // key: as finite as the window, where a row that the query does not see, of
  // another sequence too, need not be)
  int fs0[PK];  // sequence starts of the units of the step being formed
  auto form_src = [&](int st, Unit u, uint32_t row) -> const char* {
    Unit v = u;
    int s0v = fs0[0];
#pragma unroll
    for (int s = 1; s < PK; ++s) {
      const Unit y = advance(v);
      if (s <= fsub) v = y, s0v = fs0[s];
    }
    const int j = max(v.t - 32 * v.r - (R - 1) + (int)(row % R), max(s0v, v.t - p.ws + 1));
    // rows of the step's own queries are still in the stage: the unit whose
    // query is j (units ascend in (t, h))
    const int st_u = PK == 1 ? 0 : min(max((j - u.t) * G - u.h, 0), PK - 1);
    return j >= u.t ? stage + ((st & 1) * PK + st_u) * SS + RKV : ring + (j & rmask) * RKV;
  };
  auto form_read = [&](int st, Unit x) {
    const char* const sr = stage + ((st & 1) * PK + fsub) * SS;
    fm.lane = (uint32_t)fresh_lane();
    fm.q = *(const u32x4*)(sr + 16 * (fm.lane % SK));
    fm.gr = *(const u32x4*)(sr + RBK + 16 * (fm.lane % SV));
  };
  auto form_read_block = [&](auto kk, int st, Unit x) {  // source rows of formed block k
    constexpr int k = decltype(kk)::value;
    if constexpr (k < UA) fm.src[k] = *(const u32x4*)(form_src(st, x, form_row(k, SK)) + 16 * (fm.lane % SK));
    else fm.src[k] = *(const u32x4*)(form_src(st, x, form_row(k - UA, SV)) + RBK + 16 * (fm.lane % SV));
  };
  // block k of the formed rows (A blocks, then B blocks) into tile buffer buf
  auto form_block = [&](auto kk, int buf) {
    constexpr int k = decltype(kk)::value;
    constexpr bool isa = k < UA;
    constexpr int segs = isa ? SK : SV, W = isa ? C::WK : C::WV;
    char* const tile = lds + buf * TAB + (isa ? 0 : C::TK);
    const uint32_t row = form_row(isa ? k : k - UA, segs), sg = fm.lane % segs;
    const u32x4 x = isa ? fm.q : fm.gr;
    const u32x4 y = fm.src[k];
    if constexpr (F32) {
      bf16x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bf16 h_, l_;
        split_bf16(__uint_as_float(x[e]) * __uint_as_float(y[e]), h_, l_);
        hi[e] = h_;
        lo[e] = l_;
      }
      char* const dst = tile + row * W + ((8 * sg) ^ swz<W>(row));
      *(bf16x4*)dst = hi;
      *(bf16x4*)(dst + (isa ? C::LOK : C::LOV)) = lo;
    } else {
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = mul_bf16_pair(x[e], y[e]);
      *(u32x4*)(tile + row * W + ((16 * sg) ^ swz<W>(row))) = o;
    }
  };

  // Sequence of t: its start s0 and the first token past it (dense: a boundary
  // every seqlen; packed: the cu walk, one load per boundary crossed).
  int seq = 0, s0 = 0, snext = 0;
  if (p.cu != nullptr) {
    int lo = 0, hi = p.num_seqs - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (p.cu[mid] <= tfirst) lo = mid;
      else hi = mid - 1;
    }
    seq = lo;
    snext = tfirst;  // the first step loads the start and the next boundary
  } else {
    s0 = (tfirst / p.seqlen) * p.seqlen;
    snext = s0 + p.seqlen;
  }
  // Per-unit scalars (lse, dl, delta): one lane per unit, 64 units at a time
  // and one block ahead, kept in a wave-private LDS table.
  floatx4 nx{};
  auto load_block = [&](int blk) {
    const int u = min(64 * blk + lane, nunits - 1);
    const int th = u / nr, tq = tfirst + th / G, hq = g * G + th % G;
    const int64_t thq = (int64_t)tq * p.hq + hq;
    nx[0] = p.lse[(int64_t)tq * p.lse_st + hq];
    nx[1] = p.dl[thq];
    nx[2] = p.delta[thq];
  };
  auto store_block = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(nx));
    scal[lane] = nx;
  };
  auto form_starts = [&](Unit u) {  // of the units of the step from u on (ascending calls)
#pragma unroll
    for (int s = 0; s < PK; ++s, u = advance(u)) {
      const int t = min(u.t, tlast);
      if (t >= snext) {  // crossed into another sequence (uniform, rare)
        if (p.cu == nullptr) {
          s0 = (t / p.seqlen) * p.seqlen;
          snext = s0 + p.seqlen;
        } else {
          while (seq + 1 < p.num_seqs && p.cu[seq + 1] <= t) ++seq;
          const int c = p.cu[seq];
          s0 = min(max(c, 0), t);
          // well formed (cu[seq] <= t): the start holds up to the next boundary
          snext = c > t ? t + 1 : (seq + 1 < p.num_seqs ? p.cu[seq + 1] : 0x7fffffff);
        }
        s0 = __builtin_amdgcn_readfirstlane(s0);
        snext = __builtin_amdgcn_readfirstlane(snext);
      }
      fs0[s] = s0;
    }
  };
  load_block(0);
  store_block();
  if (nunits > 64) load_block(1);
  form_starts(cur);
  to_ring(0, cur);
  form_read(0, cur);
  static_for<0, UA + UB>([&](auto k) {
    form_read_block(k, 0, cur);
    form_block(k, 0);
  });

  // masked rows start their scores at -inf (p = 0); a scale of 0 gets a tiny
  // factor instead, so that -inf times it stays -inf (dS carries the scale)
  const float sl2s = p.scale == 0.f ? 1e-30f : p.scale * kLog2e;
  const float smask = p.scale < 0.f ? INFINITY : -INFINITY;
  typename C::Addr ad = C::addresses(lds, lds + C::TK, 0, lane);

  int st = 0;
  auto step = [&](auto actc) {
    const int sl = (st * PK) & 63;
    if (sl == 0 && st > 0) {  // next block of scalars into the table, load the one after
      store_block();
      if (st * PK + 64 < nunits) load_block(st * PK / 64 + 1);
    }
    if (wid == kDmaWave) wait_vmcnt<0>();  // the rows of step st+1 have landed
    block_barrier();  // tiles of st formed, ring rows up to its queries copied, rows of st+1 staged, the other buffer free
    const Unit nx2 = after(nx1);
    dma_step(st + 2);
    int cs0[PK];
#pragma unroll
    for (int s = 0; s < PK; ++s) cs0[s] = fs0[s];
    form_starts(nx1);

    float lse2[PK], dpm[PK], dsm[PK];
    int ut[PK], lo2[PK], ilo[PK];
    bool masked = false;
    Unit u = cur;
#pragma unroll
    for (int s = 0; s < PK; ++s, u = advance(u)) {
      ut[s] = u.t;
      const int t = min(u.t, tlast), s0 = cs0[s];
      const floatx4 sv4 = lds_read_now(scal + sl + s);
      const bool single = t == s0 || (p.ws == 1 && p.wl == 1);
      lse2[s] = uniform_f(sv4[0] * kLog2e);
      dpm[s] = single ? 0.f : p.scale;
      dsm[s] = uniform_f(single ? sv4[1] * p.scale : -sv4[2] * p.scale);
      // keys [lo2, t] are valid (none for a unit past the walk); rows from ilo on
      lo2[s] = PK > 1 && st * PK + s >= nunits ? 0x7fffffff : max(s0, t - p.wl + 1);
      ilo[s] = max(s0, t - p.ws + 1) - (t - 32 * u.r - (R - 1));
      masked = masked || ilo[s] > 0;
    }
    float bias[SETS][PK];  // infinite (p = 0) for keys outside the unit's long window
#pragma unroll
    for (int c = 0; c < SETS; ++c) {
      const int kw = k0 + 128 * c + 32 * wid + n;
#pragma unroll
      for (int s = 0; s < PK; ++s) bias[c][s] = kw <= ut[s] && kw >= lo2[s] ? lse2[s] : INFINITY;
    }
    const int nbuf = (st + 1) & 1;
    auto sinit = [&](int, int e) {
      constexpr int kSub = 16 / PK;  // registers per unit
      const int row = (8 * (e >> 2) + (e & 3)) % R + 4 * half;
      return row < ilo[e / kSub] ? smask : 0.f;
    };
    auto prob = [&](int c, int e, float s) { return fast_exp2(fmaf(s, sl2s, -bias[c][e / (16 / PK)])); };
    auto grad = [&](int, int e, float pr, float dp) { return pr * fmaf(dp, dpm[e / (16 / PK)], dsm[e / (16 / PK)]); };
    // forming the next step's rows beside phase 4: the reads at its first
    // item, the blocks spread over the later ones (after the last step: stale
    // rows into a tile that nothing reads; a branch here would cut the step
    // into blocks and copy accumulators between them)
    auto fill = [&](auto ii) {
      constexpr int i = decltype(ii)::value, NB = UA + UB, T4 = C::T4;
      constexpr int first = T4 / 4;
      if constexpr (i == 0) form_read(st + 1, nx1);
      static_for<0, NB>([&](auto kk) {
        constexpr int k = decltype(kk)::value;
        constexpr int at = first + k * (T4 - first) / NB;  // item that forms block k
        // wide rows: two items earlier its source is read (all at once they
        // take the registers that the fragments leave)
        if constexpr ((DK > 256 ? (at > 2 ? at - 2 : 0) : 0) == i) form_read_block(kk, st + 1, nx1);
      });
      static_for<0, NB>([&](auto kk) {
        constexpr int k = decltype(kk)::value;
        if constexpr (first + k * (T4 - first) / NB == i) form_block(kk, nbuf);
      });
    };
    core.template step<decltype(actc)::value>(ad, masked, sinit, prob, grad, fill);
    to_ring(st + 1, nx1);  // (its slots are read from the next step's formation on)
    cur = nx1;
    nx1 = nx2;
    ad.advance((st & 1) ? -TAB : TAB);  // the other buffer
    ++st;
  };
  // Set c of a wave is reached by the steps of one range [a_c, e_c): from the
  // query kc that is its first key to the last whose long window, cut at its
  // sequence start, holds its last.  The steps outside a set's range leave its
  // products out -- they would come out as zero, or NaN for values that its keys do
  // not depend on --, one loop per choice of sets: a choice per step would copy
  // accumulators or branch at every product.  Every wave takes nsteps steps
  // (barriers).
  const int64_t upt = (int64_t)G * nr;
  auto range = [&](int c, int& a, int& e) {
    const int kc = k0 + 128 * c + 32 * wid, kl = min(kc + 31, last);
    if (kc > last) {  // no key: never reached
      a = e = nsteps;
      return;
    }
    const int tend = min(seq_end(kl) - 1, kl + p.wl - 1);
    a = __builtin_amdgcn_readfirstlane((int)max((int64_t)0, min((int64_t)nsteps, (kc - tfirst) * upt / PK)));
    e = __builtin_amdgcn_readfirstlane(
        (int)max((int64_t)0, min((int64_t)nsteps, ((tend + 1 - tfirst) * upt + PK - 1) / PK)));
  };
  int a0, e0;
  range(0, a0, e0);
  while (st < a0) step(std::integral_constant<int, 0>{});
  if constexpr (SETS == 2) {
    int a1, e1;
    range(1, a1, e1);
    while (st < min(a1, e0)) step(std::integral_constant<int, 1>{});
    while (st < e0) step(std::integral_constant<int, 3>{});
    while (st < a1) step(std::integral_constant<int, 0>{});
    while (st < e1) step(std::integral_constant<int, 2>{});
  } else {
    while (st < e0) step(std::integral_constant<int, 1>{});
  }
  while (st < nsteps) step(std::integral_constant<int, 0>{});
  write_out();
}

// dk2 and dv2 = the sum of the pieces' fp32 sums in piece order; 4 values per thread
__global__ __launch_bounds__(256) void bwd_dkv2_sum_kernel(BwdParams p, int splits) {
  const int64_t i = (int64_t)bid_x() * 256 + tid_x();
  const int64_t rows = (int64_t)p.tokens * p.hk;
  const int w = p.d + p.dv;
  const int64_t row = i / (w / 4);
  if (row >= rows) return;
  const int c = (int)(i % (w / 4)) * 4;
  const float* src = p.dkv2s + row * w + c;
  floatx4 acc = *(const floatx4*)src;
  for (int k = 1; k < splits; ++k) acc += *(const floatx4*)(src + (int64_t)k * rows * w);
  const int64_t t = row / p.hk, g = row % p.hk;
  const bool isk = c < p.d;
  void* base = isk ? p.dk2 : p.dv2;
  const int64_t off = isk ? t * p.dk_st + g * p.dk_sh + c : t * p.dv_st + g * p.dv_sh + c - p.d;
  if (p.f32) {
    *(floatx4*)((float*)base + off) = acc;
  } else {
    bf16x4 b;
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = (bf16)acc[e];
    *(bf16x4*)((bf16*)base + off) = b;
  }
}

// Pieces per walk.  One workgroup runs per CU, so the pass takes ceil(blocks *
// s / cus) rounds of walk / s steps, each piece paying about kPieceSteps steps
// of start-up (ring, fragments, first tiles, sums): the s with the least time,
// at least kMinSteps steps a piece and no more pieces than the scratch holds.
struct Dkv2Plan {
  int pieces;
  double time;  // in steps
};
Dkv2Plan dkv2_pieces(int64_t blocks, int64_t steps, int64_t cus, int64_t room) {
  constexpr int kMaxPieces = 16, kPieceSteps = 24, kMinSteps = 32;
  Dkv2Plan best{1, 0};
  for (int s = 1; s <= kMaxPieces; ++s) {
    if (s > 1 && (s > room || steps / s < kMinSteps)) break;
    const double rounds = (double)((blocks * s + cus - 1) / cus);
    const double t = rounds * ((double)steps / s + kPieceSteps);
    if (s == 1 || t < 0.98 * best.time) best = {s, t};
  }
  return best;
}
// ... of workgroups of KB keys, steps of PK units
Dkv2Plan dkv2_plan(const BwdParams& p, size_t scratch_bytes, int KB, int PK) {
  const int64_t blocks = ((int64_t)p.tokens + KB - 1) / KB * p.hk;
  const int64_t queries = std::min<int64_t>((int64_t)KB + p.wl - 1, p.cu ? p.tokens : std::max(p.seqlen, KB));
  const int nr = PK > 1 ? 1 : (p.ws + 31) / 32;
  const int64_t room = p.dkv2s ? (int64_t)scratch_bytes / dkv2_piece_bytes(p.tokens, p.hk, p.d, p.dv) : 1;
  return dkv2_pieces(blocks, queries * p.group * nr / PK, device_cu_count(), room);
}

template <int DK, int DV, int SETS, int PK, bool F32, int KB0, int KBN, int VBN>
hipError_t launch_dkv2_slice(const BwdParams& p, const Dkv2Geo& geo, hipStream_t stream) {
  const size_t lds = Dkv2Lds<DK, DV, PK, F32>::bytes(geo.ring);
  auto kern = bwd_dkv2_kernel<DK, DV, SETS, PK, F32, KB0, KBN, VBN>;
  hipError_t e = set_lds_limit((const void*)kern, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(geo.nblocks), dim3(256), lds, stream, p, geo);
  return hipGetLastError();
}

template <int DK, int DV, int SETS, int PK, bool F32>
hipError_t launch_dkv2_t(const BwdParams& p, size_t scratch_bytes, hipStream_t stream) {
  constexpr int KB = 128 * SETS;
  Dkv2Geo geo{};
  geo.nr = PK > 1 ? 1 : (p.ws + 31) / 32;
  geo.ring = DK > 256 ? 32 : geo.nr <= 2 ? 64 : 128;
  geo.kblocks = (p.tokens + KB - 1) / KB;
  const int64_t blocks = (int64_t)geo.kblocks * p.hk;
  // fp32 walks stay whole: their sums then depend on a key's own sequence only
  // (a packed batch equals its sequences one by one, bit for bit)
  geo.splits = F32 ? 1 : dkv2_plan(p, scratch_bytes, KB, PK).pieces;
  geo.nblocks = (int)(blocks * geo.splits);
  hipError_t e;
  if constexpr (DK > 256) {
    // accumulators of 512 + 256 columns take 384 registers: two launches
    constexpr int kFirst = 4;
    e = launch_dkv2_slice<DK, DV, SETS, PK, F32, 0, kFirst, DV / 32>(p, geo, stream);
    if (e == hipSuccess) e = launch_dkv2_slice<DK, DV, SETS, PK, F32, kFirst, DK / 32 - kFirst, 0>(p, geo, stream);
  } else {
    e = launch_dkv2_slice<DK, DV, SETS, PK, F32, 0, DK / 32, DV / 32>(p, geo, stream);
  }
  if (e != hipSuccess || geo.splits == 1) return e;
  const int64_t threads = (int64_t)p.tokens * p.hk * ((DK + DV) / 4);
  hipLaunchKernelGGL(bwd_dkv2_sum_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, p, geo.splits);
  return hipGetLastError();
}

// Short windows of at most 16 (8) keys: two (four) units per 32-row step.  A
// 16-row MFMA then holds one unit or, with four, a pair of heads of one query
// (even groups only): the sums of a key do not depend on where its sequence
// starts in the batch.
inline int dkv2_units(const BwdParams& p) { return p.ws <= 8 && p.group % 2 == 0 ? 4 : p.ws <= 16 ? 2 : 1; }

template <int DK, int DV, int SETS, bool F32 = false>
hipError_t launch_dkv2_pk(const BwdParams& p, size_t scratch_bytes, hipStream_t stream) {
  switch (dkv2_units(p)) {
    case 4: return launch_dkv2_t<DK, DV, SETS, 4, F32>(p, scratch_bytes, stream);
    case 2: return launch_dkv2_t<DK, DV, SETS, 2, F32>(p, scratch_bytes, stream);
    default: return launch_dkv2_t<DK, DV, SETS, 1, F32>(p, scratch_bytes, stream);
  }
}

}  // namespace

}  // namespace sa
