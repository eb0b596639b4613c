// Wave-level step shared by the backward passes that accumulate two gradients
// from one score tile.
//
// A step works on one 32-row tile pair in LDS (K rows of DK, V rows of DV
// bf16) and SETS blocks of 32 "x" rows held in registers as MFMA fragments
// (kx: DK wide, vx: DV wide):
//
//   1  S[c]  = Kt · kx[c]^T                       DK/16 MFMAs per set
//   2  dP[c] = Vt · vx[c]^T     with P[c] = exp2(S[c] sl2 - bias)
//   3  av[c] += Vt^T · P[c]     with dS[c] = P (dP dpm + dsm)
//   4  ak[c] += Kt^T · dS[c]    with the caller's next-step work
//
// Why sets: every MFMA takes one 1 KB operand fragment from LDS, which at one
// fragment per MFMA asks for 128 B per cycle and CU -- all that LDS delivers --
// at the full matrix rate.  With SETS = 2 each fragment feeds two MFMAs.  (At the
// rates reached LDS is not the bound: active in 10-24 % of the cycles, matrix cores
// in 19-38 %.)  The accumulators of both gradients and both sets take the
// accumulation registers, so one wave runs per SIMD; the vector work of a
// phase is therefore placed between the MFMAs of the phase that does not need
// its result (P beside the dP products, dS beside the av products), one group
// per MFMA, and the fragments are read kAhead items ahead across phases.
//
// Tile rows are unpadded and swizzled (swz): the row reads (ds_read_b128, 16
// rows per cycle) and the transposing reads (ds_read_b64_tr_b16, 4 rows x 64
// bytes) both touch every bank once.
#pragma once

#include "sa_mfma.h"

namespace sa {

// XOR mask (bytes, on the 16-byte segment index) of LDS tile row `row` of W
// bytes.  W >= 256: 16 consecutive rows get 16 different segments, 4
// consecutive rows different 64-byte groups; W = 128 (two rows per 256 bytes
// of banks): the same over row pairs.
template <int W>
__device__ __forceinline__ int swz(int row) {
  static_assert(W >= 128 && (W & (W - 1)) == 0, "row bytes");
  if constexpr (W >= 256) return ((row & 3) << 6) | (((row >> 2) & 3) << 4);
  else return ((row & 2) << 5) | (((row >> 2) & 3) << 4);
}

// Wait until at most N of this wave's LDS operations are outstanding, tied to
// the four registers of a fragment.
template <int N>
__device__ __forceinline__ void lds_wait_frag(u32x4& f) {
  static_assert(N >= 0 && N < 16, "lgkmcnt is 4 bits");
  asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(f) : "i"(N));
}
template <int N>
__device__ __forceinline__ void lds_wait_frag2(u32x2& a, u32x2& b) {
  static_assert(N >= 0 && N < 16, "lgkmcnt is 4 bits");
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a), "+v"(b) : "i"(N));
}
// 16 bytes of LDS read and waited for in one asm block.  (For a plain LDS read
// the compiler first waits for the wave's outstanding global->LDS DMAs.)
__device__ __forceinline__ floatx4 lds_read_now(const floatx4* p) {
  floatx4 r;
  asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(r) : "v"(lds_addr(p)) : "memory");
  return r;
}
template <int OFF>
__device__ __forceinline__ u32x4 lds_read_b128(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "16-bit LDS offset");
  u32x4 r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "i"(OFF));
  return r;
}
template <int OFF>
__device__ __forceinline__ u32x2 lds_read_tr(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "16-bit LDS offset");
  u32x2 r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "i"(OFF));
  return r;
}

// MFMAs in asm: with the result in ordinary registers (mfma_v; mfma_v0 starts
// from 0) or in an accumulation register (mfma_a).  Where a kernel may use the
// accumulation registers the compiler gives them to every MFMA result: the
// scores then compete with the gradients for those 256 and are copied out for
// the vector work (85 registers spilled at widths of 128, two sets).
// The compiler knows nothing of these instructions' hazards: NOP puts the two
// wait states before them that an operand written by vector code needs, and a
// result read by vector code needs mfma_settle() first.
template <bool NOP>
__device__ __forceinline__ void mfma_v(floatx16& c, const bf16x8& a, const bf16x8& b) {
  if constexpr (NOP) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_v0(floatx16& c, const bf16x8& a, const bf16x8& b) {
  asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
}
template <bool NOP>
__device__ __forceinline__ void mfma_a(floatx16& c, const bf16x8& a, const bf16x8& b) {
  if constexpr (NOP) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
// Wait states between the last MFMA into x and its first use by vector code,
// tied to x.  An 8-pass MFMA (32x32x16) asks for 11; the callers issue at least
// one more MFMA in between, which itself waits for the 8 passes of the one
// before, and 8 states here.
__device__ __forceinline__ void mfma_settle(floatx16& x) { asm volatile("s_nop 7" : "+v"(x)); }
// Element e of an accumulator, read from its accumulation register where it is
// used (left to the compiler, all accumulators are copied to ordinary
// registers on the loop exit and the loop spills its fragments for them).
// Preceded by acc_settle() after the last MFMA.
__device__ __forceinline__ float acc_get(const floatx16& a, int e) {
  float x;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(a[e]));
  return x;
}
__device__ __forceinline__ void acc_settle() { asm volatile("s_nop 15\n\ts_nop 3" ::: "memory"); }

// F32: every operand as hi + lo bf16 terms (split_bf16), each product on three
// term pairs; the lo tile rows follow the 32 (TR) hi rows of each tile.
// KB0, KBN: the 32-column blocks of the score width whose ak is accumulated;
// VBN: the blocks of av (DV / 32, or 0: no av).  A width whose accumulators do
// not fit the registers takes one launch per slice, which forms the scores anew.
template <int DK, int DV, int SETS, bool F32, int KB0 = 0, int KBN = DK / 32, int VBN = DV / 32>
struct BwdCore {
  static constexpr int TR = 32;                            // rows of a tile
  static constexpr int WK = 2 * DK, WV = 2 * DV;           // bytes of a tile row
  static constexpr int TK = TR * WK * (F32 ? 2 : 1);       // bytes of a K tile (hi, then lo rows)
  static constexpr int TV = TR * WV * (F32 ? 2 : 1);
  static constexpr int LOK = TR * WK, LOV = TR * WV;       // offset of the lo rows
  // items read ahead (with one set an item lasts one MFMA: further ahead)
  static constexpr int kAhead = F32 ? 3 : SETS == 1 ? 5 : DK + DV >= 256 ? 3 : 4;
  static constexpr int T1 = DK / 16, T2 = DV / 16, T3 = 2 * VBN, T4 = 2 * KBN;
  static_assert(VBN == 0 || VBN == DV / 32, "all of av or none");
  static constexpr int NT = T1 + T2 + T3 + T4;
  static constexpr int NX = F32 ? 2 : 1;                   // terms per operand

  bf16x8 kx[SETS][T1], vx[SETS][T2];
  bf16x8 kxl[F32 ? SETS : 1][F32 ? T1 : 1], vxl[F32 ? SETS : 1][F32 ? T2 : 1];
  floatx16 ak[SETS][KBN], av[SETS][VBN ? VBN : 1];

  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int c = 0; c < SETS; ++c) {
#pragma unroll
      for (int i = 0; i < KBN; ++i) ak[c][i] = floatx16{};
#pragma unroll
      for (int i = 0; i < VBN; ++i) av[c][i] = floatx16{};
    }
  }

  // Lane base addresses of one tile pair: rows row0 .. row0+31 of the K tile
  // at `kt` and the V tile at `vt` (256-byte aligned).
  struct Addr {
    uint32_t kr, vr;  // row reads: row row0 + n, segment `half`
    uint32_t kc, vc;  // transposing reads: row row0 + 4 half + e, 64-byte group 0
    __device__ __forceinline__ void advance(int bytes) { kr += bytes, vr += bytes, kc += bytes, vc += bytes; }
  };
  __device__ static __forceinline__ Addr addresses(const char* kt, const char* vt, int row0, int lane) {
    const int n = lane & 31, half = lane >> 5, g16 = (lane >> 4) & 1, i16 = lane & 15;
    const int e = i16 >> 2, q = i16 & 3;
    const int rr = row0 + n, rc = row0 + 4 * half + e;
    const int cb = 32 * g16 + 16 * (q >> 1);
    Addr a;
    a.kr = lds_addr(kt) + rr * WK + ((16 * half) ^ swz<WK>(rr));
    a.vr = lds_addr(vt) + rr * WV + ((16 * half) ^ swz<WV>(rr));
    a.kc = lds_addr(kt) + rc * WK + (cb ^ swz<WK>(rc)) + 8 * (q & 1);
    a.vc = lds_addr(vt) + rc * WV + (cb ^ swz<WV>(rc)) + 8 * (q & 1);
    return a;
  }

  // LDS operations issued for item i
  static constexpr int ops(int i) { return (i < T1 + T2 ? 1 : 2) * NX; }
  static constexpr int ops_after(int i) {  // of the items in flight behind item i
    int s = 0;
    for (int k = i + 1; k <= i + kAhead && k < NT; ++k) s += ops(k);
    return s;
  }

  struct Frag {
    u32x4 r;          // row fragment
    u32x2 a, b;       // transposed fragment (two reads)
  };
  template <int I>
  __device__ static __forceinline__ void read(const Addr& ad, Frag& h, Frag& l) {
    if constexpr (I < T1 + T2) {
      constexpr bool isk = I < T1;
      constexpr int t = isk ? I : I - T1;
      constexpr int xm = (isk ? WK : WV) >= 256 ? 32 * (t & 7) : 32 * t;   // inside the swizzled bits
      constexpr int off = (isk ? WK : WV) >= 256 ? 32 * (t & ~7) : 0;
      const uint32_t a = (isk ? ad.kr : ad.vr) ^ xm;
      h.r = lds_read_b128<off>(a);
      if constexpr (F32) l.r = lds_read_b128<off + (isk ? LOK : LOV)>(a);
    } else {
      constexpr bool isk = I >= T1 + T2 + T3;
      constexpr int D = isk ? DK : DV, W = 2 * D;
      constexpr int s = isk ? I - T1 - T2 - T3 : I - T1 - T2;
      constexpr int NB = isk ? KBN : VBN ? VBN : 1;
      constexpr int t = s / NB, db = s % NB + (isk ? KB0 : 0);
      constexpr int xm = W >= 256 ? 64 * (db & 3) : 64 * db;
      constexpr int off = (W >= 256 ? 256 * (db >> 2) : 0) + 16 * t * W;
      const uint32_t a = (isk ? ad.kc : ad.vc) ^ xm, b = a ^ 32;
      h.a = lds_read_tr<off>(a);
      h.b = lds_read_tr<off + 8 * W>(b);
      if constexpr (F32) {
        l.a = lds_read_tr<off + (isk ? LOK : LOV)>(a);
        l.b = lds_read_tr<off + 8 * W + (isk ? LOK : LOV)>(b);
      }
    }
  }
  template <int I, int N>
  __device__ static __forceinline__ bf16x8 get(Frag& f) {
    if constexpr (I < T1 + T2) {
      lds_wait_frag<N>(f.r);
      return __builtin_bit_cast(bf16x8, f.r);
    } else {
      lds_wait_frag2<N>(f.a, f.b);
      return __builtin_bit_cast(bf16x8, u32x4{f.a[0], f.a[1], f.b[0], f.b[1]});
    }
  }
  // One step for the sets in ACT (a bit mask; 0: the caller's work only).  sinit(c, e): start value of score
  // register e of set c (0, or the value that masks it) when `masked`.  prob(c, e, s):
  // the probability of register e of set c; grad(c, e, p, dp): its dS.
  // fill(item): the caller's work beside item 0 .. T4-1 of phase 4.
  template <int ACT, typename SI, typename PF, typename GF, typename FF>
  __device__ __forceinline__ void step(const Addr& ad, bool masked, SI&& sinit, PF&& prob, GF&& grad, FF&& fill) {
    if constexpr (ACT == 0) {  // the caller's work only
      static_for<0, T4>([&](auto i) { fill(i); });
      return;
    }
    floatx16 s[SETS], dp[SETS];
    uint32_t pk[SETS][8], pl[F32 ? SETS : 1][8];
    Frag fh[NT], fl[F32 ? NT : 1];
    auto frl = [&](int i) -> Frag& { return fl[F32 ? i : 0]; };
    static_for<0, kAhead>([&](auto i) { read<decltype(i)::value>(ad, fh[i], frl(i)); });
    // score start values: 0, or in a masked step what masks their rows
    auto first = [&](auto cc, const bf16x8& h) {
      constexpr int c = decltype(cc)::value;
      if (masked) {
#pragma unroll
        for (int e = 0; e < 16; ++e) s[c][e] = sinit(c, e);
        mfma_v<true>(s[c], h, kx[c][0]);
      } else {
        mfma_v0(s[c], h, kx[c][0]);
      }
    };
    static_for<0, NT>([&](auto ii) {
      constexpr int I = decltype(ii)::value;
      if constexpr (I + kAhead < NT) read<I + kAhead>(ad, fh[I + kAhead], frl(I + kAhead));
      bf16x8 h, l;
      if constexpr (F32) {
        // the hi reads of an item are issued before its lo reads
        constexpr int lo = I < T1 + T2 ? 1 : 2;
        h = get<I, ops_after(I) + lo>(fh[I]);
        l = get<I, ops_after(I)>(frl(I));
      } else {
        h = get<I, ops_after(I)>(fh[I]);
        l = h;
      }
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, SETS>([&](auto cc) {
        constexpr int c = decltype(cc)::value, cl = F32 ? c : 0;
        if constexpr ((ACT >> c) & 1) {
          // first use of vector results: the start scores, the packed P and dS.
          // (fp32 and width 512: fragments are moved out of accumulation registers)
          constexpr bool nop = F32 || DK > 256 || I == 0 || I == T1 + T2 || I == T1 + T2 + T3;
          if constexpr (I < T1) {
            if constexpr (I == 0) first(cc, h);
            else mfma_v<nop>(s[c], h, kx[c][I]);
            if constexpr (F32) {
              mfma_v<nop>(s[c], h, kxl[cl][F32 ? I : 0]);
              mfma_v<nop>(s[c], l, kx[c][I]);
            }
          } else if constexpr (I < T1 + T2) {
            constexpr int t = I - T1;
            if constexpr (t == 0) mfma_v0(dp[c], h, vx[c][t]);
            else mfma_v<nop>(dp[c], h, vx[c][t]);
            if constexpr (F32) {
              mfma_v<nop>(dp[c], h, vxl[cl][F32 ? t : 0]);
              mfma_v<nop>(dp[c], l, vx[c][t]);
            }
          } else {
            constexpr bool isk = I >= T1 + T2 + T3;
            constexpr int NB = isk ? KBN : VBN ? VBN : 1;
            constexpr int q = isk ? I - T1 - T2 - T3 : I - T1 - T2;
            constexpr int t = q / NB, db = q % NB;
            if constexpr (VBN == 0 && I == T1 + T2) {  // no av phase to form dS beside
              asm volatile("s_nop 15" : "+v"(dp[c]));
#pragma unroll
              for (int e = 0; e < 16; ++e) dp[c][e] = grad(c, e, s[c][e], dp[c][e]);
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                if constexpr (F32) pack_bf16_split(dp[c][2 * i], dp[c][2 * i + 1], pk[c][i], pl[cl][i]);
                else pk[c][i] = pack_bf16(dp[c][2 * i], dp[c][2 * i + 1]);
              }
            }
            const bf16x8 b = __builtin_bit_cast(bf16x8, u32x4{pk[c][4 * t], pk[c][4 * t + 1], pk[c][4 * t + 2], pk[c][4 * t + 3]});
            const bf16x8 bl = __builtin_bit_cast(bf16x8, u32x4{pl[cl][4 * t], pl[cl][4 * t + 1], pl[cl][4 * t + 2], pl[cl][4 * t + 3]});
            floatx16& acc = isk ? ak[c][isk ? db : 0] : av[c][isk ? 0 : db];
            mfma_a<nop>(acc, h, b);
            if constexpr (F32) {
              mfma_a<nop>(acc, h, bl);
              mfma_a<nop>(acc, l, b);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
          // the set's vector work beside this MFMA (pair i of 8: registers 2i, 2i+1)
          if constexpr (I >= T1 && I < T1 + T2) {
            if constexpr (I == T1) mfma_settle(s[c]);
            // (pairs are packed one item later: the exponentials' latency)
            auto pack = [&](auto item) {
              static_for<0, 8>([&](auto ee) {
                constexpr int i = decltype(ee)::value;
                if constexpr (i * T2 / 8 == decltype(item)::value) {
                  if constexpr (F32) pack_bf16_split(s[c][2 * i], s[c][2 * i + 1], pk[c][i], pl[cl][i]);
                  else pk[c][i] = pack_bf16(s[c][2 * i], s[c][2 * i + 1]);
                }
              });
            };
            static_for<0, 8>([&](auto ee) {
              constexpr int i = decltype(ee)::value;
              if constexpr (i * T2 / 8 == I - T1) {
                s[c][2 * i] = prob(c, 2 * i, s[c][2 * i]);
                s[c][2 * i + 1] = prob(c, 2 * i + 1, s[c][2 * i + 1]);
              }
            });
            if constexpr (VBN > 0 && I > T1) pack(std::integral_constant<int, I - T1 - 1>{});
            if constexpr (VBN > 0 && I == T1 + T2 - 1) pack(std::integral_constant<int, T2 - 1>{});
            __builtin_amdgcn_sched_barrier(0);
          } else if constexpr (I >= T1 + T2 && I < T1 + T2 + T3) {
            if constexpr (I == T1 + T2) mfma_settle(dp[c]);
            // pairs 4t .. of the packed P feed this phase's MFMAs: dS stays in
            // dp until the last of them has been issued
            static_for<0, 8>([&](auto ee) {
              constexpr int i = decltype(ee)::value;
              if constexpr (i * T3 / 8 == I - T1 - T2) {
                dp[c][2 * i] = grad(c, 2 * i, s[c][2 * i], dp[c][2 * i]);
                dp[c][2 * i + 1] = grad(c, 2 * i + 1, s[c][2 * i + 1], dp[c][2 * i + 1]);
              }
            });
            if constexpr (I == T1 + T2 + T3 - 1) {
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                if constexpr (F32) pack_bf16_split(dp[c][2 * i], dp[c][2 * i + 1], pk[c][i], pl[cl][i]);
                else pk[c][i] = pack_bf16(dp[c][2 * i], dp[c][2 * i + 1]);
              }
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      });
      if constexpr (I >= T1 + T2 + T3) {
        fill(std::integral_constant<int, I - T1 - T2 - T3>{});
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  }
};

}  // namespace sa
