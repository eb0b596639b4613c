// dq / dk1 / dv1 pass of the matrix-core backward: the gradients that sum over
// long keys, from one score tile (archlab/architectures/simplicial_kernels.py:75-101).
//
// A workgroup of 4 waves owns U consecutive units (query t, head h of one KV
// group); a wave holds SETS x 32 of their rows j as MFMA fragments, A rows
// bf16(q_th ⊙ k1_j) and B rows bf16(dout_th ⊙ v1_j): one unit's 32 short keys
// per set or, with short windows of at most 16, PK = 2 units of 16 rows.  The
// waves walk the chunks of 32 long keys that the units reach, whose K2 / V2 rows
// stream into LDS (double-buffered DMAs, one barrier per chunk).  Per set
// (BwdCore, keys x rows j):
//     S = K2 · A^T,  dP = V2 · B^T,  O''^T += V2^T · P,  dA^T += K2^T · dS
// After the walk dA and O'' go through LDS, where
//     dq_th = Σ_j dA_j ⊙ k1_j     dk1_j += Σ_th dA_j ⊙ q_th     dv1_j += Σ_th O''_j ⊙ dout_th
// are formed for the whole workgroup: dq is final, the dk1 / dv1 rows of a
// workgroup are fp32 partials that bwd_dk1_dv1_sum_kernel adds in block order
// (no atomics).
//
// Measured, forward + backward of the determinant form of 256-wide heads (score
// width 512, values 256; 1024 tokens, 8 / 2 heads, windows 32 x 256): 271 ms on
// the portable kernels, 1.70 ms with this pass (0.65 ms in its two column
// slices) and the dk2 / dv2 pass (0.71 ms).  What bounds it there (counters): the
// single wave per SIMD waits in 49 % of its cycles, at the start for one load after
// another of its A and B rows, at the end for one LDS read after another of the
// sums, and nothing runs beside them; matrix cores busy in 19-20 %.
// At widths of 64 and 128 with at most 16 short keys it takes the place of the
// dq pass with dk1 partials and the dv1 pass, whose 32-row tiles such windows
// half fill: 2 x 4099 tokens, 16 / 4 heads, width 128, 16 x 512 keys 7.06 ->
// 5.08 ms forward + backward, error against 64 bits 0.0044 before and after
// (waits 37 %, matrix cores 30 %).  Its partials take less than the scratch that
// the dk1 partials had.
//
// Partials past the workspace: the blocks run in phases (dq_phase), each
// followed by the sum of the keys it completes; a phase starts with the blocks of
// the last unfinished keys again.  At widths of 64 and 128, where passes without
// partials stand beside this one, only where a phase takes more than half of the
// CUs.  Against those passes, backward with 16 short keys, width 128: phases of 512
// workgroups (2048 tokens, 32 / 1 heads, 9 phases) 19.1 -> 14.9 ms, of 256 (4096,
// 16 / 1, 18 phases) 11.0 -> 10.2; of 128 (2048, 16 / 1) 8.9 -> 9.0, of 88 (1500, 8
// / 1) 5.0 -> 5.2.
#include "sa_bwd_core.h"
#include "sa_bwd_walk.h"
#include "sa_launch.h"
#include "sa_backward.h"

#include <algorithm>

namespace sa {

namespace {

struct DqGeo {
  int nblocks;  // workgroups of the launch
  int b0, nb;   // blocks [b0, b0 + nb) of every KV head
  int nrows;    // short-key rows of a block's partial
  float* part;  // [hk][nb][nrows][DK + DV]
};

template <int DK, int DV, int SETS, int PK, int KBN>
struct DqLds {
  static constexpr int S = 4 * SETS, U = S * PK, R = 32 / PK;
  static constexpr int TAB = 32 * 2 * (DK + DV);                // one K2 + V2 tile pair
  static constexpr int CS = 32 * KBN < 128 || DV < 128 ? 64 : 128;  // columns per epilogue slab
  static constexpr int MAIN = 2 * TAB > S * 32 * CS * 4 ? 2 * TAB : S * 32 * CS * 4;
  static constexpr int ROWS = U * 2 * (DK + DV);                // q and dout rows of the units
  static constexpr int LO1 = U * 4;                             // first short key of the units
  static constexpr size_t BYTES = MAIN + ROWS + LO1;
};

// First token of token t's sequence (clamped like the forward's).
__device__ __forceinline__ int seq_start_of(const BwdParams& p, int t) {
  if (p.cu == nullptr) return (t / p.seqlen) * p.seqlen;
  int lo = 0, hi = p.num_seqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (p.cu[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  return min(max(p.cu[lo], 0), t);
}

template <int DK, int DV, int SETS, int PK, int KB0, int KBN, int VBN>
__global__ __launch_bounds__(256, 1) void bwd_dq_core_kernel(BwdParams p, DqGeo geo) {
  using C = BwdCore<DK, DV, SETS, false, KB0, KBN, VBN>;
  using L = DqLds<DK, DV, SETS, PK, KBN>;
  constexpr int U = L::U, R = L::R, CS = L::CS, TAB = L::TAB;
  extern __shared__ __attribute__((aligned(256))) char lds[];
  bf16* const qs = (bf16*)(lds + L::MAIN);                 // [U][DK]
  bf16* const gs = qs + U * DK;                            // [U][DV]
  int* const lo1s = (int*)(lds + L::MAIN + L::ROWS);       // [U]

  const int tid = tid_x(), lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, n = lane & 31;
  const int lb = xcd_remap(bid_x(), geo.nblocks);
  const int b = geo.b0 + lb % geo.nb, g = lb / geo.nb;
  const int last = p.tokens - 1, G = p.group;
  const int u0 = b * U;  // first unit (the host bounds tokens * group)
  const int tq0 = u0 / G, h0 = u0 % G;
  const int tq1 = min(last, (u0 + U - 1) / G);
  const int64_t kvg_k = (int64_t)g * p.k_sh, kvg_v = (int64_t)g * p.v_sh;

  // the units' q and dout rows, for the partial sums, and their first short keys
  if (tid < U) {
    const int t = min((u0 + tid) / G, last);
    lo1s[tid] = max(seq_start_of(p, t), t - p.ws + 1);
  }
  for (int i = tid; i < U * (DK + DV) / 8; i += 256) {
    const int u = i / ((DK + DV) / 8), s = i % ((DK + DV) / 8);
    const int t = min((u0 + u) / G, last), h = g * G + (u0 + u) % G;
    const bool isq = s < DK / 8;
    const bf16* src = isq ? (const bf16*)p.q + (int64_t)t * p.q_st + (int64_t)h * p.q_sh + 8 * s
                          : (const bf16*)p.dout + (int64_t)t * p.do_st + (int64_t)h * p.do_sh + 8 * (s - DK / 8);
    bf16* dst = isq ? qs + u * DK + 8 * s : gs + u * DV + 8 * (s - DK / 8);
    *(u32x4*)dst = *(const u32x4*)src;
  }

  // Walk: the keys that any of the units reaches
  const int lo = __builtin_amdgcn_readfirstlane(max(seq_start_of(p, tq0), tq0 - p.wl + 1));
  const int lo_last = __builtin_amdgcn_readfirstlane(max(seq_start_of(p, tq1), tq1 - p.wl + 1));
  const int nch = (tq1 - lo) / 32 + 1;

  // this lane's unit per set
  int ut[SETS], ulo[SETS], us0[SETS];
  int64_t uth[SETS];
  bool uok[SETS];
#pragma unroll
  for (int c = 0; c < SETS; ++c) {
    const int u = u0 + (wid * SETS + c) * PK + n / R;
    uok[c] = u / G <= last;
    ut[c] = min(u / G, last);
    us0[c] = seq_start_of(p, ut[c]);
    ulo[c] = max(us0[c], ut[c] - p.wl + 1);
    uth[c] = g * G + u % G;
  }

  // K2 / V2 rows of a chunk by DMA: wave w fetches every fourth 1 KB of the
  // tiles; a lane's 16 bytes are the swizzled segment of its row
  constexpr int NIK = C::TK / 4096, NIV = C::TV / 4096;
  static_assert(NIK >= 1 && NIV >= 1, "whole DMAs per wave");
  auto seg_of = [&](int k, int W, int& row) {  // source byte of the lane within its row
    const int pos = 1024 * (4 * k + wid) + 16 * lane;
    row = pos / W;
    return pos % W;
  };
  uint32_t koff[NIK], voff[NIV];
  auto offsets = [&](int rmax) {
#pragma unroll
    for (int k = 0; k < NIK; ++k) {
      int row;
      const int s = seg_of(k, C::WK, row);
      koff[k] = (uint32_t)min(row, rmax) * (uint32_t)(2 * p.k_st) + (uint32_t)(s ^ swz<C::WK>(row));
    }
#pragma unroll
    for (int k = 0; k < NIV; ++k) {
      int row;
      const int s = seg_of(k, C::WV, row);
      voff[k] = (uint32_t)min(row, rmax) * (uint32_t)(2 * p.v_st) + (uint32_t)(s ^ swz<C::WV>(row));
    }
  };
  auto dma_chunk = [&](int ch) {
    const int k0 = lo + 32 * ch;
    // (the walk's last chunk: rows past its last query repeat that query's key,
    // so that masked keys bring in no value that no unit sees)
    if (k0 + 31 > tq1) offsets(tq1 - k0);
    char* const buf = lds + (ch & 1) * TAB;
    const char* kp = (const char*)uniform_ptr((const bf16*)p.k2 + (int64_t)k0 * p.k_st + kvg_k);
    const char* vp = (const char*)uniform_ptr((const bf16*)p.v2 + (int64_t)k0 * p.v_st + kvg_v);
#pragma unroll
    for (int k = 0; k < NIK; ++k) dma16(kp + koff[k], buf + 1024 * (4 * k + wid));
#pragma unroll
    for (int k = 0; k < NIV; ++k) dma16(vp + voff[k], buf + C::TK + 1024 * (4 * k + wid));
  };

  const float sl2s = p.scale == 0.f ? 1e-30f : p.scale * kLog2e;
  const float smask = p.scale < 0.f ? INFINITY : -INFINITY;
  C core;

  offsets(31);
  dma_chunk(0);
  float bias[SETS], dpm[SETS], dsm[SETS];
#pragma unroll
  for (int c = 0; c < SETS; ++c) {
    const int j = ut[c] - (R - 1) + n % R;
    const bool ok = uok[c] && j >= max(us0[c], ut[c] - p.ws + 1);
    const int jc = max(j, 0);
    const bf16* qr = (const bf16*)p.q + (int64_t)ut[c] * p.q_st + uth[c] * p.q_sh + 8 * half;
    const bf16* gr = (const bf16*)p.dout + (int64_t)ut[c] * p.do_st + uth[c] * p.do_sh + 8 * half;
    const bf16* k1r = (const bf16*)p.k1 + (int64_t)jc * p.k_st + kvg_k + 8 * half;
    const bf16* v1r = (const bf16*)p.v1 + (int64_t)jc * p.v_st + kvg_v + 8 * half;
    auto form = [&](const bf16* a, const bf16* bb) {
      const u32x4 x = *(const u32x4*)a, y = *(const u32x4*)bb;
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = ok ? mul_bf16_pair(x[e], y[e]) : 0u;
      return __builtin_bit_cast(bf16x8, o);
    };
#pragma unroll
    for (int t = 0; t < DK / 16; ++t) core.kx[c][t] = form(qr + 16 * t, k1r + 16 * t);
#pragma unroll
    for (int t = 0; t < DV / 16; ++t) core.vx[c][t] = form(gr + 16 * t, v1r + 16 * t);
    const int64_t thq = (int64_t)ut[c] * p.hq + uth[c];
    const float lse = p.lse[(int64_t)ut[c] * p.lse_st + uth[c]];
    const bool single = ut[c] == us0[c] || (p.ws == 1 && p.wl == 1);
    bias[c] = ok ? lse * kLog2e : INFINITY;  // (p = 0 in rows outside the short window)
    dpm[c] = single ? 0.f : p.scale;
    dsm[c] = single ? p.dl[thq] * p.scale : -p.delta[thq] * p.scale;
  }
  core.clear();
  typename C::Addr ad = C::addresses(lds, lds + C::TK, 0, lane);
  for (int ch = 0; ch < nch; ++ch) {
    wait_vmcnt<0>();
    block_barrier();  // chunk ch has landed, the other buffer is free
    if (ch + 1 < nch) dma_chunk(ch + 1);
    const int k0 = lo + 32 * ch;
    const bool masked = k0 < lo_last || k0 + 31 > tq0;
    auto sinit = [&](int c, int e) {
      const int kr = k0 + 8 * (e >> 2) + (e & 3) + 4 * half;
      return kr < ulo[c] || kr > ut[c] ? smask : 0.f;
    };
    auto prob = [&](int c, int, float s) { return fast_exp2(fmaf(s, sl2s, -bias[c])); };
    auto grad = [&](int c, int, float pr, float dp) { return pr * fmaf(dp, dpm[c], dsm[c]); };
    core.template step<(1 << SETS) - 1>(ad, masked, sinit, prob, grad, [](auto) {});
    ad.advance((ch & 1) ? -TAB : TAB);
  }
  acc_settle();
  __syncthreads();  // every wave is done with the tiles: slabs take their place

  const int lf = fresh_lane(), tf = 64 * wid + lf;
  float* const slab = (float*)lds;  // [S][32][CS], 16-byte segment s of row n at s ^ (n % 16)
  constexpr int C4 = CS / 4, TRG = 256 / C4, NRT = (R - 1 + U + TRG - 1) / TRG;
  const int d4 = tf % C4, rg = tf / C4;
  // the block's partial rows of 32 x nblk columns from d0 (K: dA with q; V: O'' with dout)
  auto partial = [&](const bf16* xs, int width, int col, int pcol) {
    floatx4 acc[NRT];
#pragma unroll
    for (int i = 0; i < NRT; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    int t = tq0, h = h0;
    for (int u = 0; u < U && t <= last; ++u) {
      const bf16x4 x4 = *(const bf16x4*)(xs + u * width + col);
      const floatx4 x = {(float)x4[0], (float)x4[1], (float)x4[2], (float)x4[3]};
#pragma unroll
      for (int i = 0; i < NRT; ++i) {
        const int nn = rg + TRG * i - (t - tq0);
        if (nn < 0 || nn >= R) continue;
        const int row = u % PK * R + nn;
        acc[i] += *(const floatx4*)(slab + (u / PK * 32 + row) * CS + 4 * (d4 ^ (row & 15))) * x;
      }
      if (++h == G) h = 0, ++t;
    }
    float* const dst = geo.part + ((int64_t)g * geo.nb + (b - geo.b0)) * geo.nrows * (DK + DV) + pcol;
#pragma unroll
    for (int i = 0; i < NRT; ++i)
      if (rg + TRG * i < geo.nrows) *(floatx4*)(dst + (int64_t)(rg + TRG * i) * (DK + DV)) = acc[i];
  };
  auto put = [&](const floatx16& a, int c, int db) {  // one 32-column block of a set into the slab
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      floatx4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = acc_get(a, 4 * q4 + e);
      const int row = lf & 31;
      *(floatx4*)(slab + ((wid * SETS + c) * 32 + row) * CS + 4 * ((8 * db + 2 * q4 + (lf >> 5)) ^ (row & 15))) = x;
    }
  };
  static_for<0, 32 * KBN / CS>([&](auto ss) {
    constexpr int s = decltype(ss)::value;
    if (s > 0) __syncthreads();
#pragma unroll
    for (int c = 0; c < SETS; ++c) {
#pragma unroll
      for (int i = 0; i < CS / 32; ++i) put(core.ak[c][s * (CS / 32) + i], c, i);
    }
    __syncthreads();
    const int col = 32 * KB0 + CS * s + 4 * d4;
    partial(qs, DK, col, col);
    for (int u = rg; u < U; u += TRG) {  // dq of one unit: its rows times k1
      const int t = (u0 + u) / G, h = g * G + (u0 + u) % G;
      if (t > last) continue;
      floatx4 acc = {0.f, 0.f, 0.f, 0.f};
      // (dA is 0 in rows before the window: they take its first key, which is
      // as finite as the window, not one the query does not see)
      const int j0 = t - (R - 1), lo1 = lo1s[u];
#pragma unroll 8
      for (int i = 0; i < R; ++i) {
        const bf16x4 y = *(const bf16x4*)((const bf16*)p.k1 + (int64_t)max(j0 + i, lo1) * p.k_st + kvg_k + col);
        const int row = u % PK * R + i;
        const floatx4 x = *(const floatx4*)(slab + (u / PK * 32 + row) * CS + 4 * (d4 ^ (row & 15)));
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(x[e], (float)y[e], acc[e]);
      }
      bf16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (bf16)acc[e];
      *(bf16x4*)((bf16*)p.dq + (int64_t)t * p.dq_st + (int64_t)h * p.dq_sh + col) = o;
    }
  });
  static_for<0, 32 * VBN / CS>([&](auto ss) {
    constexpr int s = decltype(ss)::value;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < SETS; ++c) {
#pragma unroll
      for (int i = 0; i < CS / 32; ++i) put(core.av[c][s * (CS / 32) + i], c, i);
    }
    __syncthreads();
    partial(gs, DV, CS * s + 4 * d4, DK + CS * s + 4 * d4);
  });
}

// dk1 and dv1 of the keys [j0, j1): their blocks' partials in block order; 4
// values per thread.
__global__ __launch_bounds__(256) void bwd_dk1_dv1_sum_kernel(BwdParams p, DqGeo geo, int U, int R, int j0, int j1) {
  const int w = p.d + p.dv;
  const int64_t i = (int64_t)bid_x() * 256 + tid_x();
  const int64_t jg = i / (w / 4);
  if (jg >= (int64_t)(j1 - j0) * p.hk) return;
  const int c = (int)(i % (w / 4)) * 4;
  const int g = (int)(jg % p.hk), j = j0 + (int)(jg / p.hk);
  const int G = p.group;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  const int thi = min(j + R - 1, p.tokens - 1);
  const int blo = (int)((int64_t)j * G / U), bhi = (int)(((int64_t)thi * G + G - 1) / U);
  for (int b = blo; b <= bhi; ++b) {
    const int row = j - (int)((int64_t)b * U / G) + R - 1;
    acc += *(const floatx4*)(geo.part + (((int64_t)g * geo.nb + (b - geo.b0)) * geo.nrows + row) * w + c);
  }
  const bool isk = c < p.d;
  bf16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (bf16)acc[e];
  bf16* const dst = isk ? (bf16*)p.dk1 + (int64_t)j * p.dk_st + (int64_t)g * p.dk_sh + c
                        : (bf16*)p.dv1 + (int64_t)j * p.dv_st + (int64_t)g * p.dv_sh + c - p.d;
  *(bf16x4*)dst = o;
}

template <int DK, int DV, int SETS, int PK, int KB0, int KBN, int VBN>
hipError_t launch_dq_slice(const BwdParams& p, const DqGeo& geo, hipStream_t stream) {
  constexpr size_t lds = DqLds<DK, DV, SETS, PK, KBN>::BYTES;
  auto kern = bwd_dq_core_kernel<DK, DV, SETS, PK, KB0, KBN, VBN>;
  hipError_t e = set_lds_limit((const void*)kern, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(geo.nblocks), dim3(256), lds, stream, p, geo);
  return hipGetLastError();
}

// Queries that a block of U units of group G may span.
inline int block_queries(int U, int G) { return U % G == 0 ? U / G : G % U == 0 ? 1 : (U + G - 2) / G + 1; }

template <int DK, int DV, int SETS, int PK>
hipError_t launch_dq_t(const BwdParams& p, size_t scratch_bytes, hipStream_t stream) {
  constexpr int U = 4 * SETS * PK, R = 32 / PK;
  if (p.ws > R) return hipErrorNotSupported;
  DqGeo geo{};
  geo.nrows = R - 1 + block_queries(U, p.group);
  geo.part = p.dkv2s;
  const int64_t bytes = (int64_t)p.hk * geo.nrows * (DK + DV) * sizeof(float);  // of a block of every KV head
  const int64_t cap = (int64_t)(scratch_bytes / bytes);
  constexpr int reach = R - 1;  // queries after its own that a key waits for
  // (score width 512: the portable kernels otherwise)
  const int64_t least = DK > 256 ? 1 : device_cu_count() / 2 / p.hk + 1;
  if (!dq_phases_pay(p.tokens, p.group, U, reach, cap, least)) return hipErrorNotSupported;
  for (int j0 = 0; j0 < p.tokens;) {
    const DqPhase ph = dq_phase(j0, p.tokens, p.group, U, reach, cap);
    geo.b0 = ph.b0;
    geo.nb = ph.nb;
    geo.nblocks = geo.nb * p.hk;
    const int j1 = ph.j1;
    hipError_t e;
    if constexpr (DK > 256) {
      // accumulators of 512 + 256 columns take 384 registers: two launches
      constexpr int kFirst = 4;
      e = launch_dq_slice<DK, DV, SETS, PK, 0, kFirst, DV / 32>(p, geo, stream);
      if (e == hipSuccess) e = launch_dq_slice<DK, DV, SETS, PK, kFirst, DK / 32 - kFirst, 0>(p, geo, stream);
    } else {
      e = launch_dq_slice<DK, DV, SETS, PK, 0, DK / 32, DV / 32>(p, geo, stream);
    }
    if (e != hipSuccess) return e;
    const int64_t threads = (int64_t)(j1 - j0) * p.hk * ((DK + DV) / 4);
    hipLaunchKernelGGL(bwd_dk1_dv1_sum_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, p, geo,
                       U, R, j0, j1);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    j0 = j1;
  }
  return hipSuccess;
}

template <int DK, int DV, int SETS>
hipError_t launch_dq_pk(const BwdParams& p, size_t scratch_bytes, hipStream_t stream) {
  if (p.ws <= 16) return launch_dq_t<DK, DV, SETS, 2>(p, scratch_bytes, stream);
  return launch_dq_t<DK, DV, SETS, 1>(p, scratch_bytes, stream);
}

}  // namespace

// Partials of a call in one phase at score width 512.
size_t dq_core_partial_bytes(int tokens, int hq, int hk, int d, int dv, int ws) {
  const int U = 4 * (ws <= 16 ? 2 : 1), R = ws <= 16 ? 16 : 32, G = hq / hk;
  const size_t blocks = ((size_t)tokens * G + U - 1) / U;
  return blocks * hk * (R - 1 + block_queries(U, G)) * (size_t)(d + dv) * sizeof(float);
}

hipError_t launch_bwd_dq_core(const BwdParams& p, size_t scratch_bytes, hipStream_t stream) {
  if (!bwd_mfma_ok(p) || p.f32 || !p.dkv2s) return hipErrorNotSupported;
  // 32-bit row offsets within a chunk, and unit numbers
  if (64 * std::max(p.k_st, p.v_st) >= (int64_t)1 << 31 || (int64_t)p.tokens * p.group >= (int64_t)1 << 30)
    return hipErrorNotSupported;
  if (std::min(p.k_st, p.v_st) < 0) return hipErrorNotSupported;
  if (p.d == 512 && p.ws <= 32) return launch_dq_pk<512, 256, 1>(p, scratch_bytes, stream);
  // At most 16 short keys: the dq and dv1 passes of their own spend half of
  // their 32-row MFMAs outside the window (times above).
  if (p.ws <= 16 && p.d == 128 && p.dv == 128) return launch_dq_t<128, 128, 2, 2>(p, scratch_bytes, stream);
  if (p.ws <= 16 && p.d == 64 && p.dv == 64) return launch_dq_t<64, 64, 2, 2>(p, scratch_bytes, stream);
  return hipErrorNotSupported;
}

}  // namespace sa
