// Paged forward for an fp32 query over caches that are not both bf16 (fp32,
// fp16, or mixed: the reference reads any float cache, simplicial_paged.py:42-52,
// and its contiguous fp32 decodes, simplicial_decode.py, simplicial_packed.py:238-338),
// on the fp32 matrix instructions: every product and sum in fp32.
//
// A workgroup owns (token, KV group, split, task block); a task is 32 rows a_j =
// q ⊙ k1_j: one query head's 32-row group of short keys or, with at most 16
// short keys, two heads x 16.  Each wave takes one task and walks the split's
// 32-key chunks, whose K2 / V2 rows the workgroup converts to fp32 in LDS:
//     S^T = K · A^T     D/2 v_mfma_f32_32x32x2_f32 (lane: row, registers: keys)
//     O^T += V^T · P^T  16 D/32 of them; MFMA r takes key 8 (r/4) + r % 4 from
//                       lanes 0-31 and that key + 4 from lanes 32-63, which is
//                       how S^T left P in the registers
// Every row keeps its own running maximum; rows, splits and row groups merge
// by their log-sum-exp weights (paged_combine_kernel, a fixed order).
//
// What bounds it: with many tokens the fp32 matrix rate (a chunk is 128 MFMAs of
// 64 cycles at width 128, against 32 KB of rows); for a few tokens the chain of
// rows, products and merge, a tile segment after another since its loads are not
// issued ahead (the decode below: matrix cores busy in 18 % of the cycles, waves
// waiting in 48 %).  So the long axis is cut into as many splits as
// give each SIMD one to four waves.  4 rows x 8 KV heads, GQA 4, 16 x 1025 keys,
// width 128: 1630 us on the portable kernel (one workgroup per query head, scalar
// products), 46 us here, of which the merge is 4.
#include "sa_generic.h"
#include "sa_grid.h"
#include "sa_mfma.h"
#include "sa_launch.h"

#include <algorithm>
#include <type_traits>

namespace sa {

struct PagedF32Params {
  const float* q;
  int64_t q_st, q_sh;
  PagedRows rows;
  const void* tseq;
  const void* tpos;
  const int32_t* caps;
  int seq64, pos64, num_seqs;
  int tokens, hq, hk, group;
  int ws, wl, nc, nr;
  int rpu;      // rows per unit: 16 (two heads per task) or 32
  int tasks;    // tasks per (token, KV group)
  int tblocks;  // task blocks
  int splits;
  float sl2;    // scale * log2(e)
  int direct;   // splits * nr == 1: write out / lse
  float* part_o;
  float* part_m;
  float* part_z;
  float* out;
  int64_t o_st, o_sh;
  float* lse;
};

template <typename T>
__device__ __forceinline__ floatx4 load4(const T* p) {
  if constexpr (std::is_same_v<T, float>) {
    return *(const floatx4*)p;
  } else {
    typedef T tx4 __attribute__((ext_vector_type(4)));
    const tx4 x = *(const tx4*)p;
    return floatx4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
  }
}

template <int D, typename SCT, typename LCT>
__global__ __launch_bounds__(256, D >= 256 ? 1 : 2) void paged_f32_kernel(PagedF32Params p) {
  constexpr int SEGS = D / 4;  // 16-byte segments per fp32 row
  extern __shared__ __attribute__((aligned(256))) char lds[];
  float* const kt = (float*)lds;         // [32][D], segment s of row r at s ^ (r % 16)
  float* const vt = kt + 32 * D;
  int64_t* const roff = (int64_t*)(vt + 32 * D);  // [32] row offsets of the chunk
  const int tid = tid_x(), lane = tid & 63, nthreads = (int)__builtin_amdgcn_workgroup_size_x();
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), nw = nthreads >> 6;
  const int n = lane & 31, half = lane >> 5;

  int b = bid_x();
  const int tb = b % p.tblocks;
  b /= p.tblocks;
  const int split = b % p.splits;
  b /= p.splits;
  const int g = b % p.hk, token = b / p.hk;

  const bool tables = p.rows.stable != nullptr;  // (uniform)
  PagedRowsOf<false> rows{p.rows};
  rows.seq = p.tseq ? clamp64(load_index(p.tseq, token, p.seq64), 0, p.num_seqs - 1) : token;
  const int pos = p.tpos ? (int)load_index(p.tpos, token, p.pos64) : p.wl - 1;
  int ws = p.ws, wl = p.wl;
  if (p.caps) {
    ws = max(1, min(ws, p.caps[2 * token]));
    wl = max(1, min(wl, p.caps[2 * token + 1]));
  }
  const int lo1 = max(0, pos - ws + 1), lo2 = max(0, pos - wl + 1);
  const int kstart = pos - p.wl + 1;  // chunk grid origin
  const int cfirst = (lo2 - kstart) / kChunk;
  const int per = (p.nc - cfirst + p.splits - 1) / p.splits;
  const int cbeg = cfirst + split * per, cend = pos < 0 ? cbeg : min(p.nc, cbeg + per);

  // this lane's row: head hi of the group, short key j
  const int task = tb * nw + wid;
  const int r = p.rpu == 32 ? task / p.group : 0;
  const int hi = p.rpu == 32 ? task % p.group : 2 * task + (n >> 4);
  const int j = pos - 32 * r - (p.rpu == 32 ? n : n & 15);
  const bool head_ok = task < p.tasks && hi < p.group;
  const bool row_ok = head_ok && j >= lo1 && j <= pos && cbeg < cend;
  const int h = g * p.group + (head_ok ? hi : 0);
  const SCT* const sc = (const SCT*)rows.sc;
  const LCT* const lc = (const LCT*)rows.lc;
  auto at = [&](auto off) {  // off(rows) of the caches' form
    PagedRowsOf<true> seq_rows{rows};
    return tables ? off(rows) : off(seq_rows);
  };
  const int64_t soff = at([&](const auto& x) { return x.s_off(max(j, 0), g); });

  floatx4 a[D / 8];  // A rows: d = 8 u + 4 half + e; during the last P·V the v1 rows
  floatx16 o[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) o[i] = floatx16{};
  float m = -INFINITY, z = 0.f;  // this lane's row (z: its 16 keys per chunk)

  for (int c = cbeg; c < cend; ++c) {
    const int k0 = kstart + kChunk * c;
    __syncthreads();  // the previous chunk is consumed
    if (tid < kChunk) roff[tid] = at([&](const auto& x) { return x.l_off(min(max(k0 + tid, lo2), pos), g); });
    __syncthreads();
    if (c == cbeg) {  // beside the first tile's loads
      const float* const qr = p.q + (int64_t)token * p.q_st + (int64_t)h * p.q_sh;
#pragma unroll
      for (int u = 0; u < D / 8; ++u) {
        const floatx4 x = *(const floatx4*)(qr + 8 * u + 4 * half) * load4(sc + soff + 8 * u + 4 * half);
        a[u] = row_ok ? x : floatx4{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll 8
    for (int i = tid; i < 32 * SEGS; i += nthreads) {
      const int row = i / SEGS, seg = i % SEGS;
      const LCT* const src = lc + roff[row] + 4 * seg;
      const int dst = row * D + 4 * (seg ^ (row & 15));
      // keys outside the window: zero rows (their p is 0, V may be anything)
      const bool in = k0 + row >= lo2 && k0 + row <= pos;
      const floatx4 kf = load4(src), vf = load4(src + rows.lc_a), zero{};
      *(floatx4*)(kt + dst) = in ? kf : zero;
      *(floatx4*)(vt + dst) = in ? vf : zero;
    }
    __syncthreads();
    floatx16 s = floatx16{};
#pragma unroll
    for (int u = 0; u < D / 8; ++u) {
      const floatx4 kf = *(const floatx4*)(kt + n * D + 4 * ((2 * u + half) ^ (n & 15)));
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], a[u][e], s, 0, 0, 0);
    }
    const int klo = lo2 - k0 - 4 * half, khi = pos - k0 - 4 * half;
    float cmax = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int kr = 8 * (e >> 2) + (e & 3);
      s[e] = kr < klo || kr > khi ? -INFINITY : s[e] * p.sl2;
      cmax = fmaxf(cmax, s[e]);
    }
    // A row whose scores so far are all -inf (they overflowed: a chunk of the walk
    // holds a valid key) keeps sums of 0: its exponents are taken against 0.
    const float mn = fmaxf(m, pair_max(cmax)), ref = mn == -INFINITY ? 0.f : mn, alpha = fast_exp2(m - ref);
    m = mn;
    float zs = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = fast_exp2(s[e] - ref);
      zs += s[e];
    }
    z = z * alpha + zs;
#pragma unroll
    for (int i = 0; i < D / 32; ++i) o[i] *= alpha;
    if (c + 1 == cend) {
#pragma unroll
      for (int u = 0; u < D / 8; ++u) a[u] = load4(sc + soff + rows.sc_a + 8 * u + 4 * half);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int key = 8 * (e >> 2) + 4 * half + (e & 3);
#pragma unroll
      for (int i = 0; i < D / 32; ++i) {
        const int d = 32 * i + n;
        const float v = vt[key * D + 4 * ((d >> 2) ^ (key & 15)) + (d & 3)];
        o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, s[e], o[i], 0, 0, 0);
      }
    }
  }
  __syncthreads();  // tile reads done: the merge scratch takes their place

  // rows of a head merged by their weights: out = sum_n w_n v1_n ⊙ O_n / sum_n w_n z_n
  const bool two = p.rpu != 32;
  auto group_max = [&](float x) {
    x = fmaxf(x, dpp_mov<kDppXor1>(x));
    x = fmaxf(x, dpp_mov<kDppXor2>(x));
    x = fmaxf(x, dpp_mov<kDppHalfMirror>(x));
    x = fmaxf(x, dpp_mov<kDppMirror>(x));
    return two ? x : row_pair_max(x);
  };
  auto group_sum = [&](float x) {
    x += dpp_mov<kDppXor1>(x);
    x += dpp_mov<kDppXor2>(x);
    x += dpp_mov<kDppHalfMirror>(x);
    x += dpp_mov<kDppMirror>(x);
    return two ? x : row_pair_sum(x);
  };
  const float M = group_max(row_ok ? m : -INFINITY);
  const float wgt = row_ok && M > -INFINITY ? fast_exp2(m - M) : 0.f;
  const float zr = pair_sum(z);
  const float Z = group_sum(row_ok ? wgt * zr : 0.f);
  float* const red = (float*)lds + wid * (64 * 36);
  const int64_t th = (int64_t)p.tokens * p.hq;
  const int64_t pbase = (int64_t)(split * p.nr + r) * th + (int64_t)token * p.hq;
  // head of half x of the wave's rows (one head when rpu == 32)
  const int h0 = g * p.group + (two ? 2 * task : hi);
  const bool ok0 = task < p.tasks, ok1 = two && 2 * task + 1 < p.group && ok0;
  const float Z0 = uniform_f(Z), Z1 = __shfl(Z, 16), M0 = uniform_f(M), M1 = __shfl(M, 16);
#pragma unroll
  for (int sl = 0; sl < D / 64; ++sl) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int dd = 32 * (i >> 2) + 8 * (i & 3) + 4 * half;
      const floatx4 v = a[8 * sl + i];
#pragma unroll
      for (int e = 0; e < 4; ++e) red[(dd + e) * 36 + n] = row_ok ? wgt * v[e] * o[2 * sl + (i >> 2)][4 * (i & 3) + e] : 0.f;
    }
    // `red` is private to the wave, whose LDS accesses execute in order
    float acc[2] = {0.f, 0.f};
    const floatx4* const row4 = (const floatx4*)(red + lane * 36);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const floatx4 x = row4[i];
      acc[i >> 2] += (x[0] + x[1]) + (x[2] + x[3]);
    }
    if (!two) acc[0] += acc[1];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (!(k ? ok1 : ok0)) continue;
      const int hh = h0 + k;
      if (p.direct) p.out[(int64_t)token * p.o_st + (int64_t)hh * p.o_sh + 64 * sl + lane] = acc[k] / (k ? Z1 : Z0);
      else p.part_o[(pbase + hh) * D + 64 * sl + lane] = acc[k];
    }
  }
  if (lane < 2 && (lane ? ok1 : ok0)) {
    const float Mk = lane ? M1 : M0, Zk = lane ? Z1 : Z0;
    if (p.direct) {
      if (p.lse) p.lse[(int64_t)token * p.hq + h0 + lane] = (Mk + __log2f(Zk)) * kLn2;
    } else {
      p.part_m[pbase + h0 + lane] = Mk;
      p.part_z[pbase + h0 + lane] = Zk;
    }
  }
}

// ---------------------------------------------------------------------------
// Host side

namespace {

// The portable kernel needs no workspace; calls whose partials would pass this
// size stay there (more than one row group) or take fewer splits.
constexpr size_t kF32PartialCap = (size_t)256 << 20;

struct F32Plan {
  int rpu, nr, tasks, nw;
};
F32Plan f32_plan(const sa_paged_args* a) {
  F32Plan f{};
  const int group = a->heads_q / a->heads_kv;
  f.rpu = a->short_window <= 16 ? 16 : 32;
  f.nr = (a->short_window + 31) / 32;
  f.tasks = f.rpu == 16 ? (group + 1) / 2 : group * f.nr;
  f.nw = f.tasks >= 4 ? 4 : f.tasks >= 2 ? 2 : 1;
  return f;
}
size_t f32_partial_bytes(const sa_paged_args* a, size_t P) {
  const size_t th = (size_t)a->tokens * a->heads_q;
  return ((P * th * a->head_dim * 4 + 255) & ~(size_t)255) + 2 * ((P * th * 4 + 255) & ~(size_t)255);
}

}  // namespace

bool paged_f32_route(const sa_paged_args* a) {
  if ((a->flags & SA_FLAG_FORCE_GENERIC) || a->q_dtype != SA_DTYPE_F32) return false;
  if (a->cache_dtype == SA_DTYPE_BF16 && a->long_cache_dtype == SA_DTYPE_BF16) return false;
  if (a->head_dim != 64 && a->head_dim != 128 && a->head_dim != 256) return false;
  // rows are read four elements at a time
  for (int i = 0; i < 4; ++i)
    if ((a->sc_stride[i] % 4) || (a->lc_stride[i] % 4)) return false;
  if ((a->q_stride_t % 4) || (a->q_stride_h % 4)) return false;
  if (((uintptr_t)a->q | (uintptr_t)a->short_cache | (uintptr_t)a->long_cache) & 15) return false;
  const F32Plan f = f32_plan(a);
  if (!grid_fits((int64_t)a->tokens * a->heads_kv * ((f.tasks + f.nw - 1) / f.nw), 64 * f.nw)) return false;
  return f.nr == 1 || f32_partial_bytes(a, f.nr) <= kF32PartialCap;
}

void paged_without_partials(sa_paged_args* a) {
  a->splits = 1;
  if (f32_plan(a).nr > 1) a->flags |= SA_FLAG_FORCE_GENERIC;
}

// Chunks per split: of the grids that fill one, two and four waves per SIMD the
// one with the least (chunks in turn on a SIMD, which shares its matrix unit)
// + 3 chunks' worth of loads, reductions and launch per round of two waves.
int paged_f32_splits(const sa_paged_args* a) {
  const F32Plan f = f32_plan(a);
  const int64_t nc = ((int64_t)a->long_window + kChunk - 1) / kChunk;
  const int64_t waves = (int64_t)a->tokens * a->heads_kv * ((f.tasks + f.nw - 1) / f.nw) * f.nw;
  int64_t s = a->splits;
  if (s <= 0) {
    const int64_t simds = 4 * (int64_t)device_cu_count();
    int64_t best = INT64_MAX;
    for (int k = 1; k <= 4; k *= 2) {
      const int64_t want = std::max<int64_t>(1, std::min(nc, k * simds / waves));
      const int64_t per = (nc + want - 1) / want, splits = (nc + per - 1) / per;  // no split stays empty
      const int64_t turns = (waves * splits + simds - 1) / simds;
      const int64_t cost = turns * per + 3 * ((turns + 1) / 2);
      if (cost < best) best = cost, s = splits;
    }
  }
  s = std::min(s, nc);
  while (s > 1 && f32_partial_bytes(a, (size_t)s * f.nr) > kF32PartialCap) s = (s + 1) / 2;
  return (int)s;
}

size_t paged_f32_workspace_bytes(const sa_paged_args* a, int splits) {
  const size_t P = (size_t)splits * f32_plan(a).nr;
  return P == 1 ? 0 : f32_partial_bytes(a, P);
}

template <int D, typename SCT, typename LCT>
static hipError_t launch_f32_t(const PagedF32Params& p, int nw, hipStream_t stream) {
  const size_t tiles = 2 * 32 * (size_t)D * 4 + 32 * 8, red = (size_t)nw * 64 * 36 * 4;
  const size_t lds = std::max(tiles, red);
  auto kern = paged_f32_kernel<D, SCT, LCT>;
  hipError_t e = set_lds_limit((const void*)kern, lds);
  if (e != hipSuccess) return e;
  const int64_t nb = (int64_t)p.tokens * p.hk * p.splits * p.tblocks;
  hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(64 * nw), lds, stream, p);
  return hipGetLastError();
}
template <int D, typename SCT>
static hipError_t launch_f32_l(const PagedF32Params& p, int lt, int nw, hipStream_t s) {
  if (lt == SA_DTYPE_F32) return launch_f32_t<D, SCT, float>(p, nw, s);
  if (lt == SA_DTYPE_F16) return launch_f32_t<D, SCT, _Float16>(p, nw, s);
  if constexpr (!std::is_same_v<SCT, bf16>) return launch_f32_t<D, SCT, bf16>(p, nw, s);
  return hipErrorInvalidValue;  // both bf16: the bf16 kernel's
}
template <int D>
static hipError_t launch_f32_d(const PagedF32Params& p, int st, int lt, int nw, hipStream_t s) {
  if (st == SA_DTYPE_F32) return launch_f32_l<D, float>(p, lt, nw, s);
  if (st == SA_DTYPE_F16) return launch_f32_l<D, _Float16>(p, lt, nw, s);
  return launch_f32_l<D, bf16>(p, lt, nw, s);
}

hipError_t launch_paged_f32(const sa_paged_args* a, int splits, void* ws, size_t ws_bytes, hipStream_t stream) {
  const F32Plan f = f32_plan(a);
  PagedF32Params p{};
  p.q = (const float*)a->q;
  p.q_st = a->q_stride_t;
  p.q_sh = a->q_stride_h;
  p.rows = paged_rows(a);
  p.tseq = a->token_seq;
  p.tpos = a->token_pos;
  p.caps = a->token_window_caps;
  p.seq64 = a->token_index_dtype == SA_INDEX_I64;
  p.pos64 = a->token_pos_index_dtype == SA_INDEX_I64;
  p.num_seqs = a->num_seqs;
  p.tokens = a->tokens;
  p.hq = a->heads_q;
  p.hk = a->heads_kv;
  p.group = a->heads_q / a->heads_kv;
  p.ws = a->short_window;
  p.wl = a->long_window;
  p.nc = (int)(((int64_t)a->long_window + kChunk - 1) / kChunk);
  p.nr = f.nr;
  p.rpu = f.rpu;
  p.tasks = f.tasks;
  p.tblocks = (f.tasks + f.nw - 1) / f.nw;
  p.splits = splits;
  p.sl2 = a->scale * kLog2e;
  p.direct = splits * f.nr == 1;
  p.out = a->out;
  p.o_st = a->o_stride_t;
  p.o_sh = a->o_stride_h;
  p.lse = a->lse;
  const size_t P = (size_t)splits * f.nr, th = (size_t)a->tokens * a->heads_q;
  if (!p.direct) {
    if (ws_bytes < f32_partial_bytes(a, P) || ((uintptr_t)ws & 255)) return hipErrorInvalidValue;
    char* const w = (char*)ws;
    const size_t ob = (P * th * (size_t)a->head_dim * 4 + 255) & ~(size_t)255;
    const size_t mb = (P * th * 4 + 255) & ~(size_t)255;
    p.part_o = (float*)w;
    p.part_m = (float*)(w + ob);
    p.part_z = (float*)(w + ob + mb);
  }
  const int st = a->cache_dtype, lt = a->long_cache_dtype;
  hipError_t e = a->head_dim == 64    ? launch_f32_d<64>(p, st, lt, f.nw, stream)
                 : a->head_dim == 128 ? launch_f32_d<128>(p, st, lt, f.nw, stream)
                                      : launch_f32_d<256>(p, st, lt, f.nw, stream);
  if (e != hipSuccess || p.direct) return e;
  return launch_paged_combine(p.part_o, p.part_m, p.part_z, (int)P, a, stream);
}

}  // namespace sa
