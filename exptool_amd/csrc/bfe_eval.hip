// Evaluation: coefficient folding and the batch / field evaluators.
#include <math.h>

#include <algorithm>
#include <vector>

#include "bfe_field.hpp"

namespace bfe {

struct SLFoldArgs {
  double mul[kMaxLM];  // per-pair multiplier: N_lm times halofac (0 for skipped l)
  int lmax, nmax_use;
};

// Four lanes per (R radial nodes from i0, (l, m) pair p in m-major order), lane q
// summing radial orders q, q + 4, ...: the sums of a table row are shared by the
// nodes that read it (a node takes rows i and i + 1 of E and D and three rows of G),
// so R nodes cost 3 R + 4 rows instead of 7 R.  The four partial sums are combined
// across the lanes, D1/D2 formed, and the blocks rounded once to float32 (layout in
// bfe_field.hpp; the last node, never a cell start, is zero).  What bounds it is the
// latency and number of the row gathers: lmax 6, nmax 20, numr 2000, one set / 12
// sets, with one node a group of lanes and seven rows each 12.3 / 75 us, one, two and
// four nodes with shared rows 15.6 / 91, 10.5 / 55 and 10.3 / 47; small tables take
// one (sl_fold_rows).
struct SLFoldIn {
  const double* S;       // fold inputs
  const double* coef;
  int nmax, numr, nset;
  float* out;
  int64_t coef_stride, out_stride;
};
constexpr int kFoldLanes = 4;
// Nodes i0 .. i0 + R - 1 of the pair at place j of the l-major order, into the
// node blocks at o (2 np float4 a node) and the density blocks at od.
template <int R>
__device__ __forceinline__ void sl_fold_nodes(const SLFoldIn& f, const SLFoldArgs& a, int i0, int j,
                                              int q, const double* __restrict__ c, float4* o,
                                              float4* od) {
  const int np = sl_npairs(a.lmax), nmax = f.nmax, numr = f.numr;
  // lanes in l-major order, so that neighbours read the same rows
  int l = 0, m = j;
  while (m > l) m -= ++l;
  const int p = m * (a.lmax + 1) - m * (m - 1) / 2 + l - m;
  const double mul = a.mul[p];
  const bool two = m > 0;
  const double* cc = c + (size_t)(l * l + (two ? 2 * m - 1 : 0)) * nmax;
  const double* cs = c + (size_t)(l * l + 2 * m) * nmax;
  const size_t plane = (size_t)(a.lmax + 1) * numr * nmax;
  const double* E = f.S + (size_t)l * numr * nmax;
  // rows of E and D: i0 .. i0 + R; of G: i0 - 1 .. i0 + R (the first node is
  // centred on row 1, so there row -1 stands for row 2); rows past the table
  // repeat its last
  int re[R + 1], rg[R + 2];
#pragma unroll
  for (int k = 0; k <= R; ++k) re[k] = (i0 + k < numr ? i0 + k : numr - 1) * nmax;
#pragma unroll
  for (int k = 0; k < R + 2; ++k) {
    const int r = i0 + k - 1;
    rg[k] = (r < 0 ? 2 : r < numr ? r : numr - 1) * nmax;
  }
  double e[R + 1][2], d[R + 1][2], w[R + 2][2];
#pragma unroll
  for (int k = 0; k <= R; ++k) e[k][0] = e[k][1] = d[k][0] = d[k][1] = 0.0;
#pragma unroll
  for (int k = 0; k < R + 2; ++k) w[k][0] = w[k][1] = 0.0;
  for (int n = q; n < a.nmax_use; n += kFoldLanes) {
    const double c0 = cc[n] * mul;
    const double c1 = two ? cs[n] * mul : 0.0;
    const double *En = E + n, *Dn = En + plane, *Gn = Dn + plane;
#pragma unroll
    for (int k = 0; k <= R; ++k) {
      const double te = En[re[k]], td = Dn[re[k]];
      e[k][0] += c0 * te;
      e[k][1] += c1 * te;
      d[k][0] += c0 * td;
      d[k][1] += c1 * td;
    }
#pragma unroll
    for (int k = 0; k < R + 2; ++k) {
      const double tg = Gn[rg[k]];
      w[k][0] += c0 * tg;
      w[k][1] += c1 * tg;
    }
  }
  // fixed-order combination: (q0 + q1) + (q2 + q3) on every lane of the group
  auto sum = [](double v) {
    v += __shfl_xor(v, 1, kFoldLanes);
    return v + __shfl_xor(v, 2, kFoldLanes);
  };
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int k = 0; k <= R; ++k) {
      e[k][h] = sum(e[k][h]);
      d[k][h] = sum(d[k][h]);
    }
#pragma unroll
    for (int k = 0; k < R + 2; ++k) w[k][h] = sum(w[k][h]);
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = i0 + k;
    if (i >= numr) break;
    const size_t at = (size_t)k * np + p;
    const bool last = i == numr - 1;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (q == 0) {
      // node i and the step to node i+1, so that the evaluation interpolates
      // with one FMA: E_i + x2 (E_i+1 - E_i)
      if (!last)
        v = make_float4((float)e[k][0], (float)e[k][1], (float)(e[k + 1][0] - e[k][0]),
                        (float)(e[k + 1][1] - e[k][1]));
      o[2 * at] = v;
    } else if (q == 1) {
      // rows c - 1, c, c + 1 about c = max(i, 1)
      const bool first = k == 0 && i0 == 0;
      double b[2], z[2], t[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        b[h] = first ? w[1][h] : w[k][h];
        z[h] = first ? w[2][h] : w[k + 1][h];
        t[h] = first ? w[0][h] : w[k + 2][h];
      }
      if (!last)
        v = make_float4((float)(0.5 * (t[0] - b[0])), (float)(0.5 * (t[1] - b[1])),
                        (float)(b[0] - 2.0 * z[0] + t[0]), (float)(b[1] - 2.0 * z[1] + t[1]));
      o[2 * at + 1] = v;
    } else if (q == 2) {
      if (!last)
        v = make_float4((float)d[k][0], (float)d[k][1], (float)d[k + 1][0], (float)d[k + 1][1]);
      od[at] = v;
    }
  }
}

template <int R>
__device__ __forceinline__ void sl_fold_block(const SLFoldIn& f, const SLFoldArgs& a, unsigned block,
                                              int set) {
  const int np = sl_npairs(a.lmax);
  const unsigned gid = block * blockDim.x + threadIdx.x;
  const unsigned idx = gid / kFoldLanes;
  const int g = (int)(idx / (unsigned)np);
  const int i0 = g * R;
  // groups of four lanes are whole within a wave, so a group leaves together
  if (i0 >= f.numr) return;
  float4* o = reinterpret_cast<float4*>(f.out + (size_t)set * f.out_stride);
  sl_fold_nodes<R>(f, a, i0, (int)(idx - (unsigned)g * (unsigned)np), (int)(gid & (kFoldLanes - 1)),
                   f.coef + (size_t)set * f.coef_stride, o + (size_t)i0 * np * 2,
                   o + (size_t)f.numr * np * 2 + (size_t)i0 * np);
}

template <int R>
__global__ __launch_bounds__(256) void sl_fold_kernel(SLFoldIn f, SLFoldArgs a) {
  sl_fold_block<R>(f, a, blockIdx.x, blockIdx.y);
}

struct EOFFoldArgs {
  double mmul[kMaxM + 1];  // per-m multiplier (range / no_odd mask)
  int nuse;
  int numx, numy;          // grid, for the float64 edge blocks
};

// The float64 edge blocks of the folded field (after the float32 blocks of
// each set): the m = 0 cos sums [pot, rforce, zforce, dens] of edge node e
// (eof_edge_index) from its float64 fold inputs E[f][n][edge], as the float32
// blocks sum them for m = 0.  One serial chain of norder reads a lane, so the
// reads of six orders go out together; with the density a test inside the loop
// each order waited for its own (density fold at mmax 2, 257 x 129 nodes, 24.2 ->
// 20.1 us).
template <bool DENS>
__device__ __forceinline__ void eof_fold_edge(const double* __restrict__ E, int64_t nedge,
                                              int64_t e, const double* __restrict__ cf, int mmax,
                                              int norder, const EOFFoldArgs& a,
                                              float* __restrict__ out_set) {
  double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 6
  for (int n = 0; n < a.nuse; ++n) {
    const double c = cf[n];
#pragma unroll
    for (int f = 0; f < (DENS ? 4 : 3); ++f) s[f] += c * E[((size_t)f * norder + n) * nedge + e];
  }
  const double mul = a.mmul[0];
  double4* o = reinterpret_cast<double4*>(out_set + eof_fold32_floats(a.numx, a.numy, mmax)) + e;
  *o = make_double4(s[0] * mul, s[1] * mul, s[2] * mul, s[3] * mul);
}

// A block of eight waves folds kFoldNodes nodes: lane = node, so the
// function-major float32 tables are read coalesced (sums in float64), and a wave
// takes one row group q at a time (q = m for cos m = 0..mmax, mmax + m for sin
// m = 1..mmax), so the coefficients are scalar loads.  Each row group is one half
// [pot, rf, zf, dens] of the 8-float block [potC, rfC, zfC, dC, potS, rfS, zfS, dS]
// of its m (the sin half of m = 0 is zero); four m at a time, the halves are put
// together in LDS and leave as 128 bytes of a node, where 16-byte stores cost an
// L2 request each.  grid.x = ceil(nedge / 512) blocks a set for the float64 edge
// blocks (eof_fold_edge) of the m = 0 cos rows, first so that they do not trail,
// then the node blocks, each XCD (block index modulo eight) a contiguous range of
// them; grid.y = groups of SETS coefficient sets, which share the reads of the
// tables.  What bounds it is memory: 93 MB of tables at mmax 6, norder 18, 257 x
// 129 nodes (one set 21.5 -> 19 us), and 7.4 MB of results a set (12 sets: one set
// a thread 230 us; four sets 92, their stores made whole 72; six sets 69).
constexpr int kFoldNodes = 64;
constexpr int kFoldThreads = 512;
constexpr int kFoldM = 4;            // m per group: one row group a wave
constexpr int kEofFoldSets = 6;
struct EOFFoldIn {
  const float* T[4];
  const double *ccos, *csin;
  int mmax, norder, nset, per_xcd;
  int64_t nodes, nedge;
  const double* E;
  float* out;
  int64_t coef_stride, out_stride;
};
// The pointers come as arguments of their own: read from the struct they lose
// __restrict__, and with it the scalar loads of the coefficients (six sets 69 -> 115 us).
template <int SETS>
__device__ __forceinline__ void eof_fold_block(
    const float* __restrict__ T0, const float* __restrict__ T1, const float* __restrict__ T2,
    const double* __restrict__ ccos, const double* __restrict__ csin,
    const double* __restrict__ E, float* __restrict__ out, const EOFFoldIn& f, const EOFFoldArgs& a,
    unsigned block, int set0) {
  __shared__ float4 s_fold[SETS][kFoldNodes][2 * kFoldM];
  const int mmax = f.mmax, norder = f.norder, nset = f.nset, per_xcd = f.per_xcd;
  const int64_t nodes = f.nodes, nedge = f.nedge, coef_stride = f.coef_stride, out_stride = f.out_stride;
  const unsigned eblocks = (unsigned)((nedge + kFoldThreads - 1) / kFoldThreads) * SETS;
  if (block < eblocks) {
    const int k = set0 + (int)(block % SETS);
    const int64_t e = (int64_t)(block / SETS) * kFoldThreads + threadIdx.x;
    if (k < nset && e < nedge)
      eof_fold_edge<false>(E, nedge, e, ccos + (size_t)k * coef_stride, mmax, norder, a,
                           out + (size_t)k * out_stride);
    return;
  }
  const unsigned b = block - eblocks;
  const int64_t node0 = ((int64_t)(b & 7) * per_xcd + (b >> 3)) * kFoldNodes;
  if (node0 >= nodes) return;
  const int lane = threadIdx.x & 63;
  const int64_t node = node0 + lane < nodes ? node0 + lane : nodes - 1;
  const unsigned nn = nodes - node0 < kFoldNodes ? (unsigned)(nodes - node0) : kFoldNodes;
  for (int m0 = 0; m0 <= mmax; m0 += kFoldM) {
    const int wave = uni(threadIdx.x >> 6), m = m0 + (wave & (kFoldM - 1));
    const bool sn = wave >= kFoldM;
    if (m <= mmax && !(sn && m == 0)) {
      const int q = sn ? mmax + m : m;
      const double* cf[SETS];
#pragma unroll
      for (int k = 0; k < SETS; ++k)   // a group past the last set repeats it and writes nothing
        cf[k] = (sn ? csin : ccos) + (size_t)(set0 + k < nset ? set0 + k : nset - 1) * coef_stride +
                (size_t)m * norder;
      const double mul = a.mmul[m];
      const size_t row = (size_t)q * norder * nodes + node;
      const float* t0 = T0 + row;
      const float* t1 = T1 + row;
      const float* t2 = T2 + row;
      double v[SETS][3];
#pragma unroll
      for (int k = 0; k < SETS; ++k)
#pragma unroll
        for (int f = 0; f < 3; ++f) v[k][f] = 0.0;
#pragma unroll 6
      for (int n = 0; n < a.nuse; ++n) {
        const size_t o = (size_t)n * nodes;
        const float t[3] = {t0[o], t1[o], t2[o]};
#pragma unroll
        for (int k = 0; k < SETS; ++k) {
          const double c = cf[k][n];
#pragma unroll
          for (int f = 0; f < 3; ++f) v[k][f] += c * t[f];
        }
      }
      // slot j of a node at j ^ (node & 7): eight lanes' stores on eight bank groups
      const int j = 2 * (m - m0) + (sn ? 1 : 0), sw = lane & 7;
#pragma unroll
      for (int k = 0; k < SETS; ++k) {
        s_fold[k][lane][j ^ sw] =
            make_float4((float)(v[k][0] * mul), (float)(v[k][1] * mul), (float)(v[k][2] * mul), 0.f);
        if (m == 0) s_fold[k][lane][1 ^ sw] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
    __syncthreads();
    const unsigned len = 2u * (unsigned)(mmax + 1 - m0 < kFoldM ? mmax + 1 - m0 : kFoldM);
#pragma unroll
    for (int k = 0; k < SETS; ++k) {
      if (set0 + k >= nset) break;
      float4* o = reinterpret_cast<float4*>(out + (size_t)(set0 + k) * out_stride) +
                  (size_t)node0 * (2 * (mmax + 1)) + 2 * m0;
      for (unsigned f = threadIdx.x; f < nn * len; f += kFoldThreads) {
        const unsigned d = f / len, j = f - d * len;
        o[d * (2u * (unsigned)(mmax + 1)) + j] = s_fold[k][d][j ^ (d & 7)];
      }
    }
    __syncthreads();
  }
}

template <int SETS>
__global__ __launch_bounds__(kFoldThreads) void eof_fold_kernel(EOFFoldIn f, EOFFoldArgs a) {
  eof_fold_block<SETS>(f.T[0], f.T[1], f.T[2], f.ccos, f.csin, f.E, f.out, f, a, blockIdx.x, blockIdx.y * SETS);
}

// One set with the density: one thread per (row group, node), the row groups one
// after the other (q as above), so that a block reads 1 KB of a table row and the
// grid streams the rows in turn.  Bound by those reads (124 MB at mmax 6, 257 x
// 129 nodes): tables not in the cache 70 us, by blocks of 64 nodes 73 - 77; in the
// cache, where the 16-byte stores cost, 38.4 and 36.2.  mmax 12: 124 / 136 and 69.8 /
// 67.6, mmax 2: 31.5 / 35.8 and 19.0 / 19.8.
__global__ __launch_bounds__(256) void eof_fold_rows_kernel(
    const float* __restrict__ T0, const float* __restrict__ T1, const float* __restrict__ T2,
    const float* __restrict__ T3, const double* __restrict__ ccos, const double* __restrict__ csin,
    const double* __restrict__ E, float* __restrict__ out, EOFFoldIn f, EOFFoldArgs a, unsigned chunks) {
  const unsigned eblocks = (unsigned)((f.nedge + 255) / 256);
  if (blockIdx.x < eblocks) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < f.nedge) eof_fold_edge<true>(E, f.nedge, e, ccos, f.mmax, f.norder, a, out);
    return;
  }
  const unsigned b = blockIdx.x - eblocks;
  const int q = (int)(b / chunks);
  const int64_t nodes = f.nodes, node = (int64_t)(b - (unsigned)q * chunks) * 256 + threadIdx.x;
  if (node >= nodes) return;
  const bool sn = q > f.mmax;
  const int m = sn ? q - f.mmax : q;
  const double* cf = (sn ? csin : ccos) + (size_t)m * f.norder;
  const double mul = a.mmul[m];
  const size_t row = (size_t)q * f.norder * nodes + node;
  const float *t0 = T0 + row, *t1 = T1 + row, *t2 = T2 + row, *t3 = T3 + row;
  double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 6
  for (int n = 0; n < a.nuse; ++n) {
    const double c = cf[n];
    const size_t o = (size_t)n * nodes;
    v[0] += c * t0[o];
    v[1] += c * t1[o];
    v[2] += c * t2[o];
    v[3] += c * t3[o];
  }
  float4* o = reinterpret_cast<float4*>(out) + ((size_t)node * (f.mmax + 1) + m) * 2;
  o[sn ? 1 : 0] = make_float4((float)(v[0] * mul), (float)(v[1] * mul), (float)(v[2] * mul), (float)(v[3] * mul));
  if (q == 0) o[1] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Both folds of one frozen field in one launch: the SL fold waits on its own
// gathers and runs in the shadow of the EOF fold's table reads (23 us; as two
// launches on two streams 21 and 12 us and 15 us of events between them).
template <int R>
__global__ __launch_bounds__(kFoldThreads) void field_fold_kernel(SLFoldIn sf, SLFoldArgs sa,
                                                                  unsigned slblocks, EOFFoldIn ef,
                                                                  EOFFoldArgs ea) {
  if (blockIdx.x < slblocks) sl_fold_block<R>(sf, sa, blockIdx.x, 0);
  else eof_fold_block<1>(ef.T[0], ef.T[1], ef.T[2], ef.ccos, ef.csin, ef.E, ef.out, ef, ea,
                         blockIdx.x - slblocks, 0);
}

static int ensure_folded(Context* c, float** d, size_t* have, size_t floats, hipStream_t s) {
  if (*d && *have >= floats) return 0;
  if (*d) {
    BFE_HIP(c, hipStreamSynchronize(s));
    (void)hipFree(*d);
    *d = nullptr;
    *have = 0;
  }
  BFE_HIP(c, hipMalloc(d, floats * sizeof(float)));
  *have = floats;
  return 0;
}

static size_t sl_fold_floats(const Context* c) { return (size_t)c->numr * sl_npairs(c->lmax) * 12; }
// float32 blocks of every node, then the float64 m = 0 cos blocks (four
// values, eight floats) of the edge nodes
static size_t eof_fold_floats(const Context* c) {
  return (size_t)eof_fold32_floats(c->numx, c->numy, c->mmax) +
         (size_t)eof_edge_count(c->numx, c->numy) * 8;
}

// The arguments of the SL fold of nset coefficient sets (stride (lmax+1)^2 nmax)
// into out (stride sl_fold_floats); returns its lanes.
static int64_t sl_fold_args(Context* c, const double* coef, int nset, double halofac, int lmax_use,
                            int nmax_use, int L1, int L2, bool no_odd, float* out, SLFoldIn* f,
                            SLFoldArgs* args) {
  SLFoldArgs& a = *args;
  double lmul[kMaxL + 1];
  for (int l = 0; l <= kMaxL; ++l) {
    bool keep = l <= lmax_use;
    if (l >= 1 && (l > L2 || l < L1)) keep = false;
    if (l >= 1 && no_odd && (l & 1)) keep = false;
    lmul[l] = keep ? halofac : 0.0;
  }
  a.lmax = c->lmax;
  a.nmax_use = nmax_use;
  // N_lm (spheresl.py:858-861) folded into the table
  for (int m = 0, p = 0; m <= c->lmax; ++m)
    for (int l = m; l <= c->lmax; ++l, ++p) {
      double ratio = 1.0;
      for (int k = 1; k <= m; ++k) ratio /= (double)(l - k + 1) * (double)(l + k);
      double N = sqrt((0.5 * l + 0.25) / kPi * ratio);
      if (m > 0) N *= 1.4142135623730951;
      a.mul[p] = lmul[l] * N;
    }
  *f = SLFoldIn{c->sl_fold64, coef, c->nmax, c->numr, nset, out,
                (int64_t)(c->lmax + 1) * (c->lmax + 1) * c->nmax, (int64_t)sl_fold_floats(c)};
  const int rows = sl_fold_rows(c->numr, c->lmax);
  return (int64_t)((c->numr + rows - 1) / rows) * sl_npairs(c->lmax) * kFoldLanes;
}

static int sl_fold_into(Context* c, const double* coef, int nset, double halofac, int lmax_use,
                        int nmax_use, int L1, int L2, bool no_odd, float* out, hipStream_t s) {
  SLFoldIn f;
  SLFoldArgs a;
  const int64_t lanes = sl_fold_args(c, coef, nset, halofac, lmax_use, nmax_use, L1, L2, no_odd, out, &f, &a);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((lanes + 255) / 256), (unsigned)nset), dim3(256), 0, s, f, a);
  };
  if (sl_fold_rows(c->numr, c->lmax) == 2) go(sl_fold_kernel<2>);
  else go(sl_fold_kernel<1>);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

static int sl_fold(Context* c, int slot, const double* coef, double halofac, int lmax_use,
                   int nmax_use, int L1, int L2, bool no_odd, hipStream_t s) {
  SLFolded& f = c->slf[slot];
  int rc = ensure_folded(c, &f.d, &f.floats, sl_fold_floats(c), s);
  if (rc) return rc;
  rc = sl_fold_into(c, coef, 1, halofac, lmax_use, nmax_use, L1, L2, no_odd, f.d, s);
  if (rc) return rc;
  f.valid = true;
  return 0;
}

// The arguments of the EOF fold, likewise; returns the blocks of `sets` sets.
static unsigned eof_fold_args(Context* c, const double* ccos, const double* csin, int nset, int sets,
                              int mmax_use, int nuse, int m1, int m2, bool no_odd, bool compat_mask,
                              bool dens, float* out, EOFFoldIn* f, EOFFoldArgs* args) {
  const int64_t nodes = (int64_t)(c->numx + 1) * (c->numy + 1);
  EOFFoldArgs& a = *args;
  for (int m = 0; m <= kMaxM; ++m) {
    double mul = 1.0;
    if (m > mmax_use || m > m2 || m < m1) mul = 0.0;
    if (no_odd && m >= 1 && (m & 1)) {
      // eof.force_eval mask = |cos(pi m / 2)| (eof.py:833): ~6e-17 for odd m
      mul *= compat_mask ? fabs(cos((kPi / 2.0) * m)) : 0.0;
    }
    a.mmul[m] = mul;
  }
  a.nuse = nuse;
  a.numx = c->numx;
  a.numy = c->numy;
  const int64_t nedge = eof_edge_count(c->numx, c->numy);
  const int64_t chunks = (nodes + kFoldNodes - 1) / kFoldNodes;
  const int per_xcd = (int)((chunks + 7) / 8);
  *f = EOFFoldIn{{c->eof_fold32[0], c->eof_fold32[1], c->eof_fold32[2],
                  dens ? c->eof_fold32[3] : c->eof_fold32[0]},
                 ccos, csin, c->mmax, c->norder, nset, per_xcd, nodes, nedge, c->eof_edge64, out,
                 (int64_t)(c->mmax + 1) * c->norder, (int64_t)eof_fold_floats(c)};
  return 8u * (unsigned)per_xcd + (unsigned)((nedge + kFoldThreads - 1) / kFoldThreads) * sets;
}

static int eof_fold_into(Context* c, const double* ccos, const double* csin, int nset, int mmax_use,
                         int nuse, int m1, int m2, bool no_odd, bool compat_mask, bool dens, float* out,
                         hipStream_t s) {
  EOFFoldIn f;
  EOFFoldArgs a;
  auto go = [&](auto kernel, int sets) {
    const unsigned grid = eof_fold_args(c, ccos, csin, nset, sets, mmax_use, nuse, m1, m2, no_odd,
                                        compat_mask, false, out, &f, &a);
    hipLaunchKernelGGL(kernel, dim3(grid, (unsigned)((nset + sets - 1) / sets)), dim3(kFoldThreads), 0, s, f, a);
  };
  if (dens) {   // one set
    eof_fold_args(c, ccos, csin, 1, 1, mmax_use, nuse, m1, m2, no_odd, compat_mask, true, out, &f, &a);
    const unsigned chunks = (unsigned)((f.nodes + 255) / 256);
    const unsigned grid = (unsigned)((f.nedge + 255) / 256) + (2u * (unsigned)f.mmax + 1) * chunks;
    hipLaunchKernelGGL(eof_fold_rows_kernel, dim3(grid), dim3(256), 0, s, f.T[0], f.T[1], f.T[2], f.T[3], ccos,
                       csin, f.E, out, f, a, chunks);
  } else if (nset > 1) {
    go(eof_fold_kernel<kEofFoldSets>, kEofFoldSets);
  } else {
    go(eof_fold_kernel<1>, 1);
  }
  BFE_HIP(c, hipGetLastError());
  return 0;
}

static int eof_fold(Context* c, int slot, const double* ccos, const double* csin, int mmax_use,
                    int nuse, int m1, int m2, bool no_odd, bool compat_mask, bool dens,
                    hipStream_t s) {
  EOFFolded& f = c->eoff[slot];
  int rc = ensure_folded(c, &f.d, &f.floats, eof_fold_floats(c), s);
  if (rc) return rc;
  rc = eof_fold_into(c, ccos, csin, 1, mmax_use, nuse, m1, m2, no_odd, compat_mask, dens, f.d, s);
  if (rc) return rc;
  f.valid = true;
  return 0;
}

// ---------------------------------------------------------------------------
// batch evaluators
// ---------------------------------------------------------------------------
template <bool DENS>
__global__ __launch_bounds__(256) void sl_eval_kernel(
    const float* __restrict__ px, const float* __restrict__ py, const float* __restrict__ pz,
    int64_t n, SLGeom g, const float* __restrict__ F, int L, uint32_t flags, double densfac, float* den0, float* den1, float* pot0, float* pot1,
    float* potr, float* pott, float* potp) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const double x = px[p], y = py[p], z = pz[p];
  const double r = sqrt(x * x + y * y + z * z);  // no floor (spheresl.py:1257)
  const double costh = z / r;                     // NaN at r = 0, as the reference
  double c1, s1;
  planar_angle(x, y, c1, s1);
  SLOut o;
  sl_eval_folded<DENS>(g, F, L, r, costh, c1, s1, flags, o);
  if (den0) den0[p] = (float)(o.den0 * densfac);
  if (den1) den1[p] = (float)(o.den1 * densfac);
  if (pot0) pot0[p] = (float)o.pot0;
  if (pot1) pot1[p] = (float)o.pot1;
  if (potr) potr[p] = (float)o.potr;
  if (pott) pott[p] = (float)o.pott;
  if (potp) potp[p] = (float)o.potp;
}

template <bool DENS>
__global__ __launch_bounds__(256) void eof_eval_kernel(
    const float* __restrict__ px, const float* __restrict__ py, const float* __restrict__ pz,
    int64_t n, EOFGeom g, const float* __restrict__ F, float* p0, float* p, float* fr,
    float* fp, float* fz, float* d0, float* d) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double x = px[i], y = py[i], z = pz[i];
  const double R = sqrt(x * x + y * y + 1.e-10);  // eof.py:1070
  double c1, s1;
  planar_angle(x, y, c1, s1);
  EOFOut o;
  eof_eval_folded<DENS>(g, F, R, z, c1, s1, o);
  if (p0) p0[i] = (float)o.p0;
  if (p) p[i] = (float)o.p;
  if (fr) fr[i] = (float)o.fr;
  if (fp) fp[i] = (float)o.fp;
  if (fz) fz[i] = (float)o.fz;
  if (DENS) {
    if (d0) d0[i] = (float)o.d0;
    if (d) d[i] = (float)o.d;
  }
}

// Point forms: the caller gives the coordinates the reference's point
// evaluators take, in float64, and receives float64 rows of n values.
// spheresl.force_eval / all_eval (spheresl.py:1107-1234, :987-1102) at
// (r, cos theta, phi): out rows den0, den1 (l >= 1), pot0, pot1, potr, pott,
// potp; densities are written only with DENS (zero rows otherwise).
template <bool DENS>
__global__ __launch_bounds__(256) void sl_eval_sph_kernel(
    const double* __restrict__ pr, const double* __restrict__ pct, const double* __restrict__ pph,
    int64_t n, SLGeom g, const float* __restrict__ F, int L, uint32_t flags, double densfac,
    double* __restrict__ out) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  double s1, c1;
  sincos(pph[p], &s1, &c1);
  SLOut o;
  sl_eval_folded<DENS>(g, F, L, pr[p], pct[p], c1, s1, flags, o);
  out[p] = DENS ? o.den0 * densfac : 0.0;
  out[n + p] = DENS ? o.den1 * densfac : 0.0;
  out[2 * n + p] = o.pot0;
  out[3 * n + p] = o.pot1;
  out[4 * n + p] = o.potr;
  out[5 * n + p] = o.pott;
  out[6 * n + p] = o.potp;
}

// eof.force_eval / accumulated_eval (eof.py:756-872, :874-929) at planar
// radius R (as given), z, phi: out rows p0, p (m >= 1), fr, fp, fz, d0,
// d (m >= 1), fr0, fz0 (the m = 0 parts of fr, fz).
template <bool DENS>
__global__ __launch_bounds__(256) void eof_eval_cyl_kernel(
    const double* __restrict__ pR, const double* __restrict__ pz, const double* __restrict__ pph,
    int64_t n, EOFGeom g, const float* __restrict__ F, double* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s1, c1;
  sincos(pph[i], &s1, &c1);
  EOFOut o;
  eof_eval_folded<DENS>(g, F, pR[i], pz[i], c1, s1, o);
  out[i] = o.p0;
  out[n + i] = o.p;
  out[2 * n + i] = o.fr;
  out[3 * n + i] = o.fp;
  out[4 * n + i] = o.fz;
  out[5 * n + i] = DENS ? o.d0 : 0.0;
  out[6 * n + i] = DENS ? o.d : 0.0;
  out[7 * n + i] = o.fr0;
  out[8 * n + i] = o.fz0;
}

// The point forms for few points: a block per point folds the coefficients into
// the blocks of the point's own cell (the sums of the whole-table folds, in the
// same order) and evaluates it from LDS.  A whole-table fold is 93 MB of table
// reads and a launch of its own; a point needs 4 nodes of the disc's 33 153 and
// one of the halo's 2 000.  Disc calls, whole-table fold / by cells: 24 points
// 25.8 / 16.0 us, 512 31.1 / 16.8, 1 024 30.9 / 27.6, 2 048 31.0 / 48.9, hence
// point_blocks = 512.
template <bool DENS>
__global__ __launch_bounds__(256) void sl_points_kernel(
    SLFoldIn f, SLFoldArgs a, const double* __restrict__ pr, const double* __restrict__ pct,
    const double* __restrict__ pph, int64_t n, SLGeom g, uint32_t flags, double densfac,
    double* __restrict__ out) {
  __shared__ float4 sA[2 * kMaxLM], sD[kMaxLM];
  const int64_t p = blockIdx.x;
  const double r = pr[p];
  const SLCell cell = sl_locate(r, g.cmap, g.scale, g.xi, g.numr, g.idxi, g.xi0, g.xin);
  const int lanes = sl_npairs(a.lmax) * kFoldLanes;
  for (int t = threadIdx.x; t < lanes; t += 256)
    sl_fold_nodes<1>(f, a, cell.i, t / kFoldLanes, t & (kFoldLanes - 1), f.coef, sA, sD);
  __syncthreads();
  if (threadIdx.x != 0) return;
  double s1, c1;
  sincos(pph[p], &s1, &c1);
  SLOut o;
  sl_eval_cell<DENS>(g, (const float4*)sA, sD, a.lmax, cell, pct[p], c1, s1, flags, o);
  out[p] = DENS ? o.den0 * densfac : 0.0;
  out[n + p] = DENS ? o.den1 * densfac : 0.0;
  out[2 * n + p] = o.pot0;
  out[3 * n + p] = o.pot1;
  out[4 * n + p] = o.potr;
  out[5 * n + p] = o.pott;
  out[6 * n + p] = o.potp;
}

template <bool DENS>
__global__ __launch_bounds__(256) void eof_points_kernel(
    const float* __restrict__ T0, const float* __restrict__ T1, const float* __restrict__ T2,
    const float* __restrict__ T3, const double* __restrict__ ccos, const double* __restrict__ csin,
    const double* __restrict__ E, int64_t nodes, int64_t nedge, int norder, EOFFoldArgs a,
    const double* __restrict__ pR, const double* __restrict__ pz, const double* __restrict__ pph,
    int64_t n, EOFGeom g, double* __restrict__ out) {
  __shared__ float4 sF[4][2 * (kMaxM + 1)];   // corner, (m, cos / sin): [pot, rf, zf, dens]
  __shared__ double4 sE[4];                   // m = 0 in float64, last grid column or row
  const int64_t i = blockIdx.x;
  const EOFCell cell = eof_locate(pR[i], pz[i], g.cmap, g.ascale, g.ihscale, g.xmin, g.idx, g.ymin,
                                  g.idy, g.numx, g.numy);
  const bool edge = cell.ix == g.numx - 1 || cell.iy == g.numy - 1;
  const int rows = 2 * g.mmax + 1;
  // lane: value (pot, rf, zf, dens), corner (ix + c / 2, iy + c % 2), row group
  for (int t = threadIdx.x; t < 16 * (rows + 1); t += 256) {
    const int f = t & 3, c = (t >> 2) & 3, q = t >> 4;
    const bool live = f < 3 || DENS;
    const int x = cell.ix + (c >> 1), y = cell.iy + (c & 1);
    if (q < rows) {
      const bool sn = q > g.mmax;
      const int m = sn ? q - g.mmax : q;
      const double* cf = (sn ? csin : ccos) + (size_t)m * norder;
      const float* T = (f == 0 ? T0 : f == 1 ? T1 : f == 2 ? T2 : T3) + (size_t)q * norder * nodes +
                       (size_t)x * (g.numy + 1) + y;
      double v = 0.0;
      if (live) {
#pragma unroll 6
        for (int k = 0; k < a.nuse; ++k) v += cf[k] * T[(size_t)k * nodes];
      }
      reinterpret_cast<float*>(&sF[c][2 * m + (sn ? 1 : 0)])[f] = live ? (float)(v * a.mmul[m]) : 0.f;
    } else if (edge) {
      const double* e = E + (size_t)f * norder * nedge + eof_edge_index(x, y, g.numx, g.numy);
      double v = 0.0;
      if (live) {
#pragma unroll 6
        for (int k = 0; k < a.nuse; ++k) v += ccos[k] * e[(size_t)k * nedge];
      }
      reinterpret_cast<double*>(&sE[c])[f] = v * a.mmul[0];
    }
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  auto wide = [](const float4& v) { return make_double4(v.x, v.y, v.z, v.w); };
  EOFCorners0 q0;
  q0.a = edge ? sE[0] : wide(sF[0][0]);
  q0.b = edge ? sE[1] : wide(sF[1][0]);
  q0.c = edge ? sE[2] : wide(sF[2][0]);
  q0.e = edge ? sE[3] : wide(sF[3][0]);
  double s1, c1;
  sincos(pph[i], &s1, &c1);
  EOFOut o;
  eof_eval_corners<DENS>(cell, g.mmax, q0, sF[0], sF[1], sF[2], sF[3], c1, s1, o);
  out[i] = o.p0;
  out[n + i] = o.p;
  out[2 * n + i] = o.fr;
  out[3 * n + i] = o.fp;
  out[4 * n + i] = o.fz;
  out[5 * n + i] = DENS ? o.d0 : 0.0;
  out[6 * n + i] = DENS ? o.d : 0.0;
  out[7 * n + i] = o.fr0;
  out[8 * n + i] = o.fz0;
}

// Fields.return_forces_cart at n points.  pts (may be NULL): the points in
// table-cell order as float4 (x, y, z, input index bits), outputs scattered
// back to input order; block b then takes logical block xcd_block(nb) so that
// each XCD evaluates a contiguous range of cells.  Without pts, point j of
// px/py/pz.  In cell order a block's points usually share a few SL radial
// nodes: when their force blocks fit in kStageFloat4, the block copies them
// to LDS and the SL sums read them there.  pts2 (may be NULL): a second set of n2
// points in its own cell order, numbered after the first.  Bound by vector ALU
// issue (77 % busy) and address units (71 %) where the chip is full: 2M points 131
// us with FOUR waves a SIMD (128 registers, 20 B spilled), 139 with three (144);
// fewer points by one wave's own latency, where three are faster
// (eval_four_waves).  The three-wave build states no number of waves: told three,
// the compiler takes as many registers in another order of the same instructions,
// 5 to 9 % slower (200 000 points 33.4 us, untold 31.3; 400 000 47.1 and 43.9).
template <bool FOUR>
__global__ __launch_bounds__(256, FOUR ? 4 : 1) void field_eval_kernel(
    const float* __restrict__ px, const float* __restrict__ py, const float* __restrict__ pz,
    int64_t n, const float4* __restrict__ pts, const float4* __restrict__ pts2, int64_t n2,
    FieldTables T, float* fx, float* fy, float* fz, float* pot, float* comp,
    float4* __restrict__ quad, int64_t total) {
  __shared__ float4 stage[kStageFloat4];
  __shared__ int smin[4], smax[4];
  // the second set's blocks follow the first's, whose number is a multiple of eight
  const unsigned b1 = 8 * (unsigned)((n + 2047) / 2048);
  const bool second = pts2 && blockIdx.x >= b1;
  const int64_t base = second ? n : 0;
  const unsigned b = second ? blockIdx.x - b1 : blockIdx.x;
  if (second) {
    pts = pts2;
    n = n2;
  }
  const int64_t j = (pts ? xcd_block((n + 255) / 256, b) : (int64_t)b) * 256 + threadIdx.x;
  if (pts && (j - threadIdx.x) >= n) return;   // whole block past the end (XCD mapping)
  const bool live = j < n;
  float qx = 0.f, qy = 0.f, qz = 0.f;
  int64_t i = 0;
  if (live) {
    if (pts) {
      const float4 q = pts[j];
      qx = q.x; qy = q.y; qz = q.z;
      i = base + (int64_t)__float_as_int(q.w);
    } else {
      qx = px[j]; qy = py[j]; qz = pz[j];
      i = j;
    }
  }
  bool staged = false;
  int imin = 0;
  SLCell cell{0.0, 0, 0.0, 0.0};
  if (pts) {
    if (live) cell = field_sl_cell(T.slg, qx, qy, qz);
    staged = stage_sl_nodes(T, live, cell.i, stage, smin, smax, imin);
  }
  if (!live) return;
  double cv[8];
  if (staged)
    field_eval_point<true>(T, qx, qy, qz, cv, &cell, stage, imin);
  else
    field_eval_point(T, qx, qy, qz, cv);
  if (quad) {
    // one 16-byte store per point; quad_split_kernel makes the four arrays
    quad[i] = make_float4((float)(cv[0] + cv[1]), (float)(cv[2] + cv[3]), (float)(cv[4] + cv[5]),
                          (float)(cv[6] + cv[7]));
    return;
  }
  if (fx) fx[i] = (float)(cv[0] + cv[1]);
  if (fy) fy[i] = (float)(cv[2] + cv[3]);
  if (fz) fz[i] = (float)(cv[4] + cv[5]);
  if (pot) pot[i] = (float)(cv[6] + cv[7]);
  if (comp) {
#pragma unroll
    for (int k = 0; k < 8; ++k) comp[(size_t)k * total + i] = (float)cv[k];
  }
}

// Fields.return_forces_cart at n points in input order, by split blocks
// (field_eval_split): for point counts that give the one-lane kernel less
// than a few waves per SIMD.  Points n1.. come from the second arrays.  Wave
// w writes output w of the block's points.
template <int LM, int MM>
__global__ __launch_bounds__(kSplitThreads) __attribute__((amdgpu_waves_per_eu(4))) void
field_eval_split_kernel(
    const float* __restrict__ px, const float* __restrict__ py, const float* __restrict__ pz,
    int64_t n1, const float* __restrict__ qx, const float* __restrict__ qy,
    const float* __restrict__ qz, int64_t n, FieldTables T, float* fx, float* fy, float* fz,
    float* pot, float* comp) {
  extern __shared__ __align__(16) double split_sm[];
  const SplitWave w = split_wave();
  const int64_t i = (int64_t)blockIdx.x * kSplitPts + w.lane;
  const bool live = i < n;
  float x = 1.f, y = 0.f, z = 0.f;
  if (live) {
    const bool a = i < n1;
    const int64_t k = a ? i : i - n1;
    x = (a ? px : qx)[k];
    y = (a ? py : qy)[k];
    z = (a ? pz : qz)[k];
  }
  double cv[8];
  field_eval_split<LM, MM>(T, x, y, z, w, split_sm, cv);
  if (!live) return;
  if (w.wave == 0 && fx) fx[i] = (float)(cv[0] + cv[1]);
  if (w.wave == 1 && fy) fy[i] = (float)(cv[2] + cv[3]);
  if (w.wave == 2 && fz) fz[i] = (float)(cv[4] + cv[5]);
  if (w.wave == 3 && pot) pot[i] = (float)(cv[6] + cv[7]);
  if (comp) {
    double v = cv[0];
#pragma unroll
    for (int k = 1; k < 8; ++k) v = w.wave == k ? cv[k] : v;
    comp[(size_t)w.wave * n + i] = (float)v;
  }
}

// Batched frozen fields (one coefficient set per snapshot): point j of the
// (snapshot, cell) order belongs to snapshot sorted[j] / ncell and uses that
// snapshot's folded tables.
__global__ __launch_bounds__(256) void field_eval_batch_kernel(
    int64_t n, const float4* __restrict__ pts, const uint32_t* __restrict__ sorted, uint32_t ncell,
    FieldTables T, const float* __restrict__ slB, int64_t sl_stride,
    const float* __restrict__ eofB, int64_t eof_stride, float* fx, float* fy, float* fz,
    float* pot, float4* __restrict__ quad) {
  __shared__ float4 stage[kStageFloat4];
  __shared__ int smin[4], smax[4];
  const int64_t nb = (n + 255) / 256;
  const int64_t j = xcd_block(nb) * 256 + threadIdx.x;
  if (j - threadIdx.x >= n) return;   // whole block past the end (XCD mapping)
  const bool live = j < n;
  float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
  int snap = 0;
  if (live) {
    q = pts[j];
    snap = (int)(sorted[j] / ncell);
  }
  // SL nodes are staged when all the block's points belong to one snapshot
  int s0, s1;
  block_minmax(live ? snap : 0x7fffffff, live ? snap : -1, smin, smax, s0, s1);
  __syncthreads();   // smin/smax are reused below
  T.slF = slB + (size_t)(live ? snap : s0) * sl_stride;
  T.eofF = eofB + (size_t)(live ? snap : s0) * eof_stride;
  SLCell cell{0.0, 0, 0.0, 0.0};
  bool staged = false;
  int imin = 0;
  if (s0 == s1) {
    if (live) cell = field_sl_cell(T.slg, q.x, q.y, q.z);
    staged = stage_sl_nodes(T, live, cell.i, stage, smin, smax, imin);
  }
  if (!live) return;
  const int64_t i = (int64_t)__float_as_int(q.w);
  double cv[8];
  if (staged)
    field_eval_point<true>(T, q.x, q.y, q.z, cv, &cell, stage, imin);
  else
    field_eval_point(T, q.x, q.y, q.z, cv);
  quad[i] = make_float4((float)(cv[0] + cv[1]), (float)(cv[2] + cv[3]), (float)(cv[4] + cv[5]),
                        (float)(cv[6] + cv[7]));
}

static int ensure_batch(Context* c, float** d, size_t* have, size_t floats) {
  if (*d && *have >= floats) return 0;
  if (*d) {
    BFE_HIP(c, hipDeviceSynchronize());
    (void)hipFree(*d);
    *d = nullptr;
    *have = 0;
  }
  BFE_HIP(c, hipMalloc(d, floats * sizeof(float)));
  *have = floats;
  return 0;
}

void batch_free(Context* c) {
  if (c->batch_sl) (void)hipFree(c->batch_sl);
  if (c->batch_eof) (void)hipFree(c->batch_eof);
  if (c->batch_off) (void)hipFree(c->batch_off);
  c->batch_sl = nullptr;
  c->batch_eof = nullptr;
  c->batch_off = nullptr;
  c->batch_sl_floats = c->batch_eof_floats = 0;
  c->batch_off_cap = 0;
}

int field_tables(Context* c, double rotpos, FieldTables& T) {
  if (!c->slf[1].valid || !c->eoff[1].valid)
    return set_error(c, BFE_ENOTABLE, "field not set (call bfe_field_set)");
  T.slg = sl_geom(c);
  T.eg = eof_geom(c);
  T.slF = c->slf[1].d;
  T.eofF = c->eoff[1].d;
  T.lmax = c->lmax;
  T.flags = (uint32_t)c->field_flags;
  T.ximin = *std::min_element(c->h_xi.begin(), c->h_xi.end());
  T.crot = cos(rotpos);
  T.srot = sin(rotpos);
  return 0;
}

}  // namespace bfe

using namespace bfe;

static unsigned nblocks256(int64_t n) { return (unsigned)((n + 255) / 256); }

extern "C" int bfe_sl_eval(bfe_ctx* h, const float* x, const float* y, const float* z, int64_t n,
                           const double* coef, int L1, int L2, uint32_t flags, float* den0,
                           float* den1, float* pot0, float* pot1, float* potr, float* pott,
                           float* potp, void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (!c->sl_ok) return set_error(c, BFE_ENOTABLE, "sl_eval: SL tables not set");
  if (n < 0 || !coef) return set_error(c, BFE_EINVAL, "sl_eval: bad n or NULL coef");
  if (n > 0 && (!x || !y || !z)) return set_error(c, BFE_EINVAL, "sl_eval: NULL input");
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  const bool dens = den0 || den1;
  int rc = sl_fold(c, 0, coef, 1.0, c->lmax, c->nmax, L1, L2, (flags & BFE_NO_ODD) != 0, s);
  if (rc) return rc;
  if (n == 0) return 0;
  const SLFolded& f = c->slf[0];
  const double densfac = (flags & BFE_COMPAT_SL_DENS) ? 0.25 * kPi : 0.25 / kPi;
  const uint32_t ef = flags & (BFE_COMPAT_SL_DENS | BFE_COMPAT_SL_EDGE | BFE_COMPAT_SL_COS_L);
  if (dens)
    hipLaunchKernelGGL(sl_eval_kernel<true>, dim3(nblocks256(n)), dim3(256), 0, s, x, y, z, n,
                       sl_geom(c), f.d, c->lmax, ef, densfac, den0, den1, pot0, pot1, potr, pott,
                       potp);
  else
    hipLaunchKernelGGL(sl_eval_kernel<false>, dim3(nblocks256(n)), dim3(256), 0, s, x, y, z, n,
                       sl_geom(c), f.d, c->lmax, ef, densfac, den0, den1, pot0, pot1, potr, pott,
                       potp);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

extern "C" int bfe_eof_eval(bfe_ctx* h, const float* x, const float* y, const float* z, int64_t n,
                            const double* cos_coef, const double* sin_coef, int m1, int m2,
                            uint32_t flags, float* p0, float* p, float* fr, float* fp, float* fz,
                            float* d0, float* d, void* stream) {
  (void)flags;
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (!c->eof_ok) return set_error(c, BFE_ENOTABLE, "eof_eval: EOF tables not set");
  if (n < 0 || !cos_coef || !sin_coef) return set_error(c, BFE_EINVAL, "eof_eval: bad n or NULL coef");
  if (n > 0 && (!x || !y || !z)) return set_error(c, BFE_EINVAL, "eof_eval: NULL input");
  const bool dens = d0 || d;
  if (dens && !c->eof_dens) return set_error(c, BFE_ENOTABLE, "eof_eval: no density tables");
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  int rc = eof_fold(c, 0, cos_coef, sin_coef, c->mmax, c->norder, m1, m2, false, false, dens, s);
  if (rc) return rc;
  if (n == 0) return 0;
  const EOFFolded& f = c->eoff[0];
  if (dens)
    hipLaunchKernelGGL(eof_eval_kernel<true>, dim3(nblocks256(n)), dim3(256), 0, s, x, y, z, n,
                       eof_geom(c), f.d, p0, p, fr, fp, fz, d0, d);
  else
    hipLaunchKernelGGL(eof_eval_kernel<false>, dim3(nblocks256(n)), dim3(256), 0, s, x, y, z, n,
                       eof_geom(c), f.d, p0, p, fr, fp, fz, d0, d);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

extern "C" int bfe_sl_eval_sph(bfe_ctx* h, const double* r, const double* costh,
                               const double* phi, int64_t n, const double* coef, int lmax_use,
                               int nmax_use, uint32_t flags, double* out, void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (!c->sl_ok) return set_error(c, BFE_ENOTABLE, "sl_eval_sph: SL tables not set");
  if (n < 0 || !coef) return set_error(c, BFE_EINVAL, "sl_eval_sph: bad n or NULL coef");
  if (n > 0 && (!r || !costh || !phi || !out))
    return set_error(c, BFE_EINVAL, "sl_eval_sph: NULL input or output");
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  const int ll = lmax_use < 0 ? c->lmax : std::min(lmax_use, c->lmax);
  const int nn = nmax_use < 0 ? c->nmax : std::min(nmax_use, c->nmax);
  if (n == 0) return 0;
  const bool no_odd = (flags & BFE_NO_ODD) != 0;
  const uint32_t pf = flags & (BFE_COMPAT_SL_EDGE | BFE_COMPAT_SL_COS_L);
  if (n <= c->point_blocks) {
    SLFoldIn in;
    SLFoldArgs a;
    sl_fold_args(c, coef, 1, 1.0, ll, nn, -(1 << 30), 1 << 30, no_odd, nullptr, &in, &a);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(256), 0, s, in, a, r, costh, phi, n, sl_geom(c), pf,
                         0.25 / kPi, out);
    };
    if (flags & BFE_EVAL_DENS) go(sl_points_kernel<true>);
    else go(sl_points_kernel<false>);
    BFE_HIP(c, hipGetLastError());
    return 0;
  }
  int rc = sl_fold(c, 0, coef, 1.0, ll, nn, -(1 << 30), 1 << 30, no_odd, s);
  if (rc) return rc;
  const SLFolded& f = c->slf[0];
  if (flags & BFE_EVAL_DENS)
    hipLaunchKernelGGL(sl_eval_sph_kernel<true>, dim3(nblocks256(n)), dim3(256), 0, s, r, costh,
                       phi, n, sl_geom(c), f.d, c->lmax, pf, 0.25 / kPi, out);
  else
    hipLaunchKernelGGL(sl_eval_sph_kernel<false>, dim3(nblocks256(n)), dim3(256), 0, s, r, costh,
                       phi, n, sl_geom(c), f.d, c->lmax, pf, 0.25 / kPi, out);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

extern "C" int bfe_eof_eval_cyl(bfe_ctx* h, const double* R, const double* z, const double* phi,
                                int64_t n, const double* cos_coef, const double* sin_coef,
                                int mmax_use, int nmax_use, uint32_t flags, double* out,
                                void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (!c->eof_ok) return set_error(c, BFE_ENOTABLE, "eof_eval_cyl: EOF tables not set");
  if (n < 0 || !cos_coef || !sin_coef)
    return set_error(c, BFE_EINVAL, "eof_eval_cyl: bad n or NULL coef");
  if (n > 0 && (!R || !z || !phi || !out))
    return set_error(c, BFE_EINVAL, "eof_eval_cyl: NULL input or output");
  const bool dens = (flags & BFE_EVAL_DENS) != 0;
  if (dens && !c->eof_dens) return set_error(c, BFE_ENOTABLE, "eof_eval_cyl: no density tables");
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  const int mm = mmax_use < 0 ? c->mmax : std::min(mmax_use, c->mmax);
  const int nn = nmax_use < 0 ? c->norder : std::min(nmax_use, c->norder);
  if (n == 0) return 0;
  const bool no_odd = (flags & BFE_NO_ODD) != 0, mask = (flags & BFE_COMPAT_EOF_MASK) != 0;
  if (n <= c->point_blocks) {
    EOFFoldIn in;
    EOFFoldArgs a;
    eof_fold_args(c, cos_coef, sin_coef, 1, 1, mm, nn, 0, 1 << 30, no_odd, mask, dens, nullptr, &in, &a);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(256), 0, s, in.T[0], in.T[1], in.T[2], in.T[3],
                         cos_coef, sin_coef, in.E, in.nodes, in.nedge, c->norder, a, R, z, phi, n,
                         eof_geom(c), out);
    };
    if (dens) go(eof_points_kernel<true>);
    else go(eof_points_kernel<false>);
    BFE_HIP(c, hipGetLastError());
    return 0;
  }
  int rc = eof_fold(c, 0, cos_coef, sin_coef, mm, nn, 0, 1 << 30, no_odd, mask, dens, s);
  if (rc) return rc;
  const EOFFolded& f = c->eoff[0];
  if (dens)
    hipLaunchKernelGGL(eof_eval_cyl_kernel<true>, dim3(nblocks256(n)), dim3(256), 0, s, R, z, phi,
                       n, eof_geom(c), f.d, out);
  else
    hipLaunchKernelGGL(eof_eval_cyl_kernel<false>, dim3(nblocks256(n)), dim3(256), 0, s, R, z,
                       phi, n, eof_geom(c), f.d, out);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

namespace bfe {

// Fold one coefficient set into the frozen field (bfe_field_set).
static int field_set_run(Context* c, const double* eof_cos, const double* eof_sin,
                         const double* sl_coef, double halofac, int disk_m, int disk_n,
                         int halo_l, int halo_n, uint32_t flags, hipStream_t s) {
  const int mm = disk_m < 0 ? c->mmax : std::min(disk_m, c->mmax);
  const int nn = disk_n < 0 ? c->norder : std::min(disk_n, c->norder);
  const int ll = halo_l < 0 ? c->lmax : std::min(halo_l, c->lmax);
  const int hn = halo_n < 0 ? c->nmax : std::min(halo_n, c->nmax);
  const bool no_odd = (flags & BFE_NO_ODD) != 0;
  int rc = ensure_folded(c, &c->slf[1].d, &c->slf[1].floats, sl_fold_floats(c), s);
  if (!rc) rc = ensure_folded(c, &c->eoff[1].d, &c->eoff[1].floats, eof_fold_floats(c), s);
  if (rc) return rc;
  SLFoldIn sf;
  SLFoldArgs sa;
  EOFFoldIn ef;
  EOFFoldArgs ea;
  const int64_t lanes = sl_fold_args(c, sl_coef, 1, halofac, ll, hn, -(1 << 30), 1 << 30, no_odd,
                                     c->slf[1].d, &sf, &sa);
  const unsigned eb = eof_fold_args(c, eof_cos, eof_sin, 1, 1, mm, nn, 0, 1 << 30, no_odd,
                                    (flags & BFE_COMPAT_EOF_MASK) != 0, false, c->eoff[1].d, &ef, &ea);
  const unsigned sb = (unsigned)((lanes + kFoldThreads - 1) / kFoldThreads);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(sb + eb), dim3(kFoldThreads), 0, s, sf, sa, sb, ef, ea);
  };
  if (sl_fold_rows(c->numr, c->lmax) == 2) go(field_fold_kernel<2>);
  else go(field_fold_kernel<1>);
  BFE_HIP(c, hipGetLastError());
  c->slf[1].valid = c->eoff[1].valid = true;
  c->field_halofac = halofac;
  c->field_flags = (int)(flags & (BFE_COMPAT_SL_COS_L | BFE_COMPAT_SL_EDGE));
  return 0;
}

// Evaluate n points: sorted (pts, the index in .w) or in input order.
// (fx, fy, fz, pot) rows of the float4 quad array, coalesced both ways.
__global__ __launch_bounds__(256) void quad_split_kernel(const float4* __restrict__ quad, int64_t n,
                                                         float* fx, float* fy, float* fz,
                                                         float* pot) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const float4 v = quad[i];
    if (fx) fx[i] = v.x;
    if (fy) fy[i] = v.y;
    if (fz) fz[i] = v.z;
    if (pot) pot[i] = v.w;
  }
}

// Evaluate n points: sorted (pts, the index in .w) or in input order.  In
// sorted order the outputs land at scattered indices; without comp, each
// point writes one float4 to scratch (one 16-byte store instead of four
// 4-byte ones, a quarter of the partial-line HBM writes) and a coalesced
// pass splits it into fx, fy, fz, pot.
static int field_eval_run(Context* c, const FieldTables& T, const float* x, const float* y,
                          const float* z, int64_t n, const float4* pts, float* fx, float* fy,
                          float* fz, float* pot, float* comp, hipStream_t s,
                          const float4* pts2 = nullptr, int64_t n1 = 0) {
  if (n == 0) return 0;
  float4* quad = nullptr;
  if (pts && !comp && (fx || fy || fz || pot)) {
    int rc = ensure_scratch(c, (size_t)n * sizeof(float4));
    if (rc) return rc;
    quad = (float4*)c->scratch;
  }
  const unsigned grid = pts2 ? xcd_grid(nblocks256(n1)) + xcd_grid(nblocks256(n - n1))
                        : pts ? xcd_grid(nblocks256(n)) : nblocks256(n);
  timer_begin(c, "field_eval", s);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, s, x, y, z, pts2 ? n1 : n, pts, pts2, n - n1, T,
                       fx, fy, fz, pot, comp, quad, n);
  };
  if (eval_four_waves(n, (T.flags & BFE_COMPAT_SL_COS_L) != 0)) go(field_eval_kernel<true>);
  else go(field_eval_kernel<false>);
  timer_end(c, "field_eval", s);
  BFE_HIP(c, hipGetLastError());
  if (quad) {
    hipLaunchKernelGGL(quad_split_kernel, dim3(nblocks256(n)), dim3(256), 0, s, quad, n, fx, fy,
                       fz, pot);
    BFE_HIP(c, hipGetLastError());
  }
  return 0;
}

// The same in input order by split blocks: n1 points of x, y, z, then n - n1
// of x2, y2, z2.
static int field_eval_split_run(Context* c, const FieldTables& T, const float* x, const float* y,
                                const float* z, int64_t n1, const float* x2, const float* y2,
                                const float* z2, int64_t n, float* fx, float* fy, float* fz,
                                float* pot, float* comp, hipStream_t s) {
  const unsigned grid = (unsigned)((n + kSplitPts - 1) / kSplitPts);
  const size_t lds = (size_t)split_lds_doubles(c->mmax, c->lmax) * sizeof(double);
  timer_begin(c, "field_eval", s);
  if (split_fixed(c->lmax, c->mmax))
    hipLaunchKernelGGL((field_eval_split_kernel<6, 6>), dim3(grid), dim3(kSplitThreads), lds, s, x, y,
                       z, n1, x2, y2, z2, n, T, fx, fy, fz, pot, comp);
  else
    hipLaunchKernelGGL((field_eval_split_kernel<-1, -1>), dim3(grid), dim3(kSplitThreads), lds, s, x,
                       y, z, n1, x2, y2, z2, n, T, fx, fy, fz, pot, comp);
  timer_end(c, "field_eval", s);
  BFE_HIP(c, hipGetLastError());
  return 0;
}

}  // namespace bfe

extern "C" int bfe_field_set(bfe_ctx* h, const double* eof_cos, const double* eof_sin,
                             const double* sl_coef, double halofac, int disk_m, int disk_n,
                             int halo_l, int halo_n, uint32_t flags, void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (!c->sl_ok || !c->eof_ok) return set_error(c, BFE_ENOTABLE, "field_set: tables not set");
  if (!eof_cos || !eof_sin || !sl_coef) return set_error(c, BFE_EINVAL, "field_set: NULL coef");
  BFE_HIP(c, hipSetDevice(c->device));
  return field_set_run(c, eof_cos, eof_sin, sl_coef, halofac, disk_m, disk_n, halo_l, halo_n,
                       flags, (hipStream_t)stream);
}

extern "C" int bfe_field_eval_cart(bfe_ctx* h, const float* x, const float* y, const float* z,
                                   int64_t n, double rotpos, float* fx, float* fy, float* fz,
                                   float* pot, float* comp, void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (n < 0) return set_error(c, BFE_EINVAL, "field_eval: n < 0");
  if (n > 0 && (!x || !y || !z)) return set_error(c, BFE_EINVAL, "field_eval: NULL input");
  FieldTables T;
  int rc = field_tables(c, rotpos, T);
  if (rc) return rc;
  if (n == 0) return 0;
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  const EvalForm form = eval_form(n, c->lmax, c->mmax, split_ok(T), c->order_min, c->split_eval_max);
  if (form == kEvalSplit)
    return field_eval_split_run(c, T, x, y, z, n, x, y, z, n, fx, fy, fz, pot, comp, s);
  const float4* pts = nullptr;
  if (form == kEvalOrdered) {
    rc = order_points(c, T, x, y, z, n, s, nullptr, nullptr, 1, nullptr, &pts);
    if (rc) return rc;
  }
  return field_eval_run(c, T, x, y, z, n, pts, fx, fy, fz, pot, comp, s);
}

// Fields.total_coefficients followed by Fields.return_forces_cart at the
// same particles (potential.py:98-252, :445-497).  Two concurrent branches,
// each folding its coefficients as soon as they are reduced:
//   caller stream  disc EOF accumulate, then the EOF fold (the longer branch,
//                  launched first);
//   internal       halo SL accumulate (second buffer set), then the SL fold;
// then, after the join, the evaluation: in the two orders that the accumulates
// sorted their particles to (ordering all points once more for it took 80 us of
// 427 at 1M + 1M), or, where one of them sums in input order, in an order of
// all points made on the caller's stream.  Few particles take one stream with
// both accumulates, reductions and folds each in one launch.  Results equal
// bfe_accumulate_disc_halo + bfe_field_set + bfe_field_eval_cart over the
// concatenated points.
extern "C" int bfe_forces_disc_halo(bfe_ctx* h, const float* dx, const float* dy,
                                    const float* dz, const float* dm, int64_t nd, const float* hx,
                                    const float* hy, const float* hz, const float* hm, int64_t nh,
                                    uint32_t acc_flags, double* cos_out, double* sin_out,
                                    double* coef_out, double halofac, int disk_m, int disk_n,
                                    int halo_l, int halo_n, uint32_t field_flags, double rotpos,
                                    float* fx, float* fy, float* fz, float* pot, float* comp,
                                    void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (!c->eof_ok || !c->sl_ok) return set_error(c, BFE_ENOTABLE, "forces_disc_halo: tables not set");
  if (!cos_out || !sin_out || !coef_out)
    return set_error(c, BFE_EINVAL, "forces_disc_halo: NULL coefficient output");
  if (nd < 0 || nh < 0) return set_error(c, BFE_EINVAL, "forces_disc_halo: n < 0");
  if ((nd > 0 && (!dx || !dy || !dz || !dm)) || (nh > 0 && (!hx || !hy || !hz || !hm)))
    return set_error(c, BFE_EINVAL, "forces_disc_halo: NULL input");
  if (nd + nh > (int64_t)0x7fffffff) return set_error(c, BFE_ELIMIT, "forces_disc_halo: nd + nh > 2^31 - 1");
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream, s1 = nullptr;
  const int64_t n = nd + nh;
  bool done = false;
  int rc = accumulate_both_small(c, dx, dy, dz, dm, nd, hx, hy, hz, hm, nh, acc_flags, cos_out, sin_out,
                                 coef_out, s, &done);
  if (rc) return rc;
  // the two inputs are evaluated as one set: by split blocks, or ordered
  const float4 *pts = nullptr, *pts2 = nullptr;
  FieldTables G;
  G.slg = sl_geom(c);
  G.eg = eof_geom(c);
  G.lmax = c->lmax;
  G.flags = field_flags & (BFE_COMPAT_SL_COS_L | BFE_COMPAT_SL_EDGE);
  const bool split = eval_split_two(n, c->lmax, c->mmax, split_ok(G), c->order_min, c->split_eval_max);
  if (done) {
    rc = field_set_run(c, cos_out, sin_out, coef_out, halofac, disk_m, disk_n, halo_l, halo_n,
                       field_flags, s);
    if (!rc && !split) rc = order_points2(c, G, dx, dy, dz, nd, hx, hy, hz, nh, s, &pts);
    if (rc) return rc;
  } else {
    const int mm = disk_m < 0 ? c->mmax : std::min(disk_m, c->mmax);
    const int nn = disk_n < 0 ? c->norder : std::min(disk_n, c->norder);
    const int ll = halo_l < 0 ? c->lmax : std::min(halo_l, c->lmax);
    const int hn = halo_n < 0 ? c->nmax : std::min(halo_n, c->nmax);
    const bool no_odd = (field_flags & BFE_NO_ODD) != 0;
    rc = fork_begin(c, s, &s1);
    if (rc) return rc;
    const float4 *dpts = nullptr, *hpts = nullptr;
    int r0 = 0, r1 = 0;
    // disc: accumulate and fold on the caller's stream
    auto disc = [&](const float4** order) {
      r0 = eof_accumulate_one(c, dx, dy, dz, dm, nd, cos_out, sin_out, s, order);
      if (!r0) r0 = eof_fold(c, 1, cos_out, sin_out, mm, nn, 0, 1 << 30, no_odd,
                             (field_flags & BFE_COMPAT_EOF_MASK) != 0, false, s);
    };
    // halo: accumulate and fold on the first internal stream, behind the sort of the
    // points where it is asked for
    auto halo = [&](bool sort, const float4** order) {
      swap_work(c);
      if (sort) r1 = order_points2(c, G, dx, dy, dz, nd, hx, hy, hz, nh, s1, &pts);
      if (!r1) r1 = sl_accumulate_one(c, hx, hy, hz, hm, nh, acc_flags, coef_out, s1, order);
      swap_work(c);
      if (!r1) r1 = sl_fold(c, 1, coef_out, halofac, ll, hn, -(1 << 30), 1 << 30, no_odd, s1);
    };
    const bool halo_sorts = sl_cell_ordered(c, nh, acc_flags);
    if (!split && halo_sorts && eof_cell_ordered(c, nd)) {
      // both orders serve the evaluation: the disc's EOF cells (few SL nodes and EOF
      // cells a block) and the halo's evaluation cells.  The disc's branch is the
      // longer and goes first
      disc(&dpts);
      halo(false, &hpts);
      pts = dpts;
      pts2 = hpts;
    } else if (halo_sorts || split || nd < nh || n == 0) {
      halo(false, nullptr);
      disc(nullptr);
      if (!r0 && n > 0 && !split) r0 = order_points2(c, G, dx, dy, dz, nd, hx, hy, hz, nh, s, &pts);
    } else {
      // The points' order takes the buffers that a halo summed in input order leaves
      // free, on its stream: that kernel's two blocks a CU (216 registers) leave the
      // disc's sort and deposit little room, so the disc's branch is the longer unless
      // the halo has more particles.  Order behind the disc's fold / before the halo's
      // sums, us at disc | halo particles: (6, 6) 300 000 | 30 000 214 / 169; (8, 8)
      // 300 000 | 300 000 364 / 352, 300 000 | 150 000 283 / 262; (10, 6) 300 000 |
      // 300 000 367 / 352, 30 000 | 300 000 287 / 311.
      halo(true, nullptr);
      disc(nullptr);
    }
    rc = fork_end(c, s);
    if (r0 || r1 || rc) return r0 ? r0 : (r1 ? r1 : rc);
  }
  c->field_halofac = halofac;
  c->field_flags = (int)(field_flags & (BFE_COMPAT_SL_COS_L | BFE_COMPAT_SL_EDGE));
  FieldTables T;
  rc = field_tables(c, rotpos, T);
  if (rc || n == 0) return rc;
  if (split)
    return field_eval_split_run(c, T, dx, dy, dz, nd, hx, hy, hz, n, fx, fy, fz, pot, comp, s);
  return field_eval_run(c, T, nullptr, nullptr, nullptr, n, pts, fx, fy, fz, pot, comp, s, pts2, nd);
}

extern "C" int bfe_field_set_batch(bfe_ctx* h, const double* eof_cos, const double* eof_sin,
                                   const double* sl_coef, int nsnap, double halofac, int disk_m,
                                   int disk_n, int halo_l, int halo_n, uint32_t flags,
                                   void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (!c->sl_ok || !c->eof_ok) return set_error(c, BFE_ENOTABLE, "field_set_batch: tables not set");
  if (!eof_cos || !eof_sin || !sl_coef) return set_error(c, BFE_EINVAL, "field_set_batch: NULL coef");
  if (nsnap < 1 || nsnap > 65535) return set_error(c, BFE_EINVAL, "field_set_batch: nsnap outside [1, 65535]");
  const int mm = disk_m < 0 ? c->mmax : std::min(disk_m, c->mmax);
  const int nn = disk_n < 0 ? c->norder : std::min(disk_n, c->norder);
  const int ll = halo_l < 0 ? c->lmax : std::min(halo_l, c->lmax);
  const int hn = halo_n < 0 ? c->nmax : std::min(halo_n, c->nmax);
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  c->batch_nsnap = 0;
  const size_t slf = sl_fold_floats(c), eoff = eof_fold_floats(c);
  int rc = ensure_batch(c, &c->batch_sl, &c->batch_sl_floats, slf * nsnap);
  if (rc) return rc;
  rc = ensure_batch(c, &c->batch_eof, &c->batch_eof_floats, eoff * nsnap);
  if (rc) return rc;
  const bool no_odd = (flags & BFE_NO_ODD) != 0;
  rc = eof_fold_into(c, eof_cos, eof_sin, nsnap, mm, nn, 0, 1 << 30, no_odd,
                     (flags & BFE_COMPAT_EOF_MASK) != 0, false, c->batch_eof, s);
  if (rc) return rc;
  rc = sl_fold_into(c, sl_coef, nsnap, halofac, ll, hn, -(1 << 30), 1 << 30, no_odd, c->batch_sl, s);
  if (rc) return rc;
  c->batch_nsnap = nsnap;
  c->batch_flags = (int)(flags & (BFE_COMPAT_SL_COS_L | BFE_COMPAT_SL_EDGE));
  return 0;
}

extern "C" int bfe_field_eval_batch(bfe_ctx* h, const float* x, const float* y, const float* z,
                                    const int64_t* offsets, int nsnap, double rotpos, float* fx,
                                    float* fy, float* fz, float* pot, void* stream) {
  if (!h) return BFE_EINVAL;
  Context* c = &h->c;
  if (!c->sl_ok || !c->eof_ok) return set_error(c, BFE_ENOTABLE, "field_eval_batch: tables not set");
  if (c->batch_nsnap < 1) return set_error(c, BFE_ENOTABLE, "field_eval_batch: no batch field (bfe_field_set_batch)");
  if (c->batch_sl_floats < sl_fold_floats(c) * (size_t)c->batch_nsnap ||
      c->batch_eof_floats < eof_fold_floats(c) * (size_t)c->batch_nsnap)
    return set_error(c, BFE_ENOTABLE, "field_eval_batch: batch field folded for other tables (call bfe_field_set_batch again)");
  if (!offsets || nsnap != c->batch_nsnap)
    return set_error(c, BFE_EINVAL, "field_eval_batch: need offsets for the %d snapshots of the batch field",
                     c->batch_nsnap);
  if (offsets[0] != 0) return set_error(c, BFE_EINVAL, "field_eval_batch: offsets[0] must be 0");
  for (int q = 0; q < nsnap; ++q)
    if (offsets[q + 1] < offsets[q]) return set_error(c, BFE_EINVAL, "field_eval_batch: offsets must not decrease");
  const int64_t n = offsets[nsnap];
  if (n > 0 && (!x || !y || !z)) return set_error(c, BFE_EINVAL, "field_eval_batch: NULL input");
  if (n == 0) return 0;
  BFE_HIP(c, hipSetDevice(c->device));
  hipStream_t s = (hipStream_t)stream;
  if (c->batch_off_cap < (size_t)nsnap + 1) {
    if (c->batch_off) {
      BFE_HIP(c, hipDeviceSynchronize());
      (void)hipFree(c->batch_off);
      c->batch_off = nullptr;
    }
    BFE_HIP(c, hipMalloc(&c->batch_off, ((size_t)nsnap + 1) * sizeof(int64_t)));
    c->batch_off_cap = (size_t)nsnap + 1;
  }
  BatchPieces d;
  d.off = c->batch_off;
  int rc = batch_pieces(c, offsets, nsnap, {}, 0, d, s);
  if (rc) return rc;
  const size_t slf = sl_fold_floats(c), eoff = eof_fold_floats(c);
  FieldTables T;
  T.slg = sl_geom(c);
  T.eg = eof_geom(c);
  T.slF = c->batch_sl;
  T.eofF = c->batch_eof;
  T.lmax = c->lmax;
  T.flags = (uint32_t)c->batch_flags;
  T.ximin = *std::min_element(c->h_xi.begin(), c->h_xi.end());
  T.crot = cos(rotpos);
  T.srot = sin(rotpos);
  const uint32_t* sorted = nullptr;
  const float4* pts = nullptr;
  rc = order_points(c, T, x, y, z, n, s, nullptr, c->batch_off, nsnap, &sorted, &pts, offsets);
  if (rc) return rc;
  // results go through a float4 per point, split coalesced (as field_eval_run)
  rc = ensure_scratch(c, (size_t)n * sizeof(float4));
  if (rc) return rc;
  float4* quad = (float4*)c->scratch;
  hipLaunchKernelGGL(field_eval_batch_kernel, dim3(xcd_grid(nblocks256(n))), dim3(256), 0, s, n,
                     pts, sorted, order_cell_count(T, nsnap), T, c->batch_sl, (int64_t)slf, c->batch_eof,
                     (int64_t)eoff, fx, fy, fz, pot, quad);
  BFE_HIP(c, hipGetLastError());
  hipLaunchKernelGGL(quad_split_kernel, dim3(nblocks256(n)), dim3(256), 0, s, quad, n, fx, fy, fz,
                     pot);
  BFE_HIP(c, hipGetLastError());
  return 0;
}
