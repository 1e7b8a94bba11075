// Learned CLOUDSC surrogate and the hybrid dispatcher (declared in include/cloudsc_surrogate.h).
//
// The surrogate maps one column's CLOUDSC inputs (14 features x KLEV) to its main outputs (6 targets x KLEV) with
// the BF16 MLP of mlp.hip.  Feature and target matrices are built directly from the IFS blocked fields
// (NPROMA, KLEV[,n], NGPBLKS) through LDS-tiled transposes, so that both the blocked reads and the row-major
// matrix writes are coalesced.  The hybrid entry reruns a seeded random subset of columns, and every column its
// gate flags, through the plain kernel: those columns are gathered into a compact blocked field set and run by
// cloudsc_blocked_sp_c's kernel, and the output kernels take them from there.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/cloudsc_surrogate.h"
#include "capi_util.h"
#include "cloudsc_kernel.h"
#include "mlp_internal.h"
#include "synth.h"

namespace cloudsc_gpu {
}

using cloudsc_capi::fail;
using mlp::bf16;
using cloudsc_gpu::KDims;
using cloudsc_gpu::KPtrs;

namespace surr {

constexpr int NF = CLOUDSC_SURR_NFEAT, NT = CLOUDSC_SURR_NTARG;
constexpr int TILE = 64;  // columns x matrix entries per transpose tile
// Standardised features and training targets are clipped to +-CLIP standard deviations: the heavy tails of the
// tendencies (rare columns with values thousands of standard deviations out) would otherwise dominate the loss.
constexpr float CLIP = 10.0f;

inline int pad128(int n) { return (n + 127) / 128 * 128; }
inline int pad256(int n) { return (n + 255) / 256 * 256; }

// Saturation constants (TTHF, fcttre.func.h) for the relative-humidity feature and the gate.
struct Sat {
  float r2es, r3les, r3ies, r4les, r4ies, rtt, rtice, rtwat_rtice_r, retv;
};

struct Dims {
  int ngptot, nproma, klev, ngpblks;
  Sat th;
};

// Saturation specific humidity over the mixed phase, FOEEWM / p limited to 0.5 (fcttre.func.h, cloudsc.F90:1087).
__device__ __forceinline__ float qsat_mix(const Sat& c, float t, float pap) {
  const float x = (fmaxf(c.rtice, fminf(c.rtt, t)) - c.rtice) * c.rtwat_rtice_r;
  const float alfa = fminf(1.0f, x * x);
  const float es = c.r2es * (alfa * expf(c.r3les * (t - c.rtt) / (t - c.r4les)) +
                             (1.0f - alfa) * expf(c.r3ies * (t - c.rtt) / (t - c.r4ies)));
  const float e = fminf(es / pap, 0.5f);
  return e / (1.0f - c.retv * e);
}

// A column's place in the blocked fields: first element of its block in a (NPROMA, L, NGPBLKS) array is blk * L * NPROMA.
struct Col {
  size_t blk;
  int jl;
};
__device__ __forceinline__ Col column(int c, int nproma) {
  const int b = c / nproma;
  return Col{(size_t)b, c - b * nproma};
}
// Element (column, level k) of a (NPROMA, L, n, NGPBLKS) field, species s.
__device__ __forceinline__ size_t fidx(const Col& c, int k, int s, int n, int L, int nproma) {
  return ((c.blk * n + s) * L + k) * nproma + c.jl;
}

__device__ __forceinline__ float slog(float x) { return log10f(fmaxf(x, 0.0f) + 1e-10f); }

// Where the first word of a feature or target is: level k of species s of a (NPROMA, L, n, NGPBLKS) array.
struct Src {
  const float* p;
  int s, n, k, L;
};
// Selects, no branches: f and t are uniform over a wave.
__device__ __forceinline__ Src feature_src(const KPtrs<float>& p, int f, int k, int L) {
  const bool cld = f >= 3 && f <= 6, tend = f == 10 || f == 11;
  const float* q = p.plude;                 // 13
  q = f == 0 ? p.pt : q;
  q = f == 1 || f == 12 ? p.pq : q;         // 12: relative humidity, with T and PAP of the same place
  q = f == 2 ? p.pa : q;
  q = cld ? p.pclv : q;
  q = f == 7 ? p.tcml_t : q;
  q = f == 8 ? p.tcml_q : q;
  q = f == 9 ? p.tcml_a : q;
  q = tend ? p.tcml_cld : q;
  return Src{q, cld ? f - 3 : (tend ? f - 10 : 0), cld || tend ? 5 : 1, k, L};
}
__device__ __forceinline__ Src target_src(const KPtrs<float>& p, int t, int k, int L) {
  const bool cld = t == 3 || t == 4;
  const float* q = p.pfplsl;                // 5: with PFPLSN of the same place
  q = t == 0 ? p.tloc_t : q;
  q = t == 1 ? p.tloc_q : q;
  q = t == 2 ? p.tloc_a : q;
  q = cld ? p.tloc_cld : q;
  return Src{q, cld ? t - 3 : 0, cld ? 5 : 1, t == 5 ? k + 1 : k, t == 5 ? L + 1 : L};
}
__device__ __forceinline__ float load(const Src& s, const Col& c, int np) { return s.p[fidx(c, s.k, s.s, s.n, s.L, np)]; }

// Raw feature f from its words: a, and for the relative humidity T and PAP in b and c.
__device__ __forceinline__ float feature_value(const Dims& d, int f, float a, float b, float c) {
  if (f == 12) return a / qsat_mix(d.th, b, c);  // relative humidity over the mixed phase
  if ((f >= 3 && f <= 6) || f == 13) return slog(a);
  return a;
}
__device__ __forceinline__ float feature(const KPtrs<float>& p, const Dims& d, int col, int f, int k) {
  const Col c = column(col, d.nproma);
  Src s = feature_src(p, f, k, d.klev);
  const float a = load(s, c, d.nproma);
  float t = 0.0f, pap = 1.0f;
  if (f == 12) {
    s.p = p.pt;
    t = load(s, c, d.nproma);
    s.p = p.pap;
    pap = load(s, c, d.nproma);
  }
  return feature_value(d, f, a, t, pap);
}
// Raw target t at level k of a column (outputs of the plain kernel).
__device__ __forceinline__ float target(const KPtrs<float>& p, const Dims& d, int col, int t, int k) {
  const Col c = column(col, d.nproma);
  Src s = target_src(p, t, k, d.klev);
  const float a = load(s, c, d.nproma);
  if (t < 5) return a;
  s.p = p.pfplsn;
  return a + load(s, c, d.nproma);
}

// The two transposes from the blocked fields into row-major matrices: 256 lanes, a tile of 64 columns x 64 matrix entries
// through LDS; columns beyond NGPTOT and padding entries are 0.  Each wave takes 16 entries with its lanes over the
// columns; the entry (quantity and level) is uniform over the wave.  A kernel of loads and few operations: the words of
// 16 entries are in flight together, which needs the array of an entry chosen as a scalar address ahead of one load
// (a load in each branch of the choice waits for its data where the branches meet), and from entry to entry only the
// offset moves on (a division and a 64-bit product per entry cost more than the loads).  Features of 65,536 columns x
// L137 (720 MB): 366 -> 224 us; with 16-byte stores of the matrix, in another run, 234 -> 217, and with non-temporal
// loads 200 (3.6 TB/s); of 4,096 columns 21.7 -> 20.5 us.  Targets of 4,096 columns 21 -> 12 us.
constexpr int ENT = 16;

// Feature matrix X [M x nin] (bf16, standardised) for columns col0 .. col0+M-1.  NT: the loads carry the non-temporal hint
// (the rule stands at launch_features_rows).
template <bool NT>
__global__ __launch_bounds__(256) void features(KPtrs<float> p, Dims d, int col0, int M, int nin,
                                                const float* __restrict__ mu, const float* __restrict__ rsd,
                                                bf16* __restrict__ X) {
  __shared__ float tile[TILE][TILE + 1];
  const int c0 = blockIdx.x * TILE, e0 = blockIdx.y * TILE;
  const int tx = threadIdx.x & 63, ty = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int L = d.klev, np = d.nproma, nfk = NF * L;
  const bool live = c0 + tx < M && col0 + c0 + tx < d.ngptot;
  const Col c = column(live ? col0 + c0 + tx : 0, np);
  const int eb = e0 + ENT * ty, f0 = min(eb / L, NF - 1), k0 = eb - f0 * L;
  float a[ENT], t[ENT], pap[ENT];
  {
    int f = f0, k = min(k0, L - 1);  // entries past the last repeat its level
    Src s = feature_src(p, f, k, L);
    size_t o = fidx(c, k, s.s, s.n, L, np);
#pragma unroll
    for (int i = 0; i < ENT; ++i) {
      a[i] = NT ? __builtin_nontemporal_load(s.p + o) : s.p[o];
      t[i] = pap[i] = 0.0f;
      if (k + 1 < L) {
        ++k;
        o += np;
      } else if (f + 1 < NF) {
        k = 0;
        s = feature_src(p, ++f, 0, L);
        o = fidx(c, 0, s.s, s.n, L, np);
      }
    }
  }
  if (eb < 13 * L && eb + ENT > 12 * L) {  // relative humidity among the entries
#pragma unroll
    for (int i = 0; i < ENT; ++i) {
      const size_t o = fidx(c, min(max(eb + i - 12 * L, 0), L - 1), 0, 1, L, np);
      t[i] = p.pt[o];
      pap[i] = p.pap[o];
    }
  }
  int f = f0, k = k0;
#pragma unroll
  for (int i = 0; i < ENT; ++i) {
    const int e = eb + i;
    float v = 0.0f;
    if (e < nfk && live) v = fminf(fmaxf((feature_value(d, f, a[i], t[i], pap[i]) - mu[e]) * rsd[e], -CLIP), CLIP);
    tile[ENT * ty + i][tx] = v;
    if (++k == L) {
      k = 0;
      ++f;
    }
  }
  __syncthreads();
  typedef bf16 __attribute__((ext_vector_type(8))) bf16x8;
  const int q = 8 * (tx & 7), e = e0 + q;  // write X rows: 8 lanes x 8 entries to each (nin is a multiple of 128)
#pragma unroll
  for (int i = 8 * ty + (tx >> 3); i < TILE; i += 32) {
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (bf16)tile[q + j][i];
    if (c0 + i < M && e < nin) *reinterpret_cast<bf16x8*>(X + (size_t)(c0 + i) * nin + e) = v;
  }
}

// Target matrix T [M x nout] (fp32, standardised) for columns col0 .. col0+M-1.
__global__ __launch_bounds__(256) void targets(KPtrs<float> p, Dims d, int col0, int M, int nout,
                                               const float* __restrict__ mu, const float* __restrict__ rsd,
                                               float* __restrict__ T) {
  __shared__ float tile[TILE][TILE + 1];
  const int c0 = blockIdx.x * TILE, e0 = blockIdx.y * TILE;
  const int tx = threadIdx.x & 63, ty = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int L = d.klev, np = d.nproma, ntk = NT * L;
  const bool live = c0 + tx < M && col0 + c0 + tx < d.ngptot;
  const Col c = column(live ? col0 + c0 + tx : 0, np);
  const int eb = e0 + ENT * ty, t0 = min(eb / L, NT - 1), k0 = eb - t0 * L;
  float a[ENT], b[ENT];
  {
    int t = t0, k = min(k0, L - 1);
    Src s = target_src(p, t, k, L);
    size_t o = fidx(c, s.k, s.s, s.n, s.L, np);
#pragma unroll
    for (int i = 0; i < ENT; ++i) {
      a[i] = s.p[o];
      b[i] = 0.0f;
      if (k + 1 < L) {
        ++k;
        o += np;
      } else if (t + 1 < NT) {
        k = 0;
        s = target_src(p, ++t, 0, L);
        o = fidx(c, s.k, s.s, s.n, s.L, np);
      }
    }
  }
  if (eb + ENT > 5 * L) {  // precipitation flux among the entries
#pragma unroll
    for (int i = 0; i < ENT; ++i) b[i] = p.pfplsn[fidx(c, min(max(eb + i - 5 * L, 0), L - 1) + 1, 0, 1, L + 1, np)];
  }
#pragma unroll
  for (int i = 0; i < ENT; ++i) {
    const int e = eb + i;
    float v = 0.0f;
    if (e < ntk && live) {
      const float raw = e < 5 * L ? a[i] : a[i] + b[i];
      v = fminf(fmaxf((raw - mu[e]) * rsd[e], -CLIP), CLIP);
    }
    tile[ENT * ty + i][tx] = v;
  }
  __syncthreads();
#pragma unroll 4
  for (int i = ty; i < TILE; i += 4) {
    const int c = c0 + i, e = e0 + tx;
    if (c < M && e < nout) T[(size_t)c * nout + e] = tile[tx][i];
  }
}

// Where a tendency goes: as Src, t = 0 .. 4.
struct Dst {
  float* p;
  int s, n;
};
__device__ __forceinline__ Dst tendency_dst(const KPtrs<float>& p, int t) {
  float* q = p.tloc_cld;
  q = t == 0 ? p.tloc_t : q;
  q = t == 1 ? p.tloc_q : q;
  q = t == 2 ? p.tloc_a : q;
  return Dst{q, t >= 3 ? t - 3 : 0, t >= 3 ? 5 : 1};
}

constexpr int NP_C = 128;  // NPROMA of the compact field set of the hybrid entry

// Network output Y [M x nout] (standardised) -> tendencies and precipitation fluxes of columns col0 .. col0+M-1, by the
// transpose of `features` the other way.  MERGE: a column with rank[column] >= 0 takes that column of the compact field
// set pc (the plain kernel's results) instead.  Writing the plain results over the network's afterwards touched every
// line a rerun column is in a second time, for 4 of its bytes: 780 us for 3 % of 262,144 columns x L137.  65,536 columns
// (630 MB): 146 us; with the diagnostics below, 11 of the 22 fields written, stored per entry here, 285 us.
template <bool MERGE>
__global__ __launch_bounds__(256) void outputs(KPtrs<float> p, KPtrs<float> pc, const int* __restrict__ rank, Dims d,
                                               int col0, int M, int nout, const float* __restrict__ mu,
                                               const float* __restrict__ sd, const float* __restrict__ Y, float rtt,
                                               float rlvtt, float rlstt) {
  __shared__ float tile[TILE][TILE + 1];
  const int c0 = blockIdx.x * TILE, e0 = blockIdx.y * TILE;
  const int tx = threadIdx.x & 63, ty = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int L = d.klev, np = d.nproma, ntk = NT * L;
  {
    const int e = min(e0 + tx, ntk - 1);
    const float s = sd[e], m = mu[e];
    float y[ENT];
#pragma unroll
    for (int i = 0; i < ENT; ++i) y[i] = Y[(size_t)min(c0 + ENT * ty + i, M - 1) * nout + e];  // lanes over entries
#pragma unroll
    for (int i = 0; i < ENT; ++i) tile[tx][ENT * ty + i] = y[i] * s + m;
  }
  __syncthreads();
  const int eb = e0 + ENT * ty, col = col0 + c0 + tx;
  if (eb >= ntk || c0 + tx >= M || col >= d.ngptot) return;
  const Col c = column(col, np);
  const int r = MERGE ? rank[col] : -1;
  const Col q = column(r < 0 ? 0 : r, NP_C);
  float v[ENT];
#pragma unroll
  for (int i = 0; i < ENT; ++i) v[i] = tile[ENT * ty + i][tx];
  if (eb < 5 * L) {  // tendencies
    const int t0 = eb / L, k0 = eb - t0 * L;
    float w[ENT];  // rain and snow, which the network does not predict, go with cloud liquid and ice
#pragma unroll
    for (int i = 0; i < ENT; ++i) w[i] = 0.0f;
    if (MERGE && r >= 0) {
      int t = t0, k = k0;
      Dst x = tendency_dst(pc, t);
      size_t o = fidx(q, k, x.s, x.n, L, NP_C);
#pragma unroll
      for (int i = 0; i < ENT; ++i) {
        if (eb + i < 5 * L) {
          v[i] = x.p[o];
          if (t >= 3) w[i] = x.p[o + (size_t)2 * L * NP_C];
        }
        if (k + 1 < L) {
          ++k;
          o += NP_C;
        } else if (t + 1 < 5) {
          k = 0;
          x = tendency_dst(pc, ++t);
          o = fidx(q, 0, x.s, x.n, L, NP_C);
        }
      }
    }
    int t = t0, k = k0;
    Dst x = tendency_dst(p, t);
    size_t o = fidx(c, k, x.s, x.n, L, np);
#pragma unroll
    for (int i = 0; i < ENT; ++i) {
      if (eb + i < 5 * L) {
        x.p[o] = v[i];
        if (t >= 3) x.p[o + (size_t)2 * L * np] = w[i];
      }
      if (k + 1 < L) {
        ++k;
        o += np;
      } else if (t + 1 < 5) {
        k = 0;
        x = tendency_dst(p, ++t);
        o = fidx(c, 0, x.s, x.n, L, np);
      }
    }
  }
  if (eb + ENT > 5 * L) {  // precipitation at the lower half level, as rain above freezing, else as snow
    const int kb = eb - 5 * L;
    float t[ENT], hl[ENT], hs[ENT], fs[ENT], top[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < ENT; ++i) t[i] = p.pt[fidx(c, min(max(kb + i, 0), L - 1), 0, 1, L, np)];
#pragma unroll
    for (int i = 0; i < ENT; ++i) {
      const float pr = fmaxf(v[i], 0.0f);
      const bool liquid = t[i] > rtt;
      v[i] = liquid ? pr : 0.0f;
      fs[i] = liquid ? 0.0f : pr;
      hl[i] = -rlvtt * v[i];
      hs[i] = -rlstt * fs[i];
    }
    if (MERGE && r >= 0) {
#pragma unroll
      for (int i = 0; i < ENT; ++i) {
        const size_t h = fidx(q, min(max(kb + i, 0), L - 1) + 1, 0, 1, L + 1, NP_C);
        v[i] = pc.pfplsl[h];
        fs[i] = pc.pfplsn[h];
        hl[i] = pc.pfhpsl[h];
        hs[i] = pc.pfhpsn[h];
      }
      const size_t h = fidx(q, 0, 0, 1, L + 1, NP_C);
      top[0] = pc.pfplsl[h];
      top[1] = pc.pfplsn[h];
      top[2] = pc.pfhpsl[h];
      top[3] = pc.pfhpsn[h];
    }
    auto store = [&](int k, float a, float b, float e, float f) {
      const size_t h = fidx(c, k, 0, 1, L + 1, np);
      p.pfplsl[h] = a;
      p.pfplsn[h] = b;
      p.pfhpsl[h] = e;
      p.pfhpsn[h] = f;
    };
#pragma unroll
    for (int i = 0; i < ENT; ++i)
      if (kb + i >= 0 && kb + i < L) store(kb + i + 1, v[i], fs[i], hl[i], hs[i]);
    if (kb <= 0) store(0, top[0], top[1], top[2], top[3]);
  }
}

// The outputs that the network does not predict: 0 (MERGE: or the compact set's, as above) in the ten flux diagnostics,
// in PCOVPTOT from NCLDTOP on (the plain kernel's write set) and in PRAINFRAC_TOPRFZ.  A lane takes W consecutive columns
// (4 where NPROMA and the arrays' addresses allow 16-byte stores) of array blockIdx.y over LEV levels, 8 at a time, so
// that a rerun column's words are in flight together.  1.6 GB for 262,144 columns: 329 us with 3 % of them merged.
constexpr int LEV = 32;
template <bool MERGE, int W>
__global__ __launch_bounds__(256) void diagnostics(KPtrs<float> p, KPtrs<float> pc, const int* __restrict__ rank, Dims d,
                                                   int ncldtop) {
  const int a = blockIdx.y, np = d.nproma;
  auto array = [&](const KPtrs<float>& g) {
    float* q = g.prainfrac_toprfz;  // 11
    q = a == 0 ? g.pfsqlf : q;
    q = a == 1 ? g.pfsqif : q;
    q = a == 2 ? g.pfcqnng : q;
    q = a == 3 ? g.pfcqlng : q;
    q = a == 4 ? g.pfsqrf : q;
    q = a == 5 ? g.pfsqsf : q;
    q = a == 6 ? g.pfcqrng : q;
    q = a == 7 ? g.pfcqsng : q;
    q = a == 8 ? g.pfsqltur : q;
    q = a == 9 ? g.pfsqitur : q;
    q = a == 10 ? g.pcovptot : q;
    return q;
  };
  const int R = a < 10 ? d.klev + 1 : (a == 10 ? d.klev : 1);  // levels
  const int klo = a == 10 ? ncldtop - 1 : 0;
  const int k0 = max(klo, (int)blockIdx.z * LEV), k1 = min(R, (int)(blockIdx.z + 1) * LEV);
  const int col = (blockIdx.x * 256 + threadIdx.x) * W;
  if (col >= d.ngptot) return;
  const int live = min(W, d.ngptot - col);
  const Col c = column(col, np);
  float* out = array(p) + c.blk * R * np + c.jl;
  int r[W];
  bool any = false;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    r[i] = MERGE && i < live ? rank[col + i] : -1;
    any |= r[i] >= 0;
  }
  const float* comp = array(pc);
  constexpr int U = 8;
  for (int k = k0; k < k1; k += U) {
    typedef float fw __attribute__((ext_vector_type(W)));
    float v[U][W] = {};
    if (MERGE && any) {
#pragma unroll
      for (int i = 0; i < W; ++i)
        if (r[i] >= 0) {
          const Col q = column(r[i], NP_C);
#pragma unroll
          for (int u = 0; u < U; ++u) v[u][i] = comp[fidx(q, min(k + u, R - 1), 0, 1, R, NP_C)];
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k + u >= k1) break;
      float* o = out + (size_t)(k + u) * np;
      if (live == W) {
        fw x;
#pragma unroll
        for (int i = 0; i < W; ++i) x[i] = v[u][i];
        *reinterpret_cast<fw*>(o) = x;
      } else {
        for (int i = 0; i < live; ++i) o[i] = v[u][i];
      }
    }
  }
}

// Mean and standard deviation over all columns of raw feature (kind 0) or target (kind 1) entry e = blockIdx.x.
__global__ __launch_bounds__(256) void moments(KPtrs<float> p, Dims d, int kind, float* __restrict__ mu,
                                               float* __restrict__ sd) {
  const int e = blockIdx.x, k = e % d.klev, f = e / d.klev;
  double s = 0.0, s2 = 0.0;
  for (int c = threadIdx.x; c < d.ngptot; c += 256) {
    const double v = kind == 0 ? feature(p, d, c, f, k) : target(p, d, c, f, k);
    s += v;
    s2 += v * v;
  }
  __shared__ double r1[256], r2[256];
  r1[threadIdx.x] = s;
  r2[threadIdx.x] = s2;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      r1[threadIdx.x] += r1[threadIdx.x + h];
      r2[threadIdx.x] += r2[threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double m = r1[0] / d.ngptot;
    const double var = std::max(r2[0] / d.ngptot - m * m, 0.0);
    mu[e] = (float)m;
    sd[e] = (float)std::sqrt(var);  // raw; floors are applied on the host (cloudsc_surrogate_fit_norm)
  }
}

__global__ void reciprocal(const float* __restrict__ a, float* __restrict__ r, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) r[i] = 1.0f / a[i];
}

__global__ void add_scalar(float* __restrict__ acc, const float* __restrict__ x) {
  if (threadIdx.x == 0 && blockIdx.x == 0) acc[0] += x[0];
}

// PRAINFRAC_TOPRFZ is zeroed for all KLON columns of every block, the padding of the last block included
// (cloudsc.F90:1010); the network path writes the active columns in `diagnostics`.
__global__ void zero_padding_columns(float* __restrict__ prainfrac, int ngptot, int ntotal) {
  const int c = ngptot + blockIdx.x * blockDim.x + threadIdx.x;
  if (c < ntotal) prainfrac[c] = 0.0f;
}

__global__ void fill_f32(float* p, float v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) p[0] = v;
}

// Gate score and rerun selection (262,144 columns x L137, 430 MB: 169 us loading q and p only below 238 K, one level at a
// time; 105 us with 8 levels' words in flight).  Score: max over levels with T < 238 K of q / qsat_mix (FOEEWM with FOEALFA,
// fcttre.func.h).  With flags, each column's selection (seeded 1 % draw or score above the threshold) is stored and
// each group of 256 columns writes how many it selected, for the compaction below.
__global__ __launch_bounds__(256) void select_columns(KPtrs<float> p, Dims d, float frac, uint64_t seed, float thr,
                                                      float* __restrict__ score, uint8_t* __restrict__ flags,
                                                      int* __restrict__ group_counts) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  bool sel = false;
  if (c < d.ngptot) {
    float sc = 0.0f;
    const Col col = column(c, d.nproma);
    size_t o = fidx(col, 0, 0, 1, d.klev, d.nproma);
    auto level = [&](float t, float q, float pap) {
      if (t < 238.0f) sc = fmaxf(sc, q / qsat_mix(d.th, t, pap));
    };
    int k = 0;
    for (; k + 8 <= d.klev; k += 8) {  // the words of 8 levels in flight
      float t[8], q[8], pap[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        t[i] = p.pt[o + (size_t)i * d.nproma];
        q[i] = p.pq[o + (size_t)i * d.nproma];
        pap[i] = p.pap[o + (size_t)i * d.nproma];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) level(t[i], q[i], pap[i]);
      o += (size_t)8 * d.nproma;
    }
    for (; k < d.klev; ++k, o += d.nproma) level(p.pt[o], p.pq[o], p.pap[o]);
    if (score) score[c] = sc;
    if (flags) {
      const synth::Draw u = synth::draw(seed, 0x52455255u /* "RERU" */, (uint32_t)c, 0u);
      sel = u.u0 < (double)frac || sc > thr;
      flags[c] = sel ? 1 : 0;
    }
  }
  if (!flags) return;
  __shared__ int wcount[4];
  const uint64_t b = __ballot(sel);
  if ((threadIdx.x & 63) == 0) wcount[threadIdx.x >> 6] = __popcll(b);
  __syncthreads();
  if (threadIdx.x == 0) group_counts[blockIdx.x] = wcount[0] + wcount[1] + wcount[2] + wcount[3];
}

// Exclusive prefix sum of the n group counts in place (one group of 1024 lanes); *total = their sum.
__global__ __launch_bounds__(1024) void scan_counts(int* __restrict__ counts, int n, int* __restrict__ total) {
  __shared__ int part[1024];
  const int t = threadIdx.x, per = (n + 1023) / 1024, lo = min(n, t * per), hi = min(n, lo + per);
  int sum = 0;
  for (int i = lo; i < hi; ++i) sum += counts[i];
  part[t] = sum;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {  // inclusive scan of the per-lane sums
    const int v = t >= off ? part[t - off] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int run = part[t] - sum;  // exclusive start of this lane's range
  for (int i = lo; i < hi; ++i) {
    const int ci = counts[i];
    counts[i] = run;
    run += ci;
  }
  if (t == 1023) *total = part[1023];
}

// The selected columns in ascending order: list[offset of the group + rank within it] = column, and that place by
// column (-1: not selected).  Ascending order
// keeps neighbouring lanes of the gather and scatter on neighbouring blocks of the fields.
__global__ __launch_bounds__(256) void compact_columns(const uint8_t* __restrict__ flags, const int* __restrict__ offsets,
                                                       int ngptot, int* __restrict__ list, int* __restrict__ rank_of) {
  const int c = blockIdx.x * 256 + threadIdx.x, w = threadIdx.x >> 6;
  const bool sel = c < ngptot && flags[c];
  const uint64_t b = __ballot(sel);
  __shared__ int wcount[4];
  if ((threadIdx.x & 63) == 0) wcount[w] = __popcll(b);
  __syncthreads();
  int base = offsets[blockIdx.x];
  for (int i = 0; i < w; ++i) base += wcount[i];
  const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0));
  if (sel) list[base + rank] = c;
  if (c < ngptot) rank_of[c] = sel ? base + rank : -1;
}

// Column copies between a blocked field set (NPROMA = np_full) and a compact one (NPROMA = np_c), for one
// 2-D slice (NPROMA, L) of each array: element (column, level) at blk*stride + off + level*NPROMA + jl.
struct Slice {
  uint32_t* full;
  uint32_t* comp;
  long full_stride, comp_stride;  // elements per block
  long full_off, comp_off;
  int L;
};
constexpr int MAX_SLICES = 64;
struct Slices {
  Slice s[MAX_SLICES];
  int n;
};

__global__ __launch_bounds__(256) void copy_columns(Slices sl, const int* __restrict__ list, int nsel, int np_full,
                                                    int np_c, int to_compact) {
  const Slice S = sl.s[blockIdx.y];
  const long total = (long)nsel * S.L;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long)gridDim.x * 256) {
    const int j = (int)(i % nsel), lev = (int)(i / nsel);
    const int c = list[j];
    const int bf = c / np_full, jf = c - bf * np_full;
    const int bc = j / np_c, jc = j - bc * np_c;
    uint32_t* f = S.full + bf * S.full_stride + S.full_off + (long)lev * np_full + jf;
    uint32_t* q = S.comp + bc * S.comp_stride + S.comp_off + (long)lev * np_c + jc;
    if (to_compact)
      *q = *f;
    else
      *f = *q;
  }
}

}  // namespace surr

// ---------------------------------------------------------------------------------------------------------
struct cloudsc_surrogate {
  cloudsc_mlp* net = nullptr;
  int klev = 0, nin = 0, nout = 0, max_batch = 0;
  float *mu_x = nullptr, *sd_x = nullptr, *rsd_x = nullptr, *mu_y = nullptr, *sd_y = nullptr, *rsd_y = nullptr;
  float* wgt = nullptr;  // per output entry: 1 for the 6*KLEV targets, 0 for padding
  bf16* X = nullptr;
  float *T = nullptr, *Y = nullptr, *loss_acc = nullptr;
  // hybrid: selection list and the compact field set
  int* list = nullptr;
  int* count = nullptr;
  int list_cap = 0;
  int* count_host = nullptr;  // pinned
  hipEvent_t counted = nullptr, joined = nullptr;
  hipStream_t side = nullptr;  // the rerun columns, beside the network's first batch
  void* comp = nullptr;
  size_t comp_bytes = 0;
  std::vector<void*> allocs;
};

namespace {

int salloc(cloudsc_surrogate* s, size_t bytes, void** p) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) return fail(CLOUDSC_ENOMEM, "cloudsc_surrogate: hipMalloc", e);
  s->allocs.push_back(*p);
  return CLOUDSC_OK;
}

int check_fields(const cloudsc_surrogate* s, const cloudsc_params_t* q, int ngptot, int nproma, int klev,
                 int ngpblks, const KPtrs<float>& p) {
  if (!s || !q) return fail(CLOUDSC_ENULL, "cloudsc_surrogate: NULL object or parameters");
  const int rc = cloudsc_capi::check_config(q);  // the plain kernel reruns columns: the same switches apply
  if (rc) return rc;
  if (klev != s->klev) return fail(CLOUDSC_EDIMS, "cloudsc_surrogate: KLEV differs from the surrogate's");
  if (nproma < 1 || ngptot < 1 || ngpblks != (ngptot + nproma - 1) / nproma)
    return fail(CLOUDSC_EDIMS, "cloudsc_surrogate: need NGPBLKS = ceil(NGPTOT/NPROMA)");
  const void* req[] = {p.pt, p.pq, p.tcml_t, p.tcml_q, p.tcml_a, p.tcml_cld, p.tloc_t, p.tloc_q, p.tloc_a,
                       p.tloc_cld, p.pap, p.paph, p.plude, p.pa, p.pclv, p.pcovptot, p.prainfrac_toprfz,
                       p.pfplsl, p.pfplsn, p.pfhpsl, p.pfhpsn, p.pfsqlf, p.pfsqif, p.pfcqnng, p.pfcqlng,
                       p.pfsqrf, p.pfsqsf, p.pfcqrng, p.pfcqsng, p.pfsqltur, p.pfsqitur};
  for (const void* x : req)
    if (!x) return fail(CLOUDSC_ENULL, "cloudsc_surrogate: NULL array");
  return CLOUDSC_OK;
}

inline unsigned nblk(long n, int b) { return (unsigned)((n + b - 1) / b); }

surr::Sat sat_consts(const cloudsc_params_t* q) {
  if (!q) return surr::Sat{};
  return surr::Sat{(float)q->r2es, (float)q->r3les, (float)q->r3ies, (float)q->r4les, (float)q->r4ies,
                   (float)q->rtt,  (float)q->rtice, (float)q->rtwat_rtice_r, (float)q->retv};
}

// The loads of the features carry the non-temporal hint for the batches of 8,192 columns or more whose rows are whole
// lines (NPROMA a multiple of 64): prediction for 16,384 columns 159 -> 149 us, for 50,000 607 -> 579, for 131,072
// 2,074 -> 2,055.  Smaller batches can leave the state in the caches for the next call (4,096 columns 55 -> 56 us,
// training in batches of 1,024 slower by 1.5 %); a line of a ragged row is read by two waves (no gain with NPROMA 75 and
// 100); and the first batch of a hybrid call is gathered from right after (60,000 columns 980 -> 993 us): `reread`.
void launch_features_rows(cloudsc_surrogate* s, const KPtrs<float>& p, const surr::Dims& d, int c0, int M,
                          bool reread, hipStream_t st) {
  auto* kernel = !reread && d.nproma % 64 == 0 && M >= 8192 ? surr::features<true> : surr::features<false>;
  hipLaunchKernelGGL(kernel, dim3(nblk(M, surr::TILE), nblk(s->nin, surr::TILE)), dim3(256), 0, st, p, d, c0, M,
                     s->nin, s->mu_x, s->rsd_x, s->X);
}

void launch_features(cloudsc_surrogate* s, const KPtrs<float>& p, const surr::Dims& d, int c0, bool reread,
                     hipStream_t st) {
  launch_features_rows(s, p, d, c0, surr::pad128(std::min(s->max_batch, d.ngptot - c0)), reread, st);
}

// Network prediction for all columns, in batches of max_batch, the first of whose features are already there; with rank,
// columns of rank >= 0 are taken from the compact field set pc instead, which is complete at the event `ready`.
hipError_t predict(cloudsc_surrogate* s, const cloudsc_params_t* q, const KPtrs<float>& p, const surr::Dims& d,
                   const KPtrs<float>& pc, const int* rank, hipEvent_t ready, hipStream_t st) {
  hipError_t e = hipSuccess;
  const int ntotal = d.ngpblks * d.nproma;
  if (ntotal > d.ngptot)
    hipLaunchKernelGGL(surr::zero_padding_columns, dim3(nblk(ntotal - d.ngptot, 256)), dim3(256), 0, st,
                       p.prainfrac_toprfz, d.ngptot, ntotal);
  uintptr_t bits = (uintptr_t)d.nproma * 4;
  for (const float* x : {p.pfsqlf, p.pfsqif, p.pfcqnng, p.pfcqlng, p.pfsqrf, p.pfsqsf, p.pfcqrng, p.pfcqsng, p.pfsqltur,
                         p.pfsqitur, p.pcovptot, p.prainfrac_toprfz})
    bits |= (uintptr_t)x;
  const bool vec = bits % 16 == 0;
  auto* diag = rank ? (vec ? surr::diagnostics<true, 4> : surr::diagnostics<true, 1>)
                    : (vec ? surr::diagnostics<false, 4> : surr::diagnostics<false, 1>);
  for (int c0 = 0; c0 < d.ngptot && e == hipSuccess; c0 += s->max_batch) {
    const int n = std::min(s->max_batch, d.ngptot - c0);
    if (c0 > 0) launch_features(s, p, d, c0, false, st);
    e = mlp::forward(s->net, s->X, surr::pad128(n), s->Y, nullptr, nullptr, st);
    if (e == hipSuccess && c0 == 0 && ready) e = hipStreamWaitEvent(st, ready, 0);
    if (e != hipSuccess) break;
    hipLaunchKernelGGL(rank ? surr::outputs<true> : surr::outputs<false>,
                       dim3(nblk(n, surr::TILE), nblk(surr::NT * d.klev, surr::TILE)), dim3(256), 0, st, p, pc, rank, d,
                       c0, n, s->nout, s->mu_y, s->sd_y, s->Y, (float)q->rtt, (float)q->rlvtt, (float)q->rlstt);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(diag, dim3(nblk(d.ngptot, vec ? 1024 : 256), 12, nblk(d.klev + 1, surr::LEV)), dim3(256), 0, st, p,
                     pc, rank, d, q->ncldtop);
  return hipGetLastError();
}

}  // namespace

#define SURR_PTRS                                                                                                 \
  KPtrs<float> p;                                                                                                 \
  p.pt = pt; p.pq = pq; p.tcml_t = ptendency_cml_t; p.tcml_q = ptendency_cml_q; p.tcml_a = ptendency_cml_a;       \
  p.tcml_cld = ptendency_cml_cld; p.tloc_t = ptendency_loc_t; p.tloc_q = ptendency_loc_q;                         \
  p.tloc_a = ptendency_loc_a; p.tloc_cld = ptendency_loc_cld; p.pvfl = pvfl; p.pvfi = pvfi; p.pap = pap;          \
  p.paph = paph; p.plsm = plsm; p.ldcum = ldcum; p.ktype = ktype; p.peis = peis; p.plu = plu; p.plude = plude;    \
  p.pludeli = pludeli; p.psnde = psnde; p.pmfu = pmfu; p.pmfd = pmfd; p.pa = pa; p.pclv = pclv;                   \
  p.pcovptot = pcovptot; p.prainfrac_toprfz = prainfrac_toprfz; p.pfsqlf = pfsqlf; p.pfsqif = pfsqif;             \
  p.pfcqnng = pfcqnng; p.pfcqlng = pfcqlng; p.pfsqrf = pfsqrf; p.pfsqsf = pfsqsf; p.pfcqrng = pfcqrng;             \
  p.pfcqsng = pfcqsng; p.pfsqltur = pfsqltur; p.pfsqitur = pfsqitur; p.pfplsl = pfplsl; p.pfplsn = pfplsn;         \
  p.pfhpsl = pfhpsl; p.pfhpsn = pfhpsn;                                                                           \
  const surr::Dims d{ngptot, nproma, klev, ngpblks, sat_consts(ydparams)};                                                              \
  hipStream_t st = (hipStream_t)stream;                                                                           \
  (void)ptsphy

extern "C" {

int cloudsc_surrogate_create(cloudsc_surrogate_t** out, int klev, int n_hidden, int n_hidden_layers, int max_batch,
                             uint64_t seed) {
  if (!out) return fail(CLOUDSC_ENULL, "cloudsc_surrogate_create: NULL output");
  *out = nullptr;
  if (klev < 2 || max_batch < 128 || max_batch % 128)
    return fail(CLOUDSC_EDIMS, "cloudsc_surrogate_create: KLEV >= 2 and max_batch a positive multiple of 128");
  cloudsc_surrogate* s = new cloudsc_surrogate();
  s->klev = klev;
  s->nin = surr::pad128(surr::NF * klev);
  s->nout = surr::pad256(surr::NT * klev);  // the output product then runs on the 256 x 256-tile GEMM
  s->max_batch = max_batch;
  int rc = cloudsc_mlp_create(&s->net, s->nin, n_hidden, n_hidden_layers, s->nout, max_batch, seed);
  auto F = [&](size_t n, float** p) { return salloc(s, n * sizeof(float), (void**)p); };
  if (!rc)
    rc = F(s->nin, &s->mu_x) || F(s->nin, &s->sd_x) || F(s->nin, &s->rsd_x) || F(s->nout, &s->mu_y) ||
         F(s->nout, &s->sd_y) || F(s->nout, &s->rsd_y) || F(s->nout, &s->wgt) ||
         salloc(s, (size_t)max_batch * s->nin * sizeof(bf16), (void**)&s->X) ||
         F((size_t)max_batch * s->nout, &s->T) || F((size_t)max_batch * s->nout, &s->Y) || F(1, &s->loss_acc) ||
         salloc(s, sizeof(int), (void**)&s->count);
  if (!rc && (hipHostMalloc((void**)&s->count_host, sizeof(int), hipHostMallocDefault) != hipSuccess ||
              hipEventCreateWithFlags(&s->counted, hipEventDisableTiming) != hipSuccess ||
              hipEventCreateWithFlags(&s->joined, hipEventDisableTiming) != hipSuccess ||
              hipStreamCreateWithFlags(&s->side, hipStreamNonBlocking) != hipSuccess))
    rc = fail(CLOUDSC_ENOMEM, "cloudsc_surrogate_create: pinned count, events or stream");
  if (rc) {
    cloudsc_surrogate_destroy(s);
    return rc < 0 ? rc : CLOUDSC_ENOMEM;
  }
  // identity statistics until fitted; unit weights on the real targets
  std::vector<float> zx(s->nin, 0.0f), ox(s->nin, 1.0f), zy(s->nout, 0.0f), oy(s->nout, 1.0f), w(s->nout, 0.0f);
  for (int i = 0; i < surr::NT * klev; ++i) w[i] = 1.0f;
  hipError_t e = hipMemcpy(s->mu_x, zx.data(), s->nin * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(s->sd_x, ox.data(), s->nin * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(s->rsd_x, ox.data(), s->nin * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(s->mu_y, zy.data(), s->nout * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(s->sd_y, oy.data(), s->nout * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(s->rsd_y, oy.data(), s->nout * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(s->wgt, w.data(), s->nout * 4, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    cloudsc_surrogate_destroy(s);
    return fail(CLOUDSC_EHIP, "cloudsc_surrogate_create: initialisation", e);
  }
  *out = s;
  return CLOUDSC_OK;
}

int cloudsc_surrogate_destroy(cloudsc_surrogate_t* s) {
  if (!s) return CLOUDSC_OK;
  cloudsc_mlp_destroy(s->net);
  for (void* p : s->allocs) (void)hipFree(p);
  if (s->list) (void)hipFree(s->list);
  if (s->comp) (void)hipFree(s->comp);
  if (s->count_host) (void)hipHostFree(s->count_host);
  if (s->counted) (void)hipEventDestroy(s->counted);
  if (s->joined) (void)hipEventDestroy(s->joined);
  if (s->side) (void)hipStreamDestroy(s->side);
  delete s;
  return CLOUDSC_OK;
}

cloudsc_mlp_t* cloudsc_surrogate_mlp(cloudsc_surrogate_t* s) { return s ? s->net : nullptr; }

int cloudsc_surrogate_dims(const cloudsc_surrogate_t* s, int* klev, int* n_in, int* n_out, int* max_batch) {
  if (!s) return fail(CLOUDSC_ENULL, "cloudsc_surrogate_dims: NULL object");
  if (klev) *klev = s->klev;
  if (n_in) *n_in = s->nin;
  if (n_out) *n_out = s->nout;
  if (max_batch) *max_batch = s->max_batch;
  return CLOUDSC_OK;
}

int cloudsc_surrogate_norm(cloudsc_surrogate_t* s, float* mu_x, float* sd_x, float* mu_y, float* sd_y, float* wgt_y,
                           int get) {
  if (!s || !mu_x || !sd_x || !mu_y || !sd_y) return fail(CLOUDSC_ENULL, "cloudsc_surrogate_norm: NULL argument");
  const size_t nx = (size_t)surr::NF * s->klev * 4, ny = (size_t)surr::NT * s->klev * 4;
  hipError_t e = hipDeviceSynchronize();
  if (get) {
    if (e == hipSuccess) e = hipMemcpy(mu_x, s->mu_x, nx, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(sd_x, s->sd_x, nx, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(mu_y, s->mu_y, ny, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(sd_y, s->sd_y, ny, hipMemcpyDeviceToHost);
    if (e == hipSuccess && wgt_y) e = hipMemcpy(wgt_y, s->wgt, ny, hipMemcpyDeviceToHost);
  } else {
    if (e == hipSuccess) e = hipMemcpy(s->mu_x, mu_x, nx, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(s->sd_x, sd_x, nx, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(s->mu_y, mu_y, ny, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(s->sd_y, sd_y, ny, hipMemcpyHostToDevice);
    if (e == hipSuccess && wgt_y) e = hipMemcpy(s->wgt, wgt_y, ny, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(surr::reciprocal, dim3(nblk(s->nin, 256)), dim3(256), 0, 0, s->sd_x, s->rsd_x,
                         surr::NF * s->klev);
      hipLaunchKernelGGL(surr::reciprocal, dim3(nblk(s->nout, 256)), dim3(256), 0, 0, s->sd_y, s->rsd_y,
                         surr::NT * s->klev);
      e = hipDeviceSynchronize();
    }
  }
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_surrogate_norm", e);
  return CLOUDSC_OK;
}

int cloudsc_surrogate_fit_norm(cloudsc_surrogate_t* s, CLOUDSC_BLOCKED_ARGS(float)) {
  SURR_PTRS;
  int rc = check_fields(s, ydparams, ngptot, nproma, klev, ngpblks, p);
  if (rc) return rc;
  hipLaunchKernelGGL(surr::moments, dim3(surr::NF * klev), dim3(256), 0, st, p, d, 0, s->mu_x, s->sd_x);
  hipLaunchKernelGGL(surr::moments, dim3(surr::NT * klev), dim3(256), 0, st, p, d, 1, s->mu_y, s->sd_y);
  const int nx = surr::NF * klev, ny = surr::NT * klev;
  std::vector<float> mx(nx), sx(nx), my(ny), sy(ny), w(s->nout, 0.0f);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(mx.data(), s->mu_x, nx * 4, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipMemcpyAsync(sx.data(), s->sd_x, nx * 4, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipMemcpyAsync(my.data(), s->mu_y, ny * 4, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipMemcpyAsync(sy.data(), s->sd_y, ny * 4, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_surrogate_fit_norm", e);
  // Features: constant entries (the model-top pressure, levels without a quantity) are not scaled; the others
  // get at least 1e-3 of their feature's largest level spread.
  for (int f = 0; f < surr::NF; ++f) {
    float top = 0.0f;
    for (int k = 0; k < klev; ++k) top = std::max(top, sx[f * klev + k]);
    for (int k = 0; k < klev; ++k) {
      float& v = sx[f * klev + k];
      v = (v <= 1e-6f * std::fabs(mx[f * klev + k]) || v <= 1e-30f) ? 1.0f : std::max(v, 1e-3f * top);
    }
  }
  // Targets: entries whose spread is below 1e-3 of their target's largest level spread (tendencies above
  // NCLDTOP, levels where a process never acts) are not trained (weight 0) and are predicted at their mean.
  for (int t = 0; t < surr::NT; ++t) {
    float top = 0.0f;
    for (int k = 0; k < klev; ++k) top = std::max(top, sy[t * klev + k]);
    for (int k = 0; k < klev; ++k) {
      float& v = sy[t * klev + k];
      const bool live = top > 0.0f && v > 1e-3f * top;
      w[t * klev + k] = live ? 1.0f : 0.0f;
      v = live ? v : (top > 0.0f ? 1e-3f * top : 1.0f);
    }
  }
  e = hipMemcpyAsync(s->sd_x, sx.data(), nx * 4, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipMemcpyAsync(s->sd_y, sy.data(), ny * 4, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipMemcpyAsync(s->wgt, w.data(), s->nout * 4, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(surr::reciprocal, dim3(nblk(s->nin, 256)), dim3(256), 0, st, s->sd_x, s->rsd_x, nx);
    hipLaunchKernelGGL(surr::reciprocal, dim3(nblk(s->nout, 256)), dim3(256), 0, st, s->sd_y, s->rsd_y, ny);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_surrogate_fit_norm", e);
  return CLOUDSC_OK;
}

int cloudsc_surrogate_train(cloudsc_surrogate_t* s, float lr, int batch, float* loss, CLOUDSC_BLOCKED_ARGS(float)) {
  SURR_PTRS;
  int rc = check_fields(s, ydparams, ngptot, nproma, klev, ngpblks, p);
  if (rc) return rc;
  hipLaunchKernelGGL(surr::fill_f32, dim3(1), dim3(64), 0, st, s->loss_acc, 0.0f);
  if (batch < 128 || batch % 128 || batch > s->max_batch)
    return fail(CLOUDSC_EDIMS, "cloudsc_surrogate_train: batch must be a multiple of 128 and <= max_batch");
  int nb = 0;
  const int M = batch;
  hipError_t e = hipGetLastError();
  for (int c0 = 0; c0 + M <= ngptot && e == hipSuccess; c0 += M, ++nb) {
    launch_features_rows(s, p, d, c0, M, false, st);
    hipLaunchKernelGGL(surr::targets, dim3(nblk(M, surr::TILE), nblk(s->nout, surr::TILE)), dim3(256), 0, st, p, d,
                       c0, M, s->nout, s->mu_y, s->rsd_y, s->T);
    e = hipGetLastError();
    if (e != hipSuccess) break;
    rc = mlp::train_step(s->net, s->X, s->T, s->wgt, M, lr, st);
    if (rc) return rc;
    hipLaunchKernelGGL(surr::add_scalar, dim3(1), dim3(64), 0, st, s->loss_acc, s->net->loss);
    e = hipGetLastError();
  }
  float h = 0.0f;
  if (e == hipSuccess) e = hipMemcpyAsync(&h, s->loss_acc, sizeof(float), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_surrogate_train", e);
  if (loss) *loss = nb ? h / nb : 0.0f;
  return CLOUDSC_OK;
}

int cloudsc_surrogate_predict_sp(cloudsc_surrogate_t* s, CLOUDSC_BLOCKED_ARGS(float)) {
  SURR_PTRS;
  int rc = check_fields(s, ydparams, ngptot, nproma, klev, ngpblks, p);
  if (rc) return rc;
  launch_features(s, p, d, 0, false, st);
  hipError_t e = predict(s, ydparams, p, d, p, nullptr, nullptr, st);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_surrogate_predict_sp", e);
  return CLOUDSC_OK;
}

int cloudsc_surrogate_gate_scores(cloudsc_surrogate_t* s, float* score, CLOUDSC_BLOCKED_ARGS(float)) {
  SURR_PTRS;
  int rc = check_fields(s, ydparams, ngptot, nproma, klev, ngpblks, p);
  if (rc) return rc;
  if (!score) return fail(CLOUDSC_ENULL, "cloudsc_surrogate_gate_scores: NULL score");
  hipLaunchKernelGGL(surr::select_columns, dim3(nblk(ngptot, 256)), dim3(256), 0, st, p, d, 0.0f, (uint64_t)0, 0.0f,
                     score, (uint8_t*)nullptr, (int*)nullptr);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_surrogate_gate_scores", e);
  return CLOUDSC_OK;
}

int cloudsc_hybrid_sp_c(cloudsc_surrogate_t* s, float rerun_fraction, uint64_t rerun_seed, float gate_threshold,
                        int* n_plain, CLOUDSC_BLOCKED_ARGS(float)) {
  SURR_PTRS;
  int rc = check_fields(s, ydparams, ngptot, nproma, klev, ngpblks, p);
  if (rc) return rc;
  if (!p.pvfl || !p.pvfi || !p.plsm || !p.ldcum || !p.ktype || !p.peis || !p.plu || !p.pludeli || !p.psnde ||
      !p.pmfu || !p.pmfd)
    return fail(CLOUDSC_ENULL, "cloudsc_hybrid_sp_c: NULL array on the default path");
  const cloudsc_params_t* q = ydparams;
  // 1. columns for the plain kernel
  // selection list and ranks (2 ngptot ints), per-group counts and offsets, per-column flags: one allocation
  hipError_t e = hipSuccess;
  const int ngroups = (int)nblk(ngptot, 256);
  if (s->list_cap < ngptot) {
    if (s->list) (void)hipFree(s->list);
    s->list = nullptr;
    s->list_cap = 0;
    e = hipMalloc((void**)&s->list, (size_t)(2L * ngptot + ngroups) * sizeof(int) + (size_t)ngptot);
    if (e != hipSuccess) return fail(CLOUDSC_ENOMEM, "cloudsc_hybrid_sp_c: hipMalloc", e);
    s->list_cap = ngptot;
  }
  int* rank = s->list + ngptot;
  int* group_offsets = rank + ngptot;
  uint8_t* flags = reinterpret_cast<uint8_t*>(group_offsets + ngroups);
  hipLaunchKernelGGL(surr::select_columns, dim3(ngroups), dim3(256), 0, st, p, d, rerun_fraction, rerun_seed,
                     gate_threshold, (float*)nullptr, flags, group_offsets);
  hipLaunchKernelGGL(surr::scan_counts, dim3(1), dim3(1024), 0, st, group_offsets, ngroups, s->count);
  hipLaunchKernelGGL(surr::compact_columns, dim3(ngroups), dim3(256), 0, st, flags, group_offsets, ngptot, s->list, rank);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(s->count_host, s->count, sizeof(int), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipEventRecord(s->counted, st);
  if (e == hipSuccess) {
    launch_features(s, p, d, 0, true, st);  // runs while the host learns the count
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipEventSynchronize(s->counted);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_hybrid_sp_c: selection", e);
  const int nsel = *s->count_host;
  if (n_plain) *n_plain = nsel;
  if (nsel == 0) {
    e = predict(s, q, p, d, p, nullptr, nullptr, st);
    if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_hybrid_sp_c: prediction", e);
    return CLOUDSC_OK;
  }
  // 2. compact field set of the selected columns
  constexpr int NP_C = surr::NP_C;
  const int ncb = (nsel + NP_C - 1) / NP_C;
  const long L = klev, c2 = (long)NP_C * L, ch = (long)NP_C * (L + 1), c1 = NP_C;
  struct Arr {
    void* full;
    int n, L;   // species, levels per species
    bool in;
  };
  Arr arrs[] = {{(void*)p.pt, 1, (int)L, true},        {(void*)p.pq, 1, (int)L, true},
                {(void*)p.tcml_t, 1, (int)L, true},    {(void*)p.tcml_q, 1, (int)L, true},
                {(void*)p.tcml_a, 1, (int)L, true},    {(void*)p.tcml_cld, 5, (int)L, true},
                {(void*)p.tloc_t, 1, (int)L, false},    {(void*)p.tloc_q, 1, (int)L, false},
                {(void*)p.tloc_a, 1, (int)L, false},    {(void*)p.tloc_cld, 5, (int)L, false},
                {(void*)p.pvfl, 1, (int)L, true},      {(void*)p.pvfi, 1, (int)L, true},
                {(void*)p.pap, 1, (int)L, true},       {(void*)p.paph, 1, (int)L + 1, true},
                {(void*)p.plsm, 1, 1, true},           {(void*)p.ldcum, 1, 1, true},
                {(void*)p.ktype, 1, 1, true},          {(void*)p.peis, 1, 1, true},
                {(void*)p.plu, 1, (int)L, true},       {(void*)p.plude, 1, (int)L, true},
                {(void*)p.pludeli, 4, (int)L, true},   {(void*)p.psnde, 2, (int)L, true},
                {(void*)p.pmfu, 1, (int)L, true},      {(void*)p.pmfd, 1, (int)L, true},
                {(void*)p.pa, 1, (int)L, true},        {(void*)p.pclv, 5, (int)L, true},
                {(void*)p.pcovptot, 1, (int)L, false},  {(void*)p.prainfrac_toprfz, 1, 1, false},
                {(void*)p.pfsqlf, 1, (int)L + 1, false}, {(void*)p.pfsqif, 1, (int)L + 1, false},
                {(void*)p.pfcqnng, 1, (int)L + 1, false}, {(void*)p.pfcqlng, 1, (int)L + 1, false},
                {(void*)p.pfsqrf, 1, (int)L + 1, false}, {(void*)p.pfsqsf, 1, (int)L + 1, false},
                {(void*)p.pfcqrng, 1, (int)L + 1, false}, {(void*)p.pfcqsng, 1, (int)L + 1, false},
                {(void*)p.pfsqltur, 1, (int)L + 1, false}, {(void*)p.pfsqitur, 1, (int)L + 1, false},
                {(void*)p.pfplsl, 1, (int)L + 1, false}, {(void*)p.pfplsn, 1, (int)L + 1, false},
                {(void*)p.pfhpsl, 1, (int)L + 1, false}, {(void*)p.pfhpsn, 1, (int)L + 1, false}};
  const int narr = sizeof(arrs) / sizeof(arrs[0]);
  size_t offs[sizeof(arrs) / sizeof(arrs[0])], need = 0;
  for (int i = 0; i < narr; ++i) {
    offs[i] = need;
    need += (((size_t)ncb * NP_C * arrs[i].n * arrs[i].L * 4) + 255) & ~(size_t)255;
  }
  if (s->comp_bytes < need) {
    if (s->comp) (void)hipFree(s->comp);
    s->comp = nullptr;
    s->comp_bytes = 0;
    e = hipMalloc(&s->comp, need);
    if (e != hipSuccess) return fail(CLOUDSC_ENOMEM, "cloudsc_hybrid_sp_c: hipMalloc", e);
    s->comp_bytes = need;
  }
  char* cb = (char*)s->comp;
  surr::Slices sl;
  auto add_slices = [&](int i) {
    const Arr& a = arrs[i];
    for (int sp = 0; sp < a.n; ++sp) {
      surr::Slice& x = sl.s[sl.n++];
      x.full = (uint32_t*)a.full;
      x.comp = (uint32_t*)(cb + offs[i]);
      x.full_stride = (long)nproma * a.n * a.L;
      x.comp_stride = (long)NP_C * a.n * a.L;
      x.full_off = (long)nproma * sp * a.L;
      x.comp_off = (long)NP_C * sp * a.L;
      x.L = a.L;
    }
  };
  sl.n = 0;
  for (int i = 0; i < narr; ++i)
    if (arrs[i].in) add_slices(i);
  const unsigned gx = std::min<unsigned>(nblk((long)nsel * (L + 1), 256), 4096u);
  // Steps 2 and 3 run beside the network's first batch: the gather is bound by memory where the products are by the matrix
  // cores, and the plain kernel has too few columns to occupy the chip.  The side stream starts where the count is known
  // (behind all earlier work of st) and st waits for it before the first outputs.  262,144 columns, 3 % rerun: 5.90 -> 5.26
  // ms.
  hipStream_t side = s->side;
  // An error return leaves nothing on the side stream that still reads the caller's fields.
  struct Idle {
    hipStream_t s;
    ~Idle() {
      if (s) (void)hipStreamSynchronize(s);
    }
  } unjoined{side};
  e = hipStreamWaitEvent(side, s->counted, 0);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_hybrid_sp_c: side stream", e);
  hipLaunchKernelGGL(surr::copy_columns, dim3(gx, sl.n), dim3(256), 0, side, sl, s->list, nsel, nproma, NP_C, 1);
  e = hipGetLastError();
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_hybrid_sp_c: gather", e);
  // 3. plain kernel on the compact set
  auto C = [&](int i) { return (float*)(cb + offs[i]); };
  KPtrs<float> pc;
  pc.pt = C(0); pc.pq = C(1); pc.tcml_t = C(2); pc.tcml_q = C(3); pc.tcml_a = C(4); pc.tcml_cld = C(5);
  pc.tloc_t = C(6); pc.tloc_q = C(7); pc.tloc_a = C(8); pc.tloc_cld = C(9); pc.pvfl = C(10); pc.pvfi = C(11);
  pc.pap = C(12); pc.paph = C(13); pc.plsm = C(14); pc.ldcum = (const int32_t*)C(15);
  pc.ktype = (const int32_t*)C(16); pc.peis = C(17); pc.plu = C(18); pc.plude = C(19); pc.pludeli = C(20);
  pc.psnde = C(21); pc.pmfu = C(22); pc.pmfd = C(23); pc.pa = C(24); pc.pclv = C(25); pc.pcovptot = C(26);
  pc.prainfrac_toprfz = C(27); pc.pfsqlf = C(28); pc.pfsqif = C(29); pc.pfcqnng = C(30); pc.pfcqlng = C(31);
  pc.pfsqrf = C(32); pc.pfsqsf = C(33); pc.pfcqrng = C(34); pc.pfcqsng = C(35); pc.pfsqltur = C(36);
  pc.pfsqitur = C(37); pc.pfplsl = C(38); pc.pfplsn = C(39); pc.pfhpsl = C(40); pc.pfhpsn = C(41);
  const KDims kd{nsel, NP_C, klev, ncb, 1, NP_C};
  e = cloudsc_gpu::launch_cloudsc<float, float>(*q, (double)ptsphy, pc, kd, 0, side);
  if (e == hipSuccess) e = hipEventRecord(s->joined, side);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_hybrid_sp_c: plain kernel", e);
  // 4. network on every other column
  e = predict(s, q, p, d, pc, rank, s->joined, st);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_hybrid_sp_c: prediction", e);
  // 5. PLUDE, a feature that the plain kernel also updates
  sl.n = 0;
  add_slices(19);
  hipLaunchKernelGGL(surr::copy_columns, dim3(gx, sl.n), dim3(256), 0, st, sl, s->list, nsel, nproma, NP_C, 0);
  e = hipGetLastError();
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_hybrid_sp_c: scatter", e);
  unjoined.s = nullptr;
  return CLOUDSC_OK;
}

}  // extern "C"
