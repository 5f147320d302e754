// k_qr.hip -- the exact patch fits (SPRG_FP64, and the fast forms' refits):
// mth::decomposeQR / solveFromQR (mth/mthQR.cc:19-163) operation for
// operation -- Householder reflectors from sequential column sums, an
// EXPLICIT Q formed by reflect_rows, y = Q^T b as a sequential dot product,
// back substitution, evaluation at the entity's node
// (spr/sprRecoverField.cc:283-353).  The size field downstream amplifies an
// ulp of the recovered field by 1e4 and more, so every rounding of that
// sequence is kept: sums in the same order, no fused multiply-add (the
// library is built with -ffp-contract=off), correctly rounded square root
// and division.
//
// The sums are sequential, so the work is spread over independent sums, not
// inside one:
//   R       a lane owns a COLUMN of the patch matrix, in registers: the NT
//           columns' sums and updates run side by side, and a wave holds
//           64 / NT patches (6 of the 10-term fit);
//   Q       a lane owns ROWS of Q (every row evolves independently under the
//           reflectors; only its first NT entries survive to the solve);
//   Q^T b   a lane owns a component.
// What is left of the reference's work: the first reflector's dot products
// are its own entries (q_j starts as e_j), and the last reflector changes
// only entry NT-1 of the NT that are kept.  (The sums' zero terms are left
// out or in as it suits: adding +-0 changes no value but the sign of a zero.)
//
// Up to 32 rows one launch does it all, the reflectors in LDS.  Above, Q is
// nearly all the work (m x m x 9 x 4 operations), and a row of Q fills the
// registers, so there are three launches: k_qr_reflect leaves the reflectors
// in memory, k_qr_rows reads them as scalars (VALU operands that take no
// vector registers) and leaves Q's columns, k_qr_solve finishes.
//
// Measured, 14.0M patches of a 10.4M-tet mesh, 9 components: 225 ms with one
// lane group per patch running the sums, 81.4 ms so; sets of 16 rows (6.1M)
// 24.8 -> 8.8 ms, of 24 rows (6.1M) 69.8 -> 17.9 ms, of 65 to 96 rows (1.7M)
// 123.6 -> 54.6 ms (reflectors 13.4, Q 33.3, solve 7.9).  Bounds: the FP64
// issue of the separate multiplies and adds (no fused ones exist here): VALU
// busy 66% in the small fits; Q's two waves per SIMD (96 doubles a lane) wait
// for the scalar loads.  Q with the reflectors in LDS, a wave's lanes filled
// with the rows of two sets, took 1.6 times as long.
#include <algorithm>

#include "exact_common.h"
#include "fit_common.h"

namespace sprg {
namespace {

// The two factors of monomial k among (1, x, y, z): poly_terms' products.
__device__ __forceinline__ void term_pair(int k, int* a, int* b)
{
  // 1, x, y, z, xy, yz, zx, xx, yy, zz
  *a = k < 4 ? k : k < 7 ? k - 3 : k - 6;
  *b = k < 4 ? 0 : k == 4 ? 2 : k == 5 ? 3 : k == 6 ? 1 : k - 6;
}

// The one point of an affine tet with vertices v (sample_tet's operations).
__device__ __forceinline__ void sample_p1(const MeshView& m, const int4& v, double* X)
{
  const int32_t node[4] = {v.x, v.y, v.z, v.w};
  double xi[3], N[10], x[3] = {0, 0, 0};
  rule_point(1, 0, xi);
  tet_values(1, xi, N);
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int j = 0; j < 3; ++j) x[j] += m.xyz[3 * (int64_t)node[n] + j] * N[n];
  X[0] = 1;
  X[1] = x[0];
  X[2] = x[1];
  X[3] = x[2];
}

// Samples of tet t (getSamplePoints, spr/sprRecoverField.cc:193-211): point
// l < q of the MESH order's rule (the order-1 rule ignores l), mapped by the
// coordinate field in the summation order of apf/apfElement.cc:106-114; each
// node is loaded once for the tet's points.  Row l goes to X[4 l ..] as
// (1, x, y, z).
template <int ORDER>
__device__ __forceinline__ void sample_tet(const MeshView& m, int32_t t, int q, double* X)
{
  constexpr int NN = ORDER == 1 ? 4 : 10;
  constexpr int NQ = ORDER == 1 ? 1 : 4;  // distinct points
  const int64_t tt = t;
  int64_t node[NN];
  const int4 v = *reinterpret_cast<const int4*>(m.tv + 4 * tt);
  node[0] = v.x; node[1] = v.y; node[2] = v.z; node[3] = v.w;
#pragma unroll
  for (int k = 4; k < NN; ++k) node[k] = m.nv + (int64_t)m.te[6 * tt + (k - 4)];
  double x[NQ][3];
#pragma unroll
  for (int l = 0; l < NQ; ++l) x[l][0] = x[l][1] = x[l][2] = 0;
#pragma unroll
  for (int n = 0; n < NN; ++n) {
    const double* p = m.xyz + 3 * node[n];
    const double p0 = p[0], p1 = p[1], p2 = p[2];
#pragma unroll
    for (int l = 0; l < NQ; ++l) {
      double xi[3], N[10];
      rule_point(ORDER, l, xi);
      tet_values(ORDER, xi, N);
      x[l][0] += p0 * N[n];
      x[l][1] += p1 * N[n];
      x[l][2] += p2 * N[n];
    }
  }
  if constexpr (ORDER == 1) {
    for (int l = 0; l < q; ++l) {
      X[4 * l] = 1;
      X[4 * l + 1] = x[0][0];
      X[4 * l + 2] = x[0][1];
      X[4 * l + 3] = x[0][2];
    }
  } else {
#pragma unroll
    for (int l = 0; l < NQ; ++l)
      if (l < q) {
        X[4 * l] = 1;
        X[4 * l + 1] = x[l][0];
        X[4 * l + 2] = x[l][1];
        X[4 * l + 3] = x[l][2];
      }
  }
}

// A patch whose R lost rank: regular sets go to the expansion queue; sets
// whose rank was already decided are inconsistent.  Every lane of the wave
// calls it.
template <int MODE>
__device__ __forceinline__ void rank_failed(const FitArgs& a, bool failed, int64_t p)
{
  if (MODE == FIT_REGULAR) {
    wave_append(1, failed ? 1 : 0, a.L.count + 2 * NBUCKET, a.L.xq, (int32_t)p);
  } else if (failed) {
    atomicOr(a.L.status, ST_INTERNAL);
  }
}

// Back substitution (backsubUT, mth/mthQR.cc:131-148) with the packed upper
// triangle rt(i, j), j >= i, and the polynomial at the node.
template <int NT, class RT>
__device__ __forceinline__ double backsub_eval(const double* y, RT rt, const double* node)
{
  double t[10], x[NT];
  poly_terms(NT == 4 ? 1 : 2, node, t);
#pragma unroll
  for (int ii = 0; ii < NT; ++ii) {
    const int i = NT - ii - 1;
    x[i] = y[i];
#pragma unroll
    for (int j = i + 1; j < NT; ++j) x[i] -= rt(i, j) * x[j];
    x[i] /= rt(i, i);
  }
  double v = 0;
#pragma unroll
  for (int i = 0; i < NT; ++i) v += x[i] * t[i];
  return v;
}

// ---------------------------------------------------------------------------
// up to 32 rows

// R of up to MMAX rows, a column per lane (decomposeQR, mth/mthQR.cc:19-63,
// restricted to what the solve uses): false as soon as a column norm falls
// below 1e-10 (mth/mthQR.cc:31).  KEEP: reflector k stays in sV[k MMAX + k ..],
// R's triangle in sRt; else each takes the place of the one before.  Every
// lane of the wave calls it.
template <int NT, int MMAX, bool KEEP>
__device__ __forceinline__ bool small_r(double (&r)[MMAX], double* sV, double* sN, double* sRt, int gl, bool on,
                                        bool act)
{
  constexpr int G = NT, DIVS = (MMAX + G - 1) / G;
  constexpr int KS = KEEP ? MMAX : 0;  // the reflectors' stride
  bool ok = act;
  double s = 0;  // the squares of the column, rows k on
#pragma unroll
  for (int i = 0; i < MMAX; ++i) s += r[i] * r[i];
#pragma unroll
  for (int k = 0; k < NT; ++k) {
    // get_reflector on every lane's column; column k's is the one kept
    const double cn = sqrt(s);
    const double vk = r[k] + sgn(r[k]) * cn;
    s = vk * vk;
#pragma unroll
    for (int i = k + 1; i < MMAX; ++i) s += r[i] * r[i];
    if (on && gl == k) {
      sN[0] = cn;
      sN[1] = sqrt(s);
      sV[k * KS + k] = vk;
#pragma unroll
      for (int i = k + 1; i < MMAX; ++i) sV[k * KS + i] = r[i];
    }
    __syncthreads();
    ok = ok && !(sN[0] < 1e-10);
    const double rn = sN[1];
    // the lanes' divisions side by side (rows before k, whatever they
    // hold, are not stored)
    double w[DIVS];
#pragma unroll
    for (int u = 0; u < DIVS; ++u) {
      const int i = gl + u * G;
      w[u] = sV[k * KS + (i < MMAX ? i : MMAX - 1)] / rn;
      asm volatile("" : "+v"(w[u]));  // formed here, not under the stores' conditions
    }
#pragma unroll
    for (int u = 0; u < DIVS; ++u) {
      const int i = gl + u * G;
      if (on && i >= k && i < MMAX) sV[k * KS + i] = w[u];
    }
    __syncthreads();
    double v[MMAX];
#pragma unroll
    for (int i = k; i < MMAX; ++i) v[i] = sV[k * KS + i];
    if (!KEEP) __syncthreads();  // read by every lane before the next takes its place
    double dot = 0;
#pragma unroll
    for (int i = k; i < MMAX; ++i) dot += r[i] * v[i];
    const double d2 = 2 * dot;
    // the update, and the squares the next reflector starts from
    s = 0;
#pragma unroll
    for (int i = k; i < MMAX; ++i) {
      r[i] -= d2 * v[i];
      if (i > k) s += r[i] * r[i];
    }
    // row k is final (columns before k hold leftovers there)
    if (KEEP && on && gl >= k) sRt[tri(gl, k)] = r[k];
  }
  return ok;
}

// Rows of Q a lane holds at once, and the passes that cover MMAX rows: as
// many rows as the registers take (each reflector entry read from LDS then
// serves several rows, and the rows' independent sums hide each other's
// latency).
constexpr int small_rpl(int mmax)
{
  return mmax == 24 ? 3 : 2;
}
constexpr int small_waves(int nt, int mmax) { return mmax == 16 ? 3 : 2; }

// A wave's LDS (doubles): per patch its samples, then the reflectors V
// [NT][MMAX], then Q's columns [MMAX][NT]; R's triangle; two norms; its tets.
// The stride keeps the patches' equal offsets 16 bytes apart modulo the banks.
constexpr int small_stride(int nt, int mmax) { return (nt * mmax + nt * (nt + 1) / 2 + 2 + mmax / 2 + 31) / 32 * 32 + 2; }
constexpr int small_lds(int nt, int mmax) { return 64 / nt * small_stride(nt, mmax); }

// The fits of one bucket's list, the launch's blocks (one wave each) taking
// 64 / NT patches in turn; this one is block `block` of them.
template <int NT, int MMAX, int MODE>
__device__ __forceinline__ void small_fit(const FitArgs& a, int bucket, double* sm, int block)
{
  constexpr int ORDER = NT == 4 ? 1 : 2;
  constexpr int G = NT, P = 64 / G;  // lanes per patch, patches per wave
  constexpr int RPL = small_rpl(MMAX);
  constexpr int NPASS = (MMAX + G * RPL - 1) / (G * RPL);
  constexpr int VS = NT * MMAX, NRT = NT * (NT + 1) / 2;
  constexpr int S = small_stride(NT, MMAX);
  const int lane = threadIdx.x;
  const int g = lane / G < P ? lane / G : P - 1;
  int gl = lane - g * G;
  const bool on = gl < G;  // the lanes past P * G own nothing
  const int col = on ? gl : G - 1;
  double* const sV = sm + g * S;
  double* const sRt = sV + VS;
  double* const sN = sRt + NRT;
  int32_t* const sS = reinterpret_cast<int32_t*>(sN + 2);
  int fa, fb;
  term_pair(col, &fa, &fb);
  const MeshView& m = a.m;
  const int q = a.q, nc = a.nc;
  int nitems;
  const int32_t* const list = fit_list<MODE>(a, bucket, &nitems);
  for (int base = block * P; base < nitems; base += gridDim.x * P) {
    asm volatile("" : "+v"(gl));  // its many comparisons stay inside the loop (hoisted, they spill)
    const bool act = base + g < nitems;
    int64_t p = 0;
    int ns = 0;
    const int32_t* set = nullptr;
    if (act) fit_item<MODE>(a, list[base + g], &p, &set, &ns);
    const int rows = ns * q;  // <= MMAX
    if (NT == 4 && q == 1) {
      // up to MMAX / 4 tets a lane: every id, then every tet's vertices, then
      // the coordinates, instead of three round trips for each (with the
      // values below eight at a time, 275k sets of 24 rows and nine
      // components take 255 us; a load after another took 412)
      constexpr int K = (MMAX + G - 1) / G;
      int32_t t[K];
      int4 v[K];
#pragma unroll
      for (int k = 0; k < K; ++k) t[k] = ns > 0 ? set[gl + k * G < ns ? gl + k * G : 0] : 0;
#pragma unroll
      for (int k = 0; k < K; ++k) v[k] = *reinterpret_cast<const int4*>(m.tv + 4 * (int64_t)t[k]);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int s = gl + k * G;
        if (on && s < ns) {
          sS[s] = t[k];
          sample_p1(m, v[k], sV + 4 * s);
        }
      }
    } else if (on) {
      for (int s = gl; s < ns; s += G) {
        const int32_t t = set[s];
        sS[s] = t;
        sample_tet<ORDER>(m, t, q, sV + 4 * s * q);
      }
    }
    __syncthreads();
    // R: this lane's column
    double r[MMAX];
#pragma unroll
    for (int i = 0; i < MMAX; ++i) {
      const double v = sV[4 * i + fa] * sV[4 * i + fb];
      r[i] = i < rows ? v : 0.0;
    }
    __syncthreads();
    const bool ok = small_r<NT, MMAX, true>(r, sV, sN, sRt, gl, on, act);
    rank_failed<MODE>(a, act && !ok && gl == 0, p);
    // Q: rows gl, gl + G, ... of each pass
    double Qr[NPASS][RPL][NT];
#pragma unroll
    for (int ps = 0; ps < NPASS; ++ps) {
      double x[RPL][MMAX], t2[RPL];
#pragma unroll
      for (int u = 0; u < RPL; ++u) {
        const int j = (ps * RPL + u) * G + gl;
        t2[u] = 2 * (j < MMAX ? sV[j] : 0.0);  // 2 e_j . v_0
      }
#pragma unroll
      for (int l = 0; l < MMAX; ++l) {
        const double v = sV[l];
#pragma unroll
        for (int u = 0; u < RPL; ++u) {
          constexpr int G_ = G;
          const int j0 = (ps * RPL + u) * G_;  // the lane's row is j0 + gl
          const double pr = t2[u] * v;
          x[u][l] = (l >= j0 && l < j0 + G_) ? (gl == l - j0 ? 1.0 : 0.0) - pr : -pr;
        }
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int k = 1; k < NT; ++k) {
        double dot[RPL];
#pragma unroll
        for (int u = 0; u < RPL; ++u) dot[u] = 0;
#pragma unroll
        for (int l = k; l < MMAX; ++l) {
          const double v = sV[k * MMAX + l];
#pragma unroll
          for (int u = 0; u < RPL; ++u) dot[u] += x[u][l] * v;
        }
#pragma unroll
        for (int u = 0; u < RPL; ++u) {
          t2[u] = 2 * dot[u];
          asm volatile("" : "+v"(t2[u]));  // formed here, not where Q is stored
        }
        // the reflector is read again for the update: held, it would cost
        // MMAX more registers
        asm volatile("" ::: "memory");
#pragma unroll
        for (int l = k; l < (k == NT - 1 ? NT : MMAX); ++l) {
          const double v = sV[k * MMAX + l];
#pragma unroll
          for (int u = 0; u < RPL; ++u) x[u][l] -= t2[u] * v;
        }
        asm volatile("" ::: "memory");
      }
#pragma unroll
      for (int u = 0; u < RPL; ++u)
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          Qr[ps][u][i] = x[u][i];
          asm volatile("" : "+v"(Qr[ps][u][i]));
        }
    }
    __syncthreads();
#pragma unroll
    for (int ps = 0; ps < NPASS; ++ps)
#pragma unroll
      for (int u = 0; u < RPL; ++u) {
        const int j = (ps * RPL + u) * G + gl;
        if (on && j < rows)
#pragma unroll
          for (int i = 0; i < NT; ++i) sV[j * NT + i] = Qr[ps][u][i];
      }
    __syncthreads();
    // y = Q^T b (mth/mth_def.h:221-232), sequential over the rows; a lane
    // per component reads its own values and solves for them
    if (on && ok) {
      const double node[3] = {m.xyz[3 * p], m.xyz[3 * p + 1], m.xyz[3 * p + 2]};
      for (int c = gl; c < nc; c += G) {
        double y[NT];
#pragma unroll
        for (int i = 0; i < NT; ++i) y[i] = 0;
        auto add_row = [&](int r_, double b) {
#pragma unroll
          for (int i = 0; i < NT; ++i) y[i] += sV[r_ * NT + i] * b;
        };
        if (q == 4) {
          // the next tet's four values in flight while one is summed
          double b[4], bn[4];
          const double* src = a.ip + (int64_t)sS[0] * 4 * nc + c;
#pragma unroll
          for (int l = 0; l < 4; ++l) bn[l] = src[l * nc];
          for (int s = 0; s < ns; ++s) {
#pragma unroll
            for (int l = 0; l < 4; ++l) b[l] = bn[l];
            src = a.ip + (int64_t)sS[s + 1 < ns ? s + 1 : s] * 4 * nc + c;
#pragma unroll
            for (int l = 0; l < 4; ++l) bn[l] = src[l * nc];
#pragma unroll
            for (int l = 0; l < 4; ++l) add_row(4 * s + l, b[l]);
          }
        } else if (NT == 4 && q == 1) {
          // eight tets' values in flight while eight are summed
          double b[8], bn[8];
          auto fetch = [&](int s0) {
#pragma unroll
            for (int l = 0; l < 8; ++l) bn[l] = a.ip[(int64_t)sS[s0 + l < ns ? s0 + l : 0] * nc + c];
          };
          fetch(0);
          for (int s0 = 0; s0 < ns; s0 += 8) {
#pragma unroll
            for (int l = 0; l < 8; ++l) b[l] = bn[l];
            if (s0 + 8 < ns) fetch(s0 + 8);
#pragma unroll
            for (int l = 0; l < 8; ++l)
              if (s0 + l < ns) add_row(s0 + l, b[l]);
          }
        } else {
          for (int s = 0; s < ns; ++s)
            for (int l = 0; l < q; ++l) add_row(s * q + l, a.ip[((int64_t)sS[s] * q + l) * nc + c]);
        }
        a.out[p * nc + c] = backsub_eval<NT>(y, [&](int i, int j) { return sRt[tri(j, i)]; }, node);
      }
    }
    __syncthreads();
  }
}

template <int NT, int MMAX, int MODE>
__global__ __launch_bounds__(64, small_waves(NT, MMAX)) void k_qr_small(FitArgs a, int bucket)
{
  constexpr int SM = small_lds(NT, MMAX);
  __shared__ double sm[SM];
  small_fit<NT, MMAX, MODE>(a, bucket, sm, blockIdx.x);
}

// The three lists in one launch: the ones whose lengths only the device
// knows (most calls have few sets there or none, and an empty launch costs
// what a full one waits for), and the initial sets of small meshes.  A list
// starts at the block after the last that the one before it needs, so that
// short lists run side by side.
template <int NT, int MODE>
__global__ __launch_bounds__(64, 2) void k_qr_small_lists(FitArgs a)
{
  constexpr int SM = small_lds(NT, 32);
  __shared__ double sm[SM];
  constexpr int P = 64 / NT;
  const int nb = gridDim.x;
  int block = blockIdx.x, n;
  small_fit<NT, 16, MODE>(a, 0, sm, block);
  fit_list<MODE>(a, 0, &n);
  block = (block + nb - (n + P - 1) / P % nb) % nb;
  small_fit<NT, 24, MODE>(a, 1, sm, block);
  fit_list<MODE>(a, 1, &n);
  block = (block + nb - (n + P - 1) / P % nb) % nb;
  small_fit<NT, 32, MODE>(a, 2, sm, block);
}

// ---------------------------------------------------------------------------
// The reference's rank test of the initial sets that the fast forms could not
// certify (xq entries with bit 31), before the expansion: six sets a wave.
// A set of full rank becomes the patch's set; any other goes on to the
// expansion without the test (x_len X_TESTED, bit 31 cleared).  Sets above 32
// rows and short ones stay as they are (x_len 0).
// (The expansion's own test takes a wave per set, its sums on one lane: 15.9
// ms for the 452,700 edge sets of a lattice box at n = 40, and 4.5 ms more to
// queue them one by one; 1.08 ms here.)
constexpr int TEST_ROWS = 32;

template <int NT>
__global__ __launch_bounds__(64, 2) void k_rank_test(FitArgs a)
{
  constexpr int ORDER = NT == 4 ? 1 : 2;
  constexpr int G = NT, P = 64 / G, MMAX = TEST_ROWS;
  constexpr int VS = 4 * MMAX;  // samples, then a reflector
  constexpr int S = (VS + 2 + 31) / 32 * 32 + 2;
  __shared__ double sm[P * S];
  const int lane = threadIdx.x;
  const int g = lane / G < P ? lane / G : P - 1;
  int gl = lane - g * G;
  const bool on = gl < G;
  const int col = on ? gl : G - 1;
  double* const sV = sm + g * S;
  double* const sN = sV + VS;
  int fa, fb;
  term_pair(col, &fa, &fb);
  const MeshView& m = a.m;
  const int q = a.q;
  const int nq = a.L.count[2 * NBUCKET];
  for (int base = blockIdx.x * P; base < nq; base += gridDim.x * P) {
    asm volatile("" : "+v"(gl));
    const int it = base + g;
    const int32_t entry = it < nq ? a.L.xq[it] : 0;
    const int64_t p = entry & 0x7fffffff;
    int ns = 0;
    const int32_t* set = nullptr;
    if (entry < 0) patch_set(a, p, &set, &ns);
    const bool act = entry < 0 && ns * q >= NT && ns * q <= MMAX;
    const int rows = act ? ns * q : 0;
    int mw = rows;  // the wave's longest set
    for (int o = 32; o > 0; o >>= 1) {
      const int y = __shfl(mw, lane ^ o);
      mw = y > mw ? y : mw;
    }
    mw = __builtin_amdgcn_readlane(mw, 0);
    bool ok = false;
    if (mw > 0) {  // wave-uniform
      if (on && act)
        for (int s = gl; s < ns; s += G) sample_tet<ORDER>(m, set[s], q, sV + 4 * s * q);
      __syncthreads();
      auto test = [&](auto size) {
        constexpr int M = decltype(size)::value;
        double r[M];
#pragma unroll
        for (int i = 0; i < M; ++i) {
          const double v = sV[4 * i + fa] * sV[4 * i + fb];
          r[i] = i < rows ? v : 0.0;
        }
        __syncthreads();
        ok = small_r<NT, M, false>(r, sV, sN, nullptr, gl, on, act);
      };
      if (mw <= 16)
        test(std::integral_constant<int, 16>());
      else if (mw <= 24)
        test(std::integral_constant<int, 24>());
      else
        test(std::integral_constant<int, 32>());
    }
    // places in x_set for the wave's full-rank sets, one atomic per wave
    const bool head = on && gl == 0 && it < nq;
    const int len = head && ok ? ns : 0;
    int end = len;  // inclusive sum over the lanes
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl(end, lane - o);
      if (lane >= o) end += y;
    }
    const int total = __builtin_amdgcn_readlane(end, 63);
    int64_t off = 0;
    if (total > 0) {
      int lo = 0, hi = 0;
      if (lane == 0) {
        const unsigned long long at = atomicAdd((unsigned long long*)a.L.x_cursor, (unsigned long long)total);
        lo = (int)(uint32_t)at;
        hi = (int)(uint32_t)(at >> 32);
      }
      lo = __builtin_amdgcn_readlane(lo, 0);
      hi = __builtin_amdgcn_readlane(hi, 0);
      off = (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo) + end - len;
    }
    if (head) {
      const bool room = off + len <= a.L.x_cap;
      if (len > 0 && !room) atomicOr(a.L.status, ST_XSET_OVERFLOW);
      a.L.x_len[it] = len == 0 && act ? X_TESTED : room ? len : 0;
      if (len > 0 && room) {
        a.L.x_patch[it] = (int32_t)p;
        a.L.x_off[it] = off;
        for (int i = 0; i < len; ++i) a.L.x_set[off + i] = set[i];
      }
      if (act && !ok) a.L.xq[it] = (int32_t)p;
    }
    const uint64_t tested = __ballot(head && act);
    if (lane == 0 && tested) atomicAdd(a.L.status + 4, __popcll(tested));
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// 33 to 192 rows: the regular sets of a bucket, a chunk at a time

// Workspace of one set: the reflectors [NT][MMAX] (zero outside rows
// k..m-1, up to the next multiple of 8 rows), then R's top [NT][NT], whose
// last row's first entry says whether R kept full rank.
constexpr int qr_ws_doubles(int nt, int mmax) { return nt * mmax + nt * nt; }
constexpr int qr_waves(int mmax) { return (mmax + 63) / 64; }
// with Q's first NT columns [MMAX][NT]
constexpr size_t qr_set_bytes(int nt, int mmax) { return sizeof(double) * (qr_ws_doubles(nt, mmax) + (size_t)mmax * nt); }

// Lanes per patch: one per column (of the 4-term fit, whose patches would
// take too much LDS sixteen to a wave, twice that).
constexpr int reflect_lanes(int nt) { return nt == 4 ? 8 : nt; }

// The reflectors of the sets items[first, first + cap) of the bucket.  The
// row loop runs over a column that shifts up by one entry per reflector, so
// that every register index is fixed and the reflector loop stays rolled;
// blocks of rows past the wave's longest set are skipped.
template <int NT, int MMAX>
__global__ __launch_bounds__(64, MMAX <= 96 ? 2 : 1) void k_qr_reflect(FitArgs a, int bucket, int first, int cap,
                                                                       double* __restrict__ ws)
{
  constexpr int ORDER = NT == 4 ? 1 : 2;
  constexpr int G = reflect_lanes(NT), P = 64 / G, B = 16, D = 5, E = 8;
  constexpr int WS = qr_ws_doubles(NT, MMAX);
  constexpr int S = 4 * MMAX + 2;  // samples, then the current reflector
  static_assert(MMAX % B == 0, "whole blocks of rows");
  __shared__ double sm[P * S];
  __shared__ double sNorm[P][2];
  const int lane = threadIdx.x;
  const int g = lane / G < P ? lane / G : P - 1;
  int gl = lane - g * G;
  const bool on = gl < G;
  const int col = gl < NT ? gl : NT - 1;
  double* const sV = sm + g * S;
  double* const sN = sNorm[g];
  int fa, fb;
  term_pair(col, &fa, &fb);
  const MeshView& m = a.m;
  const int q = a.q;
  int nitems;
  const int32_t* const list = fit_list<FIT_REGULAR>(a, bucket, &nitems);
  const int left = nitems - first, n = left < cap ? left : cap;
  for (int base = blockIdx.x * P; base < n; base += gridDim.x * P) {
    asm volatile("" : "+v"(gl));
    const bool act = base + g < n;
    int64_t p = 0;
    int ns = 0;
    const int32_t* set = nullptr;
    if (act) fit_item<FIT_REGULAR>(a, list[first + base + g], &p, &set, &ns);
    const int rows = ns * q;
    int mw = rows;  // the wave's longest set
    for (int o = 32; o > 0; o >>= 1) {
      const int y = __shfl(mw, lane ^ o);
      mw = y > mw ? y : mw;
    }
    mw = __builtin_amdgcn_readlane(mw, 0);
    double* const W = ws + (int64_t)(base + g) * WS;  // touched by active patches only
    if (on)
      for (int s = gl; s < ns; s += G) sample_tet<ORDER>(m, set[s], q, sV + 4 * s * q);
    __syncthreads();
    double r[MMAX];
#pragma unroll
    for (int i0 = 0; i0 < MMAX; i0 += B) {
#pragma unroll
      for (int i = i0; i < i0 + B; ++i) r[i] = 0;
      if (i0 < mw) {
#pragma unroll
        for (int i = i0; i < i0 + B; ++i) {
          const double v = sV[4 * i + fa] * sV[4 * i + fb];
          r[i] = i < rows ? v : 0.0;
        }
      }
    }
    __syncthreads();
    bool ok = act;
    double s = 0;  // the squares of the column, rows k on
#pragma unroll
    for (int i0 = 0; i0 < MMAX; i0 += B)
      if (i0 < mw) {
#pragma unroll
        for (int i = i0; i < i0 + B; ++i) {
          s += r[i] * r[i];
          asm volatile("" : "+v"(r[i]));  // the squares are formed again below: MMAX of them would not fit
        }
      }
#pragma unroll 1
    for (int k = 0; k < NT; ++k) {
      const int mk = mw - k;  // r[i] is row k + i
      const double cn = sqrt(s);
      const double vk = r[0] + sgn(r[0]) * cn;
      s = vk * vk;
#pragma unroll
      for (int i0 = 0; i0 < MMAX; i0 += B)
        if (i0 < mk) {
#pragma unroll
          for (int i = i0; i < i0 + B; ++i)
            if (i > 0) s += r[i] * r[i];
        }
      if (on && gl == k) {
        sN[0] = cn;
        sN[1] = sqrt(s);
#pragma unroll
        for (int i0 = 0; i0 < MMAX; i0 += B)
          if (i0 <= mk) {
#pragma unroll
            for (int i = i0; i < i0 + B; ++i) sV[i] = i == 0 ? vk : r[i];
          }
      }
      __syncthreads();
      ok = ok && !(sN[0] < 1e-10);
      const double rn = sN[1];
      {
        // the normalised reflector, D divisions of a lane side by side
        const int end = rows - k, pad = ((rows + 7) & ~7) - k;
        double* const Vk = W + k * MMAX;
        if (on && act && gl < k) Vk[gl] = 0;
#pragma unroll 1
        for (int i0 = 0; i0 < mk + 7; i0 += D * G) {
          double w[D];
#pragma unroll
          for (int u = 0; u < D; ++u) {
            const int i = i0 + u * G + gl;
            w[u] = sV[i < MMAX ? i : MMAX - 1] / rn;
            asm volatile("" : "+v"(w[u]));  // formed here, not under the stores' conditions
          }
#pragma unroll
          for (int u = 0; u < D; ++u) {
            const int i = i0 + u * G + gl;
            if (on && act && i < pad) {
              if (i < end) sV[i] = w[u];
              Vk[k + i] = i < end ? w[u] : 0.0;
            }
          }
        }
      }
      __syncthreads();
      // the reflector is read from LDS eight entries ahead of their use,
      // twice (the column leaves no room to hold it)
      double v[E], vn[E];
      auto fetch = [&](int i0) {
#pragma unroll
        for (int u = 0; u < E; ++u) vn[u] = sV[i0 + u];
      };
      auto arrive = [&]() {
#pragma unroll
        for (int u = 0; u < E; ++u) v[u] = vn[u];
        asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
        asm volatile("" ::: "memory");
      };
      fetch(0);
      double dot = 0;
#pragma unroll
      for (int i0 = 0; i0 < MMAX; i0 += E)
        if (i0 < mk) {
          arrive();
          fetch(i0 + E);
#pragma unroll
          for (int u = 0; u < E; ++u) dot += r[i0 + u] * v[u];
          asm volatile("" : "+v"(dot));
        }
      const double d2 = 2 * dot;
      fetch(0);
      const double top = r[0] - d2 * sV[0];
      if (on && act && gl >= k && gl < NT) W[NT * MMAX + k * NT + gl] = top;
      // the update, each row one place up, and the squares the next
      // reflector starts from; a block starting at mk still hands its (zero)
      // first row to the block before
      s = 0;
#pragma unroll
      for (int i0 = 0; i0 < MMAX; i0 += E)
        if (i0 <= mk) {
          arrive();
          fetch(i0 + E);
#pragma unroll
          for (int u = 0; u < E; ++u)
            if (i0 + u > 0) {
              r[i0 + u - 1] = r[i0 + u] - d2 * v[u];
              s += r[i0 + u - 1] * r[i0 + u - 1];
              asm volatile("" : "+v"(r[i0 + u - 1]));
            }
          asm volatile("" : "+v"(s));
        }
      r[MMAX - 1] = 0;
      __syncthreads();
    }
    if (act && gl == 0) W[NT * MMAX + (NT - 1) * NT] = ok ? 1.0 : 0.0;
    rank_failed<FIT_REGULAR>(a, act && !ok && gl == 0, p);
    __syncthreads();
  }
}

// Q of the same sets: a block per set, a wave per 64 rows, a row per lane; the
// first NT entries of each row are kept.  The reflectors are read at addresses
// that are the same for the whole wave, as scalars; the block's waves read the
// same ones at about the same time, and the four sets that a CU holds then
// keep two reflectors each in the scalar cache, so a sweep finds the reflector
// of the sweep before it there.
template <int NT, int MMAX>
__global__ __launch_bounds__(64 * qr_waves(MMAX), MMAX <= 96 ? 2 : 1) void k_qr_rows(
    FitArgs a, int bucket, int first, int cap, const double* __restrict__ ws, double* __restrict__ qs)
{
  constexpr int WS = qr_ws_doubles(NT, MMAX), B = 8;
  int tid = threadIdx.x;
  const int r0 = 64 * __builtin_amdgcn_readlane(tid >> 6, 0);  // the wave's first row
  int nitems;
  const int32_t* const list = fit_list<FIT_REGULAR>(a, bucket, &nitems);
  const int left = nitems - first, n = left < cap ? left : cap;
  for (int it = blockIdx.x; it < n; it += gridDim.x) {
    asm volatile("" : "+v"(tid));  // what depends on it stays inside the loop (hoisted, it costs the row its registers)
    const int lane = tid & 63;
    const double* __restrict__ V = ws + (int64_t)it * WS;
    if (V[NT * MMAX + (NT - 1) * NT] == 0) continue;  // R lost rank: queued for the expansion
    int64_t p;
    int ns;
    const int32_t* set;
    fit_item<FIT_REGULAR>(a, list[first + it], &p, &set, &ns);
    const int rows = ns * a.q;
    if (r0 >= rows) continue;
    const int j = r0 + lane;  // this lane's row
    double x[MMAX];
    double t2 = 2 * (j < rows ? V[j] : 0.0);  // 2 e_j . v_0
    double dot = 0;
    // Reflector k's update and reflector k + 1's dot product in one sweep,
    // eight rows at a time; the next eight rows' entries of both are in
    // flight meanwhile.  (Scalar loads return in any order, so a wait is a
    // wait for all: the loads are issued once the first row has used the
    // current entries.)
    auto sweep = [&](const double* __restrict__ v, auto first_sweep) {
      double a0[B], a1[B], n0[B], n1[B];
      auto load = [&](int l0) {
#pragma unroll
        for (int u = 0; u < B; ++u) {
          n0[u] = v[l0 + u];
          n1[u] = v[MMAX + l0 + u];
        }
      };
      load(0);
#pragma unroll
      for (int l0 = 0; l0 < MMAX; l0 += B)
        if (l0 < rows) {
#pragma unroll
          for (int u = 0; u < B; ++u) {
            a0[u] = n0[u];
            a1[u] = n1[u];
          }
#pragma unroll
          for (int u = 0; u < B; ++u) {
            const int l = l0 + u;
            x[l] = (first_sweep ? (l == j ? 1.0 : 0.0) : x[l]) - t2 * a0[u];
            if (u == 0) {
              asm volatile("" : "+v"(x[l]));
              asm volatile("" ::: "memory");
              load(l0 + B < MMAX ? l0 + B : l0);
            }
            dot += x[l] * a1[u];
          }
          // keeps the loads in this block (sunk to the next, they would be
          // waited for at once)
          asm volatile("" : "+v"(dot) : "s"(n0[0]), "s"(n1[0]));
        }
    };
    // the reflector after next into this XCD's L2 meanwhile (it was
    // written through another's: its first read would wait for memory)
    double ahead = V[2 * MMAX + (lane < MMAX / 8 ? 8 * lane : 0)];
    sweep(V, std::true_type());
    asm volatile("" : "+v"(ahead));
#pragma unroll 1
    for (int k = 1; k < NT - 1; ++k) {
      t2 = 2 * dot;
      dot = 0;
      ahead = V[(k + 2 < NT ? k + 2 : k) * MMAX + (lane < MMAX / 8 ? 8 * lane : 0)];
      sweep(V + k * MMAX, std::false_type());
      asm volatile("" : "+v"(ahead));
    }
    x[NT - 1] -= (2 * dot) * V[(NT - 1) * MMAX + NT - 1];
    if (j < rows) {
      double* const Q = qs + (int64_t)it * (MMAX * NT) + j * NT;
#pragma unroll
      for (int i = 0; i < NT; ++i) Q[i] = x[i];
    }
  }
}

// y = Q^T b (mth/mth_def.h:221-232), sequential over the rows, back
// substitution and the value at the node, a thread per set and component:
// latency-bound chains, so many waves, apart from k_qr_rows' two per SIMD.
template <int NT, int MMAX>
__global__ __launch_bounds__(256) void k_qr_solve(FitArgs a, int bucket, int first, int cap,
                                                  const double* __restrict__ ws, const double* __restrict__ qs)
{
  constexpr int WS = qr_ws_doubles(NT, MMAX), L = 4;
  int nitems;
  const int32_t* const list = fit_list<FIT_REGULAR>(a, bucket, &nitems);
  const int left = nitems - first, n = left < cap ? left : cap;
  const int64_t id = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (id >= (int64_t)n * a.nc) return;
  const int it = (int)(id / a.nc), c = (int)(id % a.nc);
  const double* const Rt = ws + (int64_t)it * WS + NT * MMAX;
  if (Rt[(NT - 1) * NT] == 0) return;
  int64_t p;
  int ns;
  const int32_t* set;
  fit_item<FIT_REGULAR>(a, list[first + it], &p, &set, &ns);
  const int q = a.q;
  const double* Q = qs + (int64_t)it * (MMAX * NT);
  double y[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) y[i] = 0;
  auto add_row = [&](double b) {
#pragma unroll
    for (int i = 0; i < NT; ++i) y[i] += Q[i] * b;
    Q += NT;
  };
  if (q == 4) {
    // the next tet's values in flight while one is summed
    double b[L], bn[L];
    auto load = [&](int32_t t) {
#pragma unroll
      for (int l = 0; l < L; ++l) bn[l] = a.ip[((int64_t)t * 4 + l) * a.nc + c];
    };
    load(set[0]);
    int32_t tn = set[ns > 1 ? 1 : 0];
    for (int s = 0; s < ns; ++s) {
#pragma unroll
      for (int l = 0; l < L; ++l) b[l] = bn[l];
      load(tn);
      tn = set[s + 2 < ns ? s + 2 : ns - 1];
#pragma unroll
      for (int l = 0; l < L; ++l) add_row(b[l]);
    }
  } else {
    for (int s = 0; s < ns; ++s)
      for (int l = 0; l < q; ++l) add_row(a.ip[((int64_t)set[s] * q + l) * a.nc + c]);
  }
  const double node[3] = {a.m.xyz[3 * p], a.m.xyz[3 * p + 1], a.m.xyz[3 * p + 2]};
  a.out[p * a.nc + c] = backsub_eval<NT>(y, [&](int i, int j) { return Rt[i * NT + j]; }, node);
}

// Sets per k_qr_reflect / k_qr_rows / k_qr_solve sequence: two waves of
// k_qr_reflect (six sets each) for every SIMD and twelve rounds of k_qr_rows,
// so no launch ends in a part round, and little enough (199 MB of reflectors
// and Q at 96 rows) that each launch finds the last one's results in the
// 256 MB memory-side cache.  A step at 10.4M tets: 84.2 ms; 36,864 sets at a
// time 90.3, 18,432 86.0, 6,144 99.6.
constexpr int64_t QR_CHUNK = 12288;

template <int NT, int MMAX>
void large_fits(const FitArgs& a, int bucket, int64_t count, double* ws, size_t ws_bytes, hipStream_t s)
{
  constexpr int P = 64 / reflect_lanes(NT);
  const int cap = (int)std::min<int64_t>(QR_CHUNK, (int64_t)(ws_bytes / qr_set_bytes(NT, MMAX)));
  double* const qs = ws + (int64_t)cap * qr_ws_doubles(NT, MMAX);
  for (int64_t first = 0; first < count; first += cap) {
    const int64_t n = std::min<int64_t>(cap, count - first);
    const int64_t most = a.shape.exact_blocks;
    k_qr_reflect<NT, MMAX><<<(unsigned)std::min(most, (n + P - 1) / P), 64, 0, s>>>(a, bucket, (int)first, cap, ws);
    if (a.nc == 0) continue;  // the rank decisions alone
    k_qr_rows<NT, MMAX><<<(unsigned)std::min(most, n), 64 * qr_waves(MMAX), 0, s>>>(a, bucket, (int)first, cap, ws, qs);
    k_qr_solve<NT, MMAX><<<(unsigned)((n * a.nc + 255) / 256), 256, 0, s>>>(a, bucket, (int)first, cap, ws, qs);
  }
}

constexpr int64_t SMALL_TOGETHER = 2048;  // two waves a SIMD

template <int NT>
int regular_fits(const FitArgs& a, const int64_t* count, double* ws, size_t ws_bytes, hipStream_t s)
{
  static_assert(NSMALL == 3 && NBUCKET == 7, "the buckets below");
  for (int b = NSMALL; b < NBUCKET; ++b)
    if (count[b] && ws_bytes < qr_set_bytes(NT, bucket_rows(b)))
      return sprg_fail(SPRG_ENOMEM, "exact fit: no workspace for a set of %d rows", bucket_rows(b));
  constexpr int P = 64 / NT;
  auto blocks = [&](int b) { return (unsigned)std::min<int64_t>(a.shape.exact_blocks, (count[b] + P - 1) / P); };
  // all three in one launch while every block of it is on the chip at once
  // (729 patches: 32 us in two launches, 19 in one); beyond, each by its own
  // kernel's registers (four more waves a CU for the 16-row sets)
  const int64_t small = blocks(0) + blocks(1) + blocks(2);
  if (small > 0 && small <= SMALL_TOGETHER) {
    k_qr_small_lists<NT, FIT_REGULAR><<<(unsigned)small, 64, 0, s>>>(a);
  } else {
    if (count[0]) k_qr_small<NT, 16, FIT_REGULAR><<<blocks(0), 64, 0, s>>>(a, 0);
    if (count[1]) k_qr_small<NT, 24, FIT_REGULAR><<<blocks(1), 64, 0, s>>>(a, 1);
    if (count[2]) k_qr_small<NT, 32, FIT_REGULAR><<<blocks(2), 64, 0, s>>>(a, 2);
  }
  large_fits<NT, 64>(a, 3, count[3], ws, ws_bytes, s);
  large_fits<NT, 96>(a, 4, count[4], ws, ws_bytes, s);
  large_fits<NT, 128>(a, 5, count[5], ws, ws_bytes, s);
  large_fits<NT, 192>(a, 6, count[6], ws, ws_bytes, s);
  return hipGetLastError() == hipSuccess ? 0 : sprg_fail(SPRG_EHIP, "exact fit launch failed");
}

}  // namespace

QrWsBytes qr_ws_bytes(int nterms, const int64_t* count)
{
  QrWsBytes n;
  for (int b = NSMALL; b < NBUCKET; ++b)
    if (count[b]) {
      const size_t set = qr_set_bytes(nterms, bucket_rows(b));
      n.least = std::max(n.least, set);
      n.most = std::max(n.most, set * (size_t)std::min<int64_t>(count[b], QR_CHUNK));
    }
  return n;
}

int launch_qr_regular(const FitArgs& a, int nterms, const int64_t* count, void* ws, size_t ws_bytes, hipStream_t s)
{
  double* const w = static_cast<double*>(ws);
  return nterms == 4 ? regular_fits<4>(a, count, w, ws_bytes, s) : regular_fits<10>(a, count, w, ws_bytes, s);
}

int launch_rank_test(const FitArgs& a, int nterms, hipStream_t s)
{
  const int P = nterms == 4 ? 16 : 6;
  const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>(a.shape.expand_blocks, (a.npatch + P - 1) / P));
  if (nterms == 4)
    k_rank_test<4><<<blocks, 64, 0, s>>>(a);
  else
    k_rank_test<10><<<blocks, 64, 0, s>>>(a);
  return hipGetLastError() == hipSuccess ? 0 : sprg_fail(SPRG_EHIP, "rank test launch failed");
}

int launch_qr_lists(const FitArgs& a, int nterms, int mode, hipStream_t s)
{
  if (a.npatch == 0) return 0;
  const int P = nterms == 4 ? 16 : 6;
  const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>(a.shape.exact_blocks, (a.npatch + P - 1) / P));
  if (mode == FIT_EXPANDED) {
    if (nterms == 4)
      k_qr_small_lists<4, FIT_EXPANDED><<<blocks, 64, 0, s>>>(a);
    else
      k_qr_small_lists<10, FIT_EXPANDED><<<blocks, 64, 0, s>>>(a);
  } else {
    if (nterms == 4)
      k_qr_small_lists<4, FIT_MIXED><<<blocks, 64, 0, s>>>(a);
    else
      k_qr_small_lists<10, FIT_MIXED><<<blocks, 64, 0, s>>>(a);
  }
  if (hipGetLastError() != hipSuccess) return sprg_fail(SPRG_EHIP, "exact fit launch failed");
  return launch_exact_lists(a, nterms, mode, s);
}

}  // namespace sprg
