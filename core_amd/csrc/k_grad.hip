// k_grad.hip -- spr::getGradIPField (spr/sprGetGradIPField.cc:15-65).
//
// The Jacobian of the coordinate field, its cofactor inverse and the global
// shape gradients follow apf/apfVectorElement.cc:44-66,
// apf/apfMatrix.h:165-173 and apf/apfElement.cc:77-90 operation for
// operation; the field gradient follows ScalarElement::grad /
// VectorElement::grad / MatrixElement::grad (apf/apfScalarElement.cc:18-26,
// apf/apfVectorElement.cc:44-59, apf/apfMatrixElement.cc:24-46).  Orders,
// rule and component count are template arguments, so rule points and local
// shape gradients are constants; folding them rounds as the run-time
// evaluation does (IEEE operations in the written order, no contraction).
//
// Rules of several points: a block takes 64 tets, a wave per point.
// - The tets' nodes are gathered once for all points into LDS, the waves
//   sharing the nodes, three lanes to a node's 24 bytes (a gather costs the
//   vector cache an access per distinct line).
// - Each wave forms its point's gradients with a lane per tet: one inverse
//   Jacobian and one point's sums in registers (92 VGPRs, five waves per
//   SIMD; a thread per tet holding four points' took 248, two waves).
// - The results leave through LDS as one contiguous run, in streaming stores
//   (a lane storing its own tet's 288 bytes touches a line of its own in
//   every store).
// A one-point rule has nothing to share: a lane per tet, 256 to a block,
// loads its nodes itself, and the results leave the same way.
// Measured (calls on an order-2 mesh and field, four points): vector fields
// on 5.3M tets 0.77 -> 0.69 ms, the vector ALU 75% busy with the 560 FP64
// operations a point needs and the address unit 78%; matrix fields on 384k
// tets 0.245 -> 0.131 ms, 2.9 TB/s of stores in the kernel (a thread per
// point with run-time orders and 27 strided stores before).
#include "device.h"
#include "spr_math.h"

#include <type_traits>

namespace sprg {
namespace {

constexpr int XCD_K_GRAD = 16384;  // tets per xcd_block chunk: neighbouring tets share nodes

constexpr int grad_points(int ipo) { return ipo <= 1 ? 1 : ipo == 2 ? 4 : 5; }
constexpr int grad_tets(int ipo) { return ipo <= 1 ? 256 : 64; }  // per block
constexpr int grad_threads(int ipo) { return grad_tets(ipo) * grad_points(ipo); }
// waves per SIMD asked for: matrix fields' 27 sums take 144 VGPRs, three
// waves; four, with ten of them spilled, take 131 us a call instead of 134
constexpr int grad_waves(int ipo, int nc) { return ipo == 2 && nc == 9 ? 4 : 1; }

template <int MO, int FO, int IPO, int NCIN>
__global__ __launch_bounds__(grad_threads(IPO), grad_waves(IPO, NCIN)) void k_grad(MeshView m, const double* __restrict__ nodal,
                                                            double* __restrict__ ip)
{
  constexpr int Q = grad_points(IPO), TB = grad_tets(IPO), T = grad_threads(IPO);
  constexpr int NNM = MO == 1 ? 4 : 10;
  constexpr int NNF = FO == 1 ? 4 : 10;
  constexpr int NN = NNM > NNF ? NNM : NNF;
  constexpr int NOUT = 3 * NCIN, R = Q * NOUT, RS = R | 1;  // values per tet, their LDS stride
  // value components gathered at a time; a matrix field's rows take turns
  constexpr int GC = NCIN == 1 ? 1 : 3, NGRP = NCIN / GC;
  constexpr int XD = Q == 1 ? 0 : NNM * 3 * TB, UD = Q == 1 ? 0 : NNF * GC * TB;
  // tets whose results the buffer holds at a time
  constexpr int HELD = Q == 1 ? 2400 : XD + UD;
  constexpr int TO = TB * RS <= HELD ? TB : TB / 2 * RS <= HELD ? TB / 2 : TB / 4;
  constexpr int SD = XD + UD > TO * RS ? XD + UD : TO * RS;
  __shared__ double sm[SD];
  double* const sX = sm;       // [NNM][TB][3]
  double* const sU = sm + XD;  // [NNF][TB][GC]
  const int lt = threadIdx.x % TB;                                             // this thread's tet
  const int pt = Q == 1 ? 0 : __builtin_amdgcn_readlane((int)threadIdx.x / TB, 0);  // its wave's point
  const int64_t t0 = xcd_block(blockIdx.x, gridDim.x, XCD_K_GRAD / TB) * TB;
  const int64_t t = t0 + lt < m.nt ? t0 + lt : m.nt - 1;
  // node ids are 32-bit on any mesh
  auto node_id = [&](int n) {
    const bool vertex = NN == 4 || n < 4;
    const int32_t* const src = vertex ? m.tv + (4 * t + n) : m.te + (6 * t + (n - 4));
    return *src + (vertex ? 0 : (int32_t)m.nv);
  };
  // the wave's nodes: pt, pt + Q, ...
  constexpr int NW = (NN + Q - 1) / Q;
  int32_t node[NW];
  // value 64 r + lane of a node's [TB][G] run: with G = 3
  // three lanes read one node's 24 bytes
  auto fetch = [&](int k, int nn, const double* base, int stride, auto G, double* v) {
    if (Q * (k + 1) <= nn || pt + Q * k < nn) {
#pragma unroll
      for (int r = 0; r < G; ++r) {
        const int f = 64 * r + lt;
        const int64_t id = G == 1 ? node[k] : __shfl(node[k], f / G);
        v[r] = base[id * stride + f % G];
      }
    }
  };
  auto store = [&](int k, int nn, double* dst, auto G, const double* v) {
    if (Q * (k + 1) <= nn || pt + Q * k < nn)
#pragma unroll
      for (int r = 0; r < G; ++r) dst[(pt + Q * k) * (TB * G) + 64 * r + lt] = v[r];
  };
  using G3 = std::integral_constant<int, 3>;
  using GU = std::integral_constant<int, GC>;
  if (Q > 1) {
    // all ids, then all nodes: two round trips to memory
#pragma unroll
    for (int k = 0; k < NW; ++k) node[k] = node_id(pt + Q * k < NN ? pt + Q * k : 0);
    double xv[NW][3], uv[NW][GC];
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      fetch(k, NNM, m.xyz, 3, G3(), xv[k]);
      fetch(k, NNF, nodal, NCIN, GU(), uv[k]);
    }
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      store(k, NNM, sX, G3(), xv[k]);
      store(k, NNF, sU, GU(), uv[k]);
    }
    __syncthreads();
  }
  double out[NGRP][3 * GC];
  double jinv[9];
  // the wave's point as a constant
  auto with_point = [&](auto f) {
    if (Q == 1 || pt == 0) f(std::integral_constant<int, 0>());
    if constexpr (Q > 1) {
      if (pt == 1) f(std::integral_constant<int, 1>());
      if (pt == 2) f(std::integral_constant<int, 2>());
      if (pt == 3) f(std::integral_constant<int, 3>());
    }
    if constexpr (Q > 4)
      if (pt == 4) f(std::integral_constant<int, 4>());
  };
#pragma unroll
  for (int grp = 0; grp < NGRP; ++grp) {
    if (Q > 1 && grp > 0) {
      double uv[NW][GC];
#pragma unroll
      for (int k = 0; k < NW; ++k) fetch(k, NNF, nodal + GC * grp, NCIN, GU(), uv[k]);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < NW; ++k) store(k, NNF, sU, GU(), uv[k]);
      __syncthreads();
    }
    with_point([&](auto point) {
      constexpr int p = decltype(point)::value;
      double xi[3];
      rule_point(IPO, p, xi);
      if (grp == 0) {
        // Jacobian: J[i][j] = x_0[j]*g_0[i], then J = J + x_n[j]*g_n[i]
        double J[9];
#pragma unroll
        for (int n = 0; n < NNM; ++n) {
          double g[3];
          tet_grad(MO, xi, n, g);
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const double x = Q == 1 ? m.xyz[3 * (int64_t)node_id(n) + j] : sX[(n * TB + lt) * 3 + j];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              const double v = x * g[i];
              J[3 * i + j] = n == 0 ? v : J[3 * i + j] + v;
            }
          }
        }
        invert3(J, jinv);
      }
#pragma unroll
      for (int n = 0; n < NNF; ++n) {
        // global shape gradient of field node n
        double lg[3], gg[3];
        tet_grad(FO, xi, n, lg);
#pragma unroll
        for (int i = 0; i < 3; ++i) gg[i] = dot3(jinv + 3 * i, lg);
#pragma unroll
        for (int j = 0; j < GC; ++j) {
          const double u = Q == 1 ? nodal[(int64_t)node_id(n) * NCIN + GC * grp + j] : sU[(n * TB + lt) * GC + j];
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            const double v = NCIN == 1 ? gg[i] * u : u * gg[i];
            out[grp][GC * i + j] = n == 0 ? v : out[grp][GC * i + j] + v;
          }
        }
      }
    });
  }
  // out, tets [o0, o0 + TO) at a time: value k of a point is component
  // GC i + j for scalars and vectors (g[i][j] = du_j / dx_i) and, for matrix
  // value (grp, j), 3 grp + j + 9 d
#pragma unroll 1
  for (int o0 = 0; o0 < TB; o0 += TO) {
    __syncthreads();
    if (lt >= o0 && lt < o0 + TO) {
      double* const dst = sm + (lt - o0) * RS + pt * NOUT;
#pragma unroll
      for (int grp = 0; grp < NGRP; ++grp)
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < GC; ++j)
            dst[NCIN == 9 ? 3 * grp + j + 9 * i : GC * i + j] = out[grp][GC * i + j];
    }
    __syncthreads();
    const int64_t left = m.nt - (t0 + o0);
    const int nval = left <= 0 ? 0 : left >= TO ? TO * R : (int)left * R;
    double* const dst = ip + (t0 + o0) * R;
    auto slot = [](int d) { return d + (RS - R) * (d / R); };
    if constexpr (R % 2 == 0) {
      for (int d = 2 * threadIdx.x; d < nval; d += 2 * T) store_stream2(dst + d, sm[slot(d)], sm[slot(d) + 1]);
    } else {
      for (int d = threadIdx.x; d < nval; d += T) store_stream(dst + d, sm[slot(d)]);
    }
  }
}

template <int MO, int FO, int IPO>
void launch_grad_nc(const MeshView& m, int nc_in, const double* nodal, double* ip, hipStream_t s)
{
  const unsigned blocks = (unsigned)((m.nt + grad_tets(IPO) - 1) / grad_tets(IPO)), threads = grad_threads(IPO);
  if (nc_in == 9)
    k_grad<MO, FO, IPO, 9><<<blocks, threads, 0, s>>>(m, nodal, ip);
  else if constexpr (FO <= MO) {
    if (nc_in == 1)
      k_grad<MO, FO, IPO, 1><<<blocks, threads, 0, s>>>(m, nodal, ip);
    else
      k_grad<MO, FO, IPO, 3><<<blocks, threads, 0, s>>>(m, nodal, ip);
  }
}

template <int MO, int FO>
void launch_grad_ipo(const MeshView& m, int ip_order, int nc_in, const double* nodal, double* ip, hipStream_t s)
{
  if (ip_order <= 1)
    launch_grad_nc<MO, FO, 1>(m, nc_in, nodal, ip, s);
  else if (ip_order == 2)
    launch_grad_nc<MO, FO, 2>(m, nc_in, nodal, ip, s);
  else
    launch_grad_nc<MO, FO, 3>(m, nc_in, nodal, ip, s);
}

}  // namespace

// The caller has checked: nc_in 1, 3 or 9; field order 1 or 2 (2 only on a
// mesh with edges); ip_order 1..3; the mesh order is 1 or 2.
int launch_grad(const MeshView& m, int field_order, int nc_in, const double* nodal,
                int ip_order, double* ip, hipStream_t s)
{
  if (m.nt == 0) return 0;
  if (m.order == 1 && field_order == 2 && nc_in != 9)
    return sprg_fail(SPRG_EINVAL, "getGradIPField: an order-2 field needs mesh edges");
  if (m.order == 1 && field_order == 1)
    launch_grad_ipo<1, 1>(m, ip_order, nc_in, nodal, ip, s);
  else if (m.order == 1)
    launch_grad_ipo<1, 2>(m, ip_order, nc_in, nodal, ip, s);
  else if (field_order == 1)
    launch_grad_ipo<2, 1>(m, ip_order, nc_in, nodal, ip, s);
  else
    launch_grad_ipo<2, 2>(m, ip_order, nc_in, nodal, ip, s);
  return hipGetLastError() == hipSuccess ? 0 : sprg_fail(SPRG_EHIP, "grad launch failed");
}

}  // namespace sprg
