// rPIE's per-frame step of small frames of one mode in one workgroup: the exit wave's transform,
// the modulus and the way back (passes A, B and C of the stack) without a stack. The plane fits a
// CU's LDS and a line's values the registers. The three launches of such a batch are chains of
// launch and memory latencies on a chip that is mostly idle: 100 frames of 64² in complex64 took
// 6.9 + 9.4 + 7.6 µs and take 17.2, a call of ten epochs 630 µs and 568. With more modes, one after
// the other in the workgroup, the stack's parallel ones win (64², batches of 128: 2 modes 4 %, 4
// modes 10 % of a call), as they do where the plane needs more than 8 values a thread (96, 128: the
// kernel spills).
#pragma once

#include "kernels.hpp"

namespace ptyrs {

// Every line of the plane at once, N·TL threads.
template <typename T, int N>
using FrameShape = Lines<N, choose_e(N, 8), 1024, N, sizeof(T)>;

// Frame sides it runs at, in float.
template <typename T, int N>
constexpr bool whole_frame() {
  return sizeof(T) == 4 && N >= 32 && N <= 64;
}

// Grid (nb). The threads hold rows (row y, elements jl + TL·e) or columns (column col, elements
// cl + TL·e) of the plane and change over through LDS, whose rows are N + 8 words apart: at 64 the 8
// lanes of 8 rows that a wave writes then meet all 64 banks. The operations are those of k_pass_a,
// k_pass_b<B_RPIE> and k_pass_c_rpie_sum; the regulariser's max is taken from the tiles by every
// workgroup. Slot b's object terms go to plane b of psi, its probe direction to plane b of dP_part
// (one chunk a slot). ptyrs/src/engine/ptycho.rs:900-1086
template <typename T, int N>
__global__ __launch_bounds__((FrameShape<T, N>::NT)) void k_rpie_frame(
    cplx<T>* __restrict__ psi, const cplx<T>* __restrict__ O, int nxo,
    const cplx<T>* __restrict__ Wt, const cplx<T>* __restrict__ q,
    const int2* __restrict__ corner, const int* __restrict__ order,
    const float* __restrict__ counts, const T* __restrict__ D, const T* __restrict__ tilemax,
    int ntile, T obj_alpha, T probe_alpha, int upd_obj, int probe_dir,
    cplx<T>* __restrict__ dP_part, const cplx<T>* __restrict__ tw, T norm) {
  using S = FrameShape<T, N>;
  constexpr int E = S::E, TL = S::TL, NT = S::NT, LD = N + 8;
  constexpr int n = N * N;
  constexpr int W = S::LDS_WORDS > N * LD ? S::LDS_WORDS : N * LD;
  static_assert(S::L == N, "one workgroup holds the plane");
  static_assert(TL > 1, "the transforms' barriers order the planes' changes");
  __shared__ T lre[W], lim[W];
  __shared__ cplx<T> stw[N];
  __shared__ T red[NT];
  const int tid = threadIdx.x;
  const int y = tid / TL, jl = tid % TL, col = tid % N, cl = tid / N;
  const int b = blockIdx.x, f = order[b];
  const int2 c = corner[f];
  const size_t rn = (size_t)(c.x + y) * nxo + c.y + jl;
  const int row = y * N + jl;
  cplx<T> o[E];
#pragma unroll
  for (int e = 0; e < E; ++e) o[e] = ld(O + rn + TL * e);
  float cv[E];
#pragma unroll
  for (int e = 0; e < E; ++e) cv[e] = counts[(size_t)f * n + (cl + TL * e) * N + col];
  T omax = 0, pmax = 0;
  if (upd_obj)
    for (int i = tid; i < ntile; i += NT) pmax = tilemax[i] > pmax ? tilemax[i] : pmax;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const T o2 = norm2(o[e]);
    omax = o2 > omax ? o2 : omax;
  }
  stage_twiddles<T, N, NT>(stw, tw);
  if (probe_dir) omax = block_reduce<NT>(omax, red, MaxOp());
  if (upd_obj) pmax = block_reduce<NT>(pmax, red, MaxOp());
  T* rre = lre + S::base_row(y);
  T* rim = lim + S::base_row(y);
  T* cre = lre + S::base_col(col);
  T* cim = lim + S::base_col(col);
  // A transform leaves LDS free (its last exchange ends with a barrier), and so do the changes.
  cplx<T> v[E];
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = ld(Wt + row + TL * e) * o[e];
  line_fft<T, N, E, false, typename S::AtRow>(v, jl, rre, rim, stw);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    lre[y * LD + jl + TL * e] = v[e].x;
    lim[y * LD + jl + TL * e] = v[e].y;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e)
    v[e] = cplx<T>{lre[(cl + TL * e) * LD + col], lim[(cl + TL * e) * LD + col]};
  __syncthreads();
  line_fft<T, N, E, false, typename S::AtCol>(v, cl, cre, cim, stw);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    T s = norm;
    if (cv[e] >= 0.f)
      s = sqrt(T(cv[e]) + T(1e-7)) / (sqrt(norm2(v[e]) * norm) + T(1e-7)) * norm;
    v[e] = v[e] * s;
  }
  line_fft<T, N, E, true, typename S::AtCol>(v, cl, cre, cim, stw);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    lre[(cl + TL * e) * LD + col] = v[e].x;
    lim[(cl + TL * e) * LD + col] = v[e].y;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e)
    v[e] = cplx<T>{lre[y * LD + jl + TL * e], lim[y * LD + jl + TL * e]};
  __syncthreads();
  line_fft<T, N, E, true, typename S::AtRow>(v, jl, rre, rim, stw);
  const T inv_p = T(1) - probe_alpha, inv_o = T(1) - obj_alpha;
  const T reg = obj_alpha * pmax;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const cplx<T> w = ld(Wt + row + TL * e);
    const cplx<T> d = v[e] - w * o[e];
    if (upd_obj)
      st(psi + (size_t)b * n + row + TL * e,
         cmulc(w, d) * rcp(inv_o * D[rn + TL * e] + reg));
    if (probe_dir)
      st(dP_part + (size_t)b * n + row + TL * e,
         cmulc(ld(q + row + TL * e),
               cmulc(o[e], d) * rcp(inv_p * norm2(o[e]) + probe_alpha * omax)));
  }
}

}  // namespace ptyrs
