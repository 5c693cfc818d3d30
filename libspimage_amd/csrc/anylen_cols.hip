// Column passes of lines of any length (anylen.h), of one reconstruction:
// rec_active is not read, W of an idle slot would be projected in place.
#include "anylen.h"

namespace spx {
namespace {

template <int M, int E, int MODE>
__global__ __launch_bounds__((ColShape<M, E>::NT)) void k_any_col(ColArgs a, AnyLine c, int inverse) {
  constexpr int C = ColShape<M, E>::C, NT = ColShape<M, E>::NT;
  constexpr int NR = PlanOf<M, E>::NREG;
  using View = LdsView<M, C, true>;
  __shared__ float2 shA[View::SIZE];
  __shared__ float2 shB[SingleBuf<M>::value ? 1 : View::SIZE];
  __shared__ double red[(MODE == kColEFourier) ? 4 * 32 : 1];
  const int tid = threadIdx.x;
  const int l = tid % C, t = tid / C;
  const int ngrp = (a.geo.ncontig + C - 1) / C;
  const int blk = xcd_tile(blockIdx.x, gridDim.x);
  const int outer = blk / ngrp;
  const int x = (blk - outer * ngrp) * C + l;
  const bool act = x < a.geo.ncontig;
  const long base = (long)outer * a.geo.outer_stride + (act ? x : a.geo.ncontig - 1);
  const long st = a.geo.axis_stride;
  const View va{shA, l}, vb{shB, l};
  float2 v[NR];
  float ampv[NR];
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    if (!low_reg<M, E>(q)) continue;
    const int p = in_pos<M, E>(t, q);
    v[q] = p < c.L ? a.in[base + p * st] : make_float2(0.f, 0.f);
  }
  TwRegs<M, E> tw;
  load_tw<M, E>(a.tw, t, tw);
  Chirp<M, E> ch;
  ch.load(c, t);
  if constexpr (MODE == kColProject || MODE == kColEFourier) {
    if (MODE == kColEFourier || a.objective == 0) {
#pragma unroll
      for (int q = 0; q < NR; ++q) {
        if (!low_reg<M, E>(q)) continue;
        const int p = in_pos<M, E>(t, q);
        ampv[q] = a.ampx[base + (p < c.L ? p : 0) * st];
      }
    }
  }
  any_line<M, E>(v, MODE == kColFwd && inverse, va, vb, t, tw, ch);
  if constexpr (MODE == kColProject) {
    const bool plain = a.objective == 0 && !a.margin;
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      if (!low_reg<M, E>(q)) continue;
      const int p = in_pos<M, E>(t, q);
      const bool ok = p < c.L;
      float2 G = v[q];
      if (plain) {
        G = project_phase(G, ampv[q], a.centro != 0);
      } else if (ok) {
        const long idx = base + p * st;
        if (a.centro) G.y = 0.f;  // src/phasing.c:1061-1068
        if (a.objective == 0) {
          G = project_pixel(G, ampv[q], a, idx);
        } else {
          // src/phasing.c:1103-1109
          const float2 P = a.phased_amp[idx];
          if (__float_as_uint(P.x) != kUnmeasuredBits) G = P;
        }
      }
      v[q] = ok ? G : make_float2(0.f, 0.f);
    }
    __syncthreads();
    any_line<M, E>(v, true, va, vb, t, tw, ch);
  } else if constexpr (MODE == kColBlur) {
    const BlurLine blur(a, base);
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      if (!low_reg<M, E>(q)) continue;
      const int p = in_pos<M, E>(t, q);
      const float h = p < c.L ? blur.at(p) : 0.f;
      v[q] = p < c.L ? make_float2(v[q].x * h, v[q].y * h) : make_float2(0.f, 0.f);
    }
    __syncthreads();
    any_line<M, E>(v, true, va, vb, t, tw, ch);
  } else if constexpr (MODE == kColEFourier) {
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const int p = in_pos<M, E>(t, q);
      if (!low_reg<M, E>(q) || !act || p >= c.L) continue;
      if (a.fout) a.fout[base + p * st] = v[q];
      efourier_add(v[q], ampv[q], acc);
    }
    block_sum<4, NT>(acc, red);
    if (tid == 0) {
#pragma unroll
      for (int k = 0; k < 4; ++k) a.partials[(long)blk * 4 + k] = acc[k];
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    const int p = in_pos<M, E>(t, q);
    if (low_reg<M, E>(q) && act && p < c.L) a.W[base + p * st] = v[q];
  }
}

template <int M>
int blocks_of(const LineGeom& g) {
  constexpr int C = ColShape<M, any_col_elements(M)>::C;
  return ((g.ncontig + C - 1) / C) * g.nouter;
}

template <int M>
void col_of(const AnyLine& c, int mode, ColArgs a, hipStream_t s) {
  constexpr int E = any_col_elements(M);
  a.tw = LengthOps<M, E>::tw();
  const dim3 grid(blocks_of<M>(a.geo)), blk(ColShape<M, E>::NT);
  switch (mode) {
    case kColFwd: hipLaunchKernelGGL((k_any_col<M, E, kColFwd>), grid, blk, 0, s, a, c, 0); break;
    case kColInv: hipLaunchKernelGGL((k_any_col<M, E, kColFwd>), grid, blk, 0, s, a, c, 1); break;
    case kColProject: hipLaunchKernelGGL((k_any_col<M, E, kColProject>), grid, blk, 0, s, a, c, 0); break;
    case kColEFourier: hipLaunchKernelGGL((k_any_col<M, E, kColEFourier>), grid, blk, 0, s, a, c, 0); break;
    case kColBlur: hipLaunchKernelGGL((k_any_col<M, E, kColBlur>), grid, blk, 0, s, a, c, 0); break;
  }
}

}  // namespace

void any_col(const AnyLine& c, int mode, const ColArgs& a, hipStream_t s) {
#define SPX_CASE(M) \
  case M: col_of<M>(c, mode, a, s); break;
  SPX_ANY_SWITCH(c.M, SPX_CASE)
#undef SPX_CASE
}

int any_col_blocks(const AnyLine& c, const LineGeom& g) {
#define SPX_CASE(M) \
  case M: return blocks_of<M>(g);
  SPX_ANY_SWITCH(c.M, SPX_CASE)
#undef SPX_CASE
  return 0;
}

}  // namespace spx
