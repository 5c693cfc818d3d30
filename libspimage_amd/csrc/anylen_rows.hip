// Row passes of lines of any length (anylen.h).
#include "anylen.h"

namespace spx {
namespace {

// M-point lines per work-group as the Stockham row passes hold them
template <int M, int E, bool BLUR>
__global__ __launch_bounds__((RowShape<M, E>::NT)) void k_any_row(RowArgs a, AnyLine c, int mode) {
  constexpr int T = RowShape<M, E>::T, G = RowShape<M, E>::M, NT = RowShape<M, E>::NT;
  constexpr int NR = PlanOf<M, E>::NREG;
  using View = LdsView<M, G, false>;
  __shared__ float2 shA[View::SIZE];
  __shared__ float2 shB[SingleBuf<M>::value ? 1 : View::SIZE];
  __shared__ unsigned hsh[BLUR ? 2048 : 1];
  __shared__ float wmax[BLUR ? (NT + 63) / 64 : 1];
  const int tid = threadIdx.x;
  const int g = tid / T, t = tid - g * T;
  const int blk = xcd_tile(blockIdx.x, gridDim.x);
  const int line = blk * G + g;
  const bool act = line < a.nlines;
  const View va{shA, g}, vb{shB, g};
  const long base = (long)(act ? line : a.nlines - 1) * c.L;
  float2 v[NR];
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    const int p = in_pos<M, E>(t, q);
    if (!low_reg<M, E>(q)) continue;
    float2 x = p < c.L ? a.in[base + p] : make_float2(0.f, 0.f);
    if (!BLUR && mode == kRowAbsFwd) x = make_float2(cabsf_ref(x), 0.f);
    v[q] = x;
  }
  TwRegs<M, E> tw;
  load_tw<M, E>(a.tw, t, tw);
  Chirp<M, E> ch;
  ch.load(c, t);
  if constexpr (BLUR) {
    if (a.hist)
      for (int i = tid; i < 2048; i += NT) hsh[i] = 0u;
  }
  any_line<M, E>(v, BLUR || mode == kRowInv, va, vb, t, tw, ch);
  if constexpr (BLUR) {
    blur_out<G, NT>(a, v, blk, line, act, hsh, wmax, [&](int q) { return base + in_pos<M, E>(t, q); },
                    [&](int q) { return low_reg<M, E>(q) && in_pos<M, E>(t, q) < c.L; });
  } else {
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const int p = in_pos<M, E>(t, q);
      if (low_reg<M, E>(q) && act && p < c.L) a.out[base + p] = v[q];
    }
  }
}

// The fused real-space pass: inverse x-transform, update and constraints,
// the new iterate stored, forward x-transform (k_row_update's arithmetic for
// one reconstruction: no alg_rec, beta_rec or rec_active, so batches refuse
// these shapes).
template <int M, int E, bool DM>
__global__ __launch_bounds__((RowShape<M, E>::NT)) void k_any_update(UpdateArgs a, AnyLine c) {
  constexpr int T = RowShape<M, E>::T, G = RowShape<M, E>::M;
  constexpr int NR = PlanOf<M, E>::NREG;
  using View = LdsView<M, G, false>;
  __shared__ float2 shA[View::SIZE];
  __shared__ float2 shB[SingleBuf<M>::value ? 1 : View::SIZE];
  const int tid = threadIdx.x;
  const int g = tid / T, t = tid - g * T;
  const int blk = xcd_tile(blockIdx.x, gridDim.x);
  const int line = blk * G + g;
  const bool act = line < a.nlines;
  const View va{shA, g}, vb{shB, g};
  const long base = (long)(act ? line : a.nlines - 1) * c.L;
  TwRegs<M, E> tw;
  load_tw<M, E>(a.tw, t, tw);
  Chirp<M, E> ch;
  ch.load(c, t);
  float2 v[NR], vf[DM ? NR : 1], g0v[NR];
  bool in[NR], ok[NR];
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    if (!low_reg<M, E>(q)) continue;
    const int p = in_pos<M, E>(t, q);
    ok[q] = p < c.L;
    const long i = base + (ok[q] ? p : 0);
    v[q] = ok[q] ? a.W[i] : make_float2(0.f, 0.f);
    if constexpr (DM) vf[q] = ok[q] ? a.Wf[i] : make_float2(0.f, 0.f);
    g0v[q] = a.gcur[i];
    in[q] = a.flags[i] & kInsideSupport;
  }
  any_line<M, E>(v, true, va, vb, t, tw, ch);
  if constexpr (DM) {
    __syncthreads();
    any_line<M, E>(vf, true, va, vb, t, tw, ch);
  }
  const bool er = !(a.alg == kHIO || a.alg == kRAAR);
  const float beta = a.beta;
  const float cp = a.alg == kHIO ? -beta : 1.f - 2.f * beta;
  const float cg = a.alg == kHIO ? 1.f : beta;
  const SupportConstraints sc(a.constraints);
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    if (!low_reg<M, E>(q)) continue;
    const long i = base + in_pos<M, E>(t, q);
    const float2 P = v[q], g0 = g0v[q];
    float2 g1, gp;
    if constexpr (!DM) {
      // src/phasing.c:1128-1136 (ER), 1160-1168 (HIO), 1194-1215 (RAAR)
      gp = make_float2(P.x * a.scale, P.y * a.scale);
      float2 o = make_float2(fmaf(cp, gp.x, cg * g0.x), fmaf(cp, gp.y, cg * g0.y));
      o = er ? make_float2(0.f, 0.f) : o;
      const float2 gi = sc.apply(gp);
      g1 = make_float2(in[q] ? gi.x : o.x, in[q] ? gi.y : o.y);
    } else {
      // src/phasing.c:1243-1252; gp stays unscaled like the CPU engine
      gp = P;
      const float2 Pf = vf[q];
      const float2 gin = make_float2(g0.x + beta * ((1.f + a.gamma2) * P.x / a.nsize - a.gamma2 * g0.x),
                                     g0.y + beta * ((1.f + a.gamma2) * P.y / a.nsize - a.gamma2 * g0.y));
      g1 = in[q] ? gin : g0;
      g1.x -= beta * Pf.x / a.nsize;
      g1.y -= beta * Pf.y / a.nsize;
      const float2 gc = sc.apply(g1);
      g1 = in[q] ? gc : g1;
      // f1 of the next iteration (src/phasing.c:1260-1274)
      const float2 f1 = in[q] ? g1 : make_float2(-a.gamma1 * g1.x, -a.gamma1 * g1.y);
      vf[q] = ok[q] ? f1 : make_float2(0.f, 0.f);
    }
    if (act && ok[q]) {
      if (a.gp) a.gp[i] = gp;
      a.gnew[i] = g1;
    }
    v[q] = ok[q] ? g1 : make_float2(0.f, 0.f);
  }
  __syncthreads();
  any_line<M, E>(v, false, va, vb, t, tw, ch);
  if constexpr (DM) {
    __syncthreads();
    any_line<M, E>(vf, false, va, vb, t, tw, ch);
  }
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    if (!low_reg<M, E>(q) || !act || !ok[q]) continue;
    const long i = base + in_pos<M, E>(t, q);
    a.W[i] = v[q];
    if constexpr (DM) a.Wf[i] = vf[q];
  }
}

template <int M>
void row_of(const AnyLine& c, int mode, RowArgs a, hipStream_t s) {
  constexpr int E = any_row_elements(M), G = RowShape<M, E>::M;
  a.tw = LengthOps<M, E>::tw();
  const dim3 grid((a.nlines + G - 1) / G), blk(RowShape<M, E>::NT);
  if (mode == kRowBlurOut) hipLaunchKernelGGL((k_any_row<M, E, true>), grid, blk, 0, s, a, c, mode);
  else hipLaunchKernelGGL((k_any_row<M, E, false>), grid, blk, 0, s, a, c, mode);
}

template <int M>
void update_of(const AnyLine& c, UpdateArgs a, bool dm, hipStream_t s) {
  constexpr int E = any_row_elements(M), G = RowShape<M, E>::M;
  a.tw = LengthOps<M, E>::tw();
  const dim3 grid((a.nlines + G - 1) / G), blk(RowShape<M, E>::NT);
  if (dm) hipLaunchKernelGGL((k_any_update<M, E, true>), grid, blk, 0, s, a, c);
  else hipLaunchKernelGGL((k_any_update<M, E, false>), grid, blk, 0, s, a, c);
}

}  // namespace

void any_row(const AnyLine& c, int mode, const RowArgs& a, hipStream_t s) {
#define SPX_CASE(M) \
  case M: row_of<M>(c, mode, a, s); break;
  SPX_ANY_SWITCH(c.M, SPX_CASE)
#undef SPX_CASE
}

void any_update(const AnyLine& c, const UpdateArgs& a, bool dm, hipStream_t s) {
#define SPX_CASE(M) \
  case M: update_of<M>(c, a, dm, s); break;
  SPX_ANY_SWITCH(c.M, SPX_CASE)
#undef SPX_CASE
}

}  // namespace spx
