// Passes of lines of any length up to 4096, by Bluestein's chirp-z method.
//
// The Stockham plans cover products of 2, 3, 5 and 7; FFTW plans every length
// (reference src/fft.c:79,95,163,185).  With w[n] = exp(i pi n^2 / L),
//   X[k] = conj(w[k]) sum_n (x[n] conj(w[n])) w[k - n],
// a circular convolution of length M >= 2L - 1, M a power of two:
// a = x conj(w) padded with zeros, conv = IFFT_M(FFT_M(a) B) with
// B = FFT_M(b) / M of the chirp filter b (w at 0..L-1 and at M-L+1..M-1).
// The inverse transform is the conjugate of the forward one of conj(x).
//
// A pass keeps the padded line on chip from its first transform to its last:
// it reads L elements, does everything in registers and LDS (both transforms
// of length M, the chirps, and between a forward and an inverse transform the
// projection or the update) and writes L elements.  Only the L elements cross
// memory, so a line costs 2 M-point transforms of arithmetic and no padded
// traffic.  As separate element-wise steps and M-point passes on padded
// scratch arrays, one 1021 x 769 HIO iteration took 22 launches and 134-163
// us; the two fused passes take 27 us.  (M = 3 2^k where that is closer
// was tried: even at 768, slower at 3072, whose plans have more stages.)
//
// L <= M / 2, so the upper half of the padded line is zero on input and unused
// on output: of a thread's edge registers only those of the lower half
// (low_reg) hold data.
#pragma once
#include "passes.h"

namespace spx {

// chirp tables of one length, kept for the life of the process
struct AnyLine {
  int L = 0, M = 0;
  const float2* w = nullptr;  // L entries
  const float2* B = nullptr;  // M entries, FFT_M(b) / M
};

// one CASE per padded length of the lines without a Stockham plan (11 .. 4096)
#define SPX_ANY_SWITCH(M, CASE) \
  switch (M) {                  \
    CASE(32) CASE(64) CASE(128) CASE(256) CASE(512) CASE(1024) CASE(2048) CASE(4096) CASE(8192) \
  }

// Plans of the M-point transforms: radix-8 edges.  The row pass of M >= 4096
// gives a line 256 (512) threads of 16 elements instead of 512 (1024) of 8,
// as fewer waves wait at each barrier (1024 x 1031 ER 42 -> 33 us per
// iteration); the column pass would spill (1999 x 1999: 156 us an iteration
// with 8, 185 with the radix-16 plan).  Radix-16 plans were up to 10 % faster
// in rows but less exact: 5 HIO iterations of 1031 x 1024 end 5.8e-7 from
// the float64 result with them, 4.7e-7 with these.
constexpr int any_row_elements(int M) { return M >= 4096 ? 8 + kHalfThreads : 8; }
constexpr int any_col_elements(int) { return 8; }

template <int M, int E>
__device__ __forceinline__ constexpr bool low_reg(int q) {
  return (q % PlanOf<M, E>::E0) < PlanOf<M, E>::E0 / 2;
}

// What one thread multiplies by: the chirp at its lower positions (0 beyond
// the line) and the filter's transform at all of them.
template <int M, int E>
struct Chirp {
  float2 w[PlanOf<M, E>::NREG];
  float2 B[PlanOf<M, E>::NREG];
  __device__ __forceinline__ void load(const AnyLine& c, int t) {
#pragma unroll
    for (int q = 0; q < PlanOf<M, E>::NREG; ++q) {
      const int p = in_pos<M, E>(t, q);
      B[q] = c.B[p];
      if (low_reg<M, E>(q)) w[q] = p < c.L ? c.w[p] : make_float2(0.f, 0.f);
    }
  }
};

__device__ __forceinline__ float2 conj_if(float2 a, bool c) { return make_float2(a.x, c ? -a.y : a.y); }

// L-point transform of a line whose element in_pos(t, q) is v[q] (zero beyond
// L; the upper registers are not read), in place.  Ends like fft_line without
// a barrier.
template <int M, int E, class View>
__device__ __forceinline__ void any_line(RegLine<M, E>& v, bool inverse, const View& a, const View& b, int t,
                                         const TwRegs<M, E>& tw, const Chirp<M, E>& c) {
  constexpr int NR = PlanOf<M, E>::NREG;
  static_assert(PlanOf<M, E>::PAL, "the filter is applied at the input positions");
#pragma unroll
  for (int q = 0; q < NR; ++q) v[q] = low_reg<M, E>(q) ? twmul<+1>(conj_if(v[q], inverse), c.w[q]) : make_float2(0.f, 0.f);
  fft_line<M, E, -1>(v, a, b, t, tw);
#pragma unroll
  for (int q = 0; q < NR; ++q) v[q] = cmul(v[q], c.B[q]);
  __syncthreads();
  fft_line<M, E, +1>(v, a, b, t, tw);
#pragma unroll
  for (int q = 0; q < NR; ++q)
    if (low_reg<M, E>(q)) v[q] = conj_if(twmul<+1>(v[q], c.w[q]), inverse);
}

}  // namespace spx
