// Two-pass iterations of volumes: the 3-D transform split between a pass over
// (x, part of y) tiles and a pass over (z, the rest of y) tiles.
//
// One pass per axis moves W six times an iteration (x, y, z with the
// projection, y): 85 bytes a voxel with the iterates, amplitudes and flags.
// Here ny = 8 A and y = 8 a + b, and the y transform is split as
//   X[c + A d] = sum_b w_8^{b d} w_ny^{b c} sum_a w_A^{a c} x[8 a + b]:
//
//   real-space pass (k_vol_row), tiles of fixed z and b: the rows y = 8 a + b.
//     Inverse x, the rest of the inverse y (A-point transforms over c, after
//     the twiddles), update, constraints, the new iterate stored, and the
//     same forward.  Row c of the result is kept as row y' = 8 c + b of W.
//   Fourier-space pass (k_vol_col), tiles of fixed c and C adjacent x: the 8
//     rows y' = 8 c + b of every z.  Forward z, 8-point transforms over b,
//     projection, and back.
//
// Both passes read and write W in place, 53 bytes a voxel in two launches
// instead of four (the difference map: 89 instead of 154; counted at 256^3
// 53.7 and 107.9, as the difference map's row kernel spills 31 registers).
// HBM bounds them at 256^3 (a large copy moves 4.7 TB/s, so 190 us for an ER
// iteration beyond the Infinity Cache), the Infinity Cache and the arithmetic
// (100 instructions a voxel and pass) below.  Microseconds per HIO iteration of
// one reconstruction before and after: 64^3 14.0 -> 12.7, 80^3 20.1 both, 96^3
// 26.2 -> 25.6, 120^3 61 -> 32, 128^3 45 -> 31, 144^3 52 -> 46, 160^3 80 -> 70,
// 192^3 106 -> 97, 200^3 124 -> 106, 216^3 190 -> 165, 240^3 238 -> 180, 256^3
// 214 -> 174; difference map 64^3 26.6 -> 18.2, 128^3 88 -> 56, 256^3 465 ->
// 411; batches of 8 96^3 113 -> 78, 128^3 226 -> 161.
//
// The split: tiles of 64 KiB and less, so that two or more work-groups share
// a CU and one loads while another transforms.  At 256^3 the row tile is 32 x
// 256 and the column tile 8 x 256 x 4; a smaller A would make the column tile
// too large for two work-groups, and columns of 2 would waste the 128-byte
// lines (tile patterns without arithmetic: C = 4 6.0 TB/s, 4096-point columns
// with C = 2 2.2 TB/s).  Up to 128 the column tiles are also 4 wide: 96^3 x 8
// 49 us a pass with C = 8 (two work-groups of 56 KiB a CU), 32 us with 4.
//
// Instances exist for the lengths of vol_cfg (multiples of 8 from 64 to 256
// without a factor 7): the row pass for nx = ny = L, the column pass for nz = L.
// Other volumes, all with ny != nx among them, keep the passes per axis.
#pragma once
#include "passes.h"

#include <type_traits>

namespace spx {

struct VolCfg {
  int nline, line[3];  // radices of an x or z line, first stage first
  int ny, y[2];        // radices of the A-point part of y (inverse order)
  int rb, nt_row;      // row pass: adjacent b per work-group, threads
  int C, nt_col;       // column pass: adjacent x per work-group, threads
};

// Work-group sizes keep the butterflies of the widest stages at a whole
// number per thread, about 16 elements each (192: 512 threads for the column
// tile's 512 radix-12 butterflies; 192^3 HIO took 115 us with 384, 97 now).
constexpr VolCfg vol_cfg(int L) {
  switch (L) {
    case 64: return {2, {8, 8, 1}, 1, {8, 1}, 4, 256, 4, 256};
    case 72: return {2, {8, 9, 1}, 1, {9, 1}, 2, 162, 4, 144};
    case 80: return {2, {8, 10, 1}, 1, {10, 1}, 2, 200, 4, 160};
    case 96: return {2, {8, 12, 1}, 1, {12, 1}, 2, 192, 4, 192};
    case 120: return {2, {8, 15, 1}, 1, {15, 1}, 2, 256, 4, 256};
    case 128: return {2, {8, 16, 1}, 1, {16, 1}, 2, 256, 4, 256};
    case 144: return {2, {12, 12, 1}, 2, {6, 3}, 1, 216, 4, 192};
    case 160: return {2, {10, 16, 1}, 2, {5, 4}, 1, 320, 4, 256};
    case 192: return {2, {12, 16, 1}, 2, {6, 4}, 1, 384, 4, 512};
    case 200: return {3, {8, 5, 5}, 2, {5, 5}, 1, 512, 4, 448};
    case 216: return {3, {6, 6, 6}, 2, {9, 3}, 1, 512, 4, 384};
    case 240: return {2, {15, 16, 1}, 2, {6, 5}, 1, 480, 4, 512};
    case 256: return {2, {16, 16, 1}, 2, {8, 4}, 1, 512, 4, 512};
    default: return {};
  }
}
constexpr int kVolB = 8;

// Twiddles of length L, one table: exp(-2 pi i j k / (Ns R)) at
// (k - 1) Ns + j for the line's stages after the first, for the second stage
// of the A-point transform in inverse and in forward order, then
// exp(-2 pi i b c / ny) at b A + c.
constexpr int vol_line_ns(int L, int s) {
  int n = 1;
  for (int i = 0; i < s; ++i) n *= vol_cfg(L).line[i];
  return n;
}
constexpr int vol_line_off(int L, int s) {
  int o = 0;
  for (int i = 1; i < s; ++i) o += vol_line_ns(L, i) * (vol_cfg(L).line[i] - 1);
  return o;
}
constexpr int vol_yinv_off(int L) { return vol_line_off(L, vol_cfg(L).nline); }
constexpr int vol_yfwd_off(int L) { return vol_yinv_off(L) + vol_cfg(L).y[0] * (vol_cfg(L).y[1] - 1); }
constexpr int vol_split_off(int L) { return vol_yfwd_off(L) + vol_cfg(L).y[1] * (vol_cfg(L).y[0] - 1); }
constexpr int vol_table_size(int L) { return vol_split_off(L) + L; }

// Fourier-space layout of the amplitudes (and margins, phased amplitudes):
// the order in which the column pass reads them, [tile (c, x / C)][d][z][x % C].
// j: natural index (z, y, x) of one reconstruction; y = c + A d.
__host__ __device__ __forceinline__ long vol_amp_index(long j, int nx, int ny, int nz, int C) {
  const int A = ny / kVolB;
  const int x = (int)(j % nx);
  const long r = j / nx;
  const int y = (int)(r % ny), z = (int)(r / ny);
  const int c = y % A, d = y / A;
  return (((long)(c * (nx / C) + x / C) * kVolB + d) * nz + z) * C + x % C;
}

enum VolRowMode : int { kVolUpdate = 0, kVolUpdateDM = 1, kVolFwd = 2, kVolFwdF1 = 3 };

struct VolRowArgs {
  UpdateArgs u;      // kVolFwd*: gcur -> W (kVolFwdF1: f1 of gcur -> W)
  const float2* tw;  // table of nx
  int nz;
  int nplanes;       // nz * reconstructions
};
struct VolColArgs {
  ColArgs a;         // W, amplitudes, ... ; geometry below
  float2* W2;        // difference map: f1's array, projected by the grid's second row
  const float2* tw;  // table of nz
  int nx, ny;
  int nrec;
};

struct VolOps {
  int L;
  int C;
  void (*row)(int mode, const VolRowArgs&, hipStream_t);
  void (*col)(int mode, const VolColArgs&, hipStream_t);  // kColProject or kColEFourier
};
// null where the length has no instance
const VolOps* vol_ops(int L);
// device table of length L (engine.hip); null on a device error
const float2* vol_table(int L);

// f(i, n) for the butterflies n = tid + i NT < N of a stage
template <int N, int NT, class F>
__device__ __forceinline__ void each_of(int tid, F&& f) {
#pragma unroll
  for (int i = 0; i < (N + NT - 1) / NT; ++i) {
    const int n = tid + i * NT;
    if ((i + 1) * NT <= N || n < N) f(i, n);
  }
}
template <int N, int NT>
constexpr int per_thread = (N + NT - 1) / NT;

// element i of an array at a uniform address: the byte offset stays in 32
// bits, so that it is one register beside a scalar base (64-bit addresses of
// all of a thread's elements, kept for the stores, would be 32 or more)
template <class T>
__device__ __forceinline__ T& el(T* base, unsigned i) {
  return *reinterpret_cast<T*>(reinterpret_cast<std::conditional_t<std::is_const_v<T>, const char, char>*>(base) +
                               i * (unsigned)sizeof(T));
}

// The thread index as a value of its own for each stage: otherwise the
// stages' LDS and global offsets, which only depend on it, are computed once
// and kept in registers from the inverse transforms to the forward ones.
__device__ __forceinline__ int fresh(int tid) {
  asm volatile("" : "+v"(tid));
  return tid;
}

template <int R, int NS, int DIR>
__device__ __forceinline__ void stage_tw(float2* x, const float2* tw, int j) {
#pragma unroll
  for (int k = 1; k < R; ++k) x[k] = twmul<DIR>(x[k], tw[(k - 1) * NS + j]);
}

// waves on a SIMD when the CU holds as many work-groups as its LDS takes, at
// most 4 (128 registers a thread): the compiler is held to it
constexpr int waves_per_simd(int lds_bytes, int threads) {
  const int groups = 160 * 1024 / lds_bytes;
  const int waves = groups * ((threads + 63) / 64) / 4;
  return waves < 1 ? 1 : waves > 4 ? 4 : waves;
}

// ---------------------------------------------------------------------------
// real-space pass
// ---------------------------------------------------------------------------
template <int L>
struct VolRow {
  static constexpr VolCfg K = vol_cfg(L);
  static constexpr int A = L / kVolB, RB = K.rb, ROWS = A * RB, NT = K.nt_row;
  // one slot of padding after every PAD positions: 8 where every stage's
  // read stride is a multiple of it (slot offsets are then constants, see
  // slot()), else 16 like LdsView
  static constexpr bool pad8() {
    for (int i = 0; i < K.nline; ++i)
      if ((L / K.line[i]) % 16 == 8) return true;
    return false;
  }
  static constexpr int PAD = pad8() ? 8 : 16;
  static constexpr int LP = (L + L / PAD) | 1;
  // slot of base + off, base a multiple of MB and off a constant: the slot of
  // base plus a constant where the padding before them adds up
  template <int MB>
  __device__ static __forceinline__ int slot(int base, int off) {
    if (off % PAD == 0 || MB % PAD == 0 || (PAD % MB == 0 && off < MB)) return base + base / PAD + off + off / PAD;
    return base + off + (base + off) / PAD;
  }
  static constexpr int SIZE = ROWS * LP;
  // two buffers (one barrier per exchange) while four work-groups still fit
  static constexpr int NBUF = 2 * SIZE * 8 <= 38 * 1024 ? 2 : 1;
  static constexpr int YL = K.ny == 2 ? K.y[1] : K.y[0];  // radix next to the update
  static constexpr int NY = RB * (A / YL) * L;            // its butterflies
  static constexpr int IY = per_thread<NY, NT>;
  static_assert(IY * YL <= 32, "the support bits of a thread fit a word");
  // the radix-16 rows of 128 need 166 registers: held to the 128 of a fourth
  // wave they spill (128^3 HIO 31.5 -> 38.8 us, batches of 8 161 -> 245)
  static constexpr int WPE = L == 128 ? 3 : waves_per_simd((NBUF * SIZE + vol_table_size(L)) * 8, NT);
};

// the work-group's LDS tile: exchanges alternate over the buffers
template <int L>
struct VolTile {
  using R = VolRow<L>;
  float2* sh;
  int cur = 0;
  template <int MB = 1>
  __device__ __forceinline__ float2& at(int row, int x, int off = 0) {
    return sh[cur * R::SIZE + row * R::LP + R::template slot<MB>(x, off)];
  }
  // after every thread's writes
  __device__ __forceinline__ void written() { __syncthreads(); }
  // after a stage's reads, before its writes
  __device__ __forceinline__ void read() {
    if constexpr (R::NBUF == 2) cur ^= 1;
    else __syncthreads();
  }
};

// The x transform of the tile's rows, from stage S on.  Inverse: from global
// rows (ld(row, x)) into the tile; forward: from the tile to global rows
// (st(row, x, value)).
template <int L, int DIR, int S, class Io>
__device__ __forceinline__ void vol_x_stages(VolTile<L>& tile, int tid, const float2* tw, Io&& io) {
  using R = VolRow<L>;
  constexpr int RX = R::K.line[S], NS = vol_line_ns(L, S), NB = L / RX, N = R::ROWS * NB;
  constexpr bool gin = S == 0 && DIR > 0, last = S == R::K.nline - 1, gout = last && DIR < 0;
  float2 v[per_thread<N, R::NT>][RX];
  tid = fresh(tid);
  each_of<N, R::NT>(tid, [&](int i, int n) {
    const int row = n / NB, j = n % NB;
#pragma unroll
    for (int k = 0; k < RX; ++k) {
      if constexpr (gin) v[i][k] = io(row, j + k * NB);
      else v[i][k] = tile.at(row, j, k * NB);
    }
  });
  if constexpr (!gin) tile.read();
  each_of<N, R::NT>(tid, [&](int i, int n) {
    const int row = n / NB, j = n % NB, jj = j % NS;
    if constexpr (S > 0) stage_tw<RX, NS, DIR>(v[i], tw + vol_line_off(L, S), jj);
    dft<RX, DIR, true>(v[i]);
    const int o = (j - jj) * RX + jj;
#pragma unroll
    for (int r = 0; r < RX; ++r) {
      if constexpr (gout) io(row, o + r * NS, v[i][r]);
      else tile.template at<S == 0 ? RX : 1>(row, o, r * NS) = v[i][r];
    }
  });
  if constexpr (!gout) tile.written();
  if constexpr (!last) vol_x_stages<L, DIR, S + 1>(tile, tid, tw, io);
}

// butterfly n of a y stage of radix RY: column x, b offset rb, index j; its
// element k is tile row (j + k A / RY) RB + rb
template <int L, int RY>
struct VolYFly {
  int x, rb, j;
  __device__ __forceinline__ explicit VolYFly(int n) {
    x = n % L;
    const int m = n / L;
    rb = m % VolRow<L>::RB;
    j = m / VolRow<L>::RB;
  }
};

// From the tile (rows c, x transformed back) to the registers of the last
// inverse y stage: v[i][r] is row a = j + r A / YL of butterfly (i).
template <int L>
__device__ __forceinline__ void vol_y_inverse(VolTile<L>& tile, int tid, int b0, const float2* tw,
                                              float2 (&v)[VolRow<L>::IY][VolRow<L>::YL]) {
  using R = VolRow<L>;
  constexpr int A = R::A, RB = R::RB, YL = R::YL;
  const float2* split = tw + vol_split_off(L);
  tid = fresh(tid);
  if constexpr (R::K.ny == 2) {
    constexpr int Y0 = R::K.y[0], N = RB * (A / Y0) * L;
    float2 u[per_thread<N, R::NT>][Y0];
    each_of<N, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, Y0> f(n);
#pragma unroll
      for (int k = 0; k < Y0; ++k) u[i][k] = tile.at((f.j + k * (A / Y0)) * RB + f.rb, f.x);
    });
    tile.read();
    each_of<N, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, Y0> f(n);
#pragma unroll
      for (int k = 0; k < Y0; ++k) u[i][k] = twmul<+1>(u[i][k], split[(b0 + f.rb) * A + f.j + k * (A / Y0)]);
      dft<Y0, +1, true>(u[i]);
#pragma unroll
      for (int r = 0; r < Y0; ++r) tile.at((f.j * Y0 + r) * RB + f.rb, f.x) = u[i][r];
    });
    tile.written();
    each_of<R::NY, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, YL> f(n);
#pragma unroll
      for (int k = 0; k < YL; ++k) v[i][k] = tile.at((f.j + k * (A / YL)) * RB + f.rb, f.x);
    });
    tile.read();
    each_of<R::NY, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, YL> f(n);
      stage_tw<YL, Y0, +1>(v[i], tw + vol_yinv_off(L), f.j);
      dft<YL, +1, true>(v[i]);
    });
  } else {
    each_of<R::NY, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, YL> f(n);
#pragma unroll
      for (int k = 0; k < YL; ++k) v[i][k] = tile.at(k * RB + f.rb, f.x);
    });
    tile.read();
    each_of<R::NY, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, YL> f(n);
#pragma unroll
      for (int k = 0; k < YL; ++k) v[i][k] = twmul<+1>(v[i][k], split[(b0 + f.rb) * A + k]);
      dft<YL, +1, true>(v[i]);
    });
  }
}

// The forward counterpart: from those registers to the tile's rows c, ready
// for the x stages.
template <int L>
__device__ __forceinline__ void vol_y_forward(VolTile<L>& tile, int tid, int b0, const float2* tw,
                                              float2 (&v)[VolRow<L>::IY][VolRow<L>::YL]) {
  using R = VolRow<L>;
  constexpr int A = R::A, RB = R::RB, YL = R::YL;
  const float2* split = tw + vol_split_off(L);
  tid = fresh(tid);
  if constexpr (R::K.ny == 2) {
    constexpr int Y0 = R::K.y[0], N = RB * (A / Y0) * L;
    each_of<R::NY, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, YL> f(n);
      dft<YL, -1, true>(v[i]);
#pragma unroll
      for (int r = 0; r < YL; ++r) tile.at((f.j * YL + r) * RB + f.rb, f.x) = v[i][r];
    });
    tile.written();
    float2 u[per_thread<N, R::NT>][Y0];
    each_of<N, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, Y0> f(n);
#pragma unroll
      for (int k = 0; k < Y0; ++k) u[i][k] = tile.at((f.j + k * (A / Y0)) * RB + f.rb, f.x);
    });
    tile.read();
    each_of<N, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, Y0> f(n);
      stage_tw<Y0, YL, -1>(u[i], tw + vol_yfwd_off(L), f.j);
      dft<Y0, -1, true>(u[i]);
#pragma unroll
      for (int r = 0; r < Y0; ++r) {
        const int c = f.j + r * YL;
        tile.at(c * RB + f.rb, f.x) = twmul<-1>(u[i][r], split[(b0 + f.rb) * A + c]);
      }
    });
  } else {
    each_of<R::NY, R::NT>(tid, [&](int i, int n) {
      const VolYFly<L, YL> f(n);
      dft<YL, -1, true>(v[i]);
#pragma unroll
      for (int c = 0; c < YL; ++c) tile.at(c * RB + f.rb, f.x) = twmul<-1>(v[i][c], split[(b0 + f.rb) * A + c]);
    });
  }
  tile.written();
}

template <int L, int MODE>
__global__ __launch_bounds__((VolRow<L>::NT), (VolRow<L>::WPE)) void k_vol_row(VolRowArgs p) {
  using R = VolRow<L>;
  constexpr int A = R::A, RB = R::RB, NT = R::NT, IY = R::IY, YL = R::YL, NY = R::NY;
  constexpr bool DM = MODE == kVolUpdateDM, FWD = MODE == kVolFwd || MODE == kVolFwdF1;
  __shared__ float2 sh[R::NBUF * R::SIZE];
  __shared__ float2 tw[vol_table_size(L)];
  const UpdateArgs& a = p.u;
  const int tid = threadIdx.x;
  const int blk = xcd_tile(blockIdx.x, gridDim.x);
  const int plane = blk / (kVolB / RB), b0 = (blk - plane * (kVolB / RB)) * RB;
  const int rec = plane / p.nz;
  // tile row c RB + rb is row 8 c + b0 + rb of the plane, in W and (c read as
  // a) in the iterates
  const long base = (long)plane * (L * L) + (long)b0 * L;
  auto row_of = [&](int rr) -> unsigned { return (RB == 1 ? rr * kVolB : (rr / RB) * kVolB + rr % RB) * L; };
  if (!FWD && a.rec_active) {
    const uint8_t st = a.rec_active[rec];
    if (st != kSlotActive) {
      // kSlotIdle reconstructions keep their state (the iterate is carried
      // over to the other ping-pong buffer); kSlotVacant ones are skipped
      if (st == kSlotIdle)
        for (int i = tid; i < R::ROWS * L; i += NT) {
          const long k = base + row_of(i / L) + i % L;
          a.gnew[k] = a.gcur[k];
        }
      return;
    }
  }
  // twiddles from LDS: read from global memory, each stage would wait for
  // its own behind the barrier before it
  for (int i = tid; i < vol_table_size(L); i += NT) tw[i] = p.tw[i];
  VolTile<L> tile{sh};
  float2 v[IY][YL], vf[DM ? IY : 1][YL], g0[IY][YL];
  uint8_t fl[IY][YL];
  auto at = [&](int n, int k) -> unsigned {
    const VolYFly<L, YL> f(n);
    return row_of((f.j + k * (A / YL)) * RB + f.rb) + f.x;
  };
  const float2* gcur = a.gcur + base;
  // the update's operands: loaded early, they arrive during the inverse
  // transforms, where there are registers to keep them in meanwhile
  auto operands = [&] {
    const int tid = fresh(threadIdx.x);
    if (!FWD && (a.nt & 4)) {
      each_of<NY, NT>(tid, [&](int i, int n) {
#pragma unroll
        for (int k = 0; k < YL; ++k) g0[i][k] = ld_nt(&el(gcur, at(n, k)));
      });
    } else {
      each_of<NY, NT>(tid, [&](int i, int n) {
#pragma unroll
        for (int k = 0; k < YL; ++k) g0[i][k] = el(gcur, at(n, k));
      });
    }
    if constexpr (MODE != kVolFwd)
      each_of<NY, NT>(tid, [&](int i, int n) {
#pragma unroll
        for (int k = 0; k < YL; ++k) fl[i][k] = el(a.flags + base, at(n, k));
      });
  };
  constexpr bool early = !DM && IY * YL <= 12;
  if constexpr (FWD || early) operands();
  if constexpr (FWD) {
    each_of<NY, NT>(tid, [&](int i, int n) {
#pragma unroll
      for (int k = 0; k < YL; ++k) {
        const float2 g = g0[i][k];
        if constexpr (MODE == kVolFwd) v[i][k] = g;
        else v[i][k] = (fl[i][k] & kInsideSupport) ? g : make_float2(-a.gamma1 * g.x, -a.gamma1 * g.y);
      }
    });
  } else {
    const float2* W = a.W + base;
    vol_x_stages<L, +1, 0>(tile, tid, tw, [&](int rr, int x) { return el(W, row_of(rr) + x); });
    vol_y_inverse<L>(tile, tid, b0, tw, v);
    if constexpr (!early) operands();
    const float beta = a.beta_rec ? a.beta_rec[rec] : a.beta;
    const SupportConstraints sc(a.constraints);
    if (a.gp)
      each_of<NY, NT>(tid, [&](int i, int n) {
#pragma unroll
        for (int k = 0; k < YL; ++k)
          el(a.gp + base, at(n, k)) = DM ? v[i][k] : make_float2(v[i][k].x * a.scale, v[i][k].y * a.scale);
      });
    if constexpr (!DM) {
      const int alg = a.alg_rec ? a.alg_rec[rec] : a.alg;
      const bool er = !(alg == kHIO || alg == kRAAR);
      const float cp = alg == kHIO ? -beta : 1.f - 2.f * beta;
      const float cg = alg == kHIO ? 1.f : beta;
      each_of<NY, NT>(tid, [&](int i, int) {
#pragma unroll
        for (int k = 0; k < YL; ++k) {
          // src/phasing.c:1128-1136 (ER), 1160-1168 (HIO), 1194-1215 (RAAR)
          const float2 P = v[i][k], g = g0[i][k];
          const bool in = fl[i][k] & kInsideSupport;
          const float2 gp = make_float2(P.x * a.scale, P.y * a.scale);
          float2 o = make_float2(fmaf(cp, gp.x, cg * g.x), fmaf(cp, gp.y, cg * g.y));
          o = er ? make_float2(0.f, 0.f) : o;
          const float2 gi = sc.apply(gp);
          v[i][k] = make_float2(in ? gi.x : o.x, in ? gi.y : o.y);
        }
      });
    } else {
      // src/phasing.c:1243-1252; gp stays unscaled like the CPU engine.  The
      // part without f1 first, so that the iterate's registers are free
      // during f1's transforms
      unsigned inside = 0;
      each_of<NY, NT>(tid, [&](int i, int) {
#pragma unroll
        for (int k = 0; k < YL; ++k) {
          const float2 P = v[i][k], g = g0[i][k];
          const bool in = fl[i][k] & kInsideSupport;
          const float2 gin = make_float2(g.x + beta * ((1.f + a.gamma2) * P.x / a.nsize - a.gamma2 * g.x),
                                         g.y + beta * ((1.f + a.gamma2) * P.y / a.nsize - a.gamma2 * g.y));
          v[i][k] = in ? gin : g;
          inside |= in ? 1u << (i * YL + k) : 0u;
        }
      });
      const float2* Wf = a.Wf + base;
      vol_x_stages<L, +1, 0>(tile, tid, tw, [&](int rr, int x) { return el(Wf, row_of(rr) + x); });
      vol_y_inverse<L>(tile, tid, b0, tw, vf);
      each_of<NY, NT>(tid, [&](int i, int) {
#pragma unroll
        for (int k = 0; k < YL; ++k) {
          const bool in = inside & (1u << (i * YL + k));
          float2 g1 = v[i][k];
          g1.x -= beta * vf[i][k].x / a.nsize;
          g1.y -= beta * vf[i][k].y / a.nsize;
          const float2 gc = sc.apply(g1);
          g1 = in ? gc : g1;
          v[i][k] = g1;
          // f1 of the next iteration (src/phasing.c:1260-1274)
          vf[i][k] = in ? g1 : make_float2(-a.gamma1 * g1.x, -a.gamma1 * g1.y);
        }
      });
    }
    const int tid = fresh(threadIdx.x);
    if (a.nt & 8) {
      each_of<NY, NT>(tid, [&](int i, int n) {
#pragma unroll
        for (int k = 0; k < YL; ++k) st_nt(&el(a.gnew + base, at(n, k)), v[i][k]);
      });
    } else {
      each_of<NY, NT>(tid, [&](int i, int n) {
#pragma unroll
        for (int k = 0; k < YL; ++k) el(a.gnew + base, at(n, k)) = v[i][k];
      });
    }
  }
  float2* W = a.W + base;
  if constexpr (FWD) __syncthreads();  // the twiddles
  vol_y_forward<L>(tile, tid, b0, tw, v);
  vol_x_stages<L, -1, 0>(tile, tid, tw, [&](int rr, int x, float2 y) { el(W, row_of(rr) + x) = y; });
  if constexpr (DM) {
    float2* Wf = a.Wf + base;
    vol_y_forward<L>(tile, tid, b0, tw, vf);
    vol_x_stages<L, -1, 0>(tile, tid, tw, [&](int rr, int x, float2 y) { el(Wf, row_of(rr) + x) = y; });
  }
}

// ---------------------------------------------------------------------------
// Fourier-space pass
// ---------------------------------------------------------------------------
template <int L>
struct VolCol {
  static constexpr VolCfg K = vol_cfg(L);
  static constexpr int C = K.C, NT = K.nt_col, G = kVolB * C;  // G lines of z
  static constexpr int P = G + C;  // pitch of one z: C columns of padding keep the b stage off one bank
  static constexpr int SIZE = L * P;
  static constexpr int WPE = waves_per_simd((SIZE + vol_yinv_off(L)) * 8, NT);
};

// z stages S.. of the tile's 8 C lines in LDS (one buffer: a stage reads,
// synchronises, writes).  Forward: from global memory into the tile; inverse:
// from the tile to global memory.
template <int L, int DIR, int S>
__device__ __forceinline__ void vol_z_stages(float2* sh, int tid, const float2* tw, float2* W, unsigned plane,
                                             unsigned nx) {
  using R = VolCol<L>;
  constexpr int C = R::C, G = R::G, P = R::P;
  constexpr int RZ = R::K.line[S], NS = vol_line_ns(L, S), NB = L / RZ, N = G * NB;
  constexpr bool gin = S == 0 && DIR < 0, last = S == R::K.nline - 1, gout = last && DIR > 0;
  float2 v[per_thread<N, R::NT>][RZ];
  tid = fresh(tid);
  each_of<N, R::NT>(tid, [&](int i, int n) {
    const int g = n % G, j = n / G;
#pragma unroll
    for (int k = 0; k < RZ; ++k) {
      if constexpr (gin) v[i][k] = el(W, (j + k * NB) * plane + (g / C) * nx + g % C);
      else v[i][k] = sh[(j + k * NB) * P + g];
    }
  });
  if constexpr (!gin) __syncthreads();
  each_of<N, R::NT>(tid, [&](int i, int n) {
    const int g = n % G, j = n / G, jj = j % NS;
    if constexpr (S > 0) stage_tw<RZ, NS, DIR>(v[i], tw + vol_line_off(L, S), jj);
    dft<RZ, DIR, true>(v[i]);
    const int o = (j - jj) * RZ + jj;
#pragma unroll
    for (int r = 0; r < RZ; ++r) {
      if constexpr (gout) el(W, (o + r * NS) * plane + (g / C) * nx + g % C) = v[i][r];
      else sh[(o + r * NS) * P + g] = v[i][r];
    }
  });
  if constexpr (!gout) __syncthreads();
  if constexpr (!last) vol_z_stages<L, DIR, S + 1>(sh, tid, tw, W, plane, nx);
}

template <int L, int MODE, bool PLAIN>
__global__ __launch_bounds__((VolCol<L>::NT), (VolCol<L>::WPE)) void k_vol_col(VolColArgs p) {
  using R = VolCol<L>;
  constexpr int C = R::C, NT = R::NT, P = R::P, NY = L * C, IY = per_thread<NY, NT>;
  __shared__ float2 sh[R::SIZE];
  __shared__ float2 tw[vol_yinv_off(L)];
  __shared__ double red[(MODE == kColEFourier) ? 4 * 32 : 1];
  const ColArgs& a = p.a;
  const int tid = threadIdx.x;
  const int nxg = p.nx / C, A = p.ny / kVolB;
  const int blk = xcd_tile(blockIdx.x, gridDim.x);
  const int c = (blk / nxg) % A, xg = blk % nxg, rec = blk / (nxg * A);
  if (MODE != kColEFourier && a.rec_active && a.rec_active[rec] != kSlotActive) return;
  const long plane = (long)p.nx * p.ny, N = plane * L;
  const long base = rec * N + (long)c * kVolB * p.nx + xg * C;
  const bool second = blockIdx.y != 0;  // the difference map's f1
  float2* W = (second ? p.W2 : a.W) + base;
  for (int i = tid; i < vol_yinv_off(L); i += NT) tw[i] = p.tw[i];
  const long abase = rec * N + (long)(blk - rec * (nxg * A)) * kVolB * NY;
  // the amplitudes arrive during the transforms; thread order is memory order
  float amp[IY][kVolB];
  if (MODE == kColEFourier || PLAIN || a.objective == 0)
    each_of<NY, NT>(tid, [&](int i, int n) {
#pragma unroll
      for (int d = 0; d < kVolB; ++d) amp[i][d] = el(a.ampx + abase, d * NY + n);
    });
  vol_z_stages<L, -1, 0>(sh, tid, tw, W, plane, p.nx);
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const bool centro = a.centro != 0 && !second;  // the difference map constrains FFT(g0) only (src/phasing.c:1232-1235)
  each_of<NY, NT>(tid, [&](int i, int n) {
    const int x = n % C, z = n / C;
    float2* s = sh + z * P + x;
    float2 v[kVolB];
#pragma unroll
    for (int b = 0; b < kVolB; ++b) v[b] = s[b * C];
    dft<kVolB, -1, true>(v);
    if constexpr (MODE == kColEFourier) {
#pragma unroll
      for (int d = 0; d < kVolB; ++d) {
        if (a.fout) a.fout[rec * N + z * plane + (long)(c + A * d) * p.nx + xg * C + x] = v[d];
        efourier_add(v[d], amp[i][d], acc);
      }
    } else {
      if constexpr (PLAIN) {
#pragma unroll
        for (int d = 0; d < kVolB; ++d) v[d] = project_phase(v[d], amp[i][d], centro);
      } else {
#pragma unroll
        for (int d = 0; d < kVolB; ++d) {
          const long idx = abase + d * NY + n;
          if (centro) v[d].y = 0.f;  // src/phasing.c:1061-1068
          if (a.objective == 0) {
            v[d] = project_pixel(v[d], amp[i][d], a, idx);
          } else {
            // src/phasing.c:1103-1109
            const float2 F = a.phased_amp[idx];
            if (__float_as_uint(F.x) != kUnmeasuredBits) v[d] = F;
          }
        }
      }
      dft<kVolB, +1, true>(v);
#pragma unroll
      for (int b = 0; b < kVolB; ++b) s[b * C] = v[b];
    }
  });
  if constexpr (MODE == kColEFourier) {
    block_sum<4, NT>(acc, red);
    if (tid == 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) a.partials[(long)blk * 4 + q] = acc[q];
    }
  } else {
    __syncthreads();
    vol_z_stages<L, +1, 0>(sh, tid, tw, W, plane, p.nx);
  }
}

template <int L>
struct VolLaunch {
  static void row(int mode, const VolRowArgs& a, hipStream_t s) {
    using R = VolRow<L>;
    const dim3 grid(a.nplanes * (kVolB / R::RB)), blk(R::NT);
    switch (mode) {
      case kVolUpdate: hipLaunchKernelGGL((k_vol_row<L, kVolUpdate>), grid, blk, 0, s, a); break;
      case kVolUpdateDM: hipLaunchKernelGGL((k_vol_row<L, kVolUpdateDM>), grid, blk, 0, s, a); break;
      case kVolFwd: hipLaunchKernelGGL((k_vol_row<L, kVolFwd>), grid, blk, 0, s, a); break;
      case kVolFwdF1: hipLaunchKernelGGL((k_vol_row<L, kVolFwdF1>), grid, blk, 0, s, a); break;
    }
  }
  static void col(int mode, const VolColArgs& a, hipStream_t s) {
    using R = VolCol<L>;
    const dim3 grid((a.nx / R::C) * (a.ny / kVolB) * a.nrec, a.W2 ? 2 : 1), blk(R::NT);
    if (mode == kColEFourier) hipLaunchKernelGGL((k_vol_col<L, kColEFourier, true>), grid, blk, 0, s, a);
    else if (a.a.objective == 0 && !a.a.margin) hipLaunchKernelGGL((k_vol_col<L, kColProject, true>), grid, blk, 0, s, a);
    else hipLaunchKernelGGL((k_vol_col<L, kColProject, false>), grid, blk, 0, s, a);
  }
};

template <int L>
constexpr VolOps vol_ops_of() {
  return VolOps{L, VolCol<L>::C, &VolLaunch<L>::row, &VolLaunch<L>::col};
}

}  // namespace spx
