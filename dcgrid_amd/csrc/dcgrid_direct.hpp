// dcgrid_direct.hpp — gfx950 direct solve of a dense level's correction equation (extension).
//
// A level that covers the domain has the couplings of a box with Neumann walls: every neighbour is
// a cell of the level or, at a wall, the cell itself. Its operator A (diagonal minus neighbours) is
// diagonal in the DCT-II basis of the three axes, with eigenvalues
//     4 sin^2(pi kx / 2 nx) + 4 sin^2(pi ky / 2 ny) + 4 sin^2(pi kz / 2 nz),
// so A e = h^2 rho takes a transform along each axis, a division and the inverse transforms. The
// constant mode, which a pure Neumann system leaves free, is set to zero.
//
// Each transform is a matrix product, on the matrix cores (v_mfma_f64_16x16x4, or the f32 form):
// cells * n multiply-adds a pass, half of that through the symmetry of the cosines (a row's
// values at i and n-1-i are folded to their sum and difference, which the even and the odd
// frequencies take apart). A pass works on tiles of n x NC values staged in LDS: NC lines along the
// axis, all n entries of each. Five passes: z and y forward, x forward, division and x back in one,
// y and z back. Frequencies stay in the order the fold gives them (the even ones, then the odd).
//
// What bounds a pass (MI355X, FP64, 256 x 128 x 256 cells, 67 MB in and out): z forward 77 us (block
// order in, 27 TFLOP/s), y 26 us (2.6 TB/s of each direction), x both ways 129 us (33 TFLOP/s of the
// 69 that the instruction alone reaches), y back 32, z back 75 us; 64^3 and less 4-9 us, latency. Against
// the V-cycles of such a level (seven to nine, to 1e-8) it leaves one step at 1e-13: a projection of
// 256 x 128 x 256 cells on three dense levels 6.24 -> 0.96 ms, of 512 x 128 x 512 on four 19.2 -> 4.1 ms,
// of 512^3 cells in 32768 blocks of 8^3 (two of four levels dense) 4.82 -> 2.19 ms. In FP32 throughout, four to five
// steps stall where the V-cycles' seven to nine did, at the rounding of the residual: over 192 levels of 17 grids
// the pressure's error against 64 bits is 1.03 +- 0.04 times theirs (they fail on 40 more, which this solves).
#pragma once

#include "dcgrid_solve.hpp"

namespace dcg {

// 16 x 16 x 4 matrix product: lane l holds a = A[l % 16][k], b = B[k][l % 16] for k = l / 16, and
// of the result column l % 16, rows row(l / 16, 0..3).
template <class T>
struct Mfma;
template <>
struct Mfma<float> {
  typedef float V __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ V mac(float a, float b, V c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int q, int r) { return 4 * q + r; }
};
template <>
struct Mfma<double> {
  typedef double V __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ V mac(double a, double b, V c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int q, int r) { return q + 4 * r; }
};

// Transform of one axis length n (even): np x np matrices (np = n / 2 rounded up to 16, zero beyond
// n / 2): the even and odd rows of the orthonormal DCT-II over the first half of the axis, their
// transposes, and the eigenvalue of every frequency in fold order.
template <class T>
struct DctAxis {
  const T* fwd[2];
  const T* inv[2];
  const T* lam;
  int n, nh, np;
};
enum : int { DCT_Z_FWD, DCT_Y_FWD, DCT_X_BOTH, DCT_Y_INV, DCT_Z_INV };
template <class T>
struct DctArgs {
  DctAxis<T> ax;         // the axis of the pass
  const T *lamY, *lamZ;  // DCT_X_BOTH
  const T* in;
  T* out;
  int nx, ny, nz, rx, ry, rz;
  uint32_t cell0;  // first cell of the level in block order
  T h2;
  const SolveCtl* ctl;
};
static constexpr int kDctThreads = 512;
// Longest axis: a tile of 16 lines is 144 KB at 1024 entries in FP64. Beyond 512 cells, with these tiles,
// the direct solve is still 1.25x (1024 x 8 x 8 cells) to 9x (640 x 640 x 64) faster than the V-cycles in mixed
// arithmetic (1024 x 256 x 1024 on two levels 118 -> 54 ms), and up to 512 3.3x to 10x.
static constexpr int kDctMaxAxis = 1024;
// LDS row of NC lines. The pad spreads a fragment's four rows over the banks.
template <int NC>
static constexpr int kDctRow = NC + (NC == 16 ? 2 : 4);
template <class T, int NC>
constexpr size_t dctLds(int np) {
  return (size_t)2 * np * kDctRow<NC> * sizeof(T);
}
// Lines along z of a block column, numbered by the Morton code of (lx, ly): 16, 32 or 64 consecutive
// lines are then a consecutive part of every block's cells (whose z bits are below).
template <int BW>
__device__ __forceinline__ int lineOf(int lx, int ly) {
  int r = 0;
#pragma unroll
  for (int b = 0; b < Geo<BW>::BB; b++) r |= ((lx >> b) & 1) << (2 * b + 1) | ((ly >> b) & 1) << (2 * b);
  return r;
}
template <int BW>
__device__ __forceinline__ void linePos(int l, int& lx, int& ly) {
  lx = ly = 0;
#pragma unroll
  for (int b = 0; b < Geo<BW>::BB; b++) {
    lx |= ((l >> (2 * b + 1)) & 1) << b;
    ly |= ((l >> (2 * b)) & 1) << b;
  }
}

// Block order of the level's cells is the input of DCT_Z_FWD and the output of DCT_Z_INV. Between:
//   S1[zr][line], lines in block-column order (bx ry + by) BW^2 + lineOf(lx, ly), zr the z frequency;
//   S2[(zr ny + yr) nx + x].
template <int BW, class T, int NC, int PASS>
__global__ void __launch_bounds__(kDctThreads) k_dct(DctArgs<T> a) {
  constexpr int BB = Geo<BW>::BB, BV = Geo<BW>::BV, BL = BW * BW, ST = kDctRow<NC>;
  constexpr int NT = NC >= 32 ? 2 : 1, NG = NC / 16 / NT;
  constexpr bool FWD = PASS == DCT_Z_FWD || PASS == DCT_Y_FWD || PASS == DCT_X_BOTH;
  constexpr int WAVES = kDctThreads / 64, UMAX = 8 / NT;  // units of a wavefront at the longest axis
  using M = Mfma<T>;
  using V = typename M::V;
  extern __shared__ char ldsRaw[];
  T* X = reinterpret_cast<T*>(ldsRaw);
  if (solveDone(a.ctl)) return;
  const int n = a.ax.n, nh = a.ax.nh, np = a.ax.np;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, q = lane >> 4;
  const uint32_t NL = (uint32_t)a.nx * a.ny;
  // the tile's lines
  const uint32_t first = blockIdx.x * NC;                      // z: first line; x: first (zr, yr)
  constexpr int NZ = NC / BW;                                  // y: z frequencies of the tile
  const int bx = (int)(blockIdx.x % (uint32_t)a.rx), zr0 = (int)(blockIdx.x / (uint32_t)a.rx) * NZ;
  // ---- stage the tile: folded (forward) or as it is (inverse); rows nh.. np-1 of both halves zero
  for (int e = tid; e < 2 * (np - nh) * NC; e += kDctThreads) {
    const int r = e / NC;
    X[(r < np - nh ? nh + r : nh + np + (r - (np - nh))) * ST + e % NC] = (T)0;
  }
  auto fold = [&](int i, int c, T u, T v) {
    X[i * ST + c] = u + v;
    X[(np + i) * ST + c] = u - v;
  };
  // the cells of one z tile: per block column the part of every block that the tile's lines cover
  constexpr int PART = NC >= BL ? BV : NC * BW, QB = NC >= BL ? NC / BL : 1;
  const uint32_t col0 = first / BL, sub = NC >= BL ? 0u : first % BL;
  auto blockCells = [&](auto op) {  // op(column, z, cell of (column, z), block column, local cell)
    const int per = PART * a.rz;
    for (int e = tid; e < QB * per; e += kDctThreads) {
      const int qb = e / per, b = (e % per) / PART, t = (int)sub * BW + e % PART;
      const uint32_t col = col0 + qb;
      if (col >= NL / BL) continue;
      int lx, ly, lz;
      locPos<BB>((uint32_t)t, lx, ly, lz);
      op(qb * BL + lineOf<BW>(lx, ly) - (int)sub, b * BW + lz, a.cell0 + (col * a.rz + b) * BV + t, col, lx, ly);
    }
  };
  if (PASS == DCT_Z_FWD) {
    blockCells([&](int c, int z, uint32_t cell, uint32_t col, int lx, int ly) {
      if (z >= nh) return;
      const int m = n - 1 - z;
      fold(z, c, a.in[cell], a.in[a.cell0 + (col * a.rz + (m >> BB)) * BV + loc<BB>(lx, ly, m & (BW - 1))]);
    });
  } else if (PASS == DCT_Y_FWD) {
    const int per = a.ry * BL;
    for (int e = tid; e < NZ * per; e += kDctThreads) {
      const int zi = e / per, w = e % per;
      int lx, ly;
      linePos<BW>(w % BL, lx, ly);
      const int y = (w / BL) * BW + ly, m = n - 1 - y;
      if (y >= nh || zr0 + zi >= a.nz) continue;
      const T* s = a.in + (size_t)(zr0 + zi) * NL + (uint32_t)bx * per;
      fold(y, zi * BW + lx, s[w], s[(m >> BB) * BL + lineOf<BW>(lx, m & (BW - 1))]);
    }
  } else if (PASS == DCT_X_BOTH) {
    for (int e = tid; e < NC * nh; e += kDctThreads) {
      const int c = e / nh, x = e % nh;
      if (first + c >= (uint32_t)a.nz * a.ny) continue;
      const T* s = a.in + (size_t)(first + c) * n;
      fold(x, c, s[x], s[n - 1 - x]);
    }
  } else if (PASS == DCT_Y_INV) {
    for (int e = tid; e < NC * n; e += kDctThreads) {
      const int lx = e % BW, r = (e / BW) % n, zi = e / (BW * n);
      if (zr0 + zi >= a.nz) continue;
      X[(r < nh ? r : np + r - nh) * ST + zi * BW + lx] = a.in[((size_t)(zr0 + zi) * n + r) * a.nx + bx * BW + lx];
    }
  } else {
    for (int e = tid; e < NC * n; e += kDctThreads) {
      const int c = e % NC, r = e / NC;
      if (first + c >= NL) continue;
      X[(r < nh ? r : np + r - nh) * ST + c] = a.in[(size_t)r * NL + first + c];
    }
  }
  __syncthreads();
  // ---- products: 16 rows of `mat` with NT tiles of 16 columns of the half `h`
  const int MT = np / 16;
  auto product = [&](const T* __restrict__ mat, int h, int mt, int g, V* acc) {
    const T* ar = mat + (size_t)(16 * mt + j) * np + 4 * q;
    const T* xr = X + (h * np + 4 * q) * ST + g * NT * 16 + j;
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = V{0, 0, 0, 0};
#pragma unroll 2
    for (int s = 0; s < MT; s++) {  // step m takes entries 16 s + 4 q + m from both operands
      T av[4];
#pragma unroll
      for (int m = 0; m < 4; m++) av[m] = ar[16 * s + m];
#pragma unroll
      for (int m = 0; m < 4; m++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[t] = M::mac(av[m], xr[(16 * s + m) * ST + 16 * t], acc[t]);
    }
  };
  if (FWD) {
    V acc[UMAX][NT];
#pragma unroll
    for (int i = 0; i < UMAX; i++) {
      const int u = wave + i * WAVES;
      if (u < 2 * MT * NG) product(a.ax.fwd[u & 1], u & 1, (u >> 1) / NG, (u >> 1) % NG, acc[i]);
    }
    if (PASS == DCT_X_BOTH) __syncthreads();  // the folded tile is no longer read
#pragma unroll
    for (int i = 0; i < UMAX; i++) {
      const int u = wave + i * WAVES;
      if (u >= 2 * MT * NG) continue;
      const int h = u & 1, mt = (u >> 1) / NG, g = (u >> 1) % NG;
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const int c = (g * NT + t) * 16 + j;
        T ly = 0, lz = 0;
        if (PASS == DCT_X_BOTH && first + c < (uint32_t)a.nz * a.ny) {
          ly = a.lamY[(first + c) % (uint32_t)a.ny];
          lz = a.lamZ[(first + c) / (uint32_t)a.ny];
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int k = 16 * mt + M::row(q, r);
          const T v = acc[i][t][r];
          if (PASS == DCT_X_BOTH) {
            const T l = (k < nh ? a.ax.lam[h * nh + k] : (T)0) + ly + lz;
            X[(h * np + k) * ST + c] = k < nh && l > (T)0 ? v * (a.h2 / l) : (T)0;  // l = 0: the constant mode
          } else if (k < nh) {
            const int kr = h * nh + k;
            if (PASS == DCT_Z_FWD) {
              if (first + c < NL) a.out[(size_t)kr * NL + first + c] = v;
            } else if (zr0 + c / BW < a.nz) {
              a.out[((size_t)(zr0 + c / BW) * n + kr) * a.nx + bx * BW + c % BW] = v;
            }
          }
        }
      }
    }
    if (PASS != DCT_X_BOTH) return;
    __syncthreads();
  }
  // ---- inverse: the even and the odd frequencies' parts of entry i; entry n-1-i is their difference
  V even[UMAX / 2][NT], odd[UMAX / 2][NT];
#pragma unroll
  for (int i = 0; i < UMAX / 2; i++) {
    const int u = wave + i * WAVES;
    if (u < MT * NG) {
      product(a.ax.inv[0], 0, u / NG, u % NG, even[i]);
      product(a.ax.inv[1], 1, u / NG, u % NG, odd[i]);
    }
  }
  __syncthreads();  // the frequencies are no longer read: the tile takes the result
#pragma unroll
  for (int i = 0; i < UMAX / 2; i++) {
    const int u = wave + i * WAVES;
    if (u >= MT * NG) continue;
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const int c = ((u % NG) * NT + t) * 16 + j;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int k = 16 * (u / NG) + M::row(q, r);
        if (k >= nh) continue;
        X[k * ST + c] = even[i][t][r] + odd[i][t][r];
        X[(n - 1 - k) * ST + c] = even[i][t][r] - odd[i][t][r];
      }
    }
  }
  __syncthreads();
  if (PASS == DCT_Z_INV) {
    blockCells([&](int c, int z, uint32_t cell, uint32_t, int, int) { a.out[cell] = X[z * ST + c]; });
  } else if (PASS == DCT_Y_INV) {
    const int per = a.ry * BL;
    for (int e = tid; e < NZ * per; e += kDctThreads) {
      const int zi = e / per, w = e % per;
      int lx, ly;
      linePos<BW>(w % BL, lx, ly);
      const int y = (w / BL) * BW + ly;
      if (zr0 + zi < a.nz) a.out[(size_t)(zr0 + zi) * NL + (uint32_t)bx * per + w] = X[y * ST + zi * BW + lx];
    }
  } else {
    for (int e = tid; e < NC * n; e += kDctThreads) {
      const int c = e / n, x = e % n;
      if (first + c < (uint32_t)a.nz * a.ny) a.out[(size_t)(first + c) * n + x] = X[x * ST + c];
    }
  }
}

}  // namespace dcg
