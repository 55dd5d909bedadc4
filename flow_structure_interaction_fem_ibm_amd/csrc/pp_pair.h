// Both colours of one line direction in one launch, for the levels whose
// passes are bound by launches: a colour pass of 20k cells takes 3.3 to 3.6
// us, most of it launch and memory latency, and the next starts about 1.2 us
// later.
//
// A workgroup owns a tile of A x B lines (A along the contiguous transverse
// index).  It solves the first colour's lines of the tile and of the ring
// around it (the ring's again in the neighbouring tiles), keeps them in LDS,
// and solves the second colour's lines of the tile against them.  The result
// goes to another array, since the neighbouring tiles still read the old
// values.  Sixteen lanes hold a line in every direction, so one barrier does
// for the whole launch: FP32 32x24x24 4.6 us in x, 6.2 in y and z, where two
// colour passes take 8.2 with the gap between them; with the y and z
// reductions in LDS and lines across the lanes, as in k_yzline, 9.  Same
// equations, colours and order of operations as k_xline and k_yzline.
#pragma once
#include "pp_kernels.h"

namespace pp {

// The lines along DIR of one level: (a, b) = (j, k), (i, k) or (i, j); first
// colour: a + b even.  SPL: colour-split rows, see k_xline.
template <typename T, int DIR, bool SPL>
struct PairLines {
  const LevelArgs<T> &L;
  int hp;
  const T *__restrict__ rhs, *__restrict__ e;
  __device__ int n() const { return DIR == 0 ? L.cx : (DIR == 1 ? L.cy : L.cz); }
  __device__ int na() const { return DIR == 0 ? L.cy : L.cx; }
  __device__ int nb() const { return DIR == 2 ? L.cy : L.cz; }
  // offset of line (a, b)'s first cell, and of its cell q from there
  __device__ long start(int a, int b) const {
    const int i = DIR == 0 ? 0 : a, j = DIR == 0 ? a : (DIR == 1 ? 0 : b), k = DIR == 2 ? 0 : b;
    return SPL ? sidx(L.sx, L.sxy, hp, i, j, k) : lidx(L.sx, L.sxy, i, j, k);
  }
  __device__ long along(int q) const {
    return DIR == 0 ? (SPL ? (long)((q >> 1) + (q & 1) * hp) : (long)q) : (DIR == 1 ? q * (long)L.sx : q * L.sxy);
  }
  // LS cells of a line from cell q0 on (cells past its end: the first one's
  // memory, marked blank)
  template <int LS>
  __device__ void load(long base, int q0, uint8_t (&fl)[LS], T (&eo)[LS], T (&rv)[LS]) const {
    const int nl = n();
#pragma unroll
    for (int m = 0; m < LS; m++) {
      const long o = base + along(q0 + m < nl ? q0 + m : 0);
      fl[m] = q0 + m < nl ? L.fl[o] : FL_BLANK;
      eo[m] = e[o];
      rv[m] = rhs[o];
    }
  }
  // the four neighbouring lines' values beside them, a - 1, a + 1, b - 1, b + 1
  template <int LS>
  __device__ void load_neighbours(long base, int q0, int a, T (&v)[LS][4]) const {
    const int nl = n(), par = a & 1;
    const long dm = DIR == 0 ? -(long)L.sx : (SPL ? (par ? -(long)hp : (long)hp - 1) : -1);
    const long dp = DIR == 0 ? (long)L.sx : (SPL ? (par ? 1 - (long)hp : (long)hp) : 1);
    const long sb = DIR == 2 ? (long)L.sx : L.sxy;
#pragma unroll
    for (int m = 0; m < LS; m++) {
      const long o = base + along(q0 + m < nl ? q0 + m : 0);
      v[m][0] = e[o + dm];
      v[m][1] = e[o + dp];
      v[m][2] = e[o - sb];
      v[m][3] = e[o + sb];
    }
  }
  // coefficients of the cells along the line and, once per line, towards
  // its neighbours
  template <int LS>
  __device__ void load_coef(int q0, T (&cm)[LS], T (&cp)[LS]) const {
    const T *cml = DIR == 0 ? L.cmx : (DIR == 1 ? L.cmy : L.cmz), *cpl = DIR == 0 ? L.cpx : (DIR == 1 ? L.cpy : L.cpz);
    const int nl = n();
#pragma unroll
    for (int m = 0; m < LS; m++) {
      const int q = q0 + m < nl ? q0 + m : 0;
      cm[m] = cml[q];
      cp[m] = cpl[q];
    }
  }
  __device__ void load_cross(int a, int b, T (&t)[4]) const {
    t[0] = DIR == 0 ? L.cmy[a] : L.cmx[a];
    t[1] = DIR == 0 ? L.cpy[a] : L.cpx[a];
    t[2] = DIR == 2 ? L.cmy[b] : L.cmz[b];
    t[3] = DIR == 2 ? L.cpy[b] : L.cpz[b];
  }
  // eliminate the segment's rows; nbr(m, v) gives a cell's neighbour values
  template <int LS, typename Nbr>
  __device__ void push(const T (&cm)[LS], const T (&cp)[LS], const T (&t)[4], const uint8_t (&fl)[LS],
                       const T (&eo)[LS], const T (&rv)[LS], SegElim<T, LS> &se, Nbr nbr) const {
    constexpr uint8_t F_LM = DIR == 0 ? FL_IM : (DIR == 1 ? FL_JM : FL_KM), F_AM = DIR == 0 ? FL_JM : FL_IM,
                      F_BM = DIR == 2 ? FL_JM : FL_KM;
    constexpr uint8_t F_LP = (uint8_t)(2 * F_LM), F_AP = (uint8_t)(2 * F_AM), F_BP = (uint8_t)(2 * F_BM);
#pragma unroll
    for (int m = 0; m < LS; m++) {
      const uint8_t f = fl[m];
      const T am = (f & F_LM) ? T(0) : cm[m], ap = (f & F_LP) ? T(0) : cp[m];
      const T ama = (f & F_AM) ? T(0) : t[0], apa = (f & F_AP) ? T(0) : t[1];
      const T amb = (f & F_BM) ? T(0) : t[2], apb = (f & F_BP) ? T(0) : t[3];
      const T dl = -(am + ap), da = -(ama + apa), db = -(amb + apb);
      const T diag = DIR == 0 ? (dl + da) + db : (DIR == 1 ? (da + dl) + db : (da + db) + dl);
      T v[4];
      nbr(m, v);
      const T r = rv[m] - v[0] * ama - v[1] * apa - v[2] * amb - v[3] * apb;
      // blank rows hold the ghost value; a fluid row with every face closed
      // keeps its value
      const bool fluid = !(f & FL_BLANK), row = fluid && !(tabs(diag) < T(1.0e-12));
      se.push(m, row ? am : T(0), row ? diag : T(1), row ? ap : T(0),
              row ? r : ((fluid || (f & FL_GHOST)) ? eo[m] : T(0)));
    }
  }
  template <int LS>
  __device__ void store(long base, int q0, const T (&x)[LS], T *__restrict__ out) const {
    const int nl = n();
#pragma unroll
    for (int m = 0; m < LS; m++)
      if (q0 + m < nl) out[base + along(q0 + m)] = x[m];
  }
};

// A first-colour line of the tile at (a0, b0) with its ring: row r (0 .. B +
// 1) and place p (0 .. A / 2) in it; its index among them is r (A/2 + 1) + p.
__device__ inline void pair_first(int a0, int b0, int r, int p, int &a, int &b) {
  b = b0 - 1 + r;
  a = a0 - 1 + 2 * p + ((a0 - 1 + b) & 1);
}
template <int A>
__device__ inline int pair_index(int a0, int b0, int a, int b) {
  return (b - b0 + 1) * (A / 2 + 1) + ((a - a0 + 1) >> 1);
}

constexpr int kPairA = 8, kPairB = 4, kPairThreads = 512;
constexpr int kPairSlots = (kPairA / 2 + 1) * (kPairB + 2);
template <typename T, int LS, int DIR, bool SPL>
__global__ void __launch_bounds__(kPairThreads) k_line_pair(LevelArgs<T> L, int hp, const T *__restrict__ rhs,
                                                          const T *__restrict__ e, T *__restrict__ out, T omega) {
  constexpr int G = 16, np = G * LS, A = kPairA, B = kPairB;
  static_assert(kPairSlots * G <= kPairThreads, "a group of lanes per first-colour line");
  __shared__ T first[kPairSlots * np];
  const PairLines<T, DIR, SPL> D{L, hp, rhs, e};
  const int a0 = blockIdx.x * A, b0 = blockIdx.y * B;
  const int slot = threadIdx.x / G, sub = threadIdx.x & (G - 1), q0 = sub * LS;
  T cm[LS], cp[LS], tc[4], eo[LS], rv[LS];
  uint8_t fl[LS];
  SegElim<T, LS> se;
  D.load_coef(q0, cm, cp);
  if (slot < kPairSlots) {  // first colour: tile and ring
    const int r = slot / (A / 2 + 1);
    int a, b;
    pair_first(a0, b0, r, slot - r * (A / 2 + 1), a, b);
    const bool in = a >= 0 && a < D.na() && b >= 0 && b < D.nb();
    const int ac = in ? a : 0, bc = in ? b : 0;  // slots past the level work on line (0, 0) and keep zeros
    const long base = D.start(ac, bc);
    T v[LS][4];
    D.load_cross(ac, bc, tc);
    D.load(base, q0, fl, eo, rv);
    D.load_neighbours(base, q0, ac, v);
    D.push(cm, cp, tc, fl, eo, rv, se, [&](int m, T(&w)[4]) {
#pragma unroll
      for (int t = 0; t < 4; t++) w[t] = v[m][t];
    });
    se.template solve<G>();
#pragma unroll
    for (int m = 0; m < LS; m++) {
      eo[m] = (T(1) - omega) * eo[m] + omega * se.dp[m];
      first[slot * np + q0 + m] = in ? eo[m] : T(0);
    }
    if (in && a >= a0 && a < a0 + A && b >= b0 && b < b0 + B) D.store(base, q0, eo, out);
  }
  // second colour: the tile's lines
  const int r = slot / (A / 2), b = b0 + r, a = a0 + 2 * (slot - r * (A / 2)) + ((a0 + b + 1) & 1);
  const bool in = slot < A * B / 2 && a < D.na() && b < D.nb();
  const long base = D.start(in ? a : 0, in ? b : 0);
  if (in) {
    D.load_cross(a, b, tc);
    D.load(base, q0, fl, eo, rv);
  }
  __syncthreads();
  if (!in) return;  // whole groups of lanes
  const T *w0 = first + pair_index<A>(a0, b0, a - 1, b) * np + q0, *w1 = first + pair_index<A>(a0, b0, a + 1, b) * np + q0;
  const T *w2 = first + pair_index<A>(a0, b0, a, b - 1) * np + q0, *w3 = first + pair_index<A>(a0, b0, a, b + 1) * np + q0;
  D.push(cm, cp, tc, fl, eo, rv, se, [&](int m, T(&w)[4]) { w[0] = w0[m]; w[1] = w1[m]; w[2] = w2[m]; w[3] = w3[m]; });
  se.template solve<G>();
#pragma unroll
  for (int m = 0; m < LS; m++) eo[m] = (T(1) - omega) * eo[m] + omega * se.dp[m];
  D.store(base, q0, eo, out);
}

}  // namespace pp
