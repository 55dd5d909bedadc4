// CDNA4 (gfx950) kernels of the implicit momentum solve (itsolv_ad_x/y/z,
// calc_residual_ad; CORE_SOLVE_AD.F90:314-907) on colour-split rows.
//
// The solve works on its own copy of u, v, w, of their right-hand sides and
// of the seven row coefficients, in the row layout of the pressure solve's
// split level 0 (sidx): the even cells of a row, then its odd cells.  A
// zebra colour of y- or z-lines then owns one contiguous half of every row,
// and a thread's four consecutive cells of an x-line are two 16-byte pairs.
// In the caller's layout a y/z pass moved every cache line of the 13 fields
// to update half the cells, and an x pass read them 32 bytes apart per lane.
//
// The copy carries what the passes would otherwise test per cell: row
// coefficients across a closed face are 0, a blank row is the identity
// (coefficients 0, diagonal 1) with right-hand side 0, or on a ghost cell
// its current value, so the passes read no flags.  The outer layer holds the
// caller's values, whose edges and corners only the ghost and fresh-cell
// stencils read: a line's rows end with its last cell, and what a segment
// covers behind it is the literal identity row (a row of zero coefficients
// would still take 0 * x from its neighbours, NaN where those are not finite).
#pragma once

#include "pp_kernels.h"

namespace pp {

// longest segment of a y/z line per thread
constexpr int kAdMaxLS = 16;

// Split-row geometry and arrays of the momentum solve: total values per
// array, `row` the seven coefficients amx, apx, amy, apy, amz, apz, diagonal
// (total apart).
struct AdSplit {
  int cx, cy, cz, sx, hp;
  long sxy, total;
  double *var[3], *rw[3], *row;
};
__device__ inline long aidx(const AdSplit &A, int i, int j, int k) { return sidx(A.sx, A.sxy, A.hp, i, j, k); }
// offset of a reference-layout entry (0..n+1 per direction) in the split rows
__host__ __device__ inline long ref_to_split(const RefArgs &R, int sx, long sxy, int hp, long r) {
  const int i = (int)(r % R.ex), k = (int)(r / R.exy), j = (int)((r - R.exy * k) / R.ex);
  return sidx(sx, sxy, hp, i - 1, j - 1, k - 1);
}
__global__ void __launch_bounds__(256) k_ad_offsets(int n, RefArgs R, int sx, long sxy, int hp,
                                                    const long *__restrict__ ref, long *__restrict__ out) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q < n) out[q] = ref[q] < 0 ? -1 : ref_to_split(R, sx, sxy, hp, ref[q]);
}

// ---------------------------------------------------------------------
// One pair of row positions (the even cell 2h and the odd cell 2h + 1) per
// thread, rows (j, k) of the grid's y and z.
// u, v, w with their outer layer into the split copy, and the right-hand
// sides masked: 0 on a solid cell, the cell's value on a ghost.  HALO rows
// and the end cells i = -1, cx carry the caller's outer layer.
// ---------------------------------------------------------------------
struct AdIn {
  const double *var[3], *r[3];
};
template <int NV>
__global__ void __launch_bounds__(256) k_ad_in(RefArgs R, LevelArgs<double> L0, AdIn F, AdSplit A) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;  // cells 2h - 1 and 2h (0-based), h = 0 .. (nxc + 1) / 2
  const int j = (int)(blockIdx.y * blockDim.y + threadIdx.y) - 1, k = (int)blockIdx.z - 1;
  if (j > R.nyc) return;
  const bool inner_row = j >= 0 && j < R.nyc && k >= 0 && k < R.nzc;
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int i = 2 * h - 1 + t;
    if (i > R.nxc) return;
    const long r = (long)(i + 1) + R.ex * (j + 1) + R.exy * (k + 1);
    const long a = aidx(A, i, j, k);
    const bool cell = inner_row && i >= 0 && i < R.nxc;
    const uint8_t f = cell ? L0.fl[lidx(L0.sx, L0.sxy, i, j, k)] : (uint8_t)FL_BLANK;
#pragma unroll
    for (int q = 0; q < NV; q++) {
      const double v = F.var[q][r];
      A.var[q][a] = v;
      if (cell) A.rw[q][a] = (f & FL_BLANK) ? ((f & FL_GHOST) ? v : 0.0) : F.r[q][r];
    }
  }
}
// the interior cells of u, v, w back into the caller's fields
struct AdOut {
  double *var[3];
};
__global__ void __launch_bounds__(256) k_ad_out(RefArgs R, AdSplit A, AdOut F) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y, k = blockIdx.z;
  if (i >= R.nxc || j >= R.nyc) return;
  const long a = aidx(A, i, j, k), r = ridx(R, i, j, k);
#pragma unroll
  for (int q = 0; q < 3; q++) F.var[q][r] = A.var[q][a];
}

// ---------------------------------------------------------------------
// The operator of one cell as itsolv_ad_* and calc_residual_ad build it
// (CORE_SOLVE_AD.F90:391-421), masked: the viscous coefficients plus the
// Crank-Nicolson advection terms (half_dt = 0 for ADAMS_BASHFORTH2), 0
// across a closed face, and the diagonal 1 + (acx + acy + acz); the identity
// row on a blank cell.  A fresh cell's diagonal is 1 (killForGCMFresh,
// CORE_SOLVE_AD.F90:425-427, 866).  The face velocities are fixed during one
// solve_ad call, so the rows are built once per call.
// ---------------------------------------------------------------------
template <int NT>
__global__ void __launch_bounds__(NT) k_ad_rows(RefArgs R, LevelArgs<double> L0, FracMetrics M, double half_dt,
                                                const double *__restrict__ coef, long nref,
                                                const double *__restrict__ fu, const double *__restrict__ fv,
                                                const double *__restrict__ fw, const int8_t *__restrict__ fresh,
                                                AdSplit A) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y, k = blockIdx.z;
  if (i >= R.nxc || j >= R.nyc) return;
  const long id = ridx(R, i, j, k);
  const long a0 = aidx(A, i, j, k);
  const uint8_t f = L0.fl[lidx(L0.sx, L0.sxy, i, j, k)];
  const long st[3] = {1, R.ex, R.exy};
  const int I[3] = {i + 1, j + 1, k + 1};
  const uint8_t FM[3] = {FL_IM, FL_JM, FL_KM}, FP[3] = {FL_IP, FL_JP, FL_KP};
  const double *face[3] = {fu, fv, fw};
  const bool blank = f & FL_BLANK;
  double ac[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const int um = (f & FM[d]) ? 1 : 0, up = (f & FP[d]) ? 1 : 0;
    const int q = I[d];
    double am = coef[(2 * d) * nref + id], ap = coef[(2 * d + 1) * nref + id];
    double a = -(am + ap);
    const double fm = M.fx[d][q], fp = M.fx[d][q + 1], di = M.dinv[d][q];
    const double vm = face[d][id], vp = face[d][id + st[d]];
    double t1 = 1.0 - fm, t2 = fp;
    am = am - half_dt * vm * t1 * di;
    ap = ap + half_dt * vp * t2 * di;
    t1 = fm * (double)(1 - um);
    t2 = (1.0 - fp) * (double)(1 - up);
    a = a + half_dt * (vp * t2 - vm * t1) * di;
    A.row[(2 * d) * A.total + a0] = (blank || um) ? 0.0 : am;
    A.row[(2 * d + 1) * A.total + a0] = (blank || up) ? 0.0 : ap;
    ac[d] = a;
  }
  const double kill = fresh ? 1.0 - 1.0 * (double)fresh[id] : 1.0;
  A.row[6 * A.total + a0] = blank ? 1.0 : 1.0 + (ac[0] + ac[1] + ac[2]) * kill;
}

// ---------------------------------------------------------------------
// Reduced system of a line split into P segments, one equation per thread
// and three right-hand sides: back recurrences of the segment, then parallel
// cyclic reduction, double-buffered in LDS as three 16-byte fields per
// equation ([buf][field][slot], nslot slots; one more slot per buffer holds
// the identity equation read past the ends of a line).  Neighbouring lanes
// hold neighbouring slots, so every LDS access is a conflict-free 16-byte
// one.  Slot of segment s of this line: slot + (s - seg) * sstr.  Every
// thread of the block must call it.
// ---------------------------------------------------------------------
template <int LS>
__device__ inline void ad_reduced_solve(double2 *sh, int nslot, int slot, int sstr, int P, int seg,
                                        SegElimN<double, LS, 3> &se, double (&XL)[3], double (&XS)[3]) {
  double cl, dl[3], fl;
  se.back(cl, dl, fl);
  const int ns1 = nslot + 1;
  double2 *cur = sh, *nxt = sh + 3 * ns1;
  auto put = [&](double2 *b, int s, double A, double B, double C, double r0, double r1, double r2) {
    b[s] = make_double2(A, B);
    b[ns1 + s] = make_double2(C, r0);
    b[2 * ns1 + s] = make_double2(r1, r2);
  };
  if (slot == 0) {
    put(cur, nslot, 0.0, 1.0, 0.0, 0.0, 0.0, 0.0);
    put(nxt, nslot, 0.0, 1.0, 0.0, 0.0, 0.0, 0.0);
  }
  put(nxt, slot, se.fp[0], se.cp[0], se.dp[0][0], se.dp[1][0], se.dp[2][0], 0.0);
  __syncthreads();
  double F0n = 0.0, G0n = 0.0, D0n[3] = {0.0, 0.0, 0.0};
  if (seg + 1 < P) {
    const double2 a = nxt[slot + sstr], b = nxt[ns1 + slot + sstr], c = nxt[2 * ns1 + slot + sstr];
    F0n = a.x; G0n = a.y; D0n[0] = b.x; D0n[1] = b.y; D0n[2] = c.x;
  }
  double A = -fl, B = 1.0 + cl * F0n, C = cl * G0n, R[3];
#pragma unroll
  for (int q = 0; q < 3; q++) R[q] = dl[q] - cl * D0n[q];
  put(cur, slot, A, B, C, R[0], R[1], R[2]);
  __syncthreads();
  for (int d = 1; d < P; d <<= 1) {
    const int sm = seg >= d ? slot - d * sstr : nslot, sp = seg + d < P ? slot + d * sstr : nslot;
    const double2 am = cur[sm], bm = cur[ns1 + sm], cm = cur[2 * ns1 + sm];
    const double2 ap = cur[sp], bp = cur[ns1 + sp], cp = cur[2 * ns1 + sp];
    const double k1 = A * fast_rcp(am.y), k2 = C * fast_rcp(ap.y);
    A = -am.x * k1;
    B = B - bm.x * k1 - ap.x * k2;
    C = -bp.x * k2;
    R[0] = R[0] - bm.y * k1 - bp.y * k2;
    R[1] = R[1] - cm.x * k1 - cp.x * k2;
    R[2] = R[2] - cm.y * k1 - cp.y * k2;
    put(nxt, slot, A, B, C, R[0], R[1], R[2]);
    __syncthreads();
    double2 *t = cur; cur = nxt; nxt = t;
  }
  const double rB = fast_rcp(B);
#pragma unroll
  for (int q = 0; q < 3; q++) XS[q] = R[q] * rB;
  nxt[slot] = make_double2(XS[0], XS[1]);
  nxt[ns1 + slot] = make_double2(XS[2], 0.0);
  __syncthreads();
  XL[0] = XL[1] = XL[2] = 0.0;
  if (seg > 0) {
    const double2 a = nxt[slot - sstr], b = nxt[ns1 + slot - sstr];
    XL[0] = a.x; XL[1] = a.y; XL[2] = b.x;
  }
}

// ---------------------------------------------------------------------
// One zebra pass of y-lines (DIR = 1, plane = k) or z-lines (DIR = 2,
// plane = j) for u, v and w together: lines (i, plane) with (i + plane) % 2
// == colour, i.e. one contiguous half of each row; a block of TX lines x P
// segments of LS cells.  The three fields share the row coefficients and are
// independent until the ghost update, so one pass gives what three would.
// Past a line's end (RAG: segments reach there) a segment reads its first
// cell again, for rows that are then replaced by the identity.
// ---------------------------------------------------------------------
//
// Bound by HBM: 64 B/cell (half of the seven row coefficients 28 and of the
// three right-hand sides 12, the other colour's fields 12, the results 12);
// neighbouring planes are read again from the Infinity Cache.  A tile of 16
// lines is one 128-byte line per load and field; the cells of a segment are
// taken one at a time (see below), so that several blocks share a CU.
// 256x192x192: 150 us, 4.0 TB/s, against 387 (y) and 401 us (z) in the
// caller's layout with one block per CU and flag tests.
template <int DIR, int LS, bool RAG>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 8))) k_ad_yzline(AdSplit A, int color) {
  extern __shared__ unsigned char smem_raw[];
  const int TX = blockDim.x, P = blockDim.y;
  const int tx = threadIdx.x, seg = threadIdx.y;
  const int lb = xcd_block(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int tile = lb % gridDim.x, plane = lb / gridDim.x;
  const int par = (plane + color) & 1;
  const int h = tile * TX + tx;
  const bool ok = 2 * h + par < A.cx;
  const int n = DIR == 1 ? A.cy : A.cz;
  const int m0 = seg * LS;
  const long lstr = DIR == 1 ? (long)A.sx : A.sxy, ostr = DIR == 1 ? A.sxy : (long)A.sx;
  // uniform offset of the plane's first half-row, lane offset of the segment
  const long base = DIR == 1 ? sidx(A.sx, A.sxy, A.hp, par, 0, plane) : sidx(A.sx, A.sxy, A.hp, par, plane, 0);
  const long v = (ok ? h : 0) + (long)m0 * lstr;
  // the neighbours i - 1 and i + 1: the other half of the row
  const long dlo = par ? -(long)A.hp : (long)A.hp - 1, dhi = par ? 1 - (long)A.hp : (long)A.hp;
  const double *cxm = A.row + base, *cxp = cxm + A.total;
  const double *com = cxm + (DIR == 1 ? 4 : 2) * A.total, *cop = com + A.total;
  const double *clm = cxm + (DIR == 1 ? 2 : 4) * A.total, *clp = clm + A.total;
  const double *cd = cxm + 6 * A.total;
  SegElimN<double, LS, 3> se;
#pragma unroll
  for (int m = 0; m < LS; m++) {
    const bool in = !RAG || m0 + m < n;  // m0 < n
    const long o = in ? v + m * lstr : v;
    const double axm = cxm[o], axp = cxp[o], aom = com[o], aop = cop[o];
    double d[3];
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const double *x = A.var[q] + base;
      const double r = A.rw[q][base + o] - x[o + dlo] * axm - x[o + dhi] * axp - x[o - ostr] * aom - x[o + ostr] * aop;
      d[q] = in ? r : 0.0;
    }
    se.push(m, in ? clm[o] : 0.0, in ? cd[o] : 1.0, in ? clp[o] : 0.0, d);
    // the row's results are needed here, before the next cell's loads: left
    // alone the compiler loads the whole segment first (190 registers at
    // LS = 4, one block per CU, 204 us against 175 with LS = 4 this way)
    asm volatile("" : "+v"(se.dp[0][m]), "+v"(se.dp[1][m]), "+v"(se.dp[2][m]), "+v"(se.cp[m]), "+v"(se.fp[m])::"memory");
  }
  double XL[3], XS[3];
  ad_reduced_solve<LS>(reinterpret_cast<double2 *>(smem_raw), TX * P, seg * TX + tx, TX, P, seg, se, XL, XS);
  if (!ok) return;
#pragma unroll
  for (int q = 0; q < 3; q++) {
    se.combine(q, XL[q], XS[q]);
    double *x = A.var[q] + base;
#pragma unroll
    for (int m = 0; m < LS; m++)
      if (m0 + m < n) x[v + m * lstr] = se.dp[q][m];
  }
}

// One zebra pass of x-lines: lines (j, k) with (j + k) % 2 == colour, the P
// segments of four cells of a line on adjacent lanes (two 16-byte pairs per
// array and lane, one in each half row); TX lines per block.  256x192x192:
// 130 us, 4.65 TB/s on the 64 B/cell it must move, against 471 us with
// single 8-byte loads 32 bytes apart per lane and an LDS layout whose
// neighbouring equations met in the same banks.
template <bool RAG>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 8)))
k_ad_xline(AdSplit A, int color, int P, int TX) {
  extern __shared__ unsigned char smem_raw[];
  const int lt = threadIdx.x / P, seg = threadIdx.x - lt * P;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const int line = blk * TX + lt;
  const int nyh = (A.cy + 1) >> 1;
  const int k = line / nyh;
  const int j = 2 * (line - k * nyh) + ((k + color) & 1);
  const bool ok = k < A.cz && j < A.cy;
  const long v = ok ? sidx(A.sx, A.sxy, A.hp, 4 * seg, j, k) : sidx(A.sx, A.sxy, A.hp, 0, 0, 0);
  auto ld4 = [&](const double *p, double (&w)[4]) {
    const double2 e = *reinterpret_cast<const double2 *>(p), o = *reinterpret_cast<const double2 *>(p + A.hp);
    w[0] = e.x; w[1] = o.x; w[2] = e.y; w[3] = o.y;
  };
  double d[3][4];
#pragma unroll
  for (int q = 0; q < 3; q++) ld4(A.rw[q] + v, d[q]);
  auto off_line = [&](int c, long s) {
    double w[4];
    ld4(A.row + c * A.total + v, w);
#pragma unroll
    for (int q = 0; q < 3; q++) {
      double x[4];
      ld4(A.var[q] + v + s, x);
#pragma unroll
      for (int m = 0; m < 4; m++) d[q][m] -= x[m] * w[m];
    }
  };
  off_line(2, -(long)A.sx);
  off_line(3, A.sx);
  off_line(4, -A.sxy);
  off_line(5, A.sxy);
  double a[4], b[4], c[4];
  ld4(A.row + v, a);
  ld4(A.row + A.total + v, c);
  ld4(A.row + 6 * A.total + v, b);
  SegElimN<double, 4, 3> se;
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const bool in = !RAG || 4 * seg + m < A.cx;
    const double dm[3] = {in ? d[0][m] : 0.0, in ? d[1][m] : 0.0, in ? d[2][m] : 0.0};
    se.push(m, in ? a[m] : 0.0, in ? b[m] : 1.0, in ? c[m] : 0.0, dm);
  }
  double XL[3], XS[3];
  ad_reduced_solve<4>(reinterpret_cast<double2 *>(smem_raw), TX * P, threadIdx.x, 1, P, seg, se, XL, XS);
  if (!ok) return;
#pragma unroll
  for (int q = 0; q < 3; q++) {
    se.combine(q, XL[q], XS[q]);
    double *x = A.var[q] + v;
    if (4 * seg + 4 <= A.cx) {
      *reinterpret_cast<double2 *>(x) = make_double2(se.dp[q][0], se.dp[q][2]);
      *reinterpret_cast<double2 *>(x + A.hp) = make_double2(se.dp[q][1], se.dp[q][3]);
    } else {
#pragma unroll
      for (int m = 0; m < 4; m++)
        if (4 * seg + m < A.cx) x[(m & 1 ? A.hp : 0) + (m >> 1)] = se.dp[q][m];
    }
  }
}

// ---------------------------------------------------------------------
// calc_residual_ad for NV fields (u, v, w share the rows), the row's even
// and odd cell of one position per thread, KB rows of z per block: per-block
// maximum and argmax of each field at part[3 * (q * nblk + blk)], the argmax
// the smallest reference-layout offset of the block's maximum.  rout (may be
// null): the residual of the first field, reference layout.
// ---------------------------------------------------------------------
template <int NT, int NV>
__global__ void __launch_bounds__(NT) k_ad_residual(RefArgs R, LevelArgs<double> L0, AdSplit A, FreshRes FR,
                                                    double *__restrict__ part, long nblk, double *__restrict__ rout,
                                                    int kb) {
#pragma clang fp contract(off)
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  const int k0 = blockIdx.z * kb, k1 = min(k0 + kb, R.nzc);
  SumMax v[NV];
#pragma unroll
  for (int q = 0; q < NV; q++) v[q] = SumMax{0.0, 0.0, -1};
  const bool in = 2 * h < R.nxc && j < R.nyc;
  for (int k = k0; in && k < k1; k++) {
    const long e = sidx(A.sx, A.sxy, A.hp, 2 * h, j, k);
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int i = 2 * h + t;
      if (i >= R.nxc) break;
      const long a = t ? e + A.hp : e;
      const long am = t ? e : e + A.hp - 1, ap = t ? e + 1 : e + A.hp;
      const long id = ridx(R, i, j, k);
      const double fl = (L0.fl[lidx(L0.sx, L0.sxy, i, j, k)] & FL_BLANK) ? 0.0 : 1.0;
      const double *row = A.row;
      const double amx = row[a], apx = row[A.total + a], amy = row[2 * A.total + a], apy = row[3 * A.total + a];
      const double amz = row[4 * A.total + a], apz = row[5 * A.total + a], diag = row[6 * A.total + a];
      // GCM_correct_res_ad (GCM_FRESHCELL_AD.F90:73-137): the off-stencil
      // terms of a fresh cell, added one by one in stencil order before the
      // iblank mask
      const int fq = (FR.mask && FR.mask[id]) ? fresh_find(FR.ids, FR.n, id) : -1;
#pragma unroll
      for (int q = 0; q < NV; q++) {
        const double *x = A.var[q];
        double s = A.rw[q][a] - x[a] * diag - x[am] * amx - x[ap] * apx - x[a - A.sx] * amy - x[a + A.sx] * apy -
                   x[a - A.sxy] * amz - x[a + A.sxy] * apz;
        if (fq >= 0)
          for (int m = 0; m < 4; m++) s = s + FR.cc[4 * fq + m] * x[FR.coff[4 * fq + m]];
        s = s * fl;
        if (q == 0 && rout) rout[id] = s;
        const SumMax w{0.0, fabs(s), id};
        v[q] = v[q].arg < 0 ? w : summax_combine(v[q], w);
      }
    }
  }
  const long blk = blockIdx.x + (long)gridDim.x * (blockIdx.y + (long)gridDim.y * blockIdx.z);
#pragma unroll
  for (int q = 0; q < NV; q++) {
    const SumMax b = block_summax<NT>(v[q]);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
      double *pq = part + 3 * (nblk * q + blk);
      pq[0] = 0.0;
      pq[1] = b.mx;
      pq[2] = (double)b.arg;
    }
    __syncthreads();
  }
}
// the blocks' maxima of field blockIdx.x: out[3 * q + {0, 1, 2}] = {0, max, argmax}
__global__ void __launch_bounds__(1024) k_ad_residual_max(const double *__restrict__ part, int nblk,
                                                          double *__restrict__ out) {
  const double *p = part + 3L * nblk * blockIdx.x;
  SumMax v{0.0, -1.0, -1};
  for (int b = threadIdx.x; b < nblk; b += 1024) v = summax_combine(v, SumMax{0.0, p[3L * b + 1], (long)p[3L * b + 2]});
  v = block_summax<1024>(v);
  if (threadIdx.x == 0) {
    out[3 * blockIdx.x] = 0.0;
    out[3 * blockIdx.x + 1] = v.mx;
    out[3 * blockIdx.x + 2] = (double)v.arg;
  }
}

}  // namespace pp
