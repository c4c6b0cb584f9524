// The isotropic / VTI PML scheme on register tiles (included by elastic.hip; el_fwd_step and
// el3_fwd_step state one step): at 4th order two steps per launch, at 6th to 10th one.
//
// A workgroup of NW wavefronts holds a tile of NW*NR rows x 64 columns of one shot in registers
// (NR rows x 1 column per lane: the ten splits and six coefficients), advances it and stores the
// points whose stencils never left the tile: a step reaches 3 points in each direction with
// two-term differences and 5 with three, so 6 points on every side are halo.  x-neighbours come
// from the adjacent lanes (DPP wavefront shifts), z-neighbours from registers and, between
// wavefronts, through LDS: the edge rows of the velocity totals before the stress update, those
// of the stress totals before the velocity update.  Outside the update window the coefficients
// are zero, so the splits, zero there, stay zero without masks.
//
// What a step leaves for the adjoint is the five totals, half the bytes of the ten splits: the
// kernel writes them to a trace after every step, while the splits stay in registers between the
// launch's steps.
#include "tile_common.hpp"

namespace tile {

// Differences of ORD terms: 2 (4th order) or 3 (6th to 10th)
__host__ __device__ constexpr int steps_of(int ord) { return ord == 2 ? 2 : 1; }   // steps per launch (at most)
constexpr int TK = steps_of(2);
constexpr int H = 6;               // halo points per side: 3 per step with 2 terms, 5 with 3
constexpr int OX = WAVE - 2 * H;   // stored columns
constexpr int out_rows(int rows) { return rows - 2 * H; }
constexpr unsigned DROP = 0x80000000u;   // a lane offset past every buffer (all under 2 GiB): access dropped

// x / b from rb = 1.0 / (double)b, for quotients of 2^-126 and more the same bits as the division: rb and
// the product are each within 2^-53 of their exact values, relatively, and a quotient of two floats lies
// at least 2^-49 of its size from any value halfway between two floats, so the last rounding falls as
// the division's.  Smaller quotients can lie on such a value, and then may round to its other side:
// 1.4e-45 apart, as far from the quotient as the division's.  15 cycles a wavefront against 50 for the
// division sequence.
__device__ __forceinline__ float quot(float x, double rb) { return (float)((double)x * rb); }

struct Grid { int ntx, ntz; };

// the ORD-term staggered differences and their transposes: along x by wavefront shifts, along z
// about row r of an accessor
template <int ORD>
struct Fd {
  float c0, c1, c2;
  __device__ __forceinline__ float dxf(float v) const {
    const float l1 = from_left(v), r1 = from_right(v), r2 = from_right(r1);
    const float s = c0 * (r1 - v) + c1 * (r2 - l1);
    return ORD == 2 ? s : s + c2 * (from_right(r2) - from_left(l1));
  }
  __device__ __forceinline__ float dxb(float v) const {
    const float l1 = from_left(v), l2 = from_left(l1), r1 = from_right(v);
    const float s = c0 * (v - l1) + c1 * (r1 - l2);
    return ORD == 2 ? s : s + c2 * (from_right(r1) - from_left(l2));
  }
  __device__ __forceinline__ float dxfT(float v) const {
    const float l1 = from_left(v), l2 = from_left(l1), r1 = from_right(v);
    const float s = c0 * (l1 - v) + c1 * (l2 - r1);
    return ORD == 2 ? s : s + c2 * (from_left(l2) - from_right(r1));
  }
  __device__ __forceinline__ float dxbT(float v) const {
    const float l1 = from_left(v), r1 = from_right(v), r2 = from_right(r1);
    const float s = c0 * (v - r1) + c1 * (l1 - r2);
    return ORD == 2 ? s : s + c2 * (from_left(l1) - from_right(r2));
  }
  template <class W> __device__ __forceinline__ float dzf(const W &w, int r) const {
    const float s = c0 * (w(r + 1) - w(r)) + c1 * (w(r + 2) - w(r - 1));
    return ORD == 2 ? s : s + c2 * (w(r + 3) - w(r - 2));
  }
  template <class W> __device__ __forceinline__ float dzb(const W &w, int r) const {
    const float s = c0 * (w(r) - w(r - 1)) + c1 * (w(r + 1) - w(r - 2));
    return ORD == 2 ? s : s + c2 * (w(r + 2) - w(r - 3));
  }
  template <class W> __device__ __forceinline__ float dzfT(const W &w, int r) const {
    const float s = c0 * (w(r - 1) - w(r)) + c1 * (w(r - 2) - w(r + 1));
    return ORD == 2 ? s : s + c2 * (w(r - 3) - w(r + 2));
  }
  template <class W> __device__ __forceinline__ float dzbT(const W &w, int r) const {
    const float s = c0 * (w(r) - w(r + 1)) + c1 * (w(r - 1) - w(r + 2));
    return ORD == 2 ? s : s + c2 * (w(r - 2) - w(r + 3));
  }
};

// A wavefront's NR rows with the A rows above and the B below them from its neighbours, through an
// LDS buffer of A + B rows per wavefront (its first B and its last A), written by put before a
// barrier and read by get after it.  dzb and dzfT take A = ORD, B = ORD - 1, dzf and dzbT the reverse.
template <int A, int B, int NR>
struct Rows {
  const float (&v)[NR];
  float a[A], b[B];
  template <int Q>
  static __device__ __forceinline__ void put(float (*buf)[Q][WAVE], int wv, int slot, int lane, const float (&v)[NR]) {
#pragma unroll
    for (int j = 0; j < B; ++j) buf[wv + 1][slot + j][lane] = v[j];
#pragma unroll
    for (int j = 0; j < A; ++j) buf[wv + 1][slot + B + j][lane] = v[NR - A + j];
  }
  template <int Q>
  __device__ __forceinline__ Rows(const float (*buf)[Q][WAVE], int wv, int slot, int lane, const float (&v_)[NR]) : v(v_) {
#pragma unroll
    for (int j = 0; j < A; ++j) a[j] = buf[wv][slot + B + j][lane];
#pragma unroll
    for (int j = 0; j < B; ++j) b[j] = buf[wv + 2][slot + j][lane];
  }
  __device__ __forceinline__ float operator()(int r) const { return r < 0 ? a[r + A] : r >= NR ? b[r - NR] : v[r]; }
};

struct FwdIO {
  const float *in;
  float *out;
  int t, n;              // first step and number of steps (1 .. TK)
  float *trace;          // [n][5][S][Z][pitch] totals after each step, or NULL
  ElRec rec;             // rec.map NULL: no records
};

template <int ORD, int NR, int NW>
__global__ __launch_bounds__(NW *WAVE, 4) void el_fwd_tile(ElDev d, Grid g, FwdIO io) {
  static_assert(NR == 4 && H == 6, "rows nn-2 .. nn+1, which the free surface ties together, are wavefront 1 of the first tiles");
  using Up = Rows<ORD, ORD - 1, NR>;
  using Dn = Rows<ORD - 1, ORD, NR>;
  constexpr int Q = 2 * ORD - 1;   // LDS rows of either
  const int nn = ORD == 2 ? 2 : d.nn;
  constexpr int OZ = out_rows(NR * NW);
  constexpr int QN = 2 * (2 * ORD - 1);
  __shared__ float sv[NW + 2][QN][WAVE], ss[NW + 2][QN][WAVE];
  int tx, tzi, s;
  place(g, tx, tzi, s);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < QN; ++q) sv[0][q][lane] = sv[NW + 1][q][lane] = ss[0][q][lane] = ss[NW + 1][q][lane] = 0.f;
  }
  const int x0 = nn + tx * OX, z0 = nn + tzi * OZ;            // first stored column and row
  const int c = x0 - H + lane, zt = z0 - H + wv * NR;       // this lane's column, this wavefront's first row
  const int zw1 = d.Z - nn - 1, xw1 = d.X - nn - 1;   // the window's last row and column
  const unsigned rowb = 4u * (unsigned)d.pitch, planeb = 4u * (unsigned)d.plane, fieldb = 4u * (unsigned)d.field;
  const unsigned vin = c >= 0 && c < d.X ? 4u * (unsigned)c : DROP;
  const bool own = c >= x0 && c < min(x0 + OX, xw1 + 1);
  const unsigned vout = own ? 4u * (unsigned)c : DROP;
  const bool cwin = c >= nn && c <= xw1;
  auto bits = [&](int lo, int hi) -> unsigned {   // rows lo .. hi-1 of this wavefront
    const int a = min(max(lo - zt, 0), NR), b = min(max(hi - zt, 0), NR);
    return b > a ? ((1u << b) - 1u) & ~((1u << a) - 1u) : 0u;
  };
  const unsigned ownbits = bits(z0, min(z0 + OZ, zw1 + 1));
  auto off = [&](int row) -> unsigned { return (unsigned)min(max(row, 0), d.Z - 1) * rowb; };
  const Fd<ORD> D{d.c0, d.c1, ORD == 2 ? 0.f : d.c2};

  // ten splits; rows outside the grid repeat an edge row, whose splits are zero as theirs would be
  float f[NFIELD][NR];
  {
    const rsrc_t rIn = rsrc(io.in + (long long)s * d.plane, (NFIELD - 1) * fieldb + planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int q = 0; q < NFIELD; ++q) f[q][r] = bld(rIn, vin, (unsigned)q * fieldb + off(zt + r));
  }
  float C[4][NR], bx[NR], bz[NR];
  {
    const rsrc_t rC = rsrc(d.coef, (unsigned)NCOEF * planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const unsigned v = cwin && zt + r >= nn && zt + r <= zw1 ? vin : DROP;   // (dropped loads return 0)
#pragma unroll
      for (int q = 0; q < 4; ++q) C[q][r] = bld(rC, v, (unsigned)q * planeb + off(zt + r));
      bx[r] = bld(rC, v, BX * planeb + off(zt + r));
      bz[r] = bld(rC, v, BZ * planeb + off(zt + r));
    }
  }
  const int cc = min(max(c, 0), d.X - 1);
  const float pxn = d.pml_x[cc], pxi = d.pml_x[2 * d.pitch + cc];
  const double rpx = 1.0 / (double)d.pml_x[d.pitch + cc], rdx = 1.0 / (double)d.dx, rdz = 1.0 / (double)d.dz;
  auto pz = [&](int k, int r) -> float { return scalar_ld(d.pml_z + k * d.Z + min(max(zt + r, 0), d.Z - 1)); };
  double rpz[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) rpz[r] = 1.0 / (double)pz(1, r);
  const int zs = scalar_ld(d.src_z + s), xs = scalar_ld(d.src_x + s);
  const bool src_here = zs >= zt && zs < zt + NR;
  const bool fsw = d.fsurf && tzi == 0 && wv == 1;          // this wavefront's rows are nn-2 .. nn+1
  unsigned rbits = 0;
  if (io.rec.map) {
    const bool mine = lane < NR && ((ownbits >> (lane & 31)) & 1u);
    rbits = (unsigned)__ballot(mine && io.rec.map[mine ? zt + lane : 0] > 0);
  }
  const bool one_row = rbits && !(rbits & (rbits - 1));
  int ridx = -1;
  auto slot_of = [&](int r) -> int {
    return __builtin_bit_cast(int, bld(rsrc(io.rec.map + d.Z, planeb), vout, off(zt + r)));
  };
  if (one_row) ridx = slot_of(__builtin_ctz(rbits));

#pragma unroll 1
  for (int i = 0; i < io.n; ++i) {
    const float wsrc = src_here ? scalar_ld(d.src + (long long)s * d.nt + io.t + i) : 0.f;
    // velocity totals, the free-surface rows nn-2 and nn-1 from rows nn and nn+1
    float vx[NR], vz[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) { vx[r] = f[VX_X][r] + f[VX_Z][r]; vz[r] = f[VZ_X][r] + f[VZ_Z][r]; }
    if (fsw) {
      const bool jj1 = c + 1 >= nn && c + 1 <= xw1;
      const float vz2n = from_right(vz[2]);
      const float vz1m_n = jj1 ? vz2n : 0.0f;
      const float vz1m = cwin ? vz[2] : vz[1];
      if (cwin) {
        vx[1] = (((vz1m_n - vz1m) + vz2n) - vz[2]) + vx[3];
        vz[0] = vz1m;
      }
      vz[1] = vz1m;
    }
    Dn::put(sv, wv, 0, lane, vx);
    Up::put(sv, wv, Q, lane, vz);
    lds_barrier();
    {
      const Dn VXr(sv, wv, 0, lane, vx);
      const Up VZr(sv, wv, Q, lane, vz);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        __builtin_amdgcn_sched_barrier(0);
        const float dxb_vx = D.dxb(vx[r]), dzb_vz = D.dzb(VZr, r);
        const float dxf_vz = D.dxf(vz[r]), dzf_vx = D.dzf(VXr, r);
        const float pzn = pz(0, r), pzi = pz(2, r);
        f[TXX_X][r] = (pxn * f[TXX_X][r] + d.dt_dx * (C[0][r] * dxb_vx)) * pxi;
        f[TXX_Z][r] = (pzn * f[TXX_Z][r] + d.dt_dz * (C[1][r] * dzb_vz)) * pzi;
        f[TZZ_X][r] = (pxn * f[TZZ_X][r] + d.dt_dx * (C[1][r] * dxb_vx)) * pxi;
        f[TZZ_Z][r] = (pzn * f[TZZ_Z][r] + d.dt_dz * (C[2][r] * dzb_vz)) * pzi;
        f[TXZ_X][r] = (pxn * f[TXZ_X][r] + d.dt_dx * (C[3][r] * dxf_vz)) * pxi;
        f[TXZ_Z][r] = (pzn * f[TXZ_Z][r] + d.dt_dz * (C[3][r] * dzf_vx)) * pzi;
      }
    }
    if (src_here) {
      const float mxx = d.src_m[3 * s], mzz = d.src_m[3 * s + 1], mxz = d.src_m[3 * s + 2];
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if (zs == zt + r && c == xs) {
          f[TXX_X][r] = f[TXX_X][r] + mxx * wsrc; f[TXX_Z][r] = f[TXX_Z][r] + mxx * wsrc;
          f[TZZ_X][r] = f[TZZ_X][r] + mzz * wsrc; f[TZZ_Z][r] = f[TZZ_Z][r] + mzz * wsrc;
          f[TXZ_X][r] = f[TXZ_X][r] + mxz * wsrc; f[TXZ_Z][r] = f[TXZ_Z][r] + mxz * wsrc;
        }
    }
    // stress totals, kept as they are for the records and the trace; the free surface after that
    float xx[NR], zz[NR], xz[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      xx[r] = f[TXX_X][r] + f[TXX_Z][r]; zz[r] = f[TZZ_X][r] + f[TZZ_Z][r]; xz[r] = f[TXZ_X][r] + f[TXZ_Z][r];
    }
    const long long ro = ((long long)s * d.nt + io.t + i) * d.nrec;
    const unsigned rbytes = 4u * (unsigned)d.nrec;
    auto rec_off = [&](int r) -> unsigned {
      const int m = one_row ? ridx : slot_of(r);
      return own && m >= 0 ? 4u * (unsigned)m : DROP;
    };
    if (rbits) {
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if ((rbits >> r) & 1u) {
          const unsigned v = rec_off(r);
          bst(xx[r], rsrc(io.rec.r[TXX] + ro, rbytes), v, 0u);
          bst(d.fsurf && zt + r == nn ? 0.0f : zz[r], rsrc(io.rec.r[TZZ] + ro, rbytes), v, 0u);
          bst(xz[r], rsrc(io.rec.r[TXZ] + ro, rbytes), v, 0u);
        }
    }
    const rsrc_t rT = rsrc(io.trace ? io.trace + (long long)i * NFIELD5 * d.field + (long long)s * d.plane : nullptr,
                           io.trace ? (NFIELD5 - 1) * fieldb + planeb : 0u);
    if (io.trace) {
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if ((ownbits >> r) & 1u) {
          bst(xx[r], rT, vout, TXX * fieldb + off(zt + r));
          bst(zz[r], rT, vout, TZZ * fieldb + off(zt + r));
          bst(xz[r], rT, vout, TXZ * fieldb + off(zt + r));
        }
    }
    if (fsw) {
      zz[1] = -zz[3]; zz[2] = 0.0f;
      xz[1] = -xz[2]; xz[0] = -xz[3];
    }
    Dn::put(ss, wv, 0, lane, zz);
    Up::put(ss, wv, Q, lane, xz);
    lds_barrier();
    {
      const Dn ZZr(ss, wv, 0, lane, zz);
      const Up XZr(ss, wv, Q, lane, xz);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        __builtin_amdgcn_sched_barrier(0);
        const float dxf_txx = D.dxf(xx[r]), dzb_txz = D.dzb(XZr, r);
        const float dxb_txz = D.dxb(xz[r]), dzf_tzz = D.dzf(ZZr, r);
        const float pzn = pz(0, r);
        f[VX_X][r] = quot(pxn * f[VX_X][r] + quot((d.dt * bx[r]) * dxf_txx, rdx), rpx);
        f[VX_Z][r] = quot(pzn * f[VX_Z][r] + quot((d.dt * bx[r]) * dzb_txz, rdz), rpz[r]);
        f[VZ_X][r] = quot(pxn * f[VZ_X][r] + quot((d.dt * bz[r]) * dxb_txz, rdx), rpx);
        f[VZ_Z][r] = quot(pzn * f[VZ_Z][r] + quot((d.dt * bz[r]) * dzf_tzz, rdz), rpz[r]);
      }
    }
    if (src_here && d.src_fz) {   // vertical force: half of f w into each vz split
      const float hf = 0.5f * (scalar_ld(d.src_fz + s) * wsrc);
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if (zs == zt + r && c == xs) {
          f[VZ_X][r] = f[VZ_X][r] + hf;
          f[VZ_Z][r] = f[VZ_Z][r] + hf;
        }
    }
    if (rbits) {
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if ((rbits >> r) & 1u) {
          const unsigned v = rec_off(r);
          bst(f[VX_X][r] + f[VX_Z][r], rsrc(io.rec.r[VX] + ro, rbytes), v, 0u);
          bst(f[VZ_X][r] + f[VZ_Z][r], rsrc(io.rec.r[VZ] + ro, rbytes), v, 0u);
        }
    }
    if (io.trace) {
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if ((ownbits >> r) & 1u) {
          bst(f[VX_X][r] + f[VX_Z][r], rT, vout, VX * fieldb + off(zt + r));
          bst(f[VZ_X][r] + f[VZ_Z][r], rT, vout, VZ * fieldb + off(zt + r));
        }
    }
  }
  if (io.out) {
    const rsrc_t rOut = rsrc(io.out + (long long)s * d.plane, (NFIELD - 1) * fieldb + planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if ((ownbits >> r) & 1u) {
#pragma unroll
        for (int q = 0; q < NFIELD; ++q) bst(f[q][r], rOut, vout, (unsigned)q * fieldb + off(zt + r));
      }
  }
}

struct AdjIO {
  const float *lin;
  float *lout;
  int t, n;              // latest step and number of steps (1 .. TK), going down
  int spg;               // shots per group
  const float *fv[TK];   // totals [5][S][Z][pitch] before each step (velocities) ...
  const float *fs[TK];   // ... and after it (stresses)
  float *gacc, *gsrc;    // [groups][NCOEF][Z][pitch] gradient sums; [S][nt] or NULL
  ElInj inj;             // inj.map NULL: no record adjoints
};

__device__ __forceinline__ float keep(int m, float v) {
  return __builtin_bit_cast(float, __builtin_bit_cast(int, v) & m);
}
__device__ __forceinline__ float pick(int m, float a, float b) {   // bits of a where m is set, else of b
  return __builtin_bit_cast(float, (__builtin_bit_cast(int, a) & m) | (__builtin_bit_cast(int, b) & ~m));
}

// The adjoint (el_adj_step lists the transposes) over the same tiles.  A workgroup takes the shots
// of a group one after the other and keeps their gradient sums of its points in registers: one
// read and write of the gradient planes per launch.  Per point and step that is 40 B of splits, 20 B
// of totals and 24 / shots B of gradients, against 80 + 20 + 12 for a step at a time; the halo's
// re-reads come from the L2.  A tile's loads, its arithmetic (about 200 VALU operations a row and
// step, 24 of them wavefront shifts) and its stores follow each other with one workgroup per CU; at
// 48 rows the traffic alone is two thirds of the time.  All of it has to stay within 168 registers,
// three wavefronts per SIMD: with 224 (two) 150 us per step against 135 on 242 x 680 with 32 shots,
// and el_adj_step took 251; 362 x 1040, 48 shots: 474, 409, 779.  Adjoint splits outside the window, which
// el_adj_step keeps at zero, take values here, but nothing reads them: the coefficients there are
// zero, and they are not stored.
template <int ORD, int NR, int NW>
__global__ __launch_bounds__(NW *WAVE, NW / 4) void el_adj_tile(ElDev d, Grid g, AdjIO io) {
  static_assert(NR == 4 && H == 6, "rows nn-2 .. nn+1, which the free surface ties together, are wavefront 1 of the first tiles");
  using Up = Rows<ORD, ORD - 1, NR>;
  using Dn = Rows<ORD - 1, ORD, NR>;
  constexpr int Q = 2 * ORD - 1;   // LDS rows of either
  const int nn = ORD == 2 ? 2 : d.nn;
  constexpr int OZ = out_rows(NR * NW);
  __shared__ float sv[NW + 2][6 * (2 * ORD - 1)][WAVE], ss[NW + 2][2 * (2 * ORD - 1)][WAVE];
  int tx, tzi, grp;
  place(g, tx, tzi, grp);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < 6 * Q; ++q) sv[0][q][lane] = sv[NW + 1][q][lane] = 0.f;
#pragma unroll
    for (int q = 0; q < 2 * Q; ++q) ss[0][q][lane] = ss[NW + 1][q][lane] = 0.f;
  }
  const int x0 = nn + tx * OX, z0 = nn + tzi * OZ;
  const int c = x0 - H + lane, zt = z0 - H + wv * NR;
  const int zw1 = d.Z - nn - 1, xw1 = d.X - nn - 1;   // the window's last row and column
  const unsigned rowb = 4u * (unsigned)d.pitch, planeb = 4u * (unsigned)d.plane, fieldb = 4u * (unsigned)d.field;
  const bool own = c >= x0 && c < min(x0 + OX, xw1 + 1);
  const bool cwin = c >= nn && c <= xw1;
  auto bits = [&](int lo, int hi) -> unsigned {   // rows lo .. hi-1 of this wavefront
    const int a = min(max(lo - zt, 0), NR), b = min(max(hi - zt, 0), NR);
    return b > a ? ((1u << b) - 1u) & ~((1u << a) - 1u) : 0u;
  };
  const unsigned ownbits = bits(z0, min(z0 + OZ, zw1 + 1));
  // byte offset of this lane's point of row r in a plane (outside the grid: none, loads return 0),
  // and the same where the workgroup stores the point
  unsigned vi[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r)
    vi[r] = c >= 0 && c < d.X && zt + r >= 0 && zt + r < d.Z ? (unsigned)(zt + r) * rowb + 4u * (unsigned)c : DROP;
  auto vo = [&](int r) -> unsigned { return own && ((ownbits >> r) & 1u) ? vi[r] : DROP; };
  const Fd<ORD> D{d.c0, d.c1, ORD == 2 ? 0.f : d.c2};
  float C[4][NR], bx[NR], bz[NR];
  {
    const rsrc_t rC = rsrc(d.coef, (unsigned)NCOEF * planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const unsigned v = cwin && zt + r >= nn && zt + r <= zw1 ? vi[r] : DROP;
#pragma unroll
      for (int q = 0; q < 4; ++q) C[q][r] = bld(rC, v, (unsigned)q * planeb);
      bx[r] = bld(rC, v, BX * planeb);
      bz[r] = bld(rC, v, BZ * planeb);
    }
  }
  // absorbing-boundary factors: per column, and per row in scalar registers
  const int cc = min(max(c, 0), d.X - 1);
  const float pxn = d.pml_x[cc], pxd = d.pml_x[d.pitch + cc], pxi = d.pml_x[2 * d.pitch + cc];
  const float sx_keep = pxn * pxi, sx_a = d.dt_dx * pxi, vx_keep = pxn / pxd, vx_w = d.dt / (d.dx * pxd);
  auto uni = [](float v) -> float {
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
  };
  float sz_keep[NR], sz_a[NR], vz_keep[NR], vz_w[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int row = min(max(zt + r, 0), d.Z - 1);
    const float pzn = scalar_ld(d.pml_z + row), pzd = scalar_ld(d.pml_z + d.Z + row), pzi = scalar_ld(d.pml_z + 2 * d.Z + row);
    sz_keep[r] = uni(pzn * pzi); sz_a[r] = uni(d.dt_dz * pzi);
    vz_keep[r] = uni(pzn / pzd); vz_w[r] = uni(d.dt / (d.dz * pzd));
  }
  // masks: the free surface's wavefront (rows nn-2 .. nn+1), window columns c, c + 1 and c - 1
  int mfs = __builtin_amdgcn_readfirstlane(d.fsurf && tzi == 0 && wv == 1 ? -1 : 0);
  asm volatile("" : "+s"(mfs));
  auto in_win = [&](int x) -> int { int m = x >= nn && x <= xw1 ? -1 : 0; asm volatile("" : "+v"(m)); return m; };
  const int mcw = in_win(c), mj1 = in_win(c + 1), mm1 = in_win(c - 1), mfc = mfs & mcw;
  unsigned rbits = 0;   // rows with receivers: of the halo, too
  if (io.inj.map) {
    const bool mine = lane < NR && zt + lane >= nn && zt + lane <= zw1;
    rbits = (unsigned)__ballot(mine && io.inj.map[mine ? zt + lane : 0] > 0);
  }
  float G[6][NR];
#pragma unroll
  for (int q = 0; q < 6; ++q)
#pragma unroll
    for (int r = 0; r < NR; ++r) G[q][r] = 0.f;

  const int s_end = min((grp + 1) * io.spg, d.S);
#pragma unroll 1
  for (int s = grp * io.spg; s < s_end; ++s) {
    const int zs = scalar_ld(d.src_z + s), xs = scalar_ld(d.src_x + s);
    const bool src_here = io.gsrc && zs >= zt && zs < zt + NR && ((ownbits >> (zs - zt)) & 1u) && xs >= x0 && xs < x0 + OX;
    float f[NFIELD][NR];
    {
      const rsrc_t rIn = rsrc(io.lin + (long long)s * d.plane, (NFIELD - 1) * fieldb + planeb);
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int q = 0; q < NFIELD; ++q) f[q][r] = bld(rIn, vi[r], (unsigned)q * fieldb);
    }
#pragma unroll 1
    for (int i = 0; i < io.n; ++i) {
      const int t = io.t - i;
      float vx[NR], vz[NR], xx[NR], zz[NR], xz[NR];
      {
        const rsrc_t rV = rsrc(io.fv[i] + (long long)s * d.plane, (NFIELD5 - 1) * fieldb + planeb);
        const rsrc_t rS = rsrc(io.fs[i] + (long long)s * d.plane, (NFIELD5 - 1) * fieldb + planeb);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          vx[r] = bld(rV, vi[r], VX * fieldb);
          vz[r] = bld(rV, vi[r], VZ * fieldb);
        }
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          xx[r] = bld(rS, vi[r], TXX * fieldb);
          zz[r] = bld(rS, vi[r], TZZ * fieldb);
          xz[r] = bld(rS, vi[r], TXZ * fieldb);
        }
      }
      if (rbits) {   // record adjoints of step t, to both splits
        const long long ro = ((long long)s * d.nt + t) * d.nrec;
        auto adj = [&](int q, unsigned v) -> float {
          const float *p = io.inj.g[q];
          return bld(rsrc(p ? p + ro : nullptr, p ? 4u * (unsigned)d.nrec : 0u), v, 0u);
        };
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if ((rbits >> r) & 1u) {
            const int m = __builtin_bit_cast(int, bld(rsrc(io.inj.map + d.Z, planeb), vi[r], 0u));
            const unsigned v = cwin && m >= 0 ? 4u * (unsigned)m : DROP;
            const float axx = adj(TXX, v), azz = adj(TZZ, d.fsurf && zt + r == nn ? DROP : v), axz = adj(TXZ, v);
            const float avx = adj(VX, v), avz = adj(VZ, v);
            f[TXX_X][r] += axx; f[TXX_Z][r] += axx; f[TZZ_X][r] += azz; f[TZZ_Z][r] += azz;
            f[TXZ_X][r] += axz; f[TXZ_Z][r] += axz; f[VX_X][r] += avx; f[VX_Z][r] += avx;
            f[VZ_X][r] += avz; f[VZ_Z][r] += avz;
          }
      }
      float eb[NR], ed[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        asm volatile("" : "+v"(bx[r]), "+v"(bz[r]));   // (the products below, kept over the loops, would cost 8 registers)
        eb[r] = f[VX_Z][r] * (vz_w[r] * bx[r]);
        ed[r] = f[VZ_Z][r] * (vz_w[r] * bz[r]);
      }
      // forward free surface: velocity rows nn-2 and nn-1, stress rows nn-2 .. nn.  Bit
      // masks, not branches, here and below: the sides of a branch (or of a select, which becomes
      // one) share terms with what follows, and holding those cost 90 registers
      {
        const float vz2n = from_right(vz[2]);
        const float vz1m_n = keep(mj1, vz2n);
        const float vz1m = pick(mcw, vz[2], vz[1]);
        const float nx1 = (((vz1m_n - vz1m) + vz2n) - vz[2]) + vx[3];
        vx[1] = pick(mfc, nx1, vx[1]);
        vz[0] = pick(mfc, vz1m, vz[0]);
        vz[1] = pick(mfs, vz1m, vz[1]);
        zz[1] = pick(mfs, -zz[3], zz[1]); zz[2] = keep(~mfs, zz[2]);
        xz[1] = pick(mfs, -xz[2], xz[1]); xz[0] = pick(mfs, -xz[3], xz[0]);
      }
      Dn::put(sv, wv, 0, lane, eb);
      Up::put(sv, wv, Q, lane, ed);
      Dn::put(sv, wv, 2 * Q, lane, vx);
      Up::put(sv, wv, 3 * Q, lane, vz);
      Dn::put(sv, wv, 4 * Q, lane, zz);
      Up::put(sv, wv, 5 * Q, lane, xz);
      lds_barrier();
      {   // buoyancy gradients: velocity adjoints as they are now, forward stress derivatives
        const Dn ZZr(sv, wv, 4 * Q, lane, zz);
        const Up XZr(sv, wv, 5 * Q, lane, xz);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          const float dxf_txx = D.dxf(xx[r]), dzb_txz = D.dzb(XZr, r);
          const float dxb_txz = D.dxb(xz[r]), dzf_tzz = D.dzf(ZZr, r);
          G[4][r] += f[VX_X][r] * (vx_w * dxf_txx) + f[VX_Z][r] * (vz_w[r] * dzb_txz);
          G[5][r] += f[VZ_X][r] * (vx_w * dxb_txz) + f[VZ_Z][r] * (vz_w[r] * dzf_tzz);
          pin(G[4][r], G[5][r]);
        }
      }
      float P1[NR], Q2[NR], Q3[NR], P4[NR];
      {
        const Dn EB(sv, wv, 0, lane, eb), VXr(sv, wv, 2 * Q, lane, vx);
        const Up ED(sv, wv, Q, lane, ed), VZr(sv, wv, 3 * Q, lane, vz);
        float ltxz0 = 0.f, ltxz1 = 0.f, ltzz1 = 0.f;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          const float ea = f[VX_X][r] * (vx_w * bx[r]), ec = f[VZ_X][r] * (vx_w * bz[r]);
          const float lt_xx = D.dxfT(ea);
          float lt_xz = D.dzbT(EB, r) + D.dxbT(ec), lt_zz = D.dzfT(ED, r);
          // stress free surface transposed
          if (r == 0) ltxz0 = keep(mfs, lt_xz);
          if (r == 1) { ltzz1 = keep(mfs, lt_zz); ltxz1 = keep(mfs, lt_xz); }
          if (r == 2) { lt_zz = keep(~mfs, lt_zz); lt_xz = lt_xz - ltxz1; }
          if (r == 3) { lt_zz = lt_zz - ltzz1; lt_xz = lt_xz - ltxz0; }
          f[TXX_X][r] += lt_xx; f[TXX_Z][r] += lt_xx;
          f[TZZ_X][r] += lt_zz; f[TZZ_Z][r] += lt_zz;
          f[TXZ_X][r] += lt_xz; f[TXZ_Z][r] += lt_xz;
          const float lxx_x = f[TXX_X][r], lxx_z = f[TXX_Z][r];
          const float lzz_x = f[TZZ_X][r], lzz_z = f[TZZ_Z][r];
          const float lxz_x = f[TXZ_X][r], lxz_z = f[TXZ_Z][r];
          const float axx_x = sx_a * lxx_x, axx_z = sz_a[r] * lxx_z;
          const float azz_x = sx_a * lzz_x, azz_z = sz_a[r] * lzz_z;
          const float axz_x = sx_a * lxz_x, axz_z = sz_a[r] * lxz_z;
          P1[r] = C[0][r] * axx_x + C[1][r] * azz_x;
          Q2[r] = C[1][r] * axx_z + C[2][r] * azz_z;
          Q3[r] = C[3][r] * axz_x;
          P4[r] = C[3][r] * axz_z;
          const float dxb_vx = D.dxb(vx[r]), dzb_vz = D.dzb(VZr, r);
          const float dxf_vz = D.dxf(vz[r]), dzf_vx = D.dzf(VXr, r);
          G[0][r] += axx_x * dxb_vx;
          G[1][r] += axx_z * dzb_vz + azz_x * dxb_vx;
          G[2][r] += azz_z * dzb_vz;
          G[3][r] += axz_x * dxf_vz + axz_z * dzf_vx;
          pin(G[0][r], G[1][r]); pin(G[2][r], G[3][r]);
          pin(P1[r], Q2[r]); pin(Q3[r], P4[r]);
        }
      }
      Dn::put(ss, wv, 0, lane, Q2);
      Up::put(ss, wv, Q, lane, P4);
      if (src_here) {
        const float mxx = d.src_m[3 * s], mzz = d.src_m[3 * s + 1], mxz = d.src_m[3 * s + 2];
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (zs == zt + r && c == xs) {
            float gm = (mxx * (f[TXX_X][r] + f[TXX_Z][r]) + mzz * (f[TZZ_X][r] + f[TZZ_Z][r])) +
                       mxz * (f[TXZ_X][r] + f[TXZ_Z][r]);
            if (d.src_fz) gm = gm + 0.5f * (d.src_fz[s] * (f[VZ_X][r] + f[VZ_Z][r]));
            io.gsrc[(long long)s * d.nt + t] = gm;
          }
      }
      lds_barrier();
      {
        const Dn Q2r(ss, wv, 0, lane, Q2);
        const Up P4r(ss, wv, Q, lane, P4);
        float lvz0 = 0.f, lvz1 = 0.f, lvx1 = 0.f;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          float lvx = D.dxbT(P1[r]) + D.dzfT(P4r, r), lvz = D.dzbT(Q2r, r) + D.dxfT(Q3[r]);
          if (r == 0) lvz0 = lvz;
          if (r == 1) { lvz1 = lvz; lvx1 = lvx; }
          if (r == 2) lvz = lvz + keep(mfs, ((lvz1 + lvz0) - 2.0f * lvx1) + keep(mm1, 2.0f * from_left(lvx1)));
          if (r == 3) lvx = lvx + keep(mfs, lvx1);
          const float l1 = f[VX_X][r], l2 = f[VX_Z][r], l3 = f[VZ_X][r], l4 = f[VZ_Z][r];
          f[TXX_X][r] = sx_keep * f[TXX_X][r]; f[TXX_Z][r] = sz_keep[r] * f[TXX_Z][r];
          f[TZZ_X][r] = sx_keep * f[TZZ_X][r]; f[TZZ_Z][r] = sz_keep[r] * f[TZZ_Z][r];
          f[TXZ_X][r] = sx_keep * f[TXZ_X][r]; f[TXZ_Z][r] = sz_keep[r] * f[TXZ_Z][r];
          f[VX_X][r] = vx_keep * l1 + lvx; f[VX_Z][r] = vz_keep[r] * l2 + lvx;
          f[VZ_X][r] = vx_keep * l3 + lvz; f[VZ_Z][r] = vz_keep[r] * l4 + lvz;
        }
      }
    }
    const rsrc_t rOut = rsrc(io.lout + (long long)s * d.plane, (NFIELD - 1) * fieldb + planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const unsigned v = vo(r);
#pragma unroll
      for (int q = 0; q < NFIELD; ++q) bst(f[q][r], rOut, v, (unsigned)q * fieldb);
    }
  }
  const rsrc_t rG = rsrc(io.gacc + (long long)grp * NCOEF * d.Z * d.pitch, (unsigned)NCOEF * planeb);
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const unsigned v = vo(r);
#pragma unroll
    for (int q = 0; q < 6; ++q) bst(bld(rG, v, (unsigned)q * planeb) + G[q][r], rG, v, (unsigned)q * planeb);
  }
}

// ---- the damping scheme (el_abl_fwd and el3_abl_fwd state a step): five fields, 40 B per point and
// step in the state alone at one step per launch, 20 B at two; records and record adjoints, which
// were launches of their own, go with the step.  182 x 361, 6 shots, us per step: forward 12.5 + 4.2
// for the records -> 5.5, adjoint 25 + 4.6 -> 12.7.  The free-surface rows nn-2 and nn-1 are state and
// stored by the first tiles.  Those rows reach one column further
// per step (forward to the right, adjoint to the left), so 8 columns on a side are halo.
constexpr int HX5 = 8;
constexpr int OX5 = WAVE - 2 * HX5;

struct AblFwdIO {
  const float *in;
  float *out[TK];        // state after each step, or NULL
  int t, n;
  ElRec rec;             // rec.map NULL: no records
};

template <int ORD, int NR, int NW>
__global__ __launch_bounds__(NW *WAVE, 4) void abl_fwd_tile(ElDev d, Grid g, AblFwdIO io) {
  static_assert(NR == 4 && H == 6, "rows nn-2 .. nn+1, which the free surface ties together, are wavefront 1 of the first tiles");
  using Up = Rows<ORD, ORD - 1, NR>;
  using Dn = Rows<ORD - 1, ORD, NR>;
  constexpr int Q = 2 * ORD - 1;
  const int nn = ORD == 2 ? 2 : d.nn;
  constexpr int OZ = out_rows(NR * NW);
  constexpr int QN = 2 * (2 * ORD - 1);
  __shared__ float sv[NW + 2][QN][WAVE], ss[NW + 2][QN][WAVE];
  int tx, tzi, s;
  place(g, tx, tzi, s);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < QN; ++q) sv[0][q][lane] = sv[NW + 1][q][lane] = ss[0][q][lane] = ss[NW + 1][q][lane] = 0.f;
  }
  const int x0 = nn + tx * OX5, z0 = nn + tzi * OZ;
  const int c = x0 - HX5 + lane, zt = z0 - H + wv * NR;
  const int zw1 = d.Z - nn - 1, xw1 = d.X - nn - 1;
  const unsigned rowb = 4u * (unsigned)d.pitch, planeb = 4u * (unsigned)d.plane, fieldb = 4u * (unsigned)d.field;
  const bool own = c >= x0 && c < min(x0 + OX5, xw1 + 1);
  auto bits = [&](int lo, int hi) -> unsigned {   // rows lo .. hi-1 of this wavefront
    const int a = min(max(lo - zt, 0), NR), b = min(max(hi - zt, 0), NR);
    return b > a ? ((1u << b) - 1u) & ~((1u << a) - 1u) : 0u;
  };
  const unsigned ownbits = bits(z0, min(z0 + OZ, zw1 + 1));
  const bool fsw = d.fsurf && tzi == 0 && wv == 1;   // this wavefront's rows are nn-2 .. nn+1
  unsigned vi[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r)
    vi[r] = c >= 0 && c < d.X && zt + r >= 0 && zt + r < d.Z ? (unsigned)(zt + r) * rowb + 4u * (unsigned)c : DROP;
  auto vo = [&](int r) -> unsigned { return own && (((ownbits | (fsw ? 3u : 0u)) >> r) & 1u) ? vi[r] : DROP; };
  auto in_win = [&](int x) -> int { int m = x >= nn && x <= xw1 ? -1 : 0; asm volatile("" : "+v"(m)); return m; };
  int mfs = __builtin_amdgcn_readfirstlane(fsw ? -1 : 0);
  asm volatile("" : "+s"(mfs));
  const int mcw = in_win(c), mj1 = in_win(c + 1), mfc = mfs & mcw;
  const Fd<ORD> D{d.c0, d.c1, ORD == 2 ? 0.f : d.c2};
  const double rdx = 1.0 / (double)d.dx, rdz = 1.0 / (double)d.dz;

  float f[NFIELD5][NR], C[4][NR], bx[NR], bz[NR], dm[NR];
  {
    const rsrc_t rIn = rsrc(io.in + (long long)s * d.plane, (NFIELD5 - 1) * fieldb + planeb);
    const rsrc_t rC = rsrc(d.coef, (unsigned)NCOEF * planeb), rD = rsrc(d.damp, planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
#pragma unroll
      for (int q = 0; q < NFIELD5; ++q) f[q][r] = bld(rIn, vi[r], (unsigned)q * fieldb);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const unsigned v = mcw && zt + r >= nn && zt + r <= zw1 ? vi[r] : DROP;
#pragma unroll
      for (int q = 0; q < 4; ++q) C[q][r] = bld(rC, v, (unsigned)q * planeb);
      bx[r] = bld(rC, v, BX * planeb);
      bz[r] = bld(rC, v, BZ * planeb);
      dm[r] = bld(rD, vi[r], 0u);
    }
  }
  const int zs = scalar_ld(d.src_z + s), xs = scalar_ld(d.src_x + s);
  const bool src_here = zs >= zt && zs < zt + NR;
  unsigned rbits = 0;
  if (io.rec.map) {
    const bool mine = lane < NR && ((ownbits >> (lane & 31)) & 1u);
    rbits = (unsigned)__ballot(mine && io.rec.map[mine ? zt + lane : 0] > 0);
  }

#pragma unroll 1
  for (int i = 0; i < io.n; ++i) {
    const float wsrc = src_here ? scalar_ld(d.src + (long long)s * d.nt + io.t + i) : 0.f;
    auto &vx = f[VX], &vz = f[VZ], &xx = f[TXX], &zz = f[TZZ], &xz = f[TXZ];
    Dn::put(sv, wv, 0, lane, vx);
    Up::put(sv, wv, Q, lane, vz);
    lds_barrier();
    {
      const Dn VXr(sv, wv, 0, lane, vx);
      const Up VZr(sv, wv, Q, lane, vz);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        __builtin_amdgcn_sched_barrier(0);
        const float dxb_vx = D.dxb(vx[r]), dzb_vz = D.dzb(VZr, r);
        const float dxf_vz = D.dxf(vz[r]), dzf_vx = D.dzf(VXr, r);
        xx[r] = xx[r] + d.dt * (quot(C[0][r] * dxb_vx, rdx) + quot(C[1][r] * dzb_vz, rdz));
        zz[r] = zz[r] + d.dt * (quot(C[1][r] * dxb_vx, rdx) + quot(C[2][r] * dzb_vz, rdz));
        xz[r] = xz[r] + d.dt * (quot(C[3][r] * dxf_vz, rdx) + quot(C[3][r] * dzf_vx, rdz));
        pin(xx[r], zz[r]);
        asm volatile("" : "+v"(xz[r]));
      }
    }
    if (src_here) {
      const float mxx = d.src_m[3 * s], mzz = d.src_m[3 * s + 1], mxz = d.src_m[3 * s + 2];
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if (zs == zt + r && c == xs) {
          xx[r] = xx[r] + mxx * wsrc;
          zz[r] = zz[r] + mzz * wsrc;
          xz[r] = xz[r] + mxz * wsrc;
        }
    }
    zz[2] = keep(~mfs, zz[2]);   // stress free surface
    zz[1] = pick(mfc, -zz[3], zz[1]);
    xz[1] = pick(mfc, -xz[2], xz[1]);
    xz[0] = pick(mfc, -xz[3], xz[0]);
    Dn::put(ss, wv, 0, lane, zz);
    Up::put(ss, wv, Q, lane, xz);
    lds_barrier();
    {
      const Dn ZZr(ss, wv, 0, lane, zz);
      const Up XZr(ss, wv, Q, lane, xz);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        __builtin_amdgcn_sched_barrier(0);
        const float dxf_txx = D.dxf(xx[r]), dzb_txz = D.dzb(XZr, r);
        const float dxb_txz = D.dxb(xz[r]), dzf_tzz = D.dzf(ZZr, r);
        vx[r] = vx[r] + (d.dt * bx[r]) * (quot(dxf_txx, rdx) + quot(dzb_txz, rdz));
        vz[r] = vz[r] + (d.dt * bz[r]) * (quot(dxb_txz, rdx) + quot(dzf_tzz, rdz));
        pin(vx[r], vz[r]);
      }
    }
    if (src_here && d.src_fz) {   // vertical force
      const float a = scalar_ld(d.src_fz + s) * wsrc;
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if (zs == zt + r && c == xs) vz[r] = vz[r] + a;
    }
    {   // velocity free surface from the new rows, then the taper
      const float vzn = from_right(vz[2]);
      const float vz1m_n = keep(mj1, vzn), vz1m = keep(mcw, vz[2]);
      const float nx1 = (((vz1m_n - vz1m) + vzn) - vz[2]) + vx[3];
      vx[1] = pick(mfc, nx1, vx[1]);
      vz[1] = pick(mfc, vz1m, vz[1]);
      vz[0] = pick(mfc, vz1m, vz[0]);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) { vx[r] = vx[r] * dm[r]; vz[r] = vz[r] * dm[r]; }
    if (rbits) {
      const long long ro = ((long long)s * d.nt + io.t + i) * d.nrec;
      const unsigned rbytes = 4u * (unsigned)d.nrec;
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if ((rbits >> r) & 1u) {
          const int m = __builtin_bit_cast(int, bld(rsrc(io.rec.map + d.Z, planeb), vi[r], 0u));
          const unsigned v = own && m >= 0 ? 4u * (unsigned)m : DROP;
#pragma unroll
          for (int q = 0; q < NFIELD5; ++q) bst(f[q][r], rsrc(io.rec.r[q] + ro, rbytes), v, 0u);
        }
    }
    float *o = io.out[i];
    const rsrc_t rOut = rsrc(o ? o + (long long)s * d.plane : nullptr, o ? (NFIELD5 - 1) * fieldb + planeb : 0u);
    if (o) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const unsigned v = vo(r);
#pragma unroll
        for (int q = 0; q < NFIELD5; ++q) bst(f[q][r], rOut, v, (unsigned)q * fieldb);
      }
    }
  }
}

// Its adjoint (el_abl_adj and el3_abl_adj list the transposes), grouped as el_adj_tile.  Stress
// adjoints outside the window take values that nothing reads or stores; the velocity adjoints of
// the free-surface rows are state.
template <int ORD, int NR, int NW>
__global__ __launch_bounds__(NW *WAVE, NW / 4) void abl_adj_tile(ElDev d, Grid g, AdjIO io) {
  static_assert(NR == 4 && H == 6, "rows nn-2 .. nn+1, which the free surface ties together, are wavefront 1 of the first tiles");
  using Up = Rows<ORD, ORD - 1, NR>;
  using Dn = Rows<ORD - 1, ORD, NR>;
  constexpr int Q = 2 * ORD - 1;
  const int nn = ORD == 2 ? 2 : d.nn;
  constexpr int OZ = out_rows(NR * NW);
  __shared__ float sv[NW + 2][6 * (2 * ORD - 1)][WAVE], ss[NW + 2][2 * (2 * ORD - 1)][WAVE];
  int tx, tzi, grp;
  place(g, tx, tzi, grp);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < 6 * Q; ++q) sv[0][q][lane] = sv[NW + 1][q][lane] = 0.f;
#pragma unroll
    for (int q = 0; q < 2 * Q; ++q) ss[0][q][lane] = ss[NW + 1][q][lane] = 0.f;
  }
  const int x0 = nn + tx * OX5, z0 = nn + tzi * OZ;
  const int c = x0 - HX5 + lane, zt = z0 - H + wv * NR;
  const int zw1 = d.Z - nn - 1, xw1 = d.X - nn - 1;
  const unsigned rowb = 4u * (unsigned)d.pitch, planeb = 4u * (unsigned)d.plane, fieldb = 4u * (unsigned)d.field;
  const bool own = c >= x0 && c < min(x0 + OX5, xw1 + 1);
  auto bits = [&](int lo, int hi) -> unsigned {   // rows lo .. hi-1 of this wavefront
    const int a = min(max(lo - zt, 0), NR), b = min(max(hi - zt, 0), NR);
    return b > a ? ((1u << b) - 1u) & ~((1u << a) - 1u) : 0u;
  };
  const unsigned ownbits = bits(z0, min(z0 + OZ, zw1 + 1));
  const bool fsw = d.fsurf && tzi == 0 && wv == 1;   // this wavefront's rows are nn-2 .. nn+1
  unsigned vi[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r)
    vi[r] = c >= 0 && c < d.X && zt + r >= 0 && zt + r < d.Z ? (unsigned)(zt + r) * rowb + 4u * (unsigned)c : DROP;
  auto vo = [&](int r) -> unsigned { return own && ((ownbits >> r) & 1u) ? vi[r] : DROP; };
  auto in_win = [&](int x) -> int { int m = x >= nn && x <= xw1 ? -1 : 0; asm volatile("" : "+v"(m)); return m; };
  int mfs = __builtin_amdgcn_readfirstlane(fsw ? -1 : 0);
  asm volatile("" : "+s"(mfs));
  const int mcw = in_win(c), mm1 = in_win(c - 1), mfc = mfs & mcw;
  const Fd<ORD> D{d.c0, d.c1, ORD == 2 ? 0.f : d.c2};
  const double rdx = 1.0 / (double)d.dx, rdz = 1.0 / (double)d.dz;
  const float dtdx = d.dt_dx, dtdz = d.dt_dz;

  float C[4][NR], bx[NR], bz[NR], dm[NR];
  {
    const rsrc_t rC = rsrc(d.coef, (unsigned)NCOEF * planeb), rD = rsrc(d.damp, planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const unsigned v = mcw && zt + r >= nn && zt + r <= zw1 ? vi[r] : DROP;
#pragma unroll
      for (int q = 0; q < 4; ++q) C[q][r] = bld(rC, v, (unsigned)q * planeb);
      bx[r] = bld(rC, v, BX * planeb);
      bz[r] = bld(rC, v, BZ * planeb);
      dm[r] = bld(rD, vi[r], 0u);
    }
  }
  unsigned rbits = 0;   // rows with receivers: of the halo, too
  if (io.inj.map) {
    const bool mine = lane < NR && zt + lane >= nn && zt + lane <= zw1;
    rbits = (unsigned)__ballot(mine && io.inj.map[mine ? zt + lane : 0] > 0);
  }
  float G[6][NR];
#pragma unroll
  for (int q = 0; q < 6; ++q)
#pragma unroll
    for (int r = 0; r < NR; ++r) G[q][r] = 0.f;

  const int s_end = min((grp + 1) * io.spg, d.S);
#pragma unroll 1
  for (int s = grp * io.spg; s < s_end; ++s) {
    const int zs = scalar_ld(d.src_z + s), xs = scalar_ld(d.src_x + s);
    const bool src_here = io.gsrc && zs >= zt && zs < zt + NR && ((ownbits >> (zs - zt)) & 1u) && xs >= x0 && xs < x0 + OX5;
    float f[NFIELD5][NR];
    {
      const rsrc_t rIn = rsrc(io.lin + (long long)s * d.plane, (NFIELD5 - 1) * fieldb + planeb);
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int q = 0; q < NFIELD5; ++q) f[q][r] = bld(rIn, vi[r], (unsigned)q * fieldb);
    }
    auto &lx = f[VX], &lz = f[VZ];
#pragma unroll 1
    for (int i = 0; i < io.n; ++i) {
      const int t = io.t - i;
      float vx[NR], vz[NR], xx[NR], zz[NR], xz[NR];
      {
        const rsrc_t rV = rsrc(io.fv[i] + (long long)s * d.plane, (NFIELD5 - 1) * fieldb + planeb);
        const rsrc_t rS = rsrc(io.fs[i] + (long long)s * d.plane, (NFIELD5 - 1) * fieldb + planeb);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          vx[r] = bld(rV, vi[r], VX * fieldb);
          vz[r] = bld(rV, vi[r], VZ * fieldb);
        }
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          xx[r] = bld(rS, vi[r], TXX * fieldb);
          zz[r] = bld(rS, vi[r], TZZ * fieldb);
          xz[r] = bld(rS, vi[r], TXZ * fieldb);
        }
      }
      if (rbits) {   // record adjoints of step t
        const long long ro = ((long long)s * d.nt + t) * d.nrec;
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if ((rbits >> r) & 1u) {
            const int m = __builtin_bit_cast(int, bld(rsrc(io.inj.map + d.Z, planeb), vi[r], 0u));
            const unsigned v = mcw && m >= 0 ? 4u * (unsigned)m : DROP;
#pragma unroll
            for (int q = 0; q < NFIELD5; ++q) {
              const float *p = io.inj.g[q];
              f[q][r] += bld(rsrc(p ? p + ro : nullptr, p ? 4u * (unsigned)d.nrec : 0u),
                             q == TZZ && d.fsurf && zt + r == nn ? DROP : v, 0u);
            }
          }
      }
      // taper, then the velocity free surface transposed
#pragma unroll
      for (int r = 0; r < NR; ++r) { lx[r] = lx[r] * dm[r]; lz[r] = lz[r] * dm[r]; }
      {
        const float wz0 = lz[0], wz1 = lz[1], wx1 = lx[1];
        const float add = ((wz1 + wz0) - 2.0f * wx1) + keep(mm1, 2.0f * from_left(wx1));
        lz[0] = keep(~mfc, lz[0]);
        lz[1] = keep(~mfc, lz[1]);
        lx[1] = keep(~mfc, lx[1]);
        lz[2] = lz[2] + keep(mfc, add);
        lx[3] = lx[3] + keep(mfc, wx1);
      }
      float eb[NR], ed[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        asm volatile("" : "+v"(bx[r]), "+v"(bz[r]));   // (the products below, kept over the loops, would cost registers)
        eb[r] = lx[r] * quot(d.dt * bx[r], rdz);
        ed[r] = lz[r] * quot(d.dt * bz[r], rdz);
      }
      Dn::put(sv, wv, 0, lane, eb);
      Up::put(sv, wv, Q, lane, ed);
      Dn::put(sv, wv, 2 * Q, lane, vx);
      Up::put(sv, wv, 3 * Q, lane, vz);
      Dn::put(sv, wv, 4 * Q, lane, zz);
      Up::put(sv, wv, 5 * Q, lane, xz);
      lds_barrier();
      {   // buoyancy gradients
        const Dn ZZr(sv, wv, 4 * Q, lane, zz);
        const Up XZr(sv, wv, 5 * Q, lane, xz);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          const float dxf_txx = D.dxf(xx[r]), dzb_txz = D.dzb(XZr, r);
          const float dxb_txz = D.dxb(xz[r]), dzf_tzz = D.dzf(ZZr, r);
          G[4][r] += lx[r] * (d.dt * (quot(dxf_txx, rdx) + quot(dzb_txz, rdz)));
          G[5][r] += lz[r] * (d.dt * (quot(dxb_txz, rdx) + quot(dzf_tzz, rdz)));
          pin(G[4][r], G[5][r]);
        }
      }
      float P1[NR], Q2[NR], Q3[NR], P4[NR];
      {
        const Dn EB(sv, wv, 0, lane, eb), VXr(sv, wv, 2 * Q, lane, vx);
        const Up ED(sv, wv, Q, lane, ed), VZr(sv, wv, 3 * Q, lane, vz);
        float ltxz0 = 0.f, ltxz1 = 0.f, ltzz1 = 0.f;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          const float ea = lx[r] * quot(d.dt * bx[r], rdx), ec = lz[r] * quot(d.dt * bz[r], rdx);
          const float lt_xx = D.dxfT(ea);
          float lt_xz = D.dzbT(EB, r) + D.dxbT(ec), lt_zz = D.dzfT(ED, r);
          // stress free surface transposed; the stored tzz of row nn is a constant
          if (r == 0) ltxz0 = keep(mfs, lt_xz);
          if (r == 1) { ltzz1 = keep(mfs, lt_zz); ltxz1 = keep(mfs, lt_xz); }
          if (r == 2) lt_xz = lt_xz - ltxz1;
          if (r == 3) { lt_zz = lt_zz - ltzz1; lt_xz = lt_xz - ltxz0; }
          f[TXX][r] += lt_xx;
          f[TZZ][r] += lt_zz;
          f[TXZ][r] += lt_xz;
          if (r == 2) f[TZZ][r] = keep(~mfs, f[TZZ][r]);
          const float axx_x = dtdx * f[TXX][r], axx_z = dtdz * f[TXX][r];
          const float azz_x = dtdx * f[TZZ][r], azz_z = dtdz * f[TZZ][r];
          const float axz_x = dtdx * f[TXZ][r], axz_z = dtdz * f[TXZ][r];
          P1[r] = C[0][r] * axx_x + C[1][r] * azz_x;
          Q2[r] = C[1][r] * axx_z + C[2][r] * azz_z;
          Q3[r] = C[3][r] * axz_x;
          P4[r] = C[3][r] * axz_z;
          const float dxb_vx = D.dxb(vx[r]), dzb_vz = D.dzb(VZr, r);
          const float dxf_vz = D.dxf(vz[r]), dzf_vx = D.dzf(VXr, r);
          G[0][r] += axx_x * dxb_vx;
          G[1][r] += axx_z * dzb_vz + azz_x * dxb_vx;
          G[2][r] += azz_z * dzb_vz;
          G[3][r] += axz_x * dxf_vz + axz_z * dzf_vx;
          pin(G[0][r], G[1][r]); pin(G[2][r], G[3][r]);
          pin(P1[r], Q2[r]); pin(Q3[r], P4[r]);
        }
      }
      Dn::put(ss, wv, 0, lane, Q2);
      Up::put(ss, wv, Q, lane, P4);
      if (src_here) {
        const float mxx = d.src_m[3 * s], mzz = d.src_m[3 * s + 1], mxz = d.src_m[3 * s + 2];
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (zs == zt + r && c == xs) {
            float gm = (mxx * f[TXX][r] + mzz * f[TZZ][r]) + mxz * f[TXZ][r];
            if (d.src_fz) gm = gm + d.src_fz[s] * lz[r];
            io.gsrc[(long long)s * d.nt + t] = gm;
          }
      }
      lds_barrier();
      {
        const Dn Q2r(ss, wv, 0, lane, Q2);
        const Up P4r(ss, wv, Q, lane, P4);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          lx[r] += D.dxbT(P1[r]) + D.dzfT(P4r, r);
          lz[r] += D.dzbT(Q2r, r) + D.dxfT(Q3[r]);
        }
      }
    }
    const rsrc_t rOut = rsrc(io.lout + (long long)s * d.plane, (NFIELD5 - 1) * fieldb + planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const unsigned v = vo(r), w = own && fsw && r < 2 ? vi[r] : v;
#pragma unroll
      for (int q = 0; q < NFIELD5; ++q) bst(f[q][r], rOut, q >= VX ? w : v, (unsigned)q * fieldb);
    }
  }
  const rsrc_t rG = rsrc(io.gacc + (long long)grp * NCOEF * d.Z * d.pitch, (unsigned)NCOEF * planeb);
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const unsigned v = vo(r);
#pragma unroll
    for (int q = 0; q < 6; ++q) bst(bld(rG, v, (unsigned)q * planeb) + G[q][r], rG, v, (unsigned)q * planeb);
  }
}

}  // namespace tile
