// Several steps of the isotropic / VTI 4th-order PML scheme per launch on register tiles
// (included by elastic.hip; el_fwd_step states one step).
//
// A workgroup of NW wavefronts holds a tile of NW*NR rows x 64 columns of one shot in registers
// (NR rows x 1 column per lane: the ten splits and six coefficients), advances it up to TK = 2
// steps and stores the points whose stencils never left the tile: a step reaches 3 points in each
// direction (the free-surface rows 2), so 6 points on every side are halo.  x-neighbours come
// from the adjacent lanes (DPP wavefront shifts), z-neighbours from registers and, between
// wavefronts, through LDS: the edge rows of the velocity totals before the stress update, those
// of the stress totals before the velocity update.  Outside the update window the coefficients
// are zero, so the splits, zero there, stay zero without masks.
//
// What a step leaves for the adjoint is the five totals, half the bytes of the ten splits: the
// kernel writes them to a trace after every step, while the splits stay in registers between the
// launch's steps.
namespace tile {

constexpr int TK = 2;              // steps per launch (at most)
constexpr int H = 3 * TK;          // halo points per side
constexpr int OX = WAVE - 2 * H;   // stored columns
constexpr int out_rows(int rows) { return rows - 2 * H; }
constexpr unsigned DROP = 0x80000000u;   // a lane offset past every buffer (all under 2 GiB): access dropped

__device__ __forceinline__ float from_left(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_right(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}
// the exchange between wavefronts goes through LDS only: loads and stores of global memory may
// stay in flight across it
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// a value no kernel writes, at a wave-uniform address: a scalar load
template <class T>
__device__ __forceinline__ T scalar_ld(const T *p) {
  return *(const __attribute__((address_space(4))) T *)(unsigned long long)p;
}

struct Grid { int ntx, ntz; };

struct FwdIO {
  const float *in;
  float *out;
  int t, n;              // first step and number of steps (1 .. TK)
  float *trace;          // [n][5][S][Z][pitch] totals after each step, or NULL
  ElRec rec;             // rec.map NULL: no records
};

// workgroup -> (tile, shot): blocks go round-robin to the 8 XCDs, and every XCD takes a contiguous
// run of a shot's tiles, row by row, so that its L2 serves the halos neighbouring tiles share and
// joins the ends of their rows, which share cache lines, before they are written back.  (With the
// shots of one tile next to each other instead, for the sake of its coefficients: forward with a
// trace 135 against 108 us per step on 242 x 680 / 32 shots, 464 against 362 on 362 x 1040 / 48.)
__device__ __forceinline__ void place(const Grid &g, int &tx, int &tz, int &s) {
  const int n = (int)gridDim.x, b = (int)blockIdx.x;
  const int xcd = b & 7, per = n >> 3, rem = n & 7;
  const int logical = xcd * per + min(xcd, rem) + (b >> 3);
  const int nt = g.ntx * g.ntz;
  s = logical / nt;
  const int tl = logical - s * nt;
  tz = tl / g.ntx;
  tx = tl - tz * g.ntx;
}

template <int NR, int NW>
__global__ __launch_bounds__(NW *WAVE) void el_fwd_tile(ElDev d, Grid g, FwdIO io) {
  static_assert(NR == 4 && H == 6, "rows 0 .. 3, which the free surface ties together, are wavefront 1 of the first tiles");
  constexpr int OZ = out_rows(NR * NW);
  __shared__ float sv[NW + 2][6][WAVE], ss[NW + 2][6][WAVE];
  int tx, tzi, s;
  place(g, tx, tzi, s);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < 6; ++q) sv[0][q][lane] = sv[NW + 1][q][lane] = ss[0][q][lane] = ss[NW + 1][q][lane] = 0.f;
  }
  const int x0 = 2 + tx * OX, z0 = 2 + tzi * OZ;            // first stored column and row
  const int c = x0 - H + lane, zt = z0 - H + wv * NR;       // this lane's column, this wavefront's first row
  const int zw1 = d.Z - 3;
  const unsigned rowb = 4u * (unsigned)d.pitch, planeb = 4u * (unsigned)d.plane, fieldb = 4u * (unsigned)d.field;
  const unsigned vin = c >= 0 && c < d.X ? 4u * (unsigned)c : DROP;
  const bool own = c >= x0 && c < min(x0 + OX, d.X - 2);
  const unsigned vout = own ? 4u * (unsigned)c : DROP;
  const bool cwin = c >= 2 && c <= d.X - 3;
  auto bits = [&](int lo, int hi) -> unsigned {   // rows lo .. hi-1 of this wavefront
    const int a = min(max(lo - zt, 0), NR), b = min(max(hi - zt, 0), NR);
    return b > a ? ((1u << b) - 1u) & ~((1u << a) - 1u) : 0u;
  };
  const unsigned ownbits = bits(z0, min(z0 + OZ, zw1 + 1));
  auto off = [&](int row) -> unsigned { return (unsigned)min(max(row, 0), d.Z - 1) * rowb; };
  const float c0 = d.c0, c1 = d.c1;

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
      const unsigned v = cwin && zt + r >= 2 && zt + r <= zw1 ? vin : DROP;   // (dropped loads return 0)
#pragma unroll
      for (int q = 0; q < 4; ++q) C[q][r] = bld(rC, v, (unsigned)q * planeb + off(zt + r));
      bx[r] = bld(rC, v, BX * planeb + off(zt + r));
      bz[r] = bld(rC, v, BZ * planeb + off(zt + r));
    }
  }
  const int cc = min(max(c, 0), d.X - 1);
  const float pxn = d.pml_x[cc], pxd = d.pml_x[d.pitch + cc], pxi = d.pml_x[2 * d.pitch + cc];
  auto pz = [&](int k, int r) -> float { return scalar_ld(d.pml_z + k * d.Z + min(max(zt + r, 0), d.Z - 1)); };
  const int zs = scalar_ld(d.src_z + s), xs = scalar_ld(d.src_x + s);
  const bool src_here = zs >= zt && zs < zt + NR;
  const bool fsw = d.fsurf && tzi == 0 && wv == 1;          // this wavefront's rows are 0 .. 3
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
    // velocity totals, the free-surface rows 0 and 1 from rows 2 and 3
    float vx[NR], vz[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) { vx[r] = f[VX_X][r] + f[VX_Z][r]; vz[r] = f[VZ_X][r] + f[VZ_Z][r]; }
    if (fsw) {
      const bool jj1 = c + 1 >= 2 && c + 1 <= d.X - 3;
      const float vz2n = from_right(vz[2]);
      const float vz1m_n = jj1 ? vz2n : 0.0f;
      const float vz1m = cwin ? vz[2] : vz[1];
      if (cwin) {
        vx[1] = (((vz1m_n - vz1m) + vz2n) - vz[2]) + vx[3];
        vz[0] = vz1m;
      }
      vz[1] = vz1m;
    }
    sv[wv + 1][0][lane] = vx[0]; sv[wv + 1][1][lane] = vx[1]; sv[wv + 1][2][lane] = vx[NR - 1];
    sv[wv + 1][3][lane] = vz[0]; sv[wv + 1][4][lane] = vz[NR - 2]; sv[wv + 1][5][lane] = vz[NR - 1];
    lds_barrier();
    {
      const float xa = sv[wv][2][lane], xb1 = sv[wv + 2][0][lane], xb2 = sv[wv + 2][1][lane];
      const float za2 = sv[wv][4][lane], za1 = sv[wv][5][lane], zb = sv[wv + 2][3][lane];
      auto VXr = [&](int r) { return r < 0 ? xa : r == NR ? xb1 : r > NR ? xb2 : vx[r]; };
      auto VZr = [&](int r) { return r == -2 ? za2 : r == -1 ? za1 : r >= NR ? zb : vz[r]; };
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        __builtin_amdgcn_sched_barrier(0);
        const float xl1 = from_left(vx[r]), xl2 = from_left(xl1), xr1 = from_right(vx[r]);
        const float zl1 = from_left(vz[r]), zr1 = from_right(vz[r]), zr2 = from_right(zr1);
        const float dxb_vx = c0 * (vx[r] - xl1) + c1 * (xr1 - xl2);
        const float dzb_vz = c0 * (vz[r] - VZr(r - 1)) + c1 * (VZr(r + 1) - VZr(r - 2));
        const float dxf_vz = c0 * (zr1 - vz[r]) + c1 * (zr2 - zl1);
        const float dzf_vx = c0 * (VXr(r + 1) - vx[r]) + c1 * (VXr(r + 2) - VXr(r - 1));
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
          bst(d.fsurf && zt + r == 2 ? 0.0f : zz[r], rsrc(io.rec.r[TZZ] + ro, rbytes), v, 0u);
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
    ss[wv + 1][0][lane] = zz[0]; ss[wv + 1][1][lane] = zz[1]; ss[wv + 1][2][lane] = zz[NR - 1];
    ss[wv + 1][3][lane] = xz[0]; ss[wv + 1][4][lane] = xz[NR - 2]; ss[wv + 1][5][lane] = xz[NR - 1];
    lds_barrier();
    {
      const float za = ss[wv][2][lane], zb1 = ss[wv + 2][0][lane], zb2 = ss[wv + 2][1][lane];
      const float xa2 = ss[wv][4][lane], xa1 = ss[wv][5][lane], xb = ss[wv + 2][3][lane];
      auto ZZr = [&](int r) { return r < 0 ? za : r == NR ? zb1 : r > NR ? zb2 : zz[r]; };
      auto XZr = [&](int r) { return r == -2 ? xa2 : r == -1 ? xa1 : r >= NR ? xb : xz[r]; };
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        __builtin_amdgcn_sched_barrier(0);
        const float tl1 = from_left(xx[r]), tr1 = from_right(xx[r]), tr2 = from_right(tr1);
        const float ul1 = from_left(xz[r]), ul2 = from_left(ul1), ur1 = from_right(xz[r]);
        const float dxf_txx = c0 * (tr1 - xx[r]) + c1 * (tr2 - tl1);
        const float dzb_txz = c0 * (xz[r] - XZr(r - 1)) + c1 * (XZr(r + 1) - XZr(r - 2));
        const float dxb_txz = c0 * (xz[r] - ul1) + c1 * (ur1 - ul2);
        const float dzf_tzz = c0 * (ZZr(r + 1) - zz[r]) + c1 * (ZZr(r + 2) - ZZr(r - 1));
        const float pzn = pz(0, r), pzd = pz(1, r);
        f[VX_X][r] = (pxn * f[VX_X][r] + ((d.dt * bx[r]) * dxf_txx) / d.dx) / pxd;
        f[VX_Z][r] = (pzn * f[VX_Z][r] + ((d.dt * bx[r]) * dzb_txz) / d.dz) / pzd;
        f[VZ_X][r] = (pxn * f[VZ_X][r] + ((d.dt * bz[r]) * dxb_txz) / d.dx) / pxd;
        f[VZ_Z][r] = (pzn * f[VZ_Z][r] + ((d.dt * bz[r]) * dzf_tzz) / d.dz) / pzd;
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

}  // namespace tile
