// Several acoustic time steps per launch on register tiles (included by acoustic.hip).
//
// A workgroup of NW wavefronts holds a tile of NW*NR rows x 64*CPL columns of one shot in
// registers (NR rows x CPL columns per lane: p, u, w and the coefficients), advances it up to
// TK = 4 steps and stores the rows and columns whose stencils never left the tile.  A step
// reaches 3 points in each direction, so 4 * 3 = 12 points on every side are halo: a 64 x 128
// tile stores 40 x 104.  x-neighbours come from the adjacent lanes (DPP wavefront shifts),
// z-neighbours inside a wavefront from its own registers, and the three edge rows between
// wavefronts through LDS: one barrier after the pressure update and one after the velocities.
//
// The points a step leaves alone (outside the update windows, outside the grid) carry the
// coefficients 1 and 0, so the updates run on every point of the tile without branches or
// masks: 1*x - 0*d returns x.  u is zero past column X-2, as the stage leaves it.
#include "tile_common.hpp"

namespace tile {

constexpr int TK = 4;              // steps per launch (at most)
constexpr int H = 3 * TK;          // halo points per side
constexpr int out_cols(int cpl) { return cpl * WAVE - 2 * H; }    // stored columns
constexpr int out_rows(int rows) { return rows - 2 * H; }          // stored rows

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
// a lane's CPL adjacent columns
template <int CPL>
struct Cols { float v[CPL]; };
template <int CPL>
__device__ __forceinline__ Cols<CPL> ldc(rsrc_t r, unsigned voff, unsigned soff) {
  Cols<CPL> c;
  if constexpr (CPL == 2) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
    const unsigned a = v.x, b = v.y;   // (bit_cast of a vector element reads element 0)
    c.v[0] = __builtin_bit_cast(float, a);
    c.v[1] = __builtin_bit_cast(float, b);
  } else {
    c.v[0] = bld(r, voff, soff);
  }
  return c;
}
template <int CPL>
__device__ __forceinline__ void stc(const float (&x)[CPL], rsrc_t r, unsigned voff, unsigned soff) {
  if constexpr (CPL == 2) {
    const u32x2 v = {__builtin_bit_cast(unsigned, x[0]), __builtin_bit_cast(unsigned, x[1])};
    __builtin_amdgcn_raw_buffer_store_b64(v, r, voff, soff, 0);
  } else {
    bst(x[0], r, voff, soff);
  }
}

struct Grid {
  int ntx, ntz, ngroups, spg;      // tiles along x and z, shot groups, shots per group
  int spp;                         // shots per plane of the energy maps and gradients (<= spg; a group's go to its first one)
};

struct FwdIO {
  const float *in;
  float *out;
  int t, n;                        // first step and number of steps (1 .. TK)
  float *energy;                   // [groups][2][Z][pitch] or NULL
  float *img_d, *img_p;            // images of step t (the next step's one field further) or NULL
  const int *rmap;
  float *rec_p, *rec_u, *rec_w;
};

// PF_TBASE: with a device time base; the steps that it takes outside the run are skipped.  A variant of
// its own: in the others the bounds this takes, held over the loops, cost 2 to 4 % in spilled scalars
// (296 x 808, 16 shots, ms per 1000 steps: 13.5 -> 13.8 to 14.0; this one, replayed, 12.8 -> 12.7)
constexpr int PF_TBASE = 16;

template <int NR, int NW, int CPL, int F>
__global__ __launch_bounds__(NW *WAVE) void ac_fwd_tile(AcDev d, Grid g, FwdIO io) {
  static_assert(NR >= 4 && H % NR + 2 < NR, "the free-surface rows fs-1 .. fs+1 lie in one wavefront");
  constexpr bool FR = (F & PF_REC) != 0, FD = (F & PF_IMGD) != 0, FP = (F & PF_IMGP) != 0, FT = (F & PF_TBASE) != 0;
  constexpr int OZ = out_rows(NR * NW), OX = out_cols(CPL);
  typedef Cols<CPL> C;
  __shared__ C sp[NW + 2][3][WAVE], sw[NW + 2][3][WAVE];
  int tx, tzi, grp;
  place(g, tx, tzi, grp);
  // steps t + i0 .. t + i1 - 1; with a time base t is 0, one scalar less to hold over the loops
  const int t = FT ? 0 : io.t, ta = FT ? io.t + time_base(d) : 0;
  const int i0 = FT ? max(0, ta) : 0, i1 = FT ? min(ta + io.n, d.nt) : io.n;
  if (FT && i0 >= i1) return;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      sp[0][q][lane] = sp[NW + 1][q][lane] = C{};
      sw[0][q][lane] = sw[NW + 1][q][lane] = C{};
    }
  }
  const int x0 = tx * OX, z0 = d.zbase + tzi * OZ;          // first stored column and row
  const int ca = x0 - H + CPL * lane;                       // this lane's first column
  const int zt = z0 - H + wv * NR;                          // this wavefront's first row
  const int fs = d.fs;
  const unsigned rowb = 4u * (unsigned)d.pitch, planeb = 4u * (unsigned)d.plane;
  const unsigned vin = ca >= 0 && ca < d.X ? 4u * (unsigned)ca : DROP;
  const bool own = ca >= x0 && ca < min(x0 + OX, d.X);      // (H and OX are even: all of a lane's columns or none)
  const unsigned vout = own ? 4u * (unsigned)ca : DROP;
  const int zend = min(z0 + OZ, d.Z);
  // row tests of this wavefront's rows as bits
  auto bits = [&](int lo, int hi) -> unsigned {   // rows lo .. hi-1
    const int a = min(max(lo - zt, 0), NR), b = min(max(hi - zt, 0), NR);
    return b > a ? ((1u << b) - 1u) & ~((1u << a) - 1u) : 0u;
  };
  const unsigned ownbits = bits(z0, zend), wbits = bits(z0, min(zend, d.Z - 1));
  // size of a plane for the rows that are stored, 0 for the others, whose stores are dropped: no
  // branch around a row's stores (measured 4-8 % faster with records than branches)
  auto span = [&](unsigned b, int r) -> unsigned { return (b >> r) & 1u ? planeb : 0u; };
  // row offset; rows outside the grid repeat its first or last row (no row of the windows reads them)
  auto off = [&](int row) -> unsigned { return (unsigned)min(max(row, 0), d.Z - 1) * rowb; };
  const int s0 = grp * g.spg, ns = min(g.spg, d.S - s0);

  struct State { float p[NR][CPL], u[NR][CPL], w[NR][CPL]; };
  auto load = [&](State &S, int s) {
    const long long so = (long long)s * d.plane;
    const rsrc_t rP = rsrc(io.in + so, planeb), rU = rsrc(io.in + d.field + so, planeb);
    const rsrc_t rW = rsrc(io.in + 2 * d.field + so, planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const unsigned o = off(zt + r);
      const C p = ldc<CPL>(rP, vin, o), u = ldc<CPL>(rU, vin, o), w = ldc<CPL>(rW, vin, o);
#pragma unroll
      for (int q = 0; q < CPL; ++q) { S.p[r][q] = p.v[q]; S.u[r][q] = u.v[q]; S.w[r][q] = w.v[q]; }
    }
  };
  // columns past the grid (a lane's second column, odd X) and u past column X-2 are zero
  auto clip = [&](State &S) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
#pragma unroll
      for (int q = 0; q < CPL; ++q) {
        if (q) {
          S.p[r][q] = ca + q < d.X ? S.p[r][q] : 0.f;
          S.w[r][q] = ca + q < d.X ? S.w[r][q] : 0.f;
        }
        S.u[r][q] = ca + q < d.X - 1 ? S.u[r][q] : 0.f;
      }
    }
  };
  const bool right_edge = x0 - H + CPL * WAVE >= d.X - 2;   // the tile reaches column X-2 (uniform)
  const bool edge = right_edge || zt + NR > d.Z - 2;        // ... or the wavefront row Z-2

  State S;
  load(S, s0);
  float k1[NR][CPL], a1[NR][CPL], k2[NR][CPL], a2[NR][CPL], k3[NR][CPL];
  {
    const rsrc_t rC = rsrc(coef_of(d, s0), 5u * planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int row = zt + r;
      const unsigned o = off(row);
      const bool rp = row >= fs + 1 && row <= d.Z - 3, ru = row >= fs && row <= d.Z - 2;
      const bool rw = row >= fs && row <= d.Z - 3;
      const C m0 = ldc<CPL>(rC, vin, o), m1 = ldc<CPL>(rC, vin, planeb + o), m2 = ldc<CPL>(rC, vin, 2u * planeb + o);
      const C m3 = ldc<CPL>(rC, vin, 3u * planeb + o), m4 = ldc<CPL>(rC, vin, 4u * planeb + o);
#pragma unroll
      for (int q = 0; q < CPL; ++q) {
        const int c = ca + q;
        const bool cp = c >= 2 && c <= d.X - 3, cu = c >= 1 && c <= d.X - 3, cw = c >= 1 && c <= d.X - 2;
        k1[r][q] = rp && cp ? m0.v[q] : 1.f;
        a1[r][q] = rp && cp ? m1.v[q] : 0.f;
        k2[r][q] = ru && cu ? m2.v[q] : 1.f;
        k3[r][q] = rw && cw ? m4.v[q] : 1.f;
        // one factor for u and w: their windows differ in column X-2 and row Z-2 only, where
        // the edge variant of the update keeps the old value
        a2[r][q] = (ru || rw) && (cu || cw) ? m3.v[q] : 0.f;
      }
    }
  }
  // rows of this wavefront that hold receivers and are stored by this tile
  unsigned rbits = 0;
  if (FR && io.rec_p && io.rmap) {
    const bool mine = lane < NR && ((ownbits >> (lane & 31)) & 1u);
    rbits = (unsigned)__ballot(mine && io.rmap[mine ? zt + lane : 0] > 0);
  }
  // a wavefront with one receiver row (a line of receivers) reads its indices once
  const bool one_row = rbits && !(rbits & (rbits - 1));
  C ridx{};
  if (FR && one_row) ridx = ldc<CPL>(rsrc(io.rmap + d.Z, planeb), vout, off(zt + __builtin_ctz(rbits)));
  const bool fsw = d.fsurf && tzi == 0 && wv == H / NR;     // this wavefront holds rows fs-1 .. fs+1
  constexpr int RF = H % NR;                                // ... fs-1 at this local row
  float ep[FR ? NR : 1][CPL] = {}, eu[FR ? NR : 1][CPL] = {};

  clip(S);
  // The edge variant of the velocity update: a separate march for the wavefronts that need it
  // (MODE 0 / 1), or, where the energy sums leave no registers for a second copy of the loop, a
  // separate branch inside one (MODE 2).
  auto march = [&](auto mode_) __attribute__((always_inline)) {
  constexpr int MODE = decltype(mode_)::value;
  for (int j = 0; j < ns; ++j) {
    const int s = s0 + j;
    auto &p = S.p; auto &u = S.u; auto &w = S.w;
    const int zs = scalar_ld(d.src_z + s), xs = scalar_ld(d.src_x + s);
    const bool src_here = zs >= zt && zs < zt + NR;
    C wa1, wa2, wb, pa, pb1, pb2;   // rows above (a) and below (b) this wavefront's
    auto row_of = [&](const float (&x)[CPL]) { C c; for (int q = 0; q < CPL; ++q) c.v[q] = x[q]; return c; };
    auto put_w = [&]() {
      sw[wv + 1][0][lane] = row_of(w[0]);
      sw[wv + 1][1][lane] = row_of(w[NR - 2]);
      sw[wv + 1][2][lane] = row_of(w[NR - 1]);
    };
    auto get_w = [&]() {
      lds_barrier();
      wa2 = sw[wv][1][lane]; wa1 = sw[wv][2][lane]; wb = sw[wv + 2][0][lane];
    };
    auto put_p = [&]() {
      sp[wv + 1][0][lane] = row_of(p[0]);
      sp[wv + 1][1][lane] = row_of(p[1]);
      sp[wv + 1][2][lane] = row_of(p[NR - 1]);
    };
    auto W = [&](int r, int q) -> float { return r == -2 ? wa2.v[q] : r == -1 ? wa1.v[q] : r >= NR ? wb.v[q] : w[r][q]; };
    auto P = [&](int r, int q) -> float { return r < 0 ? pa.v[q] : r == NR ? pb1.v[q] : r > NR ? pb2.v[q] : p[r][q]; };
    put_w();
    get_w();
#pragma unroll 1
    for (int i = i0; i < i1; ++i) {
      // pressure
      float *const img = FD ? io.img_d + (long long)i * d.field + (long long)s * d.plane : nullptr;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        __builtin_amdgcn_sched_barrier(0);
        float dx1[CPL], dx2[CPL], dd[CPL];    // u[j] - u[j-1], u[j+1] - u[j-2]
        if constexpr (CPL == 2) {
          const float ul0 = from_left(u[r][0]), ul1 = from_left(u[r][1]), ur0 = from_right(u[r][0]);
          dx1[0] = u[r][0] - ul1; dx2[0] = u[r][1] - ul0;
          dx1[1] = u[r][1] - u[r][0]; dx2[1] = ur0 - ul1;
        } else {
          const float ul1 = from_left(u[r][0]), ul2 = from_left(ul1);
          dx1[0] = u[r][0] - ul1; dx2[0] = from_right(u[r][0]) - ul2;
        }
#pragma unroll
        for (int q = 0; q < CPL; ++q) {
          dd[q] = C1 * ((dx1[q] + w[r][q]) - W(r - 1, q)) + C2 * ((dx2[q] + W(r + 1, q)) - W(r - 2, q));
          p[r][q] = k1[r][q] * p[r][q] - a1[r][q] * dd[q];
        }
        if constexpr (FD) stc<CPL>(dd, rsrc(img, span(ownbits, r)), vout, off(zt + r));
      }
      if (src_here) {
        const float sv = scalar_ld(d.src + (long long)s * d.nt + t + i);
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (zs == zt + r) {
#pragma unroll
            for (int q = 0; q < CPL; ++q) p[r][q] = ca + q == xs ? p[r][q] + sv : p[r][q];
          }
      }
      if (fsw) {   // free surface: p[fs-1] = -p[fs+1]
#pragma unroll
        for (int q = 0; q < CPL; ++q) p[RF][q] = -p[RF + 2][q];
      }
      put_p();
      lds_barrier();
      pa = sp[wv][2][lane]; pb1 = sp[wv + 2][0][lane]; pb2 = sp[wv + 2][1][lane];
      // velocities
      auto velocities = [&](auto edge_) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          float dx1[CPL], dx2[CPL];    // p[j+1] - p[j], p[j+2] - p[j-1]
          if constexpr (CPL == 2) {
            const float pl1 = from_left(p[r][1]), pr0 = from_right(p[r][0]), pr1 = from_right(p[r][1]);
            dx1[0] = p[r][1] - p[r][0]; dx2[0] = pr0 - pl1;
            dx1[1] = pr0 - p[r][1]; dx2[1] = pr1 - p[r][0];
          } else {
            const float pr1 = from_right(p[r][0]);
            dx1[0] = pr1 - p[r][0]; dx2[0] = from_right(pr1) - from_left(p[r][0]);
          }
#pragma unroll
          for (int q = 0; q < CPL; ++q) {
            float un = k2[r][q] * u[r][q] - a2[r][q] * (C1 * dx1[q] + C2 * dx2[q]);
            float wn = k3[r][q] * w[r][q] - a2[r][q] * (C1 * (P(r + 1, q) - p[r][q]) + C2 * (P(r + 2, q) - P(r - 1, q)));
            if constexpr (decltype(edge_)::value) {
              un = ca + q <= d.X - 3 ? un : u[r][q];
              wn = zt + r <= d.Z - 3 ? wn : w[r][q];
            }
            u[r][q] = un;
            w[r][q] = wn;
          }
        }
      };
      if constexpr (MODE < 2) {
        velocities(std::integral_constant<bool, MODE == 1>{});
      } else {
        // two conditions, the second hidden from the compiler: as one if/else it hoists the
        // branches' common products, which costs 40 registers
        if (!edge) velocities(std::false_type{});
        int at_edge = __builtin_amdgcn_readfirstlane((int)edge);
        asm volatile("" : "+s"(at_edge));
        if (at_edge) velocities(std::true_type{});
      }
      if (fsw) {   // free surface: w[fs-1] = w[fs]
#pragma unroll
        for (int q = 0; q < CPL; ++q) w[RF][q] = w[RF + 1][q];
      }
      if (FR && rbits) {
        const long long ro = ((long long)s * d.nt + t + i) * d.nrec;
        const unsigned rbytes = 4u * (unsigned)d.nrec;
        const rsrc_t qP = rsrc(io.rec_p + ro, rbytes), qU = rsrc(io.rec_u + ro, rbytes), qW = rsrc(io.rec_w + ro, rbytes);
        const rsrc_t rM = rsrc(io.rmap + d.Z, planeb);
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if ((rbits >> r) & 1u) {
            C m = ridx;
            if (!one_row) m = ldc<CPL>(rM, vout, off(zt + r));
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
              const int idx = __builtin_bit_cast(int, m.v[q]);
              const unsigned v = own && ca + q < d.X && idx >= 0 ? 4u * (unsigned)idx : DROP;
              bst(p[r][q], qP, v, 0u);
              bst(u[r][q], qU, v, 0u);
              bst(w[r][q], qW, v, 0u);
            }
          }
      }
      if constexpr (FP) {
        float *const imp = io.img_p + (long long)i * d.field + (long long)s * d.plane;
#pragma unroll
        for (int r = 0; r < NR; ++r) stc<CPL>(p[r], rsrc(imp, span(ownbits, r)), vout, off(zt + r));
      }
      if constexpr (FR) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int q = 0; q < CPL; ++q) ep[r][q] += p[r][q] * p[r][q];
        if (t + i >= d.eu_from) {
#pragma unroll
          for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int q = 0; q < CPL; ++q) eu[r][q] += u[r][q] * u[r][q];
        }
      }
      if (i + 1 < i1) {
        put_w();
        get_w();
      }
    }
    {
      const long long so = (long long)s * d.plane;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const unsigned o = off(zt + r), b = span(ownbits, r);
        stc<CPL>(p[r], rsrc(io.out + so, b), vout, o);
        stc<CPL>(u[r], rsrc(io.out + d.field + so, b), vout, o);
        stc<CPL>(w[r], rsrc(io.out + 2 * d.field + so, span(wbits, r)), vout, o);
      }
    }
    if (j + 1 < ns) load(S, s + 1);
    clip(S);
  }
  };
  if constexpr (FR) march(std::integral_constant<int, 2>{});
  else if (edge) march(std::integral_constant<int, 1>{});
  else march(std::integral_constant<int, 0>{});
  if constexpr (FR) {
    if (io.energy) {
      float *const e = io.energy + (long long)(s0 / g.spp) * 2 * d.plane;
      auto add = [&](float *plane, const float (&sum)[FR ? NR : 1][CPL]) {
        C old[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) old[r] = ldc<CPL>(rsrc(plane, span(ownbits, r)), vout, off(zt + r));
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          float v[CPL];
#pragma unroll
          for (int q = 0; q < CPL; ++q) v[q] = old[r].v[q] + sum[r][q];
          stc<CPL>(v, rsrc(plane, span(ownbits, r)), vout, off(zt + r));
        }
      };
      add(e, ep);
      if (t + i1 > d.eu_from) add(e + d.plane, eu);
    }
  }
}

// ---------------------------------------------------------------------------
// adjoint: up to TK reversed steps per launch, the transposes of ac_fwd_tile's stages on the same
// tiles (ac_adj_step states them for one step)
// ---------------------------------------------------------------------------
struct AdjIO {
  const float *in;                 // adjoint of the state after step t, its receiver sources not added
  float *out;
  int t, n;                        // steps t, t-1, ..., t-n+1 are reversed
  const float *img_d, *img_p;      // images of step t (the step before one field back) or NULL
  float *grad_a1, *grad_a2, *grad_src;
  const int *rmap;
  const float *g_p, *g_u, *g_w;    // record adjoints [S][nt][R] or NULL
};

// FULL: u and w record adjoints or the wavelet gradient; A2: the rho gradient.  16 wavefronts leave 128
// VGPRs: with two columns per lane 9 are spilled (27 with FULL, some in the step loop), and scalars go to
// lanes of others; with one column 83 to 100 are used and none spilled.
template <int NR, int NW, int CPL, bool A2, bool FULL>
__global__ __launch_bounds__(NW *WAVE) void ac_adj_tile(AcDev d, Grid g, AdjIO io) {
  static_assert(NR >= 4 && H % NR + 2 < NR, "the free-surface rows fs-1 .. fs+1 lie in one wavefront");
  constexpr int OZ = out_rows(NR * NW), OX = out_cols(CPL);
  constexpr int NG = FULL ? 3 : 1;                // record components
  typedef Cols<CPL> C;
  __shared__ C sg[NW + 2][3][WAVE], sw[NW + 2][3][WAVE];    // rows of a1 lambda_p and of a2 lambda_w
  __shared__ C srec[NW][NG][TK][WAVE];            // record adjoints of a wavefront's receiver row
  int tx, tzi, grp;
  place(g, tx, tzi, grp);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      sg[0][q][lane] = sg[NW + 1][q][lane] = C{};
      sw[0][q][lane] = sw[NW + 1][q][lane] = C{};
    }
  }
  const int x0 = tx * OX, z0 = d.zbase + tzi * OZ;
  const int ca = x0 - H + CPL * lane;
  const int zt = z0 - H + wv * NR;
  const int fs = d.fs;
  const unsigned rowb = 4u * (unsigned)d.pitch, planeb = 4u * (unsigned)d.plane;
  const unsigned vin = ca >= 0 && ca < d.X ? 4u * (unsigned)ca : DROP;
  const bool own = ca >= x0 && ca < min(x0 + OX, d.X);
  const unsigned vout = own ? 4u * (unsigned)ca : DROP;
  const int zend = min(z0 + OZ, d.Z);
  auto bits = [&](int lo, int hi) -> unsigned {   // rows lo .. hi-1 of this wavefront
    const int a = min(max(lo - zt, 0), NR), b = min(max(hi - zt, 0), NR);
    return b > a ? ((1u << b) - 1u) & ~((1u << a) - 1u) : 0u;
  };
  const unsigned ownbits = bits(z0, zend), wbits = bits(z0, min(zend, d.Z - 1));
  // an access to row r only where mask b has it: with two columns per lane through the size of the
  // plane (as above), with one through the lane's offset, for which there are registers (one
  // descriptor per plane instead of one per row: 3-6 % faster, but with two columns it spills)
  auto span = [&](unsigned b, int r) -> unsigned { return CPL == 1 || ((b >> r) & 1u) ? planeb : 0u; };
  auto vrow = [&](unsigned b, int r) -> unsigned { return CPL > 1 || ((b >> r) & 1u) ? vout : DROP; };
  constexpr bool PIN = CPL == 1 || !FULL;   // (two columns with all records: 5 % slower pinned)
  auto off = [&](int row) -> unsigned { return (unsigned)min(max(row, 0), d.Z - 1) * rowb; };
  const int s0 = grp * g.spg, ns = min(g.spg, d.S - s0);

  float p[NR][CPL], u[NR][CPL], w[NR][CPL];       // lambda_p, lambda_u, lambda_w
  auto load = [&](int s) __attribute__((always_inline)) {
    const long long so = (long long)s * d.plane;
    const rsrc_t rP = rsrc(io.in + so, planeb), rU = rsrc(io.in + d.field + so, planeb);
    const rsrc_t rW = rsrc(io.in + 2 * d.field + so, planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const unsigned o = off(zt + r);
      const C x = ldc<CPL>(rP, vin, o), y = ldc<CPL>(rU, vin, o), z = ldc<CPL>(rW, vin, o);
#pragma unroll
      for (int q = 0; q < CPL; ++q) { p[r][q] = x.v[q]; u[r][q] = y.v[q]; w[r][q] = z.v[q]; }
    }
  };
  auto clip = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
#pragma unroll
      for (int q = 0; q < CPL; ++q) {
        if (q) {
          p[r][q] = ca + q < d.X ? p[r][q] : 0.f;
          w[r][q] = ca + q < d.X ? w[r][q] : 0.f;
        }
        u[r][q] = ca + q < d.X - 1 ? u[r][q] : 0.f;
      }
    }
  };
  const bool right_edge = x0 - H + CPL * WAVE >= d.X - 2;
  const bool edge = right_edge || zt + NR > d.Z - 2;

  load(s0);
  float k1[NR][CPL], a1[NR][CPL], k2[NR][CPL], a2[NR][CPL], k3[NR][CPL];
  {
    const rsrc_t rC = rsrc(coef_of(d, s0), 5u * planeb);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int row = zt + r;
      const unsigned o = off(row);
      const bool rp = row >= fs + 1 && row <= d.Z - 3, ru = row >= fs && row <= d.Z - 2;
      const bool rw = row >= fs && row <= d.Z - 3;
      const C m0 = ldc<CPL>(rC, vin, o), m1 = ldc<CPL>(rC, vin, planeb + o), m2 = ldc<CPL>(rC, vin, 2u * planeb + o);
      const C m3 = ldc<CPL>(rC, vin, 3u * planeb + o), m4 = ldc<CPL>(rC, vin, 4u * planeb + o);
#pragma unroll
      for (int q = 0; q < CPL; ++q) {
        const int c = ca + q;
        const bool cp = c >= 2 && c <= d.X - 3, cu = c >= 1 && c <= d.X - 3, cw = c >= 1 && c <= d.X - 2;
        k1[r][q] = rp && cp ? m0.v[q] : 1.f;
        a1[r][q] = rp && cp ? m1.v[q] : 0.f;
        k2[r][q] = ru && cu ? m2.v[q] : 1.f;
        k3[r][q] = rw && cw ? m4.v[q] : 1.f;
        a2[r][q] = (ru || rw) && (cu || cw) ? m3.v[q] : 0.f;   // (column X-2 and row Z-2: the edge variant)
      }
    }
  }
  // rows of this wavefront that hold receivers: their record adjoints enter every lane of the
  // tile, halo included
  unsigned rbits = 0;
  if (io.rmap) {
    const int row = zt + lane;
    const bool mine = lane < NR && row >= 0 && row < d.Z;
    rbits = (unsigned)__ballot(mine && io.rmap[mine ? row : 0] > 0);
  }
  const bool one_row = rbits && !(rbits & (rbits - 1));
  const bool fsw = d.fsurf && tzi == 0 && wv == H / NR;     // this wavefront holds rows fs-1 .. fs+1
  constexpr int RF = H % NR;
  float ga1[NR][CPL] = {}, ga2[A2 ? NR : 1][CPL] = {};

  auto march = [&](auto edge_) __attribute__((always_inline)) {
  constexpr bool EDGE = decltype(edge_)::value;
  for (int j = 0; j < ns; ++j) {
    const int s = s0 + j;
    // receiver slot of this lane's columns in a row, as a byte offset into a step's records
    auto slots = [&](int r, unsigned (&v)[CPL]) __attribute__((always_inline)) {
      const C m = ldc<CPL>(rsrc(io.rmap + d.Z, planeb), vin, off(zt + r));
#pragma unroll
      for (int q = 0; q < CPL; ++q) {
        const int idx = __builtin_bit_cast(int, m.v[q]);
        v[q] = vin != DROP && ca + q < d.X && idx >= 0 ? 4u * (unsigned)idx : DROP;
      }
    };
    const float *const gr[3] = {io.g_p, FULL ? io.g_u : nullptr, FULL ? io.g_w : nullptr};
    auto rec_at = [&](int c, int i) -> rsrc_t {   // records of component c in reversed step i
      return rsrc(gr[c] ? gr[c] + ((long long)s * d.nt + io.t - i) * d.nrec : nullptr, gr[c] ? 4u * (unsigned)d.nrec : 0u);
    };
    if (one_row) {   // a line of receivers: all steps' values of the row are fetched up front
      unsigned v[CPL];
      slots(__builtin_ctz(rbits), v);
#pragma unroll
      for (int c = 0; c < NG; ++c)
#pragma unroll
        for (int i = 0; i < TK; ++i) {
          C x{};
          if (i < io.n) {
#pragma unroll
            for (int q = 0; q < CPL; ++q) x.v[q] = bld(rec_at(c, i), v[q], 0u);
          }
          srec[wv][c][i][lane] = x;
        }
    }
    clip();
    const int zs = scalar_ld(d.src_z + s), xs = scalar_ld(d.src_x + s);
    const bool src_here = FULL && io.grad_src && zs >= zt && zs < zt + NR;
    auto row_of = [&](const float (&x)[CPL]) { C c; for (int q = 0; q < CPL; ++q) c.v[q] = x[q]; return c; };
#pragma unroll 1
    for (int i = 0; i < io.n; ++i) {
      const long long fi = (long long)s * d.plane - (long long)i * d.field;
      // pressures of rows -1 .. NR+1 after the step: one lane column leaves the registers to fetch
      // them this early
      C q0[A2 ? NR + 3 : 1];
      auto load_p = [&]() __attribute__((always_inline)) {
        const float *const imp = io.img_p + fi;
#pragma unroll
        for (int r = 0; r < NR + 3; ++r) q0[r] = ldc<CPL>(rsrc(imp, planeb), vin, off(zt + r - 1));
      };
      if constexpr (A2 && CPL == 1) load_p();
      // the record adjoints of the step
      if (rbits) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if ((rbits >> r) & 1u) {
            C x[NG];
            if (one_row) {
#pragma unroll
              for (int c = 0; c < NG; ++c) x[c] = srec[wv][c][i][lane];
            } else {
              unsigned v[CPL];
              slots(r, v);
#pragma unroll
              for (int c = 0; c < NG; ++c)
#pragma unroll
                for (int q = 0; q < CPL; ++q) x[c].v[q] = bld(rec_at(c, i), v[q], 0u);
            }
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
              p[r][q] = p[r][q] + x[0].v[q];
              if constexpr (FULL) {
                u[r][q] = u[r][q] + x[1].v[q];
                w[r][q] = w[r][q] + x[2].v[q];
              }
            }
          }
      }
      if (fsw) {   // stage 6 transposed: row fs gathers row fs-1
#pragma unroll
        for (int q = 0; q < CPL; ++q) {
          w[RF + 1][q] = w[RF + 1][q] + w[RF][q];
          w[RF][q] = 0.f;
        }
      }
      // stages 5 and 4 transposed: lambda_p3
      auto fw = [&](int r, int q) __attribute__((always_inline)) -> float {
        if (EDGE && zt + r > d.Z - 3) return 0.f;
        return a2[r][q] * w[r][q];
      };
      {
        C x, y, z;
#pragma unroll
        for (int q = 0; q < CPL; ++q) { x.v[q] = fw(0, q); y.v[q] = fw(NR - 2, q); z.v[q] = fw(NR - 1, q); }
        sw[wv + 1][0][lane] = x;
        sw[wv + 1][1][lane] = y;
        sw[wv + 1][2][lane] = z;
      }
      lds_barrier();
      C im[NR];
      if (io.grad_a1) {
        const float *const img = io.img_d + fi;
#pragma unroll
        for (int r = 0; r < NR; ++r) im[r] = ldc<CPL>(rsrc(img, span(ownbits, r)), vrow(ownbits, r), off(zt + r));
      }
      const C wa2 = sw[wv][1][lane], wa1 = sw[wv][2][lane], wb = sw[wv + 2][0][lane];
      {
        auto f = [&](int r, int q) -> float { return r == 0 ? wa2.v[q] : r == 1 ? wa1.v[q] : r == NR + 2 ? wb.v[q] : fw(r - 2, q); };
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          float fu[CPL], dx1[CPL], dx2[CPL];    // fu[j-1] - fu[j], fu[j-2] - fu[j+1]
#pragma unroll
          for (int q = 0; q < CPL; ++q) {
            fu[q] = a2[r][q] * u[r][q];
            if constexpr (EDGE) fu[q] = ca + q <= d.X - 3 ? fu[q] : 0.f;
          }
          if constexpr (CPL == 2) {
            const float l0 = from_left(fu[0]), l1 = from_left(fu[1]), r0 = from_right(fu[0]);
            dx1[0] = l1 - fu[0]; dx2[0] = l0 - fu[1];
            dx1[1] = fu[0] - fu[1]; dx2[1] = l1 - r0;
          } else {
            const float l1 = from_left(fu[0]), l2 = from_left(l1);
            dx1[0] = l1 - fu[0]; dx2[0] = l2 - from_right(fu[0]);
          }
#pragma unroll
          for (int q = 0; q < CPL; ++q) {
            const float dxt = C1 * dx1[q] + C2 * dx2[q];
            const float dzt = C1 * (f(r + 1, q) - f(r + 2, q)) + C2 * (f(r, q) - f(r + 3, q));
            p[r][q] = p[r][q] - (dxt + dzt);
            if constexpr (PIN) pin(p[r][q]);
          }
        }
      }
      if (fsw) {   // stage 3 transposed
#pragma unroll
        for (int q = 0; q < CPL; ++q) {
          p[RF + 2][q] = p[RF + 2][q] - p[RF][q];
          p[RF][q] = 0.f;
        }
      }
      if (FULL && src_here) {   // stage 2 transposed
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (zs == zt + r && ((ownbits >> r) & 1u)) {
#pragma unroll
            for (int q = 0; q < CPL; ++q)
              if (own && ca + q == xs) io.grad_src[(long long)s * d.nt + io.t - i] = p[r][q];
          }
      }
      if (io.grad_a1) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int q = 0; q < CPL; ++q) {
            ga1[r][q] -= p[r][q] * im[r].v[q];
            if constexpr (PIN) pin(ga1[r][q]);
          }
      }
      {
        C x, y, z;
#pragma unroll
        for (int q = 0; q < CPL; ++q) {
          x.v[q] = a1[0][q] * p[0][q]; y.v[q] = a1[1][q] * p[1][q]; z.v[q] = a1[NR - 1][q] * p[NR - 1][q];
        }
        sg[wv + 1][0][lane] = x;
        sg[wv + 1][1][lane] = y;
        sg[wv + 1][2][lane] = z;
      }
      if constexpr (A2) {   // zero-lag image of the velocity updates: the pressures after step t
        if constexpr (CPL > 1) load_p();
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const C &pc = q0[r + 1];
          float dx1[CPL], dx2[CPL];
          if constexpr (CPL == 2) {
            const float l1 = from_left(pc.v[1]), r0 = from_right(pc.v[0]), r1 = from_right(pc.v[1]);
            dx1[0] = pc.v[1] - pc.v[0]; dx2[0] = r0 - l1;
            dx1[1] = r0 - pc.v[1]; dx2[1] = r1 - pc.v[0];
          } else {
            const float r1 = from_right(pc.v[0]);
            dx1[0] = r1 - pc.v[0]; dx2[0] = from_right(r1) - from_left(pc.v[0]);
          }
#pragma unroll
          for (int q = 0; q < CPL; ++q) {
            float tu = u[r][q] * (C1 * dx1[q] + C2 * dx2[q]);
            float tw = w[r][q] * (C1 * (q0[r + 2].v[q] - pc.v[q]) + C2 * (q0[r + 3].v[q] - q0[r].v[q]));
            if constexpr (EDGE) {
              tu = ca + q <= d.X - 3 ? tu : 0.f;
              tw = zt + r <= d.Z - 3 ? tw : 0.f;
            }
            ga2[r][q] -= tu;
            ga2[r][q] -= tw;
          }
        }
      }
      lds_barrier();
      // stage 1 transposed and the adjoint state before the step
      const C gm = sg[wv][2][lane], gb1 = sg[wv + 2][0][lane], gb2 = sg[wv + 2][1][lane];
      {
        float gg[NR + 3][CPL];   // a1 lambda_p of rows -1 .. NR+1
#pragma unroll
        for (int r = 0; r < NR + 3; ++r)
#pragma unroll
          for (int q = 0; q < CPL; ++q)
            gg[r][q] = r == 0 ? gm.v[q] : r == NR + 1 ? gb1.v[q] : r == NR + 2 ? gb2.v[q] : a1[r - 1][q] * p[r - 1][q];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          const float (&gc)[CPL] = gg[r + 1];
          float dx1[CPL], dx2[CPL];    // g[j] - g[j+1], g[j-1] - g[j+2]
          if constexpr (CPL == 2) {
            const float l1 = from_left(gc[1]), r0 = from_right(gc[0]), r1 = from_right(gc[1]);
            dx1[0] = gc[0] - gc[1]; dx2[0] = l1 - r0;
            dx1[1] = gc[1] - r0; dx2[1] = gc[0] - r1;
          } else {
            const float r1 = from_right(gc[0]);
            dx1[0] = gc[0] - r1; dx2[0] = from_left(gc[0]) - from_right(r1);
          }
#pragma unroll
          for (int q = 0; q < CPL; ++q) {
            p[r][q] = k1[r][q] * p[r][q];
            u[r][q] = k2[r][q] * u[r][q] - (C1 * dx1[q] + C2 * dx2[q]);
            w[r][q] = k3[r][q] * w[r][q] - (C1 * (gc[q] - gg[r + 2][q]) + C2 * (gg[r][q] - gg[r + 3][q]));
            if constexpr (EDGE) {
              u[r][q] = ca + q < d.X - 1 ? u[r][q] : 0.f;
              w[r][q] = zt + r < d.Z - 1 ? w[r][q] : 0.f;
            }
          }
        }
      }
    }
    {
      const long long so = (long long)s * d.plane;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const unsigned o = off(zt + r), b = span(ownbits, r);
        stc<CPL>(p[r], rsrc(io.out + so, b), vrow(ownbits, r), o);
        stc<CPL>(u[r], rsrc(io.out + d.field + so, b), vrow(ownbits, r), o);
        stc<CPL>(w[r], rsrc(io.out + 2 * d.field + so, span(wbits, r)), vrow(wbits, r), o);
      }
    }
    if (j + 1 < ns) load(s + 1);
  }
  };
  if (edge) march(std::true_type{}); else march(std::false_type{});
  // the images of all steps and shots into the group's planes: points of the update windows only
  auto add = [&](float *plane, const float (&sum)[NR][CPL], int r0, int r1, int c0, int c1) __attribute__((always_inline)) {
    const unsigned b = ownbits & bits(r0, r1);
    C old[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) old[r] = ldc<CPL>(rsrc(plane, span(b, r)), vrow(b, r), off(zt + r));
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      float v[CPL];
#pragma unroll
      for (int q = 0; q < CPL; ++q) v[q] = old[r].v[q] + (ca + q >= c0 && ca + q < c1 ? sum[r][q] : 0.f);
      stc<CPL>(v, rsrc(plane, span(b, r)), vrow(b, r), off(zt + r));
    }
  };
  if (io.grad_a1) add(io.grad_a1 + (long long)(s0 / g.spp) * d.plane, ga1, fs + 1, d.Z - 2, 2, d.X - 2);
  if constexpr (A2) add(io.grad_a2 + (long long)(s0 / g.spp) * d.plane, ga2, fs, d.Z - 1, 1, d.X - 1);
}

}  // namespace tile
