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
namespace tile {

constexpr int TK = 4;              // steps per launch (at most)
constexpr int H = 3 * TK;          // halo points per side
constexpr int out_cols(int cpl) { return cpl * WAVE - 2 * H; }    // stored columns
constexpr int out_rows(int rows) { return rows - 2 * H; }          // stored rows

// value of the lane one to the left / right (0 past the wavefront's ends, which only halo
// columns see)
__device__ __forceinline__ float from_left(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_right(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}

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

// the exchange between wavefronts goes through LDS only: loads and stores of global memory may
// stay in flight across it
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// a value no kernel writes, at a wave-uniform address: a scalar load, outside the vector
// memory queue (a vector load here would make the wave wait for every prefetch issued before it)
template <class T>
__device__ __forceinline__ T scalar_ld(const T *p) {
  return *(const __attribute__((address_space(4))) T *)(unsigned long long)p;
}

struct Grid {
  int ntx, ntz, ngroups, spg;      // tiles along x and z, shot groups, shots per group
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

// workgroup -> (tile, shot group).  Blocks go round-robin to the 8 XCDs: every XCD takes a
// contiguous run of (tile, group) with the groups of one tile next to each other, so that the
// tile's coefficients are read from its L2 for all of them.
__device__ __forceinline__ void place(const Grid &g, int &tx, int &tz, int &grp) {
  const int n = (int)gridDim.x, b = (int)blockIdx.x;
  const int xcd = b & 7, per = n >> 3, rem = n & 7;
  const int logical = xcd * per + min(xcd, rem) + (b >> 3);
  const int tl = logical / g.ngroups;
  grp = logical - tl * g.ngroups;
  tz = tl / g.ntx;
  tx = tl - tz * g.ntx;
}

template <int NR, int NW, int CPL, int F>
__global__ __launch_bounds__(NW *WAVE) void ac_fwd_tile(AcDev d, Grid g, FwdIO io) {
  static_assert(NR >= 4 && H % NR + 2 < NR, "the free-surface rows fs-1 .. fs+1 lie in one wavefront");
  constexpr bool FR = (F & PF_REC) != 0, FD = (F & PF_IMGD) != 0, FP = (F & PF_IMGP) != 0;
  constexpr int OZ = out_rows(NR * NW), OX = out_cols(CPL);
  typedef Cols<CPL> C;
  __shared__ C sp[NW + 2][3][WAVE], sw[NW + 2][3][WAVE];
  int tx, tzi, grp;
  place(g, tx, tzi, grp);
  const int t = io.t + time_base(d);
  if (t < 0 || t + io.n > d.nt) return;   // a device time base outside the run: nothing to do
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
    for (int i = 0; i < io.n; ++i) {
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
      if (i + 1 < io.n) {
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
      float *const e = io.energy + (long long)grp * 2 * d.plane;
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
      if (t + io.n > d.eu_from) add(e + d.plane, eu);
    }
  }
}

}  // namespace tile
