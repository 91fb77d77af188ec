// lattice_kernels.hpp -- several steps of the multigrid cycle on one lattice level per launch.
//
// A level whose nodes form an m x m (x m) lattice, x fastest, and whose matrix couples a node only to
// the box of nodes around it (Q1: 3 per axis, Q2: 5) is smoothed in bricks: a workgroup loads the
// brick's right-hand side and iterate once, with a halo as wide as its steps reach, takes several
// damped-Jacobi steps in LDS, and writes the inner tile.  The prolongation into the level (or the cycle's
// entry, or the first step from x = 0) is fused in front, the defect and its restriction behind.  The
// halo's nodes are computed redundantly by neighbouring bricks; in exchange a level takes two to
// four launches per cycle instead of ten (a launch of a small level costs 3 to 4 us), reads its
// vectors once per launch instead of once per step, and takes each x from LDS.  What bounds it: on
// small levels the launch and one block's latency (3D Q1, 33^3 nodes in FP32: 8.2 us for a level's
// way down or up, 16 to 19 us as five launches), on large ones the LDS reads and vector instructions
// of the halo's repeated nodes.  V-cycles, one launch per step -> bricks (us): 3D Q1 L5 FP32 102 ->
// 56; solves: 2D Q2 L9 FP32 2110 -> 1206, 2D Q1 L9 with a coefficient 1560 -> 790, 2D Q1 L6 FP64 556 ->
// 307, 3D Q1 L7 FP64 3710 -> 2360.
//
// Matrix values: MODE 0, one row of values for every node inside the lattice (Q1 Laplacian; the
// values are kernel arguments, read as scalars); MODE 1, one per parity of the coordinates (2D Q2;
// a lane keeps the two rows of its column in registers); MODE 2, a row of its own for every node (2D
// Q1 with a variable coefficient; loaded once per launch into registers).  MODE 0 and 1 need the
// Dirichlet nodes to be exactly the lattice's boundary; then rows of boundary nodes are never used
// (dinv = 0 and filtered defects), whatever their values.
//
// Every node's row sum takes the terms of its matrix row in ascending column order with fused
// multiply-adds, and the steps' expressions are those of k_sweep, k_defect, k_restrict and
// k_prolong: the iterates are those of the banded kernels bit for bit (the general formats round their
// products before adding them and differ by that).
#pragma once

#include "device_common.hpp"
#include "mg_kernels.hpp"

namespace feat3_amd
{
namespace lat
{
  using mg::u32;
  using mg::u64;

  // where the iterate comes from: memory; dinv * rhs (the first step from zero); the same with
  // rhs = (inner) def, written for the later steps (the cycle's entry); memory + P x_coarse
  enum In : int { kMem = 0, kZero = 1, kEntry = 2, kProl = 3 };

  template<typename DT_>
  struct Args
  {
    u32 m, mc;                 // nodes per axis, of the next coarser lattice
    u32 nbx, nby;              // tiles along x and y
    int t[3];                  // tile extents (even)
    int hl;                    // halo below the tile
    int in, sweeps, write_x, restrict_;
    const DT_* x;
    const double* def;
    const DT_* rhs;
    DT_* rhs_out;
    const DT_* xc;
    DT_* xout;
    const DT_* dinv;           // MODE 2
    const u32* mask;           // MODE 2
    const DT_* coef;           // MODE 2: [tap][node]; MODE 1: [class][tap..., dinv]
    const u32* mask_c;
    DT_* rhs_c;
    DT_* x_c;                  // first step of the next level (null: not wanted)
    const DT_* dinv_c;
    const double* dot_r;       // with it: partials[block] = sum of r x over the tile (the cycle's last launch)
    double* partials;
    const int* status;
    DT_ k[27];                 // MODE 0
    DT_ d;
  };

  // taps (z, y, x ascending) of the 3D box: all, and without the six face neighbours (FP32 copies of
  // the 3D Q1 Laplacian drop those roundoff residues)
  constexpr u32 kTapsAll = 0x7FFFFFFu;
  constexpr u32 kTapsNoFaces = kTapsAll & ~((1u << 4) | (1u << 10) | (1u << 12) | (1u << 14) | (1u << 16) | (1u << 22));

  // the 1D factors of the Q2 transfers: weight of coarse node 2e + k in fine node 4e + q
  __device__ __forceinline__ float q2_weight(int q, int k)
  {
    const float w1 = k == 0 ? 0.375f : (k == 1 ? 0.75f : -0.125f);
    const float w3 = k == 0 ? -0.125f : (k == 1 ? 0.75f : 0.375f);
    const float even = k == (q >> 1) ? 1.0f : 0.0f;
    return q == 1 ? w1 : (q == 3 ? w3 : even);
  }

  // brick BX x BY (x BZ); a thread owns CZ consecutive nodes along the slowest axis
  template<typename DT_, int DIM_, int RAD_, int MODE_, int BX_, int BY_, int BZ_, int CZ_, u32 TAPS_>
  struct Brick
  {
    static constexpr int DIM = DIM_, RAD = RAD_, MODE = MODE_, BX = BX_, BY = BY_, BZ = BZ_, CZ = CZ_;
    static constexpr u32 TAPS = TAPS_;
    typedef DT_ DT;
    static constexpr int S1 = DIM_ == 3 ? BX_ * BY_ : BX_;        // stride along the slowest axis
    static constexpr int COL = DIM_ == 3 ? BZ_ : BY_;
    static constexpr int NT = S1 * COL / CZ_;
    static constexpr int PTS = S1 * COL;
    static constexpr int NL = 2 * RAD_ + 1;
    static constexpr int NC = DIM_ == 3 ? NL * NL : NL;           // taps of one layer
    static constexpr int NTAP = NL * NC;
    static constexpr int PAD = DIM_ == 3 ? S1 + BX_ + 1 : RAD_ * BX_ + RAD_;
    static constexpr int LDS = 2 * (PTS + 2 * PAD) * int(sizeof(DT_));
    static constexpr int RLO = RAD_ == 1 ? 1 : 3, RHI = RAD_ == 1 ? 0 : 2;   // reach of the restriction
    static_assert(DIM_ == 2 || RAD_ == 1, "3D bricks: Q1");
    static_assert(COL % CZ_ == 0 && NT <= 1024 && NT % 64 == 0, "whole waves");
  };

  template<typename B_>
  __global__ __launch_bounds__(B_::NT) void k_lattice(Args<typename B_::DT> a)
  {
    typedef typename B_::DT DT;
    constexpr int DIM = B_::DIM, RAD = B_::RAD, MODE = B_::MODE, BX = B_::BX, BY = B_::BY, S1 = B_::S1, CZ = B_::CZ;
    constexpr int NL = B_::NL, NC = B_::NC, NTAP = B_::NTAP, PAD = B_::PAD, NT = B_::NT;
    if(mg::stopped(a.status)) return;
    extern __shared__ double lat_lds_[];
    DT* const buf0 = reinterpret_cast<DT*>(lat_lds_) + PAD;
    DT* const buf1 = buf0 + B_::PTS + 2 * PAD;
    const int tid = int(threadIdx.x);
    const u32 blk = dev::xcd_remap(blockIdx.x, gridDim.x);
    const u32 tbx = blk % a.nbx, tby = (blk / a.nbx) % a.nby, tbz = blk / (a.nbx * a.nby);
    const int m = int(a.m);
    // lattice position of the brick's first node; the slowest axis is z (3D) or y (2D)
    const int ox = int(tbx) * a.t[0] - a.hl, oy = int(tby) * a.t[1] - a.hl;
    const int oc = DIM == 3 ? int(tbz) * a.t[2] - a.hl : oy;
    const int tc = DIM == 3 ? a.t[2] : a.t[1];
    const int q = tid % S1, l0 = (tid / S1) * CZ;
    const int lx = q % BX, ly = DIM == 3 ? q / BX : 0;
    const int gx = ox + lx, gy = DIM == 3 ? oy + ly : 0, gc0 = oc + l0;
    const u32 line = u32(m), layer = DIM == 3 ? line * line : line;
    const u32 i0 = u32(gc0) * layer + (DIM == 3 ? u32(gy) * line : 0u) + u32(gx);   // wraps outside; not used there
    const bool in_xy = u32(gx) < a.m && (DIM == 2 || u32(gy) < a.m);
    const bool mid_xy = gx >= 1 && gx <= m - 2 && (DIM == 2 || (gy >= 1 && gy <= m - 2));
    const bool own_xy = in_xy && lx >= a.hl && lx < a.hl + a.t[0] && (DIM == 2 || (ly >= a.hl && ly < a.hl + a.t[1]));
    auto inside = [&](int j) { return in_xy && u32(gc0 + j) < a.m; };
    auto owned = [&](int j) { return own_xy && l0 + j >= a.hl && l0 + j < a.hl + tc && u32(gc0 + j) < a.m; };

    // the thread's matrix rows, dinv and Dirichlet flags
    constexpr int NROW = MODE == 2 ? CZ : (MODE == 1 ? 2 : 1);
    constexpr int NREG = MODE == 0 ? 1 : NTAP;
    DT kr[NROW][NREG], dv[CZ];
    bool fixed[CZ];
    if constexpr(MODE == 0)
    {
#pragma unroll
      for(int j = 0; j < CZ; ++j)
      {
        fixed[j] = !(mid_xy && gc0 + j >= 1 && gc0 + j <= m - 2);
        dv[j] = fixed[j] ? DT(0) : a.d;
      }
    }
    else if constexpr(MODE == 1)
    {
      // class = parity of y * 2 + parity of x; the column starts at an even y
      static_assert(MODE != 1 || CZ % 2 == 0, "columns of whole periods");
      const u32 px = u32(gx) & 1u;
#pragma unroll
      for(int r = 0; r < 2; ++r)
#pragma unroll
        for(int t = 0; t < NTAP; ++t) kr[r][t] = a.coef[(u32(r) * 2u + px) * u32(NTAP + 1) + u32(t)];
      const DT d0 = a.coef[px * u32(NTAP + 1) + u32(NTAP)], d1 = a.coef[(2u + px) * u32(NTAP + 1) + u32(NTAP)];
#pragma unroll
      for(int j = 0; j < CZ; ++j)
      {
        fixed[j] = !(mid_xy && gc0 + j >= 1 && gc0 + j <= m - 2);
        dv[j] = fixed[j] ? DT(0) : ((j & 1) ? d1 : d0);
      }
    }
    else
    {
      const u64 n = u64(layer) * a.m;
#pragma unroll
      for(int j = 0; j < CZ; ++j)
      {
        const bool in = inside(j);
        const u32 i = in ? i0 + u32(j) * layer : 0u;
#pragma unroll
        for(int t = 0; t < NTAP; ++t)
        {
          const DT v = a.coef[u64(t) * n + i];
          kr[j][t] = in ? v : DT(0);
        }
        const DT d = a.dinv[i];
        const bool f = dev::masked_nn(a.mask, i);
        dv[j] = in ? d : DT(0);
        fixed[j] = !in || f;
      }
    }

    // right-hand side and first iterate
    // (one uniform branch per array, so that the column's loads are in flight together)
    DT xr[CZ], b[CZ];
    u32 at[CZ];
#pragma unroll
    for(int j = 0; j < CZ; ++j) at[j] = inside(j) ? i0 + u32(j) * layer : 0u;
    if(a.in == kEntry)
    {
      double v[CZ];
#pragma unroll
      for(int j = 0; j < CZ; ++j) v[j] = a.def[at[j]];
#pragma unroll
      for(int j = 0; j < CZ; ++j)
      {
        b[j] = inside(j) ? DT(v[j]) : DT(0);
        if(owned(j)) a.rhs_out[at[j]] = b[j];
      }
    }
    else
    {
#pragma unroll
      for(int j = 0; j < CZ; ++j) b[j] = a.rhs[at[j]];
#pragma unroll
      for(int j = 0; j < CZ; ++j) b[j] = inside(j) ? b[j] : DT(0);
    }
    double rv[CZ];   // (loaded ahead of the steps: behind them it cost the launch another memory latency)
    if(a.dot_r)
    {
#pragma unroll
      for(int j = 0; j < CZ; ++j) rv[j] = a.dot_r[at[j]];
    }
    else
    {
#pragma unroll
      for(int j = 0; j < CZ; ++j) rv[j] = 0.0;
    }
    if(a.in == kMem || a.in == kProl)
    {
#pragma unroll
      for(int j = 0; j < CZ; ++j) xr[j] = a.x[at[j]];
#pragma unroll
      for(int j = 0; j < CZ; ++j) xr[j] = inside(j) ? xr[j] : DT(0);
    }
    else
    {
#pragma unroll
      for(int j = 0; j < CZ; ++j) xr[j] = dv[j] * b[j];
    }
    if(a.in == kProl)
    {
#pragma clang fp contract(off)
      // the coarse nodes under the brick, then each node's interpolation from LDS (buf1)
      constexpr int CX = BX / 2 + 4, CY = BY / 2 + 4, CW = DIM == 3 ? B_::BZ / 2 + 4 : 1;
      static_assert(CX * CY * CW <= B_::PTS, "coarse nodes fit the buffer");
      const int mc = int(a.mc);
      const int sh = RAD == 1 ? 1 : 2;     // fine nodes per coarse step (Q1) or element (Q2)
      const int cx0 = (ox >> sh) << (sh - 1), cy0 = (oy >> sh) << (sh - 1), cz0 = DIM == 3 ? oc >> 1 : 0;
      for(int k = tid; k < CX * CY * CW; k += NT)
      {
        const int kx = k % CX, ky = (k / CX) % CY, kz = k / (CX * CY);
        const int x = cx0 + kx, y = cy0 + ky, z = cz0 + kz;
        const bool in = x >= 0 && x < mc && y >= 0 && y < mc && z >= 0 && (DIM == 2 || z < mc);
        const u32 i = in ? (DIM == 3 ? u32(z) * a.mc * a.mc : 0u) + u32(y) * a.mc + u32(x) : 0u;
        const DT v = a.xc[i];
        buf1[k] = in ? v : DT(0);
      }
      __syncthreads();
#pragma unroll
      for(int j = 0; j < CZ; ++j)
      {
        if(fixed[j]) continue;
        DT s = DT(0);
        if constexpr(RAD == 1)
        {
          const int gz = DIM == 3 ? gc0 + j : 0, y = DIM == 3 ? gy : gc0 + j;
          const DT* c = buf1 + (((DIM == 3 ? (gz >> 1) - cz0 : 0) * CY + ((y >> 1) - cy0)) * CX + ((gx >> 1) - cx0));
#pragma unroll
          for(int az = 0; az < (DIM == 3 ? 2 : 1); ++az)
#pragma unroll
            for(int ay = 0; ay < 2; ++ay)
#pragma unroll
              for(int ax = 0; ax < 2; ++ax)
              {
                const bool term = (az == 0 || (gz & 1)) && (ay == 0 || (y & 1)) && (ax == 0 || (gx & 1));
                const DT w = DT(((DIM == 3 && (gz & 1)) ? 0.5f : 1.0f) * ((y & 1) ? 0.5f : 1.0f) * ((gx & 1) ? 0.5f : 1.0f));
                const DT p = w * c[(az * CY + ay) * CX + ax];
                const DT s2 = s + p;
                s = term ? s2 : s;
              }
        }
        else
        {
          const int y = gc0 + j, qx = gx & 3, qy = y & 3;
          const DT* c = buf1 + ((2 * (y >> 2) - cy0) * CX + (2 * (gx >> 2) - cx0));
#pragma unroll
          for(int ay = 0; ay < 3; ++ay)
#pragma unroll
            for(int ax = 0; ax < 3; ++ax)
            {
              const DT wy = DT(q2_weight(qy, ay)), wx = DT(q2_weight(qx, ax));
              const DT v = wy * wx;
              const DT p = v * c[ay * CX + ax];
              const DT s2 = s + p;
              s = (wy != DT(0) && wx != DT(0)) ? s2 : s;
            }
        }
        xr[j] = xr[j] + s;
      }
    }
    DT* cur = buf0;
    DT* oth = buf1;
    {
      DT* o = cur + l0 * S1 + q;
#pragma unroll
      for(int j = 0; j < CZ; ++j) o[j * S1] = xr[j];
    }
    __syncthreads();

    // s[j] = sum over the taps of node j of the column (terms in ascending column order)
    auto row_sums = [&](const DT* src, DT (&s)[CZ]) {
      const DT* p = src + l0 * S1 + q;
#pragma unroll
      for(int j = 0; j < CZ; ++j) s[j] = DT(0);
#pragma unroll
      for(int pl = -RAD; pl < CZ + RAD; ++pl)
      {
        DT v[NC];
#pragma unroll
        for(int c = 0; c < NC; ++c)
        {
          const int dx = c % NL - RAD, dy = DIM == 3 ? c / NL - RAD : 0;
          v[c] = p[pl * S1 + dy * BX + dx];
        }
#pragma unroll
        for(int l = 0; l < NL; ++l)
        {
          const int j = pl - l + RAD;
          if(j < 0 || j >= CZ) continue;
#pragma unroll
          for(int c = 0; c < NC; ++c)
          {
            const int t = l * NC + c;
            if(DIM == 3 && !((B_::TAPS >> t) & 1u)) continue;
            const DT k = MODE == 0 ? a.k[t] : kr[MODE == 2 ? j : (j & 1)][MODE == 0 ? 0 : t];
            s[j] = mg::fmadd(k, v[c], s[j]);
          }
        }
      }
    };
    // nodes that the steps behind this one still read: the tile and e_lo / e_hi nodes around it
    auto needed = [&](int e_lo, int e_hi) {
      return lx >= a.hl - e_lo && lx < a.hl + a.t[0] + e_hi && (DIM == 2 || (ly >= a.hl - e_lo && ly < a.hl + a.t[1] + e_hi)) &&
             l0 + CZ > a.hl - e_lo && l0 < a.hl + tc + e_hi;
    };
    const int r_lo = a.restrict_ ? RAD + B_::RLO : 0, r_hi = a.restrict_ ? RAD + B_::RHI : 0;
    for(int k = 0; k < a.sweeps; ++k)
    {
      const int left = (a.sweeps - 1 - k) * RAD;
      if(needed(left + r_lo, left + r_hi))
      {
        DT s[CZ];
        row_sums(cur, s);
        DT* o = oth + l0 * S1 + q;
#pragma unroll
        for(int j = 0; j < CZ; ++j)
        {
          xr[j] = xr[j] + dv[j] * (b[j] - s[j]);
          o[j * S1] = xr[j];
        }
      }
      __syncthreads();
      DT* const t = cur; cur = oth; oth = t;
    }
    if(a.write_x)
    {
#pragma unroll
      for(int j = 0; j < CZ; ++j)
        if(owned(j)) a.xout[i0 + u32(j) * layer] = xr[j];
    }
    if(a.dot_r)
    {
      double v = 0.0;
#pragma unroll
      for(int j = 0; j < CZ; ++j)
        if(owned(j)) v += rv[j] * double(xr[j]);
      dev::block_partial(v, a.partials);
    }
    if(!a.restrict_) return;
    if(needed(B_::RLO, B_::RHI))
    {
      DT s[CZ];
      row_sums(cur, s);
      DT* o = oth + l0 * S1 + q;
#pragma unroll
      for(int j = 0; j < CZ; ++j) o[j * S1] = fixed[j] ? DT(0) : b[j] - s[j];
    }
    __syncthreads();
    {
#pragma clang fp contract(off)
      // rhs_c = filter(R def) on the tile's coarse nodes (fine node 2I), terms in ascending order
      const int hx = a.t[0] / 2, hy = a.t[1] / 2, hz = DIM == 3 ? a.t[2] / 2 : 1;
      for(int k = tid; k < hx * hy * hz; k += NT)
      {
        const int ix = k % hx, iy = (k / hx) % hy, iz = k / (hx * hy);
        const u32 cx = tbx * u32(hx) + u32(ix), cy = tby * u32(hy) + u32(iy), cz = DIM == 3 ? tbz * u32(hz) + u32(iz) : 0u;
        if(cx >= a.mc || cy >= a.mc || (DIM == 3 && cz >= a.mc)) continue;
        const DT* f = oth + (DIM == 3 ? (a.hl + 2 * iz) * S1 : 0) + (a.hl + 2 * iy) * BX + a.hl + 2 * ix;
        DT s = DT(0);
        if constexpr(RAD == 1)
        {
#pragma unroll
          for(int z = (DIM == 3 ? -1 : 0); z <= (DIM == 3 ? 1 : 0); ++z)
#pragma unroll
            for(int y = -1; y <= 1; ++y)
#pragma unroll
              for(int x = -1; x <= 1; ++x)
              {
                const DT w = DT((z ? 0.5f : 1.0f) * (y ? 0.5f : 1.0f) * (x ? 0.5f : 1.0f));
                const DT p = w * f[z * S1 + y * BX + x];
                s = s + p;
              }
        }
        else
        {
          // a vertex of the coarse mesh (even index) gathers from -3, -1, 0, 1, 3, an element's
          // middle node from -1, 0, 1
#pragma unroll
          for(int y = -3; y <= 3; ++y)
#pragma unroll
            for(int x = -3; x <= 3; ++x)
            {
              if(y == -2 || y == 2 || x == -2 || x == 2) continue;
              const bool vy = (cy & 1u) == 0u, vx = (cx & 1u) == 0u;
              const DT wy = DT(y == 0 ? 1.0f : ((y == 1 || y == -1) ? (vy ? 0.375f : 0.75f) : -0.125f));
              const DT wx = DT(x == 0 ? 1.0f : ((x == 1 || x == -1) ? (vx ? 0.375f : 0.75f) : -0.125f));
              const bool term = (vy || (y >= -1 && y <= 1)) && (vx || (x >= -1 && x <= 1));
              const DT w = wy * wx;
              const DT p = w * f[y * BX + x];
              const DT s2 = s + p;
              s = term ? s2 : s;
            }
        }
        const u32 i = (DIM == 3 ? cz * a.mc * a.mc : 0u) + cy * a.mc + cx;
        const DT r = dev::masked_nn(a.mask_c, i) ? DT(0) : s;
        a.rhs_c[i] = r;
        if(a.x_c) a.x_c[i] = a.dinv_c[i] * r;
      }
    }
  }

  // ---- large 3D levels: one step per launch, columns in registers ------------------------------
  //
  // On a large 3D lattice the bricks' halos cost more than the launches they save (129^3 nodes, FP32:
  // 29.5 us for two steps, 2.4 times the nodes).  Here a thread takes CX consecutive nodes of CZ
  // planes: it loads each line of x it needs once (CX + 2 values by vector loads, 3 lines of CZ + 2
  // planes), so a node costs 9 loaded values instead of 27, no halo is computed twice and the
  // matrix row comes from scalar registers.  The lines of a plane are taken end to end (a group may
  // run over a line's end; the nodes at line ends are boundary nodes, whose sums are not used).
  // Blocks of one XCD take consecutive planes, whose x, rhs and result fit its L2.  Measured, 129^3
  // nodes, value-coded band -> columns: FP32 step 13.6 -> 7.8 us (3 vectors, 25.8 MB: 3.3 TB/s), FP64
  // step 35.4 -> 11.4 us and outer product 35.3 -> 11.8 us (51.5 and 34.3 MB); a copy of 1 GiB runs at
  // 5.1 TB/s.  Shapes CX x CZ in FP32: 4x2 7.8, 2x4 7.8, 4x4 8.4, 4x8 11.3 us (few blocks, or few loads
  // shared); FP64: 2x4 11.4, 2x2 11.6, 4x2 12.0, 2x8 13.9 us.
  constexpr int kColThreads = 256;
  template<typename DT_> struct ColShape { static constexpr int CX = sizeof(DT_) == 4 ? 4 : 2, CZ = sizeof(DT_) == 4 ? 2 : 4; };

  // kColZero: a step from the first step's iterate dinv .* rhs, formed where it is read (no x); kColLast: a
  // step with the partials of r . out; kColProduct commits the new gamma (mg::commit_gamma)
  enum ColOp : int { kColSweep = 0, kColDefect = 1, kColProduct = 2, kColInit = 3, kColZero = 4, kColLast = 5 };

  template<typename DT_>
  struct ColArgs
  {
    u32 m, mm, groups, gblocks;   // nodes per axis and plane, groups of CX nodes per plane, blocks per z chunk
    u64 div;                      // mg::udiv_magic multiplier of m
    const DT_* x;
    const DT_* rhs;
    DT_* out;
    double* partials;             // per block: kColProduct out . x, kColInit out . out, kColLast r . out
    const double* r;              // kColLast
    mg::PcgState* st;             // kColProduct
    const int* status;
    DT_ k[27];
    DT_ d;
  };

  // W consecutive values from index i (any alignment); out of [0, n) the nearest value inside
  template<int W, typename T>
  __device__ __forceinline__ void load_line(const T* __restrict__ p, int i, int n, T (&o)[W])
  {
    if(i >= 0 && i + W <= n)
    {
      typedef T v2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
      typedef T v4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
      constexpr int Q = sizeof(T) == 4 ? W / 4 * 4 : 0;
      if constexpr(sizeof(T) == 4)
      {
#pragma unroll
        for(int k = 0; k < Q; k += 4)
        {
          const v4 v = *reinterpret_cast<const v4*>(p + i + k);
          o[k] = v[0]; o[k + 1] = v[1]; o[k + 2] = v[2]; o[k + 3] = v[3];
        }
      }
#pragma unroll
      for(int k = Q; k + 1 < W; k += 2)
      {
        const v2 v = *reinterpret_cast<const v2*>(p + i + k);
        o[k] = v[0]; o[k + 1] = v[1];
      }
    }
    else
    {
#pragma unroll
      for(int k = 0; k < W; ++k)
      {
        const int j = i + k;
        o[k] = p[j < 0 ? 0 : (j < n ? j : n - 1)];
      }
    }
  }

  template<typename DT_, u32 TAPS_, int OP_>
  __global__ __launch_bounds__(kColThreads) void k_columns(ColArgs<DT_> a)
  {
    if(mg::stopped(a.status)) return;
    constexpr int CX = ColShape<DT_>::CX, CZ = ColShape<DT_>::CZ;
    const u32 blk = dev::xcd_remap(blockIdx.x, gridDim.x);
    const u32 zc = blk / a.gblocks, g = (blk % a.gblocks) * u32(kColThreads) + threadIdx.x;
    const int m = int(a.m), mm = int(a.mm), n = mm * m;
    const int z0 = int(zc) * CZ, q0 = int(g) * CX;
    double dot = 0.0;
    if constexpr(OP_ == kColProduct) mg::commit_gamma(a.st);
    if(g < a.groups)
    {
      const u32 y0 = mg::udiv_magic(u32(q0), a.div), x0 = u32(q0) - y0 * a.m;
      // kColZero: dinv at the loaded nodes of an inner plane
      DT_ dz[3][CX + 2];
      if constexpr(OP_ == kColZero)
      {
#pragma unroll
        for(int y = 0; y < 3; ++y)
#pragma unroll
          for(int k = 0; k < CX + 2; ++k)
          {
            int lx = int(x0) + k - 1, ly = int(y0) + y - 1;
            if(lx < 0) { lx += m; --ly; }
            if(lx >= m) { lx -= m; ++ly; }
            dz[y][k] = lx >= 1 && lx + 1 < m && ly >= 1 && ly + 1 < m ? a.d : DT_(0);
          }
      }
      DT_ s[CZ][CX], xc[CZ][CX];
#pragma unroll
      for(int j = 0; j < CZ; ++j)
#pragma unroll
        for(int c = 0; c < CX; ++c) { s[j][c] = DT_(0); xc[j][c] = DT_(0); }
#pragma unroll
      for(int pl = -1; pl <= CZ; ++pl)
      {
        const int z = z0 + pl;
        if(z < 0 || z >= m) continue;   // (planes outside: only boundary nodes reach them)
        DT_ v[3][CX + 2];
#pragma unroll
        for(int y = 0; y < 3; ++y)
          load_line<CX + 2>(OP_ == kColZero ? a.rhs : a.x, z * mm + q0 + (y - 1) * m - 1, n, v[y]);
        if constexpr(OP_ == kColZero)
        {
          const bool mid = z >= 1 && z + 1 < m;
#pragma unroll
          for(int y = 0; y < 3; ++y)
#pragma unroll
            for(int k = 0; k < CX + 2; ++k) v[y][k] = (mid ? dz[y][k] : DT_(0)) * v[y][k];
        }
        if(pl >= 0 && pl < CZ)
        {
#pragma unroll
          for(int c = 0; c < CX; ++c) xc[pl][c] = v[1][c + 1];
        }
#pragma unroll
        for(int l = 0; l < 3; ++l)
        {
          const int j = pl - l + 1;
          if(j < 0 || j >= CZ) continue;
#pragma unroll
          for(int t = 0; t < 9; ++t)
          {
            if(!((TAPS_ >> (l * 9 + t)) & 1u)) continue;
#pragma unroll
            for(int c = 0; c < CX; ++c) s[j][c] = mg::fmadd(a.k[l * 9 + t], v[t / 3][c + t % 3], s[j][c]);
          }
        }
      }
#pragma unroll
      for(int j = 0; j < CZ; ++j)
      {
        const int z = z0 + j;
        if(z >= m) continue;
        const int i = z * mm + q0;
        DT_ b[CX], o[CX];
        double rv[CX];
        if constexpr(OP_ != kColProduct) load_line<CX>(a.rhs, i, n, b);
        if constexpr(OP_ == kColLast) load_line<CX>(a.r, i, n, rv);
        u32 x = x0, y = y0;
#pragma unroll
        for(int c = 0; c < CX; ++c)
        {
          const bool mid = x >= 1 && x + 1 < a.m && y >= 1 && y + 1 < a.m && z >= 1 && z + 1 < m;
          if constexpr(OP_ == kColSweep || OP_ == kColZero || OP_ == kColLast) o[c] = xc[j][c] + (mid ? a.d : DT_(0)) * (b[c] - s[j][c]);
          else if constexpr(OP_ == kColProduct) o[c] = mid ? s[j][c] : DT_(0);
          else o[c] = mid ? b[c] - s[j][c] : DT_(0);
          const bool in = q0 + c < mm;
          if constexpr(OP_ == kColProduct) dot += in ? double(o[c]) * double(xc[j][c]) : 0.0;
          if constexpr(OP_ == kColInit) dot += in ? double(o[c]) * double(o[c]) : 0.0;
          if constexpr(OP_ == kColLast) dot += in ? rv[c] * double(o[c]) : 0.0;
          ++x;
          if(x == a.m) { x = 0; ++y; }
        }
        if(q0 + CX <= mm)
        {
          typedef DT_ vc __attribute__((ext_vector_type(CX), aligned(sizeof(DT_))));
          vc w;
#pragma unroll
          for(int c = 0; c < CX; ++c) w[c] = o[c];
          *reinterpret_cast<vc*>(a.out + i) = w;
        }
        else
        {
#pragma unroll
          for(int c = 0; c < CX; ++c)
            if(q0 + c < mm) a.out[i + c] = o[c];
        }
      }
    }
    if constexpr(OP_ == kColProduct || OP_ == kColInit || OP_ == kColLast) dev::block_partial(dot, a.partials);
  }

  // x_f += P x_c on a 3D Q1 lattice: a thread takes four consecutive nodes of a line, whose coarse
  // nodes are three values of one, two or four coarse lines (terms in ascending column order; the
  // weights are powers of two).  Boundary nodes keep their value.
  template<typename DT_>
  __global__ __launch_bounds__(256) void k_prolong_q1(u32 m, u32 mc, u32 quads, u64 div, const DT_* __restrict__ xc, DT_* __restrict__ xf,
                                                      const int* status)
  {
#pragma clang fp contract(off)
    if(mg::stopped(status)) return;
    // grid: x over the quads of a plane, y the planes
    const u32 t = blockIdx.x * 256u + threadIdx.x, z = blockIdx.y + 1u;
    const u32 y = mg::udiv_magic(t, div) + 1u, x0 = (t - (y - 1u) * quads) * 4u;
    if(y + 1u >= m) return;
    const u32 oz = z & 1u, oy = y & 1u;
    const u32 cy = y >> 1, cz = z >> 1, cx = x0 >> 1;
    const bool has2 = cx + 2u < mc;
    DT_ c[2][2][3];
#pragma unroll
    for(u32 b = 0; b < 2; ++b)
#pragma unroll
      for(u32 e = 0; e < 2; ++e)
      {
        const u32 i = ((cz + (b & oz)) * mc + cy + (e & oy)) * mc + cx;
        c[b][e][0] = xc[i];
        c[b][e][1] = xc[cx + 1u < mc ? i + 1u : i];
        c[b][e][2] = xc[has2 ? i + 2u : i];
      }
    const u32 i0 = (z * m + y) * m + x0;
    const DT_ wzy = DT_((oz ? 0.5f : 1.0f) * (oy ? 0.5f : 1.0f));
    DT_ v[4];
    load_line<4>(xf, int(i0), int(m * m * m), v);
#pragma unroll
    for(u32 k = 0; k < 4; ++k)
    {
      const u32 x = x0 + k;
      DT_ s = DT_(0);
#pragma unroll
      for(u32 b = 0; b < 2; ++b)
#pragma unroll
        for(u32 e = 0; e < 2; ++e)
        {
          const DT_ w = (k & 1u) ? DT_(0.5f) * wzy : wzy;
          const DT_ s1 = s + w * c[b][e][k >> 1];
          const DT_ s2 = (k & 1u) ? s1 + w * c[b][e][(k >> 1) + 1u] : s1;
          s = ((b && !oz) || (e && !oy)) ? s : s2;
        }
      v[k] = (x < 1u || x + 1u >= m) ? v[k] : v[k] + s;
    }
    if(x0 + 4u <= m)
    {
      typedef DT_ v4 __attribute__((ext_vector_type(4), aligned(sizeof(DT_))));
      v4 w;
#pragma unroll
      for(int k = 0; k < 4; ++k) w[k] = v[k];
      *reinterpret_cast<v4*>(xf + i0) = w;
    }
    else
    {
#pragma unroll
      for(u32 k = 0; k < 4; ++k)
        if(x0 + k < m) xf[i0 + k] = v[k];
    }
  }

  // ---- setup ---------------------------------------------------------------------------------

  // The matrix row and dinv (null: not wanted) of one inner node of each class, by taps; rep, repd and flags
  // zero before.  Raises the flags 1 and 2 for an entry outside the box.  One block of 64 threads.
  template<typename DT_, typename VT_>
  __global__ __launch_bounds__(64) void k_lattice_rep(u32 m, int dim, int rad, int per, const u32* __restrict__ rp,
                                                      const u32* __restrict__ col, const VT_* __restrict__ val,
                                                      const DT_* __restrict__ dinv, int ntap, DT_* __restrict__ rep,
                                                      DT_* __restrict__ repd, int* flags)
  {
    const int nl = 2 * rad + 1;
    for(int c = 0; c < (per == 2 ? 4 : 1); ++c)
    {
      const int x = 4 + (c & 1), y = 4 + (c >> 1), z = dim == 3 ? 4 : 0;
      const u32 r = (u32(z) * m + u32(y)) * m + u32(x), e = rp[r], n = rp[r + 1] - e;
      if(n > 64u) { if(threadIdx.x == 0) atomicOr(flags, 3); return; }
      if(dinv && threadIdx.x == 0) repd[c] = dinv[r];
      if(threadIdx.x >= n) continue;
      const u32 k = col[e + threadIdx.x], kl = k / m, kz = kl / m;
      const int dx = int(k - kl * m) - x, dy = int(kl - kz * m) - y, dz = int(kz) - z, rz = dim == 3 ? rad : 0;
      if(dx < -rad || dx > rad || dy < -rad || dy > rad || dz < -rz || dz > rz) { atomicOr(flags, 3); continue; }
      rep[c * ntap + ((dz + rz) * nl + dy + rad) * nl + dx + rad] = dev::ld<DT_>(val, e + threadIdx.x);
    }
  }

  // Flags raised: 1 an entry outside the box of RAD nodes around its row's node, or a second one of the
  // same column (the general formats add both; the lattice kernels have one value per neighbour); 2 an inner row that
  // differs (any value or its dinv, as bit patterns) from its class's row in rep, a Dirichlet row with a
  // value that is not finite (the row kernels carry it into the cycle, and the solve reports it: such a
  // level keeps them, or its own table of values), or Dirichlet nodes other than the lattice's boundary.  Classes: the coordinates' parities (per = 2) or one;
  // rep[class][tap], repd[class] in the arithmetic type (dinv null: not compared).
  template<typename DT_, typename VT_>
  __global__ void k_lattice_check(u64 n, u32 m, u64 div_m, int dim, int rad, int per, const u32* __restrict__ rp, const u32* __restrict__ col,
                                  const VT_* __restrict__ val, const u32* __restrict__ mask, const DT_* __restrict__ dinv,
                                  const DT_* __restrict__ rep, const DT_* __restrict__ repd, int ntap, int* flags)
  {
    const int nl = 2 * rad + 1;
    for(u64 r = u64(blockIdx.x) * blockDim.x + threadIdx.x; r < n; r += u64(gridDim.x) * blockDim.x)
    {
      const u32 rl = mg::udiv_magic(u32(r), div_m), rz = mg::udiv_magic(rl, div_m);
      const int x = int(u32(r) - rl * m), y = int(rl - rz * m), z = int(rz);
      const bool edge = x == 0 || y == 0 || (dim == 3 && z == 0) || x == int(m) - 1 || y == int(m) - 1 || (dim == 3 && z == int(m) - 1);
      const bool dir = dev::masked(mask, r);
      int f = dir != edge ? 2 : 0;
      const int cls = per == 2 ? (y & 1) * 2 + (x & 1) : 0;
      u32 hit = 0;
      for(u32 k = rp[r]; k < rp[r + 1]; ++k)
      {
        const u32 c = col[k], cl = mg::udiv_magic(c, div_m), cz = mg::udiv_magic(cl, div_m);
        const int dx = int(c - cl * m) - x, dy = int(cl - cz * m) - y, dz = int(cz) - z;
        if(dx < -rad || dx > rad || dy < -rad || dy > rad || dz < -rad || dz > rad || (dim == 2 && dz != 0)) { f |= 3; continue; }
        const int t = ((dim == 3 ? dz + rad : 0) * nl + dy + rad) * nl + dx + rad;
        const DT_ v = dev::ld<DT_>(val, k);
        if((hit >> t) & 1u) f |= 3;
        hit |= 1u << t;
        if(dir ? !isfinite(v) : !(v == rep[cls * ntap + t])) f |= 2;
      }
      if(!dir)
        for(int t = 0; t < ntap; ++t)
          if(!((hit >> t) & 1u) && rep[cls * ntap + t] != DT_(0)) f |= 2;
      if(dinv)
      {
        const DT_ d = dinv[r];
        if(dir ? !(d == DT_(0)) : !(d == repd[cls])) f |= 2;
      }
      if(f) atomicOr(flags, f);
    }
  }

  // [tap][node] values of a 2D matrix (zero-filled before)
  template<typename DT_, typename VT_>
  __global__ void k_lattice_scatter(u64 n, u32 m, int rad, const u32* __restrict__ rp, const u32* __restrict__ col,
                                    const VT_* __restrict__ val, DT_* __restrict__ coef)
  {
    const int nl = 2 * rad + 1;
    for(u64 r = u64(blockIdx.x) * blockDim.x + threadIdx.x; r < n; r += u64(gridDim.x) * blockDim.x)
      for(u32 k = rp[r]; k < rp[r + 1]; ++k)
      {
        const int dx = int(col[k] % m) - int(r % m), dy = int(col[k] / m) - int(r / m);
        coef[u64((dy + rad) * nl + dx + rad) * n + r] = dev::ld<DT_>(val, k);
      }
  }
} // namespace lat
} // namespace feat3_amd
