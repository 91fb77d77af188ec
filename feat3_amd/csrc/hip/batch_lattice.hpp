// batch_lattice.hpp -- the batched solver's steps on 3D lattice levels whose inner rows are all alike.
//
// A node of a batched level holds ncol = B * K values (B components, K systems, system fastest).
// When the shared matrix couples the 27 nodes around a node with one row of scalar values for every
// inner node and component (a vector Laplacian on a uniform mesh), all columns take the same sums, and
// a row's loads of row pointer, columns and values go away.  A thread owns CH consecutive columns (16
// bytes) of one (x, y) line and walks along z: each plane's nine neighbours are loaded once and added
// to three running sums (the nodes above, in and below the plane), so a value is loaded 9 instead of
// 27 times, from the L1 but for the first time (a block is a tile of lines).  The next plane's values
// are loaded while one is summed.  Every sum takes its terms in ascending column order with fused
// multiply-adds: the results are those of k_sweep, k_defect and the outer kernels bit for bit (the dot
// products' grouping by blocks apart).
//
// What bounds them: the vectors, with the tiles' halos read again.  Measured on 65^3 nodes of 3 x 32
// values, from the row kernels: FP32 sweep 169 -> 83 us (3.8 TB/s of its three vectors; a large copy
// reaches 5.1), defect 158 -> 82 us, FP64 product with its dot 387 -> 142 us.
// Without the loads ahead of the sums the sweep takes 101 us.
#pragma once

#include "batch_kernels.hpp"
#include "lattice_kernels.hpp"

namespace feat3_amd
{
namespace batch
{
  enum LatOp : int { kLatSweep = 0, kLatDefect = 1, kLatProduct = 2, kLatInit = 3 };

  template<typename DT_>
  struct LatArgs
  {
    u32 m, ncol, K;
    u32 lanes, groups;         // threads per node in a block, blocks that share a node's columns
    u32 nx, ny;                // lines of a block
    u32 bx, by, zlen;          // blocks along x and y, planes per block
    const DT_* x;
    const DT_* rhs;
    DT_* out;
    double* partials;          // [block][K]: kLatProduct out . x, kLatInit out . out
    const int* any;
    DT_ k[27];
    DT_ d;
  };

  template<typename DT_, int CH_, u32 TAPS_, int OP_>
  __global__ __launch_bounds__(256, 4) void k_lat_lines(LatArgs<DT_> a)
  {
    if(idle(a.any)) return;
    const u32 id = dev::xcd_remap(blockIdx.x, gridDim.x);
    const u32 grp = id % a.groups, blk = id / a.groups;
    const u32 tx = blk % a.bx, ty = (blk / a.bx) % a.by, tz = blk / (a.bx * a.by);
    const u32 lane = threadIdx.x % a.lanes, line = threadIdx.x / a.lanes;
    const u32 x = tx * a.nx + line % a.nx, y = ty * a.ny + line / a.nx;
    const int m = int(a.m);
    double dot[CH_];
#pragma unroll
    for(int c = 0; c < CH_; ++c) dot[c] = 0.0;
    const u32 col = (grp * a.lanes + lane) * u32(CH_);
    if(line < a.nx * a.ny && x < a.m && y < a.m && col < a.ncol)
    {
      const bool mid = x >= 1 && x + 1 < a.m && y >= 1 && y + 1 < a.m;
      const u64 row = u64(a.m) * a.ncol, plane = row * a.m;
      const u64 at = u64(y) * row + u64(x) * a.ncol + col;
      // offsets of the eight neighbours in a plane (0 at the boundary, whose sums are not used)
      u64 off[9];
#pragma unroll
      for(int t = 0; t < 9; ++t)
        off[t] = mid ? at + u64(std::int64_t(t / 3 - 1) * std::int64_t(row) + std::int64_t(t % 3 - 1) * std::int64_t(a.ncol)) : at;
      const int z0 = int(tz * a.zlen), z1 = z0 + int(a.zlen) < m ? z0 + int(a.zlen) : m;
      DT_ s0[CH_], s1[CH_], s2[CH_], c1[CH_], c2[CH_];   // sums of planes pz + 1, pz, pz - 1; x of pz, pz - 1
      // the nine values of plane pz (the planes beside the lattice only feed sums of boundary nodes)
      auto load = [&](int pz, DT_ (&v)[9][CH_]) {
        const int q = pz < 0 ? 0 : pz < m ? pz : m - 1;
        const DT_* px = a.x + u64(q) * plane;
#pragma unroll
        for(int t = 0; t < 9; ++t) ldv<DT_, CH_>(px + off[t], v[t]);
      };
      auto add = [&](const DT_ (&v)[9][CH_]) {
#pragma unroll
        for(int c = 0; c < CH_; ++c) { s2[c] = s1[c]; s1[c] = s0[c]; s0[c] = DT_(0); c2[c] = c1[c]; c1[c] = v[4][c]; }
#pragma unroll
        for(int t = 0; t < 9; ++t)
        {
#pragma unroll
          for(int c = 0; c < CH_; ++c)
          {
            if((TAPS_ >> t) & 1u) s0[c] = mg::fmadd(a.k[t], v[t][c], s0[c]);
            if((TAPS_ >> (9 + t)) & 1u) s1[c] = mg::fmadd(a.k[9 + t], v[t][c], s1[c]);
            if((TAPS_ >> (18 + t)) & 1u) s2[c] = mg::fmadd(a.k[18 + t], v[t][c], s2[c]);
          }
        }
      };
#pragma unroll
      for(int c = 0; c < CH_; ++c) { s0[c] = s1[c] = DT_(0); c1[c] = DT_(0); }
      DT_ v[9][CH_], w[9][CH_], b[CH_], bn[CH_];
      load(z0 - 1, v);
      load(z0, w);
      add(v);
      load(z0 + 1, v);
      if constexpr(OP_ != kLatProduct) ldv<DT_, CH_>(a.rhs + u64(z0) * plane + at, b);
      add(w);
      auto out = [&](int z, const DT_ (&bz)[CH_]) {
        const u64 i = u64(z) * plane + at;
        const bool in = mid && z >= 1 && z + 1 < m;
        DT_ o[CH_];
#pragma unroll
        for(int c = 0; c < CH_; ++c)
        {
          if constexpr(OP_ == kLatSweep) o[c] = c2[c] + (in ? a.d : DT_(0)) * (bz[c] - s2[c]);
          else if constexpr(OP_ == kLatProduct) { o[c] = in ? s2[c] : DT_(0); dot[c] += double(o[c]) * double(c2[c]); }
          else o[c] = in ? bz[c] - s2[c] : DT_(0);
          if constexpr(OP_ == kLatInit) dot[c] += double(o[c]) * double(o[c]);
        }
        stv<DT_, CH_>(a.out + i, o);
      };
      // two planes a turn: one is loaded while the other is summed
      for(int z = z0; z < z1; z += 2)
      {
        const bool two = z + 1 < z1;
        if(two)
        {
          load(z + 2, w);
          if constexpr(OP_ != kLatProduct) ldv<DT_, CH_>(a.rhs + u64(z + 1) * plane + at, bn);
        }
        add(v);
        out(z, b);
        if(two)
        {
          if(z + 2 < z1)
          {
            load(z + 3, v);
            if constexpr(OP_ != kLatProduct) ldv<DT_, CH_>(a.rhs + u64(z + 2) * plane + at, b);
          }
          add(w);
          out(z + 1, bn);
        }
      }
    }
    if constexpr(OP_ == kLatProduct || OP_ == kLatInit)
    {
      // per system: the block's lines and components in a fixed order
      extern __shared__ double lat_red_[];
      const u32 nl = a.nx * a.ny, w = a.lanes * u32(CH_), c0 = grp * w;
      if(line < nl)
#pragma unroll
        for(int c = 0; c < CH_; ++c) lat_red_[line * w + lane * CH_ + u32(c)] = dot[c];
      __syncthreads();
      for(u32 k = threadIdx.x; k < a.K; k += blockDim.x)
      {
        // the block's columns of system k: c0 + j = k (mod K)
        double s = 0.0;
        for(u32 j = (k + a.K - c0 % a.K) % a.K; j < w; j += a.K)
#pragma unroll 8
          for(u32 l = 0; l < nl; ++l) s += lat_red_[l * w + j];
        a.partials[u64(blockIdx.x) * a.K + k] = s;
      }
    }
  }

  // x_f += filter(P x_c) for the Q1 prolongation of an m^DIM lattice (weights 1, 1/2, ... by the parities
  // of the node's coordinates, the boundary filtered), ncol values per node, CH of them per thread; the
  // terms and their order are k_prolong's, whose chain of row pointer, column and value loads this leaves
  // out.  Bounded by reading and writing x_f.  Measured, k_prolong -> this: 65^3 nodes of 96 FP32 values 79 ->
  // 47 us, 1025^2 nodes of 16 79 -> 28 us (133 MB: 5.3 TB/s).
  template<typename DT_, int CH_, int DIM_>
  __global__ __launch_bounds__(256) void k_lat_prolong(u32 m, u32 ncol, const DT_* __restrict__ xc, DT_* __restrict__ xf,
                                                       const int* any)
  {
    if(idle(any)) return;
    const u32 per = ncol / u32(CH_), i = blockIdx.x * 256u + threadIdx.x;
    const u32 x = i / per, c = (i % per) * u32(CH_), y = blockIdx.y, z = DIM_ == 3 ? blockIdx.z : 1;
    if(x < 1 || x + 1 >= m || y < 1 || y + 1 >= m || z < 1 || (DIM_ == 3 && z + 1 >= m)) return;
    const u64 mc = (m + 1) / 2;
    const u32 ox = x & 1u, oy = y & 1u, oz = DIM_ == 3 ? z & 1u : 0u;
    DT_ v[1 << DIM_][CH_], o[CH_], s[CH_];
    // the neighbours of an even coordinate are one node: loaded again, taken once
#pragma unroll
    for(u32 t = 0; t < (1u << DIM_); ++t)
    {
      const u64 cx = x / 2 + (ox & t), cy = y / 2 + (oy & (t >> 1)), cz = DIM_ == 3 ? z / 2 + (oz & (t >> 2)) : 0;
      ldv<DT_, CH_>(xc + ((cz * mc + cy) * mc + cx) * ncol + c, v[t]);
    }
    DT_* px = xf + ((u64(DIM_ == 3 ? z : 0) * m + y) * m + x) * ncol + c;
    ldv<DT_, CH_>(px, o);
    const DT_ w = (ox ? DT_(0.5) : DT_(1)) * (oy ? DT_(0.5) : DT_(1)) * (oz ? DT_(0.5) : DT_(1));
#pragma unroll
    for(int j = 0; j < CH_; ++j) s[j] = DT_(0);
#pragma unroll
    for(u32 t = 0; t < (1u << DIM_); ++t)
    {
      const bool take = (t & 1u) <= ox && ((t >> 1) & 1u) <= oy && (t >> 2) <= oz;
#pragma unroll
      for(int j = 0; j < CH_; ++j) s[j] = take ? mg::fmadd(w, v[t][j], s[j]) : s[j];
    }
#pragma unroll
    for(int j = 0; j < CH_; ++j) o[j] = o[j] + s[j];
    stv<DT_, CH_>(px, o);
  }
} // namespace batch
} // namespace feat3_amd
