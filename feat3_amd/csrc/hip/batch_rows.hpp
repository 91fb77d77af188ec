// batch_rows.hpp -- several steps of the batched solver's cycle in one pass over a 2D lattice level with
// one matrix per system.
//
// On such a level the matrices are nearly all that a step reads (9 values per node and system against one
// of x, rhs and dinv each), and every smoothing step read them again.  k_field_rows walks along y with NS
// steps in a pipeline, each one row behind the one before: a row's nine values, its right-hand side and
// its dinv are loaded once, one row ahead of their first use, and stay in registers until the last step
// has used them.  A thread is one node column and system (systems fastest, so a node's values of one
// entry are contiguous); its x neighbours' values come through LDS, a double row per step, and its own
// 3 x 3 window is kept in registers.  A block of 1024 threads is lanes systems times nx nodes; each step
// is right on one node less at both ends, so nx - 2 NS columns and ylen rows of it are stored, and its
// first 2 NS rows warm the pipeline.  The terms of every sum and their order are those of k_sweep and
// k_defect: the results are theirs bit for bit.
//
// What bounds it: the values, 604 MB of FP32 at 1025^2 nodes and 16 systems, with a quarter of them read
// twice (56 of 64 columns are stored, 79 of 87 rows).  Measured there: four sweeps 4 x 189 -> 188 us, three
// sweeps and the defect 743 -> 216 us; 513^2 nodes 146 -> 48 and 52 us, 257^2 50 -> 20 and 23 us, 129^2
// 20 -> 17 and 19 us.
#pragma once

#include "batch_kernels.hpp"

namespace feat3_amd
{
namespace batch
{
  template<typename DT_, typename VT_>
  struct FieldArgs
  {
    u32 m, K;
    u32 lanes, groups;     // systems of a block, blocks that share a node's systems
    u32 nx, bx, ylen;      // node columns of a block, blocks along x, rows stored by a block
    const VT_* val;        // [entry][k] of the full 9-point graph (rows ascending)
    const DT_* dinv;
    const DT_* rhs;
    const DT_* x;
    DT_* out;              // x after the last sweep
    DT_* def;              // DEF_: the last step is the defect of out
    const int* any;
  };

  // entries before the inner node (x, y) in the 9-point graph of an m x m lattice
  __host__ __device__ __forceinline__ u64 field_entry(u64 m, u64 x, u64 y)
  {
    return 6 * m - 4 + (y - 1) * (9 * m - 6) + 6 + 9 * (x - 1);
  }

  constexpr u32 kFieldThreads = 1024;

  template<typename DT_, typename VT_, int NS_, bool DEF_>
  __global__ __launch_bounds__(1024) void k_field_rows(FieldArgs<DT_, VT_> a)
  {
    constexpr int R = NS_ + 1;   // rows in registers: one per step and the one being loaded
    __shared__ DT_ line[NS_][2][kFieldThreads];
    if(idle(a.any)) return;
    const u32 id = dev::xcd_remap(blockIdx.x, gridDim.x);
    const u32 grp = id % a.groups, blk = id / a.groups;
    const u32 tx = blk % a.bx, ty = blk / a.bx;
    const u32 lane = threadIdx.x % a.lanes, node = threadIdx.x / a.lanes;
    const u32 k = grp * a.lanes + lane;
    const int m = int(a.m), x = int(tx * (a.nx - 2 * NS_) + node) - NS_;
    const int y0 = int(ty * a.ylen), y1 = y0 + int(a.ylen) < m ? y0 + int(a.ylen) : m;
    const bool on = node < a.nx && k < a.K && x >= 0 && x < m;
    const bool mid = on && x >= 1 && x + 1 < m;
    const bool store = on && node >= u32(NS_) && node + u32(NS_) < a.nx;
    const u32 left = threadIdx.x >= a.lanes ? threadIdx.x - a.lanes : threadIdx.x;
    const u32 right = threadIdx.x + a.lanes < kFieldThreads ? threadIdx.x + a.lanes : threadIdx.x;
    const u64 K = a.K, rowv = u64(m) * K, at = on ? u64(x) * K + k : 0;

    VT_ c[R][9];
    DT_ b[R], d[R], win[NS_][2][3];
#pragma unroll
    for(int r = 0; r < R; ++r)
    {
#pragma unroll
      for(int e = 0; e < 9; ++e) c[r][e] = VT_(0.0f);
      b[r] = d[r] = DT_(0);
    }
#pragma unroll
    for(int s = 0; s < NS_; ++s)
#pragma unroll
      for(int e = 0; e < 3; ++e) win[s][0][e] = win[s][1][e] = DT_(0);

    const int t0 = y0 - NS_ > 0 ? y0 - NS_ : 0, t1 = y1 + NS_;
    // row t of x; on the boundary plus dinv, which is 0 there or, in a row that is not finite, NaN
    auto load_x = [&](int t) {
      DT_ v = a.x[u64(t) * rowv + at];
      if(!mid || t == 0 || t + 1 == m) v += a.dinv[u64(t) * rowv + at];
      return v;
    };
    DT_ next = on ? load_x(t0) : DT_(0);
    // turn t: row t of x arrives; step s completes row t - 1 - s from its input's rows t - 2 - s .. t - s
    auto turn = [&](int t, auto phase) {
      constexpr int P = decltype(phase)::value;
      DT_ cur = next;
      if(on && t + 1 < m) next = load_x(t + 1);
      if(mid && t >= 1 && t + 1 < m)
      {
        const VT_* v = a.val + field_entry(u64(m), u64(x), u64(t)) * K + k;
#pragma unroll
        for(int e = 0; e < 9; ++e) c[P][e] = v[u64(e) * K];
        b[P] = a.rhs[u64(t) * rowv + at];
        d[P] = a.dinv[u64(t) * rowv + at];
      }
#pragma unroll
      for(int s = 0; s < NS_; ++s)
      {
        const int r = t - 1 - s;
        const int q = (P + 2 * R - 1 - s) % R;
        line[s][t & 1][threadIdx.x] = cur;
        __syncthreads();
        const DT_ l = line[s][t & 1][left], g = line[s][t & 1][right];
        DT_ sum = DT_(0);
#pragma unroll
        for(int e = 0; e < 3; ++e) sum = mg::fmadd(cvt<DT_, VT_>(c[q][e]), win[s][0][e], sum);
#pragma unroll
        for(int e = 0; e < 3; ++e) sum = mg::fmadd(cvt<DT_, VT_>(c[q][3 + e]), win[s][1][e], sum);
        sum = mg::fmadd(cvt<DT_, VT_>(c[q][6]), l, sum);
        sum = mg::fmadd(cvt<DT_, VT_>(c[q][7]), cur, sum);
        sum = mg::fmadd(cvt<DT_, VT_>(c[q][8]), g, sum);
        const bool in = mid && r >= 1 && r + 1 < m;
        const DT_ own = win[s][1][1];
        DT_ o;
        if(DEF_ && s == NS_ - 1) o = in ? b[q] - sum : DT_(0);
        else o = in ? own + d[q] * (b[q] - sum) : own;
        if(s >= NS_ - (DEF_ ? 2 : 1) && store && r >= y0 && r < y1)
          (DEF_ && s == NS_ - 1 ? a.def : a.out)[u64(r) * rowv + at] = o;
#pragma unroll
        for(int e = 0; e < 3; ++e) win[s][0][e] = win[s][1][e];
        win[s][1][0] = l; win[s][1][1] = cur; win[s][1][2] = g;
        cur = o;
      }
    };
    for(int t = t0; t < t1; t += R)
    {
      // rows past the end change nothing that is stored; the turns are the same for all threads
      turn(t, std::integral_constant<int, 0>());
      if constexpr(R > 1) { if(t + 1 < t1) turn(t + 1, std::integral_constant<int, 1 % R>()); }
      if constexpr(R > 2) { if(t + 2 < t1) turn(t + 2, std::integral_constant<int, 2 % R>()); }
      if constexpr(R > 3) { if(t + 3 < t1) turn(t + 3, std::integral_constant<int, 3 % R>()); }
      if constexpr(R > 4) { if(t + 4 < t1) turn(t + 4, std::integral_constant<int, 4 % R>()); }
    }
  }
} // namespace batch
} // namespace feat3_amd
