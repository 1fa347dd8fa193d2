// D-ILU triangular solves by columns, one launch per sweep (p3d_column.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "p3d_internal.hpp"
#include "p3d_kernels.hpp"

namespace p3d {

// LDS of one column at most.  Phi factors that are not all equal, or a phi cut,
// take a table of 8 bytes per plane beside the 34 KB of rows: beyond about 3780
// planes the tile schedules run.  Equal factors without a cut and stored
// couplings need no table.
constexpr size_t kColLdsMax = 64 * 1024;

struct ColArgs {
  int NI = 0, NJ = 0, c = 0;  // columns of 8x8 points, planes
  int tk_log2 = 0, planes = 0;  // tile-major placement of r and z (TileMap)
  int rounds = 0;               // rounds of 32 steps
  int rows_alloc = 0;           // rows of a column in dinv_s and y_s
  int face_rows = 0;            // rows of a column's faces
  int pf_n = 0;                 // entries of the phi-factor tables
  int skip = 0;                 // steps before the backward sweep's first plane
  int mode = 0;                 // phi factors: by plane, equal but for the cut, equal
  float u_d = 0.f, u_k = 0.f;   // the equal FDPH, FDPL = FDPU
  IluBlocks bl{};
  const int* order = nullptr;      // columns by anti-diagonal inside their block
  const float* dinv_s = nullptr;   // [column][row][lane]: plane row - 32 - ii - 2 jj
  float* y_s = nullptr;            // the forward result, placed as dinv_s
  unsigned long long* face_i = nullptr;  // [column][row][8]: {value, stamp} of the step row - 8
  unsigned long long* face_j = nullptr;
  const float2* pf_lo = nullptr;  // (FDPH, FDPL) by plane + 21, zero outside
  const float2* pf_up = nullptr;  // (FDPH, FDPU) from plane c + skip - 1 downwards, likewise
  // stored couplings: {k, j, i, dinv} by step and lane of the forward and the
  // backward march, and those of the phi wrap (a x b)
  const float4 *lo_s = nullptr, *up_s = nullptr;
  const float *wrap_lo = nullptr, *wrap_up = nullptr;
  unsigned* ctr = nullptr;        // stamps of the next forward, backward sweep
  unsigned* failed = nullptr;     // set once a wait ran into its bound
  unsigned polls = 0;             // that bound
  void* dummy = nullptr;          // where rows outside the vectors are stored
};

struct ColumnPlan {
  int ready = 0;
  int dev = 0, ncu = 0;  // device and its CUs
  ColArgs a;
  int* order = nullptr;
  float *dinv_s = nullptr, *y_s = nullptr;
  unsigned long long* face = nullptr;
  float2* pf = nullptr;
  unsigned* ctr = nullptr;
  void* dummy = nullptr;
  float4* cs = nullptr;  // stored couplings, forward then backward
};

// dinv: the D-ILU's inverse pivots in natural order; tk_log2: planes per
// tile of the r and z placement; failed: device word that is set once a wait
// runs into its bound.  Returns 0 when the sweeps can run.
int build_column_plan(ColumnPlan& plan, const Metric& m, const Grid3& g, const IluBlocks& bl,
                      int tk_log2, const float* dinv, unsigned* failed);
// The same with stored couplings; co's wrap planes have to outlive the plan,
// whose word column_failure_flag is.
int build_column_plan_stored(ColumnPlan& plan, const Grid3& g, const CoefArrays& co, bool wrap,
                             const float* dinv);
void free_column_plan(ColumnPlan& plan);

// Room on the device for the column sweeps of one call, from before its first
// launch until its last one has ended.  Without it (claim false) the call takes
// the tile schedules.
struct ColumnUse {
  int dev = 0, ncol = 0;
  bool claim(const ColumnPlan& plan);
  void release();
  ColumnUse() = default;
  ColumnUse(const ColumnUse&) = delete;
  ColumnUse& operator=(const ColumnUse&) = delete;
  ~ColumnUse() { release(); }
};

// What it counts with: columns of launches under way on a device of ncu CUs.
extern "C" int p3d_columns_claim(int dev, int ncol, int ncu);
extern "C" void p3d_columns_release(int dev, int ncol);

// z = (LU)^-1 r on tile-major r and z, two launches.  ap (tile-major, with
// guard): r -= alpha ap first, alpha from guard.
template <typename T>
void launch_dilu_columns(const ColumnPlan& plan, const Metric& m, const Grid3& g, T* r, T* z,
                         const CgState* guard, const T* ap, hipStream_t s);

// x = (LU)^-1 x on natural order, stored couplings, two launches.  r32 (N
// floats) receives x as it was, rounded to FP32 as the sweep uses it.
void launch_dilu_columns_stored(const ColumnPlan& plan, const Grid3& g, double* x, float* r32,
                                hipStream_t s);

// The plan's own device word, not 0 once a wait of its sweeps ran into its bound
// (build_column_plan_stored).
const unsigned* column_failure_flag(const ColumnPlan& plan);

}  // namespace p3d
