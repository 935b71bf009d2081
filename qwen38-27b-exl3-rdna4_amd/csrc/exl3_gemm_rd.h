// exl3_gemm_rd.h -- host side of the register-decode GEMM (exl3_gemm_rd.hip).
#pragma once
#include "exl3_device.h"

constexpr int RD_MAX_ROWS = 128, RD_MAX_TILES = 4096;

// A launch of M rows through groups of `widths` columns: tiles of all rows (R row tiles of 32) x 128
// columns, each tile's K in units of 256, shared by `grid` workgroups, each group its own range of
// them.  A function of the shape only.
struct RdPlan {
    bool use;                                  // false: the shape is not served
    int R, grid;
    int G[EXL3_MAX_GROUPS], w0[EXL3_MAX_GROUPS], tile0[EXL3_MAX_GROUPS];
    size_t part_bytes;                         // fp32 partial tiles (and one zeroed counter per tile)
};

RdPlan rd_plan(int M, int K, const int* widths, int groups);

int launch_gemm_rd(const RdPlan& pl, int bits, int cb, const uint16_t* const* xf, const void* const* trellis, uint16_t* const* y,
                   int64_t ldy, const uint16_t* const* svh, const int* widths, int groups, int M, int K, void* part,
                   uint32_t* counters, hipStream_t s);
