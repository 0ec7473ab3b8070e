// Multilevel field update in fast arithmetic (field_fast.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.hpp"

namespace ion {

constexpr int ML_MAX_P = 20;                         // sample points per axis
constexpr size_t ML_WS_FLOATS = (size_t)16 << 20;    // most of the workspace of a field update (64 MB)

// Sample points of the blocks of one level along the three axes, relative to
// the block's first cell.
struct MlGrid {
    int P[3];
    int n;           // P[0] P[1] P[2]
    uint32_t shift;  // block side = LOD block side << shift
    uint32_t side;   // blocks per axis
    uint32_t groups; // workgroups of k_ml_coarse
    float x[3][ML_MAX_P];
};

// Everything the kernels need beside the FieldArgs; a pure function of the
// lattice and the LOD depth (ml_plan). Offsets are in floats from ws.
struct MlArgs {
    FieldArgs f;
    const float4* qu;        // LOD sums, [n_lod]
    float* ws;
    uint32_t nd, lo, n_lod, zext;
    uint32_t b[3];           // cells per LOD block side
    uint32_t levels;         // coarse levels: 2 .. D - 1
    MlGrid fine, coarse[2];  // the LOD blocks; levels 2 and 3 of the block tree
    uint32_t cells[3];       // rows of the cell tables (z: up to whole groups of R cells)
    uint32_t ld;             // weights of a row of the tables
    uint32_t t_cell[3];      // fine sample points -> cells: [cells][ld] (x, y), [P][cells] (z)
    uint32_t t_up[2][3];     // coarse sample points -> fine ones: [1 << shift][P][ld]
    uint32_t t0, t_end;      // begin and end of the tables
    uint32_t samples[2];     // [block][6][n] field samples of the coarse levels
    uint32_t ws_floats;
    uint32_t leaf;           // the cells are the sample points
    // cells of one LOD block: tiles of colw wavefronts of 64 columns, R cells a thread along z
    uint32_t R, nzt, colw, ntile, threads;
    uint32_t rows;           // rows of cells that a tile's columns touch at most
    uint32_t gc;             // components interpolated at a time
    uint32_t nt;             // far sources: tiles of 16 sample points per wavefront and pass
    uint32_t v_off, w_off, list_off, lds;  // LDS layout (floats), total bytes
};

// Header of the workspace: the modes, then from ML_DENSE floats on the LOD
// sources at every LOD index, whole z layers (depth 3 and 4).
constexpr uint32_t ML_DENSE = 16;

// Plan of the lattice of f; false if the multilevel update does not take it.
bool ml_plan(const FieldArgs& f, MlArgs* a);
// Floats of the workspace (0: none).
size_t ml_workspace(const FieldArgs& f);
// Tables and coarse levels, then the cells (nothing unless *f.mode).
hipError_t launch_field_fast(const MlArgs& a, hipStream_t s);

}  // namespace ion
