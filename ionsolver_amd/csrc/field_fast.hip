// The dynamic E/B field update (update_e_b_dynamic, sim_kernels.cl:897-993) in
// fast arithmetic: E += q r/|r|^3, B += q v x r/|r|^3 over the LOD sources.
//
// The field of distant sources varies slowly over a block of cells, so it is
// summed at a few sample points of the block only and interpolated. The LOD
// blocks (8^D) are the leaves of a tree whose level l has 8^l blocks; a source
// is near a block if it lies in the 3^3 blocks of that level around it. Each
// source is taken once per cell, on the coarsest level where it is not near:
//   levels 2 .. D-1  k_ml_coarse: sources near the parent block but not near
//                    the block, at the block's sample points (on level 2 all
//                    that are not near);
//   level D          k_ml_cells / k_ml_leaf: the same, plus the interpolated
//                    samples of the coarser blocks above; then at the cells the
//                    26 LOD blocks around the own one (which is left out, as
//                    in the reference), plus the interpolated samples.
// Sample points are Chebyshev points, as many per axis as bring the
// interpolation error below the rounding of the float sums (grid_of); the
// weights are computed in double. A block of up to 9 or so cells a side has as
// many points as cells: its cells are the sample points (k_ml_leaf).
//
// Why: a direct sum costs 13 VALU instructions and one v_rsq_f32 for each cell
// and source, 16.1 ms at 256^3 with 3511 sources (VALU issue); this split
// leaves about 24 sources a cell and 145 a sample point: 1.15 ms (coarse levels
// 0.29, the rest 0.81 ms, of which the near sources 0.12, the far ones 0.2, the
// interpolation between the levels 0.2 and to the cells 0.13, the fields' own
// traffic 0.22). Its error against the sum in double is smaller, 1e-7 against
// 3.4e-7 (fewer float additions in a row). 240 x 336 x 144, blocks of
// 15 x 21 x 9 cells: 17.5 -> 2.85 ms; 128^3 2.56 -> 0.60 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "field_fast.hpp"
#include "judge.hpp"

namespace ion {

namespace {

constexpr int COARSE_T = 512;                     // threads of a coarse workgroup
constexpr int COARSE_NT = 4;                      // tiles of 16 sample points per wavefront
constexpr int COARSE_SG = 2;                      // groups of wavefronts that share the sources
constexpr int COARSE_PTS = COARSE_T / 64 / COARSE_SG * COARSE_NT * 16;  // sample points per workgroup
constexpr int LIST_FAR = 216, LIST_NEAR = 28;     // sources of a leaf: 6^3 candidates, 3^3 around the block
constexpr int LIST_CNT = 10;  // lengths, counts of the 4 wavefronts of candidates
constexpr uint32_t LEAF_T = 512;
constexpr uint32_t ML_LDS = 80 * 1024;  // two workgroups of k_ml_cells on a CU

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) float* cfloat_p;  // tables: read through the scalar cache

struct Src {
    float4 p;  // centre, charge
    float4 v;  // mean velocity
};

// Sources of the sample points in LDS, relative to the centre of their block:
// place and |s|^2, [4][CAP], and the columns that all of their fields are linear
// in, [CAP][12]: q, q s (3), J = q v (3), J x s (3).
template <int CAP> struct FarList {
    float s[4][CAP];
    float col[CAP][12];
    __device__ __forceinline__ void put(int i, const Src& a, const float org[3]) {
        const float x = a.p.x - org[0], y = a.p.y - org[1], z = a.p.z - org[2], q = a.p.w;
        const float jx = q * a.v.x, jy = q * a.v.y, jz = q * a.v.z;
        s[0][i] = x;
        s[1][i] = y;
        s[2][i] = z;
        s[3][i] = __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z));
        float4* const c = (float4*)col[i];
        c[0] = make_float4(q, q * x, q * y, q * z);
        c[1] = make_float4(jx, jy, jz, jy * z - jz * y);
        c[2] = make_float4(jz * x - jx * z, jx * y - jy * x, 0.0f, 0.0f);
    }
    // fills up a list of m sources to whole steps of far_sums (i: 0 .. 15)
    __device__ __forceinline__ void pad(int m, int i) {
        if (m + i >= ((m + 15) & ~15)) return;
        s[0][m + i] = 4.0e6f;
        s[1][m + i] = s[2][m + i] = 0.0f;
        s[3][m + i] = 1.6e13f;
        float4* const c = (float4*)col[m + i];
        c[0] = c[1] = c[2] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
};

typedef FarList<(LIST_FAR + 15) / 16 * 16> LeafList;

// A tile of 16 sample points, one of them a lane & 15, relative to the block's
// centre: operand of |r|^2 = |x|^2 + (-2 x, 1) . (s, |s|^2)
struct Points {
    float v;   // component lane >> 4 of (-2 x, 1)
    float xx;  // |x|^2
    __device__ __forceinline__ void set(float x, float y, float z) {
        const int k = ((int)threadIdx.x & 63) >> 4;
        v = k == 0 ? -2.0f * x : k == 1 ? -2.0f * y : k == 2 ? -2.0f * z : 1.0f;
        xx = __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z));
    }
};

// Field sums of NT tiles of sample points over a list of m sources, 16 at a
// time. |r|^2 of 16 points and 16 sources is a matrix product; its lanes hold
// point lane & 15 and sources 4 r + (lane >> 4), which is, r by r, the left
// operand of the product of 1/|r|^3 with the columns of four sources in a row,
// and
//   E = x (sum q / r^3) - sum q s / r^3,  B = (sum J / r^3) x x - sum J x s / r^3.
// What stays on the VALU per pair of a wavefront are 2 instructions and a
// v_rsq_f32 (12 cycles) beside 40 cycles of the matrix unit, where the sum of the
// vectors takes 21 and one (50 cycles). k_ml_coarse has the matrix units busy 45 %
// of its time and the VALU 15 %.
// A product adds its four terms one after the other, so a sum is taken in the
// order of the list: a source too weak to change it leaves it as it is,
// wherever in the list it stands.
// Of a point x and a source s that is not near, (|x|^2 + |s|^2) / |r|^2 is at
// most 3.2 on cubic blocks and 7 on the most uneven ones that get a plan (16 x 16
// x 5 cells), |s| / |r| at most 1.7 and 2.3: |r|^2 loses up to 1.7 and 2.8 bits to
// cancellation, the differences of the fields about one.
template <int NT, int CAP>
__device__ __forceinline__ void far_sums(const FarList<CAP>& list, int m, const Points* p, f32x4* c) {
    const int lane = (int)threadIdx.x & 63, n = min(lane & 15, 11), k = lane >> 4;
    const int row = 4 * (lane & 3) + ((lane & 15) >> 2);  // row 4 k + r: source 4 r + k
    for (int i = 0; i < m; i += 16) {
        const float sv = list.s[k][i + row];
        float col[4];
#pragma unroll
        for (int r = 0; r < 4; r++) col[r] = list.col[i + 4 * r + k][n];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const f32x4 r2 = __builtin_amdgcn_mfma_f32_16x16x4f32(sv, p[t].v, (f32x4){p[t].xx, p[t].xx, p[t].xx, p[t].xx}, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float inv = __builtin_amdgcn_rsqf(r2[r]);
                c[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(inv * inv * inv, col[r], c[t], 0, 0, 0);
            }
        }
    }
}
// The product of a tile as [16 points][17] in LDS (a lane holds points
// 4 (lane >> 4) + r of column lane & 15)
__device__ __forceinline__ void put_tile(float* t, const f32x4 c) {
    const int lane = (int)threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < 4; r++) t[(4 * (lane >> 4) + r) * 17 + (lane & 15)] = c[r];
}
// Component o of the fields of a point at (x, y, z) from its row of the product
__device__ __forceinline__ float field_of(const float* t, int o, float x, float y, float z) {
    switch (o) {
        case 0: return __builtin_fmaf(x, t[0], -t[1]);
        case 1: return __builtin_fmaf(y, t[0], -t[2]);
        case 2: return __builtin_fmaf(z, t[0], -t[3]);
        case 3: return __builtin_fmaf(t[5], z, -__builtin_fmaf(t[6], y, t[7]));
        case 4: return __builtin_fmaf(t[6], x, -__builtin_fmaf(t[4], z, t[8]));
        default: return __builtin_fmaf(t[4], y, -__builtin_fmaf(t[5], x, t[9]));
    }
}

// Whether this update runs (few or non-finite sources: the direct kernels)
__device__ __forceinline__ bool multilevel(const MlArgs& a) { return a.f.mode[MODE_FAST] != 0u; }

// The source at (X, Y, Z) of the LOD grid (Z up to zext: the last indices of
// the range lie above the domain), and whether the field update reads it:
// indices from lo to n_lod, charges that are not zero.
__device__ __forceinline__ bool source_at(const MlArgs& a, int X, int Y, int Z, Src* s) {
    const uint32_t d = (uint32_t)X + ((uint32_t)Y + (uint32_t)Z * a.nd) * a.nd;
    if (d < a.lo || d >= a.n_lod) return false;
    const float4 e = a.qu[d];
    if (e.x == 0.0f) return false;
    const float dx = (float)a.b[0], dy = (float)a.b[1], dz = (float)a.b[2];
    s->p = make_float4((float)X * dx + 0.5f * dx, (float)Y * dy + 0.5f * dy, (float)Z * dz + 0.5f * dz, e.x);
    s->v = make_float4(e.y, e.z, e.w, 0.0f);
    return true;
}

// The sample points of a grid into LDS: the kernel arguments lie in host
// memory, and a load per lane from there costs microseconds.
__device__ __forceinline__ void stage_points(const MlGrid& g, float (*x)[ML_MAX_P]) {
    for (int i = (int)threadIdx.x; i < 3 * ML_MAX_P; i += (int)blockDim.x) x[i / ML_MAX_P][i % ML_MAX_P] = (&g.x[0][0])[i];
}

__device__ __forceinline__ bool within1(int a, int b) { return (uint32_t)(a - b + 1) <= 2u; }

// Weight of point i of x[0 .. P) at u (Lagrange)
__device__ float lagrange(const float* x, int P, int i, double u) {
    double num = 1.0, den = 1.0;
    for (int j = 0; j < P; j++) {
        if (j == i) continue;
        num *= u - (double)x[j];
        den *= (double)x[i] - (double)x[j];
    }
    return (float)(num / den);
}

// Interpolation tables: rows of a.ld weights (padded with zeros) for one point
// each; the cells' along z transposed, so that the weights of consecutive
// cells lie together.
__device__ void ml_tables(const MlArgs& a, uint32_t t, const float (*x)[3][ML_MAX_P]) {
    if (t >= a.t_end) return;
    const uint32_t ld = a.ld;
    for (int k = 0; k < 3; k++) {
        const int P = a.fine.P[k];
        const uint32_t cells = a.cells[k];
        uint32_t i = t - a.t_cell[k];
        if (t >= a.t_cell[k] && i < cells * (k < 2 ? ld : (uint32_t)P)) {
            if (k < 2) a.ws[t] = (int)(i % ld) < P ? lagrange(x[0][k], P, i % ld, (double)(i / ld)) : 0.0f;
            else a.ws[t] = lagrange(x[0][k], P, i / cells, (double)(i % cells));
        }
        for (uint32_t l = 0; l < a.levels; l++) {
            const MlGrid& c = a.coarse[l];
            i = t - a.t_up[l][k];
            if (t < a.t_up[l][k] || i >= (uint32_t)((1 << c.shift) * P) * ld) continue;
            const uint32_t off = i / (P * ld), p = i / ld % P;
            a.ws[t] = (int)(i % ld) < c.P[k]
                          ? lagrange(x[1 + l][k], c.P[k], i % ld, (double)(off * a.b[k]) + (double)x[0][k][p])
                          : 0.0f;
        }
    }
}

// Samples of the coarse levels: a workgroup takes COARSE_PTS points of a block
// (level 2 first: its blocks have the longest source lists); the last
// workgroups compute the tables. The sources are gathered into LDS COARSE_T
// candidates at a time, in index order; two groups of wavefronts take those of
// even and odd number (of the candidate, not of the source: which charges are
// there does not move a source to the other group) and are summed at the end.
__global__ void __launch_bounds__(COARSE_T) __attribute__((amdgpu_waves_per_eu(4))) k_ml_coarse(MlArgs a) {
    constexpr int WPG = COARSE_T / 64 / COARSE_SG;  // wavefronts of a group
    __shared__ __align__(16) union {
        FarList<COARSE_T / COARSE_SG> list[COARSE_SG];
        float tile[COARSE_T / 64][COARSE_NT][16 * 17];
    } sh;
    __shared__ uint32_t wtot[COARSE_SG][COARSE_T / 64];
    __shared__ float xs[3][3][ML_MAX_P];
    if (!multilevel(a)) return;
    uint32_t blk = blockIdx.x;
    uint32_t li = 0;
    while (li < a.levels && blk >= a.coarse[li].groups) blk -= a.coarse[li++].groups;
    const int tid = (int)threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (li == a.levels) {
        stage_points(a.fine, xs[0]);
        for (uint32_t l = 0; l < a.levels; l++) stage_points(a.coarse[l], xs[1 + l]);
        __syncthreads();
        ml_tables(a, a.t0 + blk * COARSE_T + tid, xs);
        return;
    }
    const MlGrid& g = a.coarse[li];
    stage_points(g, xs[0]);
    __syncthreads();
    const int parts = (g.n + COARSE_PTS - 1) / COARSE_PTS;
    const int p0 = ((int)blk % parts * WPG + wv % WPG) * COARSE_NT * 16;  // first point of the wavefront
    blk /= parts;
    const int side = (int)g.side, shift = (int)g.shift;
    const int C[3] = {(int)blk % side, (int)blk / side % side, (int)blk / (side * side)};
    // candidates: the sources near the parent block (on level 2, all)
    int lo3[3], n3[3];
    float half[3], org[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int end = (int)(k == 2 ? a.zext : a.nd);
        lo3[k] = li == 0 ? 0 : max(0, ((C[k] >> 1) - 1) * (2 << shift));
        n3[k] = (li == 0 ? end : min(end, ((C[k] >> 1) + 2) * (2 << shift))) - lo3[k];
        half[k] = 0.5f * (float)(a.b[k] << shift);
        org[k] = (float)(C[k] * (int)(a.b[k] << shift)) + half[k];
    }
    const int total = n3[0] * n3[1] * n3[2], grp = wv / WPG;
    auto at = [&](int i, float* x) {
        x[0] = xs[0][0][i % g.P[0]] - half[0];
        x[1] = xs[0][1][i / g.P[0] % g.P[1]] - half[1];
        x[2] = xs[0][2][i / (g.P[0] * g.P[1])] - half[2];
    };
    Points pt[COARSE_NT];
    f32x4 acc[COARSE_NT];
#pragma unroll
    for (int t = 0; t < COARSE_NT; t++) {
        float x[3];
        at(min(p0 + t * 16 + (lane & 15), g.n - 1), x);
        pt[t].set(x[0], x[1], x[2]);
        acc[t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (int base = 0; base < total; base += COARSE_T) {
        const int j = base + tid;
        Src s;
        bool keep = false;
        if (j < total) {
            const int X = lo3[0] + j % n3[0], Y = lo3[1] + j / n3[0] % n3[1], Z = lo3[2] + j / (n3[0] * n3[1]);
            keep = !(within1(X >> shift, C[0]) && within1(Y >> shift, C[1]) && within1(Z >> shift, C[2])) &&
                   source_at(a, X, Y, Z, &s);
        }
        static_assert(COARSE_SG == 2, "lists of even and odd candidates");
        const uint64_t mask = __ballot(keep), even = 0x5555555555555555ull;
        __syncthreads();
        if (lane < COARSE_SG) wtot[lane][wv] = (uint32_t)__popcll(mask & even << lane);
        __syncthreads();
        const int mine = lane & 1;
        int off = __popcll(mask & even << mine & ((1ull << lane) - 1ull)), m[COARSE_SG] = {0, 0};
        for (int w = 0; w < COARSE_T / 64; w++) {
            if (w < wv) off += (int)wtot[mine][w];
#pragma unroll
            for (int h = 0; h < COARSE_SG; h++) m[h] += (int)wtot[h][w];
        }
        if (keep) sh.list[mine].put(off, s, org);
        if (tid < 16 * COARSE_SG) sh.list[tid >> 4].pad(tid < 16 ? m[0] : m[1], tid & 15);
        __syncthreads();
        if (p0 < g.n) far_sums<COARSE_NT>(sh.list[grp], __builtin_amdgcn_readfirstlane(grp == 0 ? m[0] : m[1]), pt, acc);
    }
    // sum of the groups, in order
    float* const out = a.ws + a.samples[li] + (size_t)blk * 6 * g.n;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < COARSE_NT; t++) put_tile(sh.tile[wv][t], acc[t]);
    __syncthreads();
    // a lane: point lane & 15 of a tile, components lane >> 4 and, below 2, that + 4
#pragma unroll
    for (int t = 0; t < COARSE_NT; t++) {
        const int p = p0 + t * 16 + (lane & 15);
        if (t % COARSE_SG != grp || p >= g.n) continue;
        float x[3];
        at(p, x);
        for (int o = lane >> 4; o < 6; o += 4) {
            float v = 0.0f;
#pragma unroll
            for (int h = 0; h < COARSE_SG; h++)
                v += field_of(&sh.tile[h * WPG + wv % WPG][t][(lane & 15) * 17], o, x[0], x[1], x[2]);
            out[o * g.n + p] = v;
        }
    }
}

// Interpolation along one axis: each line of c values gives nout values
// M[o] . in, where row o of M has CM weights (zero from c on) that are the same
// for every thread: they come as scalar operands. in(line, &stride): the first
// of a line's values and their distance.
template <int CM, class In, class Out>
__device__ __forceinline__ void lines(int nlines, int c, int nout, cfloat_p M, In in, Out out) {
    for (int line = (int)threadIdx.x; line < nlines; line += (int)blockDim.x) {
        int stride;
        const float* const p = in(line, &stride);
        float v[CM];
#pragma unroll
        for (int k = 0; k < CM; k++) v[k] = k < c ? p[k * stride] : 0.0f;
        float w[CM], s[2];
#pragma unroll
        for (int k = 0; k < CM; k++) w[k] = M[k];
        for (int o = 0; o < nout; o++) {
            // short rows: the next one's loads run beside this one's sum (long
            // ones would not fit the scalar registers twice)
            const cfloat_p next = M + min(o + 1, nout - 1) * CM;
            float wn[CM];
            if (CM <= 12)
#pragma unroll
                for (int k = 0; k < CM; k++) wn[k] = next[k];
            s[0] = w[0] * v[0];
            s[1] = w[1] * v[1];
#pragma unroll
            for (int k = 2; k < CM; k++) s[k & 1] = __builtin_fmaf(w[k], v[k], s[k & 1]);
            out(line, o, s[0] + s[1]);
#pragma unroll
            for (int k = 0; k < CM; k++) w[k] = CM <= 12 ? wn[k] : next[k];
        }
    }
}

// S[6][n] = the coarse levels' samples above LOD block (X, Y, Z), interpolated
// to its sample points, one axis after the other through tmp (a.gc components
// at a time).
template <int CM>
__device__ __forceinline__ void from_coarse(const MlArgs& a, uint32_t X, uint32_t Y, uint32_t Z, float* S, float* tmp) {
    const int Px = a.fine.P[0], Py = a.fine.P[1], Pz = a.fine.P[2], n = a.fine.n, G = (int)a.gc;
    for (uint32_t l = 0; l < a.levels; l++) {
        const MlGrid& g = a.coarse[l];
        const uint32_t sh = g.shift, m = (1u << sh) - 1u;
        const int cx = g.P[0], cy = g.P[1], cz = g.P[2];
        const float* const in =
            a.ws + a.samples[l] + (size_t)((X >> sh) + ((Y >> sh) + (Z >> sh) * g.side) * g.side) * 6 * g.n;
        const cfloat_p Mx = (cfloat_p)(a.ws + a.t_up[l][0] + (X & m) * Px * CM);
        const cfloat_p My = (cfloat_p)(a.ws + a.t_up[l][1] + (Y & m) * Py * CM);
        const cfloat_p Mz = (cfloat_p)(a.ws + a.t_up[l][2] + (Z & m) * Pz * CM);
        float* const t1 = tmp;
        float* const t2 = tmp + G * cz * cy * Px;
        for (int c0 = 0; c0 < 6; c0 += G) {
            lines<CM>(
                G * cz * cy, cx, Px, Mx,
                [&](int i, int* st) {
                    *st = 1;
                    return in + (size_t)c0 * g.n + i * cx;
                },
                [&](int i, int o, float v) { t1[i * Px + o] = v; });
            __syncthreads();
            lines<CM>(
                G * cz * Px, cy, Py, My,
                [&](int i, int* st) {
                    *st = Px;
                    return t1 + i / Px * cy * Px + i % Px;
                },
                [&](int i, int o, float v) { t2[(i / Px * Py + o) * Px + i % Px] = v; });
            __syncthreads();
            lines<CM>(
                G * Px * Py, cz, Pz, Mz,
                [&](int i, int* st) {
                    *st = Px * Py;
                    return t2 + i / (Px * Py) * cz * Px * Py + i % (Px * Py);
                },
                [&](int i, int o, float v) {
                    float* const d = S + (c0 + i / (Px * Py)) * n + o * Px * Py + i % (Px * Py);
                    *d = l == 0 ? v : *d + v;
                });
        }
    }
    __syncthreads();
}

// S[6][n] += the sources of a list at the sample points, NT tiles of 16 points
// a wavefront and pass; tile: 16 * 17 floats of LDS per wavefront.
template <int NT>
__device__ __forceinline__ void far_points(const MlArgs& a, const float (*xs)[ML_MAX_P], const LeafList& list, int m, float* S,
                                           float* tile) {
    const int lane = (int)threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int n = a.fine.n, Px = a.fine.P[0], Py = a.fine.P[1];
    float* const tl = tile + wv * 16 * 17;
    auto at = [&](int i, float* x) {
        x[0] = xs[0][i % Px] - 0.5f * (float)a.b[0];
        x[1] = xs[1][i / Px % Py] - 0.5f * (float)a.b[1];
        x[2] = xs[2][i / (Px * Py)] - 0.5f * (float)a.b[2];
    };
    for (int p0 = wv * NT * 16; p0 < n; p0 += (int)(blockDim.x >> 6) * NT * 16) {
        Points pt[NT];
        f32x4 c[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            float x[3];
            at(min(p0 + t * 16 + (lane & 15), n - 1), x);
            pt[t].set(x[0], x[1], x[2]);
            c[t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        }
        far_sums<NT>(list, m, pt, c);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            put_tile(tl, c[t]);
            __builtin_amdgcn_wave_barrier();
            const int p = p0 + t * 16 + (lane & 15);
            if (p < n) {
                float x[3];
                at(p, x);
                for (int o = lane >> 4; o < 6; o += 4) S[o * n + p] += field_of(tl + (lane & 15) * 17, o, x[0], x[1], x[2]);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}
__device__ __forceinline__ void far_points(const MlArgs& a, const float (*xs)[ML_MAX_P], const LeafList& list, int m, float* S,
                                           float* tile) {
    if (a.nt == 3) far_points<3>(a, xs, list, m, S, tile);
    else if (a.nt == 4) far_points<4>(a, xs, list, m, S, tile);
    else far_points<6>(a, xs, list, m, S, tile);
    __syncthreads();
}

// Source lists of LOD block (X, Y, Z) into LDS, in index order: near the parent
// block (far: not near the block itself; with ALL everything but the block
// itself), and the blocks around it (near). cnt: lengths; then counts per
// wavefront of candidates.
template <bool ALL>
__device__ __forceinline__ void leaf_lists(const MlArgs& a, int X, int Y, int Z, LeafList* far, Src* near, int* cnt) {
    constexpr int W = (LIST_FAR + 63) / 64;
    const int lane = (int)threadIdx.x & 63, waves = (int)blockDim.x >> 6;
    const float org[3] = {((float)X + 0.5f) * (float)a.b[0], ((float)Y + 0.5f) * (float)a.b[1],
                          ((float)Z + 0.5f) * (float)a.b[2]};
    Src s[W];  // the candidates of this lane: W of them for a single wavefront, else fewer
    uint64_t mf[W], mn[W];
#pragma unroll
    for (int u = 0; u < W; u++) {
        const int w = (int)(threadIdx.x >> 6) + u * waves, j = w * 64 + lane;
        mf[u] = mn[u] = 0;
        if (w >= W) continue;
        const int sx = ((X >> 1) - 1) * 2 + j % 6, sy = ((Y >> 1) - 1) * 2 + j / 6 % 6, sz = ((Z >> 1) - 1) * 2 + j / 36;
        const bool in = j < LIST_FAR && sx >= 0 && sy >= 0 && sz >= 0 && sx < (int)a.nd && sy < (int)a.nd &&
                        sz < (int)a.zext && !(sx == X && sy == Y && sz == Z) && source_at(a, sx, sy, sz, &s[u]);
        const bool nb = !ALL && within1(sx, X) && within1(sy, Y) && within1(sz, Z);
        mf[u] = __ballot(in && !nb);
        mn[u] = __ballot(in && nb);
        if (lane == 0) {
            cnt[2 + 2 * w] = __popcll(mf[u]);
            cnt[3 + 2 * w] = __popcll(mn[u]);
        }
    }
    __syncthreads();
    const uint64_t below = (1ull << lane) - 1ull, self = 1ull << lane;
    int nf = 0;
    for (int w = 0; w < W; w++) nf += cnt[2 + 2 * w];
#pragma unroll
    for (int u = 0; u < W; u++) {
        const int w = (int)(threadIdx.x >> 6) + u * waves;
        if (w >= W) continue;
        int of = __popcll(mf[u] & below), on = __popcll(mn[u] & below);
        for (int k = 0; k < w; k++) {
            of += cnt[2 + 2 * k];
            on += cnt[3 + 2 * k];
        }
        if (mf[u] & self) far->put(of, s[u], org);
        if (mn[u] & self) near[on] = s[u];
    }
    if (threadIdx.x < 16) far->pad(nf, (int)threadIdx.x);
    if (threadIdx.x == 0) {
        cnt[0] = nf;
        int nn = 0;
        for (int w = 0; w < W; w++) nn += cnt[3 + 2 * w];
        cnt[1] = nn;
    }
    __syncthreads();
}

// LOD blocks go to the XCDs (workgroup b runs on XCD b % 8) in runs: neighbours
// share coarse samples, and lines of the fields, in one L2.
__device__ __forceinline__ uint32_t block_of_xcd(uint32_t nblk) { return blockIdx.x % 8u * (nblk / 8u) + blockIdx.x / 8u; }

// LOD blocks whose cells are the sample points.
template <int CM>
__global__ void __launch_bounds__(LEAF_T) k_ml_leaf(MlArgs a) {
    extern __shared__ __align__(16) float lds[];
    __shared__ float xs[3][ML_MAX_P];
    if (!multilevel(a)) return;
    const int tid = (int)threadIdx.x, T = (int)blockDim.x, n = a.fine.n;
    LeafList* const far = (LeafList*)(lds + a.list_off);
    int* const cnt = (int*)(far + 1);
    const uint32_t blk = block_of_xcd(a.nd * a.nd * a.nd), X = blk % a.nd, Y = blk / a.nd % a.nd, Z = blk / (a.nd * a.nd);
    const int bx = (int)a.b[0], by = (int)a.b[1];
    const uint64_t base_cell = (uint64_t)X * a.b[0] + ((uint64_t)Y * a.b[1] + (uint64_t)Z * a.b[2] * a.f.ny) * a.f.nx;
    auto cell = [&](int i) {
        return base_cell + i % bx + ((uint64_t)(i / bx % by) + (uint64_t)(i / (bx * by)) * a.f.ny) * a.f.nx;
    };
    bool any = false;  // a block of solid cells has nothing to write
    for (int i = tid; i < n; i += T) any |= (a.f.flags[cell(i)] & 0x1F) != 0x01;
    if (!__syncthreads_or(any)) return;
    stage_points(a.fine, xs);
    leaf_lists<true>(a, (int)X, (int)Y, (int)Z, far, nullptr, cnt);
    from_coarse<CM>(a, X, Y, Z, lds, lds + a.v_off);
    far_points(a, xs, *far, __builtin_amdgcn_readfirstlane(cnt[0]), lds, lds + a.v_off);
    for (int i = tid; i < n; i += T) {
        const uint64_t c = cell(i);
        if ((a.f.flags[c] & 0x1F) == 0x01) continue;
        float v[6];
#pragma unroll
        for (int k = 0; k < 6; k++) v[k] = lds[k * n + i];
        write_cell(a.f, c, v, nullptr);
    }
}

// LOD blocks of more cells: the sample points first (far sources), then the
// cells, a thread taking R cells of a column along z. The samples go to the
// columns axis by axis, GC components at a time through LDS (x: V, y: W); the
// last axis runs in the thread, its weights the same for the whole wavefront.
template <int R, int CM, int GC>
__global__ void __launch_bounds__(512) k_ml_cells(MlArgs a) {
    extern __shared__ __align__(16) float lds[];
    __shared__ float xs[3][ML_MAX_P];
    if (!multilevel(a)) return;
    const int tid = (int)threadIdx.x, T = (int)blockDim.x;
    LeafList* const far = (LeafList*)(lds + a.list_off);
    Src* const near = (Src*)(far + 1);
    int* const cnt = (int*)(near + LIST_NEAR);
    const uint32_t blk = block_of_xcd(a.nd * a.nd * a.nd), X = blk % a.nd, Y = blk / a.nd % a.nd, Z = blk / (a.nd * a.nd);
    const int bx = (int)a.b[0], by = (int)a.b[1], bz = (int)a.b[2];
    const int Px = a.fine.P[0], Py = a.fine.P[1], Pz = a.fine.P[2], n = a.fine.n;
    float* const S = lds;
    const uint64_t base_cell = (uint64_t)X * a.b[0] + ((uint64_t)Y * a.b[1] + (uint64_t)Z * a.b[2] * a.f.ny) * a.f.nx;
    const uint64_t nxy = (uint64_t)a.f.nx * a.f.ny;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int zg = wave / (int)a.colw, cw = wave % (int)a.colw;  // this wave's z group and columns
    const int W = (int)a.colw * 64;                            // columns of a tile
    const int zt = T / W, ncol = bx * by, tiles = (int)(a.ntile * a.nzt);
    // the cells of a tile that have a field: R bits
    auto live_of = [&](int tile) -> uint32_t {
        const int col = tile % (int)a.ntile * W + cw * 64 + lane, z0 = (tile / (int)a.ntile * zt + zg) * R;
        const uint64_t cell0 = base_cell + col % bx + (uint64_t)(col / bx) * a.f.nx + z0 * nxy;
        uint8_t f[R];
#pragma unroll
        for (int r = 0; r < R; r++) f[r] = col < ncol && z0 + r < bz ? a.f.flags[cell0 + r * nxy] : 0x01;
        uint32_t live = 0;
#pragma unroll
        for (int r = 0; r < R; r++) live |= ((f[r] & 0x1F) != 0x01 ? 1u : 0u) << r;
        return live;
    };
    uint32_t live0 = live_of(0), any = live0;
    for (int tile = 1; tile < tiles; tile++) any |= live_of(tile);
    if (!__syncthreads_or(any != 0u)) return;  // a block of solid cells has nothing to write
    stage_points(a.fine, xs);
    leaf_lists<false>(a, (int)X, (int)Y, (int)Z, far, near, cnt);
    from_coarse<CM>(a, X, Y, Z, S, lds + a.v_off);
    far_points(a, xs, *far, __builtin_amdgcn_readfirstlane(cnt[0]), S, lds + a.v_off);
    const int m = __builtin_amdgcn_readfirstlane(cnt[1]);
    for (int tile = 0; tile < tiles; tile++) {
        const int col0 = tile % (int)a.ntile * W, col = col0 + cw * 64 + lane;
        const int z0 = (tile / (int)a.ntile * zt + zg) * R;
        const int x = col % bx, y = col / bx;
        const uint32_t live = tile == 0 ? live0 : live_of(tile);
        const uint64_t cell0 = base_cell + x + (uint64_t)y * a.f.nx + z0 * nxy;
        float acc[R][6];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 6; c++) acc[r][c] = 0.0f;
        float* const V = lds + a.v_off;
        float* const Wb = lds + a.w_off;
        const int y0 = col0 / bx, rows = min((col0 + W - 1) / bx, by - 1) - y0 + 1;  // of the tile's columns
        const int at = min(col, ncol - 1) - y0 * bx, ws = (int)a.rows * bx;
        const cfloat_p Mx = (cfloat_p)(a.ws + a.t_cell[0]);
        const cfloat_p My = (cfloat_p)(a.ws + a.t_cell[1] + y0 * CM);
        const cfloat_p Mz = (cfloat_p)(a.ws + a.t_cell[2] + z0);
#pragma unroll
        for (int c0 = 0; c0 < 6; c0 += GC) {
            lines<CM>(
                GC * Pz * Py, Px, bx, Mx,
                [&](int i, int* st) {
                    *st = 1;
                    return S + c0 * n + i * Px;
                },
                [&](int i, int o, float v) { V[i * bx + o] = v; });
            __syncthreads();
            lines<CM>(
                GC * Pz * bx, Py, rows, My,
                [&](int i, int* st) {
                    *st = bx;
                    return V + i / bx * Py * bx + i % bx;
                },
                [&](int i, int o, float v) { Wb[i / bx * ws + o * bx + i % bx] = v; });
            __syncthreads();
            float mz[R];
#pragma unroll
            for (int r = 0; r < R; r++) mz[r] = Mz[r];
            for (int k = 0; k < Pz; k++) {
                const cfloat_p next = Mz + min(k + 1, Pz - 1) * (int)a.cells[2];
                float mn[R];
#pragma unroll
                for (int r = 0; r < R; r++) mn[r] = next[r];
#pragma unroll
                for (int c = 0; c < GC; c++) {
                    const float w = Wb[(c * Pz + k) * ws + at];
#pragma unroll
                    for (int r = 0; r < R; r++) acc[r][c0 + c] = __builtin_fmaf(mz[r], w, acc[r][c0 + c]);
                }
#pragma unroll
                for (int r = 0; r < R; r++) mz[r] = mn[r];
            }
        }
        // the sources around the block at the cells of the column: the terms
        // of x and y alone once for the R cells
        if (__any(live != 0u)) {
            const float cx = (float)((int)X * bx + x), cy = (float)((int)Y * by + y), cz = (float)((int)Z * bz + z0);
            for (int i = 0; i < m; i++) {
                const float4 p = near[i].p, v = near[i].v;
                const float rx = cx - p.x, ry = cy - p.y, rz0 = cz - p.z;
                const float sxy = __builtin_fmaf(rx, rx, ry * ry);
                const float vz = __builtin_fmaf(v.x, ry, -v.y * rx), m1 = v.z * ry, m2 = v.z * rx;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const float rz = rz0 + (float)r;
                    const float inv = __builtin_amdgcn_rsqf(__builtin_fmaf(rz, rz, sxy));
                    const float t = p.w * (inv * inv * inv);
                    acc[r][0] = __builtin_fmaf(t, rx, acc[r][0]);
                    acc[r][1] = __builtin_fmaf(t, ry, acc[r][1]);
                    acc[r][2] = __builtin_fmaf(t, rz, acc[r][2]);
                    acc[r][3] = __builtin_fmaf(t, __builtin_fmaf(v.y, rz, -m1), acc[r][3]);
                    acc[r][4] = __builtin_fmaf(t, __builtin_fmaf(-v.x, rz, m2), acc[r][4]);
                    acc[r][5] = __builtin_fmaf(t, vz, acc[r][5]);
                }
            }
        }
        // E, then B: all of the column's loads before its stores
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float* const stat = h ? a.f.b_stat : a.f.e_stat;
            float* const dyn = h ? a.f.b_dyn : a.f.e_dyn;
            const float k = h ? a.f.kmu : a.f.ke;
            float st[R][3];
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < 3; c++) st[r][c] = live >> r & 1u ? stat[cell0 + r * nxy + c * a.f.N] : 0.0f;
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < 3; c++)
                    if (live >> r & 1u) dyn[cell0 + r * nxy + c * a.f.N] = st[r][c] + k * acc[r][3 * h + c];
        }
    }
}

}  // namespace

// Sample points: as many per axis as the interpolation error asks for. The
// nearest source that a block's samples hold lies 2 block sides from its
// centre along an axis, and 1.5 sides from every cell; a function that is
// singular at distance d straight ahead of (beside) an interval of half width
// h is interpolated to rho^-P with rho = r + sqrt(r^2 - 1) (r + sqrt(r^2 + 1)),
// r = d / h. Cubic blocks get 9 points a side on level D, 10 on D - 1 and 11 on
// D - 2; interpolated in double on 16^3 LOD blocks, the field of the sources that
// a level takes is then off by 1e-7, 5e-8 and 2e-8 of itself (a point fewer: 4e-7,
// 6e-7 and 1.4e-7). With the rounding of the sums the update is within 2e-7 to 4e-7
// of the sum in double on blocks of 4 to 24 cells a side, cubic and uneven, a direct
// one within 1.2e-6 (depth 4; 1.6e-7 to 3.4e-7 and 4.5e-7 at depth 3).
static bool grid_of(const uint32_t b[3], uint32_t shift, uint32_t side, double tol, MlGrid* g) {
    g->shift = shift;
    g->side = side;
    g->n = 1;
    const double shortest = std::min(b[0], std::min(b[1], b[2])) * (double)(1u << shift);
    for (int k = 0; k < 3; k++) {
        const int w = (int)(b[k] << shift);
        const double h = std::max(0.5 * (w - 1), 0.25);
        const double r1 = 1.5 * shortest / h, r2 = 2.0 * w / h;
        const double rho = std::min(r1 + std::sqrt(r1 * r1 + 1.0), r2 + std::sqrt(r2 * r2 - 1.0));
        const int P = std::min((int)std::ceil(std::log(1.0 / tol) / std::log(rho)), w);
        if (P > ML_MAX_P) return false;
        g->P[k] = P;
        g->n *= P;
        for (int i = 0; i < P; i++) {
            if (P == w) g->x[k][i] = (float)i;
            else  // Chebyshev points, stretched so that the outer ones are the first and last cell
                g->x[k][i] = (float)(0.5 * (w - 1) * (1.0 - std::cos((2 * i + 1) * M_PI / (2 * P)) / std::cos(M_PI / (2 * P))));
        }
    }
    g->groups = side * side * side * (uint32_t)((g->n + COARSE_PTS - 1) / COARSE_PTS);
    return true;
}

// The rule. Depth 3 and 4: below depth 3 all or almost all sources are near,
// deeper trees have their near field on the cells. Sources enough and finite
// (MODE_FAST): at least 1/32 of the LOD blocks, 128 of 4096, where the direct
// sum of 256^3 takes 0.62 ms and this update, which has its interpolation
// whatever the sources, 0.60 ms (1.15 ms with all of them; direct 16.9 ms). At
// depth 3 (439 sources) uneven blocks (ld > 12: many points) pay from some
// 400 000 cells on: 64 x 80 x 48 0.103 ms, direct 0.078 ms; 80 x 64 x 96 0.121 and
// 0.134 ms; even ones always do (48^3 0.058 and 0.065 ms). Blocks so uneven or so
// large that the points do not fit take the direct sum.
static bool tree(const FieldArgs& f) { return !f.f64 && !f.near && (f.D == 3 || f.D == 4); }

static size_t header(uint32_t nd, uint32_t zext) { return ML_DENSE + (size_t)zext * nd * nd * 4; }

static bool plan(const FieldArgs& f, MlArgs* a) {
    if (!tree(f)) return false;
    *a = MlArgs{};
    a->f = f;
    a->qu = f.qu;
    a->ws = f.ml_ws;
    const uint32_t D = f.D, nd = 1u << D, levels = D - 2;
    a->nd = nd;
    for (uint32_t i = 0; i <= D; i++) a->n_lod += 1u << (3 * i);
    a->lo = a->n_lod - nd * nd * nd;
    a->zext = (a->n_lod + nd * nd - 1) / (nd * nd);
    a->b[0] = f.nx / nd;
    a->b[1] = f.ny / nd;
    a->b[2] = f.nz / nd;
    a->levels = levels;
    const uint32_t cells = a->b[0] * a->b[1] * a->b[2];
    int most = 0;  // sample points of an axis
    if (!grid_of(a->b, 0, nd, 5e-8, &a->fine)) return false;
    for (uint32_t l = 0; l < levels; l++)
        if (!grid_of(a->b, D - 2 - l, 4u << l, l + 1 == levels ? 5e-8 : 1e-8, &a->coarse[l])) return false;
    for (int k = 0; k < 3; k++) {
        most = std::max(most, a->fine.P[k]);
        for (uint32_t l = 0; l < levels; l++) most = std::max(most, a->coarse[l].P[k]);
    }
    a->ld = most <= 12 ? 12 : most <= 16 ? 16 : ML_MAX_P;
    a->leaf = (uint32_t)a->fine.n == cells;
    // work split
    if (a->leaf) {
        a->threads = std::min(cells <= 1024 ? LEAF_T / 2 : LEAF_T, (cells + 63) / 64 * 64);
    } else {
        // columns of R cells; the z groups of a tile, then its columns, up to 8 wavefronts
        const uint32_t ncolw = (a->b[0] * a->b[1] + 63) / 64, nzg = (a->b[2] + 7) / 8, zt = std::min(nzg, 8u);
        a->R = std::max(4u, (a->b[2] + nzg - 1) / nzg);
        a->nzt = (nzg + zt - 1) / zt;
        a->ntile = (ncolw + 8 / zt - 1) / (8 / zt);
        a->colw = (ncolw + a->ntile - 1) / a->ntile;
        a->threads = 64 * a->colw * zt;
        a->cells[0] = a->b[0];
        a->cells[1] = a->b[1];
        a->cells[2] = a->nzt * zt * a->R;
    }
    // workspace: header, sources, tables, samples
    size_t at = header(nd, a->zext);
    a->t0 = (uint32_t)at;
    for (int k = 0; k < 3; k++) {
        a->t_cell[k] = (uint32_t)at;
        at += (size_t)a->cells[k] * (k < 2 ? a->ld : (uint32_t)a->fine.P[k]);
        for (uint32_t l = 0; l < levels; l++) {
            a->t_up[l][k] = (uint32_t)at;
            at += (size_t)(1u << a->coarse[l].shift) * a->fine.P[k] * a->ld;
        }
    }
    a->t_end = (uint32_t)at;
    for (uint32_t l = 0; l < levels; l++) {
        a->samples[l] = (uint32_t)at;
        at += (size_t)a->coarse[l].side * a->coarse[l].side * a->coarse[l].side * 6 * a->coarse[l].n;
    }
    if (at > ML_WS_FLOATS) return false;
    a->ws_floats = (uint32_t)at;
    // LDS: samples, scratch (from_coarse: two half-interpolated grids;
    // far_points: tiles; then V and W), source lists; three components at a
    // time where that leaves room for two workgroups, else one
    a->rows = a->leaf ? 0 : std::min((a->colw * 64 - 1) / a->b[0] + 2, a->b[1]);
    for (uint32_t gc : {3u, 1u}) {
        if (gc == 3 && a->ld != 12) continue;
        a->gc = gc;
        size_t tmp = (size_t)a->threads / 64 * 16 * 17;
        for (uint32_t l = 0; l < levels; l++) {
            const MlGrid& g = a->coarse[l];
            tmp = std::max(tmp, (size_t)gc * g.P[2] * a->fine.P[0] * (g.P[1] + a->fine.P[1]));
        }
        const size_t V = a->leaf ? 0 : (size_t)gc * a->fine.P[2] * a->fine.P[1] * a->b[0];
        a->v_off = 6 * a->fine.n;
        a->w_off = (uint32_t)(a->v_off + V);
        a->list_off = (uint32_t)(a->v_off + std::max(V + (size_t)gc * a->fine.P[2] * a->rows * a->b[0], tmp) + 3) & ~3u;
        a->lds = a->list_off * 4 + (uint32_t)(sizeof(LeafList) + LIST_NEAR * sizeof(Src)) + LIST_CNT * 4;
        if (a->lds <= ML_LDS) break;
    }
    if (a->lds > ML_LDS) return false;
    // far_points: tiles of 16 points per wavefront and pass, the split with the fewest idle
    uint32_t best = ~0u;
    for (uint32_t nt : {6u, 4u, 3u}) {
        const uint32_t per = nt * 16 * (a->threads / 64), cost = (a->fine.n + per - 1) / per * nt;
        if (cost < best) {
            best = cost;
            a->nt = nt;
        }
    }
    return true;
}

bool ml_plan(const FieldArgs& f, MlArgs* a) {
    return f.ml_ws != nullptr && plan(f, a) && (f.D == 4 || a->ld == 12 || f.N >= 400000u);
}

size_t ml_workspace(const FieldArgs& f) {
    if (!tree(f)) return 0;
    MlArgs a;
    if (plan(f, &a)) return a.ws_floats;
    const uint32_t nd = 1u << f.D;
    return header(nd, nd + 4);  // the header alone (zext is nd + 2 or nd + 3)
}

hipError_t launch_field_fast(const MlArgs& a, hipStream_t s) {
    uint32_t gc = (a.t_end - a.t0 + COARSE_T - 1) / COARSE_T;
    for (uint32_t l = 0; l < a.levels; l++) gc += a.coarse[l].groups;
    hipLaunchKernelGGL(k_ml_coarse, dim3(gc), dim3(COARSE_T), 0, s, a);
    const dim3 g(a.nd * a.nd * a.nd), b(a.threads);
    if (a.leaf) {
        if (a.ld == 12) hipLaunchKernelGGL(k_ml_leaf<12>, g, b, a.lds, s, a);
        else if (a.ld == 16) hipLaunchKernelGGL(k_ml_leaf<16>, g, b, a.lds, s, a);
        else hipLaunchKernelGGL(k_ml_leaf<ML_MAX_P>, g, b, a.lds, s, a);
    } else {
#define ION_CELLS(R)                                                                        \
    do {                                                                                    \
        if (a.gc == 3) hipLaunchKernelGGL((k_ml_cells<R, 12, 3>), g, b, a.lds, s, a);       \
        else if (a.ld == 12) hipLaunchKernelGGL((k_ml_cells<R, 12, 1>), g, b, a.lds, s, a); \
        else if (a.ld == 16) hipLaunchKernelGGL((k_ml_cells<R, 16, 1>), g, b, a.lds, s, a); \
        else hipLaunchKernelGGL((k_ml_cells<R, ML_MAX_P, 1>), g, b, a.lds, s, a);           \
    } while (0)
        switch (a.R) {
            case 4: ION_CELLS(4); break;
            case 5: ION_CELLS(5); break;
            case 6: ION_CELLS(6); break;
            case 7: ION_CELLS(7); break;
            default: ION_CELLS(8); break;
        }
#undef ION_CELLS
    }
    return hipGetLastError();
}

}  // namespace ion
