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
//                    in the reference) one by one, plus the interpolated
//                    samples.
// Sample points are Chebyshev points, as many per axis as bring the
// interpolation error below the rounding of the float sums (ml_plan); the
// weights are computed in double. A block of up to 9 or so cells a side has as
// many points as cells: its cells are the sample points (k_ml_leaf).
//
// Why: a direct sum costs 13 VALU instructions and one v_rsq_f32 for each cell
// and source, 16.1 ms at 256^3 with 3511 sources (111 TFLOP/s, VALU issue);
// this split leaves about 24 sources a cell and 145 a sample point and takes
// 1.23 ms (levels 2 and 3 0.42 ms, the rest 0.80 ms), with a smaller error
// against the sum in double (8e-8 against 4.5e-7: fewer float additions in a
// row). 240 x 336 x 144 (blocks of 15 x 21 x 9 cells): 17.4 -> 3.0 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "field_fast.hpp"
#include "judge.hpp"

namespace ion {

namespace {

constexpr int COARSE_T = 1024, COARSE_G = 256;  // threads of a coarse workgroup, threads per source group
constexpr int COARSE_K = 2;                     // sample points per thread
constexpr int COARSE_PTS = COARSE_K * COARSE_G; // sample points per workgroup
constexpr uint32_t LIST_FAR = 216, LIST_NEAR = 32;  // sources of a leaf: 6^3 candidates, 3^3 around the block
constexpr uint32_t LEAF_T = 256;
constexpr uint32_t ML_LDS = 80 * 1024;  // two workgroups of k_ml_cells on a CU

typedef const __attribute__((address_space(4))) float* cfloat_p;  // tables: read through the scalar cache

struct Src {
    float4 p;  // centre, charge
    float4 v;  // mean velocity
};

// t = q / |r|^3; e += t r, b += t (v x r)
__device__ __forceinline__ void interact(const float4 p, const float4 v, float x, float y, float z, float* a) {
    const float rx = x - p.x, ry = y - p.y, rz = z - p.z;
    const float inv = __builtin_amdgcn_rsqf(__builtin_fmaf(rx, rx, __builtin_fmaf(ry, ry, rz * rz)));
    const float t = p.w * (inv * inv * inv);
    a[0] = __builtin_fmaf(t, rx, a[0]);
    a[1] = __builtin_fmaf(t, ry, a[1]);
    a[2] = __builtin_fmaf(t, rz, a[2]);
    a[3] = __builtin_fmaf(t, __builtin_fmaf(v.y, rz, -v.z * ry), a[3]);
    a[4] = __builtin_fmaf(t, __builtin_fmaf(v.z, rx, -v.x * rz), a[4]);
    a[5] = __builtin_fmaf(t, __builtin_fmaf(v.x, ry, -v.y * rx), a[5]);
}

__device__ __forceinline__ bool multilevel(const MlArgs& a) { return a.levels > 0 && __float_as_uint(a.ws[0]) != 0u; }

// LOD index of the source at (X, Y, Z) of the LOD grid (Z up to zext: the last
// indices of the range lie above the domain), and whether the field update
// reads it: indices from lo to n_lod, charges that are not zero.
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
__device__ void ml_tables(const MlArgs& a, uint32_t t) {
    if (t >= a.t_end) return;
    const uint32_t ld = a.ld;
    for (int k = 0; k < 3; k++) {
        const int P = a.fine.P[k];
        const uint32_t cells = a.cells[k];
        uint32_t i = t - a.t_cell[k];
        if (t >= a.t_cell[k] && i < cells * (k < 2 ? ld : (uint32_t)P)) {
            if (k < 2) a.ws[t] = (int)(i % ld) < P ? lagrange(a.fine.x[k], P, i % ld, (double)(i / ld)) : 0.0f;
            else a.ws[t] = lagrange(a.fine.x[k], P, i / cells, (double)(i % cells));
        }
        for (uint32_t l = 0; l < a.levels; l++) {
            const MlGrid& c = a.coarse[l];
            i = t - a.t_up[l][k];
            if (t < a.t_up[l][k] || i >= (uint32_t)((1 << c.shift) * P) * ld) continue;
            const uint32_t off = i / (P * ld), p = i / ld % P;
            a.ws[t] = (int)(i % ld) < c.P[k]
                          ? lagrange(c.x[k], c.P[k], i % ld, (double)(off * a.b[k]) + (double)a.fine.x[k][p])
                          : 0.0f;
        }
    }
}

// Samples of the coarse levels: a workgroup takes COARSE_PTS points of a block
// (level 2 first: its blocks have the longest source lists); the last
// workgroups compute the tables. The sources are gathered into LDS COARSE_T
// candidates at a time, in index order; the four groups of threads take every
// fourth one and are summed at the end.
// Bound by VALU issue: 21 instructions and a v_rsq_f32 per point and source.
__global__ void __launch_bounds__(COARSE_T) __attribute__((amdgpu_waves_per_eu(8))) k_ml_coarse(MlArgs a) {
    constexpr int GROUPS = COARSE_T / COARSE_G;
    __shared__ __align__(16) union {
        Src list[COARSE_T];
        float part[GROUPS - 1][COARSE_K * 6][COARSE_G];
    } sh;
    __shared__ uint32_t wtot[COARSE_T / 64];
    if (!multilevel(a)) return;
    uint32_t blk = blockIdx.x;
    uint32_t li = 0;
    while (li < a.levels && blk >= a.coarse[li].groups) blk -= a.coarse[li++].groups;
    const int tid = (int)threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (li == a.levels) {
        ml_tables(a, 16 + blk * COARSE_T + tid);
        return;
    }
    const MlGrid& g = a.coarse[li];
    const int parts = (g.n + COARSE_PTS - 1) / COARSE_PTS, n0 = (int)blk % parts * COARSE_PTS;
    blk /= parts;
    const int side = (int)g.side, shift = (int)g.shift;
    const int C[3] = {(int)blk % side, (int)blk / side % side, (int)blk / (side * side)};
    // candidates: the sources near the parent block (on level 2, all)
    int lo3[3], n3[3];
    for (int k = 0; k < 3; k++) {
        const int end = (int)(k == 2 ? a.zext : a.nd);
        lo3[k] = li == 0 ? 0 : max(0, ((C[k] >> 1) - 1) * (2 << shift));
        n3[k] = (li == 0 ? end : min(end, ((C[k] >> 1) + 2) * (2 << shift))) - lo3[k];
    }
    const int total = n3[0] * n3[1] * n3[2];
    const int grp = wv / (COARSE_G / 64), gt = tid % COARSE_G;
    float px[COARSE_K], py[COARSE_K], pz[COARSE_K], acc[COARSE_K][6];
#pragma unroll
    for (int k = 0; k < COARSE_K; k++) {
        const int i = min(n0 + k * COARSE_G + gt, g.n - 1);
        px[k] = (float)(C[0] * (int)(a.b[0] << shift)) + g.x[0][i % g.P[0]];
        py[k] = (float)(C[1] * (int)(a.b[1] << shift)) + g.x[1][i / g.P[0] % g.P[1]];
        pz[k] = (float)(C[2] * (int)(a.b[2] << shift)) + g.x[2][i / (g.P[0] * g.P[1])];
#pragma unroll
        for (int c = 0; c < 6; c++) acc[k][c] = 0.0f;
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
        const uint64_t mask = __ballot(keep);
        __syncthreads();
        if (lane == 0) wtot[wv] = (uint32_t)__popcll(mask);
        __syncthreads();
        int off = __popcll(mask & ((1ull << lane) - 1ull)), m = 0;
        for (int w = 0; w < COARSE_T / 64; w++) {
            if (w < wv) off += (int)wtot[w];
            m += (int)wtot[w];
        }
        if (keep) sh.list[off] = s;
        __syncthreads();
        m = __builtin_amdgcn_readfirstlane(m);
        for (int i = grp; i < m; i += GROUPS) {
            const float4 p = sh.list[i].p, v = sh.list[i].v;
#pragma unroll
            for (int k = 0; k < COARSE_K; k++) interact(p, v, px[k], py[k], pz[k], acc[k]);
        }
    }
    // sum of the groups, in order
    float* const out = a.ws + a.samples[li] + (size_t)blk * 6 * g.n;
    __syncthreads();
    if (grp > 0) {
#pragma unroll
        for (int k = 0; k < COARSE_K; k++)
#pragma unroll
            for (int c = 0; c < 6; c++) sh.part[grp - 1][k * 6 + c][gt] = acc[k][c];
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
        for (int k = 0; k < COARSE_K; k++) {
            const int i = n0 + k * COARSE_G + gt;
            if (i >= g.n) continue;
#pragma unroll
            for (int c = 0; c < 6; c++) {
                float v = acc[k][c];
#pragma unroll
                for (int h = 0; h < GROUPS - 1; h++) v += sh.part[h][k * 6 + c][gt];
                out[c * g.n + i] = v;
            }
        }
    }
}

// Interpolation along one axis: each line of c values in[k * stride] gives nout
// values M[o] . in, where row o of M has CM weights (zero from c on) that are
// the same for every thread: they come as scalar operands.
template <int CM, class In, class Out>
__device__ __forceinline__ void lines(int nlines, int c, int nout, cfloat_p M, In in, Out out) {
    for (int line = (int)threadIdx.x; line < nlines; line += (int)blockDim.x) {
        int stride;
        const float* const p = in(line, &stride);
        float v[CM];
#pragma unroll
        for (int k = 0; k < CM; k++) v[k] = k < c ? p[k * stride] : 0.0f;
        for (int o = 0; o < nout; o++) {
            float s = M[o * CM] * v[0];
#pragma unroll
            for (int k = 1; k < CM; k++) s = __builtin_fmaf(M[o * CM + k], v[k], s);
            out(line, o, s);
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

// S[6][n] += the far sources at the sample points: groups of threads take
// every a.pg-th source, K points a thread and pass.
template <int K>
__device__ __forceinline__ void far_points(const MlArgs& a, const float org[3], const Src* list, int m, float* S) {
    const int G = (int)(a.threads / a.pg), gt = (int)threadIdx.x % G;
    const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x / G);  // groups are whole wavefronts
    const int n = a.fine.n, Px = a.fine.P[0], Py = a.fine.P[1];
    for (int n0 = 0; n0 < n; n0 += K * G) {
        float px[K], py[K], pz[K], s[K][6];
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int i = min(n0 + k * G + gt, n - 1);
            px[k] = org[0] + a.fine.x[0][i % Px];
            py[k] = org[1] + a.fine.x[1][i / Px % Py];
            pz[k] = org[2] + a.fine.x[2][i / (Px * Py)];
#pragma unroll
            for (int c = 0; c < 6; c++) s[k][c] = 0.0f;
        }
        for (int i = grp; i < m; i += (int)a.pg) {
            const float4 p = list[i].p, v = list[i].v;
#pragma unroll
            for (int k = 0; k < K; k++) interact(p, v, px[k], py[k], pz[k], s[k]);
        }
        for (int h = 0; h < (int)a.pg; h++) {  // one group after the other
            if (h == grp) {
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const int i = n0 + k * G + gt;
                    if (i < n)
#pragma unroll
                        for (int c = 0; c < 6; c++) S[c * n + i] += s[k][c];
                }
            }
            __syncthreads();
        }
    }
}

// Source lists of LOD block (X, Y, Z) into LDS, in index order, by the first
// wavefront: near the parent but not near the block (far), and the blocks
// around it without itself (near).
__device__ __forceinline__ void leaf_lists(const MlArgs& a, int X, int Y, int Z, Src* far, Src* near, uint32_t* cnt) {
    if (threadIdx.x < 64) {
        const uint32_t lane = threadIdx.x;
        uint32_t nf = 0, nn = 0;
        for (uint32_t j0 = 0; j0 < LIST_FAR; j0 += 64) {
            const int j = (int)(j0 + lane);
            const int sx = ((X >> 1) - 1) * 2 + j % 6, sy = ((Y >> 1) - 1) * 2 + j / 6 % 6, sz = ((Z >> 1) - 1) * 2 + j / 36;
            Src s;
            const bool in = j < (int)LIST_FAR && sx >= 0 && sy >= 0 && sz >= 0 && sx < (int)a.nd && sy < (int)a.nd &&
                            sz < (int)a.zext && !(sx == X && sy == Y && sz == Z) && source_at(a, sx, sy, sz, &s);
            const bool nb = within1(sx, X) && within1(sy, Y) && within1(sz, Z);
            const uint64_t mf = __ballot(in && !nb), mn = __ballot(in && nb), below = (1ull << lane) - 1ull;
            if (in && !nb) far[nf + (uint32_t)__popcll(mf & below)] = s;
            if (in && nb) near[nn + (uint32_t)__popcll(mn & below)] = s;
            nf += (uint32_t)__popcll(mf);
            nn += (uint32_t)__popcll(mn);
        }
        if (lane == 0) {
            cnt[0] = nf;
            cnt[1] = nn;
        }
    }
    __syncthreads();
}

// Chunk of the compacted list of all sources for the direct sum; the own LOD
// block's entry becomes one that adds zero.
__device__ __forceinline__ uint32_t all_sources(const MlArgs& a, uint32_t own, uint32_t base, Src* list) {
    const uint32_t m = min(LIST_FAR, *a.f.src_count - base);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < m; i += blockDim.x) {
        Src s{a.f.src_pq[base + i], a.f.src_vd[base + i]};
        if (__float_as_uint(s.v.w) == own) {
            s.p = make_float4(-4.0e6f, 0.0f, 0.0f, 0.0f);
            s.v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        list[i] = s;
    }
    __syncthreads();
    return m;
}

// The cell's fields: raw sums, or E_dyn / B_dyn (compared with the surrogate's
// sums they replace, for the judge).
__device__ __forceinline__ void write_cell(const FieldArgs& f, uint64_t n, const float* v, float* jd) {
    const uint64_t N = f.N;
    if (f.raw != nullptr) {
#pragma unroll
        for (int c = 0; c < 6; c++) f.raw[(uint64_t)c * N + n] = v[c];
        return;
    }
#pragma unroll
    for (int c = 0; c < 6; c++) {
        float* const dyn = (c < 3 ? f.e_dyn : f.b_dyn) + (uint64_t)(c % 3) * N + n;
        const float* const stat = (c < 3 ? f.e_stat : f.b_stat) + (uint64_t)(c % 3) * N + n;
        if (f.judge != nullptr) {
            const float d = *dyn - v[c];
            jd[c < 3 ? 0 : 2] = __builtin_fmaf(d, d, jd[c < 3 ? 0 : 2]);
            jd[c < 3 ? 1 : 3] = __builtin_fmaf(v[c], v[c], jd[c < 3 ? 1 : 3]);
        }
        *dyn = *stat + (c < 3 ? f.ke : f.kmu) * v[c];
    }
}

// LOD blocks whose cells are the sample points: K cells per thread.
template <int K, int CM>
__global__ void __launch_bounds__(LEAF_T) k_ml_leaf(MlArgs a) {
    extern __shared__ __align__(16) float lds[];
    const uint32_t tid = threadIdx.x, T = blockDim.x;
    Src* const far = (Src*)(lds + a.list_off);
    Src* const near = far + LIST_FAR;
    uint32_t* const cnt = (uint32_t*)(near + LIST_NEAR);
    const uint32_t blk = blockIdx.x, X = blk % a.nd, Y = blk / a.nd % a.nd, Z = blk / (a.nd * a.nd);
    float px[K], py[K], pz[K], acc[K][6];
    uint64_t cell[K];
    bool live[K];
    bool any = false;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const uint32_t i = tid + (uint32_t)k * T;
        const uint32_t x = X * a.b[0] + i % a.b[0], y = Y * a.b[1] + i / a.b[0] % a.b[1], z = Z * a.b[2] + i / (a.b[0] * a.b[1]);
        live[k] = i < (uint32_t)a.fine.n;
        cell[k] = (uint64_t)x + ((uint64_t)y + (uint64_t)z * a.f.ny) * a.f.nx;
        if (live[k]) live[k] = (a.f.flags[cell[k]] & 0x1F) != 0x01;
        any |= live[k];
        px[k] = (float)x;
        py[k] = (float)y;
        pz[k] = (float)z;
    }
    float jd[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (__syncthreads_or(any)) {
#pragma unroll
        for (int k = 0; k < K; k++)
#pragma unroll
            for (int c = 0; c < 6; c++) acc[k][c] = 0.0f;
        auto sweep = [&](const Src* list, uint32_t m) {
            for (uint32_t i = 0; i < m; i++) {
                const float4 p = list[i].p, v = list[i].v;
#pragma unroll
                for (int k = 0; k < K; k++) interact(p, v, px[k], py[k], pz[k], acc[k]);
            }
        };
        if (multilevel(a)) {
            leaf_lists(a, (int)X, (int)Y, (int)Z, far, near, cnt);
            from_coarse<CM>(a, X, Y, Z, lds, lds + a.v_off);
#pragma unroll
            for (int k = 0; k < K; k++) {
                const uint32_t i = min(tid + (uint32_t)k * T, (uint32_t)a.fine.n - 1u);
#pragma unroll
                for (int c = 0; c < 6; c++) acc[k][c] = lds[c * a.fine.n + (int)i];
            }
            if (__any(any)) {
                sweep(far, cnt[0]);
                sweep(near, cnt[1]);
            }
        } else {
            const uint32_t count = *a.f.src_count;
            for (uint32_t base = 0; base < count; base += LIST_FAR) sweep(far, all_sources(a, blk, base, far));
        }
#pragma unroll
        for (int k = 0; k < K; k++)
            if (live[k]) write_cell(a.f, cell[k], acc[k], jd);
    }
    if (a.f.judge != nullptr) judge_block_sums(jd, a.f.judge);
}

// LOD blocks of more cells: the sample points first (far sources), then the
// cells, a thread taking R cells of a column along z. The samples go to the
// columns axis by axis, GC components at a time through LDS (x: V, y: W); the
// last axis runs in the thread, its weights the same for the whole wavefront.
template <int R, int CM, int GC>
__global__ void __launch_bounds__(512) k_ml_cells(MlArgs a) {
    extern __shared__ __align__(16) float lds[];
    const int tid = (int)threadIdx.x, T = (int)blockDim.x;
    Src* const far = (Src*)(lds + a.list_off);
    Src* const near = far + LIST_FAR;
    uint32_t* const cnt = (uint32_t*)(near + LIST_NEAR);
    const uint32_t blk = blockIdx.x, X = blk % a.nd, Y = blk / a.nd % a.nd, Z = blk / (a.nd * a.nd);
    const int bx = (int)a.b[0], by = (int)a.b[1], bz = (int)a.b[2];
    const int Px = a.fine.P[0], Py = a.fine.P[1], Pz = a.fine.P[2], n = a.fine.n;
    float* const S = lds;
    float jd[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint64_t base_cell = (uint64_t)X * a.b[0] + ((uint64_t)Y * a.b[1] + (uint64_t)Z * a.b[2] * a.f.ny) * a.f.nx;
    const uint64_t nxy = (uint64_t)a.f.nx * a.f.ny;
    const bool ml = multilevel(a);
    // a block of solid cells has nothing to write
    bool any = false;
    for (int col = tid; col < bx * by; col += T) {
        const uint64_t c0 = base_cell + col % bx + (uint64_t)(col / bx) * a.f.nx;
        for (int z = 0; z < bz; z++) any |= (a.f.flags[c0 + z * nxy] & 0x1F) != 0x01;
    }
    if (__syncthreads_or(any)) {
        if (ml) {
            leaf_lists(a, (int)X, (int)Y, (int)Z, far, near, cnt);
            from_coarse<CM>(a, X, Y, Z, S, lds + a.v_off);
            const float org[3] = {(float)((int)X * bx), (float)((int)Y * by), (float)((int)Z * bz)};
            const int m = __builtin_amdgcn_readfirstlane((int)cnt[0]);
            if (a.pk == 2) far_points<2>(a, org, far, m, S);
            else if (a.pk == 3) far_points<3>(a, org, far, m, S);
            else far_points<4>(a, org, far, m, S);
        }
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int zg = wave / (int)a.colw, cw = wave % (int)a.colw;  // this wave's z group and columns
        const int W = (int)a.colw * 64;                            // columns of a tile
        const int zt = (int)a.threads / W, ncol = bx * by;
        for (int tile = 0; tile < (int)(a.ntile * a.nzt); tile++) {
            const int col0 = tile % (int)a.ntile * W, col = col0 + cw * 64 + lane;
            const int z0 = (tile / (int)a.ntile * zt + zg) * R;
            const int x = col % bx, y = col / bx;
            uint32_t live = 0;
            const uint64_t cell0 = base_cell + x + (uint64_t)y * a.f.nx + z0 * nxy;
#pragma unroll
            for (int r = 0; r < R; r++)
                if (col < ncol && z0 + r < bz && (a.f.flags[cell0 + r * nxy] & 0x1F) != 0x01) live |= 1u << r;
            float acc[R][6];
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < 6; c++) acc[r][c] = 0.0f;
            const float cx = (float)((int)X * bx + x), cy = (float)((int)Y * by + y), cz = (float)((int)Z * bz + z0);
            // R cells of the column against the sources of a list
            auto sweep = [&](const Src* list, int m) {
                for (int i = 0; i < m; i++) {
                    const float4 p = list[i].p, v = list[i].v;
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
            };
            if (ml) {
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
                    for (int k = 0; k < Pz; k++) {
                        const cfloat_p mz = Mz + k * (int)a.cells[2];
#pragma unroll
                        for (int c = 0; c < GC; c++) {
                            const float w = Wb[(c * Pz + k) * ws + at];
#pragma unroll
                            for (int r = 0; r < R; r++) acc[r][c0 + c] = __builtin_fmaf(mz[r], w, acc[r][c0 + c]);
                        }
                    }
                }
                if (__any(live != 0u)) sweep(near, __builtin_amdgcn_readfirstlane((int)cnt[1]));
            } else {
                const uint32_t count = *a.f.src_count;
                for (uint32_t base = 0; base < count; base += LIST_FAR) {
                    const uint32_t m = all_sources(a, blk, base, far);
                    if (__any(live != 0u)) sweep(far, (int)m);
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++)
                if (live >> r & 1u) write_cell(a.f, cell0 + r * nxy, acc[r], jd);
        }
    }
    if (a.f.judge != nullptr) judge_block_sums(jd, a.f.judge);
}

}  // namespace

// Sample points: as many per axis as the interpolation error asks for. The
// nearest source that a block's samples hold lies 2 block sides from its
// centre along an axis, and 1.5 sides from every cell; a function that is
// singular at distance d straight ahead of (beside) an interval of half width
// h is interpolated to rho^-P with rho = r + sqrt(r^2 - 1) (r + sqrt(r^2 + 1)),
// r = d / h. The bounds below gave, against the sum at every cell in double on
// 16^3 LOD blocks, relative errors of the far field of 2e-8 on level D, 3e-8
// on D - 1 and 1e-8 on D - 2 (9, 10 and 11 points for cubic blocks), below the
// 1e-7 to 2e-7 of the float sums themselves.
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
    return true;
}

static bool plan(const FieldArgs& f, uint32_t levels, MlArgs* a) {
    *a = MlArgs{};
    a->f = f;
    a->qu = f.qu;
    a->ws = f.ml_ws;
    const uint32_t D = f.D, nd = 1u << D;
    a->nd = nd;
    for (uint32_t i = 0; i <= D; i++) a->n_lod += 1u << (3 * i);
    a->lo = a->n_lod - nd * nd * nd;
    a->zext = (a->n_lod + nd * nd - 1) / (nd * nd);
    a->b[0] = f.nx / nd;
    a->b[1] = f.ny / nd;
    a->b[2] = f.nz / nd;
    a->levels = levels;
    const uint32_t cells = a->b[0] * a->b[1] * a->b[2];
    if (levels > 0) {
        if (!grid_of(a->b, 0, nd, 5e-8, &a->fine)) return false;
        for (uint32_t l = 0; l < levels; l++)
            if (!grid_of(a->b, D - 2 - l, 4u << l, l + 1 == levels ? 1e-8 : 2e-9, &a->coarse[l])) return false;
        a->leaf = (uint32_t)a->fine.n == cells && cells <= 4 * LEAF_T;
    }
    // work split
    if (a->leaf) {
        a->threads = std::min(LEAF_T, (cells + 63) / 64 * 64);
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
    int most = 0;  // sample points of an axis
    for (int k = 0; k < 3; k++) {
        most = std::max(most, a->fine.P[k]);
        for (uint32_t l = 0; l < levels; l++) most = std::max(most, a->coarse[l].P[k]);
    }
    a->ld = most <= 12 ? 12 : ML_MAX_P;
    // workspace: header, tables, samples
    size_t at = 16;
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
    // LDS: samples, scratch (from_coarse: two half-interpolated grids; then V
    // and W), source lists; three components at a time where that leaves room
    // for two workgroups, else one
    a->rows = a->leaf ? 0 : std::min((a->colw * 64 - 1) / a->b[0] + 2, a->b[1]);
    for (uint32_t gc : {3u, 1u}) {
        if (gc == 3 && a->ld != 12) continue;
        a->gc = gc;
        size_t tmp = 0;
        for (uint32_t l = 0; l < levels; l++) {
            const MlGrid& g = a->coarse[l];
            tmp = std::max(tmp, (size_t)gc * g.P[2] * a->fine.P[0] * (g.P[1] + a->fine.P[1]));
        }
        const size_t V = a->leaf ? 0 : (size_t)gc * a->fine.P[2] * a->fine.P[1] * a->b[0];
        a->v_off = 6 * a->fine.n;
        a->w_off = (uint32_t)(a->v_off + V);
        a->list_off = (uint32_t)(a->v_off + std::max(V + (size_t)gc * a->fine.P[2] * a->rows * a->b[0], tmp) + 3) & ~3u;
        a->lds = a->list_off * 4 + (LIST_FAR + LIST_NEAR) * (uint32_t)sizeof(Src) + 16;
        if (a->lds <= ML_LDS) break;
    }
    if (a->lds > ML_LDS) return false;
    // far_points: K points a thread in pg groups, the split with the fewest idle lanes
    if (levels > 0 && !a->leaf) {
        uint32_t best = ~0u;
        for (uint32_t pg : {1u, 2u, 4u})
            for (uint32_t k : {4u, 3u, 2u}) {
                if (a->threads % (64 * pg)) continue;
                const uint32_t per = k * (a->threads / pg), slots = (a->fine.n + per - 1) / per * per * pg;
                // of equal ones, more points a thread: fewer LDS reads per interaction
                const uint32_t cost = slots / pg;
                if (cost < best) {
                    best = cost;
                    a->pg = pg;
                    a->pk = k;
                }
            }
    }
    for (uint32_t l = 0; l < levels; l++) {
        MlGrid& g = a->coarse[l];
        g.groups = g.side * g.side * g.side * (uint32_t)((g.n + COARSE_PTS - 1) / COARSE_PTS);
    }
    return true;
}

// Levels 2 .. D - 1: of depth 3 and 4. (Below depth 3 all or almost all
// sources are near; deeper trees have their near field on the cells.) Blocks
// so uneven or so large that the points do not fit take the direct sum.
bool ml_plan(const FieldArgs& f, MlArgs* a) {
    if (f.f64 || f.near || f.D > 4) return false;
    return (f.D >= 3 && plan(f, f.D - 2, a)) || plan(f, 0, a);
}

uint32_t ml_blocks(const MlArgs& a) { return a.nd * a.nd * a.nd; }

hipError_t launch_field_fast(const MlArgs& a, hipStream_t s) {
    if (a.levels > 0) {
        uint32_t g = (a.t_end - 16 + COARSE_T - 1) / COARSE_T;
        for (uint32_t l = 0; l < a.levels; l++) g += a.coarse[l].groups;
        hipLaunchKernelGGL(k_ml_coarse, dim3(g), dim3(COARSE_T), 0, s, a);
    }
    const dim3 g(ml_blocks(a)), b(a.threads);
    if (a.leaf) {
        // cells of at most 12 points an axis, coarse levels of up to 24
#define ION_LEAF(K)                                                                    \
    do {                                                                               \
        if (a.ld == 12) hipLaunchKernelGGL((k_ml_leaf<K, 12>), g, b, a.lds, s, a);     \
        else hipLaunchKernelGGL((k_ml_leaf<K, ML_MAX_P>), g, b, a.lds, s, a);          \
    } while (0)
        switch ((a.fine.n + a.threads - 1) / a.threads) {
            case 1: ION_LEAF(1); break;
            case 2: ION_LEAF(2); break;
            case 3: ION_LEAF(3); break;
            default: ION_LEAF(4); break;
        }
#undef ION_LEAF
    } else {
#define ION_CELLS(R)                                                                        \
    do {                                                                                    \
        if (a.gc == 3) hipLaunchKernelGGL((k_ml_cells<R, 12, 3>), g, b, a.lds, s, a);       \
        else if (a.ld == 12) hipLaunchKernelGGL((k_ml_cells<R, 12, 1>), g, b, a.lds, s, a); \
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
