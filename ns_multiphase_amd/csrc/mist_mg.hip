// mist_mg.hip -- variable-density pressure Poisson multigrid on gfx950.
//
// Operator (src/Pressure.jl:909-1033 scaling): (A p)_c = sum_f c_f (p_nb - p_c) with
// c_f = dt / (den_f h^2), wall faces dropped, periodic faces wrapped, b = div(u*)
// (src/Pressure.jl:16-22). V-cycle of mg_vc_lin! (src/Multigrid.jl:678-764): red-black
// Gauss-Seidel (src/Pressure.jl:1096-1133, colour (i+j+k)%2, red first, omega 1), 8-cell
// average restriction (src/Multigrid.jl:183-197), trilinear prolongation from coarse centres
// (src/Multigrid.jl:5-54). Coarse face coefficients are the mean of the fine faces covering
// them (MIST_COARSE_FACE_AVERAGE), or the reference's face densities of the liquid fraction
// restricted to the level (MIST_COARSE_RESTRICTED_VF, src/Multigrid.jl:725-737). The outer
// loop evaluates the FP64 residual in flux form and applies one V-cycle in
// precision T (double, or float for the mixed mode) to it per iteration, until
// max|b - A p| <= tol; the solution is shifted to zero mean.
//
// Storage: interior cells only (n_x n_y n_z per level, x fastest); neighbours across a wall
// have a zero coefficient and read the cell itself, so no ghost layers are needed. The levels
// relaxed by per-level launches store each x-row as its red cells then its black cells, so a
// one-colour sweep reads and writes unit-stride vectors; the coarse end (one work-group, in
// LDS) and the FP64 outer arrays use the plain order.
#include <algorithm>
#include <cmath>
#include <vector>

#include "mist_internal.h"

namespace mist {

struct LevelGeom {
    int n[3];
    int per[3];
    int coarsened[3];  // coarser than the level above along axis d
    int split;         // rows stored red half then black half (n[0] even)
    __host__ __device__ int64_t size() const { return (int64_t)n[0] * n[1] * n[2]; }
};

// storage index of cell (i, j, k); red = (i+1)+(j+1)+(k+1) even = i+j+k odd (second half)
__host__ __device__ __forceinline__ int64_t lidx(const LevelGeom& g, int i, int j, int k) {
    const int64_t row = (int64_t)g.n[0] * (j + (int64_t)g.n[1] * k);
    if (!g.split) return row + i;
    return row + (((i + j + k) & 1) ? (g.n[0] >> 1) : 0) + (i >> 1);
}

// cell (i, j, k) stored at index q
__device__ __forceinline__ void lcell(const LevelGeom& g, int64_t q, int& i, int& j, int& k) {
    const int64_t row = q / g.n[0];
    const int r = (int)(q - row * g.n[0]);
    j = (int)(row % g.n[1]);
    k = (int)(row / g.n[1]);
    if (!g.split) {
        i = r;
        return;
    }
    const int hn = g.n[0] >> 1;
    const int half = r >= hn ? 1 : 0;
    i = 2 * (r - half * hn) + ((half + j + k) & 1);
}

// A tile of a split level: SPLIT_H pairs of x-cells by SPLIT_J rows of one plane, the cells one
// work-group of k_rbgs_split relaxes. Away from the interface all open faces of a tile's cells
// have one coefficient per axis (the same bits: they come from one density); the sweeps then
// take it from this table instead of reading three coefficient arrays per cell.
constexpr int SPLIT_H = 64, SPLIT_J = 4;
template <class T>
struct UTile {
    T c[3];
    T uniform;  // 1: c holds the coefficient of every open face along each axis
};
struct SplitGrid {
    int gx, gy, nb;  // tiles along x and y, and in all
    __host__ __device__ explicit SplitGrid(const LevelGeom& g)
        : gx((g.n[0] + 2 * SPLIT_H - 1) / (2 * SPLIT_H)), gy((g.n[1] + SPLIT_J - 1) / SPLIT_J), nb(gx * gy * g.n[2]) {}
};

template <class T>
struct LevelBuf {
    T* c[3] = {nullptr, nullptr, nullptr};
    T* e = nullptr;
    T* b = nullptr;
    T* r = nullptr;
    UTile<T>* ut = nullptr;  // split levels: coefficients of the uniform tiles
};

struct MGState {
    std::vector<LevelGeom> g;         // plain order (the FP64 outer arrays use g[0])
    std::vector<LevelGeom> gq[2];     // storage of the FP64 and FP32 hierarchies
    std::vector<LevelBuf<double>> d;  // FP64 hierarchy
    std::vector<LevelBuf<float>> s;   // FP32 hierarchy
    double* c64[3] = {nullptr, nullptr, nullptr};  // fine FP64 operator
    UTile<double>* ut64 = nullptr;                 // its tile table
    double* p64 = nullptr;
    double* b64 = nullptr;
    std::vector<double*> vfl;  // restricted liquid fraction per level (plain order; 1..)
    double dt = 0.0;           // of the solve being set up
    double* part = nullptr;
    double* h_part = nullptr;  // pinned
    int nblocks = 0;
    int64_t nfine = 0;
    int first_small[2] = {0, 0};              // first level solved in one block (FP64, FP32)
    size_t small_lds[2] = {0, 0};             // its LDS bytes
    void* small_desc[2] = {nullptr, nullptr};  // SmallLevels<T> in device memory
    bool small_odd[2] = {false, false};        // its cells need k_small_vcycle's numbering for odd rows
    hipGraph_t graph[2] = {nullptr, nullptr};  // one defect-correction iteration
    hipGraphExec_t exec[2] = {nullptr, nullptr};
    std::vector<void*> allocs;
};

void mg_free(MGState* s) {
    if (!s) return;
    for (int q = 0; q < 2; ++q) {
        if (s->exec[q]) (void)hipGraphExecDestroy(s->exec[q]);
        if (s->graph[q]) (void)hipGraphDestroy(s->graph[q]);
    }
    for (void* p : s->allocs) (void)hipFree(p);
    if (s->h_part) (void)hipHostFree(s->h_part);
    delete s;
}

// ---- kernels ---------------------------------------------------------------------------
// Neighbours (storage indices) and face coefficients of cell (i, j, k): faces x-, x+, y-, y+,
// z-, z+; C[d][c] is the face between c and its lower neighbour along d. A neighbour across a
// wall is the cell itself with coefficient 0; across a periodic side, the wrapped cell.
template <class T, bool MAY_SPLIT = true>
__device__ __forceinline__ void stencil(const LevelGeom& g, T* const* C, int i, int j, int k, int64_t cell, int64_t nb[6],
                                       T cf[6]) {
    auto lidx = [&](int a, int b, int c) -> int64_t {
        if constexpr (MAY_SPLIT) return ::mist::lidx(g, a, b, c);
        return a + (int64_t)g.n[0] * (b + (int64_t)g.n[1] * c);
    };
    const int q[3] = {i, j, k};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int nd = g.n[d];
        int up[3] = {i, j, k}, dn[3] = {i, j, k};
        // every load is issued whether the face is open or not (a closed one reads the cell
        // itself): a load under a branch would make the wave wait for it before the next one
        const bool ou = q[d] + 1 < nd || g.per[d], od = q[d] > 0 || g.per[d];
        up[d] = ou ? (q[d] + 1 < nd ? q[d] + 1 : 0) : q[d];
        dn[d] = od ? (q[d] > 0 ? q[d] - 1 : nd - 1) : q[d];
        nb[2 * d + 1] = lidx(up[0], up[1], up[2]);
        nb[2 * d] = lidx(dn[0], dn[1], dn[2]);
        const T cu = C[d][nb[2 * d + 1]];
        cf[2 * d] = C[d][cell];
        cf[2 * d + 1] = ou ? cu : T(0);
    }
}

// One colour of a red-black Gauss-Seidel sweep (rbgs_update!, src/Pressure.jl:1096-1133)
template <class T>
__global__ void k_rbgs(LevelGeom g, T* cx, T* cy, T* cz, T* e, const T* b, int color) {
    T* C[3] = {cx, cy, cz};
    const int hx = (g.n[0] + 1) / 2;
    const int64_t tot = (int64_t)hx * g.n[1] * g.n[2];
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
        const int h = (int)(q % hx);
        const int64_t row = q / hx;
        const int j = (int)(row % g.n[1]);
        const int k = (int)(row / g.n[1]);
        const int i = 2 * h + ((color + 1 + j + k) & 1);  // ((i+1)+(j+1)+(k+1)) % 2 == color
        if (i >= g.n[0]) continue;
        const int64_t cell = lidx(g, i, j, k);
        int64_t nb[6];
        T cf[6];
        stencil(g, C, i, j, k, cell, nb, cf);
        const T S = ((((cf[0] + cf[1]) + cf[2]) + cf[3]) + cf[4]) + cf[5];
        if (!(S > T(0))) continue;
        const T sum = ((((cf[0] * e[nb[0]] + cf[1] * e[nb[1]]) + cf[2] * e[nb[2]]) + cf[3] * e[nb[3]]) +
                       cf[4] * e[nb[4]]) + cf[5] * e[nb[5]];
        e[cell] = (sum - b[cell]) / S;
    }
}

// Work-group `bid` of `nb` takes logical tile xcd_tile(bid, nb): the dispatcher hands consecutive
// work-groups to the 8 XCDs in turn, so each XCD gets one contiguous run of tiles and the rows
// and planes shared by neighbouring tiles meet in one L2.
__device__ __forceinline__ int xcd_tile(int bid, int nb) {
    const int per = nb >> 3, rem = nb & 7, x = bid & 7;
    return x * per + min(x, rem) + (bid >> 3);
}

// Neighbours (storage index) of the cell of `color` at position h of row (j, k) of a split level,
// i = 2h + p: its x-neighbours sit at h-1+p and h+p of the other half of the same row, its y- and
// z-neighbours at h of the other half of the adjacent rows, so every load and the store are
// unit-stride across the wave; no index divisions. A closed (wall) face has the cell itself.
struct SplitCell {
    int cell, nxm, nxp, nym, nyp, nzm, nzp;  // a level holds fewer than 2^30 cells
    bool oxm, oxp, oym, oyp, ozm, ozp;
    __device__ __forceinline__ SplitCell(const LevelGeom& g, int h, int j, int k, int color) {
        const int hn = g.n[0] >> 1;
        const int p = (color + 1 + j + k) & 1;
        const int i = 2 * h + p;
        const int sy = g.n[0], sz = g.n[0] * g.n[1];
        const int row = sy * j + sz * k;
        const int own_off = color == 0 ? hn : 0;
        cell = row + own_off + h;
        const int oth = row + (hn - own_off);
        nxm = nxp = nym = nyp = nzm = nzp = cell;
        oxm = oxp = oym = oyp = ozm = ozp = true;
        if (i > 0) nxm = oth + h - 1 + p; else if (g.per[0]) nxm = oth + hn - 1; else oxm = false;
        if (i < g.n[0] - 1) nxp = oth + h + p; else if (g.per[0]) nxp = oth; else oxp = false;
        if (j > 0) nym = oth - sy + h; else if (g.per[1]) nym = oth + sy * (g.n[1] - 1) + h; else oym = false;
        if (j < g.n[1] - 1) nyp = oth + sy + h; else if (g.per[1]) nyp = oth - sy * (g.n[1] - 1) + h; else oyp = false;
        if (k > 0) nzm = oth - sz + h; else if (g.per[2]) nzm = oth + sz * (g.n[2] - 1) + h; else ozm = false;
        if (k < g.n[2] - 1) nzp = oth + sz + h; else if (g.per[2]) nzp = oth - sz * (g.n[2] - 1) + h; else ozp = false;
    }
};

// The six face coefficients of a cell, from its tile's table entry or from the arrays.
template <class T>
__device__ __forceinline__ void split_coefs(const SplitCell& s, const UTile<T>& u, const T* __restrict__ cx,
                                            const T* __restrict__ cy, const T* __restrict__ cz, T (&c)[6]) {
    if (u.uniform != T(0)) {
        c[0] = s.oxm ? u.c[0] : T(0); c[1] = s.oxp ? u.c[0] : T(0);
        c[2] = s.oym ? u.c[1] : T(0); c[3] = s.oyp ? u.c[1] : T(0);
        c[4] = s.ozm ? u.c[2] : T(0); c[5] = s.ozp ? u.c[2] : T(0);
    } else {
        const T x = cx[s.nxp], y = cy[s.nyp], z = cz[s.nzp];  // a closed face reads the cell itself
        c[0] = cx[s.cell]; c[1] = s.oxp ? x : T(0);
        c[2] = cy[s.cell]; c[3] = s.oyp ? y : T(0);
        c[4] = cz[s.cell]; c[5] = s.ozp ? z : T(0);
    }
}

// One colour of a sweep on a split level: a work-group relaxes SPLIT_K tiles stacked in z, each
// thread one cell of each, their loads all issued before the first store (the reads are of the
// other colour). PASS 1, the first colour pass of a V-cycle's pre-smoothing, takes e as zero, so
// that it is neither read nor cleared beforehand; PASS 2, the pass after it, reads what that wrote; both set
// cells without an open face, which no pass relaxes, to zero. PASS 0 are the others. Bound by memory: a colour pass reads the
// other colour's e and its own b and writes its own e, and in a tile that the interface crosses
// the three coefficient arrays too (1.5 against 4.5 values per cell of the level). Per colour, with
// the interface across the level: 256^3 FP32 60 -> 26 us, 128^3 FP64 13 -> 9.5 us (one plane per
// thread and always the arrays before).
template <class T, int SPLIT_K, int PASS>
__global__ __launch_bounds__(256) void k_rbgs_split(LevelGeom g, const T* __restrict__ cx, const T* __restrict__ cy,
                                                    const T* __restrict__ cz, const UTile<T>* __restrict__ ut, T* e,
                                                    const T* __restrict__ b, int color) {
    const SplitGrid G(g);
    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int bx = t % G.gx, by = (t / G.gx) % G.gy, k0 = (t / (G.gx * G.gy)) * SPLIT_K;
    const int h = bx * SPLIT_H + threadIdx.x;
    const int j = by * SPLIT_J + __builtin_amdgcn_readfirstlane(threadIdx.y);  // a wave is one row
    const int hn = g.n[0] >> 1, sy = g.n[0], sz = g.n[0] * g.n[1];
    if (h >= hn || j >= g.n[1]) return;
    // The other colour's values sit at the own position h of the row and of the four adjacent rows
    // and at one more position of the row (SplitCell); the value of plane k +- 1 is also the
    // x-neighbour there, so a stack of planes needs (SPLIT_K + 2) + 3 SPLIT_K of them. A closed
    // face reads a value next to it, which its zero coefficient removes.
    const T* O = e + (color == 0 ? 0 : hn);
    T* own = e + (color == 0 ? hn : 0);
    const T* bo = b + (color == 0 ? hn : 0);
    const int jm = j > 0 ? j - 1 : (g.per[1] ? g.n[1] - 1 : j), jp = j + 1 < g.n[1] ? j + 1 : (g.per[1] ? 0 : j);
    T zc[SPLIT_K + 2], xo[SPLIT_K], ym[SPLIT_K], yp[SPLIT_K], vb[SPLIT_K];
#pragma unroll
    for (int z = 0; z < SPLIT_K; ++z) {
        const int k = min(k0 + z, g.n[2] - 1);
        vb[z] = bo[sy * j + sz * k + h];
        if constexpr (PASS != 1) {
            const int p = (color + 1 + j + k) & 1;
            int hx = p ? h + 1 : h - 1;
            if (hx < 0) hx = g.per[0] ? hn - 1 : h;
            if (hx >= hn) hx = g.per[0] ? 0 : h;
            xo[z] = O[sy * j + sz * k + hx];
            ym[z] = O[sy * jm + sz * k + h];
            yp[z] = O[sy * jp + sz * k + h];
        }
    }
    if constexpr (PASS != 1) {
#pragma unroll
        for (int z = -1; z <= SPLIT_K; ++z) {
            int k = k0 + z;
            if (k < 0) k = g.per[2] ? g.n[2] - 1 : 0;
            if (k >= g.n[2]) k = k == g.n[2] && g.per[2] ? 0 : g.n[2] - 1;
            zc[z + 1] = O[sy * j + sz * k + h];
        }
    }
    T v[SPLIT_K];
    bool on[SPLIT_K];
#pragma unroll
    for (int z = 0; z < SPLIT_K; ++z) {
        const int k = min(k0 + z, g.n[2] - 1);
        const UTile<T> u = ut[bx + G.gx * (by + G.gy * k)];
        T c[6];
        const int p = (color + 1 + j + k) & 1;
        if (u.uniform != T(0)) {
            const int i = 2 * h + p;
            c[0] = i > 0 || g.per[0] ? u.c[0] : T(0); c[1] = i < g.n[0] - 1 || g.per[0] ? u.c[0] : T(0);
            c[2] = j > 0 || g.per[1] ? u.c[1] : T(0); c[3] = j < g.n[1] - 1 || g.per[1] ? u.c[1] : T(0);
            c[4] = k > 0 || g.per[2] ? u.c[2] : T(0); c[5] = k < g.n[2] - 1 || g.per[2] ? u.c[2] : T(0);
        } else {
            split_coefs(SplitCell(g, h, j, k, color), u, cx, cy, cz, c);
        }
        const T S = ((((c[0] + c[1]) + c[2]) + c[3]) + c[4]) + c[5];
        T sum = T(0);
        if constexpr (PASS != 1) {
            const T xm = p ? zc[z + 1] : xo[z], xp = p ? xo[z] : zc[z + 1];
            sum = ((((c[0] * xm + c[1] * xp) + c[2] * ym[z]) + c[3] * yp[z]) + c[4] * zc[z]) + c[5] * zc[z + 2];
        }
        on[z] = S > T(0);
        v[z] = (sum - vb[z]) / S;
        if constexpr (PASS != 0) {
            if (!on[z]) v[z] = T(0);
            on[z] = true;
        }
    }
#pragma unroll
    for (int z = 0; z < SPLIT_K; ++z)
        if (on[z] && k0 + z < g.n[2]) own[sy * j + sz * (k0 + z) + h] = v[z];
}

// K red-black sweeps of a split level in one launch, for the levels that are small enough for a
// launch per colour to be mostly latency (a colour pass takes 4-5 us on any level below 64^3). A work-group holds e of its output tile of BX x BY x BZ
// cells and a halo of 2K cells in LDS, each colour pass is valid one cell further inside, and
// after the 2K passes the tile is final: the iterates are those of the colour passes over the
// whole level, bit for bit. Work-groups read each other's tiles of `ein`, so the result goes to
// another array. A thread owns the same pairs of x-neighbours in every pass and keeps their
// coefficients and b in registers. Bound by latency and, above 64^3, by the halo's extra loads and
// relaxations (6 times the output cells). Two sweeps of 64^3 take 14 us in FP64 and 10 in FP32
// against 18 with a launch per colour, of 32^3 8 and 6.5 against 17; of 80x48x112 in FP64 26
// against 19. FIRST: ein counts as zero and is not read. Needs even extents
// along periodic axes (the wrapped halo keeps the colours).
template <int K_, int BH_, int BY_, int BZ_>
struct LdsTile {
    static constexpr int K = K_, NT = 512, HALO = 2 * K_;
    static constexpr int BH = BH_, BY = BY_, BZ = BZ_;  // output: BH pairs of x-cells by BY by BZ
    static constexpr int EH = BH + HALO, EY = BY + 2 * HALO, EZ = BZ + 2 * HALO;
    static constexpr int N = EH * EY * EZ, S = (N + NT - 1) / NT;
};
__device__ __forceinline__ bool wrap_into(int& c, int n, int per) {
    if (c >= 0 && c < n) return true;
    if (!per) return false;
    c %= n;
    if (c < 0) c += n;
    return true;
}

template <class T, class C, bool FIRST>
__global__ __launch_bounds__(C::NT) void k_rbgs_lds(LevelGeom g, int tx, int ty, const T* __restrict__ cx,
                                                    const T* __restrict__ cy, const T* __restrict__ cz,
                                                    const UTile<T>* __restrict__ ut, const T* __restrict__ ein,
                                                    T* __restrict__ eout, const T* __restrict__ b) {
    constexpr int K = C::K, SY = C::EH, SZ = C::EH * C::EY;
    __shared__ T p[2][C::N];  // [colour: 0 red, 1 black][pair]
    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int h0 = (t % tx) * C::BH - C::HALO / 2, j0 = ((t / tx) % ty) * C::BY - C::HALO,
              k0 = (t / (tx * ty)) * C::BZ - C::HALO;
    const int hn = g.n[0] >> 1, sy = g.n[0], sz = g.n[0] * g.n[1];
    // whether one coefficient per axis serves every cell of the block: the table entries of the
    // level's tiles that the halo box meets are uniform and equal
    // (a periodic box may meet a cut-off last tile between the positions looked at)
    const SplitGrid G(g);
    bool same = !(g.per[0] && hn % SPLIT_H) && !(g.per[1] && g.n[1] % SPLIT_J);
    UTile<T> u;
    {
        // tile positions along x and rows of tiles along y that the box can meet, planes along z
        constexpr int TX = (C::EH + SPLIT_H - 2) / SPLIT_H + 1, TY = (C::EY + SPLIT_J - 2) / SPLIT_J + 1;
        constexpr int NE = TX * TY * C::EZ;
        u = ut[(min(max(h0, 0), hn - 1) / SPLIT_H) + G.gx * ((min(max(j0, 0), g.n[1] - 1) / SPLIT_J) + G.gy * min(max(k0, 0), g.n[2] - 1))];
        for (int q = threadIdx.x; q < NE; q += C::NT) {
            // along an axis the box meets the tiles of its positions 0, STEP, 2 STEP, .. and its last
            int h = h0 + min((q % TX) * SPLIT_H, C::EH - 1), j = j0 + min(((q / TX) % TY) * SPLIT_J, C::EY - 1),
                k = k0 + q / (TX * TY);
            // each axis by itself: a box wider than the level has all its positions along one axis
            // beyond walls, and still meets the tiles across another axis' periodic side
            if (!wrap_into(h, hn, g.per[0])) h = min(max(h, 0), hn - 1);
            if (!wrap_into(j, g.n[1], g.per[1])) j = min(max(j, 0), g.n[1] - 1);
            if (!wrap_into(k, g.n[2], g.per[2])) k = min(max(k, 0), g.n[2] - 1);
            const UTile<T> w = ut[h / SPLIT_H + G.gx * (j / SPLIT_J + G.gy * k)];
            same = same && w.uniform != T(0) && w.c[0] == u.c[0] && w.c[1] == u.c[1] && w.c[2] == u.c[2];
        }
    }
    T cf[C::S][2][6], S[C::S][2], bb[C::S][2], ev[C::S][2];
    int off[C::S];       // offset of the red cell in its pair
    int depth[C::S][2];  // distance of the cell to the halo's rim: passes it can take part in (0: none)
    int store[C::S];     // storage row + h of an output pair, -1 elsewhere
    // every load is issued before any is used; positions outside the level read the nearest cell
#pragma unroll
    for (int s = 0; s < C::S; ++s) {
        const int q = min((int)threadIdx.x + s * C::NT, C::N - 1);
        const int eh = q % C::EH, ey = (q / C::EH) % C::EY, ez = q / SZ;
        int h = h0 + eh, j = j0 + ey, k = k0 + ez;
        const bool in = wrap_into(h, hn, g.per[0]) && wrap_into(j, g.n[1], g.per[1]) && wrap_into(k, g.n[2], g.per[2]);
        const bool mine = (int)threadIdx.x + s * C::NT < C::N && in;
        h = min(max(h, 0), hn - 1);
        j = min(max(j, 0), g.n[1] - 1);
        k = min(max(k, 0), g.n[2] - 1);
        const int row = sy * j + sz * k + h;
        if constexpr (!FIRST) {
            ev[s][0] = ein[row + hn];
            ev[s][1] = ein[row];
            if (!in) ev[s][0] = ev[s][1] = T(0);
        }
        off[s] = (1 + j + k) & 1;
        const int dyz = min(min(ey, C::EY - 1 - ey), min(ez, C::EZ - 1 - ez));
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int ex = 2 * eh + (c == 0 ? off[s] : 1 - off[s]);
            depth[s][c] = mine ? min(dyz, min(ex, 2 * C::EH - 1 - ex)) : 0;
            bb[s][c] = b[row + (c == 0 ? hn : 0)];
        }
        store[s] = mine && eh >= C::HALO / 2 && eh < C::HALO / 2 + C::BH && ey >= C::HALO && ey < C::HALO + C::BY &&
                           ez >= C::HALO && ez < C::HALO + C::BZ
                       ? row
                       : -1;
    }
    same = __syncthreads_and(same);
#pragma unroll
    for (int s = 0; s < C::S; ++s) {
        const int q = min((int)threadIdx.x + s * C::NT, C::N - 1);
        int h = h0 + q % C::EH, j = j0 + (q / C::EH) % C::EY, k = k0 + q / SZ;
        (void)(wrap_into(h, hn, g.per[0]) && wrap_into(j, g.n[1], g.per[1]) && wrap_into(k, g.n[2], g.per[2]));
        h = min(max(h, 0), hn - 1);
        j = min(max(j, 0), g.n[1] - 1);
        k = min(max(k, 0), g.n[2] - 1);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const SplitCell sc(g, h, j, k, c);
            T* F = cf[s][c];
            if (same) {
                F[0] = sc.oxm ? u.c[0] : T(0); F[1] = sc.oxp ? u.c[0] : T(0);
                F[2] = sc.oym ? u.c[1] : T(0); F[3] = sc.oyp ? u.c[1] : T(0);
                F[4] = sc.ozm ? u.c[2] : T(0); F[5] = sc.ozp ? u.c[2] : T(0);
            } else {
                F[0] = cx[sc.cell]; F[1] = cx[sc.nxp];
                F[2] = cy[sc.cell]; F[3] = cy[sc.nyp];
                F[4] = cz[sc.cell]; F[5] = cz[sc.nzp];
                if (!sc.oxp) F[1] = T(0);
                if (!sc.oyp) F[3] = T(0);
                if (!sc.ozp) F[5] = T(0);
            }
        }
    }
#pragma unroll
    for (int s = 0; s < C::S; ++s) {
        const int q = threadIdx.x + s * C::NT;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const T* F = cf[s][c];
            S[s][c] = ((((F[0] + F[1]) + F[2]) + F[3]) + F[4]) + F[5];
            if (!(S[s][c] > T(0))) depth[s][c] = 0;
            if (q < C::N) p[c][q] = FIRST ? T(0) : ev[s][c];
        }
    }
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < 2 * K; ++pass) {
        constexpr int RED = 0;
        const int c = pass & 1;
        const T* o = p[c == RED ? 1 : 0];  // the other colour
#pragma unroll
        for (int s = 0; s < C::S; ++s) {
            if (depth[s][c] <= pass) continue;
            const int q = threadIdx.x + s * C::NT;  // < C::N: a position past the tile has depth 0
            const int x = q + (c == RED ? off[s] : 1 - off[s]);
            const T* F = cf[s][c];
            const T sum = ((((F[0] * o[x - 1] + F[1] * o[x]) + F[2] * o[q - SY]) + F[3] * o[q + SY]) +
                           F[4] * o[q - SZ]) + F[5] * o[q + SZ];
            p[c][q] = (sum - bb[s][c]) / S[s][c];
        }
        __syncthreads();
    }
#pragma unroll
    for (int s = 0; s < C::S; ++s)
        if (store[s] >= 0) {
            const int q = threadIdx.x + s * C::NT;
            eout[store[s] + hn] = p[0][q];
            eout[store[s]] = p[1][q];
        }
}

// The right-hand side of a split level's coarser level in one launch: the residual of the eight
// fine cells of each coarse cell (k_resid's arithmetic), averaged as k_restrict does (256^3 FP32:
// 108 -> 61 us for the two launches before, which stored the residual). One thread
// per coarse cell, its fine cells the pairs at h = I of four rows, so the loads are unit-stride.
template <class T>
__global__ __launch_bounds__(256) void k_resid_restrict(LevelGeom g, LevelGeom gc, const T* __restrict__ cx,
                                                        const T* __restrict__ cy, const T* __restrict__ cz,
                                                        const UTile<T>* __restrict__ ut, const T* __restrict__ e,
                                                        const T* __restrict__ b, T* __restrict__ bc) {
    const SplitGrid G(g);
    const int cgy = (gc.n[1] + SPLIT_J - 1) / SPLIT_J;
    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int I = (t % G.gx) * SPLIT_H + threadIdx.x;
    const int J = ((t / G.gx) % cgy) * SPLIT_J + __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int K = t / (G.gx * cgy);
    if (I >= gc.n[0] || J >= gc.n[1]) return;
    T sum = T(0);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int bb = 0; bb < 2; ++bb) {
            const int j = 2 * J + bb, k = 2 * K + c;
            const UTile<T> u = ut[(t % G.gx) + G.gx * ((j / SPLIT_J) + G.gy * k)];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int color = (1 + a + j + k) & 1;  // of cell i = 2 I + a (0: i + j + k odd)
                const SplitCell s(g, I, j, k, color);
                T f[6];
                split_coefs(s, u, cx, cy, cz, f);
                const T pc = e[s.cell];
                const T xm = s.oxm ? e[s.nxm] : pc, xp = s.oxp ? e[s.nxp] : pc;
                const T ym = s.oym ? e[s.nym] : pc, yp = s.oyp ? e[s.nyp] : pc;
                const T zm = s.ozm ? e[s.nzm] : pc, zp = s.ozp ? e[s.nzp] : pc;
                const T Ap = ((((f[0] * (xm - pc) + f[1] * (xp - pc)) + f[2] * (ym - pc)) + f[3] * (yp - pc)) +
                              f[4] * (zm - pc)) + f[5] * (zp - pc);
                sum += b[s.cell] - Ap;
            }
        }
    bc[lidx(gc, I, J, K)] = sum * (T(1) / T(8));
}

// k_prolong_add onto a split level, one thread per pair of x-cells: the two cells share their
// coarse rows, so twelve coarse values serve both (256^3 FP32: 82 -> 53 us).
template <class T>
__global__ __launch_bounds__(256) void k_prolong_split(LevelGeom gc, LevelGeom g, const T* __restrict__ ec, T* ef) {
    const SplitGrid G(g);
    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int h = (t % G.gx) * SPLIT_H + threadIdx.x;
    const int j = ((t / G.gx) % G.gy) * SPLIT_J + __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int k = t / (G.gx * G.gy);
    const int hn = g.n[0] >> 1;
    if (h >= hn || j >= g.n[1]) return;
    // coarse cells below and above a fine cell along an axis, and their weights
    auto pick = [&](int q, int n, int per, int& lo, int& hi, T& w1, T& w2) {
        const int Q = q / 2;
        if ((q & 1) == 0) { lo = Q - 1; hi = Q; w1 = T(0.75); w2 = T(0.25); }
        else { lo = Q; hi = Q + 1; w1 = T(0.25); w2 = T(0.75); }
        if (lo < 0) lo = per ? n - 1 : 0;
        if (hi >= n) hi = per ? 0 : n - 1;
    };
    int jl, jh, kl, kh;
    T wy1, wy2, wz1, wz2;
    pick(j, gc.n[1], gc.per[1], jl, jh, wy1, wy2);
    pick(k, gc.n[2], gc.per[2], kl, kh, wz1, wz2);
    const int im = h > 0 ? h - 1 : (gc.per[0] ? gc.n[0] - 1 : 0), ip = h + 1 < gc.n[0] ? h + 1 : (gc.per[0] ? 0 : gc.n[0] - 1);
    T E[3][2][2];  // [h-1, h, h+1][lo, hi of y][lo, hi of z]
#pragma unroll
    for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            const int J = y ? jh : jl, K = z ? kh : kl;
            E[0][y][z] = ec[lidx(gc, im, J, K)];
            E[1][y][z] = ec[lidx(gc, h, J, K)];
            E[2][y][z] = ec[lidx(gc, ip, J, K)];
        }
    const int row = g.n[0] * (j + g.n[1] * k);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const T w1 = a ? T(0.25) : T(0.75), w2 = a ? T(0.75) : T(0.25);  // of the upper and lower coarse cell
        const T v = wz1 * (wy1 * (w1 * E[a + 1][1][1] + w2 * E[a][1][1]) + wy2 * (w1 * E[a + 1][0][1] + w2 * E[a][0][1])) +
                    wz2 * (wy1 * (w1 * E[a + 1][1][0] + w2 * E[a][1][0]) + wy2 * (w1 * E[a + 1][0][0] + w2 * E[a][0][0]));
        const int q = row + (((a + j + k) & 1) ? hn : 0) + h;
        ef[q] += v;
    }
}

// The tile table of a level from its coefficients (in the level's storage): one work-group per
// tile, the smallest and largest coefficient of the open faces of the tile's cells along each axis.
template <class T>
__global__ __launch_bounds__(256) void k_uniform_tiles(LevelGeom g, const T* cx, const T* cy, const T* cz, UTile<T>* ut) {
    __shared__ T s_mn[4][3], s_mx[4][3];
    __shared__ int s_bad;
    const SplitGrid G(g);
    const int t = blockIdx.x;
    const int j = ((t / G.gx) % G.gy) * SPLIT_J + threadIdx.y;
    const int k = t / (G.gx * G.gy);
    const int tid = threadIdx.x + SPLIT_H * threadIdx.y;
    const T big = T(3e38);
    T mn[3] = {big, big, big}, mx[3] = {-big, -big, -big};
    bool bad = false;
    if (tid == 0) s_bad = 0;
    __syncthreads();
    for (int a = 0; a < 2; ++a) {
        const int i = 2 * ((t % G.gx) * SPLIT_H + (int)threadIdx.x) + a;
        if (i >= g.n[0] || j >= g.n[1]) continue;
        const T* C[3] = {cx, cy, cz};
        const int q[3] = {i, j, k};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            auto take = [&](T v) {
                bad = bad || !(v > -big && v < big);
                mn[d] = v < mn[d] ? v : mn[d];
                mx[d] = v > mx[d] ? v : mx[d];
            };
            int up[3] = {i, j, k};
            if (q[d] > 0 || g.per[d]) take(C[d][lidx(g, i, j, k)]);
            if (q[d] + 1 < g.n[d] || g.per[d]) {
                up[d] = q[d] + 1 < g.n[d] ? q[d] + 1 : 0;
                take(C[d][lidx(g, up[0], up[1], up[2])]);
            }
        }
    }
    if (bad) atomicOr(&s_bad, 1);
    for (int a = 0; a < 3; ++a)
        for (int o = 32; o >= 1; o >>= 1) {
            const T m = __shfl_xor(mn[a], o), M = __shfl_xor(mx[a], o);
            mn[a] = m < mn[a] ? m : mn[a];
            mx[a] = M > mx[a] ? M : mx[a];
        }
    if ((tid & 63) == 0)
        for (int a = 0; a < 3; ++a) {
            s_mn[tid >> 6][a] = mn[a];
            s_mx[tid >> 6][a] = mx[a];
        }
    __syncthreads();
    if (tid == 0) {
        UTile<T> u;
        u.uniform = s_bad ? T(0) : T(1);
        for (int a = 0; a < 3; ++a) {
            T m = s_mn[0][a], M = s_mx[0][a];
            for (int w = 1; w < 4; ++w) {
                m = s_mn[w][a] < m ? s_mn[w][a] : m;
                M = s_mx[w][a] > M ? s_mx[w][a] : M;
            }
            if (m < M) u.uniform = T(0);
            u.c[a] = m <= M ? m : T(0);  // no open face along the axis: never used
        }
        ut[t] = u;
    }
}

template <class T>
__global__ void k_resid(LevelGeom g, T* cx, T* cy, T* cz, const T* e, const T* b, T* r) {
    T* C[3] = {cx, cy, cz};
    const int64_t tot = g.size();
    for (int64_t cell = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; cell < tot;
         cell += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        lcell(g, cell, i, j, k);
        int64_t nb[6];
        T cf[6];
        stencil(g, C, i, j, k, cell, nb, cf);
        const T pc = e[cell];
        const T Ap = ((((cf[0] * (e[nb[0]] - pc) + cf[1] * (e[nb[1]] - pc)) + cf[2] * (e[nb[2]] - pc)) +
                       cf[3] * (e[nb[3]] - pc)) + cf[4] * (e[nb[4]] - pc)) + cf[5] * (e[nb[5]] - pc);
        r[cell] = b[cell] - Ap;
    }
}

template <class T>
__global__ void k_restrict(LevelGeom F, LevelGeom C, const T* rf, T* bc) {
    const int f0 = C.coarsened[0] ? 2 : 1, f1 = C.coarsened[1] ? 2 : 1, f2 = C.coarsened[2] ? 2 : 1;
    const T inv = T(1) / T(f0 * f1 * f2);
    const int64_t tot = C.size();
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
        int I, J, K;
        lcell(C, q, I, J, K);
        T s = T(0);
        for (int c = 0; c < f2; ++c)
            for (int b = 0; b < f1; ++b)
                for (int a = 0; a < f0; ++a) s += rf[lidx(F, I * f0 + a, J * f1 + b, K * f2 + c)];
        bc[q] = s * inv;
    }
}

template <class T>
__global__ void k_prolong_add(LevelGeom C, LevelGeom F, const T* ec, T* ef) {
    const int64_t tot = F.size();
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
        int qq[3];
        lcell(F, q, qq[0], qq[1], qq[2]);
        int lo[3], hi[3];
        T w1[3], w2[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (!C.coarsened[d]) { lo[d] = hi[d] = qq[d]; w1[d] = T(1); w2[d] = T(0); continue; }
            const int Q = qq[d] / 2;
            if ((qq[d] & 1) == 0) { lo[d] = Q - 1; hi[d] = Q; w1[d] = T(0.75); w2[d] = T(0.25); }
            else { lo[d] = Q; hi[d] = Q + 1; w1[d] = T(0.25); w2[d] = T(0.75); }
            if (lo[d] < 0) lo[d] = C.per[d] ? C.n[d] - 1 : 0;
            if (hi[d] >= C.n[d]) hi[d] = C.per[d] ? 0 : C.n[d] - 1;
        }
        auto E = [&](int a, int b, int c) { return ec[lidx(C, a, b, c)]; };
        const T v = w1[2] * (w1[1] * (w1[0] * E(hi[0], hi[1], hi[2]) + w2[0] * E(lo[0], hi[1], hi[2])) +
                             w2[1] * (w1[0] * E(hi[0], lo[1], hi[2]) + w2[0] * E(lo[0], lo[1], hi[2]))) +
                    w2[2] * (w1[1] * (w1[0] * E(hi[0], hi[1], lo[2]) + w2[0] * E(lo[0], hi[1], lo[2])) +
                             w2[1] * (w1[0] * E(hi[0], lo[1], lo[2]) + w2[0] * E(lo[0], lo[1], lo[2])));
        ef[q] += v;
    }
}

template <class T>
__global__ void k_coarsen_coef(LevelGeom F, LevelGeom C, int d, const T* cf, T* cc) {
    const int f[3] = {C.coarsened[0] ? 2 : 1, C.coarsened[1] ? 2 : 1, C.coarsened[2] ? 2 : 1};
    const int d1 = (d + 1) % 3, d2 = (d + 2) % 3;
    const T scale = T(1) / T(f[d] * f[d]) / T(f[d1] * f[d2]);
    const int64_t tot = C.size();
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
        int Q[3];
        lcell(C, q, Q[0], Q[1], Q[2]);
        T s = T(0);
        for (int b = 0; b < f[d2]; ++b)
            for (int a = 0; a < f[d1]; ++a) {
                int x[3];
                x[d] = Q[d] * f[d];
                x[d1] = Q[d1] * f[d1] + a;
                x[d2] = Q[d2] * f[d2] + b;
                s += cf[lidx(F, x[0], x[1], x[2])];
            }
        cc[q] = s * scale;
    }
}

// The liquid fraction of level C (plain order): the mean of the finer level's over each coarse
// cell, summed in i, then j, then k order and scaled by 1/8 (restrict!,
// src/Multigrid.jl:183-197). From the context's VF (interior cells) when `src` is null.
__global__ void k_restrict_vf(DevMesh m, LevelGeom F, LevelGeom C, const double* vf_field, const double* src,
                              double* dst) {
    const int f0 = C.coarsened[0] ? 2 : 1, f1 = C.coarsened[1] ? 2 : 1, f2 = C.coarsened[2] ? 2 : 1;
    const double inv = 1.0 / (double)(f0 * f1 * f2);
    const int64_t tot = C.size();
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
        const int I = (int)(q % C.n[0]);
        const int J = (int)((q / C.n[0]) % C.n[1]);
        const int K = (int)(q / ((int64_t)C.n[0] * C.n[1]));
        double s = 0.0;
        for (int c = 0; c < f2; ++c)
            for (int b = 0; b < f1; ++b)
                for (int a = 0; a < f0; ++a) {
                    const int i = I * f0 + a, j = J * f1 + b, k = K * f2 + c;
                    s += src ? src[i + (int64_t)F.n[0] * (j + (int64_t)F.n[1] * k)]
                             : vf_field[m.vof(i + 1, j + 1, k + 1)];
                }
        dst[q] = s * inv;
    }
}

// Face coefficients of level C along d from its liquid fraction vf (plain order), in the
// level's storage: compute_dens! (src/Tools.jl:1212-1232) gives the face density
// rho_liq v + rho_gas (1 - v), v = clamp((vf_c + vf_{c-1}) / 2, 0, 1), and the coefficient is
// dt / (den h^2) as on the fine level; wall faces 0, periodic faces wrapped.
template <class T>
__global__ void k_coef_from_vf(LevelGeom C, int d, double dt, double rl, double rg, double h2, const double* vf,
                               T* c) {
    const int64_t tot = C.size();
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
        int Q[3];
        lcell(C, q, Q[0], Q[1], Q[2]);
        int lo[3] = {Q[0], Q[1], Q[2]};
        bool wall = false;
        if (Q[d] > 0) lo[d] = Q[d] - 1;
        else if (C.per[d]) lo[d] = C.n[d] - 1;
        else wall = true;
        if (wall) {
            c[q] = T(0);
            continue;
        }
        const double a = vf[Q[0] + (int64_t)C.n[0] * (Q[1] + (int64_t)C.n[1] * Q[2])];
        const double b = vf[lo[0] + (int64_t)C.n[0] * (lo[1] + (int64_t)C.n[1] * lo[2])];
        const double v = fmin(1.0, fmax(0.0, (a + b) / 2));
        const double den = rl * v + rg * (1 - v);
        c[q] = (T)(dt / (den * h2));
    }
}

// fine coefficients from the face densities (FP64), plus the rhs and initial guess
__global__ void k_fine_setup(DevMesh m, LevelGeom g, double dt, const double* denx, const double* deny,
                             const double* denz, const double* rhs, const double* P, double* cx, double* cy,
                             double* cz, double* b, double* p) {
    const int64_t tot = g.size();
    const double h2[3] = {m.dx * m.dx, m.dy * m.dy, m.dz * m.dz};
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(q % g.n[0]) + 1;
        const int j = (int)((q / g.n[0]) % g.n[1]) + 1;
        const int k = (int)(q / ((int64_t)g.n[0] * g.n[1])) + 1;
        const int a = i - 1 + m.ng, bb = j - 1 + m.ng, c = k - 1 + m.ng;
        const double dx = denx[a + (int64_t)(m.cnx + 1) * (bb + (int64_t)m.cny * c)];
        const double dy = deny[a + (int64_t)m.cnx * (bb + (int64_t)(m.cny + 1) * c)];
        const double dz = denz[a + (int64_t)m.cnx * (bb + (int64_t)m.cny * c)];
        cx[q] = (i > 1 || g.per[0]) ? dt / (dx * h2[0]) : 0.0;
        cy[q] = (j > 1 || g.per[1]) ? dt / (dy * h2[1]) : 0.0;
        cz[q] = (k > 1 || g.per[2]) ? dt / (dz * h2[2]) : 0.0;
        b[q] = rhs[m.cell(i, j, k)];
        p[q] = P[m.cell(i, j, k)];
    }
}

// level storage of g from a plain-order FP64 array
template <class T>
__global__ void k_to_level(LevelGeom g, const double* a, T* b) {
    const int64_t n = g.size();
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        lcell(g, q, i, j, k);
        b[q] = (T)a[i + (int64_t)g.n[0] * (j + (int64_t)g.n[1] * k)];
    }
}

// p64 += e (p64 in plain order, e in the storage of g)
template <class T>
__global__ void k_add_correction(LevelGeom g, const T* e, double* p) {
    const int64_t n = g.size();
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        lcell(g, q, i, j, k);
        p[i + (int64_t)g.n[0] * (j + (int64_t)g.n[1] * k)] += (double)e[q];
    }
}

template <class T>
__global__ void k_zero(T* a, int64_t n) {
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x)
        a[q] = T(0);
}

__global__ void k_shift(double* a, int64_t n, const double* sum) {
    const double mean = *sum / (double)n;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x)
        a[q] -= mean;
}

constexpr int MG_RED = 256;
__device__ double mg_block_sum(double v, bool maxabs) {
    __shared__ double s[MG_RED];
    s[threadIdx.x] = v;
    __syncthreads();
    for (int w = MG_RED / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            s[threadIdx.x] = maxabs ? fmax(s[threadIdx.x], s[threadIdx.x + w]) : s[threadIdx.x] + s[threadIdx.x + w];
        __syncthreads();
    }
    const double r = s[0];
    __syncthreads();
    return r;
}

// The outer loop's FP64 residual r = b - A p (plain order, flux form) handed straight to the
// V-cycle of precision T: bT = (T) r in the storage of gT, max |r| of the block into
// part[blockIdx.x]; r itself is not stored, and the V-cycle takes its e as zero. A work-group
// takes OUTER_K tiles stacked in z, the coefficients of a uniform tile from the table (24 bytes
// per cell instead of 48). Bound by memory: 256^3 210 -> 130 us, 128^3 23 -> 17 us.
constexpr int OUTER_K = 4;
template <class T>
__global__ __launch_bounds__(MG_RED) void k_outer_resid(LevelGeom g, LevelGeom gT, const double* __restrict__ cx,
                                                       const double* __restrict__ cy, const double* __restrict__ cz,
                                                       const UTile<double>* __restrict__ ut, const double* __restrict__ p,
                                                       const double* __restrict__ b, T* __restrict__ bT, double* part) {
    static_assert(MG_RED == SPLIT_H * SPLIT_J, "one thread per pair of cells of a tile");
    const SplitGrid G(g);
    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int bx = t % G.gx, by = (t / G.gx) % G.gy, k0 = (t / (G.gx * G.gy)) * OUTER_K;
    const int j = by * SPLIT_J + __builtin_amdgcn_readfirstlane(threadIdx.x / SPLIT_H);  // a wave is one row
    const int sy = g.n[0], sz = g.n[0] * g.n[1];
    double vmax = 0.0;
    if (j < g.n[1]) {
        const bool oym = j > 0 || g.per[1], oyp = j + 1 < g.n[1] || g.per[1];
        const int jm = j > 0 ? j - 1 : (g.per[1] ? g.n[1] - 1 : j), jp = j + 1 < g.n[1] ? j + 1 : (g.per[1] ? 0 : j);
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const int i = bx * (2 * SPLIT_H) + a * SPLIT_H + (threadIdx.x & (SPLIT_H - 1));
            if (i >= g.n[0]) continue;
            const bool oxm = i > 0 || g.per[0], oxp = i + 1 < g.n[0] || g.per[0];
            const int im = i > 0 ? i - 1 : (g.per[0] ? g.n[0] - 1 : i), ip = i + 1 < g.n[0] ? i + 1 : (g.per[0] ? 0 : i);
            double pc[OUTER_K + 2], nx[OUTER_K][4], vb[OUTER_K];
#pragma unroll
            for (int z = -1; z <= OUTER_K; ++z) {
                int k = k0 + z;
                if (k < 0) k = g.per[2] ? g.n[2] - 1 : 0;
                if (k >= g.n[2]) k = k == g.n[2] && g.per[2] ? 0 : g.n[2] - 1;
                pc[z + 1] = p[i + sy * j + sz * k];
            }
#pragma unroll
            for (int z = 0; z < OUTER_K; ++z) {
                const int pl = sz * min(k0 + z, g.n[2] - 1);
                nx[z][0] = p[im + sy * j + pl];
                nx[z][1] = p[ip + sy * j + pl];
                nx[z][2] = p[i + sy * jm + pl];
                nx[z][3] = p[i + sy * jp + pl];
                vb[z] = b[i + sy * j + pl];
            }
#pragma unroll
            for (int z = 0; z < OUTER_K; ++z) {
                const int k = k0 + z;
                if (k >= g.n[2]) break;
                const UTile<double> u = ut[bx + G.gx * (by + G.gy * k)];
                const bool ozm = k > 0 || g.per[2], ozp = k + 1 < g.n[2] || g.per[2];
                double c[6];
                if (u.uniform != 0.0) {
                    c[0] = oxm ? u.c[0] : 0.0; c[1] = oxp ? u.c[0] : 0.0;
                    c[2] = oym ? u.c[1] : 0.0; c[3] = oyp ? u.c[1] : 0.0;
                    c[4] = ozm ? u.c[2] : 0.0; c[5] = ozp ? u.c[2] : 0.0;
                } else {
                    const int q = i + sy * j + sz * k;
                    const double x = cx[ip + sy * j + sz * k], y = cy[i + sy * jp + sz * k],
                                 w = cz[i + sy * j + sz * (ozp ? (k + 1 < g.n[2] ? k + 1 : 0) : k)];
                    c[0] = cx[q]; c[1] = oxp ? x : 0.0;
                    c[2] = cy[q]; c[3] = oyp ? y : 0.0;
                    c[4] = cz[q]; c[5] = ozp ? w : 0.0;
                }
                const double v = pc[z + 1];
                const double Ap = ((((c[0] * (nx[z][0] - v) + c[1] * (nx[z][1] - v)) + c[2] * (nx[z][2] - v)) +
                                    c[3] * (nx[z][3] - v)) + c[4] * (pc[z] - v)) + c[5] * (pc[z + 2] - v);
                const double r = vb[z] - Ap;
                bT[lidx(gT, i, j, k)] = (T)r;
                vmax = fmax(vmax, fabs(r));
            }
        }
    }
    const double m = mg_block_sum(vmax, true);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// The same residual a cell per thread in plain order, without the table: meshes whose rows or planes do
// not fill a tile (tile_resid). Clears eT too if given, for a V-cycle whose first sweep reads it. A
// residual of 1x512x512 took 62 us by tiles and 8 this way, of 16x256x256 24 and 15, of a 1024^2 plane
// 20 and 17.
template <class T>
__global__ __launch_bounds__(MG_RED) void k_outer_resid_cells(LevelGeom g, LevelGeom gT, const double* cx,
                                                             const double* cy, const double* cz, const double* p,
                                                             const double* b, T* bT, T* eT,
                                                             double* part) {
    const double* C[3] = {cx, cy, cz};
    const int64_t tot = g.size();
    double vmax = 0.0;
    for (int64_t cell = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; cell < tot;
         cell += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(cell % g.n[0]);
        const int64_t row = cell / g.n[0];
        const int j = (int)(row % g.n[1]), k = (int)(row / g.n[1]);
        int64_t nb[6];
        double cf[6];
        stencil<double, false>(g, const_cast<double* const*>(C), i, j, k, cell, nb, cf);
        const double pc = p[cell];
        const double Ap = ((((cf[0] * (p[nb[0]] - pc) + cf[1] * (p[nb[1]] - pc)) + cf[2] * (p[nb[2]] - pc)) +
                            cf[3] * (p[nb[3]] - pc)) + cf[4] * (p[nb[4]] - pc)) + cf[5] * (p[nb[5]] - pc);
        const double r = b[cell] - Ap;
        const int64_t qs = lidx(gT, i, j, k);
        bT[qs] = (T)r;
        if (eT) eT[qs] = T(0);
        vmax = fmax(vmax, fabs(r));
    }
    const double m = mg_block_sum(vmax, true);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

template <class T>
__global__ __launch_bounds__(MG_RED) void k_sum_part(const T* a, int64_t n, int maxabs, double* part) {
    double v = 0.0;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x)
        v = maxabs ? fmax(v, fabs((double)a[q])) : v + (double)a[q];
    const double r = mg_block_sum(v, maxabs != 0);
    if (threadIdx.x == 0) part[blockIdx.x] = r;
}

__global__ __launch_bounds__(MG_RED) void k_sum_final(const double* part, int n, int maxabs, double* out) {
    double v = 0.0;
    for (int q = threadIdx.x; q < n; q += blockDim.x) v = maxabs ? fmax(v, part[q]) : v + part[q];
    const double r = mg_block_sum(v, maxabs != 0);
    if (threadIdx.x == 0) *out = r;
}

// ---- the coarse end of the V-cycle in one work-group --------------------------------------
// Levels from `first` down to the coarsest run in one block of MG_SMALL_THREADS threads with
// e, b and r of every such level in LDS (coefficients stay in global memory): the same
// smoothing, residual, restriction and prolongation as the per-level kernels, separated by
// block barriers instead of launches. The coarsest level removes the mean of b, zeroes e and
// runs `coarse_sweeps` red-black sweeps.
constexpr int MG_SMALL_THREADS = 1024;
constexpr int MG_SMALL_MAXLEV = 12;
constexpr size_t MG_SMALL_LDS = 120 * 1024;

template <class T>
struct SmallLevels {
    int count;  // number of levels handled in the block
    int nu1, nu2, coarse_sweeps;
    LevelGeom g[MG_SMALL_MAXLEV];
    T* c[MG_SMALL_MAXLEV][3];
    int off[MG_SMALL_MAXLEV];  // LDS element offset of level l: e, then b, then r
    const T* b_top;            // b of the first level (global, from the restriction)
    T* e_top;                  // e of the first level (global, for the prolongation)
};

// The two cells of one colour that a thread relaxes on a level of at most 4 * MG_SMALL_THREADS
// cells, with their stencils: loaded once per level visit, then every sweep reads
// only the neighbours' e from LDS.
template <class T>
struct CellSet {
    int cell[2];
    int nb[2][6];
    T cf[2][6];
    T S[2], b[2];
    bool on[2];
};

// Loads the cells of one colour with the numbers first and first + stride.
// The numbers are half of each row, rounded up, times the rows: of a level of odd rows that can be more
// than two per thread (all of it where rows have one cell). ODD, for those, numbers every second cell of
// each plane, or of the level where planes are odd too, which is at most one more than half of the cells
// (in one instance for all levels the second way cost the common one 3 us of 78 in FP64).
template <bool ODD, class T>
__device__ __forceinline__ void load_cells(const LevelGeom& g, T* const* C, const T* b, int color, int first,
                                           int stride, CellSet<T>& cs) {
    const bool by_row = !ODD || g.n[0] % 2 == 0;
    const int plane = g.n[0] * g.n[1];
    const int run = by_row ? g.n[0] : (plane % 2 ? plane * g.n[2] : plane), half = (run + 1) / 2;
    const int tot = half * (by_row ? g.n[1] * g.n[2] : (plane % 2 ? 1 : g.n[2]));
#pragma unroll
    for (int s = 0; s < 2; ++s) {  // every load issued, a slot without a cell reads cell (0, 0, 0)'s
        const int q = first + s * stride;
        const int h = q % half, r = q / half;
        int i, j, k;
        if (by_row) {
            j = r % g.n[1];
            k = r / g.n[1];
            i = 2 * h + ((color + 1 + j + k) & 1);
        } else {
            const int x = 2 * h + ((color + 1 + r) & 1);  // position in the plane or the level
            const int row = x / g.n[0];
            i = x < run ? x - row * g.n[0] : g.n[0];
            j = row % g.n[1];
            k = plane % 2 ? row / g.n[1] : r;
        }
        const bool on = q < tot && i < g.n[0];
        if (!on) i = j = k = 0;
        const int cell = i + g.n[0] * (j + g.n[1] * k);
        int64_t nb[6];
        T cf[6];
        stencil<T, false>(g, C, i, j, k, cell, nb, cf);
        const T S = ((((cf[0] + cf[1]) + cf[2]) + cf[3]) + cf[4]) + cf[5];
        cs.on[s] = on && S > T(0);
        cs.cell[s] = cell;
        cs.S[s] = cs.on[s] ? S : T(1);
        cs.b[s] = b[cell];
#pragma unroll
        for (int f = 0; f < 6; ++f) { cs.nb[s][f] = (int)nb[f]; cs.cf[s][f] = cf[f]; }
    }
}

template <class T>
__device__ __forceinline__ void relax_cells(T* e, const CellSet<T>& cs) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (!cs.on[s]) continue;
        const T* cf = cs.cf[s];
        const int* nb = cs.nb[s];
        const T sum = ((((cf[0] * e[nb[0]] + cf[1] * e[nb[1]]) + cf[2] * e[nb[2]]) + cf[3] * e[nb[3]]) +
                       cf[4] * e[nb[4]]) + cf[5] * e[nb[5]];
        e[cs.cell[s]] = (sum - cs.b[s]) / cs.S[s];
    }
}

// Orders the LDS accesses of one wave (its lanes run in lockstep; the fences keep the
// compiler from moving loads above the previous phase's stores).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// `sweeps` red-black sweeps of a level in LDS. Levels of at most 64 cells run on wave 0 alone
// with wave-level ordering; larger ones (at most 2 * MG_SMALL_THREADS numbers per colour) on the
// whole block with a barrier per colour.
template <bool ODD, class T>
__device__ __forceinline__ void blk_smooth(const LevelGeom& g, T* const* C, T* e, const T* b, int sweeps) {
    if (sweeps <= 0) return;
    const int tid = threadIdx.x;
    if (g.size() <= 64) {
        if (tid < 64) {
            CellSet<T> red, black;
            load_cells<ODD>(g, C, b, 0, tid, 64, red);
            load_cells<ODD>(g, C, b, 1, tid, 64, black);
            for (int sw = 0; sw < sweeps; ++sw) {
                relax_cells(e, red);
                wave_sync();
                relax_cells(e, black);
                wave_sync();
            }
        }
        __syncthreads();
        return;
    }
    CellSet<T> red, black;
    load_cells<ODD>(g, C, b, 0, tid, MG_SMALL_THREADS, red);
    load_cells<ODD>(g, C, b, 1, tid, MG_SMALL_THREADS, black);
    for (int sw = 0; sw < sweeps; ++sw) {
        relax_cells(e, red);
        __syncthreads();
        relax_cells(e, black);
        __syncthreads();
    }
}

template <class T, bool ODD>
__global__ __launch_bounds__(MG_SMALL_THREADS) void k_small_vcycle(const SmallLevels<T>* P) {
    extern __shared__ double lds_raw[];
    T* lds = reinterpret_cast<T*>(lds_raw);
    const int tid = threadIdx.x;
    const int nl = P->count;
    {
        const int n = (int)P->g[0].size();
        T* e = lds + P->off[0];
        T* b = e + n;
        for (int q = tid; q < n; q += MG_SMALL_THREADS) {
            b[q] = P->b_top[q];
            e[q] = T(0);
        }
        __syncthreads();
    }
    // down: smooth, residual, restrict
    for (int l = 0; l + 1 < nl; ++l) {
        const LevelGeom g = P->g[l];
        const int n = (int)g.size();
        T* C[3] = {P->c[l][0], P->c[l][1], P->c[l][2]};
        T* e = lds + P->off[l];
        T* b = e + n;
        T* r = b + n;
        blk_smooth<ODD>(g, C, e, b, P->nu1);
        for (int cell = tid; cell < n; cell += MG_SMALL_THREADS) {
            const int i = cell % g.n[0], j = (cell / g.n[0]) % g.n[1], k = cell / (g.n[0] * g.n[1]);
            int64_t nb[6];
            T cf[6];
            stencil<T, false>(g, C, i, j, k, cell, nb, cf);
            const T pc = e[cell];
            const T Ap = ((((cf[0] * (e[nb[0]] - pc) + cf[1] * (e[nb[1]] - pc)) + cf[2] * (e[nb[2]] - pc)) +
                           cf[3] * (e[nb[3]] - pc)) + cf[4] * (e[nb[4]] - pc)) + cf[5] * (e[nb[5]] - pc);
            r[cell] = b[cell] - Ap;
        }
        __syncthreads();
        const LevelGeom gc = P->g[l + 1];
        const int nc = (int)gc.size();
        T* ec = lds + P->off[l + 1];
        T* bc = ec + nc;
        const int f0 = gc.coarsened[0] ? 2 : 1, f1 = gc.coarsened[1] ? 2 : 1, f2 = gc.coarsened[2] ? 2 : 1;
        const T inv = T(1) / T(f0 * f1 * f2);
        for (int q = tid; q < nc; q += MG_SMALL_THREADS) {
            const int I = q % gc.n[0], J = (q / gc.n[0]) % gc.n[1], K = q / (gc.n[0] * gc.n[1]);
            T sum = T(0);
            for (int c = 0; c < f2; ++c)
                for (int bb = 0; bb < f1; ++bb)
                    for (int a = 0; a < f0; ++a)
                        sum += r[(I * f0 + a) + g.n[0] * ((J * f1 + bb) + g.n[1] * (K * f2 + c))];
            bc[q] = sum * inv;
            ec[q] = T(0);
        }
        __syncthreads();
    }
    // coarsest: consistent right-hand side, then sweeps from zero
    {
        const int l = nl - 1;
        const LevelGeom g = P->g[l];
        const int n = (int)g.size();
        T* C[3] = {P->c[l][0], P->c[l][1], P->c[l][2]};
        T* e = lds + P->off[l];
        T* b = e + n;
        __shared__ double red[MG_SMALL_THREADS / 64];
        double v = 0.0;
        for (int q = tid; q < n; q += MG_SMALL_THREADS) v += (double)b[q];
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
        if ((tid & 63) == 0) red[tid >> 6] = v;
        __syncthreads();
        double tot = 0.0;
        for (int w = 0; w < MG_SMALL_THREADS / 64; ++w) tot += red[w];
        const T mean = (T)(tot / (double)n);
        for (int q = tid; q < n; q += MG_SMALL_THREADS) {
            b[q] -= mean;
            e[q] = T(0);
        }
        __syncthreads();
        blk_smooth<ODD>(g, C, e, (const T*)b, P->coarse_sweeps);
    }
    // up: prolongate and smooth
    for (int l = nl - 2; l >= 0; --l) {
        const LevelGeom g = P->g[l], gc = P->g[l + 1];
        const int n = (int)g.size();
        T* C[3] = {P->c[l][0], P->c[l][1], P->c[l][2]};
        T* e = lds + P->off[l];
        T* b = e + n;
        const T* ec = lds + P->off[l + 1];
        for (int q = tid; q < n; q += MG_SMALL_THREADS) {
            const int qq[3] = {q % g.n[0], (q / g.n[0]) % g.n[1], q / (g.n[0] * g.n[1])};
            int lo[3], hi[3];
            T w1[3], w2[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                if (!gc.coarsened[d]) { lo[d] = hi[d] = qq[d]; w1[d] = T(1); w2[d] = T(0); continue; }
                const int Q = qq[d] / 2;
                if ((qq[d] & 1) == 0) { lo[d] = Q - 1; hi[d] = Q; w1[d] = T(0.75); w2[d] = T(0.25); }
                else { lo[d] = Q; hi[d] = Q + 1; w1[d] = T(0.25); w2[d] = T(0.75); }
                if (lo[d] < 0) lo[d] = gc.per[d] ? gc.n[d] - 1 : 0;
                if (hi[d] >= gc.n[d]) hi[d] = gc.per[d] ? 0 : gc.n[d] - 1;
            }
            auto E = [&](int a, int bb, int c) { return ec[a + gc.n[0] * (bb + gc.n[1] * c)]; };
            const T v = w1[2] * (w1[1] * (w1[0] * E(hi[0], hi[1], hi[2]) + w2[0] * E(lo[0], hi[1], hi[2])) +
                                 w2[1] * (w1[0] * E(hi[0], lo[1], hi[2]) + w2[0] * E(lo[0], lo[1], hi[2]))) +
                        w2[2] * (w1[1] * (w1[0] * E(hi[0], hi[1], lo[2]) + w2[0] * E(lo[0], hi[1], lo[2])) +
                                 w2[1] * (w1[0] * E(hi[0], lo[1], lo[2]) + w2[0] * E(lo[0], lo[1], lo[2])));
            e[q] += v;
        }
        __syncthreads();
        blk_smooth<ODD>(g, C, e, (const T*)b, P->nu2);
    }
    {
        const int n = (int)P->g[0].size();
        const T* e = lds + P->off[0];
        for (int q = tid; q < n; q += MG_SMALL_THREADS) P->e_top[q] = e[q];
    }
}

__global__ void k_store_p(DevMesh m, LevelGeom g, const double* p, double* P) {
    const int64_t tot = g.size();
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(q % g.n[0]) + 1;
        const int j = (int)((q / g.n[0]) % g.n[1]) + 1;
        const int k = (int)(q / ((int64_t)g.n[0] * g.n[1])) + 1;
        P[m.cell(i, j, k)] = p[q];
    }
}

// ---- host driver -----------------------------------------------------------------------
static inline int gridn(int64_t n, int b = 256) {
    int64_t g = (n + b - 1) / b;
    return (int)std::max<int64_t>(1, std::min<int64_t>(g, 65536));
}

#define MGL(kernel, grid, block, ...)                                                    \
    do {                                                                                 \
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, ctx->stream, __VA_ARGS__); \
        MIST_HIP_TRY(hipGetLastError());                                                 \
    } while (0)

template <class T>
static int alloc_level(mist_ctx* ctx, MGState* s, const LevelGeom& g, LevelBuf<T>& L) {
    const size_t bytes = (size_t)g.size() * sizeof(T);
    void** ptrs[6] = {(void**)&L.c[0], (void**)&L.c[1], (void**)&L.c[2], (void**)&L.e, (void**)&L.b, (void**)&L.r};
    for (void** p : ptrs) {
        if (hipMalloc(p, bytes) != hipSuccess) { ctx->err = "multigrid: device allocation failed"; return MIST_ERR_OOM; }
        s->allocs.push_back(*p);
    }
    return MIST_OK;
}

// The coarse end of the hierarchy that fits in MG_SMALL_LDS bytes of LDS (e, b, r per level)
// goes to k_small_vcycle; its descriptor is copied to device memory once.
template <class T>
static int build_small(mist_ctx* ctx, MGState* s, std::vector<LevelBuf<T>>& L, int q) {
    const int nlev = (int)s->g.size();
    int first = nlev - 1;
    size_t bytes = 3 * sizeof(T) * (size_t)s->g[first].size();
    const int64_t maxcells = 4 * MG_SMALL_THREADS;  // two cells per thread and colour
    while (first > 0 && nlev - first < MG_SMALL_MAXLEV && s->g[first - 1].size() <= maxcells &&
           bytes + 3 * sizeof(T) * (size_t)s->g[first - 1].size() <= MG_SMALL_LDS) {
        --first;
        bytes += 3 * sizeof(T) * (size_t)s->g[first].size();
    }
    if (bytes > MG_SMALL_LDS || s->g[first].size() > maxcells) { ctx->err = "multigrid: coarsest level too large for one work-group (raise mg_lvl)"; return MIST_ERR_PARAM; }
    SmallLevels<T> h{};
    h.count = nlev - first;
    h.nu1 = (int)ctx->p.mg_nu1;
    h.nu2 = (int)ctx->p.mg_nu2;
    h.coarse_sweeps = (int)ctx->p.mg_coarse_sweeps;
    int off = 0;
    for (int l = first; l < nlev; ++l) {
        h.g[l - first] = s->g[l];
        for (int d = 0; d < 3; ++d) h.c[l - first][d] = L[l].c[d];
        h.off[l - first] = off;
        off += 3 * (int)s->g[l].size();
    }
    h.b_top = L[first].b;
    h.e_top = L[first].e;
    void* dsc = nullptr;
    if (hipMalloc(&dsc, sizeof(h)) != hipSuccess) { ctx->err = "multigrid: device allocation failed"; return MIST_ERR_OOM; }
    s->allocs.push_back(dsc);
    MIST_HIP_TRY(hipMemcpy(dsc, &h, sizeof(h), hipMemcpyHostToDevice));
    s->small_odd[q] = false;
    for (int l = first; l < nlev; ++l)
        s->small_odd[q] |= (s->g[l].n[0] + 1) / 2 * s->g[l].n[1] * s->g[l].n[2] > 2 * MG_SMALL_THREADS;
    const void* kernel = s->small_odd[q] ? (const void*)k_small_vcycle<T, true> : (const void*)k_small_vcycle<T, false>;
    MIST_HIP_TRY(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    s->first_small[q] = first;
    s->small_lds[q] = bytes;
    s->small_desc[q] = dsc;
    return MIST_OK;
}

// Rows of at least ROW_CELLS cells fill a wave of the kernels that take pairs of a row (k_rbgs_split,
// k_resid_restrict, k_prolong_split) or a tile of k_outer_resid at least by half. Shorter rows keep the
// kernels that take cells in storage order, but for the levels of the LDS sweeps and small ones, whose launches
// cost more than their lanes (LDS_SMALL_CELLS; 32x512x1 1.45 split, 1.49 ms plain). A solve of four
// cycles in plain order against split rows, FP64 and mixed: 2x512x512 4.0 against 15.0 and 3.1 against
// 12.4 ms, 16x256x256 3.4 : 5.5 and 2.8 : 3.9, 32x256x256 4.9 : 5.6 and 3.8 : 3.9, 64x256x256 8.2 : 6.8 and 6.1 : 4.9.
constexpr int ROW_CELLS = 64;

// Whether the outer residual goes by tiles (k_outer_resid), and its work-groups, a partial each.
static bool tile_resid(const LevelGeom& g) { return g.n[0] >= ROW_CELLS && g.n[2] > 1; }
// Whether it leaves e of the V-cycle's first level (storage gT) cleared, for sweeps that read it at once.
static bool resid_clears(const LevelGeom& g, const LevelGeom& gT) { return !tile_resid(g) && !gT.split; }
static int outer_blocks(const LevelGeom& g) {
    if (!tile_resid(g)) return std::min(4096, gridn(g.size(), MG_RED));
    const SplitGrid G(g);
    return G.gx * G.gy * ((g.n[2] + OUTER_K - 1) / OUTER_K);
}

// Levels whose LDS tiles are at most one per compute unit, LDS_TILES, take two sweeps per launch; the others a
// launch per colour. A second round of work-groups costs what the first does: in whole solves of four
// cycles (FP64) the finest level's fused sweeps take 1.01 of a colour launch's time at 256 tiles (64^3; mixed
// 0.91) and 1.18-1.25 at 288 (64x64x72, 128x32x72; mixed 1.10-1.16), and of a shape of two planes with
// 1024 tiles (512x256x2) 1.38; two rows of a tile's eight are not worth it at any count (64x2x256, 128 tiles: 1.12).
// Levels of at most LDS_SMALL_CELLS whose tiles of a quarter of that size are as few
// take those, which leaves more work-groups and half the work for each (32^3 in FP64: 8 us against 11.5).
constexpr int LDS_TILES = 256;
constexpr int64_t LDS_SMALL_CELLS = 70000, LDS_SMALL_TILES = 288;
using LdsOne = LdsTile<1, 8, 8, 8>;
using LdsSmall = LdsTile<2, 4, 8, 4>;
using LdsLarge = LdsTile<2, 8, 8, 8>;
template <class C>
static int64_t lds_tiles(const LevelGeom& g) {
    return (int64_t)((g.n[0] / 2 + C::BH - 1) / C::BH) * ((g.n[1] + C::BY - 1) / C::BY) * ((g.n[2] + C::BZ - 1) / C::BZ);
}
static bool lds_small(const LevelGeom& g) { return g.size() <= LDS_SMALL_CELLS && lds_tiles<LdsSmall>(g) <= LDS_SMALL_TILES; }
static bool lds_fits(const LevelGeom& g) {
    if (g.n[0] % 2 || g.n[1] < 2 || g.n[2] < 2) return false;
    for (int d = 1; d < 3; ++d)
        if (g.per[d] && g.n[d] % 2) return false;
    return lds_small(g) || (g.n[1] >= 4 && g.n[2] >= 4 && lds_tiles<LdsLarge>(g) <= LDS_TILES);
}

static int build_state(mist_ctx* ctx) {
    if (ctx->mg) return MIST_OK;
    const mist_params& p = ctx->p;
    MGState* s = new MGState();
    LevelGeom g0{};
    g0.n[0] = (int)p.Nx; g0.n[1] = (int)p.Ny; g0.n[2] = (int)p.Nz;
    g0.per[0] = p.xper && p.Nx > 1; g0.per[1] = p.yper && p.Ny > 1; g0.per[2] = p.zper && p.Nz > 1;
    int64_t nlev = p.mg_lvl;
    if (nlev <= 1) {
        nlev = 1;
        int n[3] = {g0.n[0], g0.n[1], g0.n[2]};
        for (;;) {
            const int mx = std::max(n[0], std::max(n[1], n[2]));
            bool ok = mx > 4;
            for (int d = 0; d < 3; ++d) if (n[d] > 1 && (n[d] % 2)) ok = false;
            if (!ok) break;
            for (int d = 0; d < 3; ++d) if (n[d] > 1) n[d] /= 2;
            ++nlev;
        }
    }
    s->g.push_back(g0);
    for (int64_t l = 1; l < nlev; ++l) {
        LevelGeom c{};
        const LevelGeom& f = s->g.back();
        for (int d = 0; d < 3; ++d) {
            if (f.n[d] > 1 && (f.n[d] % 2)) { mg_free(s); ctx->err = "multigrid: odd extent cannot be coarsened"; return MIST_ERR_PARAM; }
            c.coarsened[d] = f.n[d] > 1;
            c.n[d] = f.n[d] > 1 ? f.n[d] / 2 : 1;
            c.per[d] = f.per[d] && c.n[d] > 1;
        }
        s->g.push_back(c);
    }
    s->d.resize(s->g.size());
    s->s.resize(s->g.size());
    s->vfl.assign(s->g.size(), nullptr);
    if (p.mg_coarse_op == MIST_COARSE_RESTRICTED_VF)
        for (size_t l = 1; l < s->g.size(); ++l) {
            if (hipMalloc((void**)&s->vfl[l], (size_t)s->g[l].size() * sizeof(double)) != hipSuccess) { mg_free(s); ctx->err = "multigrid: device allocation failed"; return MIST_ERR_OOM; }
            s->allocs.push_back(s->vfl[l]);
        }
    int st;
    for (size_t l = 0; l < s->g.size(); ++l) {
        if ((st = alloc_level(ctx, s, s->g[l], s->d[l]))) { mg_free(s); return st; }
        if ((st = alloc_level(ctx, s, s->g[l], s->s[l]))) { mg_free(s); return st; }
    }
    if ((st = build_small<double>(ctx, s, s->d, 0)) || (st = build_small<float>(ctx, s, s->s, 1))) {
        mg_free(s);
        return st;
    }
    for (int q = 0; q < 2; ++q) {
        s->gq[q] = s->g;
        for (int l = 0; l < s->first_small[q]; ++l) {
            LevelGeom& g = s->gq[q][l];
            g.split = g.n[0] % 2 == 0 && (g.n[0] >= ROW_CELLS || g.size() <= LDS_SMALL_CELLS || lds_fits(g));
            if (!g.split) continue;
            const size_t nb = (size_t)SplitGrid(g).nb;
            void** ut = q == 0 ? (void**)&s->d[l].ut : (void**)&s->s[l].ut;
            if (hipMalloc(ut, nb * (q == 0 ? sizeof(UTile<double>) : sizeof(UTile<float>))) != hipSuccess) { mg_free(s); ctx->err = "multigrid: device allocation failed"; return MIST_ERR_OOM; }
            s->allocs.push_back(*ut);
        }
    }
    s->nfine = g0.size();
    const size_t fb = (size_t)s->nfine * sizeof(double);
    double** f64[5] = {&s->c64[0], &s->c64[1], &s->c64[2], &s->p64, &s->b64};
    for (double** q : f64) {
        if (hipMalloc((void**)q, fb) != hipSuccess) { mg_free(s); ctx->err = "multigrid: device allocation failed"; return MIST_ERR_OOM; }
        s->allocs.push_back(*q);
    }
    if (tile_resid(g0)) {
        if (hipMalloc((void**)&s->ut64, (size_t)SplitGrid(g0).nb * sizeof(UTile<double>)) != hipSuccess) { mg_free(s); ctx->err = "multigrid: device allocation failed"; return MIST_ERR_OOM; }
        s->allocs.push_back(s->ut64);
    }
    s->nblocks = 4096;  // fixed: the sums' order, and with it the last bits of the means, depends on it
    // the residual has a partial per work-group, the others at most nblocks and their result behind them
    const size_t npart = std::max<size_t>(s->nblocks + 8, outer_blocks(g0));
    if (hipMalloc((void**)&s->part, npart * sizeof(double)) != hipSuccess) { mg_free(s); ctx->err = "multigrid: device allocation failed"; return MIST_ERR_OOM; }
    s->allocs.push_back(s->part);
    if (hipHostMalloc((void**)&s->h_part, 8 * sizeof(double), hipHostMallocDefault) != hipSuccess) { mg_free(s); ctx->err = "multigrid: pinned allocation failed"; return MIST_ERR_OOM; }
    ctx->mg = s;
    return MIST_OK;
}

// sum (maxabs = 0) or max |.| (maxabs = 1) of a device vector, result in s->part[nblocks]
template <class T>
static int dev_reduce(mist_ctx* ctx, const T* a, int64_t n, int maxabs) {
    MGState* s = ctx->mg;
    const int g = std::min<int>(s->nblocks, gridn(n, MG_RED));
    MGL(k_sum_part<T>, g, MG_RED, a, n, maxabs, s->part);
    MGL(k_sum_final, 1, MG_RED, (const double*)s->part, g, maxabs, s->part + s->nblocks);
    return MIST_OK;
}

template <class T, class C>
static int lds_sweeps(mist_ctx* ctx, const LevelGeom& g, const LevelBuf<T>& B, const T* ein, T* eout, bool first) {
    const int tx = (g.n[0] / 2 + C::BH - 1) / C::BH, ty = (g.n[1] + C::BY - 1) / C::BY, tz = (g.n[2] + C::BZ - 1) / C::BZ;
    const dim3 grid(tx * ty * tz);
    if (first)
        hipLaunchKernelGGL((k_rbgs_lds<T, C, true>), grid, dim3(C::NT), 0, ctx->stream, g, tx, ty, (const T*)B.c[0],
                           (const T*)B.c[1], (const T*)B.c[2], (const UTile<T>*)B.ut, ein, eout, (const T*)B.b);
    else
        hipLaunchKernelGGL((k_rbgs_lds<T, C, false>), grid, dim3(C::NT), 0, ctx->stream, g, tx, ty, (const T*)B.c[0],
                           (const T*)B.c[1], (const T*)B.c[2], (const UTile<T>*)B.ut, ein, eout, (const T*)B.b);
    MIST_HIP_TRY(hipGetLastError());
    return MIST_OK;
}

// Planes per thread of a colour pass: four from SPLIT_DEEP cells on, two from SPLIT_PAIRS on, one below, and
// no more than the level has. More planes are fewer loads, fewer planes more work-groups. Solves of
// four cycles with two planes against four: 0.97-0.99 of the time from 256k to 1M cells in either precision; above,
// mixed precision 1.03 at 128^3, 1.04 at 160x128x96, 1.07-1.09 at 4.2M cells, FP64 0.97-0.98. With one plane against two:
// 0.91-0.97 on slabs of 64k to 131k cells (smaller thicker levels take the LDS sweeps), 1.02-1.05 from 328k to 430k. A
// sweep of a 2048^2 plane in FP64 took 60 us with four planes, three of them loaded for nothing, and 34 with one.
constexpr int64_t SPLIT_DEEP = 1 << 20, SPLIT_PAIRS = 200000;
template <class T, int K, int PASS>
static int split_pass(mist_ctx* ctx, const LevelGeom& g, const LevelBuf<T>& B, T* e, int color) {
    const SplitGrid G(g);
    hipLaunchKernelGGL((k_rbgs_split<T, K, PASS>), dim3(G.gx * G.gy * ((g.n[2] + K - 1) / K)), dim3(SPLIT_H, SPLIT_J), 0,
                       ctx->stream, g, (const T*)B.c[0], (const T*)B.c[1], (const T*)B.c[2], (const UTile<T>*)B.ut, e,
                       (const T*)B.b, color);
    MIST_HIP_TRY(hipGetLastError());
    return MIST_OK;
}
// One sweep; `first`: e counts as zero.
template <class T, int K>
static int split_sweep(mist_ctx* ctx, const LevelGeom& g, const LevelBuf<T>& B, T* e, bool first) {
    if (int st = first ? split_pass<T, K, 1>(ctx, g, B, e, 0) : split_pass<T, K, 0>(ctx, g, B, e, 0)) return st;
    return first ? split_pass<T, K, 2>(ctx, g, B, e, 1) : split_pass<T, K, 0>(ctx, g, B, e, 1);
}

// `sweeps` red-black sweeps on level g, red first. *e is the array that holds e before and after
// (B.e or B.r: the fused sweeps write to the other one). With `zero`, e counts as zero before and
// its contents are not read.
template <class T>
static int smooth(mist_ctx* ctx, const LevelGeom& g, LevelBuf<T>& B, T** e, int sweeps, bool zero, bool prof) {
    const int64_t n = g.size();
    if (zero && (sweeps < 1 || !g.split)) {
        MGL(k_zero<T>, gridn(n), 256, *e, n);
        zero = false;
    }
    const bool fused = g.split && lds_fits(g);
    int st;
    for (int sw = 0; sw < sweeps;) {
        hipEvent_t ev = prof ? prof_begin(ctx, MIST_PROF_MG_RBGS) : nullptr;
        const bool first = zero && sw == 0;
        int k = 1;
        if (fused) {
            T* out = *e == B.e ? B.r : B.e;
            k = sweeps - sw >= 2 ? 2 : 1;
            if (k == 1) st = lds_sweeps<T, LdsOne>(ctx, g, B, *e, out, first);
            else if (lds_small(g)) st = lds_sweeps<T, LdsSmall>(ctx, g, B, *e, out, first);
            else st = lds_sweeps<T, LdsLarge>(ctx, g, B, *e, out, first);
            if (st) return st;
            *e = out;
        } else if (g.split) {
            if (n >= SPLIT_DEEP && g.n[2] >= 4) st = split_sweep<T, 4>(ctx, g, B, *e, first);
            else if (n >= SPLIT_PAIRS && g.n[2] >= 2) st = split_sweep<T, 2>(ctx, g, B, *e, first);
            else st = split_sweep<T, 1>(ctx, g, B, *e, first);
            if (st) return st;
        } else {
            const int64_t nh = (int64_t)((g.n[0] + 1) / 2) * g.n[1] * g.n[2];
            for (int c = 0; c < 2; ++c)
                MGL(k_rbgs<T>, gridn(nh), 256, g, B.c[0], B.c[1], B.c[2], *e, (const T*)B.b, c);
        }
        prof_end(ctx, MIST_PROF_MG_RBGS, ev, nullptr, k * n);
        sw += k;
    }
    return MIST_OK;
}

// One V-cycle from level l on L[l].b with e = 0; *eres is the array the level's e ends in.
template <class T>
static int vcycle(mist_ctx* ctx, std::vector<LevelBuf<T>>& L, size_t l, T** eres) {
    MGState* s = ctx->mg;
    const int q = sizeof(T) == sizeof(double) ? 0 : 1;
    const LevelGeom& g = s->gq[q][l];
    LevelBuf<T>& B = L[l];
    const int nu1 = (int)ctx->p.mg_nu1, nu2 = (int)ctx->p.mg_nu2;
    const int64_t n = g.size();
    if ((int)l == s->first_small[q]) {
        const SmallLevels<T>* desc = (const SmallLevels<T>*)s->small_desc[q];
        if (s->small_odd[q])
            hipLaunchKernelGGL((k_small_vcycle<T, true>), dim3(1), dim3(MG_SMALL_THREADS), s->small_lds[q], ctx->stream, desc);
        else
            hipLaunchKernelGGL((k_small_vcycle<T, false>), dim3(1), dim3(MG_SMALL_THREADS), s->small_lds[q], ctx->stream, desc);
        MIST_HIP_TRY(hipGetLastError());
        *eres = B.e;
        return MIST_OK;
    }
    int st;
    T* e = B.e;
    const bool cleared = l == 0 && resid_clears(s->g[0], g);
    if ((st = smooth(ctx, g, B, &e, nu1, !cleared, l == 0))) return st;
    const LevelGeom& gc = s->gq[q][l + 1];
    const bool fused = g.split && gc.coarsened[0] && gc.coarsened[1] && gc.coarsened[2];
    if (fused) {
        const int blocks = SplitGrid(g).gx * ((gc.n[1] + SPLIT_J - 1) / SPLIT_J) * gc.n[2];
        hipLaunchKernelGGL(k_resid_restrict<T>, dim3(blocks), dim3(SPLIT_H, SPLIT_J), 0, ctx->stream, g, gc,
                           (const T*)B.c[0], (const T*)B.c[1], (const T*)B.c[2], (const UTile<T>*)B.ut, (const T*)e,
                           (const T*)B.b, L[l + 1].b);
        MIST_HIP_TRY(hipGetLastError());
    } else {
        T* r = e == B.e ? B.r : B.e;
        MGL(k_resid<T>, gridn(n), 256, g, B.c[0], B.c[1], B.c[2], (const T*)e, (const T*)B.b, r);
        MGL(k_restrict<T>, gridn(gc.size()), 256, g, gc, (const T*)r, L[l + 1].b);
    }
    T* ec = nullptr;
    if ((st = vcycle(ctx, L, l + 1, &ec))) return st;
    if (fused) {
        hipLaunchKernelGGL(k_prolong_split<T>, dim3(SplitGrid(g).nb), dim3(SPLIT_H, SPLIT_J), 0, ctx->stream, gc, g,
                           (const T*)ec, e);
        MIST_HIP_TRY(hipGetLastError());
    } else {
        MGL(k_prolong_add<T>, gridn(n), 256, gc, g, (const T*)ec, e);
    }
    st = smooth(ctx, g, B, &e, nu2, false, l == 0);
    *eres = e;
    return st;
}

template <class T>
static int setup_coefs(mist_ctx* ctx, std::vector<LevelBuf<T>>& L) {
    MGState* s = ctx->mg;
    const std::vector<LevelGeom>& G = s->gq[sizeof(T) == sizeof(double) ? 0 : 1];
    for (int d = 0; d < 3; ++d) MGL(k_to_level<T>, gridn(s->nfine), 256, G[0], (const double*)s->c64[d], L[0].c[d]);
    if (ctx->p.mg_coarse_op == MIST_COARSE_RESTRICTED_VF) {
        double h[3] = {ctx->m.dx, ctx->m.dy, ctx->m.dz};
        for (size_t l = 1; l < L.size(); ++l) {
            MGL(k_restrict_vf, gridn(G[l].size()), 256, ctx->m, s->g[l - 1], s->g[l],
                (const double*)ctx->f[MIST_FIELD_VOF], l == 1 ? (const double*)nullptr : (const double*)s->vfl[l - 1],
                s->vfl[l]);
            for (int d = 0; d < 3; ++d) {
                if (G[l].coarsened[d]) h[d] *= 2.0;
                MGL(k_coef_from_vf<T>, gridn(G[l].size()), 256, G[l], d, s->dt, ctx->p.rho_liq, ctx->p.rho_gas,
                    h[d] * h[d], (const double*)s->vfl[l], L[l].c[d]);
            }
        }
        return MIST_OK;
    }
    for (size_t l = 1; l < L.size(); ++l)
        for (int d = 0; d < 3; ++d)
            MGL(k_coarsen_coef<T>, gridn(G[l].size()), 256, G[l - 1], G[l], d, (const T*)L[l - 1].c[d], L[l].c[d]);
    return MIST_OK;
}

// The hierarchy's coefficients, the tile tables of its split levels and that of the FP64 operator.
template <class T>
static int tile_table(mist_ctx* ctx, const LevelGeom& g, T* const* c, UTile<T>* ut) {
    hipLaunchKernelGGL(k_uniform_tiles<T>, dim3(SplitGrid(g).nb), dim3(SPLIT_H, SPLIT_J), 0, ctx->stream, g,
                       (const T*)c[0], (const T*)c[1], (const T*)c[2], ut);
    MIST_HIP_TRY(hipGetLastError());
    return MIST_OK;
}
template <class T>
static int setup_hierarchy(mist_ctx* ctx, std::vector<LevelBuf<T>>& L) {
    int st = setup_coefs(ctx, L);
    if (st) return st;
    const LevelGeom& g0 = ctx->mg->g[0];
    if (tile_resid(g0) && (st = tile_table<double>(ctx, g0, ctx->mg->c64, ctx->mg->ut64))) return st;
    const std::vector<LevelGeom>& G = ctx->mg->gq[sizeof(T) == sizeof(double) ? 0 : 1];
    for (size_t l = 0; l < L.size(); ++l)
        if (G[l].split && (st = tile_table<T>(ctx, G[l], L[l].c, L[l].ut))) return st;
    return MIST_OK;
}

// FP64 residual of the outer loop handed to the V-cycle of precision T as b of level 0 (whose e the V-cycle
// takes as zero without reading it, or resid_clears), and max|r| into s->h_part[0]
template <class T>
static int outer_residual(mist_ctx* ctx, std::vector<LevelBuf<T>>& L) {
    MGState* s = ctx->mg;
    const int g = outer_blocks(s->g[0]);
    hipEvent_t ev = prof_begin(ctx, MIST_PROF_MG_RESID);
    const LevelGeom& g0 = s->g[0];
    const LevelGeom& gT = s->gq[sizeof(T) == sizeof(double) ? 0 : 1][0];
    const double *cx = s->c64[0], *cy = s->c64[1], *cz = s->c64[2], *p = s->p64, *b = s->b64;
    if (tile_resid(g0))
        MGL(k_outer_resid<T>, g, MG_RED, g0, gT, cx, cy, cz, (const UTile<double>*)s->ut64, p, b, L[0].b, s->part);
    else
        MGL(k_outer_resid_cells<T>, g, MG_RED, g0, gT, cx, cy, cz, p, b, L[0].b, resid_clears(g0, gT) ? L[0].e : nullptr,
            s->part);
    prof_end(ctx, MIST_PROF_MG_RESID, ev, nullptr, s->nfine);
    // straight into pinned memory, which the device writes and the host reads after the wait
    MGL(k_sum_final, 1, MG_RED, (const double*)s->part, g, 1, s->h_part);
    return MIST_OK;
}

// One defect-correction iteration: e = V-cycle(r) in precision T, p += e, the new residual
// handed to the next V-cycle.
template <class T>
static int outer_iteration(mist_ctx* ctx, std::vector<LevelBuf<T>>& L) {
    MGState* s = ctx->mg;
    const int64_t n = s->nfine;
    const LevelGeom& g0 = s->gq[sizeof(T) == sizeof(double) ? 0 : 1][0];
    T* e = nullptr;
    int st = vcycle(ctx, L, 0, &e);
    if (st) return st;
    MGL(k_add_correction<T>, gridn(n), 256, g0, (const T*)e, s->p64);
    return outer_residual(ctx, L);
}

template <class T>
static int solve_t(mist_ctx* ctx, std::vector<LevelBuf<T>>& L, double tol, int64_t* cycles, double* resid) {
    MGState* s = ctx->mg;
    int st = setup_hierarchy(ctx, L);
    if (st) return st;
    const int q = sizeof(T) == sizeof(double) ? 0 : 1;
    const int64_t maxc = ctx->p.mg_max_cycles > 0 ? ctx->p.mg_max_cycles : 10000;
    int64_t cyc = 0;
    double res = 0.0;
    int status = MIST_OK;
    if ((st = outer_residual(ctx, L))) return st;
    for (;;) {
        MIST_HIP_TRY(hipStreamSynchronize(ctx->stream));
        res = *(volatile double*)s->h_part;
        if (!(res > tol)) break;  // also stops on NaN, reported through the residual
        if (cyc >= maxc) { status = MIST_ERR_NOCONV; break; }
        if (ctx->prof.on) {
            // per-kernel timing needs the kernels launched one by one
            if ((st = outer_iteration(ctx, L))) return st;
        } else {
            // the ~200 launches of an iteration replayed as one graph (captured once)
            if (!s->exec[q]) {
                MIST_HIP_TRY(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
                st = outer_iteration(ctx, L);
                hipGraph_t g = nullptr;
                const hipError_t ec = hipStreamEndCapture(ctx->stream, &g);
                if (st) {
                    if (g) (void)hipGraphDestroy(g);
                    return st;
                }
                MIST_HIP_TRY(ec);
                s->graph[q] = g;
                MIST_HIP_TRY(hipGraphInstantiate(&s->exec[q], g, nullptr, nullptr, 0));
            }
            MIST_HIP_TRY(hipGraphLaunch(s->exec[q], ctx->stream));
        }
        ++cyc;
    }
    if (res != res) status = MIST_ERR_NOCONV;
    *cycles = cyc;
    *resid = res;
    return status;
}

int pressure_solve(mist_ctx* ctx, double dt, double tol, int precision, int64_t* cycles, double* resid) {
    int st = build_state(ctx);
    if (st) return st;
    MGState* s = ctx->mg;
    const int64_t n = s->nfine;
    s->dt = dt;
    MGL(k_fine_setup, gridn(n), 256, ctx->m, s->g[0], dt, (const double*)ctx->f[MIST_FIELD_DENX],
        (const double*)ctx->f[MIST_FIELD_DENY], (const double*)ctx->f[MIST_FIELD_DENZ],
        (const double*)ctx->f[MIST_FIELD_RHS], (const double*)ctx->f[MIST_FIELD_P], s->c64[0], s->c64[1], s->c64[2],
        s->b64, s->p64);
    // compatibility: remove the mean of b (constants are the null space of A)
    if ((st = dev_reduce<double>(ctx, s->b64, n, 0))) return st;
    MGL(k_shift, gridn(n), 256, s->b64, n, (const double*)(s->part + s->nblocks));
    int status = precision == MIST_MG_MIXED ? solve_t<float>(ctx, s->s, tol, cycles, resid)
                                            : solve_t<double>(ctx, s->d, tol, cycles, resid);
    if (status != MIST_OK && status != MIST_ERR_NOCONV) return status;
    // zero-mean gauge, back into P, then ghosts
    if ((st = dev_reduce<double>(ctx, s->p64, n, 0))) return st;
    MGL(k_shift, gridn(n), 256, s->p64, n, (const double*)(s->part + s->nblocks));
    MGL(k_store_p, gridn(n), 256, ctx->m, s->g[0], (const double*)s->p64, (double*)ctx->f[MIST_FIELD_P]);
    if ((st = launch_neumann(ctx, MIST_FIELD_P))) return st;
    if ((st = launch_borders(ctx, MIST_FIELD_P))) return st;
    if (status == MIST_ERR_NOCONV) ctx->err = "pressure solve did not converge";
    return status;
}

}  // namespace mist
