// octofmm.hip -- liboctofmm: gfx950 kernels and the C-ABI of include/octofmm.h.
//
// Data path (one level pass):
//   1. stage_records: the caller's AoS state (M[cell][20], com[cell][3],
//      mon[cell]) becomes one 24-double partner record per cell in HBM,
//      ordered coarse-cell-major / child-minor inside each 8^3 slot.  The
//      record already holds what a partner contributes under the reference's
//      staging rules (multipole_interaction_interface.hpp:88-281): refined
//      cells give (M, com), leaf cells give a monopole at the geometric cell
//      centre.
//   2. level_kernel: one 512-lane workgroup per target sub-grid.  Wave w owns
//      a 2x2x2 block of coarse cells, lane = (coarse cell, child), so the 8
//      lanes of one coarse cell share every partner record they load.  Each
//      lane walks the coarse offsets of the opening-criterion stencil and the
//      8 children of each partner coarse cell, accumulating its 20-component
//      local expansion (and 3-component correction) in registers, and adds
//      them to L / writes L_c once at the end.
//   3. root: root_kernel splits the 512 x 512 all-pairs sweep of the root
//      sub-grid over partner chunks; root_reduce sums the chunks in a fixed
//      order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdlib>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "kernels.hpp"
#include "octofmm.h"
#include "octofmm_internal.hpp"

using namespace octofmm;

// ===========================================================================
// Kernels
// ===========================================================================
namespace {

// Workgroups are handed to the 8 XCDs round-robin; give each XCD a contiguous
// run of items so neighbouring sub-grids share an L2.
__device__ __forceinline__ int xcd_item(int b, int n) {
    const int q = n >> 3, r = n & 7;
    const int x = b & 7, i = b >> 3;
    return x * q + (x < r ? x : r) + i;
}

// A store of data nothing in the same pass or solve reads through L2 again
// (staged records, which the level kernels read once per image from HBM, and
// a leaf's final rows): non-temporal, so the lines stream out without
// displacing what the concurrent kernels reuse.
__device__ __forceinline__ void store_stream(double2* p, double2 v) {
    __builtin_nontemporal_store(v.x, &p->x);
    __builtin_nontemporal_store(v.y, &p->y);
}

// One block per 128 cells of a slot (two x-planes).  Those cells' records are
// the 128 consecutive records of the block's coarse x-layer, so the block
// loads the cells' M and centre-of-mass rows (contiguous) in 16-byte pieces
// into LDS rows of 25 doubles (an odd stride: a wave that reads one column of
// 64 rows hits every bank), two waves per 64 rows turn each row into its
// record (one half the mass, dipole, quadrupole and centre, the other the
// octupole), and the records leave as one contiguous range, consecutive
// threads in consecutive 16-byte chunks.  Loads and stores are both coalesced,
// where a lane per record spread every instruction over 64 rows.
constexpr int kStageRow = 25;

// Every branch that fills a half record sets all 12 fields in this order: with
// fields set one by one the compiler merges the branches' last stores into one
// of a varying index, which puts the array into scratch memory.
__device__ __forceinline__ void set12(double* v, double a, double b, double c, double d, double e, double f, double g,
    double h, double i, double j, double k, double l) {
    v[0] = a;
    v[1] = b;
    v[2] = c;
    v[3] = d;
    v[4] = e;
    v[5] = f;
    v[6] = g;
    v[7] = h;
    v[8] = i;
    v[9] = j;
    v[10] = k;
    v[11] = l;
}

// One half of a cell's record fields from its row (M 20, com 3): the mass,
// dipole, quadrupole and centre (fields 0..8 and 21..23) or the octupole
// (fields 9..20).
__device__ __forceinline__ void record_half(const double* row, bool octupole, bool rho, double* v) {
    if (!octupole) {
        const double m4 = row[4], m7 = row[7], tr = (m4 + m7 + row[9]) * (1.0 / 3.0);
        set12(v, row[0], 1.25 * row[1], 1.25 * row[2], 1.25 * row[3], (15.0 / 32.0) * (m4 - tr), (15.0 / 32.0) * row[5],
            (15.0 / 32.0) * row[6], (15.0 / 32.0) * (m7 - tr), (15.0 / 32.0) * row[8], row[20], row[21], row[22]);
    } else {
        double m[10];
#pragma unroll
        for (int i = 0; i < 10; ++i) m[i] = (5.0 / 64.0) * row[10 + i];
        const double tx = m[0] + m[3] + m[5], ty = m[1] + m[6] + m[8], tz = m[2] + m[7] + m[9];
        const double xxx = m[0] - 0.6 * tx, xyy = m[3] - 0.2 * tx, xzz = m[5] - 0.2 * tx;
        const double xxy = m[1] - 0.2 * ty, yyy = m[6] - 0.6 * ty, yzz = m[8] - 0.2 * ty;
        const double xxz = m[2] - 0.2 * tz, yyz = m[7] - 0.2 * tz, xyz = m[4];
        // DRHODT: coefficients of the cubic monomials
        if (rho)
            set12(v, xxx, xyy, xzz, xxy, yyy, yzz, xxz, yyz, xyz, 0.7 * tx, 0.7 * ty, 0.7 * tz);
        else
            set12(v, 0.5 * xxx, 1.5 * xyy, 1.5 * xxy, 0.5 * yyy, 1.5 * xxz, 1.5 * yyz, xxz + yyz, 3.0 * xyz, 0.0, 0.0, 0.0, 0.0);
    }
}

// The first half's fields of a leaf cell: a monopole at the geometric cell
// centre in the target's frame (multipole_interaction_interface.hpp:216-235),
// rounded operation by operation as the reference does.
__device__ __forceinline__ void record_leaf(double m, int x, int y, int z, const int* off, const double* base, double dx,
    double* v) {
#pragma clang fp contract(off)
    set12(v, m, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, (double)(x + off[0]) * dx + base[0] - kInx * dx,
        (double)(y + off[1]) * dx + base[1] - kInx * dx, (double)(z + off[2]) * dx + base[2] - kInx * dx);
}

__device__ __forceinline__ void write_half(double* row, bool octupole, const double* v) {
    if (!octupole) {
#pragma unroll
        for (int i = 0; i < 9; ++i) row[i] = v[i];
#pragma unroll
        for (int i = 0; i < 3; ++i) row[kRecY + i] = v[9 + i];
    } else {
#pragma unroll
        for (int i = 0; i < 12; ++i) row[9 + i] = v[i];
    }
}

// Loads n cells' M and centre rows (contiguous, M 16-byte aligned) into LDS rows.
__device__ __forceinline__ void load_rows(const double* M, const double* com, int n, double* s_row) {
    const int t = threadIdx.x;
    const double2* srcM = reinterpret_cast<const double2*>(M);
#pragma unroll
    for (int r = 0; r < 5; ++r) {
        const int i = t + 256 * r;
        if (i < n * 10) {
            const double2 m = srcM[i];
            double* d = s_row + (i / 10) * kStageRow + 2 * (i % 10);
            d[0] = m.x;
            d[1] = m.y;
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int i = t + 256 * r;
        if (i < n * 3) s_row[(i / 3) * kStageRow + 20 + i % 3] = com[i];
    }
}

// One launch stages up to kStageLevels levels, one after another: the levels
// of a tree that are too small to fill the chip share one (tree_launch).
__global__ __launch_bounds__(256) void stage_records(StageGroup g) {
    __shared__ double s_row[128 * kStageRow];
    int si = blockIdx.x >> 2, lvl = 0;
    const int q = blockIdx.x & 3;
    while (lvl < kStageLevels - 1 && si >= g.a[lvl].nslots) si -= g.a[lvl++].nslots;   // uniform
    const StageArgs& a = g.a[lvl];
    if (si >= a.nslots) return;                // uniform per block
    const int slot = a.list ? a.list[si] : si;
    const int k = a.kind[slot];
    const int c0 = q * 128;
    const int t = threadIdx.x;
    const size_t row0 = (size_t)slot * kCells + c0;
    // cell c0 + t's row; thread t and t + 128 share cell t
    const int cl = t & 127, octupole = t >> 7;   // octupole: uniform per wave
    double* row = s_row + cl * kStageRow;
    double v[12];                              // this half's record fields
    float f32[10];                             // and its FP32 moments (mixed precision)
    if (k == OCTOFMM_SLOT_NONLEAF) {
        load_rows(a.M + row0 * 20, a.com + row0 * 3, 128, s_row);
        __syncthreads();
        record_half(row, octupole, a.rho != 0, v);
        if (a.recm) {
#pragma unroll
            for (int i = 0; i < 10; ++i)
                f32[i] = (float)(row[10 * octupole + i] * (octupole ? record_scale(10 + i) : record_scale(i)));
        }
    } else {
        const bool leaf = k == OCTOFMM_SLOT_LEAF && !octupole;
        const int cell = c0 + cl;
        if (leaf)
            record_leaf(a.mon[row0 + cl], cell >> 6, (cell >> 3) & 7, cell & 7, a.foff + 3 * slot, a.fxbase + 3 * slot,
                a.dx, v);
        else
            set12(v, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0);
#pragma unroll
        for (int i = 1; i < 10; ++i) f32[i] = 0.0f;
        f32[0] = leaf ? (float)v[0] : 0.0f;
    }
    // the row of the block's r-th record: coarse cell r >> 3 of the layer,
    // child r & 7
    auto out = [&](double* rec) {
        double2* dst = reinterpret_cast<double2*>(rec + row0 * kRecDoubles);
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const int ch = t + 256 * i;
            const int r = ch / 12, part = ch % 12;
            const int co = r >> 3, ci = r & 7;
            const int x = (ci >> 2) & 1, y = 2 * (co >> 2) + ((ci >> 1) & 1), z = 2 * (co & 3) + (ci & 1);
            const double* src = s_row + (x * 64 + y * 8 + z) * kStageRow + 2 * part;
            store_stream(dst + ch, make_double2(src[0], src[1]));
        }
    };
    __syncthreads();   // every row read before its record overwrites it
    write_half(row, octupole, v);
    __syncthreads();
    out(a.rec);
    if (a.recm) {   // uniform: the mixed-precision records of the same cells
        __syncthreads();
        double* d = row + 5 * octupole;
#pragma unroll
        for (int i = 0; i < 5; ++i) d[i] = __builtin_bit_cast(double, make_float2(f32[2 * i], f32[2 * i + 1]));
        if (!octupole) {
#pragma unroll
            for (int i = 0; i < 3; ++i) row[2 * kRecmY01 + i] = v[9 + i];
            row[2 * kRecmY2M0 + 1] = v[0];
        } else {
            double* o = row + 2 * kRecmOct;
            o[0] = v[0];
            o[1] = v[1];
            o[2] = v[3];
            o[3] = v[4];
            o[4] = v[6];
            o[5] = v[7];
            o[6] = v[8];
            o[7] = v[9];
            o[8] = v[10];
            o[9] = v[11];
        }
        __syncthreads();
        out(a.recm);
    }
}

// Staging of the per-sub-grid entry points.  The host packs the sub-grid and
// the cells of its neighbours within the stencil's reach (12^3 cells at theta
// 0.5, a ninth of the 27 sub-grids) into pinned memory, which this kernel reads
// where it lies: one pass over PCIe in coalesced rows, with no device copy in
// between.  It writes the records the interaction kernels read, the monopoles
// and (leaf targets) the centres, and the one-target level's tables.  Slot 0 is
// the target, the neighbour in raw direction d is slot packed_slot(d); packed
// cells run over the neighbour's box, x slowest.
__host__ __device__ __forceinline__ int packed_slot(int raw) { return raw == 13 ? 0 : raw < 13 ? raw + 1 : raw; }
__host__ __device__ __forceinline__ int packed_raw(int slot) { return slot == 0 ? 13 : slot <= 13 ? slot - 1 : slot; }

// First cell and extent along one axis of the cells a neighbour hands over,
// d = -1, 0, 1 its direction.
__host__ __device__ __forceinline__ void packed_box(int d, int reach, int& lo, int& n) {
    lo = d < 0 ? kInx - reach : 0;
    n = d == 0 ? kInx : reach;
}

struct PackedArgs {
    const double* src;      // pinned host memory: per slot M [n][20], com [n][3] (refined), mon [n] (leaf);
                            // a leaf target's com [512][3] after its mon
    int32_t off[27];        // first double of each slot
    int32_t kind[27];       // octofmm_slot_kind, or -1: absent
    int32_t reach;
    int32_t rho;
    int32_t leaf_target;
    int32_t item_flags;
    double xbase[3];
    double dx;
    double* rec;            // [27][512][24]
    double* mon;            // [27][512]
    double* com;            // [512][3] a leaf target's centres
    int32_t* meta;          // items[2] nbr[27] kind[27]
    const int32_t* packs_src;   // p2m work lists in pinned memory, packs_n words, copied to packs
    int32_t* packs;
    int32_t packs_n;
    double* p2m;            // [512][8] p2m sums, cleared for leaf targets
};

__global__ __launch_bounds__(256) void stage_packed(PackedArgs a) {
    __shared__ double s_row[128 * kStageRow];
    const int slot = blockIdx.x >> 2, c0 = (blockIdx.x & 3) * 128;
    const int t = threadIdx.x;
    if (blockIdx.x == 0 && t < 27) {
        if (t < 2) a.meta[t] = t == 0 ? 0 : a.item_flags;
        a.meta[2 + t] = a.kind[packed_slot(t)] >= 0 ? packed_slot(t) : -1;
        a.meta[29 + t] = a.kind[t];
    }
    for (int i = blockIdx.x * 256 + t; i < a.packs_n; i += gridDim.x * 256) a.packs[i] = a.packs_src[i];
    if (a.leaf_target)
        for (int i = blockIdx.x * 256 + t; i < kCells * 8; i += gridDim.x * 256) a.p2m[i] = 0.0;
    const int k = a.kind[slot], raw = packed_raw(slot);
    int lo[3], n[3];
    packed_box(raw % 3 - 1, a.reach, lo[0], n[0]);
    packed_box(raw / 3 % 3 - 1, a.reach, lo[1], n[1]);
    packed_box(raw / 9 - 1, a.reach, lo[2], n[2]);
    const int ncell = n[0] * n[1] * n[2], cnt = ncell - c0 < 128 ? ncell - c0 : 128;
    if (k < 0 || cnt <= 0) return;             // uniform per block
    const double* src = a.src + a.off[slot];
    auto cell_of = [&](int i, int& x, int& y, int& z) {
        x = lo[0] + i / (n[1] * n[2]);
        y = lo[1] + i / n[2] % n[1];
        z = lo[2] + i % n[2];
    };
    const int cl = t & 127, octupole = t >> 7;
    double* row = s_row + cl * kStageRow;
    double v[12];
    if (k == OCTOFMM_SLOT_NONLEAF) {
        load_rows(src + (size_t)c0 * 20, src + (size_t)ncell * 20 + (size_t)c0 * 3, cnt, s_row);
        __syncthreads();
        record_half(row, octupole, a.rho != 0, v);   // (rows past cnt: unused)
    } else if (cl < cnt && !octupole) {
        int x, y, z;
        cell_of(c0 + cl, x, y, z);
        const int off[3] = {kInx + kInx * (raw % 3 - 1), kInx + kInx * (raw / 3 % 3 - 1), kInx + kInx * (raw / 9 - 1)};
        record_leaf(src[c0 + cl], x, y, z, off, a.xbase, a.dx, v);
        const int cell = x * 64 + y * 8 + z;
        a.mon[(size_t)slot * kCells + cell] = v[0];
        if (a.leaf_target && slot == 0) {
#pragma unroll
            for (int d = 0; d < 3; ++d) a.com[cell * 3 + d] = src[kCells + cell * 3 + d];
        }
    } else {
        set12(v, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0);
    }
    __syncthreads();
    if (cl < cnt) write_half(row, octupole, v);
    __syncthreads();
    for (int ch = t; ch < cnt * 12; ch += 256) {
        const int r = ch / 12, part = ch % 12;
        int x, y, z;
        cell_of(c0 + r, x, y, z);
        const double* from = s_row + r * kStageRow + 2 * part;
        reinterpret_cast<double2*>(a.rec + ((size_t)slot * kCells + record_of_cell(x, y, z)) * kRecDoubles)[part] =
            make_double2(from[0], from[1]);
    }
}

struct LaneGeom {
    int Cx, Cy, Cz;   // coarse cell in the sub-grid (0..3)
    int k;            // child index
    int cell;         // x*64 + y*8 + z
    int rec;          // record index inside the slot
};

// wave w (0..7 across the sub-grid) owns coarse block ((w>>2)&1, (w>>1)&1, w&1);
// t is the thread's index in the workgroup
__device__ __forceinline__ LaneGeom lane_geom(int w, int t = threadIdx.x) {
    LaneGeom g;
    const int l = t & 63;
    const int c = l >> 3;
    g.k = l & 7;
    g.Cx = ((w >> 2) & 1) * 2 + ((c >> 2) & 1);
    g.Cy = ((w >> 1) & 1) * 2 + ((c >> 1) & 1);
    g.Cz = (w & 1) * 2 + (c & 1);
    const int fx = 2 * g.Cx + ((g.k >> 2) & 1), fy = 2 * g.Cy + ((g.k >> 1) & 1), fz = 2 * g.Cz + (g.k & 1);
    g.cell = fx * 64 + fy * 8 + fz;
    g.rec = (g.Cx * 16 + g.Cy * 4 + g.Cz) * 8 + g.k;
    return g;
}

// Partner coarse cell C + delta -> (slot, coarse index in the slot); slot < 0
// when the direction is empty.
__device__ __forceinline__ int partner_base(const LaneGeom& g, int ax, int ay, int az, const int* s_nbr,
    int& nslot, int& raw) {
    const int px = g.Cx + ax, py = g.Cy + ay, pz = g.Cz + az;
    const int rx = px < 0 ? 0 : (px < 4 ? 1 : 2);
    const int ry = py < 0 ? 0 : (py < 4 ? 1 : 2);
    const int rz = pz < 0 ? 0 : (pz < 4 ? 1 : 2);
    raw = rx + 3 * ry + 9 * rz;
    nslot = s_nbr[raw];
    return ((px & 3) * 16 + (py & 3) * 4 + (pz & 3)) * 8;
}

// geometric centre xbase + i*dx, rounded as written (grid_fmm.cpp:1669-1671)
__device__ __forceinline__ double cell_centre(double xb, int i, double dx) {
#pragma clang fp contract(off)
    return xb + (double)i * dx;
}

// The final expansion of a cell in a whole-tree solve: its interactions plus
// the parent cell's expansion re-expanded about the cell's centre of mass, and
// L_c plus the parent's L_c.
template <bool RHO>
__device__ __forceinline__ void tree_final_row(const LevelArgs& a, int slot, int cell, const double* L, int ncomp,
    const double* C, bool write_c, double* Lf, double* Cf) {
    double l[20], lc[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 20; ++j) l[j] = 0.0;
    const int pn = a.parent[slot];
    if (pn >= 0) {
        const int pc = parent_cell(a.octant[slot], cell >> 7, (cell >> 4) & 3, (cell >> 1) & 3);
        double A[20];
        const double2* src = reinterpret_cast<const double2*>(a.pL + ((size_t)pn * kCells + pc) * 20);
#pragma unroll
        for (int j = 0; j < 10; ++j) {
            const double2 v = src[j];
            A[2 * j] = v.x;
            A[2 * j + 1] = v.y;
        }
        const double* Y = a.pcom + ((size_t)pn * kCells + pc) * 3;
        const double* X = a.com + ((size_t)slot * kCells + cell) * 3;
        const double dX[3] = {X[0] - Y[0], X[1] - Y[1], X[2] - Y[2]};
        local_shift(A, dX, l);
        if (RHO) {
            const double* q = a.pLc + ((size_t)pn * kCells + pc) * 3;
            lc[0] = q[0];
            lc[1] = q[1];
            lc[2] = q[2];
        }
    }
#pragma unroll
    for (int j = 0; j < 20; ++j) Lf[j] = (j < ncomp ? L[j] : 0.0) + l[j];
#pragma unroll
    for (int d = 0; d < 3; ++d) Cf[d] = RHO ? (write_c ? C[d] : 0.0) + lc[d] : 0.0;
}

// Leaf force assembly: phi = G L0, g = -G (L_1..3 + L_c).
template <bool RHO>
__device__ __forceinline__ void leaf_force(const LevelArgs& a, const double* Lf, const double* Cf, double* g4) {
    g4[0] = a.G * Lf[0];
#pragma unroll
    for (int d = 0; d < 3; ++d) g4[1 + d] = RHO ? -a.G * Lf[1 + d] - (a.correct_am ? a.G * Cf[d] : 0.0) : 0.0;
}

// Expansion epilogue of one target cell.  Outside a whole-tree solve:
// accumulate the cell's L (the ncomp leading components: 20 for M2L
// targets, 4 for leaves) and overwrite L_c when the kernel forms it
// (write_c).  In a whole-tree solve the cell's final expansion is written
// directly: interactions + the parent cell's expansion re-expanded about the
// cell's centre of mass (taylor::operator<<=, grid::compute_expansions,
// src/grid_fmm.cpp:1524-1637), L_c + the parent's L_c, and for leaf cells
// phi = G L0 and g = -G (L_1..3 + L_c).
template <bool RHO>
__device__ __forceinline__ void finish_cell(const LevelArgs& a, int slot, int cell, const double* L, int ncomp,
    const double* C, bool write_c, bool leaf_target) {
    // expansion rows are 160 bytes and 16-byte aligned: moved as 10 double2
    double2* Lo = reinterpret_cast<double2*>(a.L + ((size_t)slot * kCells + cell) * 20);
    double* Co = a.Lc + ((size_t)slot * kCells + cell) * 3;
    if (!a.l2l) {
        for (int i = 0; i < ncomp / 2; ++i) {
            double2 v = a.overwrite ? make_double2(0.0, 0.0) : Lo[i];
            v.x += L[2 * i];
            v.y += L[2 * i + 1];
            Lo[i] = v;
        }
        if (RHO && write_c) {
            Co[0] = C[0];
            Co[1] = C[1];
            Co[2] = C[2];
        }
        return;
    }
    double Lf[20], Cf[3];
    tree_final_row<RHO>(a, slot, cell, L, ncomp, C, write_c, Lf, Cf);
    if (!leaf_target || a.leaf_rows) {
#pragma unroll
        for (int j = 0; j < 10; ++j) Lo[j] = make_double2(Lf[2 * j], Lf[2 * j + 1]);
    }
    if (RHO) {
#pragma unroll
        for (int d = 0; d < 3; ++d) Co[d] = Cf[d];
    }
    if (a.g && leaf_target) {
        double2* go = reinterpret_cast<double2*>(a.g + ((size_t)slot * kCells + cell) * 4);
        double g4[4];
        leaf_force<RHO>(a, Lf, Cf, g4);
        if (RHO) {
            go[0] = make_double2(g4[0], g4[1]);
            go[1] = make_double2(g4[2], g4[3]);
        } else {
            reinterpret_cast<double*>(go)[0] = g4[0];   // DRHODT: phi slot only
        }
    }
}

// Mixed-precision kernels: the expansion of a target's FP64 pairs, once they
// are all in s, and after the FP32 ones the correction, whose sums go on.
template <bool RHO>
__device__ __forceinline__ void finish_fp64_part(const Acc<RHO>& s, double* L) {
    double f[kFolded], C[3];
    acc_fold_expansion<RHO>(s, f);
    f[18] = f[19] = f[20] = 0.0;
    acc_finish<RHO>(f, L, C);
}

template <bool RHO>
__device__ __forceinline__ void finish_correction(const Acc<RHO>& s, const double* __restrict__ trec, double* C) {
    if constexpr (RHO) {
        double c[3] = {s.u[6], s.u[7], s.u[8]};
        fold_w(trec, 1.0 / trec[0], s.u, c);
#pragma unroll
        for (int d = 0; d < 3; ++d) C[d] = kCorrectionScale * c[d];
    } else {
        C[0] = C[1] = C[2] = 0.0;
    }
}

// A target's neighbour slots and their kinds in LDS, for near_pairs (the far
// pairs read the neighbour row through scalar loads).  Every thread of the
// workgroup calls it.
__device__ __forceinline__ void near_tables(const LevelArgs& a, int slot, int* s_nbr, int* s_kind) {
    if (threadIdx.x < 27) {
        const int n = a.nbr[(size_t)slot * 27 + threadIdx.x];
        s_nbr[threadIdx.x] = n;
        s_kind[threadIdx.x] = n >= 0 ? a.kind[n] : -1;
    }
    __syncthreads();
}

// Near pairs of a target cell over the coarse offsets di = first, first + step,
// ...: partners in leaf slots, which carry only their monopole.
template <bool RHO>
__device__ __forceinline__ void near_pairs(const LevelArgs& a, const LaneGeom& g, const int* s_nbr, const int* s_kind,
    int first, int step, double X0, double X1, double X2, Acc<RHO>& s) {
    const Tables* __restrict__ tab = a.tab;
    for (int di = first; di < tab->ndelta; di += step) {
        const int ax = tab->delta[di][0], ay = tab->delta[di][1], az = tab->delta[di][2];
        unsigned nb = (unsigned)(tab->nearbits[di] >> (8 * g.k)) & 0xffu;
        int ns, raw;
        const int cb = partner_base(g, ax, ay, az, s_nbr, ns, raw);
        if (ns < 0 || s_kind[raw] != OCTOFMM_SLOT_LEAF) nb = 0;
        const double* pb = a.rec + ((size_t)(ns < 0 ? 0 : ns) * kCells + cb) * kRecDoubles;
        if (__builtin_amdgcn_ballot_w64(nb != 0) == 0) continue;
        // the 8 partners' loads in flight together: one after another the
        // waits for them were most of what a block beside leaves took longer
        // (a 2048-slot level of mixed kinds takes 755 us in place of 790, a
        // 105-slot one at theta 0.34 227 in place of 244)
        double q[8][4];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const double* p = pb + j * kRecDoubles;
            q[j][0] = p[0];
#pragma unroll
            for (int d = 0; d < 3; ++d) q[j][1 + d] = p[kRecY + d];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if ((nb >> j) & 1u) m2l_near<RHO>(q[j][0], q[j][1], q[j][2], q[j][3], X0, X1, X2, s);
    }
}

// Mapping 0.  MIXED: the FP64 pairs of every offset come first, then the FP32
// ones (a.mixbits), so that the FP64 sums are done before the FP32 expansion
// takes their registers.
template <bool RHO, bool MIXED>
__device__ void m2l_item(const LevelArgs& a, int slot, int flags, const int* s_nbr, const int* s_kind, int w) {
    const LaneGeom g = lane_geom(w);
    const Tables* __restrict__ tab = a.tab;
    const double* trec = a.rec + ((size_t)slot * kCells + g.rec) * kRecDoubles;
    const double X0 = trec[kRecY], X1 = trec[kRecY + 1], X2 = trec[kRecY + 2];
    Acc<RHO> s;
    acc_clear(s);
    const int nd = tab->ndelta;
    // far pass, software-pipelined: the record of the next pair is loaded
    // (by every lane, from a valid address) while the current one is computed
    auto far_base = [&](int di, const double* rec, unsigned& fb) -> const double* {
        const int ax = tab->delta[di][0], ay = tab->delta[di][1], az = tab->delta[di][2];
        fb = (unsigned)(tab->farbits[di] >> (8 * g.k)) & 0xffu;
        int ns, raw;
        const int cb = partner_base(g, ax, ay, az, s_nbr, ns, raw);
        if (ns < 0) fb = 0;
        return rec + ((size_t)(ns < 0 ? 0 : ns) * kCells + cb) * kRecDoubles;
    };
    if constexpr (!MIXED) {
        unsigned fb;
        const double* pb = far_base(0, a.rec, fb);
        Rec nxt;
        load_rec(pb, nxt);
        for (int di = 0; di < nd; ++di) {
            unsigned fbn = 0;
            const double* pbn = pb;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const Rec cur = nxt;
                if (j < 7) {
                    load_rec(pb + (j + 1) * kRecDoubles, nxt);
                } else if (di + 1 < nd) {
                    pbn = far_base(di + 1, a.rec, fbn);
                    load_rec(pbn, nxt);
                }
                if (fb & (1u << j)) m2l_far_rec<RHO>(cur, X0, X1, X2, s);
            }
            pb = pbn;
            fb = fbn;
        }
    } else {
        for (int di = 0; di < nd; ++di) {
            unsigned fb;
            const double* pb = far_base(di, a.rec, fb);
            fb &= ~((unsigned)(a.mixbits[di] >> (8 * g.k)));
#pragma unroll 1
            for (int j = 0; j < 8; ++j)
                if (fb & (1u << j)) m2l_far<RHO>(pb + j * kRecDoubles, X0, X1, X2, s);
        }
    }
    if (flags & kItemNear) near_pairs<RHO>(a, g, s_nbr, s_kind, 0, 1, X0, X1, X2, s);
    double f[kFolded], L[20], C[3];
    if constexpr (!MIXED) {
        acc_fold<RHO>(s, trec, f);
        acc_finish<RHO>(f, L, C);
    } else {
        finish_fp64_part<RHO>(s, L);
        for (int di = 0; di < nd; ++di) {
            unsigned fb;
            const double* pb = far_base(di, a.recm, fb);
            fb &= (unsigned)(a.mixbits[di] >> (8 * g.k));
            float Lf[20];
#pragma unroll
            for (int i = 0; i < 20; ++i) Lf[i] = 0.0f;
#pragma unroll 1
            for (int j = 0; j < 8; ++j) {
                if (fb & (1u << j)) {
                    Rec cur;
                    load_rec(pb + j * kRecDoubles, cur);
                    m2l_far_m32<RHO>(cur.v, X0, X1, X2, Lf, s.u);
                }
            }
            // the coarse offset's FP32 partial sums join the FP64 expansion
#pragma unroll
            for (int i = 0; i < 20; ++i) L[i] += (double)Lf[i];
        }
        finish_correction<RHO>(s, trec, C);
    }
    finish_cell<RHO>(a, slot, g.cell, L, 20, C, true, false);
}

// Mapping 5: the coarse offsets of one 2x2x2 coarse block are split over
// SPLIT waves of a workgroup (wave s takes offsets s, s + SPLIT, ...), so a
// sub-grid runs on 8 * SPLIT waves; this shortens the serial time of one
// item for levels with few sub-grids.  Waves s > 0 leave their partial
// expansions in LDS and wave 0 adds them in the order s = 1, 2, ... before
// writing the result.
template <bool RHO, int SPLIT>
__device__ void m2l_item_split(const LevelArgs& a, int slot, int flags, const int* s_nbr, const int* s_kind, int w,
    int sl, double* __restrict__ s_part) {
    const LaneGeom g = lane_geom(w);
    const int lane = threadIdx.x & 63;
    const Tables* __restrict__ tab = a.tab;
    const double* trec = a.rec + ((size_t)slot * kCells + g.rec) * kRecDoubles;
    const double X0 = trec[kRecY], X1 = trec[kRecY + 1], X2 = trec[kRecY + 2];
    Acc<RHO> s;
    acc_clear(s);
    const int nd = tab->ndelta;
    for (int di = sl; di < nd; di += SPLIT) {
        const int ax = tab->delta[di][0], ay = tab->delta[di][1], az = tab->delta[di][2];
        unsigned fb = (unsigned)(tab->farbits[di] >> (8 * g.k)) & 0xffu;
        int ns, raw;
        const int cb = partner_base(g, ax, ay, az, s_nbr, ns, raw);
        if (ns < 0) fb = 0;
        const double* pb = a.rec + ((size_t)(ns < 0 ? 0 : ns) * kCells + cb) * kRecDoubles;
        Rec nxt;
        load_rec(pb, nxt);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const Rec cur = nxt;
            if (j < 7) load_rec(pb + (j + 1) * kRecDoubles, nxt);
            if (fb & (1u << j)) m2l_far_rec<RHO>(cur, X0, X1, X2, s);
        }
    }
    if (flags & kItemNear) near_pairs<RHO>(a, g, s_nbr, s_kind, sl, SPLIT, X0, X1, X2, s);
    double f[kFolded];
    acc_fold<RHO>(s, trec, f);
    if (sl > 0) {
        double* o = s_part + ((size_t)(sl - 1) * 64 + lane) * kFolded;
#pragma unroll
        for (int i = 0; i < kFolded; ++i) o[i] = f[i];
    }
    __syncthreads();
    if (sl == 0) {
        for (int q = 0; q < SPLIT - 1; ++q) {
            const double* o = s_part + ((size_t)q * 64 + lane) * kFolded;
#pragma unroll
            for (int i = 0; i < kFolded; ++i) f[i] += o[i];
        }
        double L[20], C[3];
        acc_finish<RHO>(f, L, C);
        finish_cell<RHO>(a, slot, g.cell, L, 20, C, true, false);
    }
}

// Mapping-5 kernel: one workgroup of SPLIT waves per 2x2x2 coarse block.
template <bool RHO, int SPLIT>
__global__ __launch_bounds__(64 * SPLIT) void level_kernel_split(LevelArgs a) {
    __shared__ int s_nbr[27];
    __shared__ int s_kind[27];
    __shared__ double s_part[(SPLIT - 1) * 64 * kFolded];
    const int v = xcd_item(blockIdx.x, gridDim.x);
    const int item = v >> 3, w = v & 7;
    const int2 it = a.items[a.item0 + item];
    if (threadIdx.x < 27) {
        const int n = a.nbr[(size_t)it.x * 27 + threadIdx.x];
        s_nbr[threadIdx.x] = n;
        s_kind[threadIdx.x] = n >= 0 ? a.kind[n] : -1;
    }
    __syncthreads();
    if (it.y & kItemLeaf) return;
    m2l_item_split<RHO, SPLIT>(a, it.x, it.y, s_nbr, s_kind, w, (int)(threadIdx.x >> 6), s_part);
}

// Waits for this wave's LDS writes (lgkmcnt(0), global loads left in flight)
// and keeps the compiler from moving LDS accesses across the point.  The
// lanes of a wave execute each LDS instruction together and in order, so the
// written records are then visible to every lane of the wave.
__device__ __forceinline__ void lds_wave_sync() {
    __builtin_amdgcn_s_waitcnt(0xC07F);   // vmcnt = 63, expcnt = 7, lgkmcnt = 0
    __builtin_amdgcn_wave_barrier();
}

// Mapping 3: the partner records of each coarse offset staged once per wave
// in LDS by direct global->LDS loads
// (global_load_lds_dwordx4): the 64 partner records a wave needs for one
// coarse offset (8 partner coarse cells x 8 children, 12 KiB) go from L2
// into the wave's LDS image without passing through registers, 16 bytes per
// lane and instruction; the 8 lanes of a coarse cell then read each record as
// an LDS broadcast.  Each group of 96 chunks is followed by one unused pad
// chunk so the 8 groups read together fall into different banks.
constexpr int kDirGroup = 97;              // 96 chunks + 1 pad
constexpr int kDirWave = 8 * kDirGroup;    // 776 double2 = 12.1 KiB per wave

typedef __attribute__((address_space(3))) void* lds_ptr;
// Read-only data seen through the constant address space: uniform loads stay
// scalar even after the kernel has issued LDS-direct loads.
// Forms the 8 values in scalar registers at this point, so that the scalar
// loads they depend on are in flight together (the constraint exists only in
// the device pass).
__device__ __forceinline__ void form_sgprs(const unsigned (&v)[8]) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" ::"s"(v[0]), "s"(v[1]), "s"(v[2]), "s"(v[3]), "s"(v[4]), "s"(v[5]), "s"(v[6]), "s"(v[7]));
#else
    (void)v;
#endif
}

// A uniform address formed in scalar registers at this point: a load that
// adds a 32-bit lane offset to it then takes the scalar-base form, with no
// per-lane 64-bit address arithmetic (the constraint exists only in the
// device pass).
__device__ __forceinline__ const char* uniform_ptr(const char* p) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(p));
#endif
    return p;
}

template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T* as_const(const T* p) {
    return (const __attribute__((address_space(4))) T*)p;
}

// SPLIT = 1: mapping 3, the wave walks every offset of its coarse block.
// SPLIT = 2, 4 or 8: mapping 7, the SPLIT waves of the workgroup share one
// coarse block and wave sl walks offsets sl, sl + SPLIT, ... (far and near);
// the other waves then hand their partial sums to wave 0 through their own
// images, and wave 0 adds them in wave order, so the sum is the same on every
// run.
//
// MIXED (mixed-precision plans): a far offset all of whose far pairs are
// evaluated in FP32 (a.mixorder) stages the mixed-precision records instead and
// runs m2l_far_m32 on them, with the offset's FP32 partial sums added to the
// FP64 expansion after its 8 children; the other far offsets run in FP64.
// The precision is uniform over the wave for each offset, so no lane waits
// for the other precision's arithmetic.
//
// WIDE (mapping 7 on small levels): the entries are split further over `parts` workgroups
// (this one is `part`), and wave 0 leaves the folded sums of its 64 cells in
// `sums` ([kFolded][64]) for level_reduce.
template <bool RHO, int SPLIT = 1, bool MIXED = false, bool WIDE = false>
__device__ void m2l_item_direct(const LevelArgs& a, int slot, int flags, const int* s_nbr, const int* s_kind,
    int w, double2* __restrict__ s_stage, int sl = 0, int part = 0, double* __restrict__ sums = nullptr) {
    static_assert(!(MIXED && WIDE), "the wide form is FP64");
    // this wave's image (wave-uniform address)
    double2* stage = s_stage + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * kDirWave;
    // an opaque copy of the lane index: lane values formed from it are formed
    // where they are used instead of being held across the pair loop, where
    // the RHO kernels run at their register limit
    auto lane = []() -> int {
        int t;
        asm volatile("v_mov_b32 %0, %1" : "=v"(t) : "v"((int)threadIdx.x));
        return t & 63;
    };
    const auto* tab = as_const(a.tab);
    const int wu = __builtin_amdgcn_readfirstlane(w);
    const double* trec = a.rec + ((size_t)slot * kCells + lane_geom(wu).rec) * kRecDoubles;
    const double X0 = trec[kRecY], X1 = trec[kRecY + 1], X2 = trec[kRecY + 2];
    Acc<RHO> s;
    acc_clear(s);
    const int bx = ((wu >> 2) & 1) * 2, by = ((wu >> 1) & 1) * 2, bz = (wu & 1) * 2;
    const auto* nbr_row = as_const(a.nbr + (size_t)__builtin_amdgcn_readfirstlane(slot) * 27);
    // record index (slot * 512 + first child) of the partner coarse cell of
    // group gi (coarse cell gi of the wave's block) at offset a; empty
    // directions are marked in bit gi of `empty`.  32-bit indices keep the 8
    // bases of the next image in 8 scalar registers across the pair loop.
    auto group_rec = [&](int gi, int ax, int ay, int az, unsigned& empty) -> unsigned {
        const int px = bx + ((gi >> 2) & 1) + ax, py = by + ((gi >> 1) & 1) + ay, pz = bz + (gi & 1) + az;
        const int raw = (px < 0 ? 0 : (px < 4 ? 1 : 2)) + 3 * (py < 0 ? 0 : (py < 4 ? 1 : 2)) +
            9 * (pz < 0 ? 0 : (pz < 4 ? 1 : 2));
        const int ns = nbr_row[raw];
        const int cb = ((px & 3) * 16 + (py & 3) * 4 + (pz & 3)) * 8;
        if (ns < 0) empty |= 1u << gi;
        return (unsigned)(ns < 0 ? 0 : ns) * (unsigned)kCells + (unsigned)cb;
    };
    // only the offsets with a far pair are staged (delta 0 is all near / self),
    // in the order of the far schedule
    const int nfd = tab->nsched;
    const int step = WIDE ? SPLIT * a.parts : SPLIT;
    const int q0 = SPLIT == 1 ? 0 : __builtin_amdgcn_readfirstlane(WIDE ? part * SPLIT + sl : sl);
    // The wave's entries are those at positions q0, q0 + step, ... of the
    // schedule; a mixed-precision plan orders it (a.mixorder) with its n64 FP64
    // entries first, so that the FP64 sums are done before the FP32 expansion
    // takes their registers.
    const int n64 = MIXED ? a.mix_n64 : nfd;
    const auto* mixorder = as_const(a.mixorder);
    auto entry = [&](int i) -> int { return MIXED ? mixorder[i] : i; };
    // Group c (8 records = 96 chunks) is loaded by one full instruction
    // (chunks 0..63) and one on the lower 32 lanes (chunks 64..95): both are a
    // uniform base plus the lane's 16-byte offset, and the LDS destination is
    // uniform too, so a refill costs one address add per load instruction.
    // The 8 partner bases of an offset are formed ahead of its refill, their
    // neighbour-slot loads in flight together (one wait, taken while the
    // current image is still arriving, instead of one wait per group).
    unsigned nrec[8];
    int f32_next = 0;           // nonzero: that entry is staged from the mixed-precision records
    unsigned empty_next = 0;    // groups of that entry whose partner (a) slot is empty
    unsigned emptyb_next = 0;   // the same for offset b of a split entry (formed by issue())
    int entry_next = 0;         // the schedule entry bases() last formed
    auto bases = [&](int i) {
        const int e = tab->sched[entry(i)];
        const int di = e & 0xff;
        const int ax = tab->delta[di][0], ay = tab->delta[di][1], az = tab->delta[di][2];
        unsigned empty = 0;
#pragma unroll
        for (int gi = 0; gi < 8; ++gi) nrec[gi] = group_rec(gi, ax, ay, az, empty);
        form_sgprs(nrec);
        empty_next = empty;
        entry_next = e;
        f32_next = i >= n64;
    };
    // The full-wave loads of all groups come first and the half-wave loads
    // follow in one branch of their own: with a full and a half load of one
    // group on the two sides of a branch, the compiler may merge them into one
    // load whose LDS base differs by lane and is then taken from lane 0, which
    // sends the other lanes' chunks to the wrong place.
    //
    // A split entry (kinds 1 and 2) stages 4 records of offset a's partner
    // and 4 of offset b's per group, in two loads on lanes 0..47: lane l
    // moves chunk l % 12 of the half's (l / 12)-th child with the given bit
    // on the entry's axis.  Offset b is -a; its partner bases are formed once
    // a's loads are issued (split entries
    // always stage the FP64 records).  The LDS bases of all loads, and the lane
    // offsets of the split loads, come from opaque copies, so that they are
    // formed here and not held across the pair loop, where the kernel runs at
    // its register limit.
    auto issue = [&]() {
        const int kind = (entry_next >> 16) & 0xff;
        double2* st = stage;
        asm volatile("" : "+s"(st));
        const int lo = lane();
        if (kind == 0) {
            const char* rb = reinterpret_cast<const char*>(MIXED && f32_next != 0 ? a.recm : a.rec);
            const unsigned loff = (unsigned)lo * 16u;
#pragma unroll
            for (int gi = 0; gi < 8; ++gi)
                __builtin_amdgcn_global_load_lds(uniform_ptr(rb + (size_t)nrec[gi] * kRecBytes) + loff,
                                                 (lds_ptr)(st + gi * kDirGroup), 16, 0, 0);
            if (lo < 32) {
#pragma unroll
                for (int gi = 0; gi < 8; ++gi)
                    __builtin_amdgcn_global_load_lds(uniform_ptr(rb + (size_t)nrec[gi] * kRecBytes + 1024) + loff,
                                                     (lds_ptr)(st + gi * kDirGroup + 64), 16, 0, 0);
            }
        } else {
            const char* rb = reinterpret_cast<const char*>(a.rec);
            const int axis = entry_next >> 24;
            const int r = lo / 12, part = lo - 12 * r;
            const int low = (1 << axis) - 1;
            const int jr = ((r & ~low) << 1) | (r & low);   // r-th child with a 0 bit on the axis
            const int va = kind == 1 ? 1 : 0;               // the axis bit of a's staged children
            const unsigned offa = (unsigned)(((jr | (va << axis)) * 12 + part) * 16);
            const unsigned offb = (unsigned)(((jr | ((1 - va) << axis)) * 12 + part) * 16);
            if (lo < 48) {
#pragma unroll
                for (int gi = 0; gi < 8; ++gi)
                    __builtin_amdgcn_global_load_lds(uniform_ptr(rb + (size_t)nrec[gi] * kRecBytes) + offa,
                                                     (lds_ptr)(st + gi * kDirGroup), 16, 0, 0);
            }
            const int di = entry_next & 0xff;
            const int ax = tab->delta[di][0], ay = tab->delta[di][1], az = tab->delta[di][2];
            unsigned brec[8];
            unsigned emptyb = 0;
#pragma unroll
            for (int gi = 0; gi < 8; ++gi) brec[gi] = group_rec(gi, -ax, -ay, -az, emptyb);
            form_sgprs(brec);
            emptyb_next = emptyb;
            if (lo < 48) {
#pragma unroll
                for (int gi = 0; gi < 8; ++gi)
                    __builtin_amdgcn_global_load_lds(uniform_ptr(rb + (size_t)brec[gi] * kRecBytes) + offb,
                                                     (lds_ptr)(st + gi * kDirGroup + 48), 16, 0, 0);
            }
        }
    };
    if (flags & kItemNear) near_pairs<RHO>(a, lane_geom(wu), s_nbr, s_kind, q0, step, X0, X1, X2, s);
    // the lane's group of 8 records in the image
    const double2* group = stage + (lane() >> 3) * kDirGroup;
    // One image: image(lanes of step j, records) between the arrival of
    // position i's records and the refill with those of position i + step.
    auto walk = [&](int i, auto&& image) {
        // the lanes that read record j of the image: those of the classes in
        // byte j of the entry's step masks, unless their group's partner slot
        // is empty; kind 2 classes on the far side of the axis read records
        // 4..7 as their records 0..3.  The masks are formed in scalar
        // registers, one 64-bit lane mask per step (lane = group * 8 + class).
        const int q = entry(i);
        const uint64_t ra = tab->sched_rowa[q], rb = tab->sched_rowb[q];
        // (emptyb_next is formed between the branches of issue(), after which
        // the compiler no longer knows it to be uniform)
        const uint64_t ea = spread_groups(empty_next);
        const uint64_t eb = spread_groups(__builtin_amdgcn_readfirstlane(emptyb_next));
        const double2* recs =
            __builtin_amdgcn_inverse_ballot_w64(repeat_bytes(tab->sched_half[q] & 0xffu)) ? group + 48 : group;
        if (i + step < nfd) bases(i + step);
        __builtin_amdgcn_s_waitcnt(0x3F70);   // vmcnt(0): this wave's image is in LDS
        __builtin_amdgcn_wave_barrier();
        image([&](int j) -> uint64_t { return step_lanes(ra, rb, ea, eb, j); }, recs);
        lds_wave_sync();   // every read of the image done before it is refilled
        if (i + step < nfd) issue();
    };
    int i = q0;
    if (i < nfd) {
        bases(i);
        issue();
    }
    for (; i < n64; i += step)
        walk(i, [&](auto&& step_mask, const double2* recs) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (__builtin_amdgcn_inverse_ballot_w64(step_mask(j))) {
                    Rec cur;
#pragma unroll
                    for (int c = 0; c < 12; ++c) cur.v[c] = recs[j * 12 + c];
                    m2l_far_rec<RHO>(cur, X0, X1, X2, s);
                }
            }
        });
    constexpr int kParts = MIXED ? 23 : kFolded;   // partial sums the waves hand over
    double f[kParts];
    if constexpr (!MIXED) {
        acc_fold<RHO>(s, trec, f);
    } else {
        finish_fp64_part<RHO>(s, f);
        for (; i < nfd; i += step)
            walk(i, [&](auto&& step_mask, const double2* recs) {
                float Lf[20];
#pragma unroll
                for (int c = 0; c < 20; ++c) Lf[c] = 0.0f;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (__builtin_amdgcn_inverse_ballot_w64(step_mask(j)))
                        m2l_far_m32<RHO>(recs + j * 12, X0, X1, X2, Lf, s.u);
                // the offset's FP32 partial sums join the FP64 expansion
#pragma unroll
                for (int c = 0; c < 20; ++c) f[c] += (double)Lf[c];
            });
        finish_correction<RHO>(s, trec, f + 20);
    }
    if constexpr (SPLIT > 1) {
        // no refill is in flight and every read of the image is done, so the
        // image can hold this wave's 64 x kParts partial sums (at most 11.5 KiB)
        double* mine = reinterpret_cast<double*>(stage) + (threadIdx.x & 63) * kParts;
        if (sl != 0) {
#pragma unroll
            for (int i = 0; i < kParts; ++i) mine[i] = f[i];
        }
        __syncthreads();
        if (sl != 0) return;
        for (int o = 1; o < SPLIT; ++o) {
            const double* po = reinterpret_cast<const double*>(s_stage + o * kDirWave) + (threadIdx.x & 63) * kParts;
#pragma unroll
            for (int i = 0; i < kParts; ++i) f[i] += po[i];
        }
    }
    if constexpr (WIDE) {
#pragma unroll
        for (int c = 0; c < kFolded; ++c) sums[c * 64 + (threadIdx.x & 63)] = f[c];
        return;
    }
    // The lane's geometry again, from an opaque copy of the thread index: the
    // far loop needs none of it, and formed here it is not held in registers
    // across that loop (where the RHO kernels run at the register limit).
    int t2;
    asm volatile("v_mov_b32 %0, %1" : "=v"(t2) : "v"((int)threadIdx.x));
    const int cell = lane_geom(wu, t2).cell;
    if constexpr (!MIXED) {
        double L[20], C[3];
        acc_finish<RHO>(f, L, C);
        finish_cell<RHO>(a, slot, cell, L, 20, C, true, false);
    } else {
        finish_cell<RHO>(a, slot, cell, f, 20, f + 20, true, false);
    }
}

// Leaf targets (monopole kernels), list-driven for any opening angle: one
// 512-lane workgroup per leaf sub-grid.
// The monopoles of the sub-grid and of its leaf neighbours within the stencil
// reach are staged once into an LDS window (zeros for refined or missing
// neighbours, whose cells the monopole kernel does not see).  Wave w takes
// child class k = w over the 64 coarse cells, so the partner offsets of its
// p2p loop -- and the four constants (-1/r, d/r^3) per offset -- are the same
// for every lane: each pair is one LDS read and four FMAs with scalar
// operands (monopole_kernel_templates.hpp:16-23, kokkos_kernel.hpp:255-284;
// the 1/dx and -1/dx^2 factors are applied once per cell).  Refined
// neighbours contribute through p2m with their full multipoles over the same
// stencil, far and near alike (monopole_kernel_templates.hpp:69-239): those
// sums come from p2m_kernel, launched before this kernel on the same stream.

// The p2m sums (p2m_kernel) of cell `cell` of p2m item `ordinal` join the p2p
// ones.  Leaf items with p2m come first among the leaf items, so the item's
// place among them indexes p2m_out.
__device__ __forceinline__ void add_p2m(const LevelArgs& a, int ordinal, int cell, double* L, double* C) {
    const double2* ps = reinterpret_cast<const double2*>(a.p2m_out + ((size_t)ordinal * kCells + cell) * 8);
    const double2 v0 = ps[0], v1 = ps[1], v2 = ps[2], v3 = ps[3];
    L[0] += v0.x;
    L[1] += v0.y;
    L[2] += v1.x;
    L[3] += v1.y;
    C[0] = v2.x;
    C[1] = v2.y;
    C[2] = v3.x;
}

template <bool RHO>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void leaf_kernel(LevelArgs a) {
    extern __shared__ double s_win[];
    __shared__ int s_nbr[27];
    __shared__ int s_kind[27];
    const int ordinal = xcd_item(blockIdx.x, gridDim.x);
    const int2 it = a.items[a.item0 + ordinal];
    const int slot = it.x;
    if (threadIdx.x < 27) {
        const int n = a.nbr[(size_t)slot * 27 + threadIdx.x];
        s_nbr[threadIdx.x] = n;
        s_kind[threadIdx.x] = n >= 0 ? a.kind[n] : -1;
    }
    __syncthreads();
    const Tables* __restrict__ tab = a.tab;
    const int h = tab->p2p_halo, W = kInx + 2 * h;
    for (int i = threadIdx.x; i < W * W * W; i += 512) {
        const int x = i / (W * W) - h, y = (i / W) % W - h, z = i % W - h;
        const int raw = (x < 0 ? 0 : x < kInx ? 1 : 2) + 3 * (y < 0 ? 0 : y < kInx ? 1 : 2) +
            9 * (z < 0 ? 0 : z < kInx ? 1 : 2);
        const int ns = s_nbr[raw];
        double m = 0.0;
        if (ns >= 0 && s_kind[raw] == OCTOFMM_SLOT_LEAF)
            m = a.mon[(size_t)ns * kCells + ((x + kInx) & 7) * 64 + ((y + kInx) & 7) * 8 + ((z + kInx) & 7)];
        s_win[i] = m;
    }
    __syncthreads();
    const int k = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = threadIdx.x & 63;
    const int tx = 2 * (l >> 4) + ((k >> 2) & 1), ty = 2 * ((l >> 2) & 3) + ((k >> 1) & 1), tz = 2 * (l & 3) + (k & 1);
    const int cell = tx * 64 + ty * 8 + tz;
    double p0 = 0.0, p1 = 0.0, p2 = 0.0, p3 = 0.0;
    const double* wp = s_win + ((tx + h) * W + (ty + h)) * W + (tz + h) - 2048;
    const int32_t* __restrict__ list = tab->p2plist[k];
    const char* __restrict__ fc = reinterpret_cast<const char*>(tab->p2pconst);
    const int n = tab->np2p_k[k];
#pragma unroll 8
    for (int q = 0; q < n; ++q) {
        const int e = list[q];
        const double* f = reinterpret_cast<const double*>(fc + (e & 0xffff));
        const double m = wp[e >> 16];
        p0 = fma(f[0], m, p0);
        p1 = fma(f[1], m, p1);
        p2 = fma(f[2], m, p2);
        p3 = fma(f[3], m, p3);
    }
    const double s1 = a.inv_dx * a.neg_inv_dx;
    double L[4] = {p0 * a.inv_dx, p1 * s1, p2 * s1, p3 * s1};
    double C[3] = {0.0, 0.0, 0.0};
    const bool p2m = (it.y & kItemP2M) != 0;
    if (p2m) add_p2m(a, ordinal, cell, L, C);
    finish_cell<RHO>(a, slot, cell, L, 4, C, p2m, true);
}

// Two consecutive doubles in one 16-byte load, from an address that need not
// be 16-byte aligned.
typedef double double2_a8 __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ void load2(const double* __restrict__ p, double* v) {
    const double2_a8 d = *reinterpret_cast<const double2_a8*>(p);
    v[0] = d.x;
    v[1] = d.y;
}

// LDS layout of the 14^3 monopole window of leaf_cube_kernel: 8 parity planes
// (x & 1, y & 1, z & 1) of 7^3 cells each, row stride 12 and plane stride 80
// doubles.  At each partner offset a wave's 64 lanes read cells 2C + const
// over the 4^3 coarse cells C, i.e. consecutive cells of one parity plane:
// with strides 1, 12 and 80 (mod 32: 1, 12, 16) the 32 lanes of each half-wave
// hit 32 distinct 8-byte bank pairs.  In the plain x-slowest layout the lanes'
// stride of 2 cells put 4 of them on every bank pair in use.
constexpr int kWinSY = 12, kWinSX = 80, kWinPlane = 7 * kWinSX;
__device__ __forceinline__ int cube_win(int wx, int wy, int wz) {
    return (((wx & 1) << 2) | ((wy & 1) << 1) | (wz & 1)) * kWinPlane + (wx >> 1) * kWinSX + (wy >> 1) * kWinSY + (wz >> 1);
}

// Sums of the p2p constants over one target's partners: potential, x, and the
// odd y and z sums by |offset| 1, 2, 3.
struct P2pSums {
    double p, x, y[3], z[3];
};

// One row (or fold of two opposite rows) of a plane: even sums E[|dz|], odd
// sums O[|dz|]; f = Tables::p2pfold[|dx|][|dy|].  Returns sum E / r^3.
__device__ __forceinline__ double p2p_row(const __attribute__((address_space(4))) double* f, const double* E, const double* O, P2pSums& s) {
    s.p = fma(f[3], E[3], fma(f[2], E[2], fma(f[1], E[1], fma(f[0], E[0], s.p))));
#pragma unroll
    for (int j = 0; j < 3; ++j) s.z[j] = fma(f[5 + j], O[1 + j], s.z[j]);
    return fma(f[7], E[3], fma(f[6], E[2], fma(f[5], E[1], f[4] * E[0])));
}

// Forms the sums at this point (the constraint exists only in the device pass).
__device__ __forceinline__ void form_vgprs(P2pSums& s) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(s.p), "+v"(s.x), "+v"(s.y[0]), "+v"(s.y[1]), "+v"(s.y[2]), "+v"(s.z[0]), "+v"(s.z[1]), "+v"(s.z[2]));
#else
    (void)s;
#endif
}

// p2p of one lane's two targets, the children (0, ky, kz) and (1, ky, kz) of
// coarse cell (Cx, Cy, Cz), over the 6^3 block of cells 2C - 2 .. 2C + 3, all
// within one window.  Per axis a target of child bit 0 sees the offsets
// -2 .. 3, of child bit 1 -3 .. 2: two opposite pairs, 0, and one end e = +-3.
// 1/r and 1/r^3 are even in every offset, so opposite cells are added (for
// the even sums) and subtracted (for the odd ones) before they meet their
// constant, first along z for each row, then along y for each pair of rows.
// The folded rows of a plane serve both targets.
__device__ __forceinline__ void p2p_cube(const double* s_win, int Cx, int Cy, int Cz, int ky, int kz,
    const Tables* tab, P2pSums* s) {
    // window coordinate of the targets' row centre: 2C + 3 + k; "same" rows
    // and columns (offsets 0, +-2) lie in its parity plane, "other" ones
    // (+-1, and the end +-3) in the opposite one
    const int zs = (1 - kz) * kWinPlane + Cz + kz;                 // offset -2
    const int zo = kz * kWinPlane + Cz + 1;                         // offset -1
    const int ze = zo + (kz ? -1 : 2);                              // the end
    const int ys = (1 - ky) * 2 * kWinPlane + (Cy + ky) * kWinSY;   // offset -2
    const int yo = ky * 2 * kWinPlane + (Cy + 1) * kWinSY;          // offset -1
    const int ye = yo + (ky ? -1 : 2) * kWinSY;                     // the end
    const double* w = s_win + Cx * kWinSX;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        s[t].p = s[t].x = 0.0;
#pragma unroll
        for (int j = 0; j < 3; ++j) s[t].y[j] = s[t].z[j] = 0.0;
    }
#pragma unroll
    for (int px = 0; px < 6; ++px) {   // plane x = 2C - 2 + px
        const double* wx = w + ((1 + px) & 1) * 4 * kWinPlane + ((1 + px) >> 1) * kWinSX;
        auto row = [&](int y, double* E, double* O) {
            const double* r = wx + y;
            const double a = r[zo], b = r[zo + 1], c = r[zs], d = r[zs + 2], e = r[ze];
            E[0] = r[zs + 1];
            E[1] = b + a;
            O[1] = b - a;
            E[2] = d + c;
            O[2] = d - c;
            E[3] = O[3] = e;
        };
        double u[2] = {0.0, 0.0};   // sum / r^3 over the plane, even in y and z
        // constants of this plane by |dx| (the opaque pointer, the scheduling
        // fences and form_vgprs keep each group of rows to its own loads and
        // sums: without them all planes' rows and constants are held at once
        // and spill)
        const char* fold = uniform_ptr(reinterpret_cast<const char*>(&tab->p2pfold[0][0][0]));
        auto consts = [&](int t, int ay) {
            const int ax = px - 2 - t < 0 ? 2 + t - px : px - 2 - t;
            return as_const(reinterpret_cast<const double*>(fold)) + (ax * 4 + ay) * 8;
        };
        __builtin_amdgcn_sched_barrier(0);
        {
            double E[4], O[4];
            row(ys + kWinSY, E, O);
#pragma unroll
            for (int t = 0; t < 2; ++t) u[t] += p2p_row(consts(t, 0), E, O, s[t]);
        }
        __builtin_amdgcn_sched_barrier(0);
        {
            double E[4], O[4];
            row(ye, E, O);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const double v = p2p_row(consts(t, 3), E, O, s[t]);
                u[t] += v;
                s[t].y[2] += v;
            }
        }
#pragma unroll
        for (int dy = 1; dy < 3; ++dy) {
            __builtin_amdgcn_sched_barrier(0);
            const int lo = dy == 1 ? yo : ys, step = dy == 1 ? kWinSY : 2 * kWinSY;
            double E[4], O[4], F[4], P[4];
            row(lo, E, O);
            row(lo + step, F, P);
            double D[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                D[j] = F[j] - E[j];
                E[j] += F[j];
            }
#pragma unroll
            for (int j = 1; j < 4; ++j) O[j] += P[j];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const auto* f = consts(t, dy);
                u[t] += p2p_row(f, E, O, s[t]);
                s[t].y[dy - 1] =
                    fma(f[7], D[3], fma(f[6], D[2], fma(f[5], D[1], fma(f[4], D[0], s[t].y[dy - 1]))));
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
            if (px != 2 + t) s[t].x = fma((double)(px - 2 - t), u[t], s[t].x);
#pragma unroll
        for (int t = 0; t < 2; ++t) form_vgprs(s[t]);
    }
    const double ey = ky ? -3.0 : 3.0, ez = kz ? -3.0 : 3.0;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        s[t].y[0] = fma(ey, s[t].y[2], fma(2.0, s[t].y[1], s[t].y[0]));
        s[t].z[0] = fma(ez, s[t].z[2], fma(2.0, s[t].z[1], s[t].z[0]));
    }
}

// Leaf targets at theta = 0.5 (Tables::p2p_cube): one 4-wave workgroup per
// leaf, wave = child bits (ky, kz), lane = coarse cell, two targets (kx = 0,
// 1) per lane.  FP64 VALU issue and LDS reads bound the p2p loop: per target
// it takes ~460 FP64 operations and 108 LDS reads, where one target per lane
// with a multiply-add per constant took 864 and 216.
//
// In a whole-tree solve the final rows (L 20, L_c 3, g 4 doubles a cell) go
// through LDS and leave as the sub-grid's contiguous blocks, consecutive lanes
// in consecutive 16-byte chunks: the L rows of two x planes at a time (20 KiB),
// with the first of them L_c and g of 256 cells.  Written straight from the
// lanes each store would touch 64 rows.  Each staged row, L_c triple and g
// quadruple is shifted by one more element every 16 cells: without that the
// lanes' rows (2 cells apart in z, 16 in y) fall on a quarter of the banks.
//
// A leaf alternates between waiting for its window, FP64 work and 110 KiB of
// stores; alone on the chip 5568 leaves take 200 us, 3.4 TB/s with the VALU a
// third busy, so what counts is how many leaves share a CU.  The staging fits in
// the window's 35 KiB and the kernel in 128 registers, so 4 do (a staging of
// all even or odd planes at once, 40 KiB, left room for 3): a solve of 9361
// leaves takes 1290 us in place of 1313.
template <bool RHO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void leaf_cube_kernel(LeafGroup g) {
    extern __shared__ double s_win[];
    __shared__ int s_nbr[27];
    __shared__ int s_kind[27];
    int at = blockIdx.x, lvl = 0;
    while (lvl < kLeafLevels - 1 && at >= g.n[lvl]) at -= g.n[lvl++];   // uniform
    const LevelArgs& a = g.a[lvl];
    const int ordinal = xcd_item(at, g.n[lvl]);
    const int2 it = a.items[a.item0 + ordinal];
    const int slot = __builtin_amdgcn_readfirstlane(it.x);
    const int th = threadIdx.x;
    if (th < 27) {
        const int n = a.nbr[(size_t)slot * 27 + th];
        s_nbr[th] = n;
        s_kind[th] = n >= 0 ? a.kind[n] : -1;
    }
    __syncthreads();
    // the monopole window, one thread per row of 14 cells along z (3 of the
    // slot below, 8, 3 of the slot above): all of a row's loads are in flight
    // at once and its index arithmetic is done once (a thread per cell spent
    // as many VALU instructions on it as half the p2p loop).  Zeros for refined
    // or missing neighbours.
    if (th < 14 * 14) {
        const int wx = th / 14, wy = th % 14;
        const int x = wx - 3, y = wy - 3;
        const int rxy = (x < 0 ? 0 : x < kInx ? 1 : 2) + 3 * (y < 0 ? 0 : y < kInx ? 1 : 2);
        const size_t at = (size_t)((x & 7) * 64 + (y & 7) * 8);
        const double* src[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int ns = s_nbr[rxy + 9 * q];
            src[q] = ns >= 0 && s_kind[rxy + 9 * q] == OCTOFMM_SLOT_LEAF ? a.mon + (size_t)ns * kCells + at : nullptr;
        }
        double m[14];
#pragma unroll
        for (int i = 0; i < 14; ++i) m[i] = 0.0;
        // (the caller's monopoles are 8-byte aligned only)
        if (src[0]) {
            m[0] = src[0][5];
            load2(src[0] + 6, m + 1);
        }
        if (src[1]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) load2(src[1] + 2 * i, m + 3 + 2 * i);
        }
        if (src[2]) {
            load2(src[2], m + 11);
            m[13] = src[2][2];
        }
        double* row = s_win + cube_win(wx, wy, 0);
#pragma unroll
        for (int i = 0; i < 14; ++i) row[(i & 1) * kWinPlane + (i >> 1)] = m[i];
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(th >> 6);
    const int ky = wave >> 1, kz = wave & 1;
    const int l = th & 63;
    const int Cx = l >> 4, Cy = (l >> 2) & 3, Cz = l & 3;
    P2pSums s[2];
    p2p_cube(s_win, Cx, Cy, Cz, ky, kz, a.tab, s);
    const int cell0 = Cx * 128 + (2 * Cy + ky) * 8 + 2 * Cz + kz;   // kx = 0; kx = 1 is 64 further
    const double s1 = a.inv_dx * a.neg_inv_dx;
    const bool p2m = (it.y & kItemP2M) != 0;
    auto sums = [&](int t, double* L, double* C) {
        L[0] = s[t].p * a.inv_dx;
        L[1] = s[t].x * s1;
        L[2] = s[t].y[0] * s1;
        L[3] = s[t].z[0] * s1;
        C[0] = C[1] = C[2] = 0.0;
        if (p2m) add_p2m(a, ordinal, cell0 + 64 * t, L, C);
    };
    if (!a.l2l) {   // uniform
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            double L[4], C[3];
            sums(t, L, C);
            finish_cell<RHO>(a, slot, cell0 + 64 * t, L, 4, C, p2m, true);
        }
        return;
    }
    // both targets lie in one parent cell
    double A[20], Y[3] = {0.0, 0.0, 0.0}, lc[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 20; ++j) A[j] = 0.0;
    const int pn = a.parent[slot];
    if (pn >= 0) {   // uniform
        const size_t pr = (size_t)pn * kCells + parent_cell(a.octant[slot], Cx, Cy, Cz);
        const double2* src = reinterpret_cast<const double2*>(a.pL + pr * 20);
#pragma unroll
        for (int j = 0; j < 10; ++j) {
            const double2 v = src[j];
            A[2 * j] = v.x;
            A[2 * j + 1] = v.y;
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            Y[d] = a.pcom[pr * 3 + d];
            if (RHO) lc[d] = a.pLc[pr * 3 + d];
        }
    }
    // staged: L rows of 128 cells, L_c and g of 256, each shifted by one more
    // element every 16 cells
    double2* b2 = reinterpret_cast<double2*>(s_win);
    double* bc = s_win + 128 * 20 + 16;
    double2* bg = reinterpret_cast<double2*>(bc + 256 * 3 + 16);
    const int r = Cx * 64 + (cell0 & 63);   // cell r + 64 (r / 64 + kx)
    double2* row = b2 + (r & 127) * 10 + ((r & 127) >> 4);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        double dX[3];
        if constexpr (RHO) {
            // the centres the upward pass of this solve stored (12 KiB a leaf), formed again
            const auto* xb = as_const(a.xbase) + 3 * slot;
            dX[0] = cell_centre(xb[0], 2 * Cx + t, a.dx) - Y[0];
            dX[1] = cell_centre(xb[1], 2 * Cy + ky, a.dx) - Y[1];
            dX[2] = cell_centre(xb[2], 2 * Cz + kz, a.dx) - Y[2];
        } else {
            const double* X = a.com + ((size_t)slot * kCells + cell0 + 64 * t) * 3;
#pragma unroll
            for (int d = 0; d < 3; ++d) dX[d] = X[d] - Y[d];
        }
        double L[4], C[3], Lf[20], Cf[3], g4[4];
        sums(t, L, C);
        local_shift(A, dX, Lf);
#pragma unroll
        for (int j = 0; j < 4; ++j) Lf[j] += L[j];
#pragma unroll
        for (int d = 0; d < 3; ++d) Cf[d] = RHO ? C[d] + lc[d] : 0.0;
        leaf_force<RHO>(a, Lf, Cf, g4);
        if constexpr (!RHO) {   // phi slot only
            if (a.g) a.g[((size_t)slot * kCells + cell0 + 64 * t) * 4] = g4[0];
        }
        __syncthreads();   // the window (then the rows before) read
        if constexpr (RHO) {
            double* c = bc + r * 3 + (r >> 4);
            c[0] = Cf[0];
            c[1] = Cf[1];
            c[2] = Cf[2];
            double2* g = bg + r * 2 + (r >> 4);
            g[0] = make_double2(g4[0], g4[1]);
            g[1] = make_double2(g4[2], g4[3]);
        }
        double2* dst = reinterpret_cast<double2*>(a.L + (size_t)slot * kCells * 20) + 640 * t;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (a.leaf_rows) {   // uniform
                if (h == 1) __syncthreads();
                if ((Cx >> 1) == h) {
#pragma unroll
                    for (int j = 0; j < 10; ++j) row[j] = make_double2(Lf[2 * j], Lf[2 * j + 1]);
                }
            }
            if (a.leaf_rows || h == 0) __syncthreads();
            if (a.leaf_rows) {
#pragma unroll
                for (int i = 0; i < 5; ++i) {   // 128 rows x 10 chunks
                    const int ch = th + 256 * i;
                    store_stream(dst + h * 2560 + ch + ch / 640 * 640, b2[ch + ch / 160]);
                }
            }
            if (RHO && h == 0) {
                double2* lcd = reinterpret_cast<double2*>(a.Lc + (size_t)slot * kCells * 3) + 96 * t;
#pragma unroll
                for (int i = 0; i < 2; ++i) {   // 384 chunks: doubles 2 ch and 2 ch + 1
                    const int ch = th + 256 * i, d0 = 2 * ch + ch / 24;
                    if (ch < 384) store_stream(lcd + ch + ch / 96 * 96, make_double2(bc[d0], bc[d0 + 1]));
                }
                if (a.g) {   // uniform
                    double2* gg = reinterpret_cast<double2*>(a.g + (size_t)slot * kCells * 4) + 128 * t;
#pragma unroll
                    for (int i = 0; i < 2; ++i) {   // 512 chunks
                        const int ch = th + 256 * i;
                        store_stream(gg + ch + ch / 128 * 128, bg[ch + (ch >> 5)]);
                    }
                }
            }
        }
    }
}

// p2m: for leaf targets with refined neighbours, the pairs whose partner cell
// lies in a refined neighbour slot (far and near alike,
// monopole_kernel_templates.hpp:69-239), which are the M2L pair set of the
// target's cells restricted to those slots.  Only coarse cells at the faces,
// edges and corners towards refined neighbours have any, and between 1 and 26
// partner coarse cells each at theta 0.5, so the host lists them when the plan
// is made (build_p2m_packs): a unit is one coarse cell of one leaf, a pack is 8
// units of like length, from any leaves.  One workgroup of 4 waves takes a
// pack: lane = (unit, child), wave sl takes the units' entries sl, sl + 4, ...,
// staging each entry's 8 x 8 partner records into its LDS image by direct loads
// and reading them as 8-lane broadcasts; the waves hand their sums to wave 0,
// which adds them in wave order.  Walked by 2x2x2 coarse blocks of a leaf
// instead, half the lanes of a face's blocks and 7 of 8 of a corner's idled and
// half the workgroups found nothing to do.
// Bound by the FP64 VALU like the M2L kernel, and by its share of the chip
// while it runs beside that one: a 2048-slot level of mixed kinds takes 741 us
// in place of 803, the solve of a 10,697-sub-grid tree 1338 in place of 1416.
//
// FULL: every pair of an entry's 8 x 8 cells is in the stencil (theta 0.5).
template <bool RHO, bool FULL>
__device__ __forceinline__ void p2m_pack(const LevelArgs& a, int pack, double2* s_stage) {
    const int sl = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    double2* stage = s_stage + sl * kDirWave;
    const int l = threadIdx.x & 63, k = l & 7;
    const auto* hdr = as_const(a.p2m_hdr) + 2 * __builtin_amdgcn_readfirstlane(pack);
    const int first = hdr[0], n = hdr[1];
    const int unit = a.p2m_units[(size_t)pack * 8 + (l >> 3)];   // -1: none
    const int C = unit & 63, ordinal = unit < 0 ? 0 : unit >> 6;
    const int cell = (2 * (C >> 4) + (k >> 2)) * 64 + (2 * ((C >> 2) & 3) + ((k >> 1) & 1)) * 8 + 2 * (C & 3) + (k & 1);
    const double* xc = a.com + ((size_t)a.items[a.leaf0 + ordinal].x * kCells + cell) * 3;
    const double X0 = xc[0], X1 = xc[1], X2 = xc[2];
    Acc<RHO> s;
    acc_clear(s);
    // the records of entry e's 8 partner coarse cells; bit g of `absent` where
    // unit g has fewer entries
    unsigned nrec[8];
    unsigned absent_next = 0;
    auto bases = [&](int e) {
        const auto* row = as_const(a.p2m_idx) + (size_t)(first + e) * 8;
        unsigned absent = 0;
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const int r = row[g];
            if (r < 0) absent |= 1u << g;
            nrec[g] = (unsigned)(r < 0 ? 0 : r);
        }
        form_sgprs(nrec);
        absent_next = absent;
    };
    // the full-wave loads of every group first, the half-wave loads after
    // them in a branch of their own (as in m2l_item_direct)
    const char* rb = reinterpret_cast<const char*>(a.rec);
    const unsigned loff = (unsigned)l * 16u;
    auto issue = [&]() {
#pragma unroll
        for (int g = 0; g < 8; ++g)
            __builtin_amdgcn_global_load_lds(uniform_ptr(rb + (size_t)nrec[g] * kRecBytes) + loff,
                                             (lds_ptr)(stage + g * kDirGroup), 16, 0, 0);
        if (l < 32) {
#pragma unroll
            for (int g = 0; g < 8; ++g)
                __builtin_amdgcn_global_load_lds(uniform_ptr(rb + (size_t)nrec[g] * kRecBytes + 1024) + loff,
                                                 (lds_ptr)(stage + g * kDirGroup + 64), 16, 0, 0);
        }
    };
    const double2* group = stage + (l >> 3) * kDirGroup;
    if (sl < n) {
        bases(sl);
        issue();
    }
    for (int e = sl; e < n; e += 4) {
        const uint64_t here = ~spread_groups(absent_next);
        // the lane's pairs of this entry (byte k of the offset's pair bits)
        unsigned mine = 0xffu;
        if constexpr (!FULL) {
            const int di = a.p2m_di[(size_t)(first + e) * 8 + (l >> 3)];
            mine = (unsigned)((a.tab->farbits[di] | a.tab->nearbits[di]) >> (8 * k)) & 0xffu;
        }
        if (e + 4 < n) bases(e + 4);
        __builtin_amdgcn_s_waitcnt(0x3F70);   // vmcnt(0): this wave's image is in LDS
        __builtin_amdgcn_wave_barrier();
        if (__builtin_amdgcn_inverse_ballot_w64(here)) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (FULL || (mine & (1u << j))) {
                    Rec cur;
#pragma unroll
                    for (int i = 0; i < 12; ++i) cur.v[i] = group[j * 12 + i];
                    p2m_pair_rec<RHO>(cur, X0, X1, X2, s);
                }
            }
        }
        lds_wave_sync();   // every read of the image done before it is refilled
        if (e + 4 < n) issue();
    }
    // waves 1..3 hand their sums to wave 0 through their own images
    double L[4], C3[3];
    p2m_finish<RHO>(s, L, C3);
    double* part = reinterpret_cast<double*>(stage) + l * 7;
    if (sl != 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) part[i] = L[i];
#pragma unroll
        for (int i = 0; i < 3; ++i) part[4 + i] = C3[i];
    }
    __syncthreads();
    if (sl != 0 || unit < 0) return;
    for (int o = 1; o < 4; ++o) {
        const double* po = reinterpret_cast<const double*>(s_stage + o * kDirWave) + l * 7;
#pragma unroll
        for (int i = 0; i < 4; ++i) L[i] += po[i];
#pragma unroll
        for (int i = 0; i < 3; ++i) C3[i] += po[4 + i];
    }
    double2* out = reinterpret_cast<double2*>(a.p2m_out + ((size_t)ordinal * kCells + cell) * 8);
    out[0] = make_double2(L[0], L[1]);
    out[1] = make_double2(L[2], L[3]);
    out[2] = make_double2(C3[0], C3[1]);
    out[3] = make_double2(C3[2], 0.0);
}

template <bool RHO, bool FULL>
__global__ __launch_bounds__(256) void p2m_kernel(LevelArgs a) {
    __shared__ double2 s_stage[4 * kDirWave];
    p2m_pack<RHO, FULL>(a, xcd_item(blockIdx.x, gridDim.x), s_stage);
}

template <bool RHO>
void launch_p2m(int npacks, hipStream_t st, const LevelArgs& la, const Tables& tab) {
    if (npacks <= 0) return;
    if (tab.p2p_cube)
        hipLaunchKernelGGL((p2m_kernel<RHO, true>), dim3(npacks), dim3(256), 0, st, la);
    else
        hipLaunchKernelGGL((p2m_kernel<RHO, false>), dim3(npacks), dim3(256), 0, st, la);
}

// Leaf items of n <= kLeafLevels levels in one launch (theta 0.5).
template <bool RHO>
void launch_leaf_cube(const LevelArgs* la, int n, hipStream_t st) {
    // the window's parity planes; the staged results take less
    constexpr size_t lds = sizeof(double) * 8 * kWinPlane;
    static_assert(8 * kWinPlane >= (128 * 20 + 16) + (256 * 3 + 16) + 2 * (256 * 2 + 16));
    LeafGroup g;
    int nitems = 0;
    for (int i = 0; i < kLeafLevels; ++i) {
        g.a[i] = la[i < n ? i : 0];
        g.n[i] = i < n ? la[i].nitems : 0;
        nitems += g.n[i];
    }
    if (nitems > 0) hipLaunchKernelGGL(leaf_cube_kernel<RHO>, dim3(nitems), dim3(256), lds, st, g);
}

template <bool RHO>
void launch_leaf(int nitems, hipStream_t st, const LevelArgs& la, const Tables& tab) {
    if (tab.p2p_cube) {
        launch_leaf_cube<RHO>(&la, 1, st);
    } else {
        const int W = kInx + 2 * tab.p2p_halo;
        hipLaunchKernelGGL(leaf_kernel<RHO>, dim3(nitems), dim3(512), sizeof(double) * W * W * W, st, la);
    }
}

// One target sub-grid is split over 8 / WAVES workgroups of WAVES waves.  The
// workgroup index is first spread over the XCDs (contiguous runs per XCD),
// so the parts of one sub-grid and its neighbours share an L2.
template <bool RHO, int WAVES, bool MIXED = false>
__global__ __launch_bounds__(64 * WAVES) void level_kernel(LevelArgs a) {
    constexpr int kParts = 8 / WAVES;
    __shared__ int s_nbr[27];
    __shared__ int s_kind[27];
    const int v = xcd_item(blockIdx.x, gridDim.x);
    const int item = v / kParts;
    const int w = (v % kParts) * WAVES + (threadIdx.x >> 6);
    const int2 it = a.items[a.item0 + item];
    if (threadIdx.x < 27) {
        const int n = a.nbr[(size_t)it.x * 27 + threadIdx.x];
        s_nbr[threadIdx.x] = n;
        s_kind[threadIdx.x] = n >= 0 ? a.kind[n] : -1;
    }
    __syncthreads();
    if (it.y & kItemLeaf)
        return;   // leaf items run in leaf_kernel
    m2l_item<RHO, MIXED>(a, it.x, it.y, s_nbr, s_kind, w);
}

// Mapping-3 kernel (direct global->LDS staging); one wave per 2x2x2 coarse block.
template <bool RHO, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(3))) void level_kernel_direct(LevelArgs a) {
    constexpr int kParts = 8 / WAVES;
    __shared__ int s_nbr[27];
    __shared__ int s_kind[27];
    __shared__ double2 s_stage[WAVES * kDirWave];
    const int v = xcd_item(blockIdx.x, gridDim.x);
    const int item = v / kParts;
    const int w = (v % kParts) * WAVES + (threadIdx.x >> 6);
    const int2 it = a.items[a.item0 + item];
    if (it.y & kItemNear) near_tables(a, it.x, s_nbr, s_kind);   // uniform per workgroup
    if (it.y & kItemLeaf) return;
    m2l_item_direct<RHO>(a, it.x, it.y, s_nbr, s_kind, w, s_stage);
}

// Mapping-7 kernel: one workgroup of SPLIT waves per 2x2x2 coarse block, the
// coarse offsets split over the waves (mapping 3's staging in each).
template <bool RHO, int SPLIT, bool MIXED = false>
__global__ __launch_bounds__(64 * SPLIT) __attribute__((amdgpu_waves_per_eu(3))) void level_kernel_dsplit(LevelArgs a) {
    __shared__ int s_nbr[27];
    __shared__ int s_kind[27];
    __shared__ double2 s_stage[SPLIT * kDirWave];
    const int v = xcd_item(blockIdx.x, gridDim.x);
    const int item = v >> 3, w = v & 7;
    const int2 it = a.items[a.item0 + item];
    if (it.y & kItemNear) near_tables(a, it.x, s_nbr, s_kind);   // uniform per workgroup
    if (it.y & kItemLeaf) return;   // uniform per workgroup
    m2l_item_direct<RHO, SPLIT, MIXED>(a, it.x, it.y, s_nbr, s_kind, w, s_stage, (int)(threadIdx.x >> 6));
}

// Variant 704 on levels with few sub-grids: each 2x2x2 coarse block's entries
// over a.parts workgroups of 4 waves, whose folded sums meet in level_reduce.
// In the plain form a level of n targets has 8 n workgroups, whose waves each
// walk 6 or 7 images one after another (~3 us an image alone on a SIMD): below
// one workgroup per CU the rest of the chip stands idle meanwhile.  Measured
// (theta 0.5 / 0.34): 1 target 25.3 / 74.6 -> 10.7 / 15.1 us, 8 targets 26.0 /
// 75.2 -> 16.5 / 29.3 us, 18 targets 26.4 / 76.2 -> 21.5 / 47.3 us.
template <bool RHO>
__device__ __forceinline__ void wide_part(const LevelArgs& a, int v, int* s_nbr, int* s_kind, double2* s_stage) {
    const int block = v / a.parts, part = v - block * a.parts;
    const int2 it = a.items[a.item0 + (block >> 3)];
    if (it.y & kItemNear) near_tables(a, it.x, s_nbr, s_kind);   // uniform per workgroup
    m2l_item_direct<RHO, 4, false, true>(a, it.x, it.y, s_nbr, s_kind, block & 7, s_stage, (int)(threadIdx.x >> 6), part,
        a.wide_sums + (size_t)v * (kFolded * 64));
}

template <bool RHO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void level_kernel_wide(LevelArgs a) {
    __shared__ int s_nbr[27];
    __shared__ int s_kind[27];
    __shared__ double2 s_stage[4 * kDirWave];
    wide_part<RHO>(a, xcd_item(blockIdx.x, gridDim.x), s_nbr, s_kind, s_stage);
}

// Sums the parts of one coarse block of a target (one wave, lane = cell) in
// part order and writes the cells' results.
template <bool RHO>
__global__ __launch_bounds__(64) void level_reduce(LevelArgs a) {
    const int block = blockIdx.x;
    const int slot = a.items[a.item0 + (block >> 3)].x;
    const double* src = a.wide_sums + (size_t)block * a.parts * (kFolded * 64) + threadIdx.x;
    double f[kFolded], L[20], C[3];
#pragma unroll
    for (int c = 0; c < kFolded; ++c) f[c] = src[c * 64];
    for (int p = 1; p < a.parts; ++p) {
        src += kFolded * 64;
#pragma unroll
        for (int c = 0; c < kFolded; ++c) f[c] += src[c * 64];
    }
    acc_finish<RHO>(f, L, C);
    finish_cell<RHO>(a, slot, lane_geom(block & 7).cell, L, 20, C, true, false);
}

// Workgroups per coarse block of variant 704 on a level of n targets (0: the
// plain form).  The sums' way through memory and the second kernel cost ~5 us,
// about what two images take, and a second workgroup on some CUs takes back part
// of what a split saves.  With the 26 entries of theta 0.5 two parts take three
// images off a wave: 20 targets 26.3 us plain, 26.1 in two parts, 22 targets
// 26.4 and 26.4, 24 targets 26.3 and 27.0, 28 targets 26.4 and 27.5, so they end
// at 22; shorter schedules (theta above 0.577) save less and end at 16 (theta
// 0.6: 16 targets 21.0 and 18.0 us, 20 targets 21.1 and 22.8; theta 0.75: 8
// targets 11.3 and 10.7, 16 targets 11.4 and 11.5, 22 targets 11.6 and 13.9).
// With the 32 of theta 0.45 they take off four: 28 targets 31.0 and 29.3 us, and
// the split ends at 1.75 workgroups per CU.  With the 92 of theta 0.34 it pays up
// to three (36 targets: 109 and 88 us, 48: 110 and 93, 49: 110 and 117).  At most
// one image per wave.
int wide_parts(int n, const Tables& tab) {
    if (n <= 0) return 0;
    const int parts = std::min((tab.nsched + 3) / 4, (tab.nsched < 48 ? 448 : 768) / (8 * n));
    if (parts == 2 && tab.nsched < 32 && n > (tab.nsched < 26 ? 16 : 22)) return 0;
    return parts >= 2 ? parts : 0;
}

// Bytes of level_kernel_wide's sums.
size_t wide_bytes(int n, int parts) { return sizeof(double) * (size_t)n * 8 * parts * kFolded * 64; }

void launch_wide_sums(int nitems, hipStream_t st, const LevelArgs& la, bool rho) {
    const dim3 grid(nitems * 8 * la.parts);
    if (rho)
        hipLaunchKernelGGL(level_kernel_wide<true>, grid, dim3(256), 0, st, la);
    else
        hipLaunchKernelGGL(level_kernel_wide<false>, grid, dim3(256), 0, st, la);
}

void launch_wide_reduce(int nitems, hipStream_t st, const LevelArgs& la, bool rho) {
    if (rho)
        hipLaunchKernelGGL(level_reduce<true>, dim3(nitems * 8), dim3(64), 0, st, la);
    else
        hipLaunchKernelGGL(level_reduce<false>, dim3(nitems * 8), dim3(64), 0, st, la);
}

// In a whole-tree solve the levels of up to 96 targets (three workgroups a CU)
// run sums first: their sums need only the level's records, so those of the
// coarse levels run side by side with the root's pairs, and of the chain from
// level to level only level_reduce with its downward pass (5 to 6 us) is left,
// where the level kernels of 8 and 32 targets took 22 and 30 us one after the
// other (329-sub-grid tree: 160 -> 125 us a solve, 10,697: 1338 -> 1307).  Larger
// levels fill the chip by themselves, and their sums would cost as much traffic
// as their results.  Workgroups per coarse block of such a level, 0 for a larger
// one: the levels fill the chip together, so a split as fine as wide_parts makes
// of a level by itself only adds sums (95.7 us, against 90.0 with at least 8
// entries, two images a wave, to a part and two workgroups a CU from one level).
int sums_first_parts(int n, const Tables& tab) {
    if (n <= 0 || n > 96) return 0;
    return std::max(1, std::min(tab.nsched / 8, 64 / n));
}

// Persistent form of the mapping-7 kernel (variants 804, 802): a grid of
// the workgroups the chip holds at once, each taking work units (sub-grid,
// coarse block) from a counter until none are left.  Workgroups are handed
// to the 8 XCDs round-robin, so workgroup b runs on XCD b % 8 and takes its
// units from that XCD's counter, over the XCD's contiguous share of the units
// (the same split xcd_item makes): neighbouring sub-grids still share an L2.
// Every workgroup leaves the loop once its XCD's counter has passed the end
// of the share, so the grid drains.
__global__ void queue_reset(uint32_t* q) {
    if (threadIdx.x < 8) q[threadIdx.x] = 0u;
}

template <bool RHO, int SPLIT, bool MIXED = false>
__global__ __launch_bounds__(64 * SPLIT) __attribute__((amdgpu_waves_per_eu(3))) void level_kernel_dqueue(LevelArgs a) {
    __shared__ int s_nbr[27];
    __shared__ int s_kind[27];
    __shared__ int s_unit;
    __shared__ double2 s_stage[SPLIT * kDirWave];
    const int n = 8 * a.nitems;                 // units: 8 coarse blocks per item
    const int x = blockIdx.x & 7;
    const int q = n >> 3, r = n & 7;
    const int lo = x * q + (x < r ? x : r), hi = lo + q + (x < r ? 1 : 0);
    for (;;) {
        if (threadIdx.x == 0) s_unit = lo + (int)atomicAdd(a.queue + x, 1u);
        __syncthreads();
        const int v = s_unit;
        if (v >= hi) break;                     // uniform
        const int2 it = a.items[a.item0 + (v >> 3)];
        if (threadIdx.x < 27) {
            const int nb = a.nbr[(size_t)it.x * 27 + threadIdx.x];
            s_nbr[threadIdx.x] = nb;
            s_kind[threadIdx.x] = nb >= 0 ? a.kind[nb] : -1;
        }
        __syncthreads();
        if (!(it.y & kItemLeaf))   // uniform per workgroup
            m2l_item_direct<RHO, SPLIT, MIXED>(a, it.x, it.y, s_nbr, s_kind, v & 7, s_stage, (int)(threadIdx.x >> 6));
        __syncthreads();   // the unit's LDS (images, tables, s_unit) is free again
    }
}

template <bool RHO, int SPLIT, bool MIXED>
void launch_dqueue(int nitems, hipStream_t st, const LevelArgs& la) {
    // workgroups the device holds at once (occupancy of this instantiation
    // times CUs), found once per process
    static const int capacity = [] {
        int dev = 0, per = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess &&
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, level_kernel_dqueue<RHO, SPLIT, MIXED>, 64 * SPLIT, 0) ==
                hipSuccess && per > 0)
            return per * prop.multiProcessorCount;
        return 256;
    }();
    const int units = 8 * nitems;
    int grid = std::min(units, capacity);
    grid = std::max(8, (grid + 7) & ~7);   // every XCD's counter has workgroups
    hipLaunchKernelGGL(queue_reset, dim3(1), dim3(64), 0, st, la.queue);
    hipLaunchKernelGGL((level_kernel_dqueue<RHO, SPLIT, MIXED>), dim3(grid), dim3(64 * SPLIT), 0, st, la);
}

template <bool RHO>
void launch_level(int variant, int nitems, hipStream_t st, const LevelArgs& la, bool mixed = false) {
    const int waves = variant % 100;
    const int parts = 8 / waves;
    const dim3 grid(nitems * parts), block(64 * waves);
    if (mixed) {
        switch (variant) {
        case 8: hipLaunchKernelGGL((level_kernel<RHO, 8, true>), grid, block, 0, st, la); break;
        case 4: hipLaunchKernelGGL((level_kernel<RHO, 4, true>), grid, block, 0, st, la); break;
        case 704:
            hipLaunchKernelGGL((level_kernel_dsplit<RHO, 4, true>), dim3(nitems * 8), dim3(256), 0, st, la);
            break;
        case 702:
            hipLaunchKernelGGL((level_kernel_dsplit<RHO, 2, true>), dim3(nitems * 8), dim3(128), 0, st, la);
            break;
        case 708:
            hipLaunchKernelGGL((level_kernel_dsplit<RHO, 8, true>), dim3(nitems * 8), dim3(512), 0, st, la);
            break;
        case 804: launch_dqueue<RHO, 4, true>(nitems, st, la); break;
        case 802: launch_dqueue<RHO, 2, true>(nitems, st, la); break;
        default: hipLaunchKernelGGL((level_kernel<RHO, 2, true>), grid, block, 0, st, la); break;
        }
        return;
    }
    switch (variant) {
    case 4: hipLaunchKernelGGL((level_kernel<RHO, 4>), grid, block, 0, st, la); break;
    case 2: hipLaunchKernelGGL((level_kernel<RHO, 2>), grid, block, 0, st, la); break;
    case 304: hipLaunchKernelGGL((level_kernel_direct<RHO, 4>), grid, block, 0, st, la); break;
    case 302: hipLaunchKernelGGL((level_kernel_direct<RHO, 2>), grid, block, 0, st, la); break;
    case 504:
        hipLaunchKernelGGL((level_kernel_split<RHO, 4>), dim3(nitems * 8), dim3(256), 0, st, la);
        break;
    case 704:
        if (la.parts > 1) {
            launch_wide_sums(nitems, st, la, RHO);
            launch_wide_reduce(nitems, st, la, RHO);
        }
        else
            hipLaunchKernelGGL((level_kernel_dsplit<RHO, 4>), dim3(nitems * 8), dim3(256), 0, st, la);
        break;
    case 702:
        hipLaunchKernelGGL((level_kernel_dsplit<RHO, 2>), dim3(nitems * 8), dim3(128), 0, st, la);
        break;
    case 708:
        hipLaunchKernelGGL((level_kernel_dsplit<RHO, 8>), dim3(nitems * 8), dim3(512), 0, st, la);
        break;
    case 804: launch_dqueue<RHO, 4, false>(nitems, st, la); break;
    case 802: launch_dqueue<RHO, 2, false>(nitems, st, la); break;
    default: hipLaunchKernelGGL((level_kernel<RHO, 8>), grid, block, 0, st, la); break;
    }
}

// Root sub-grid: every pair of its 512 cells except self and near offsets
// (kokkos_kernel.hpp:324-471).  Workgroup b takes half b & 1 of the cells, one
// per lane, over chunk b >> 1 of the partners, a row of 8 along z, whose records
// all lanes read from LDS.
template <bool RHO>
__device__ __forceinline__ void root_part(const RootArgs& a, int b, double2* s_rec) {
    const int chunk = b >> 1, t = (b & 1) * 256 + (int)threadIdx.x;
    const int px = chunk >> 3, py = chunk & 7;
    if (threadIdx.x < 96) {
        const int j = (int)threadIdx.x / 12, i = (int)threadIdx.x - 12 * j;
        s_rec[threadIdx.x] = reinterpret_cast<const double2*>(a.rec + (size_t)record_of_cell(px, py, j) * kRecDoubles)[i];
    }
    const int tx = t >> 6, ty = (t >> 3) & 7, tz = t & 7;
    const double* trec = a.rec + (size_t)record_of_cell(tx, ty, tz) * kRecDoubles;
    const double X0 = trec[kRecY], X1 = trec[kRecY + 1], X2 = trec[kRecY + 2];
    const int dx = px - tx, dy = py - ty;
    unsigned skip = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int dz = j - tz;
        const bool inbox = dx >= -5 && dx <= 5 && dy >= -5 && dy <= 5 && dz >= -5 && dz <= 5;
        if (inbox && a.tab->root_excluded[(dx + 5) * 121 + (dy + 5) * 11 + (dz + 5)]) skip |= 1u << j;
    }
    __syncthreads();
    Acc<RHO> s;
    acc_clear(s);
#pragma unroll 1
    for (int j = 0; j < 8; ++j) {
        if ((skip >> j) & 1u) continue;
        Rec r;
#pragma unroll
        for (int i = 0; i < 12; ++i) r.v[i] = s_rec[j * 12 + i];
        m2l_far_rec<RHO>(r, X0, X1, X2, s);
    }
    double f[kFolded], L[20], C[3];
    acc_fold<RHO>(s, trec, f);
    acc_finish<RHO>(f, L, C);
    double* o = a.partial + ((size_t)chunk * kCells + t) * kRecDoubles;
#pragma unroll
    for (int i = 0; i < 20; ++i) o[i] = L[i];
    o[20] = C[0];
    o[21] = C[1];
    o[22] = C[2];
}

template <bool RHO>
__global__ __launch_bounds__(256) void root_kernel(RootArgs a) {
    __shared__ double2 s_rec[96];
    root_part<RHO>(a, blockIdx.x, s_rec);
}

// What a whole-tree solve does between the staging of its coarsest levels and
// the chain of reductions from level to level, in one launch: the sums of the
// sums-first levels, the finest first, their p2m, and the root's pairs.  As
// kernels on branches of a graph they took 11, 27, 15 and 19 us, but ~8 us for
// each branch and join; in one launch 39 us.  With the small leaf levels in one
// launch as well a 329-sub-grid tree takes 95 us a solve in place of 124.
template <bool RHO, bool FULL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void tree_sums_kernel(TreeSums g) {
    __shared__ int s_nbr[27];
    __shared__ int s_kind[27];
    __shared__ double2 s_stage[4 * kDirWave];
    int b = blockIdx.x;
    for (int i = kStageLevels - 1; i >= 0; --i) {   // uniform
        const int n = g.sums[i];
        if (b < n) {
            wide_part<RHO>(g.a[i], xcd_item(b, n), s_nbr, s_kind, s_stage);
            return;
        }
        b -= n;
    }
    for (int i = kStageLevels - 1; i >= 0; --i) {
        const int n = g.packs[i];
        if (b < n) {
            p2m_pack<RHO, FULL>(g.a[i], xcd_item(b, n), s_stage);
            return;
        }
        b -= n;
    }
    root_part<RHO>(g.root, b, s_stage);
}

// One thread per output value (cell, component); the chunks are summed in
// chunk order, so the result does not depend on scheduling.  Sixteen chunks'
// loads are issued before their adds, so the thread waits on one round trip
// per sixteen chunks rather than one per chunk.
__global__ __launch_bounds__(256) void root_reduce(RootReduceArgs a) {
    const int gid = blockIdx.x * 256 + threadIdx.x;
    if (gid >= kCells * 23) return;
    const int t = gid / 23, c = gid - 23 * (gid / 23);
    const double* src = a.partial + (size_t)t * kRecDoubles + c;
    const size_t stride = (size_t)kCells * kRecDoubles;
    double s = 0.0;
    for (int q0 = 0; q0 < a.nchunks; q0 += 16) {
        double v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = q0 + i < a.nchunks ? src[(size_t)(q0 + i) * stride] : 0.0;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (q0 + i < a.nchunks) s += v[i];
    }
    if (c < 20)
        a.L[(size_t)t * 20 + c] = a.overwrite ? s : a.L[(size_t)t * 20 + c] + s;
    else if (a.rho)
        a.Lc[(size_t)t * 3 + (c - 20)] = s;
}

// Fill kernel used instead of hipMemsetAsync so the passes stay graph-safe.
// Dense FMA rate probe: 8 independent chains per lane, so the issue rate and
// not the FMA latency bounds it.  b < 1 keeps the chains bounded, away from
// overflow and denormals (they converge to c / (1 - b)).
template <typename T>
__global__ __launch_bounds__(256) void fma_rate_kernel(T* __restrict__ out, T b, T c, int iters) {
    T a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = (T)(threadIdx.x & 63) + (T)i;
#pragma unroll 4
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = fma(a[i], b, c);
    }
    T s = a[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) s += a[i];
    out[(size_t)blockIdx.x * 256 + threadIdx.x] = s;
}

__global__ void zero_fill(double* p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// Partial halo slots of a level plan (octofmm_partial_slot): a neighbour that
// hands over only some of its cells (grid::get_ilist_n_bnd order,
// multipole_interaction_interface.hpp:177,257, p2m_interaction_interface.hpp:142,239)
// becomes a full slot with zeros in every cell it did not hand over, which is
// what update_input's zero padding gives.  One block per such slot, from
// descriptors in device memory: it zeroes the slot, then writes each listed
// cell from its position in the handed-over arrays.  The host lists each cell
// once (its last occurrence), so no two threads write one cell.
struct PartialSlot {
    const double* M;        // [count][20] handed-over multipoles (non-leaf slot)
    const double* com;      // [count][3]
    const double* mon;      // [count]     (leaf slot)
    const int2* idx;        // [n] (cell, position in the handed-over arrays), each cell once
    int32_t slot;
    int32_t n;
    int32_t multipole;      // 1: multipoles and centres of mass, 0: monopoles
    int32_t pad;
};

__global__ __launch_bounds__(256) void scatter_slots(const PartialSlot* __restrict__ d, double* M, double* com,
    double* mon) {
    const PartialSlot e = d[blockIdx.x];
    const int t = threadIdx.x;
    double* Ms = M + (size_t)e.slot * kCells * 20;
    double* Cs = com + (size_t)e.slot * kCells * 3;
    double* ms = mon + (size_t)e.slot * kCells;
    if (e.multipole) {
        for (int i = t; i < kCells * 20; i += 256) Ms[i] = 0.0;
        for (int i = t; i < kCells * 3; i += 256) Cs[i] = 0.0;
    } else {
        for (int i = t; i < kCells; i += 256) ms[i] = 0.0;
    }
    __syncthreads();
    for (int i = t; i < e.n; i += 256) {
        const int2 q = e.idx[i];
        if (e.multipole) {
            const double* src = e.M + (size_t)q.y * 20;
#pragma unroll
            for (int c = 0; c < 20; ++c) Ms[q.x * 20 + c] = src[c];
            const double* sc = e.com + (size_t)q.y * 3;
            Cs[q.x * 3] = sc[0];
            Cs[q.x * 3 + 1] = sc[1];
            Cs[q.x * 3 + 2] = sc[2];
        } else {
            ms[q.x] = e.mon[q.y];
        }
    }
}

// Upward pass of one leaf: one wave, lane = coarse cell, whose 8 monopoles it
// sums about their centre of mass (for RHO, which it forms; DRHODT takes the
// stored ones) without meeting another lane.  The rows go through the wave's
// LDS (32 cells at a time) and leave as the runs of 4 cells they are in the
// parent, and for RHO the leaf cells' centres as the contiguous block they are,
// in 16-byte pieces.  Bound by what it moves, 28 KiB a leaf: 5568 leaves take 24
// us (6.5 TB/s, part of it from the caches), where 8 lanes per coarse cell, with
// seven times the instructions and stores of single doubles 24 bytes apart, took
// 43 to 54.
template <bool RHO>
__device__ __forceinline__ void m2m_leaf(const M2MArgs& a, int n, double* s_rows) {
    const int l = threadIdx.x & 63;
    const int ip = l >> 4, jp = (l >> 2) & 3, kp = l & 3;
    const auto* xb = as_const(a.xbase) + 3 * n;
    const int pn = as_const(a.parent)[n], oct = as_const(a.octant)[n];
    const size_t u0 = (size_t)n * kCells + ip * 128 + jp * 16 + kp * 2;
    double m[8];   // child (kx, ky, kz) at 4 kx + 2 ky + kz
#pragma unroll
    for (int q = 0; q < 4; ++q) load2(a.mon + u0 + (q >> 1) * 64 + (q & 1) * 8, m + 2 * q);
    if constexpr (RHO) {
        // the cells' centres: 192 pieces of two doubles for each pair of x planes
        double* com = a.com + (size_t)n * (kCells * 3);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            int first[2], step[2];
            double base[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int d = 2 * (l + 64 * j) + e, cell = d / 3, c = d - 3 * cell;
                first[e] = c == 0 ? cell >> 6 : c == 1 ? (cell >> 3) & 7 : cell & 7;
                step[e] = c == 0 ? 2 : 0;
                base[e] = c == 0 ? xb[0] : c == 1 ? xb[1] : xb[2];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const double2_a8 v = {cell_centre(base[0], first[0] + q * step[0], a.dx),
                    cell_centre(base[1], first[1] + q * step[1], a.dx)};
                __builtin_nontemporal_store(v, reinterpret_cast<double2_a8*>(com + 384 * q + 2 * (l + 64 * j)));
            }
        }
    }
    if (pn < 0) return;   // uniform
    const size_t pc = (size_t)pn * kCells + parent_cell(oct, ip, jp, kp);
    double B[20];
    if constexpr (RHO) {
        // the children's centres form a grid: their moments about Y by one axis
        // after the other, T[x][y^i z^j], from 2 weights per axis and power
        double d[3][2][4];   // axis, side, power
        const double mx0 = (m[0] + m[1]) + (m[2] + m[3]), mx1 = (m[4] + m[5]) + (m[6] + m[7]);
        const double my0 = (m[0] + m[1]) + (m[4] + m[5]), my1 = (m[2] + m[3]) + (m[6] + m[7]);
        const double mz0 = (m[0] + m[2]) + (m[4] + m[6]), mz1 = (m[1] + m[3]) + (m[5] + m[7]);
        const double mtot = mx0 + mx1;
        const double lo[3] = {mx0, my0, mz0}, hi[3] = {mx1, my1, mz1};
        const int at[3] = {2 * ip, 2 * jp, 2 * kp};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double c0 = cell_centre(xb[c], at[c], a.dx), c1 = cell_centre(xb[c], at[c] + 1, a.dx);
            const double Y = (c0 * lo[c] + c1 * hi[c]) / mtot;
            a.pcom[pc * 3 + c] = Y;
            d[c][0][1] = c0 - Y;
            d[c][1][1] = c1 - Y;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                d[c][k][2] = d[c][k][1] * d[c][k][1];
                d[c][k][3] = d[c][k][2] * d[c][k][1];
            }
        }
        double T[2][4][4];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            double Z[2][4];
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const double m0 = m[4 * x + 2 * y], m1 = m[4 * x + 2 * y + 1];
                Z[y][0] = m0 + m1;
#pragma unroll
                for (int j = 1; j < 4; ++j) Z[y][j] = fma(m1, d[2][1][j], m0 * d[2][0][j]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                T[x][0][j] = Z[0][j] + Z[1][j];
#pragma unroll
                for (int i = 1; i + j < 4; ++i) T[x][i][j] = fma(Z[1][j], d[1][1][i], Z[0][j] * d[1][0][i]);
            }
        }
        auto moment = [&](int h, int i, int j) -> double {
            return h == 0 ? T[0][i][j] + T[1][i][j] : fma(T[1][i][j], d[0][1][h], T[0][i][j] * d[0][0][h]);
        };
        auto moment_of = [&](int b, int c, int e) -> double {   // axes b, c, e (3: none)
            return moment((b == 0) + (c == 0) + (e == 0), (b == 1) + (c == 1) + (e == 1), (b == 2) + (c == 2) + (e == 2));
        };
        B[0] = moment(0, 0, 0);
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            B[1 + b] = moment_of(b, 3, 3);
#pragma unroll
            for (int c = b; c < 3; ++c) {
                B[tmap2(b, c)] = moment_of(b, c, 3);
#pragma unroll
                for (int e = c; e < 3; ++e) B[tmap3(b, c, e)] = moment_of(b, c, e);
            }
        }
    } else {
        double Y[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) Y[c] = a.pcom[pc * 3 + c];
#pragma unroll
        for (int j = 0; j < 20; ++j) B[j] = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            double X[6];   // the centres of a pair along z
            const double* src = a.com + (u0 + (q >> 1) * 64 + (q & 1) * 8) * 3;
#pragma unroll
            for (int k = 0; k < 3; ++k) load2(src + 2 * k, X + 2 * k);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const double dX[3] = {X[3 * k] - Y[0], X[3 * k + 1] - Y[1], X[3 * k + 2] - Y[2]};
                double S[20];
                monopole_shift(m[2 * q + k], dX, S);
#pragma unroll
                for (int j = 0; j < 20; ++j) B[j] += S[j];
            }
        }
    }
    double2* row = reinterpret_cast<double2*>(s_rows) + (l & 31) * 10;
    const double2* rows = reinterpret_cast<const double2*>(s_rows);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (h == 1) lds_wave_sync();   // the first half's rows are read before they are overwritten
        if ((l >> 5) == h) {
#pragma unroll
            for (int j = 0; j < 10; ++j) row[j] = make_double2(B[2 * j], B[2 * j + 1]);
        }
        lds_wave_sync();
#pragma unroll
        for (int i = 0; i < 5; ++i) {   // 32 rows x 10 pieces
            const int ch = l + 64 * i, r = 32 * h + ch / 10;
            const double2 v = rows[ch];
            double* dst = a.pM + ((size_t)pn * kCells + parent_cell(oct, r >> 4, (r >> 2) & 3, r & 3)) * 20 + 2 * (ch % 10);
            *reinterpret_cast<double2_a8*>(dst) = double2_a8{v.x, v.y};
        }
    }
}

// Upward pass of one level (grid::compute_multipoles, src/grid_fmm.cpp:1639-1803).
// The first workgroups take the leaves, four each (m2m_leaf).  Two workgroups
// take a refined node, one lane per child cell, 8 consecutive lanes per coarse
// cell: for RHO the 8 lanes form the coarse cell's mass and mass-weighted
// centre by a fixed butterfly, shift their child's multipole to it, and sum the
// shifted multipoles in child order through LDS, each lane summing and storing
// 2 or 3 components of the parent's cell.
template <bool RHO>
__global__ __launch_bounds__(256) void m2m_kernel(M2MArgs a) {
    __shared__ __attribute__((aligned(16))) double s_m2m[256 * 11];
    const int nb = (a.nleaf + 3) >> 2;
    if ((int)blockIdx.x < nb) {
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const int i = (int)blockIdx.x * 4 + wave;
        if (i < a.nleaf) m2m_leaf<RHO>(a, as_const(a.order)[i], s_m2m + wave * (32 * 20));
        return;
    }
    const int rest = (int)blockIdx.x - nb;
    const int n = as_const(a.order)[a.nleaf + (rest >> 1)];
    const int q = (((rest & 1) << 8) + (int)threadIdx.x) >> 3, ci = threadIdx.x & 7;
    const int ip = q >> 4, jp = (q >> 2) & 3, kp = q & 3;
    const int u = (2 * ip + (ci & 1)) * 64 + (2 * jp + ((ci >> 1) & 1)) * 8 + (2 * kp + ((ci >> 2) & 1));
    const int pn = a.parent[n];
    if (pn < 0) return;                        // uniform per node
    const int pc = parent_cell(a.octant[n], ip, jp, kp);
    double* Yp = a.pcom + ((size_t)pn * kCells + pc) * 3;
    double A[20];
    {
        const double2* src = reinterpret_cast<const double2*>(a.M + ((size_t)n * kCells + u) * 20);
#pragma unroll
        for (int j = 0; j < 10; ++j) {
            const double2 v = src[j];
            A[2 * j] = v.x;
            A[2 * j + 1] = v.y;
        }
    }
    const double* X = a.com + ((size_t)n * kCells + u) * 3;
    const double x0 = X[0], x1 = X[1], x2 = X[2];
    double Y[3];
    if constexpr (RHO) {
        const double mtot = sum8(A[0]);
        Y[0] = sum8(x0 * A[0]) / mtot;
        Y[1] = sum8(x1 * A[0]) / mtot;
        Y[2] = sum8(x2 * A[0]) / mtot;
        if (ci == 0) {
            Yp[0] = Y[0];
            Yp[1] = Y[1];
            Yp[2] = Y[2];
        }
    } else {
        Y[0] = Yp[0];
        Y[1] = Yp[1];
        Y[2] = Yp[2];
    }
    const double dX[3] = {x0 - Y[0], x1 - Y[1], x2 - Y[2]};
    double B[20];
    multipole_shift(A, dX, B);
    // the 8 children's shifted multipoles meet in the wave's LDS rows, 10
    // components at a time (11 doubles apart, so the 8 lanes reading one
    // component hit distinct banks; two passes of 10 halve the LDS a
    // workgroup holds, so 5 waves per SIMD fit instead of 3); lane ci of the
    // group sums components ci (and ci + 8) of each half over the children
    // in order and stores them, so the group writes the parent's 160-byte
    // row as consecutive doubles
    double* row = s_m2m + threadIdx.x * 11;
    const double* grp = s_m2m + (threadIdx.x & ~7) * 11;
    double* Mo = a.pM + ((size_t)pn * kCells + pc) * 20;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (h == 1) lds_wave_sync();   // the first half's rows are read before they are overwritten
#pragma unroll
        for (int j = 0; j < 10; ++j) row[j] = B[10 * h + j];
        lds_wave_sync();
#pragma unroll
        for (int j = ci; j < 10; j += 8) {
            double v = grp[j];
#pragma unroll
            for (int c = 1; c < 8; ++c) v += grp[c * 11 + j];
            Mo[10 * h + j] = v;
        }
    }
}


}   // namespace

// ===========================================================================
// Host side
// ===========================================================================
namespace {

constexpr int kRootChunks = 64;

// Work lists of p2m_kernel.  hdr: first row and number of rows of each pack;
// units: 8 per pack, ordinal * 64 + coarse cell, or -1; idx: per row (entry)
// and unit the partner coarse cell's first record, or -1; di: its offset.
struct P2mPacks {
    std::vector<int32_t> hdr, units, idx, di;
    int npacks() const { return (int)hdr.size() / 2; }
    // while they are made: one coarse cell of one item with n entries from
    // `first` on in rec and off, and the order of the units in the packs
    struct Unit {
        int32_t id, first, n;
    };
    std::vector<Unit> unit;
    std::vector<int32_t> rec, off, order;
    // room for any one item, so that a call with one makes them without allocating
    void reserve_one() {
        const size_t entries = (size_t)64 * kMaxDelta;
        hdr.reserve(2 * 8);
        units.reserve(64);
        idx.reserve(entries);
        di.reserve(entries);
        unit.reserve(64);
        rec.reserve(entries);
        off.reserve(entries);
        order.reserve(64);
    }
};

// The coarse cells of a sub-grid that reach into its neighbour in direction
// raw: (own coarse cell, offset, first record in the neighbour).
struct P2mReach {
    struct Hit {
        int16_t C, di, rec;
    };
    std::vector<Hit> by_raw[27];
};

void build_p2m_reach(const Tables& T, P2mReach& r) {
    for (int di = 0; di < T.ndelta; ++di) {
        if (!(T.farbits[di] | T.nearbits[di])) continue;
        for (int C = 0; C < 64; ++C) {
            const int px = (C >> 4) + T.delta[di][0], py = ((C >> 2) & 3) + T.delta[di][1], pz = (C & 3) + T.delta[di][2];
            const int raw = (px < 0 ? 0 : px < 4 ? 1 : 2) + 3 * (py < 0 ? 0 : py < 4 ? 1 : 2) +
                9 * (pz < 0 ? 0 : pz < 4 ? 1 : 2);
            if (raw != 13)
                r.by_raw[raw].push_back(
                    {(int16_t)C, (int16_t)di, (int16_t)(((px & 3) * 16 + (py & 3) * 4 + (pz & 3)) * 8)});
        }
    }
}

// refined(ordinal, raw): the slot of that item's neighbour where it is
// refined, else -1.  Units go to packs by falling length, in item order where
// equal, so a pack's 8 units are of like length and near each other.
template <typename F>
void build_p2m_packs(const P2mReach& reach, int nitems, F&& refined, P2mPacks& out) {
    std::vector<P2mPacks::Unit>& units = out.unit;
    std::vector<int32_t>&rec = out.rec, &di = out.off, &order = out.order;
    units.clear();
    rec.clear();
    di.clear();
    for (int o = 0; o < nitems; ++o) {
        int slot[27], count[64] = {}, at[64];
        for (int raw = 0; raw < 27; ++raw) {
            slot[raw] = raw == 13 ? -1 : refined(o, raw);
            if (slot[raw] < 0) continue;
            for (const P2mReach::Hit& h : reach.by_raw[raw]) ++count[h.C];
        }
        int end = (int)rec.size();
        for (int C = 0; C < 64; ++C) {
            at[C] = end;
            if (count[C] > 0) units.push_back({o * 64 + C, end, count[C]});
            end += count[C];
        }
        rec.resize(end);
        di.resize(end);
        for (int raw = 0; raw < 27; ++raw) {
            if (slot[raw] < 0) continue;
            for (const P2mReach::Hit& h : reach.by_raw[raw]) {
                rec[at[h.C]] = slot[raw] * kCells + h.rec;
                di[at[h.C]++] = h.di;
            }
        }
    }
    int end_of[kMaxDelta + 2] = {};   // counting sort: units of n entries lie before end_of[n]
    for (const P2mPacks::Unit& u : units) ++end_of[u.n];
    for (int n = kMaxDelta; n >= 0; --n) end_of[n] += end_of[n + 1];
    order.resize(units.size());
    for (size_t u = units.size(); u-- > 0;) order[--end_of[units[u].n]] = (int32_t)u;
    const size_t npacks = (units.size() + 7) / 8;
    out.hdr.resize(2 * npacks);
    int rows = 0;
    for (size_t p = 0; p < npacks; ++p) {
        out.hdr[2 * p] = rows;
        rows += out.hdr[2 * p + 1] = units[order[8 * p]].n;
    }
    out.units.assign(8 * npacks, -1);
    out.idx.assign((size_t)rows * 8, -1);
    out.di.assign((size_t)rows * 8, 0);
    for (size_t q = 0; q < order.size(); ++q) {
        const P2mPacks::Unit& u = units[order[q]];
        out.units[q] = u.id;
        const size_t first = (size_t)out.hdr[2 * (q / 8)] * 8 + q % 8;
        for (int e = 0; e < u.n; ++e) {
            out.idx[first + 8 * e] = rec[u.first + e];
            out.di[first + 8 * e] = di[u.first + e];
        }
    }
}
// record buffers end with a tail the direct-to-LDS staging may read into
// (one 16-byte pad chunk past the last record)
constexpr size_t kRecTailBytes = 4096;
// layout of the per-sub-grid workspace metadata (int32 words); the int2 work
// item comes first so it stays 8-byte aligned
constexpr int kMetaItems = 0;
constexpr int kMetaNbr = 2;
constexpr int kMetaKind = kMetaNbr + 27;
constexpr int kMetaSize = kMetaKind + 27;

// Most workgroups per coarse block of a one-target level (wide_parts)
constexpr int kWideMax = (kMaxDelta + 3) / 4;

// Device workspace of the per-sub-grid entry points: a 27-slot level (slot 0 the
// target sub-grid, packed_slot(d) its neighbour in direction d), the partial
// sums of the interaction kernels and the root kernel's chunk sums.  Every
// region starts on a 256-byte boundary of one block.
struct SubgridWorkspace {
    double* rec = nullptr;      // [27][512][24] + tail
    double* mon = nullptr;      // [27][512]
    double* com = nullptr;      // [512][3] a leaf target's centres
    double* wide = nullptr;     // [8][kWideMax][kFolded][64]
    double* partial = nullptr;  // [kRootChunks][512][24]
    double* p2m = nullptr;      // [512][8] p2m sums of a leaf target
    int32_t* meta = nullptr;    // kMetaSize
    int32_t* packs = nullptr;   // p2m work lists (kPackWords)
};

// p2m work lists of one leaf target, in words: hdr 2 x 8, units 64, then idx
// and di of at most 8 packs of kMaxDelta rows
constexpr int kPackHead = 16 + 64;
constexpr int kPackWords = kPackHead + 2 * 8 * 8 * kMaxDelta;

constexpr size_t ws_align(size_t n) { return (n + 255) & ~size_t(255); }
constexpr size_t kWsRec = 0;
constexpr size_t kWsMon = kWsRec + ws_align(sizeof(double) * 27 * kCells * kRecDoubles + kRecTailBytes);
constexpr size_t kWsCom = kWsMon + ws_align(sizeof(double) * 27 * kCells);
constexpr size_t kWsWide = kWsCom + ws_align(sizeof(double) * kCells * 3);
constexpr size_t kWsPartial = kWsWide + ws_align(sizeof(double) * 8 * kWideMax * kFolded * 64);
constexpr size_t kWsP2m = kWsPartial + ws_align(sizeof(double) * kRootChunks * kCells * kRecDoubles);
constexpr size_t kWsMeta = kWsP2m + ws_align(sizeof(double) * kCells * 8);
constexpr size_t kWsPacks = kWsMeta + ws_align(sizeof(int32_t) * kMetaSize);
constexpr size_t kWsBytes = kWsPacks + ws_align(sizeof(int32_t) * kPackWords);

SubgridWorkspace carve_workspace(char* base) {
    SubgridWorkspace w;
    w.rec = reinterpret_cast<double*>(base + kWsRec);
    w.mon = reinterpret_cast<double*>(base + kWsMon);
    w.com = reinterpret_cast<double*>(base + kWsCom);
    w.wide = reinterpret_cast<double*>(base + kWsWide);
    w.partial = reinterpret_cast<double*>(base + kWsPartial);
    w.p2m = reinterpret_cast<double*>(base + kWsP2m);
    w.meta = reinterpret_cast<int32_t*>(base + kWsMeta);
    w.packs = reinterpret_cast<int32_t*>(base + kWsPacks);
    return w;
}

}   // namespace

// Workspace of octofmm_compute_multipole_interactions_noalloc: one per-sub-grid
// workspace (kWsBytes, 12 MiB) in the code object's device memory, so that
// entry point never allocates.  Each GPU the library runs on holds its own
// copy until the process ends.  In host code `scratch` names a host-side
// stand-in, not a device address: host code uses only the address
// hipGetSymbolAddress returns for the current device (scratch_address).
static __device__ __align__(256) char scratch[kWsBytes];

namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_setup_mu;
char* g_scratch_ptr[kScratchDevices] = {};
// calls of the no-allocation entry point on one device share its scratch:
// they are serialised per device within the process
std::mutex g_scratch_call_mu[kScratchDevices];

// The device address of `scratch` on `device`, looked up once per device with
// that device current (the caller has made it current); null on failure.
char* scratch_address(int device) {
    if (device < 0 || device >= kScratchDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_setup_mu);
    if (!g_scratch_ptr[device]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        g_scratch_ptr[device] = static_cast<char*>(p);
    }
    return g_scratch_ptr[device];
}
}   // namespace

struct octofmm_context {
    int device = 0;
    double theta = 0.5;
    int flags = 0;                 // OCTOFMM_CHECK_FINITE
    Tables tab;
    Tables* d_tab = nullptr;
    hipStream_t stream = nullptr;
    std::string err;
    // per-sub-grid entry points: the device workspace (one allocation on the
    // first call) and the pinned memory, made at creation, that a call packs
    // its inputs into and gets its results from (the kernels read and write it
    // where it lies)
    SubgridWorkspace ws;
    char* d_ws = nullptr;
    char* d_scratch = nullptr;     // this device's `scratch` (set at creation)
    double* h_pin = nullptr;       // results [512][20], [512][3], the packed inputs, p2m work lists
    int reach = 0;                 // cells of a neighbour within the stencil's reach, per axis
    P2mReach p2m_reach;
    P2mPacks p2m_packs;            // work lists of a call
};

// doubles of the results at the front of the pinned memory, and the cells its
// packed inputs hold at most: the sub-grid and the halo within reach
constexpr size_t kPinOut = (size_t)kCells * 23;
static size_t pin_cells(const Tables& tab) {
    const size_t w = kInx + 4 * (size_t)tab.max_delta;
    return w * w * w;
}

struct octofmm_plan {
    octofmm_context* ctx = nullptr;
    int32_t nslots = 0, nitems = 0, type = 0, precision = 0, flags = 0;
    int32_t n_m2l = 0;             // items [0, n_m2l) are non-leaf, the rest leaf targets
    int32_t n_stage = 0;           // slots whose partner records some item reads
    int32_t stage_slots() const { return d_stage_list ? n_stage : nslots; }
    bool sums_first = false;       // whole-tree solve: level_kernel_wide and level_reduce launched apart
    int32_t* d_stage_list = nullptr;   // those slots, or null when all are read
    double dx = 0.0;
    const double* d_M = nullptr;
    const double* d_com = nullptr;
    const double* d_mon = nullptr;
    double* d_L = nullptr;
    double* d_Lc = nullptr;
    double* d_rec = nullptr;
    int32_t* d_nbr = nullptr;
    int32_t* d_kind = nullptr;
    int32_t* d_foff = nullptr;
    double* d_fxbase = nullptr;
    int2* d_items = nullptr;
    octofmm_plan_stats stats;
    int variant = 8;           // level-kernel variant (see kVariants)
    int32_t mixed_far_d2 = 4;
    std::vector<int2> h_items;     // the work items (host copy, for the tuning key)
    uint64_t* d_mixbits = nullptr;
    // mixed precision, lane mappings 3 and 7: the mixed-precision records and
    // the far schedule with the entries that stay FP64 (the first mix_n64) before
    // those evaluated in FP32 as a whole
    double* d_recm = nullptr;
    int32_t* d_mixorder = nullptr;
    int32_t mix_n64 = 0;
    uint32_t* d_queue = nullptr;   // per-XCD work counters of the persistent variants
    int32_t wide_parts = 0;        // variant 704 split further: workgroups per coarse block (0: not for this level)
    double* d_wide = nullptr;      // and their folded sums [n_m2l * 8 * wide_parts][kFolded][64] (behind d_rec)
    int32_t n_p2m = 0;             // leaf items with p2m: items [n_m2l, n_m2l + n_p2m)
    double* d_p2m_out = nullptr;   // their p2m sums [n_p2m][512][8], zeros where a cell has no p2m pair
    int32_t n_packs = 0;           // p2m work lists (P2mPacks): hdr, units, idx, di
    int32_t* d_packs = nullptr;    // (behind d_p2m_out)
    size_t packs_units = 0, packs_idx = 0, packs_di = 0;   // first words of the lists behind hdr
    int64_t mixed_far_pairs_by_offset = 0;   // FP32 far pairs under that rule
    int64_t mixed_far_pairs_by_pair = 0;     // and under the per-pair rule of mapping 0
    bool root = false;             // root sub-grid: root stencil over slot 0
    // set by a whole-tree plan: write final expansions (fused downward pass)
    bool l2l = false;
    const int32_t* t_parent = nullptr;
    const int32_t* t_octant = nullptr;
    const double* t_pL = nullptr;
    const double* t_pLc = nullptr;
    const double* t_pcom = nullptr;
    double* t_g = nullptr;
    double t_G = 1.0;
    int32_t t_correct_am = 1;
    double* d_partial = nullptr;   // root: per-chunk partial expansions
    int32_t leaf_rows = 1;         // whole-tree plans: 0 = leaf cells get g (and L_c) only
    // partial halo slots: rebuilt in the caller's slot rows before staging
    int32_t npartial = 0;
    PartialSlot* d_pslots = nullptr;
    int2* d_pidx = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    // a level with both kinds of items runs its leaf kernel on this stream,
    // forked after staging and joined before the pass ends
    hipStream_t side = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
};

namespace {

octofmm_status fail(octofmm_context* c, octofmm_status s, const char* fmt, ...) {
    if (c) {
        char buf[512];
        va_list ap;
        va_start(ap, fmt);
        std::vsnprintf(buf, sizeof(buf), fmt, ap);
        va_end(ap);
        c->err = buf;
    }
    return s;
}

#define HIPC(ctx, call)                                                                         \
    do {                                                                                        \
        hipError_t e_ = (call);                                                                 \
        if (e_ != hipSuccess)                                                                   \
            return fail((ctx), e_ == hipErrorOutOfMemory ? OCTOFMM_ERR_ALLOCATION : OCTOFMM_ERR_HIP, \
                "%s failed: %s", #call, hipGetErrorString(e_));                                 \
    } while (0)

int raw_of_flat(int f) { return f < 13 ? f : f + 1; }

// The per-sub-grid workspace of a context, allocated on its first call.
octofmm_status ensure_workspace(octofmm_context* c) {
    if (c->d_ws) return OCTOFMM_OK;
    HIPC(c, hipMalloc((void**)&c->d_ws, kWsBytes));
    c->ws = carve_workspace(c->d_ws);
    return OCTOFMM_OK;
}

bool check_neighbor(const octofmm_neighbor& nb, bool want_multipole) {
    if (nb.count < 0 || nb.count > kCells) return false;
    if (nb.count != kCells && nb.count > 0 && !nb.cells) return false;
    if (nb.cells)
        for (int i = 0; i < nb.count; ++i)
            if (nb.cells[i] < 0 || nb.cells[i] >= kCells) return false;
    (void)want_multipole;
    return true;
}

bool all_finite(const double* p, size_t n) {
    if (!p) return true;
    for (size_t i = 0; i < n; ++i)
        if (!std::isfinite(p[i])) return false;
    return true;
}

// OCTOFMM_CHECK_FINITE: the sub-grid's own arrays and every neighbour's.
octofmm_status check_finite_inputs(octofmm_context* c, const octofmm_subgrid* in, bool leaf_target) {
    if (!(c->flags & OCTOFMM_CHECK_FINITE)) return OCTOFMM_OK;
    if (!leaf_target && !all_finite(in->M, (size_t)kCells * 20))
        return fail(c, OCTOFMM_ERR_NONFINITE, "non-finite multipole in the sub-grid");
    if (!all_finite(in->com, (size_t)kCells * 3))
        return fail(c, OCTOFMM_ERR_NONFINITE, "non-finite centre of mass in the sub-grid");
    if (leaf_target && !all_finite(in->mon, kCells))
        return fail(c, OCTOFMM_ERR_NONFINITE, "non-finite monopole in the sub-grid");
    if (!std::isfinite(in->dx) || !std::isfinite(in->xbase[0]) || !std::isfinite(in->xbase[1]) ||
        !std::isfinite(in->xbase[2]))
        return fail(c, OCTOFMM_ERR_NONFINITE, "non-finite dx or xbase");
    for (int f = 0; f < 26; ++f) {
        const octofmm_neighbor& nb = in->neighbors[f];
        if (nb.kind == OCTOFMM_NEIGHBOR_EMPTY) continue;
        const size_t n = (size_t)nb.count;
        if (!all_finite(nb.M, n * 20) || !all_finite(nb.com, n * 3) || !all_finite(nb.mon, n))
            return fail(c, OCTOFMM_ERR_NONFINITE, "non-finite data in neighbour %d", f);
    }
    return OCTOFMM_OK;
}

// Packs one sub-grid descriptor into the context's pinned memory for
// stage_packed: the target's own arrays whole, of each neighbour the cells
// within the stencil's reach.  A partial halo contributes its listed cells
// (later entries win, as in update_input's loop over the list) and zeros
// elsewhere, which is what update_input's zero padding gives.
void pack_subgrid(octofmm_context* c, const octofmm_subgrid* in, bool leaf_target, bool root, int item_flags,
    PackedArgs& pa) {
    double* dst = c->h_pin + kPinOut;
    pa.src = dst;
    pa.reach = c->reach;
    pa.leaf_target = leaf_target ? 1 : 0;
    pa.item_flags = item_flags;
    pa.rho = in->type == OCTOFMM_RHO;
    pa.dx = in->dx;
    for (int k = 0; k < 3; ++k) pa.xbase[k] = in->xbase[k];
    pa.packs_n = 0;
    size_t at = 0;
    for (int sl = 0; sl < 27; ++sl) {
        pa.off[sl] = 0;
        pa.kind[sl] = -1;
    }
    if (leaf_target) {
        pa.kind[0] = OCTOFMM_SLOT_LEAF;
        std::memcpy(dst, in->mon, sizeof(double) * kCells);
        std::memcpy(dst + kCells, in->com, sizeof(double) * kCells * 3);
        at = (size_t)kCells * 4;
    } else {
        pa.kind[0] = OCTOFMM_SLOT_NONLEAF;
        std::memcpy(dst, in->M, sizeof(double) * kCells * 20);
        std::memcpy(dst + (size_t)kCells * 20, in->com, sizeof(double) * kCells * 3);
        at = (size_t)kCells * 23;
    }
    for (int f = 0; f < (root ? 0 : 26); ++f) {
        const octofmm_neighbor& nb = in->neighbors[f];
        const int raw = raw_of_flat(f), sl = packed_slot(raw);
        const bool multipole = nb.kind == OCTOFMM_NEIGHBOR_MULTIPOLE && nb.M && nb.com;
        const bool monopole = nb.kind == OCTOFMM_NEIGHBOR_MONOPOLE && nb.mon;
        if (!multipole && !monopole) continue;   // empty, or refined without data: the reference skips it
        pa.kind[sl] = multipole ? OCTOFMM_SLOT_NONLEAF : OCTOFMM_SLOT_LEAF;
        pa.off[sl] = (int32_t)at;
        int lo[3], n[3];
        packed_box(raw % 3 - 1, c->reach, lo[0], n[0]);
        packed_box(raw / 3 % 3 - 1, c->reach, lo[1], n[1]);
        packed_box(raw / 9 - 1, c->reach, lo[2], n[2]);
        const size_t ncell = (size_t)n[0] * n[1] * n[2];
        double* d0 = dst + at;
        double* d1 = d0 + ncell * 20;
        at += ncell * (multipole ? 23 : 1);
        if (nb.count == kCells && !nb.cells) {
            for (int x = lo[0]; x < lo[0] + n[0]; ++x)
                for (int y = lo[1]; y < lo[1] + n[1]; ++y) {
                    const size_t cell = (size_t)x * 64 + y * 8 + lo[2], nz = (size_t)n[2];
                    if (multipole) {
                        std::memcpy(d0, nb.M + cell * 20, sizeof(double) * 20 * nz);
                        std::memcpy(d1, nb.com + cell * 3, sizeof(double) * 3 * nz);
                        d0 += 20 * nz;
                        d1 += 3 * nz;
                    } else {
                        std::memcpy(d0, nb.mon + cell, sizeof(double) * nz);
                        d0 += nz;
                    }
                }
            continue;
        }
        int16_t last[kCells];
        for (int i = 0; i < kCells; ++i) last[i] = -1;
        for (int i = 0; i < nb.count; ++i) last[nb.cells[i]] = (int16_t)i;
        for (int x = lo[0]; x < lo[0] + n[0]; ++x)
            for (int y = lo[1]; y < lo[1] + n[1]; ++y)
                for (int z = lo[2]; z < lo[2] + n[2]; ++z) {
                    const int i = last[x * 64 + y * 8 + z];
                    if (!multipole) {
                        *d0++ = i >= 0 ? nb.mon[i] : 0.0;
                        continue;
                    }
                    for (int k = 0; k < 20; ++k) d0[k] = i >= 0 ? nb.M[(size_t)i * 20 + k] : 0.0;
                    for (int k = 0; k < 3; ++k) d1[k] = i >= 0 ? nb.com[(size_t)i * 3 + k] : 0.0;
                    d0 += 20;
                    d1 += 3;
                }
    }
}

// The p2m work lists of a packed leaf target, into the pinned memory behind
// the inputs: hdr, units, idx, di.  Returns the number of packs.
int pack_p2m(octofmm_context* c, PackedArgs& pa) {
    P2mPacks& pk = c->p2m_packs;
    build_p2m_packs(c->p2m_reach, 1,
        [&](int, int raw) { return pa.kind[packed_slot(raw)] == OCTOFMM_SLOT_NONLEAF ? packed_slot(raw) : -1; }, pk);
    int32_t* dst = reinterpret_cast<int32_t*>(c->h_pin + kPinOut + pin_cells(c->tab) * 23);
    std::copy(pk.hdr.begin(), pk.hdr.end(), dst);
    std::copy(pk.units.begin(), pk.units.end(), dst + 16);
    std::copy(pk.idx.begin(), pk.idx.end(), dst + kPackHead);
    std::copy(pk.di.begin(), pk.di.end(), dst + kPackHead + pk.idx.size());
    pa.packs_src = dst;
    pa.packs_n = kPackHead + 2 * (int)pk.idx.size();
    return pk.npacks();
}

// The kernels of one packed sub-grid on the context's stream: its interactions
// alone go to the results in the pinned memory.
octofmm_status launch_subgrid(octofmm_context* c, const SubgridWorkspace& w, PackedArgs& pa, bool root) {
    hipStream_t st = c->stream;
    const int npacks = (pa.item_flags & kItemP2M) ? pack_p2m(c, pa) : 0;
    const bool rho = pa.rho != 0;
    pa.rec = w.rec;
    pa.mon = w.mon;
    pa.com = w.com;
    pa.meta = w.meta;
    pa.packs = w.packs;
    pa.p2m = w.p2m;
    hipLaunchKernelGGL(stage_packed, dim3(root ? 4 : 27 * 4), dim3(256), 0, st, pa);
    HIPC(c, hipGetLastError());
    double* L = c->h_pin;
    double* Lc = c->h_pin + (size_t)kCells * 20;
    if (root) {
        RootArgs ra;
        ra.rec = w.rec;
        ra.tab = c->d_tab;
        ra.partial = w.partial;
        if (rho)
            hipLaunchKernelGGL(root_kernel<true>, dim3(kRootChunks * 2), dim3(256), 0, st, ra);
        else
            hipLaunchKernelGGL(root_kernel<false>, dim3(kRootChunks * 2), dim3(256), 0, st, ra);
        HIPC(c, hipGetLastError());
        RootReduceArgs rr;
        rr.partial = w.partial;
        rr.L = L;
        rr.Lc = Lc;
        rr.nchunks = kRootChunks;
        rr.rho = rho;
        rr.overwrite = 1;
        hipLaunchKernelGGL(root_reduce, dim3((kCells * 23 + 255) / 256), dim3(256), 0, st, rr);
        HIPC(c, hipGetLastError());
        return OCTOFMM_OK;
    }
    LevelArgs la;
    std::memset(&la, 0, sizeof(la));
    la.rec = w.rec;
    la.com = w.com;
    la.L = L;
    la.Lc = Lc;
    la.nbr = w.meta + kMetaNbr;
    la.kind = w.meta + kMetaKind;
    la.items = reinterpret_cast<const int2*>(w.meta + kMetaItems);
    la.tab = c->d_tab;
    la.parts = wide_parts(1, c->tab);
    la.wide_sums = w.wide;
    la.mon = w.mon;
    la.p2m_out = w.p2m;
    la.leaf0 = 0;
    la.p2m_hdr = w.packs;
    la.p2m_units = w.packs + 16;
    la.p2m_idx = w.packs + kPackHead;
    la.p2m_di = w.packs + kPackHead + (pa.packs_n - kPackHead) / 2;
    la.G = 1.0;
    la.leaf_rows = 1;
    la.overwrite = 1;
    la.nitems = 1;
    la.inv_dx = 1.0 / pa.dx;
    la.neg_inv_dx = -1.0 / pa.dx;
    if (pa.item_flags & kItemLeaf) {
        if (rho)
            launch_p2m<true>(npacks, st, la, c->tab);
        else
            launch_p2m<false>(npacks, st, la, c->tab);
        HIPC(c, hipGetLastError());
        if (rho)
            launch_leaf<true>(1, st, la, c->tab);
        else
            launch_leaf<false>(1, st, la, c->tab);
    } else if (rho) {
        launch_level<true>(704, 1, st, la);
    } else {
        launch_level<false>(704, 1, st, la);
    }
    HIPC(c, hipGetLastError());
    return OCTOFMM_OK;
}

// One per-sub-grid call through a workspace, synchronous: packs the inputs,
// runs the kernels and adds their results to the caller's L (the same single
// addition per component a device-side L += result makes); L_c is copied out
// when the call writes it.
octofmm_status run_subgrid(octofmm_context* c, const SubgridWorkspace& w, const octofmm_subgrid* in, bool leaf_target,
    bool root, int item_flags, double* L, double* L_c) {
    PackedArgs pa;
    pack_subgrid(c, in, leaf_target, root, item_flags, pa);
    const octofmm_status s = launch_subgrid(c, w, pa, root);
    const hipError_t e = hipStreamSynchronize(c->stream);   // also before an error leaves the pinned memory to the next call
    if (s != OCTOFMM_OK) return s;
    HIPC(c, e);
    const double* out = c->h_pin;
    if (leaf_target) {
        for (int i = 0; i < kCells; ++i)
            for (int k = 0; k < 4; ++k) L[i * 20 + k] += out[i * 20 + k];
    } else {
        for (int i = 0; i < kCells * 20; ++i) L[i] += out[i];
    }
    if (L_c) std::memcpy(L_c, out + (size_t)kCells * 20, sizeof(double) * kCells * 3);
    return OCTOFMM_OK;
}

}   // namespace

// ===========================================================================
// C-ABI
// ===========================================================================
extern "C" {

int32_t octofmm_abi_version(void) { return OCTOFMM_ABI_VERSION; }

const char* octofmm_status_string(octofmm_status s) {
    switch (s) {
    case OCTOFMM_OK: return "ok";
    case OCTOFMM_ERR_INVALID_ARGUMENT: return "invalid argument";
    case OCTOFMM_ERR_THETA: return "invalid theta / stencil";
    case OCTOFMM_ERR_NO_DEVICE: return "no HIP device";
    case OCTOFMM_ERR_HIP: return "HIP runtime error";
    case OCTOFMM_ERR_ALLOCATION: return "allocation failed";
    case OCTOFMM_ERR_SIZE: return "size not supported";
    case OCTOFMM_ERR_NONFINITE: return "non-finite input";
    }
    return "unknown status";
}

const char* octofmm_last_error(const octofmm_context* ctx) { return ctx ? ctx->err.c_str() : ""; }

octofmm_status octofmm_create(const octofmm_config* cfg, octofmm_context** out) {
    if (!cfg || !out) return OCTOFMM_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return OCTOFMM_ERR_NO_DEVICE;
    if (cfg->device < 0 || cfg->device >= n) return OCTOFMM_ERR_NO_DEVICE;
    octofmm_context* c = new octofmm_context();
    c->device = cfg->device;
    c->theta = cfg->theta;
    c->flags = cfg->flags;
    c->err.reserve(600);   // error texts (at most 511 characters) are stored without allocating
    char err[256];
    if (!build_tables(cfg->theta, c->tab, err, sizeof(err))) {
        delete c;
        return OCTOFMM_ERR_THETA;
    }
    if (hipSetDevice(c->device) != hipSuccess || hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
        hipHostMalloc((void**)&c->h_pin, sizeof(double) * (kPinOut + pin_cells(c->tab) * 23) + sizeof(int32_t) * kPackWords,
            hipHostMallocDefault) !=
            hipSuccess ||
        hipMalloc((void**)&c->d_tab, sizeof(Tables)) != hipSuccess ||
        hipMemcpy(c->d_tab, &c->tab, sizeof(Tables), hipMemcpyHostToDevice) != hipSuccess) {
        octofmm_destroy(c);
        return OCTOFMM_ERR_HIP;
    }
    c->reach = 2 * c->tab.max_delta;
    build_p2m_reach(c->tab, c->p2m_reach);
    c->p2m_packs.reserve_one();
    c->d_scratch = scratch_address(c->device);
    if (!c->d_scratch) {
        octofmm_destroy(c);
        return OCTOFMM_ERR_HIP;
    }
    *out = c;
    return OCTOFMM_OK;
}

octofmm_status octofmm_destroy(octofmm_context* c) {
    if (!c) return OCTOFMM_OK;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    (void)hipHostFree(c->h_pin);
    (void)hipFree(c->d_ws);
    (void)hipFree(c->d_tab);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return OCTOFMM_OK;
}

}   // extern "C"

// Argument checks of the multipole drop-ins; sets the item flags and the root
// choice of the call.
static octofmm_status check_multipole_call(octofmm_context* c, const octofmm_subgrid* in, double* L, double* L_c,
    int& flags, bool& root) {
    if (!in || !in->M || !in->com || !L) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "null input or output");
    if (in->type != OCTOFMM_RHO && in->type != OCTOFMM_DRHODT) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad type");
    if (in->type == OCTOFMM_RHO && !L_c) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "RHO needs L_c");
    root = in->use_root_stencil != 0;
    flags = 0;
    if (!root)
        for (int f = 0; f < 26; ++f) {
            const octofmm_neighbor& nb = in->neighbors[f];
            if (nb.kind < 0 || nb.kind > 2) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad neighbour kind %d", f);
            if (nb.kind != OCTOFMM_NEIGHBOR_EMPTY && !check_neighbor(nb, nb.kind == OCTOFMM_NEIGHBOR_MULTIPOLE))
                return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad neighbour %d", f);
            if (nb.kind == OCTOFMM_NEIGHBOR_MONOPOLE && nb.mon) flags |= kItemNear;
        }
    return check_finite_inputs(c, in, false);
}

extern "C" {

octofmm_status octofmm_compute_multipole_interactions(octofmm_context* c, const octofmm_subgrid* in,
    double* L, double* L_c) {
    if (!c) return OCTOFMM_ERR_INVALID_ARGUMENT;
    int flags = 0;
    bool root = false;
    octofmm_status s = check_multipole_call(c, in, L, L_c, flags, root);
    if (s != OCTOFMM_OK) return s;
    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    s = ensure_workspace(c);
    if (s != OCTOFMM_OK) return s;
    return run_subgrid(c, c->ws, in, false, root, flags, L, in->type == OCTOFMM_RHO ? L_c : nullptr);
}

// The same call with the workspace in `scratch` instead of the context's
// allocation: the same kernels, no device allocation.  What enters the result
// is written by this call first: the target, of each neighbour handed over the
// cells within the stencil's reach (partial halos expanded by the host, zeros
// in the cells they do not list) and the metadata; empty directions are marked
// absent, so what a previous call left in the scratch does not enter the result.
octofmm_status octofmm_compute_multipole_interactions_noalloc(octofmm_context* c, const octofmm_subgrid* in,
    double* L, double* L_c) {
    if (!c) return OCTOFMM_ERR_INVALID_ARGUMENT;
    int flags = 0;
    bool root = false;
    octofmm_status s = check_multipole_call(c, in, L, L_c, flags, root);
    if (s != OCTOFMM_OK) return s;
    if (!c->d_scratch) return fail(c, OCTOFMM_ERR_HIP, "no static workspace on device %d", c->device);
    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    std::lock_guard<std::mutex> lock(g_scratch_call_mu[c->device]);
    const SubgridWorkspace w = carve_workspace(c->d_scratch);
    return run_subgrid(c, w, in, false, root, flags, L, in->type == OCTOFMM_RHO ? L_c : nullptr);
}

octofmm_status octofmm_compute_monopole_interactions(octofmm_context* c, const octofmm_subgrid* in,
    int32_t contains_multipole_neighbor, double* L, double* L_c) {
    if (!c) return OCTOFMM_ERR_INVALID_ARGUMENT;
    if (!in || !in->mon || !in->com || !L) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "null input or output");
    if (in->type != OCTOFMM_RHO && in->type != OCTOFMM_DRHODT) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad type");
    const bool p2m = contains_multipole_neighbor != 0;
    if (in->type == OCTOFMM_RHO && p2m && !L_c) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "RHO with p2m needs L_c");
    for (int f = 0; f < 26; ++f) {
        const octofmm_neighbor& nb = in->neighbors[f];
        if (nb.kind < 0 || nb.kind > 2) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad neighbour kind %d", f);
        if (nb.kind != OCTOFMM_NEIGHBOR_EMPTY && !check_neighbor(nb, nb.kind == OCTOFMM_NEIGHBOR_MULTIPOLE))
            return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad neighbour %d", f);
    }
    octofmm_status s = check_finite_inputs(c, in, true);
    if (s != OCTOFMM_OK) return s;
    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    s = ensure_workspace(c);
    if (s != OCTOFMM_OK) return s;
    const int flags = kItemLeaf | (p2m ? kItemP2M : 0);
    return run_subgrid(c, c->ws, in, true, false, flags, L, in->type == OCTOFMM_RHO && p2m ? L_c : nullptr);
}

// ---------------------------------------------------------------------------
// Level plans
// ---------------------------------------------------------------------------
static void plan_free(octofmm_plan* p) {
    if (!p) return;
    if (p->gexec) (void)hipGraphExecDestroy(p->gexec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    if (p->ev_fork) (void)hipEventDestroy(p->ev_fork);
    if (p->ev_join) (void)hipEventDestroy(p->ev_join);
    if (p->side) (void)hipStreamDestroy(p->side);
    (void)hipFree(p->d_rec);
    (void)hipFree(p->d_nbr);
    (void)hipFree(p->d_kind);
    (void)hipFree(p->d_foff);
    (void)hipFree(p->d_fxbase);
    (void)hipFree(p->d_items);
    (void)hipFree(p->d_mixbits);
    (void)hipFree(p->d_recm);
    (void)hipFree(p->d_mixorder);
    (void)hipFree(p->d_queue);
    (void)hipFree(p->d_p2m_out);
    (void)hipFree(p->d_partial);
    (void)hipFree(p->d_pslots);
    (void)hipFree(p->d_pidx);
    (void)hipFree(p->d_stage_list);
    delete p;
}

// Stages the records of n <= kStageLevels plans in one launch.
static octofmm_status launch_stage(octofmm_context* c, hipStream_t st, octofmm_plan* const* plans, int n) {
    StageGroup g;
    int slots = 0;
    for (int i = 0; i < kStageLevels; ++i) {
        StageArgs& sa = g.a[i];
        const octofmm_plan* p = plans[i < n ? i : 0];
        sa.M = p->d_M;
        sa.com = p->d_com;
        sa.mon = p->d_mon;
        sa.kind = p->d_kind;
        sa.fxbase = p->d_fxbase;
        sa.foff = p->d_foff;
        sa.rec = p->d_rec;
        sa.recm = p->d_recm;
        sa.rho = p->type == OCTOFMM_RHO;
        sa.list = p->d_stage_list;
        sa.dx = p->dx;
        sa.nslots = i >= n ? 0 : p->stage_slots();
        slots += sa.nslots;
    }
    if (slots > 0) {
        hipLaunchKernelGGL(stage_records, dim3(slots * 4), dim3(256), 0, st, g);
        HIPC(c, hipGetLastError());
    }
    return OCTOFMM_OK;
}

static LevelArgs level_args(const octofmm_plan* p) {
    LevelArgs la;
    la.rec = p->d_rec;
    la.com = p->d_com;
    la.L = p->d_L;
    la.Lc = p->d_Lc;
    la.nbr = p->d_nbr;
    la.kind = p->d_kind;
    la.items = p->d_items;
    la.tab = p->ctx->d_tab;
    la.mixbits = p->d_mixbits;
    la.recm = p->d_recm;
    la.mixorder = p->d_mixorder;
    la.mix_n64 = p->mix_n64;
    la.queue = p->d_queue;
    la.parts = p->wide_parts;
    la.wide_sums = p->d_wide;
    la.mon = p->d_mon;
    la.p2m_out = p->d_p2m_out;
    la.parent = p->t_parent;
    la.octant = p->t_octant;
    la.pL = p->t_pL;
    la.pLc = p->t_pLc;
    la.pcom = p->t_pcom;
    la.g = p->t_g;
    la.G = p->t_G;
    la.l2l = p->l2l ? 1 : 0;
    la.correct_am = p->t_correct_am;
    la.leaf_rows = p->leaf_rows;
    la.overwrite = 0;
    la.xbase = p->d_fxbase;
    la.dx = p->dx;
    la.inv_dx = 1.0 / p->dx;
    la.neg_inv_dx = -1.0 / p->dx;
    la.nitems = p->n_m2l;
    la.item0 = 0;
    la.leaf0 = p->n_m2l;
    la.p2m_hdr = p->d_packs;
    la.p2m_units = p->d_packs + p->packs_units;
    la.p2m_idx = p->d_packs + p->packs_idx;
    la.p2m_di = p->d_packs + p->packs_di;
    return la;
}

static LevelArgs leaf_args(const octofmm_plan* p) {
    LevelArgs la = level_args(p);
    la.nitems = p->nitems - p->n_m2l;
    la.item0 = p->n_m2l;
    return la;
}

static RootArgs root_args(const octofmm_plan* p) {
    RootArgs ra;
    ra.rec = p->d_rec;
    ra.tab = p->ctx->d_tab;
    ra.partial = p->d_partial;
    return ra;
}

// stage_mask bit 0: stage the partner records; bit 1: the root kernel, or the
// level kernel over the multipole-target items (a sums-first level: what
// level_reduce does of it); bit 4: a sums-first level's level_kernel_wide,
// which goes before bit 1; bit 2: the leaf kernel over
// the monopole-target items; bit 3: the p2m kernel of the leaf items with
// refined neighbours, whose sums the leaf kernel reads (so bit 3 goes before
// bit 2, on the same stream or ordered before it).  Bits 1 and 2 write
// disjoint sub-grids.
static octofmm_status plan_launch(octofmm_plan* p, hipStream_t st, int stage_mask) {
    octofmm_context* c = p->ctx;
    if ((stage_mask & 1) && p->npartial > 0) {
        hipLaunchKernelGGL(scatter_slots, dim3(p->npartial), dim3(256), 0, st, p->d_pslots,
            const_cast<double*>(p->d_M), const_cast<double*>(p->d_com), const_cast<double*>(p->d_mon));
        HIPC(c, hipGetLastError());
    }
    if (stage_mask & 1) {
        const octofmm_status s = launch_stage(c, st, &p, 1);
        if (s != OCTOFMM_OK) return s;
    }
    if (p->root && (stage_mask & 2)) {
        const RootArgs ra = root_args(p);
        if (!p->sums_first) {   // else tree_sums_kernel ran its pairs
            if (p->type == OCTOFMM_RHO)
                hipLaunchKernelGGL(root_kernel<true>, dim3(kRootChunks * 2), dim3(256), 0, st, ra);
            else
                hipLaunchKernelGGL(root_kernel<false>, dim3(kRootChunks * 2), dim3(256), 0, st, ra);
        }
        HIPC(c, hipGetLastError());
        RootReduceArgs rr;
        rr.partial = p->d_partial;
        rr.L = p->d_L;
        rr.Lc = p->d_Lc;
        rr.nchunks = kRootChunks;
        rr.rho = p->type == OCTOFMM_RHO;
        rr.overwrite = p->l2l ? 1 : 0;
        hipLaunchKernelGGL(root_reduce, dim3((kCells * 23 + 255) / 256), dim3(256), 0, st, rr);
        HIPC(c, hipGetLastError());
    } else if (!p->root && (stage_mask & 30) && p->nitems > 0) {
        LevelArgs la = level_args(p);
        const bool rho = p->type == OCTOFMM_RHO;
        if ((stage_mask & 18) && p->n_m2l > 0) {
            if (p->sums_first) {
                if (stage_mask & 16) launch_wide_sums(p->n_m2l, st, la, rho);
                if (stage_mask & 2) launch_wide_reduce(p->n_m2l, st, la, rho);
            } else if (rho)
                launch_level<true>(p->variant, p->n_m2l, st, la, p->precision == OCTOFMM_PRECISION_MIXED);
            else
                launch_level<false>(p->variant, p->n_m2l, st, la, p->precision == OCTOFMM_PRECISION_MIXED);
            HIPC(c, hipGetLastError());
        }
        if ((stage_mask & 8) && p->n_p2m > 0) {
            // the leaf items with p2m lead the leaf items
            if (rho)
                launch_p2m<true>(p->n_packs, st, la, c->tab);
            else
                launch_p2m<false>(p->n_packs, st, la, c->tab);
            HIPC(c, hipGetLastError());
        }
        if ((stage_mask & 4) && p->nitems > p->n_m2l) {
            la = leaf_args(p);
            if (rho)
                launch_leaf<true>(la.nitems, st, la, c->tab);
            else
                launch_leaf<false>(la.nitems, st, la, c->tab);
            HIPC(c, hipGetLastError());
        }
    }
    return OCTOFMM_OK;
}

// The kernels of one pass over the masked stages.  A level with both kinds of
// items runs its leaf kernel (bit 2) on the plan's side stream, forked after
// the staging and joined back before returning: the two kernels write
// disjoint sub-grids, so the leaf kernel overlaps the multipole-target
// kernel instead of queueing behind it.
static bool plan_forks(const octofmm_plan* p, int mask) {
    return !p->root && p->n_m2l > 0 && p->nitems > p->n_m2l && (mask & 6) == 6;
}

static octofmm_status plan_fork_resources(octofmm_plan* p) {
    octofmm_context* c = p->ctx;
    if (p->side || !plan_forks(p, 15)) return OCTOFMM_OK;
    HIPC(c, hipStreamCreateWithFlags(&p->side, hipStreamNonBlocking));
    HIPC(c, hipEventCreateWithFlags(&p->ev_fork, hipEventDisableTiming));
    HIPC(c, hipEventCreateWithFlags(&p->ev_join, hipEventDisableTiming));
    return OCTOFMM_OK;
}

static octofmm_status plan_run(octofmm_plan* p, hipStream_t st, int mask) {
    octofmm_context* c = p->ctx;
    if (!plan_forks(p, mask) || !p->side) return plan_launch(p, st, mask);
    octofmm_status s = plan_launch(p, st, mask & 1);
    if (s != OCTOFMM_OK) return s;
    HIPC(c, hipEventRecord(p->ev_fork, st));
    HIPC(c, hipStreamWaitEvent(p->side, p->ev_fork, 0));
    s = plan_launch(p, p->side, mask & 12);
    if (s != OCTOFMM_OK) return s;
    s = plan_launch(p, st, 2);
    if (s != OCTOFMM_OK) return s;
    HIPC(c, hipEventRecord(p->ev_join, p->side));
    HIPC(c, hipStreamWaitEvent(st, p->ev_join, 0));
    return OCTOFMM_OK;
}

}   // extern "C"

// Kernel variants a plan may run: FP64 plans every variant, mixed-precision
// plans the mapping-0 forms (8, 4, 2 waves per workgroup; FP32 chosen per
// pair) and mapping 7 with its persistent form (704, 702, 708, 804, 802;
// FP32 chosen per coarse offset).
static bool variant_allowed(const octofmm_plan* p, int v) {
    bool known = false;
    for (int k : kVariants) known = known || k == v;
    const int mapping = v / 100;
    return known && !(p->precision == OCTOFMM_PRECISION_MIXED && mapping != 0 && mapping != 7 && mapping != 8);
}

// The plan's count of FP32 far pairs follows the chosen variant's rule.
static void set_mixed_count(octofmm_plan* p) {
    if (p->precision == OCTOFMM_PRECISION_MIXED)
        p->stats.mixed_far_pairs = p->variant >= 700 ? p->mixed_far_pairs_by_offset : p->mixed_far_pairs_by_pair;
}

// Tuning cache: the variant the autotuner chose, keyed by level shape (device
// architecture, solve type, precision, opening angle, counts of multipole-target
// items with and without a near pass, fused downward pass or not) and by the
// kernels the choice was timed on: the build gives their sources an id, so that
// entries a file holds from other kernels are passed over.  A plan of a
// shape seen before takes the cached choice without timing anything, so plans
// of one shape run the same kernel, and give the same bits, within a process.
// When the environment variable OCTOFMM_TUNE_CACHE names a file, the cache is
// read from it at the first lookup and every new choice is appended to it
// (one "key variant" line each), so the choices also hold across processes.
#ifndef OCTOFMM_KERNEL_ID
#define OCTOFMM_KERNEL_ID "0"
#endif
namespace {
std::mutex g_tune_mu;
std::vector<std::pair<std::string, int>> g_tune;
bool g_tune_loaded = false;

std::string tune_key(const octofmm_plan* p) {
    hipDeviceProp_t prop;
    const char* arch = hipGetDeviceProperties(&prop, p->ctx->device) == hipSuccess ? prop.gcnArchName : "unknown";
    int near = 0;
    for (const int2& it : p->h_items)
        if (!(it.y & kItemLeaf) && (it.y & kItemNear)) ++near;
    char buf[256];
    std::snprintf(buf, sizeof(buf), "%s/cu%d/t%d/p%d/d%d/th%.17g/m%d/n%d/l%d/k%s", arch,
        hipGetDeviceProperties(&prop, p->ctx->device) == hipSuccess ? prop.multiProcessorCount : 0, p->type,
        p->precision, p->precision == OCTOFMM_PRECISION_MIXED ? p->mixed_far_d2 : 0, p->ctx->theta, p->n_m2l, near,
        p->l2l ? 1 : 0, OCTOFMM_KERNEL_ID);
    for (char* q = buf; *q; ++q)
        if (*q == ' ') *q = '_';
    return buf;
}

// the variant cached for key, or 0
int tune_lookup(const std::string& key) {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    if (!g_tune_loaded) {
        g_tune_loaded = true;
        if (const char* path = std::getenv("OCTOFMM_TUNE_CACHE")) {
            if (FILE* f = std::fopen(path, "r")) {
                char k[256];
                int v = 0;
                while (std::fscanf(f, "%255s %d", k, &v) == 2) g_tune.emplace_back(k, v);
                std::fclose(f);
            }
        }
    }
    int v = 0;
    for (const auto& e : g_tune)
        if (e.first == key) v = e.second;   // the last entry of a key wins
    return v;
}

void tune_store(const std::string& key, int v) {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    g_tune.emplace_back(key, v);
    if (const char* path = std::getenv("OCTOFMM_TUNE_CACHE")) {
        if (FILE* f = std::fopen(path, "a")) {
            std::fprintf(f, "%s %d\n", key.c_str(), v);
            std::fclose(f);
        }
    }
}
}   // namespace

extern "C" {

// Times each level-kernel mapping on the live level's multipole-target items
// (the leaf kernel does not depend on it) and keeps the fastest.  The trial
// passes write into private scratch outputs, never the caller's L / L_c.
static octofmm_status plan_autotune_run(octofmm_plan* p);

static octofmm_status plan_autotune(octofmm_plan* p) {
    octofmm_context* c = p->ctx;
    double* userL = p->d_L;
    double* userLc = p->d_Lc;
    double *tL = nullptr, *tLc = nullptr;
    const size_t n = (size_t)p->nslots * kCells;
    if (hipMalloc((void**)&tL, n * 20 * sizeof(double)) != hipSuccess ||
        hipMalloc((void**)&tLc, n * 3 * sizeof(double)) != hipSuccess) {
        (void)hipFree(tL);
        return fail(c, OCTOFMM_ERR_ALLOCATION, "autotune scratch allocation failed");
    }
    p->d_L = tL;
    p->d_Lc = tLc;
    const octofmm_status s = plan_autotune_run(p);
    (void)hipStreamSynchronize(c->stream);
    p->d_L = userL;
    p->d_Lc = userLc;
    (void)hipFree(tL);
    (void)hipFree(tLc);
    return s;
}

static octofmm_status plan_autotune_run(octofmm_plan* p) {
    octofmm_context* c = p->ctx;
    hipStream_t st = c->stream;
    HIPC(c, hipStreamSynchronize(st));
    octofmm_status s = plan_launch(p, st, 1);
    if (s != OCTOFMM_OK) return s;
    hipEvent_t e0, e1;
    HIPC(c, hipEventCreate(&e0));
    HIPC(c, hipEventCreate(&e1));
    // Two rounds, the variants in list order and then in reverse, each
    // variant's times summed: the clock of a GPU that has just come out of
    // idle still rises over the first tens of milliseconds, which in one
    // round in list order favours the variants timed last.
    std::vector<std::pair<int, float>> timed;
    for (int w : kTunedVariants)
        if (variant_allowed(p, w)) timed.emplace_back(w, 0.f);
    const int nv = (int)timed.size();
    for (int round = 0; round < 2; ++round) {
        for (int i = 0; i < nv; ++i) {
            auto& t = timed[round == 0 ? i : nv - 1 - i];
            p->variant = t.first;
            s = plan_launch(p, st, 2);   // warm-up
            if (s != OCTOFMM_OK) return s;
            HIPC(c, hipEventRecord(e0, st));
            for (int l = 0; l < 3; ++l) {
                s = plan_launch(p, st, 2);
                if (s != OCTOFMM_OK) return s;
            }
            HIPC(c, hipEventRecord(e1, st));
            HIPC(c, hipEventSynchronize(e1));
            float ms = 0.f;
            HIPC(c, hipEventElapsedTime(&ms, e0, e1));
            t.second += ms;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    float best = 1e30f;
    int best_w = 8;
    for (const auto& t : timed) {
        if (t.second < best) {
            best = t.second;
            best_w = t.first;
        }
    }
    // Within 2% of the fastest the variant that re-reads the fewest bytes
    // from HBM wins (the timings of one plan creation spread by about 1%; in
    // interleaved A/B runs of 20 launches each on a 4096-sub-grid level,
    // 704 ran 1.3-1.8% faster than 702 every time, while the two-round
    // timing at plan creation still picked 702 in one process of six with a
    // 1% window): mapping 7 over 4 waves,
    // whose waves of one block stage overlapping neighbourhoods from one CU
    // at the same time (1.4x the algorithmic bytes on a 4096-sub-grid level,
    // 1.9x over 2 waves, 4.3x for mapping 3), then the other splits, mapping
    // 5, 3 and 0.
    auto rank = [](int w) {
        return w == 704 ? 0 : w / 100 == 7 ? 1 : w / 100 == 5 ? 2 : w / 100 == 3 ? 3 : 4;
    };
    float best_near = best;
    for (const auto& t : timed) {
        if (t.second > best * 1.02f) continue;
        if (rank(t.first) < rank(best_w) || (rank(t.first) == rank(best_w) && t.second < best_near)) {
            best_w = t.first;
            best_near = t.second;
        }
    }
    p->variant = best_w;
    return OCTOFMM_OK;
}

}   // extern "C"

// First half of level plan creation: checks, work items, pair counts, device
// tables.  The kernel variant and the graph come in level_plan_finish.
static octofmm_status level_plan_build(octofmm_context* c, const octofmm_level* lv, bool in_tree, octofmm_plan** out) {
    if (lv->nslots <= 0 || !lv->neighbors || !lv->kind || !lv->xbase || lv->ntargets < 0 ||
        (lv->ntargets > 0 && !lv->targets))
        return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad level description");
    if (!lv->d_M || !lv->d_com || !lv->d_mon || !lv->d_L || (lv->type == OCTOFMM_RHO && !lv->d_L_c))
        return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "null device array");
    if (lv->type != OCTOFMM_RHO && lv->type != OCTOFMM_DRHODT) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad type");
    if (lv->precision != OCTOFMM_PRECISION_FP64 && lv->precision != OCTOFMM_PRECISION_MIXED)
        return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad precision");
    if (!(lv->dx > 0.0)) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "dx must be positive");
    if ((size_t)lv->nslots * kCells * kRecDoubles * sizeof(double) >= ((size_t)1 << 40))
        return fail(c, OCTOFMM_ERR_SIZE, "level too large");
    const int ns = lv->nslots;
    for (int s = 0; s < ns; ++s) {
        if (lv->kind[s] != OCTOFMM_SLOT_NONLEAF && lv->kind[s] != OCTOFMM_SLOT_LEAF)
            return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad kind of slot %d", s);
        for (int r = 0; r < 27; ++r) {
            const int n = lv->neighbors[(size_t)s * 27 + r];
            if (n < -1 || n >= ns) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad neighbour of slot %d", s);
        }
        if (lv->neighbors[(size_t)s * 27 + 13] != s)
            return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "neighbour entry 13 of slot %d must be the slot", s);
    }
    const bool root = (lv->flags & OCTOFMM_PLAN_ROOT) != 0;
    if (root && (ns != 1 || lv->ntargets != 1 || lv->targets[0] != 0 || lv->kind[0] != OCTOFMM_SLOT_NONLEAF))
        return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "a root plan takes exactly one non-leaf slot as its target");
    // work items, heaviest kinds first: non-leaf with leaf neighbours, non-leaf,
    // leaf with refined neighbours, pure p2p leaves
    std::vector<int2> buckets[4];
    octofmm_plan_stats st;
    std::memset(&st, 0, sizeof(st));
    const Tables& T = c->tab;
    std::vector<char> seen(ns, 0);
    if (root) {
        // every pair of the root's cells except self and near offsets
        for (int t = 0; t < kCells; ++t)
            for (int q = 0; q < kCells; ++q) {
                const int dx = (q >> 6) - (t >> 6), dy = ((q >> 3) & 7) - ((t >> 3) & 7), dz = (q & 7) - (t & 7);
                const bool inbox = dx >= -5 && dx <= 5 && dy >= -5 && dy <= 5 && dz >= -5 && dz <= 5;
                if (inbox && T.root_excluded[(dx + 5) * 121 + (dy + 5) * 11 + (dz + 5)]) continue;
                st.far_pairs++;
            }
        st.n_m2l_items = 1;
    }
    for (int t = 0; t < (root ? 0 : lv->ntargets); ++t) {
        const int s = lv->targets[t];
        if (s < 0 || s >= ns) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad target %d", t);
        if (seen[s]) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "duplicate target slot %d", s);
        seen[s] = 1;
        bool has_leaf = false, has_nonleaf = false;
        for (int r = 0; r < 27; ++r) {
            if (r == 13) continue;
            const int n = lv->neighbors[(size_t)s * 27 + r];
            if (n < 0) continue;
            (lv->kind[n] == OCTOFMM_SLOT_LEAF ? has_leaf : has_nonleaf) = true;
        }
        if (lv->kind[s] == OCTOFMM_SLOT_NONLEAF) {
            buckets[has_leaf ? 0 : 1].push_back(make_int2(s, has_leaf ? kItemNear : 0));
            st.n_m2l_items++;
        } else {
            buckets[has_nonleaf ? 2 : 3].push_back(make_int2(s, kItemLeaf | (has_nonleaf ? kItemP2M : 0)));
            st.n_leaf_items++;
        }
    }
    // partial halo slots: each cell once, from its last entry (later entries
    // win, as in update_input's loop over the list)
    if (lv->npartial < 0 || (lv->npartial > 0 && !lv->partial))
        return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad partial halo list");
    if (root && lv->npartial > 0) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "a root plan has no halo");
    std::vector<PartialSlot> pslots;
    std::vector<size_t> poff;   // first (cell, position) pair of each partial slot in pidx
    std::vector<int2> pidx;
    {
        std::vector<char> listed(ns, 0);
        for (int q = 0; q < lv->npartial; ++q) {
            const octofmm_partial_slot& e = lv->partial[q];
            if (e.slot < 0 || e.slot >= ns) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad partial slot %d", q);
            if (seen[e.slot]) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "partial slot %d is a target", e.slot);
            if (listed[e.slot]) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "slot %d listed twice as partial", e.slot);
            listed[e.slot] = 1;
            if (e.count < 0 || e.count > kCells || (e.count > 0 && !e.cells))
                return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad cell list of partial slot %d", e.slot);
            const bool mp = lv->kind[e.slot] == OCTOFMM_SLOT_NONLEAF;
            if (e.count > 0 && (mp ? (!e.d_M || !e.d_com) : !e.d_mon))
                return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "null data of partial slot %d", e.slot);
            int last[kCells];
            for (int i = 0; i < kCells; ++i) last[i] = -1;
            for (int i = 0; i < e.count; ++i) {
                if (e.cells[i] < 0 || e.cells[i] >= kCells)
                    return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad cell in partial slot %d", e.slot);
                last[e.cells[i]] = i;
            }
            PartialSlot d;
            d.M = e.d_M;
            d.com = e.d_com;
            d.mon = e.d_mon;
            d.idx = nullptr;   // set once pidx is on the device
            poff.push_back(pidx.size());
            d.slot = e.slot;
            d.multipole = mp ? 1 : 0;
            d.pad = 0;
            d.n = 0;
            for (int cell = 0; cell < kCells; ++cell)
                if (last[cell] >= 0) {
                    pidx.push_back(make_int2(cell, last[cell]));
                    ++d.n;
                }
            pslots.push_back(d);
        }
    }
    // pair counts: per cell per coarse offset
    for (int b = 0; b < 4; ++b)
        for (const int2& it : buckets[b]) {
            const int s = it.x;
            for (int cx = 0; cx < 4; ++cx)
                for (int cy = 0; cy < 4; ++cy)
                    for (int cz = 0; cz < 4; ++cz)
                        for (int di = 0; di < T.ndelta; ++di) {
                            const int px = cx + T.delta[di][0], py = cy + T.delta[di][1], pz = cz + T.delta[di][2];
                            const int raw = (px < 0 ? 0 : px < 4 ? 1 : 2) + 3 * (py < 0 ? 0 : py < 4 ? 1 : 2) +
                                9 * (pz < 0 ? 0 : pz < 4 ? 1 : 2);
                            const int n = lv->neighbors[(size_t)s * 27 + raw];
                            if (n < 0) continue;
                            const int64_t nf = __builtin_popcountll(T.farbits[di]);
                            const int64_t nn = __builtin_popcountll(T.nearbits[di]);
                            if (!(it.y & kItemLeaf)) {
                                st.far_pairs += nf;
                                if (lv->kind[n] == OCTOFMM_SLOT_LEAF) st.near_pairs += nn;
                            } else if (lv->kind[n] == OCTOFMM_SLOT_LEAF) {
                                st.p2p_pairs += nf + nn;
                            } else if (it.y & kItemP2M) {
                                st.p2m_pairs += nf + nn;
                            }
                        }
        }
    const bool rho = lv->type == OCTOFMM_RHO;
    st.flops = st.far_pairs * (rho ? 407 : 273) + st.near_pairs * (rho ? 407 : 273) + st.p2p_pairs * 12 +
        st.p2m_pairs * (rho ? 318 : 205);
    std::vector<int2> items;
    for (int b = 0; b < 4; ++b) items.insert(items.end(), buckets[b].begin(), buckets[b].end());
    const int32_t n_m2l = (int32_t)(buckets[0].size() + buckets[1].size());
    // partner records are read by non-leaf targets (their own slot and every
    // neighbour) and by leaf targets with refined neighbours (those
    // neighbours); pure p2p leaves read monopoles directly
    std::vector<int32_t> stage_list;
    {
        std::vector<char> need(ns, 0);
        for (const int2& it : items) {
            const int32_t* nb = lv->neighbors + (size_t)it.x * 27;
            if (!(it.y & kItemLeaf)) {
                for (int r = 0; r < 27; ++r)
                    if (nb[r] >= 0) need[nb[r]] = 1;
            } else if (it.y & kItemP2M) {
                for (int r = 0; r < 27; ++r)
                    if (nb[r] >= 0 && lv->kind[nb[r]] == OCTOFMM_SLOT_NONLEAF) need[nb[r]] = 1;
            }
        }
        if (root) need[0] = 1;
        for (int s2 = 0; s2 < ns; ++s2)
            if (need[s2]) stage_list.push_back(s2);
    }

    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    octofmm_plan* p = new octofmm_plan();
    p->ctx = c;
    p->nslots = ns;
    p->nitems = (int32_t)items.size();
    p->n_m2l = n_m2l;
    p->n_stage = (int32_t)stage_list.size();
    p->type = lv->type;
    p->precision = lv->precision;
    p->flags = lv->flags;
    p->dx = lv->dx;
    p->d_M = lv->d_M;
    p->d_com = lv->d_com;
    p->d_mon = lv->d_mon;
    p->d_L = lv->d_L;
    p->d_Lc = lv->d_L_c;
    p->root = root;
    if (root) p->precision = OCTOFMM_PRECISION_FP64;
    p->stats = st;
    std::vector<int32_t> foff(3 * (size_t)ns, kInx);
    auto cleanup = [&](octofmm_status s, const char* what) {
        plan_free(p);
        return fail(c, s, "%s", what);
    };
    if (root && in_tree) p->sums_first = true;
    if (!root && p->precision == OCTOFMM_PRECISION_FP64) {
        // (a forced variant runs in a tree as it does in a level plan)
        if (in_tree && !std::getenv("OCTOFMM_VARIANT")) {
            p->wide_parts = sums_first_parts(n_m2l, T);
            p->sums_first = p->wide_parts > 0;
            if (p->sums_first) p->variant = 704;
        }
        if (!p->sums_first) p->wide_parts = wide_parts(n_m2l, T);
    }
    // the records and, behind them, the wide form's sums in one block
    const size_t rec_bytes = (size_t)ns * kCells * kRecDoubles * sizeof(double) + kRecTailBytes;
    if (hipMalloc((void**)&p->d_rec, rec_bytes + wide_bytes(n_m2l, p->wide_parts)) != hipSuccess)
        return cleanup(OCTOFMM_ERR_ALLOCATION, "record buffer allocation failed");
    static_assert(kRecTailBytes % sizeof(double) == 0);
    p->d_wide = p->d_rec + rec_bytes / sizeof(double);
    if (hipMalloc((void**)&p->d_nbr, sizeof(int32_t) * 27 * ns) != hipSuccess ||
        hipMalloc((void**)&p->d_kind, sizeof(int32_t) * ns) != hipSuccess ||
        hipMalloc((void**)&p->d_foff, sizeof(int32_t) * 3 * ns) != hipSuccess ||
        hipMalloc((void**)&p->d_fxbase, sizeof(double) * 3 * ns) != hipSuccess ||
        hipMalloc((void**)&p->d_items, sizeof(int2) * std::max<size_t>(1, items.size())) != hipSuccess)
        return cleanup(OCTOFMM_ERR_ALLOCATION, "plan table allocation failed");
    if (hipMemcpy(p->d_nbr, lv->neighbors, sizeof(int32_t) * 27 * ns, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->d_kind, lv->kind, sizeof(int32_t) * ns, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->d_foff, foff.data(), sizeof(int32_t) * 3 * ns, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->d_fxbase, lv->xbase, sizeof(double) * 3 * ns, hipMemcpyHostToDevice) != hipSuccess ||
        (!items.empty() &&
            hipMemcpy(p->d_items, items.data(), sizeof(int2) * items.size(), hipMemcpyHostToDevice) != hipSuccess))
        return cleanup(OCTOFMM_ERR_HIP, "plan table upload failed");
    if (root && hipMalloc((void**)&p->d_partial, sizeof(double) * kRootChunks * kCells * kRecDoubles) != hipSuccess)
        return cleanup(OCTOFMM_ERR_ALLOCATION, "root partial buffer allocation failed");
    if (!root && hipMalloc((void**)&p->d_queue, sizeof(uint32_t) * 8) != hipSuccess)
        return cleanup(OCTOFMM_ERR_ALLOCATION, "work counter allocation failed");
    p->n_p2m = (int32_t)buckets[2].size();
    if (p->n_p2m > 0) {
        const size_t bytes = sizeof(double) * (size_t)p->n_p2m * kCells * 8;
        P2mPacks pk;
        build_p2m_packs(c->p2m_reach, p->n_p2m,
            [&](int o, int raw) {
                const int n = lv->neighbors[(size_t)buckets[2][o].x * 27 + raw];
                return n >= 0 && lv->kind[n] == OCTOFMM_SLOT_NONLEAF ? n : -1;
            },
            pk);
        p->n_packs = pk.npacks();
        std::vector<int32_t> all(pk.hdr);
        p->packs_units = all.size();
        all.insert(all.end(), pk.units.begin(), pk.units.end());
        p->packs_idx = all.size();
        all.insert(all.end(), pk.idx.begin(), pk.idx.end());
        p->packs_di = all.size();
        if (!T.p2p_cube) all.insert(all.end(), pk.di.begin(), pk.di.end());
        if (hipMalloc((void**)&p->d_p2m_out, bytes + sizeof(int32_t) * all.size()) != hipSuccess)
            return cleanup(OCTOFMM_ERR_ALLOCATION, "p2m buffer allocation failed");
        p->d_packs = reinterpret_cast<int32_t*>(p->d_p2m_out + bytes / sizeof(double));
        if (hipMemset(p->d_p2m_out, 0, bytes) != hipSuccess ||
            hipMemcpy(p->d_packs, all.data(), sizeof(int32_t) * all.size(), hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(OCTOFMM_ERR_HIP, "p2m work list upload failed");
    }
    if (!pslots.empty()) {
        if (hipMalloc((void**)&p->d_pidx, sizeof(int2) * std::max<size_t>(1, pidx.size())) != hipSuccess ||
            hipMalloc((void**)&p->d_pslots, sizeof(PartialSlot) * pslots.size()) != hipSuccess)
            return cleanup(OCTOFMM_ERR_ALLOCATION, "partial halo table allocation failed");
        for (size_t q = 0; q < pslots.size(); ++q) pslots[q].idx = p->d_pidx + poff[q];
        if ((!pidx.empty() &&
                hipMemcpy(p->d_pidx, pidx.data(), sizeof(int2) * pidx.size(), hipMemcpyHostToDevice) != hipSuccess) ||
            hipMemcpy(p->d_pslots, pslots.data(), sizeof(PartialSlot) * pslots.size(), hipMemcpyHostToDevice) !=
                hipSuccess)
            return cleanup(OCTOFMM_ERR_HIP, "partial halo table upload failed");
        p->npartial = (int32_t)pslots.size();
    }
    if ((int)stage_list.size() < ns) {
        if (hipMalloc((void**)&p->d_stage_list, sizeof(int32_t) * std::max<size_t>(1, stage_list.size())) != hipSuccess ||
            (!stage_list.empty() && hipMemcpy(p->d_stage_list, stage_list.data(), sizeof(int32_t) * stage_list.size(),
                                        hipMemcpyHostToDevice) != hipSuccess))
            return cleanup(OCTOFMM_ERR_ALLOCATION, "staging list upload failed");
    }
    if (p->precision == OCTOFMM_PRECISION_MIXED) {
        // far pairs with |d|^2 > mixed_far_d2 (cell units) are evaluated in FP32
        std::vector<uint64_t> mb(T.ndelta > 0 ? T.ndelta : 1, 0);
        for (int di = 0; di < T.ndelta; ++di)
            for (int k = 0; k < 8; ++k)
                for (int j = 0; j < 8; ++j) {
                    const int bit = 8 * k + j;
                    if (!((T.farbits[di] >> bit) & 1)) continue;
                    const int dx = 2 * T.delta[di][0] + ((j >> 2) & 1) - ((k >> 2) & 1);
                    const int dy = 2 * T.delta[di][1] + ((j >> 1) & 1) - ((k >> 1) & 1);
                    const int dz = 2 * T.delta[di][2] + (j & 1) - (k & 1);
                    if (dx * dx + dy * dy + dz * dz > lv->mixed_far_d2) mb[di] |= uint64_t(1) << bit;
                }
        if (hipMalloc((void**)&p->d_mixbits, sizeof(uint64_t) * mb.size()) != hipSuccess ||
            hipMemcpy(p->d_mixbits, mb.data(), sizeof(uint64_t) * mb.size(), hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(OCTOFMM_ERR_ALLOCATION, "mixed-precision table upload failed");
        // lane mappings 3 and 7 choose the precision per far coarse offset:
        // FP32 where every far pair of the offset is an FP32 pair above.  The
        // split entries of opposite face offsets stage FP64 records only, so
        // their offsets stay FP64 (at mixed_far_d2 >= 4 they hold |d| = 2
        // pairs and would anyway)
        std::vector<int32_t> order, fp32;
        std::vector<char> whole(T.ndelta > 0 ? T.ndelta : 1, 0);
        for (int q = 0; q < T.nsched; ++q) {
            const int di = T.sched[q] & 0xff;
            const bool w = ((T.sched[q] >> 16) & 0xff) == 0 && T.farbits[di] != 0 && mb[di] == T.farbits[di];
            if (w) whole[di] = 1;
            (w ? fp32 : order).push_back(q);
        }
        p->mix_n64 = (int32_t)order.size();
        order.insert(order.end(), fp32.begin(), fp32.end());
        if (order.empty()) order.push_back(0);
        if (hipMalloc((void**)&p->d_mixorder, sizeof(int32_t) * order.size()) != hipSuccess ||
            hipMemcpy(p->d_mixorder, order.data(), sizeof(int32_t) * order.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMalloc((void**)&p->d_recm, (size_t)ns * kCells * kRecDoubles * sizeof(double) + kRecTailBytes) !=
                hipSuccess)
            return cleanup(OCTOFMM_ERR_ALLOCATION, "mixed-precision record allocation failed");
        // FP32 pair counts under both rules, summed over the M2L items
        p->mixed_far_pairs_by_pair = 0;
        p->mixed_far_pairs_by_offset = 0;
        for (const int2& it : items) {
            if (it.y & kItemLeaf) continue;
            for (int cx = 0; cx < 4; ++cx)
                for (int cy = 0; cy < 4; ++cy)
                    for (int cz = 0; cz < 4; ++cz)
                        for (int di = 0; di < T.ndelta; ++di) {
                            const int px = cx + T.delta[di][0], py = cy + T.delta[di][1], pz = cz + T.delta[di][2];
                            const int raw = (px < 0 ? 0 : px < 4 ? 1 : 2) + 3 * (py < 0 ? 0 : py < 4 ? 1 : 2) +
                                9 * (pz < 0 ? 0 : pz < 4 ? 1 : 2);
                            if (lv->neighbors[(size_t)it.x * 27 + raw] < 0) continue;
                            p->mixed_far_pairs_by_pair += __builtin_popcountll(mb[di]);
                            if (whole[di]) p->mixed_far_pairs_by_offset += __builtin_popcountll(T.farbits[di]);
                        }
        }
        set_mixed_count(p);
    }
    p->mixed_far_d2 = lv->mixed_far_d2;
    p->h_items = items;
    *out = p;
    return OCTOFMM_OK;
}

// Second half of plan creation, once the plan's epilogue is wired: the kernel
// variant (OCTOFMM_VARIANT, else with OCTOFMM_PLAN_AUTOTUNE the tuning cache
// or a timing of every variant on the live level, else the default) and, with
// OCTOFMM_PLAN_USE_GRAPH, the captured graph.  Frees the plan on failure.
static octofmm_status level_plan_finish(octofmm_plan* p, int flags) {
    octofmm_context* c = p->ctx;
    const char* forced = std::getenv("OCTOFMM_VARIANT");
    const bool forced_ok = forced && variant_allowed(p, std::atoi(forced));
    if (forced_ok) {
        p->variant = std::atoi(forced);
    } else if ((flags & OCTOFMM_PLAN_AUTOTUNE) && p->n_m2l > 0 && !p->root) {
        const std::string key = tune_key(p);
        const int cached = tune_lookup(key);
        if (cached && variant_allowed(p, cached)) {
            p->variant = cached;
        } else {
            // time each workgroup shape on the live level (outputs are scratch
            // here: the caller zeroes L before a real pass) and keep the fastest
            const octofmm_status ts = plan_autotune(p);
            if (ts != OCTOFMM_OK) {
                plan_free(p);
                return ts;
            }
            tune_store(key, p->variant);
        }
    }
    p->stats.variant = p->variant;
    set_mixed_count(p);
    if (flags & OCTOFMM_PLAN_USE_GRAPH) {
        // the side stream must exist before the capture starts
        octofmm_status fs = plan_fork_resources(p);
        if (fs != OCTOFMM_OK) {
            plan_free(p);
            return fs;
        }
        hipStream_t cs = c->stream;
        if (hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) != hipSuccess) {
            plan_free(p);
            return fail(c, OCTOFMM_ERR_HIP, "graph capture failed to start");
        }
        octofmm_status ls = plan_run(p, cs, 15);
        hipGraph_t g = nullptr;
        const hipError_t ee = hipStreamEndCapture(cs, &g);
        if (ls != OCTOFMM_OK || ee != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            plan_free(p);
            return fail(c, OCTOFMM_ERR_HIP, "graph capture failed");
        }
        p->graph = g;
        if (hipGraphInstantiate(&p->gexec, g, nullptr, nullptr, 0) != hipSuccess) {
            plan_free(p);
            return fail(c, OCTOFMM_ERR_HIP, "graph instantiation failed");
        }
    }
    return OCTOFMM_OK;
}

extern "C" {

octofmm_status octofmm_level_plan_create(octofmm_context* c, const octofmm_level* lv, octofmm_plan** out) {
    if (!c) return OCTOFMM_ERR_INVALID_ARGUMENT;
    if (!lv || !out) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "null level or plan");
    *out = nullptr;
    octofmm_plan* p = nullptr;
    octofmm_status s = level_plan_build(c, lv, false, &p);
    if (s != OCTOFMM_OK) return s;
    s = level_plan_finish(p, lv->flags);
    if (s != OCTOFMM_OK) return s;
    *out = p;
    return OCTOFMM_OK;
}

octofmm_status octofmm_level_plan_execute(octofmm_plan* p, void* stream) {
    if (!p) return OCTOFMM_ERR_INVALID_ARGUMENT;
    octofmm_context* c = p->ctx;
    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (p->gexec) {
        HIPC(c, hipGraphLaunch(p->gexec, st));
        return OCTOFMM_OK;
    }
    const octofmm_status fs = plan_fork_resources(p);   // first eager execute
    if (fs != OCTOFMM_OK) return fs;
    return plan_run(p, st, 15);
}

octofmm_status octofmm_level_plan_stats(const octofmm_plan* p, octofmm_plan_stats* s) {
    if (!p || !s) return OCTOFMM_ERR_INVALID_ARGUMENT;
    *s = p->stats;
    return OCTOFMM_OK;
}

octofmm_status octofmm_level_plan_time_stages(octofmm_plan* p, void* stream, int32_t iters, double* ms) {
    if (!p || !ms || iters <= 0) return OCTOFMM_ERR_INVALID_ARGUMENT;
    octofmm_context* c = p->ctx;
    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const octofmm_status fs = plan_fork_resources(p);
    if (fs != OCTOFMM_OK) return fs;
    hipEvent_t e0, e1;
    HIPC(c, hipEventCreate(&e0));
    HIPC(c, hipEventCreate(&e1));
    for (int stage = 0; stage < 2; ++stage) {
        HIPC(c, hipEventRecord(e0, st));
        for (int i = 0; i < iters; ++i) {
            octofmm_status s = plan_run(p, st, stage == 0 ? 1 : 14);
            if (s != OCTOFMM_OK) return s;
        }
        HIPC(c, hipEventRecord(e1, st));
        HIPC(c, hipEventSynchronize(e1));
        float f = 0.f;
        HIPC(c, hipEventElapsedTime(&f, e0, e1));
        ms[stage] = (double)f / iters;
    }
    ms[2] = 0.0;   // write-back is fused into the interaction kernel
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return OCTOFMM_OK;
}

octofmm_status octofmm_level_plan_destroy(octofmm_plan* p) {
    if (!p) return OCTOFMM_OK;
    (void)hipSetDevice(p->ctx->device);
    plan_free(p);
    return OCTOFMM_OK;
}


}   // extern "C"

// ---------------------------------------------------------------------------
// Whole-tree solve
// ---------------------------------------------------------------------------
struct octofmm_tree_plan {
    struct Level {
        int32_t nnodes = 0;
        double dx = 0.0;
        double* M = nullptr;
        double* com = nullptr;
        const double* mon = nullptr;
        double* L = nullptr;
        double* Lc = nullptr;
        double* g = nullptr;
        double* d_xbase = nullptr;    // the node tables: one block
        int32_t* d_kind = nullptr;
        int32_t* d_parent = nullptr;
        int32_t* d_octant = nullptr;
        int32_t* d_order = nullptr;   // the leaves, then the refined nodes
        int32_t nleaf = 0;
        octofmm_plan* plan = nullptr;
    };
    octofmm_context* ctx = nullptr;
    std::vector<Level> lv;
    int32_t type = 0, flags = 0, correct_am = 1;
    double G = 1.0;
    octofmm_tree_stats stats;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    // the interactions phase forks onto two more streams: [0] stages the larger
    // levels, [1] runs their p2m and the leaf kernels
    hipStream_t side[2] = {nullptr, nullptr};
    hipEvent_t ev_up = nullptr, ev_join[2] = {nullptr, nullptr};
    std::vector<hipEvent_t> ev_stage, ev_level, ev_sums, ev_p2m;
};

namespace {

void tree_free(octofmm_tree_plan* t) {
    if (!t) return;
    if (t->gexec) (void)hipGraphExecDestroy(t->gexec);
    if (t->graph) (void)hipGraphDestroy(t->graph);
    for (hipEvent_t e : {t->ev_up, t->ev_join[0], t->ev_join[1]})
        if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : t->ev_stage)
        if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : t->ev_level)
        if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : t->ev_sums)
        if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : t->ev_p2m)
        if (e) (void)hipEventDestroy(e);
    for (hipStream_t s : t->side)
        if (s) (void)hipStreamDestroy(s);
    for (auto& l : t->lv) {
        plan_free(l.plan);
        (void)hipFree(l.d_xbase);   // and the tables behind it
    }
    delete t;
}

// The sums, p2m and root pairs of the n coarsest levels.
void launch_tree_sums(octofmm_plan* const* plans, int n, hipStream_t st, bool rho, const Tables& tab) {
    TreeSums g;
    int blocks = 0;
    std::memset(&g, 0, sizeof(g));
    for (int i = 0; i < n; ++i) {
        const octofmm_plan* p = plans[i];
        if (p->root) {
            g.root = root_args(p);
            blocks += kRootChunks * 2;
            continue;
        }
        g.a[i] = level_args(p);
        g.sums[i] = p->sums_first ? p->n_m2l * 8 * p->wide_parts : 0;
        g.packs[i] = p->n_packs;
        blocks += g.sums[i] + g.packs[i];
    }
    if (blocks == 0) return;
    if (rho && tab.p2p_cube)
        hipLaunchKernelGGL((tree_sums_kernel<true, true>), dim3(blocks), dim3(256), 0, st, g);
    else if (rho)
        hipLaunchKernelGGL((tree_sums_kernel<true, false>), dim3(blocks), dim3(256), 0, st, g);
    else if (tab.p2p_cube)
        hipLaunchKernelGGL((tree_sums_kernel<false, true>), dim3(blocks), dim3(256), 0, st, g);
    else
        hipLaunchKernelGGL((tree_sums_kernel<false, false>), dim3(blocks), dim3(256), 0, st, g);
}

// The leaf items of n levels (one, but at theta 0.5).
octofmm_status launch_leaves(octofmm_tree_plan* t, const int* levels, int n, hipStream_t st) {
    octofmm_context* c = t->ctx;
    const bool rho = t->type == OCTOFMM_RHO;
    LevelArgs la[kLeafLevels];
    for (int i = 0; i < n; ++i) la[i] = leaf_args(t->lv[levels[i]].plan);
    if (!c->tab.p2p_cube) {
        if (rho)
            launch_leaf<true>(la[0].nitems, st, la[0], c->tab);
        else
            launch_leaf<false>(la[0].nitems, st, la[0], c->tab);
    } else if (rho) {
        launch_leaf_cube<true>(la, n, st);
    } else {
        launch_leaf_cube<false>(la, n, st);
    }
    HIPC(c, hipGetLastError());
    return OCTOFMM_OK;
}

// phase bit 0: upward pass; bit 1: interactions with the fused downward pass
octofmm_status tree_launch(octofmm_tree_plan* t, hipStream_t st, int phases) {
    octofmm_context* c = t->ctx;
    const int nl = (int)t->lv.size();
    if (phases & 1)
        for (int l = nl - 1; l >= 0; --l) {
            const auto& L = t->lv[l];
            if (l == 0 && t->lv[0].plan && t->lv[0].plan->root) continue;   // a refined root has no parent to sum into
            M2MArgs a;
            a.M = L.M;
            a.com = L.com;
            a.mon = L.mon;
            a.parent = L.d_parent;
            a.octant = L.d_octant;
            a.xbase = L.d_xbase;
            a.pM = l > 0 ? t->lv[l - 1].M : nullptr;
            a.pcom = l > 0 ? t->lv[l - 1].com : nullptr;
            a.dx = L.dx;
            a.order = L.d_order;
            a.nleaf = L.nleaf;
            const dim3 grid((L.nleaf + 3) / 4 + 2 * (L.nnodes - L.nleaf));
            if (t->type == OCTOFMM_RHO)
                hipLaunchKernelGGL(m2m_kernel<true>, grid, dim3(256), 0, st, a);
            else
                hipLaunchKernelGGL(m2m_kernel<false>, grid, dim3(256), 0, st, a);
            HIPC(c, hipGetLastError());
        }
    // Interactions of every level.  Each level's kernels also write the final
    // expansions (the downward pass is fused into them), so both kernels of
    // level l read the finished non-leaf sub-grids of level l - 1, which only
    // the level kernel of l - 1 writes.
    //
    // The coarsest levels, as many as one round of workgroups stages, are a
    // chain of few and small launches on the caller's stream: their staging in
    // one, their sums and p2m and the root's pairs in one (tree_sums_kernel), a
    // reduction per level, and small leaf levels with the next one's.  One
    // launch follows another there within a microsecond, where a branch and its
    // join cost about eight.  Larger levels are staged on a second stream; on a third
    // their p2m runs ahead of all that waits for a coarser level, and the leaf
    // kernels overlap the level kernels of their own levels.  (A graph puts its
    // branches on 4 queues in an order of its own, following that of the capture:
    // with the larger levels captured before the chain, the chain queued behind
    // their p2m, 1255 us a solve instead of 1211.)
    if (phases & 2) {
        bool used[2] = {};
        hipStream_t ss = t->side[0], sp = t->side[1];
        HIPC(c, hipEventRecord(t->ev_up, st));
        octofmm_plan* group[kStageLevels];
        int ng = 0;   // levels of the chain
        for (int slots = 0; ng < kStageLevels && ng < nl; ++ng) {
            slots += t->lv[ng].plan->stage_slots();
            if (ng > 0 && slots > kStageTogether) break;
            group[ng] = t->lv[ng].plan;
        }
        octofmm_status s = launch_stage(c, st, group, ng);
        if (s != OCTOFMM_OK) return s;
        launch_tree_sums(group, ng, st, t->type == OCTOFMM_RHO, c->tab);
        HIPC(c, hipGetLastError());
        for (int l = ng; l < nl; ++l) {
            if (t->lv[l].plan->stage_slots() == 0) continue;
            if (!used[0]) HIPC(c, hipStreamWaitEvent(ss, t->ev_up, 0));
            used[0] = true;
            s = launch_stage(c, ss, &t->lv[l].plan, 1);
            if (s != OCTOFMM_OK) return s;
            HIPC(c, hipEventRecord(t->ev_stage[l], ss));
        }
        for (int l = ng; l < nl; ++l) {
            octofmm_plan* p = t->lv[l].plan;
            if (!p->sums_first && p->n_p2m == 0) continue;
            HIPC(c, hipStreamWaitEvent(sp, t->ev_stage[l], 0));
            used[1] = true;
            if (p->sums_first) {
                s = plan_launch(p, sp, 16);
                if (s != OCTOFMM_OK) return s;
                HIPC(c, hipEventRecord(t->ev_sums[l], sp));
            }
            if (p->n_p2m == 0) continue;
            s = plan_launch(p, sp, 8);
            if (s != OCTOFMM_OK) return s;
            HIPC(c, hipEventRecord(t->ev_p2m[l], sp));
        }
        int leaves[kLeafLevels], nleaves = 0;   // leaf levels not launched yet
        for (int l = 0; l < nl; ++l) {
            octofmm_plan* p = t->lv[l].plan;
            if (l >= ng && p->n_m2l > 0) HIPC(c, hipStreamWaitEvent(st, p->sums_first ? t->ev_sums[l] : t->ev_stage[l], 0));
            s = plan_launch(p, st, 2);
            if (s != OCTOFMM_OK) return s;
            HIPC(c, hipEventRecord(t->ev_level[l], st));
            if (p->root || p->nitems == p->n_m2l) continue;
            // levels of few leaves wait for the next level's launch
            leaves[nleaves++] = l;
            const bool more = l + 1 < nl && t->lv[l + 1].plan->nitems > t->lv[l + 1].plan->n_m2l;
            if (more && c->tab.p2p_cube && p->nitems - p->n_m2l <= kStageTogether && nleaves < kLeafLevels) continue;
            hipStream_t q = st;
            if (p->n_m2l > 0) {   // beside this level's multipole targets
                q = sp;
                used[1] = true;
                HIPC(c, hipStreamWaitEvent(sp, t->ev_level[l - 1], 0));
            }
            for (int k = 0; k < nleaves; ++k)
                if (leaves[k] >= ng && t->lv[leaves[k]].plan->n_p2m > 0 && q != sp)
                    HIPC(c, hipStreamWaitEvent(q, t->ev_p2m[leaves[k]], 0));
            s = launch_leaves(t, leaves, nleaves, q);
            if (s != OCTOFMM_OK) return s;
            nleaves = 0;
        }
        for (int k = 0; k < 2; ++k) {
            if (!used[k]) continue;
            HIPC(c, hipEventRecord(t->ev_join[k], t->side[k]));
            HIPC(c, hipStreamWaitEvent(st, t->ev_join[k], 0));
        }
    }
    return OCTOFMM_OK;
}

}   // namespace

extern "C" {

octofmm_status octofmm_tree_plan_create(octofmm_context* c, const octofmm_tree* tr, octofmm_tree_plan** out) {
    if (!c) return OCTOFMM_ERR_INVALID_ARGUMENT;
    if (!tr || !out || tr->nlevels <= 0 || !tr->levels) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad tree");
    *out = nullptr;
    if (tr->type != OCTOFMM_RHO && tr->type != OCTOFMM_DRHODT) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad type");
    const bool rho = tr->type == OCTOFMM_RHO;
    const int nl = tr->nlevels;
    // structure: root alone on level 0, 8 children per non-leaf node, leaves at the bottom
    for (int l = 0; l < nl; ++l) {
        const octofmm_tree_level& L = tr->levels[l];
        if (L.nnodes <= 0 || !L.neighbors || !L.kind || !L.parent || !L.octant || !L.xbase || !(L.dx > 0.0))
            return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad description of level %d", l);
        if (!L.d_M || !L.d_com || !L.d_mon || !L.d_L || (rho && !L.d_L_c))
            return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "null device array on level %d", l);
        // expansion, correction and force rows are moved in 16-byte pieces
        if (((uintptr_t)L.d_L | (uintptr_t)L.d_L_c | (uintptr_t)L.d_g) & 15)
            return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "L, L_c and g of level %d must be 16-byte aligned", l);
        if (l == 0 && (L.nnodes != 1 || L.parent[0] != -1))
            return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "level 0 must hold the root alone, without a parent");
        std::vector<int> children(l + 1 < nl ? tr->levels[l + 1].nnodes : 0, 0);
        for (int n = 0; n < L.nnodes; ++n) {
            if (L.kind[n] != OCTOFMM_SLOT_NONLEAF && L.kind[n] != OCTOFMM_SLOT_LEAF)
                return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad kind of node %d on level %d", n, l);
            if (l == nl - 1 && L.kind[n] == OCTOFMM_SLOT_NONLEAF)
                return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "non-leaf node %d on the finest level", n);
            if (L.octant[n] < 0 || L.octant[n] > 7)
                return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "bad octant of node %d on level %d", n, l);
            if ((tr->flags & OCTOFMM_TREE_LEAF_G_ONLY) && L.kind[n] == OCTOFMM_SLOT_LEAF && !L.d_g)
                return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT,
                    "OCTOFMM_TREE_LEAF_G_ONLY needs d_g on level %d, which holds leaves", l);
        }
        if (l > 0) {
            const octofmm_tree_level& U = tr->levels[l - 1];
            std::vector<uint8_t> used((size_t)U.nnodes * 8, 0);
            for (int n = 0; n < L.nnodes; ++n) {
                const int pn = L.parent[n];
                if (pn < 0 || pn >= U.nnodes || U.kind[pn] != OCTOFMM_SLOT_NONLEAF)
                    return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "node %d on level %d has no non-leaf parent", n, l);
                uint8_t& u = used[(size_t)pn * 8 + L.octant[n]];
                if (u) return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "two children in one octant on level %d", l);
                u = 1;
            }
            for (int pn = 0; pn < U.nnodes; ++pn) {
                if (U.kind[pn] != OCTOFMM_SLOT_NONLEAF) continue;
                for (int o = 0; o < 8; ++o)
                    if (!used[(size_t)pn * 8 + o])
                        return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "non-leaf node %d on level %d lacks child %d",
                            pn, l - 1, o);
            }
        }
    }
    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    octofmm_tree_plan* t = new octofmm_tree_plan();
    t->ctx = c;
    t->type = tr->type;
    t->flags = tr->flags;
    t->G = tr->G;
    t->correct_am = tr->correct_am;
    std::memset(&t->stats, 0, sizeof(t->stats));
    t->stats.nlevels = nl;
    t->lv.resize(nl);
    t->ev_stage.assign(nl, nullptr);
    t->ev_level.assign(nl, nullptr);
    t->ev_sums.assign(nl, nullptr);
    t->ev_p2m.assign(nl, nullptr);
    auto cleanup = [&](octofmm_status s, const char* what) {
        tree_free(t);
        return fail(c, s, "%s", what);
    };
    {
        bool ok = hipStreamCreateWithFlags(&t->side[0], hipStreamNonBlocking) == hipSuccess &&
                  hipStreamCreateWithFlags(&t->side[1], hipStreamNonBlocking) == hipSuccess;
        for (hipEvent_t* e : {&t->ev_up, &t->ev_join[0], &t->ev_join[1]})
            ok = ok && hipEventCreateWithFlags(e, hipEventDisableTiming) == hipSuccess;
        for (int l = 0; l < nl; ++l)
            ok = ok && hipEventCreateWithFlags(&t->ev_stage[l], hipEventDisableTiming) == hipSuccess &&
                 hipEventCreateWithFlags(&t->ev_level[l], hipEventDisableTiming) == hipSuccess &&
                 hipEventCreateWithFlags(&t->ev_sums[l], hipEventDisableTiming) == hipSuccess &&
                 hipEventCreateWithFlags(&t->ev_p2m[l], hipEventDisableTiming) == hipSuccess;
        if (!ok) return cleanup(OCTOFMM_ERR_HIP, "tree stream or event creation failed");
    }
    for (int l = 0; l < nl; ++l) {
        const octofmm_tree_level& L = tr->levels[l];
        auto& D = t->lv[l];
        D.nnodes = L.nnodes;
        D.dx = L.dx;
        D.M = L.d_M;
        D.com = L.d_com;
        D.mon = L.d_mon;
        D.L = L.d_L;
        D.Lc = L.d_L_c;
        D.g = L.d_g;
        const size_t n = (size_t)L.nnodes;
        // one block: xbase, kind, parent, octant, order
        std::vector<double> tables((3 * n * sizeof(double) + 4 * n * sizeof(int32_t) + 7) / 8);
        std::copy(L.xbase, L.xbase + 3 * n, tables.begin());
        int32_t* ti = reinterpret_cast<int32_t*>(tables.data() + 3 * n);
        std::copy(L.kind, L.kind + n, ti);
        std::copy(L.parent, L.parent + n, ti + n);
        std::copy(L.octant, L.octant + n, ti + 2 * n);
        int32_t* to = ti + 3 * n;
        for (const int32_t k : {OCTOFMM_SLOT_LEAF, OCTOFMM_SLOT_NONLEAF})
            for (int i = 0; i < L.nnodes; ++i)
                if (L.kind[i] == k) *to++ = i;
        D.nleaf = (int32_t)std::count(L.kind, L.kind + n, (int32_t)OCTOFMM_SLOT_LEAF);
        const size_t bytes = tables.size() * sizeof(double);
        if (hipMalloc((void**)&D.d_xbase, bytes) != hipSuccess)
            return cleanup(OCTOFMM_ERR_ALLOCATION, "tree table allocation failed");
        D.d_kind = reinterpret_cast<int32_t*>(D.d_xbase + 3 * n);
        D.d_parent = D.d_kind + n;
        D.d_octant = D.d_parent + n;
        D.d_order = D.d_octant + n;
        if (hipMemcpy(D.d_xbase, tables.data(), bytes, hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(OCTOFMM_ERR_HIP, "tree table upload failed");
        t->stats.nodes += L.nnodes;
        for (int i = 0; i < L.nnodes; ++i) t->stats.leaves += L.kind[i] == OCTOFMM_SLOT_LEAF;
    }
    // one upward pass first, so that autotuning times the interactions on real multipoles
    {
        const octofmm_status s = tree_launch(t, c->stream, 1);
        if (s != OCTOFMM_OK) {
            tree_free(t);
            return s;
        }
        if (hipStreamSynchronize(c->stream) != hipSuccess) return cleanup(OCTOFMM_ERR_HIP, "upward pass failed");
    }
    for (int l = 0; l < nl; ++l) {
        const octofmm_tree_level& L = tr->levels[l];
        std::vector<int32_t> targets(L.nnodes);
        for (int i = 0; i < L.nnodes; ++i) targets[i] = i;
        octofmm_level lv;
        std::memset(&lv, 0, sizeof(lv));
        lv.nslots = L.nnodes;
        lv.neighbors = L.neighbors;
        lv.kind = L.kind;
        lv.xbase = L.xbase;
        lv.dx = L.dx;
        lv.ntargets = L.nnodes;
        lv.targets = targets.data();
        lv.type = tr->type;
        lv.precision = tr->precision;
        lv.mixed_far_d2 = tr->mixed_far_d2;
        lv.flags = tr->flags & OCTOFMM_PLAN_AUTOTUNE;
        if (l == 0 && L.kind[0] == OCTOFMM_SLOT_NONLEAF) {
            lv.flags = OCTOFMM_PLAN_ROOT;
            lv.precision = OCTOFMM_PRECISION_FP64;
        }
        lv.d_M = L.d_M;
        lv.d_com = L.d_com;
        lv.d_mon = L.d_mon;
        lv.d_L = L.d_L;
        lv.d_L_c = rho ? L.d_L_c : nullptr;
        // the level's plan is tuned only once its epilogue is the fused
        // downward pass it runs with in the solve
        octofmm_plan* lp = nullptr;
        octofmm_status s = level_plan_build(c, &lv, true, &lp);
        if (s == OCTOFMM_OK) {
            lp->l2l = true;
            lp->t_parent = t->lv[l].d_parent;
            lp->t_octant = t->lv[l].d_octant;
            lp->t_pL = l > 0 ? t->lv[l - 1].L : nullptr;
            lp->t_pLc = l > 0 ? t->lv[l - 1].Lc : nullptr;
            lp->t_pcom = l > 0 ? t->lv[l - 1].com : nullptr;
            lp->t_g = t->lv[l].g;
            lp->t_G = t->G;
            lp->t_correct_am = t->correct_am;
            lp->leaf_rows = (tr->flags & OCTOFMM_TREE_LEAF_G_ONLY) ? 0 : 1;
            s = level_plan_finish(lp, lp->sums_first ? 0 : lv.flags);
        }
        if (s != OCTOFMM_OK) {
            const std::string msg = c->err;
            tree_free(t);
            return fail(c, s, "level %d: %s", l, msg.c_str());
        }
        t->lv[l].plan = lp;
        const octofmm_plan_stats& ps = t->lv[l].plan->stats;
        if (t->lv[l].plan->root)
            t->stats.root_pairs += ps.far_pairs;
        else
            t->stats.far_pairs += ps.far_pairs;
        t->stats.near_pairs += ps.near_pairs;
        t->stats.p2p_pairs += ps.p2p_pairs;
        t->stats.p2m_pairs += ps.p2m_pairs;
        t->stats.flops += ps.flops;
        t->stats.mixed_far_pairs += ps.mixed_far_pairs;
    }
    if (tr->flags & OCTOFMM_PLAN_USE_GRAPH) {
        hipStream_t cs = c->stream;
        if (hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) != hipSuccess)
            return cleanup(OCTOFMM_ERR_HIP, "graph capture failed to start");
        const octofmm_status ls = tree_launch(t, cs, 7);
        hipGraph_t g = nullptr;
        const hipError_t ee = hipStreamEndCapture(cs, &g);
        if (ls != OCTOFMM_OK || ee != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            return cleanup(OCTOFMM_ERR_HIP, "graph capture failed");
        }
        t->graph = g;
        if (hipGraphInstantiate(&t->gexec, g, nullptr, nullptr, 0) != hipSuccess)
            return cleanup(OCTOFMM_ERR_HIP, "graph instantiation failed");
    }
    *out = t;
    return OCTOFMM_OK;
}

octofmm_status octofmm_tree_plan_execute(octofmm_tree_plan* t, void* stream) {
    if (!t) return OCTOFMM_ERR_INVALID_ARGUMENT;
    octofmm_context* c = t->ctx;
    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (t->gexec) {
        HIPC(c, hipGraphLaunch(t->gexec, st));
        return OCTOFMM_OK;
    }
    return tree_launch(t, st, 7);
}

octofmm_status octofmm_tree_plan_stats(const octofmm_tree_plan* t, octofmm_tree_stats* s) {
    if (!t || !s) return OCTOFMM_ERR_INVALID_ARGUMENT;
    *s = t->stats;
    return OCTOFMM_OK;
}

octofmm_status octofmm_tree_plan_time_phases(octofmm_tree_plan* t, void* stream, int32_t iters, double* ms) {
    if (!t || !ms || iters <= 0) return OCTOFMM_ERR_INVALID_ARGUMENT;
    octofmm_context* c = t->ctx;
    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    hipEvent_t e0, e1;
    HIPC(c, hipEventCreate(&e0));
    HIPC(c, hipEventCreate(&e1));
    for (int ph = 0; ph < 3; ++ph) {
        HIPC(c, hipEventRecord(e0, st));
        for (int i = 0; i < iters; ++i) {
            const octofmm_status s = tree_launch(t, st, 1 << ph);
            if (s != OCTOFMM_OK) return s;
        }
        HIPC(c, hipEventRecord(e1, st));
        HIPC(c, hipEventSynchronize(e1));
        float f = 0.f;
        HIPC(c, hipEventElapsedTime(&f, e0, e1));
        ms[ph] = (double)f / iters;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return OCTOFMM_OK;
}

octofmm_status octofmm_measure_fma_rate(octofmm_context* c, int32_t precision, double* tflops) {
    if (!c || !tflops) return OCTOFMM_ERR_INVALID_ARGUMENT;
    if (precision != OCTOFMM_PRECISION_FP64 && precision != OCTOFMM_PRECISION_MIXED)
        return fail(c, OCTOFMM_ERR_INVALID_ARGUMENT, "precision must be FP64 or MIXED (FP32)");
    HIPC(c, hipSetDevice(c->device));
    (void)hipGetLastError();   // launch checks below report this call's launches only
    // 4096 workgroups of 256 lanes (16 per CU on 256 CUs), 8 chains x 2048 steps each
    constexpr int kBlocks = 4096, kIters = 2048;
    void* out = nullptr;
    HIPC(c, hipMalloc(&out, sizeof(double) * (size_t)kBlocks * 256));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto run = [&]() {
        if (precision == OCTOFMM_PRECISION_FP64)
            hipLaunchKernelGGL(fma_rate_kernel<double>, dim3(kBlocks), dim3(256), 0, c->stream,
                static_cast<double*>(out), 0.999999, 1.0e-7, kIters);
        else
            hipLaunchKernelGGL(fma_rate_kernel<float>, dim3(kBlocks), dim3(256), 0, c->stream,
                static_cast<float*>(out), 0.999999f, 1.0e-7f, kIters);
    };
    hipError_t e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    if (e == hipSuccess) {
        run();
        e = hipEventRecord(e0, c->stream);
    }
    if (e == hipSuccess) {
        run();
        e = hipEventRecord(e1, c->stream);
    }
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    float ms = 0.f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(out);
    HIPC(c, e);
    const double fmas = (double)kBlocks * 256.0 * 8.0 * kIters;
    *tflops = ms > 0.f ? 2.0 * fmas / (ms * 1e-3) / 1e12 : 0.0;
    return OCTOFMM_OK;
}

octofmm_status octofmm_tree_plan_destroy(octofmm_tree_plan* t) {
    if (!t) return OCTOFMM_OK;
    (void)hipSetDevice(t->ctx->device);
    tree_free(t);
    return OCTOFMM_OK;
}

}   // extern "C"
