// LU-SGS sweeps (Time/TIME_LUSGS.F90:172-436 forward, :442-675 backward, and the k-omega
// sweeps of Time/TURBTWO_TIME_LUSGS_SST.F90:550-766) as a wavefront of single-wave tiles.
//
// A block's lines along j are cut into tiles of WVA (i) x WVB (k) lines, one wave per tile and
// equation set (mean flow, k-omega), one lane per line.  On row tau of its tile a lane updates
// the cell j - 1 = tau - ia - ib of its line, so all lanes of a row lie on one hyperplane
// i + j + k = const, and hands the terms 0.5*(A dQ +/- Rds dQ) of its three downstream
// neighbours on: along j in its registers, along i to the next lane of its DPP row (WVA = 16
// lanes), along k through a wave-private LDS row.  A wave needs no barrier at any point.
//
// Terms that cross a tile face go through the producing tile's edge rows in global memory.  An
// edge value is its own flag: the buffers are filled with a NaN pattern before the sweeps
// (k_wave_rhs), a consumer loads its values PD rows ahead and, where a loaded value still
// is that pattern, polls until the producer has stored it.  There are no progress counters,
// no chunks and no waits for stores to complete; each value is in one aligned 8-byte word that
// is stored and loaded at agent scope (two FP32 values, each its own flag, or one FP64 value, which
// must arrive whole: these are the instructions and cache bits of a relaxed 64-bit atomic load or
// store), so no order between stores matters.  Tiles are work items taken from an atomic
// counter with a tile's upstream tiles first, so a wait is always for a tile that has started;
// every wait is bounded (spin_limit), past it the error flag is raised and the sweep goes on.
//
// The inputs lie in tile packets: row tau of a tile holds its 64 lanes' values in groups of 16
// bytes per lane (WaveRow), so a row is read with consecutive 1 KB buffer loads (six for the
// mean flow with the FP32 operator) at a scalar offset.  Lanes without a cell on a row get an
// out-of-range offset, for which the buffer load returns zero without touching memory and the
// store is dropped; with zero inputs such a lane hands zero terms on, which is what its
// neighbours need before their first cell.
//
// What bounds it: a tile's rows follow each other.  A row of the mean flow is 190 instructions in FP64,
// 108 of them arithmetic and 36 memory operations, and takes 0.54 to 0.58 us (sweeps of 194 and 198
// rows); 175, 108 and 21 in FP32, 0.49 us (115 rows).  So with few tiles (fewer than four per SIMD) the
// chain (NJ1 + tile diagonals x the skew) x row time; with many, the memory system (144 B/cell FP32
// per sweep).  Forward and backward sweep together, before (one workgroup per block marching lines
// with a barrier per step, or tiles of 256 lines with progress counters) and now:
//     65k-cell bump channel, FP64           707 us   218 us
//     131k-cell plate, FP64 k-omega         406 us   225 us
//     0.13M-cell sector, FP64 k-omega       263 us    97 us
//     0.49M-cell sector, FP32 k-omega       395 us   164 us
//     8.1M-cell sector, FP32 k-omega       2129 us  1060 us
// Tiles of 16 x 4 lines: the i terms then stay within a DPP row of 16 lanes.
#pragma once
#include "k_time.h"
#include "k_visc.h"

constexpr int WVA = 16, WVB = 4;            // lines of a tile along i and along k
constexpr int WV_SKEW = WVA - 1 + WVB - 1;  // rows a tile has beyond NJ1
// (Each half of) an edge value not yet stored: a NaN that no operation makes of other values.  In
// FP32 operations hand it on, so a tile that gave up a wait may store it as a value; its neighbours
// then count it as missing, until their waits end by the error flag.
constexpr unsigned WV_SENTINEL = 0xFFF5A5A5u;
constexpr int WV_SPIN_LIMIT = 1 << 18;      // polls of one bounded wait (about 0.3 s)

// Values of one lane in a packet row.  The face means and the spectral radii are stored halved
// (exact), so the neighbour terms need no factor 0.5.
constexpr int WV_D = 0;       // 5: mean-flow right-hand side, then the increment
constexpr int WV_SA = 5;      // stept / F1
constexpr int WV_SB = 6;      // cvs / F1
constexpr int WV_C2 = 8;      // gamma p / rho (7 is unused)
constexpr int WV_U = 9;       // 3: velocity
constexpr int WV_RDS = 12;    // 3: Rds / 2
constexpr int WV_RF1 = 15;    // 1 / F1t (k-omega diagonal)
constexpr int WV_S = 16;      // 8: face means / 2, component d * 3 + x
constexpr int WV_K = 24;      // 2: k-omega right-hand side, then the increment
constexpr int WV_STEPT = 26;  // k-omega step
constexpr int WV_CVS = 27;    // k-omega step / Vol
constexpr int WV_S8 = 28;     // the ninth face mean
constexpr int WV_NVAL = 29;

template <typename R>
struct WaveRow {
    static constexpr int VL = 16 / (int)sizeof(R);  // values of a lane in one 16-byte group
    static constexpr int ELEMS = WV_NVAL * 64;      // elements of a row
    static constexpr int BYTES = ELEMS * (int)sizeof(R);
    static constexpr int GB = 1024;                 // bytes of a group of 64 lanes
    static constexpr int S8B = WV_S8 * 64 * (int)sizeof(R);  // byte offset of the ninth face mean
};

// Edge row: what the lanes on a tile's outgoing i and k faces hand on at one row, as 8-byte words per
// lane (one FP64 value, or two FP32 values of which the last may be padding): byte offsets.  (16-byte
// words, 3 to 5 % faster on small grids, gave results that differed from run to run: nothing promises
// that such a word arrives whole.)
template <typename R>
struct WaveEdge {
    static constexpr int ELEMS = 160;
    static constexpr int BYTES = ELEMS * (int)sizeof(R);
    static constexpr int A5 = 0, A2 = 24 * (int)sizeof(R);
    static constexpr int B5 = 32 * (int)sizeof(R), B2 = 128 * (int)sizeof(R);
    static constexpr int words(int neq) { return sizeof(R) == 8 ? neq : (neq + 1) / 2; }
};

struct WaveTile {
    int blk, ta, tb;
};

__host__ __device__ __forceinline__ int wave_rows(int nj) { return nj - 1 + WV_SKEW; }
__host__ __device__ __forceinline__ int wave_nta(int ni) { return (ni - 1 + WVA - 1) / WVA; }
__host__ __device__ __forceinline__ int wave_ntb(int nk) { return (nk - 1 + WVB - 1) / WVB; }

// First element of the packet row of cell (i, j, k), and its lane.
template <typename R>
__device__ __forceinline__ long wave_row(const BlkInfo& b, int i, int j, int k, int& lane)
{
    const int ia = (i - 1) % WVA, ib = (k - 1) % WVB;
    const int tile = (i - 1) / WVA + wave_nta(b.ni) * ((k - 1) / WVB);
    lane = ib * WVA + ia;
    return b.poff + ((long)tile * wave_rows(b.nj) + (j - 1 + ia + ib)) * WaveRow<R>::ELEMS;
}

// Element of value v of a lane inside a row.
template <typename R>
__device__ __forceinline__ int wave_elem(int v, int lane)
{
    constexpr int VL = WaveRow<R>::VL;
    return v == WV_S8 ? WV_S8 * 64 + lane : (v / VL) * 64 * VL + lane * VL + v % VL;
}

// Halved face-mean vectors of every interior cell into the packets, and the face means in the
// natural layout (see k_face_means); once per geometry upload.
template <typename R>
__global__ void __launch_bounds__(256) k_wave_geom(Fields f, const BlkInfo* __restrict__ blks,
                                                   const Seg* __restrict__ seg)
{
    const Seg s = seg[blockIdx.x];
    const BlkInfo b = blks[s.blk];
    const int NI1 = b.ni - 1, NJ1 = b.nj - 1, NK1 = b.nk - 1;
    const int lin = s.base + threadIdx.x;
    if (lin >= NI1 * NJ1 * NK1) return;
    int i, j, k;
    decode3(lin, NI1, NJ1, i, j, k);
    const long c = cidx(b, i, j, k);
    const long tot = f.tot;
    const long st[3] = {1, (long)b.nx, (long)b.nx * b.ny};
    int lane;
    R* const row = (R*)f.P + wave_row<R>(b, i, j, k, lane);
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const long o = (long)(d + 3 * q) * tot;
            const double m = 0.5 * (f.SD[o + c + st[d]] + f.SD[o + c]);
            f.SDm[o + c] = m;
            const int v = d * 3 + q;
            row[wave_elem<R>(v < 8 ? WV_S + v : WV_S8, lane)] = (R)(0.5 * m);
        }
}

// The sweeps' inputs of every cell into the packets: a workgroup owns a WT x WT tile of cells
// (i, j) at one k (schedule entry Seg{block, tile index}), forms each cell's values in its own
// thread (MF: mean flow, TURB: k-omega; the step sizes, velocities and radii either way) and
// writes them through LDS diagonal by diagonal, on which the tile's cells are consecutive lanes
// of one packet row.  The workgroups also fill both sweeps' edge rows with the
// not-yet-stored pattern and reset the item counters.
constexpr int WR_NV = 20;  // staged values
template <typename R, bool MF, bool TURB>
__global__ void __launch_bounds__(256) k_wave_rhs(trans_params p, Fields f, const BlkInfo* __restrict__ blks,
                                                  const Seg* __restrict__ seg, int* __restrict__ ctr,
                                                  uint4* __restrict__ edge, long edge_n16)
{
    __shared__ R sv[WR_NV][WT * WT];
    {
        const uint4 s4 = make_uint4(WV_SENTINEL, WV_SENTINEL, WV_SENTINEL, WV_SENTINEL);
        for (long q = (long)blockIdx.x * 256 + threadIdx.x; q < edge_n16; q += (long)gridDim.x * 256) edge[q] = s4;
        if (blockIdx.x == 0 && threadIdx.x < 2) ctr[threadIdx.x] = 0;
    }
    const Seg s = seg[blockIdx.x];
    const BlkInfo b = blks[s.blk];
    const TileCell tc = wtile_cell(s, b, threadIdx.x % WT, threadIdx.x / WT);
    if (tc.ok) {
        const long c = cidx(b, tc.i, tc.j, tc.k);
        const long tot = f.tot;
        const int t = threadIdx.x;
        // staged: 0-7 the first eight values, 8-15 the next eight, 16-19 the k-omega group
        double rhs[5], stept, cvs, f1;
        if (MF) {
            lusgs_rhs_cell(p, f, c, rhs, stept, cvs, f1);
#pragma unroll
            for (int L = 0; L < 5; L++) sv[WV_D + L][t] = (R)rhs[L];
            const double rf1 = 1.0 / f1;
            sv[WV_SA][t] = (R)(stept * rf1);
            sv[WV_SB][t] = (R)(cvs * rf1);
        } else {
            const double dtm = f.Dtm[c], dtl = p.dt_lusgs_main;
            stept = 2.0 * dtm / (3.0 * dtm / dtl + 2.0);
            cvs = stept / f.Vol[c];
        }
        const double roinv = 1.0 / f.V[c];
#pragma unroll
        for (int L = 0; L < 3; L++) sv[WV_U + L][t] = (R)(f.V[(long)(L + 1) * tot + c] * roinv);
        if (MF) {
            sv[WV_C2][t] = R(1.4) * (R)f.PP[c] * (R)roinv;
        }
#pragma unroll
        for (int d = 0; d < 3; d++) sv[WV_RDS + d][t] = (R)(0.5 * f.Rds[(long)d * tot + c]);
        if (TURB) {
            double d6, d7, f1t;
            sst_rhs_cell(p, f, b, tc.i, tc.j, tc.k, c, d6, d7, f1t);
            sv[WV_RF1][t] = R(1) / (R)f1t;
            sv[16][t] = (R)d6;
            sv[17][t] = (R)d7;
            sv[18][t] = (R)stept;
            sv[19][t] = (R)cvs;
        }
    }
    __syncthreads();
    constexpr int VL = WaveRow<R>::VL;
    struct alignas(16) Vec {
        R x[VL];
    };
    // diagonals dd = ti + tj of the tile: 16 consecutive threads per diagonal
    for (int q = threadIdx.x; q < (2 * WT - 1) * WT; q += 256) {
        const int ti = q % WT, tj = q / WT - ti;
        if (tj < 0 || tj >= WT) continue;
        const TileCell oc = wtile_cell(s, b, ti, tj);
        if (!oc.ok) continue;
        int lane;
        R* const row = (R*)f.P + wave_row<R>(b, oc.i, oc.j, oc.k, lane);
        const int o = tj * WT + ti;
#pragma unroll
        for (int g = 0; g < WR_NV / VL; g++) {
            const int v = g * VL;
            if (!MF && v < WV_C2) continue;      // k-omega alone: no mean-flow groups
            if (!TURB && v >= 16) continue;     // no k-omega group
            Vec x;
#pragma unroll
            for (int e = 0; e < VL; e++) x.x[e] = sv[v + e][o];
            *reinterpret_cast<Vec*>(row + wave_elem<R>(v < 16 ? v : v + (WV_K - 16), lane)) = x;
        }
    }
}

// NEQ increments (7: mean flow and k-omega, 5, or 2: k-omega) of a tile of cells from the packets into
// LDS, diagonal by diagonal: sv[L][tj * WT + ti] for L = 5 (NEQ 2) or 0 on.
template <typename R, int NEQ>
__device__ __forceinline__ void wave_fetch(const Fields& f, const Seg& s, const BlkInfo& b, R (*sv)[WT * WT])
{
    constexpr int VL = WaveRow<R>::VL;
    struct alignas(16) Vec {
        R x[VL];
    };
    struct alignas(2 * sizeof(R)) Two {
        R x[2];
    };
    for (int q = threadIdx.x; q < (2 * WT - 1) * WT; q += 256) {
        const int ti = q % WT, tj = q / WT - ti;
        if (tj < 0 || tj >= WT) continue;
        const TileCell ic = wtile_cell(s, b, ti, tj);
        if (!ic.ok) continue;
        int lane;
        const R* const row = (const R*)f.P + wave_row<R>(b, ic.i, ic.j, ic.k, lane);
        const int o = tj * WT + ti;
        if (NEQ != 2) {
#pragma unroll
            for (int v = WV_D; v < WV_D + 4; v += VL) {
                const Vec x = *reinterpret_cast<const Vec*>(row + wave_elem<R>(v, lane));
#pragma unroll
                for (int e = 0; e < VL; e++) sv[v - WV_D + e][o] = x.x[e];
            }
            sv[4][o] = row[wave_elem<R>(WV_D + 4, lane)];
        }
        if (NEQ != 5) {
            const Two x = *reinterpret_cast<const Two*>(row + wave_elem<R>(WV_K, lane));
            sv[5][o] = x.x[0];
            sv[6][o] = x.x[1];
        }
    }
    __syncthreads();
}

// The k-omega increments back to D (the Runge-Kutta path), tile by tile.
template <typename R>
__global__ void __launch_bounds__(256) k_wave_unskew(Fields f, const BlkInfo* __restrict__ blks,
                                                     const Seg* __restrict__ seg)
{
    __shared__ R sv[7][WT * WT];
    const Seg s = seg[blockIdx.x];
    const BlkInfo b = blks[s.blk];
    wave_fetch<R, 2>(f, s, b, sv);
    const TileCell oc = wtile_cell(s, b, threadIdx.x % WT, threadIdx.x / WT);
    if (!oc.ok) return;
    const long c = cidx(b, oc.i, oc.j, oc.k);
    for (int L = 5; L < 7; L++) f.D[(long)L * f.tot + c] = (double)sv[L][threadIdx.x];
}

// k_update_v with the increments from the packets, which go to D as well: a workgroup updates a
// WT x WT tile of cells.  Bound by memory (4.8 TB/s at 8.1M cells): 858 us, with a pass of its own for
// the increments 777 + 231 us; 0.13M cells, 24 us and 33 us.
template <typename R, int NEQ>
__global__ void __launch_bounds__(256) k_wave_update(trans_params p, int ki, int if_turb, Fields f,
                                                     const BlkInfo* __restrict__ blks, const Seg* __restrict__ seg,
                                                     NormPart* part, int shift)
{
    __shared__ R sv[7][WT * WT];
    const Seg s = seg[blockIdx.x];
    const BlkInfo b = blks[s.blk];
    wave_fetch<R, NEQ>(f, s, b, sv);
    const TileCell oc = wtile_cell(s, b, threadIdx.x % WT, threadIdx.x / WT);
    double dr[3] = {0.0, 0.0, 0.0};
    int arg = -1;
    if (oc.ok) {
        const long c = cidx(b, oc.i, oc.j, oc.k);
        arg = oc.i - 1 + (b.ni - 1) * (oc.j - 1 + (b.nj - 1) * (oc.k - 1));
        double d[7];
#pragma unroll
        for (int L = 0; L < 7; L++) {
            double* const D = f.D + (long)L * f.tot + c;
            if (L < NEQ) {
                d[L] = (double)sv[L][threadIdx.x];
                *D = d[L];
            } else {
                d[L] = *D;
            }
        }
        update_cell(p, ki, if_turb, f, c, d, shift, dr);
    }
    norm_reduce(dr, arg, part, 0);
}

// ---------------------------------------------------------------------------------------
// the sweep

typedef unsigned wv_u2 __attribute__((ext_vector_type(2)));
typedef unsigned wv_u4 __attribute__((ext_vector_type(4)));

// Raw buffer over [p, p + bytes): 32-bit data, no stride; loads outside it return zero, stores
// outside it are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t wv_rsrc(const void* p, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
constexpr int WV_OOB = (int)0x80000000u;  // beyond every buffer
constexpr int WV_SC1 = 16;                // agent scope: past the XCD's L2
constexpr int WV_POLL = WV_SC1 | (int)0x80000000u;  // the same, volatile: loaded anew every time

template <typename R>
struct WvVec;
template <>
struct WvVec<float> {
    static __device__ __forceinline__ float get(wv_u4 x, int e) { return __uint_as_float(x[e]); }
    static __device__ __forceinline__ wv_u4 put(const float* e)
    {
        return wv_u4{__float_as_uint(e[0]), __float_as_uint(e[1]), __float_as_uint(e[2]), __float_as_uint(e[3])};
    }
};
template <>
struct WvVec<double> {
    static __device__ __forceinline__ double get(wv_u4 x, int e)
    {
        return __hiloint2double((int)x[2 * e + 1], (int)x[2 * e]);
    }
    static __device__ __forceinline__ wv_u4 put(const double* e)
    {
        return wv_u4{(unsigned)__double2loint(e[0]), (unsigned)__double2hiint(e[0]), (unsigned)__double2loint(e[1]),
                     (unsigned)__double2hiint(e[1])};
    }
};

// One row's inputs of a lane, and the terms that reach it across its tile's i and k faces.
template <typename R, int NEQ>
struct WaveIn {
    R d[NEQ];
    R sa, sb;         // factors of the right-hand side and of the neighbour sum (mean flow: divided by F1)
    R c2, rf1;
    R u[3], rds[3], s[9];
    R ea[NEQ], eb[NEQ];
    bool act;       // whether the lane has a cell on the row
    int row, erow;  // byte offsets of the packet row and of the tile's edge row
};

// A lane's NEQ edge values: vo is the lane's offset (8 bytes per lane, or out of range), base the
// face's offset in the row, LANES the face's lanes.
template <typename R, int NEQ, int LANES, int AUX>
__device__ __forceinline__ void wv_edge_load(__amdgpu_buffer_rsrc_t r, int vo, int base, int row, R* e)
{
#pragma unroll
    for (int q = 0; q < WaveEdge<R>::words(NEQ); q++) {
        const wv_u2 w = __builtin_amdgcn_raw_buffer_load_b64(r, vo + base + q * LANES * 8, row, AUX);
        if constexpr (sizeof(R) == 8) {
            e[q] = __hiloint2double((int)w[1], (int)w[0]);
        } else {
            e[2 * q] = __uint_as_float(w[0]);
            if (2 * q + 1 < NEQ) e[2 * q + 1] = __uint_as_float(w[1]);
        }
    }
}
template <typename R, int NEQ, int LANES>
__device__ __forceinline__ void wv_edge_store(__amdgpu_buffer_rsrc_t r, int vo, int base, int row, const R* e)
{
#pragma unroll
    for (int q = 0; q < WaveEdge<R>::words(NEQ); q++) {
        wv_u2 w;
        if constexpr (sizeof(R) == 8)
            w = wv_u2{(unsigned)__double2loint(e[q]), (unsigned)__double2hiint(e[q])};
        else
            w = wv_u2{__float_as_uint(e[2 * q]), 2 * q + 1 < NEQ ? __float_as_uint(e[2 * q + 1 < NEQ ? 2 * q + 1 : 0]) : 0u};
        __builtin_amdgcn_raw_buffer_store_b64(w, r, vo + base + q * LANES * 8, row, WV_SC1);
    }
}
template <typename R>
__device__ __forceinline__ bool wv_pending(R x)
{
    if constexpr (sizeof(R) == 8)
        return (unsigned)__double2hiint(x) == WV_SENTINEL && (unsigned)__double2loint(x) == WV_SENTINEL;
    else
        return __float_as_uint(x) == WV_SENTINEL;
}

// x of the lane one down (forward) or up (backward) its DPP row; the row's first lane keeps `edge`.
template <bool FORWARD>
__device__ __forceinline__ int wv_shift_i(int edge, int x)
{
    return FORWARD ? __builtin_amdgcn_update_dpp(edge, x, 0x111, 0xf, 0xf, false)
                   : __builtin_amdgcn_update_dpp(edge, x, 0x101, 0xf, 0xf, false);
}
template <bool FORWARD>
__device__ __forceinline__ float wv_shift(float edge, float x)
{
    return __int_as_float(wv_shift_i<FORWARD>(__float_as_int(edge), __float_as_int(x)));
}
template <bool FORWARD>
__device__ __forceinline__ double wv_shift(double edge, double x)
{
    return __hiloint2double(wv_shift_i<FORWARD>(__double2hiint(edge), __double2hiint(x)),
                            wv_shift_i<FORWARD>(__double2loint(edge), __double2loint(x)));
}

// Orders a wave's LDS stores before its later loads (the LDS serves a wave in order; this only
// keeps the compiler from moving one across the other).
__device__ __forceinline__ void wv_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

__device__ __forceinline__ float wv_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double wv_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
// a . b with the first product rounded: that of component 0 (UF) or of component 1.
template <bool UF, typename R>
__device__ __forceinline__ R wv_dot(const R* a, const R* b)
{
    return UF ? wv_fma(a[2], b[2], wv_fma(a[1], b[1], a[0] * b[0])) : wv_fma(a[2], b[2], wv_fma(a[0], b[0], a[1] * b[1]));
}

// s_waitcnt operand: at most n vector memory operations in flight, the other counters free
constexpr int wv_vmcnt(int n)
{
    const int m = n < 63 ? n : 63;
    return (m & 15) | ((m >> 4) << 14) | 0x0F70;
}

// One tile's sweep for NEQ = 5 (mean flow) or 2 (k-omega).  lds: NEQ rows of 80 values, through
// which a lane's k term goes to the lane 16 above (forward) or below (backward); the 16 entries at
// the end that no lane stores to stay zero.
template <typename R, bool FORWARD, int NEQ, int PD, bool ALT>
__device__ __forceinline__ void wave_sweep(const Fields& f, const BlkInfo& b, int ta, int tb, R* __restrict__ lds,
                                           R* __restrict__ edge, int* __restrict__ err, int spin_limit)
{
    static_assert(NEQ == 5 || NEQ == 2, "mean flow or k-omega");
    constexpr bool MF = NEQ == 5;
    using Row = WaveRow<R>;
    using Edge = WaveEdge<R>;
    constexpr int VL = Row::VL;
    constexpr int EA = MF ? Edge::A5 : Edge::A2, EB = MF ? Edge::B5 : Edge::B2;
    // loads and stores of a step: packet groups and the ninth face mean, edge values; edge values
    // and increments
    constexpr int NE = Edge::words(NEQ);
    constexpr int NLD = (MF ? WV_K / VL : (28 - WV_C2) / VL) + 1 + 2 * NE, NST = 2 * NE + (MF ? 4 / VL + 1 : 1);
    const int NI1 = b.ni - 1, NJ1 = b.nj - 1, NK1 = b.nk - 1;
    const int nta = wave_nta(b.ni), ntb = wave_ntb(b.nk);
    const int T = wave_rows(b.nj);
    const int na = min(WVA, NI1 - ta * WVA), nb = min(WVB, NK1 - tb * WVB);
    const int nrow = na - 1 + nb - 1 + NJ1;  // rows on which some line of the tile has a cell
    const int lane = threadIdx.x & 63;
    const int ia = lane % WVA, ib = lane / WVA;
    // row on which the lane's line starts (never, for a lane without a line)
    const int start = ia < na && ib < nb ? ia + ib : INT_MAX / 2;
    const int tile = ta + nta * tb;
    const bool up_a = FORWARD ? ta > 0 : ta < nta - 1, up_b = FORWARD ? tb > 0 : tb < ntb - 1;
    const bool dn_a = FORWARD ? ta < nta - 1 : ta > 0, dn_b = FORWARD ? tb < ntb - 1 : tb > 0;
    const int tile_a = up_a ? (FORWARD ? tile - 1 : tile + 1) : tile;
    const int tile_b = up_b ? (FORWARD ? tile - nta : tile + nta) : tile;
    // the tile's packet rows, from the first byte and 8 KB on (a buffer offset's constant part
    // reaches 4 KB), and the edge rows of the upstream tiles and of the tile itself
    const R* const pk = (const R*)f.P + b.poff + (long)tile * T * Row::ELEMS;
    const __amdgpu_buffer_rsrc_t rw0 = wv_rsrc(pk, (unsigned)T * Row::BYTES);
    const __amdgpu_buffer_rsrc_t rw1 = wv_rsrc((const char*)pk + 8192, (unsigned)T * Row::BYTES - 8192);
    R* const e0 = edge + b.eoff;
    const unsigned ebytes = (unsigned)T * Edge::BYTES;
    const __amdgpu_buffer_rsrc_t ra = wv_rsrc(e0 + (long)tile_a * T * Edge::ELEMS, ebytes);
    const __amdgpu_buffer_rsrc_t rb = wv_rsrc(e0 + (long)tile_b * T * Edge::ELEMS, ebytes);
    const __amdgpu_buffer_rsrc_t ro = wv_rsrc(e0 + (long)tile * T * Edge::ELEMS, ebytes);
    // lane offsets in the edge rows, out of range for the lanes that take no part
    const bool in_a = up_a && ia == (FORWARD ? 0 : WVA - 1), in_b = up_b && ib == (FORWARD ? 0 : WVB - 1);
    const bool out_a = dn_a && ia == (FORWARD ? WVA - 1 : 0), out_b = dn_b && ib == (FORWARD ? WVB - 1 : 0);
    const int off_in_a = in_a ? ib * 8 : WV_OOB, off_in_b = in_b ? ia * 8 : WV_OOB;
    const int off_out_a = out_a ? ib * 8 : WV_OOB, off_out_b = out_b ? ia * 8 : WV_OOB;
    // the edge values of row tau were stored on the upstream tile's row tau + WVA - 1 (i) or
    // tau + WVB - 1 (k) in the forward sweep, and as many rows earlier in the backward one
    constexpr int SHA = FORWARD ? WVA - 1 : -(WVA - 1), SHB = FORWARD ? WVB - 1 : -(WVB - 1);
    R* const lds_st = lds + lane + (FORWARD ? 16 : 0);
    const R* const lds_ld = lds + lane + (FORWARD ? 0 : 16);
    if (lane < 16) {
#pragma unroll
        for (int L = 0; L < NEQ; L++) lds[L * 80 + lane + (FORWARD ? 0 : 64)] = R(0);
    }
    wv_lds_order();

    // byte offset r clamped to the tile's rows: a row outside them has no active lane, and its
    // offset must not exceed the buffers' ends, from which the range check counts down
    const int last_w = (T - 1) * Row::BYTES, last_e = (T - 1) * Edge::BYTES;
    auto clamp = [](int r, int last) __attribute__((always_inline)) { return min(max(r, 0), last); };
    auto edges = [&](auto aux, const int tau, WaveIn<R, NEQ>& x, R* ea) __attribute__((always_inline)) {
        constexpr int AUX = decltype(aux)::value;
        const int te = tau * Edge::BYTES;
        wv_edge_load<R, NEQ, WVB, AUX>(ra, x.act ? off_in_a : WV_OOB, EA, clamp(te + SHA * Edge::BYTES, last_e), ea);
        wv_edge_load<R, NEQ, WVA, AUX>(rb, x.act ? off_in_b : WV_OOB, EB, clamp(te + SHB * Edge::BYTES, last_e), x.eb);
    };
    auto load = [&](const int s, WaveIn<R, NEQ>& x) __attribute__((always_inline)) {
        const int tau = FORWARD ? s : nrow - 1 - s;
        x.act = (unsigned)(tau - start) < (unsigned)NJ1;
        const int vo = x.act ? lane * 16 : WV_OOB;
        const int v8 = x.act ? lane * (int)sizeof(R) : WV_OOB;
        const int row = clamp(tau * Row::BYTES, last_w), row4 = row + 4096;
        x.row = row;
        x.erow = clamp(tau * Edge::BYTES, last_e);
        R v[28];
#pragma unroll
        for (int g = 0; g < 28 / VL; g++) {
            const int q = g * VL;
            if (MF ? q >= WV_K : q < WV_C2) continue;
            const wv_u4 w = __builtin_amdgcn_raw_buffer_load_b128(g < 8 ? rw0 : rw1, vo + (g % 4) * Row::GB,
                                                                  (g / 4) % 2 ? row4 : row, 0);
#pragma unroll
            for (int e = 0; e < VL; e++) v[q + e] = WvVec<R>::get(w, e);
        }
        if constexpr (sizeof(R) == 8) {
            const wv_u2 w = __builtin_amdgcn_raw_buffer_load_b64(rw1, v8 + (Row::S8B - 8192 - 4096), row4, 0);
            x.s[8] = __hiloint2double((int)w[1], (int)w[0]);
        } else {
            x.s[8] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rw0, v8 + (Row::S8B - 4096), row4, 0));
        }
        if constexpr (MF) {
#pragma unroll
            for (int L = 0; L < NEQ; L++) x.d[L] = v[WV_D + L];
            x.sa = v[WV_SA];
            x.sb = v[WV_SB];
            x.c2 = v[WV_C2];
        } else {
#pragma unroll
            for (int L = 0; L < NEQ; L++) x.d[L] = v[WV_K + L];
            x.sa = v[WV_STEPT];
            x.sb = v[WV_CVS];
            x.rf1 = v[WV_RF1];
        }
#pragma unroll
        for (int q = 0; q < 3; q++) {
            x.u[q] = v[WV_U + q];
            x.rds[q] = v[WV_RDS + q];
        }
#pragma unroll
        for (int q = 0; q < 8; q++) x.s[q] = v[WV_S + q];
        edges(std::integral_constant<int, WV_SC1>{}, tau, x, x.ea);
    };

    R oa[NEQ], om[NEQ], kb[NEQ];  // previous row: terms along i and j, and the k term read back for this lane
#pragma unroll
    for (int L = 0; L < NEQ; L++) oa[L] = om[L] = kb[L] = R(0);
    WaveIn<R, NEQ> ring[PD];

    // one row: ring[Q] holds its inputs
    auto step = [&](auto uf, auto qc, const int s) __attribute__((always_inline)) {
        constexpr bool UF = decltype(uf)::value;
        constexpr int Q = decltype(qc)::value;
        WaveIn<R, NEQ>& x = ring[Q];
        // the row's loads are complete: what may still be in flight are the operations issued
        // after them, the stores of their step and whole steps since.  (A test follows every load
        // through the assembly; the compiler's own waits alone passed it too.)
        __builtin_amdgcn_s_waitcnt(wv_vmcnt(NST + (PD - 1) * (NLD + NST)));
        __builtin_amdgcn_sched_barrier(0);
        // the i terms from the row's previous lanes; the first lane of a DPP row keeps its edge value
#pragma unroll
        for (int L = 0; L < NEQ; L++) x.ea[L] = wv_shift<FORWARD>(x.ea[L], oa[L]);
        R dq[NEQ], e = R(0), hu2 = R(0);
        // incoming terms summed in i, j, k order, and the increment; the value returned is NaN if
        // any of the sums is
        auto front = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int L = 0; L < NEQ; L++) {
                const R sum = x.ea[L] + om[L] + (kb[L] + x.eb[L]);
                if constexpr (MF)
                    dq[L] = FORWARD ? wv_fma(x.d[L], x.sa, sum * x.sb) : wv_fma(-sum, x.sb, x.d[L]);
                else
                    dq[L] = FORWARD ? wv_fma(x.d[L], x.sa, sum * x.sb) * x.rf1 : wv_fma(-(sum * x.sb), x.rf1, x.d[L]);
            }
            if constexpr (!MF) {
                return dq[0] + dq[1];
            } else {
                hu2 = R(0.5) * wv_dot<UF>(x.u, x.u);
                e = wv_fma(hu2, dq[0], dq[4] - wv_dot<false>(x.u, dq + 1));
                return e;
            }
        };
        R chk = front();
        if (__builtin_expect(__any(chk != chk), 0)) {
            // some edge value was not there yet (or the flow has diverged): poll for it, and
            // refresh the rows already loaded
            const int tau = FORWARD ? s : nrow - 1 - s;
            for (int spins = 0;; spins++) {
                // the next row's as well: a wave that follows its upstream tile that closely would
                // otherwise poll on every row
                int pend = 0;
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const WaveIn<R, NEQ>& y = ring[(Q + r) % PD];
#pragma unroll
                    for (int L = 0; L < NEQ; L++) pend |= (int)wv_pending<R>(y.ea[L]) | (int)wv_pending<R>(y.eb[L]);
                }
                if (!__any(pend)) break;
                if (spins > spin_limit ||
                    ((spins & 63) == 63 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
                    __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
                R ea[NEQ];
                edges(std::integral_constant<int, WV_POLL>{}, tau, x, ea);
#pragma unroll
                for (int r = 1; r < PD; r++) {
                    WaveIn<R, NEQ>& y = ring[(Q + r) % PD];
                    edges(std::integral_constant<int, WV_POLL>{}, FORWARD ? tau + r : tau - r, y, y.ea);
                }
#pragma unroll
                for (int L = 0; L < NEQ; L++) x.ea[L] = in_a ? ea[L] : x.ea[L];
                __builtin_amdgcn_s_waitcnt(wv_vmcnt(0));  // nothing of this loop is in flight after it
            }
            (void)front();
        }
        // the flux Jacobian's product as adq_prep and adq_dir form it
        R dp = R(0), H = R(0), q4 = R(0), wd[3];
        if constexpr (MF) {
            const R Gm1 = R(1.4 - 1.0);
            dp = Gm1 * e;
            H = wv_fma(R(1) / Gm1, x.c2, hu2);
            q4 = wv_fma(-H, dq[0], wv_fma(Gm1, e, dq[4]));
#pragma unroll
            for (int q = 0; q < 3; q++) wd[q] = wv_fma(-x.u[q], dq[0], dq[q + 1]);
        }
        auto term = [&](int d, R o[NEQ]) __attribute__((always_inline)) {
            const R* S = x.s + d * 3;
            const R rd = FORWARD ? x.rds[d] : -x.rds[d];
            const R VP = wv_dot<UF>(x.u, S);
            if constexpr (MF) {
                const R Sm = wv_dot<false>(S, dq + 1);
                o[0] = wv_fma(rd, dq[0], Sm);
#pragma unroll
                for (int q = 0; q < 3; q++)
                    o[q + 1] = wv_fma(rd, dq[q + 1], wv_fma(S[q], dp, wv_fma(VP, wd[q], x.u[q] * Sm)));
                o[4] = wv_fma(rd, dq[4], wv_fma(H, Sm, VP * q4));
            } else {
#pragma unroll
                for (int L = 0; L < NEQ; L++) o[L] = wv_fma(VP, dq[L], rd * dq[L]);
            }
        };
        // the k terms first: their way through LDS overlaps the other directions
        R ok[NEQ];
        term(2, ok);
#pragma unroll
        for (int L = 0; L < NEQ; L++) lds_st[L * 80] = ok[L];
        wv_lds_order();
#pragma unroll
        for (int L = 0; L < NEQ; L++) kb[L] = lds_ld[L * 80];
        wv_lds_order();
        term(0, oa);
        term(1, om);
        const bool act = x.act;
        const int row = x.row, erow = x.erow;
        // the row PD ahead before this row's stores: memory operations complete in order, so a wait
        // for loads is also one for every older store, and the stores' way to memory is long
        load(s + PD, x);
        const int vo = act ? lane * 16 : WV_OOB;
        wv_edge_store<R, NEQ, WVA>(ro, act ? off_out_b : WV_OOB, EB, erow, ok);
        wv_edge_store<R, NEQ, WVB>(ro, act ? off_out_a : WV_OOB, EA, erow, oa);
        if constexpr (MF) {
#pragma unroll
            for (int g = 0; g < 4 / VL; g++)
                __builtin_amdgcn_raw_buffer_store_b128(WvVec<R>::put(dq + g * VL), rw0, vo + g * Row::GB, row, 0);
            if constexpr (sizeof(R) == 8) {
                const wv_u2 w = {(unsigned)__double2loint(dq[4]), (unsigned)__double2hiint(dq[4])};
                __builtin_amdgcn_raw_buffer_store_b64(w, rw0, vo + 2 * Row::GB, row, 0);
            } else {
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dq[4]), rw0, vo + Row::GB, row, 0);
            }
        } else if constexpr (sizeof(R) == 8) {
            constexpr int g = WV_K / VL;
            __builtin_amdgcn_raw_buffer_store_b128(WvVec<R>::put(dq), rw1, vo + (g % 4) * Row::GB, row + 4096, 0);
        } else {
            constexpr int g = WV_K / VL;
            const wv_u2 w = {__float_as_uint(dq[0]), __float_as_uint(dq[1])};
            __builtin_amdgcn_raw_buffer_store_b64(w, rw0, vo + (g % 4) * Row::GB, row + 4096, 0);
        }
    };
    // PD rows are in flight: a row's inputs are loaded PD steps ahead into the registers the
    // step before has freed.  Steps past the last row, and the one before the first where the
    // tile starts on an odd step of the sweep, have no active lane.
    const int par = ALT && !FORWARD ? (NI1 + NK1 - na - nb) & 1 : 0;
#pragma unroll
    for (int q = 0; q < PD; q++) load(q - par, ring[q]);
    // all of them, once: with loads of the prologue's order in flight at the loop's head, the
    // compiler's counter waits inside the loop would hold up the rows in flight there
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(wv_vmcnt(0));
    __builtin_amdgcn_sched_barrier(0);
    constexpr int UN = ALT && PD % 2 ? 2 * PD : PD;  // whole ring turns and whole alternations
    static_assert(UN <= 6, "rows per turn of the loop");
    int s = -par;
    do {  // (a tile has a row)
#define WV_STEP(q)                                                                                            \
    if constexpr (q < UN)                                                                                     \
        step(std::integral_constant<bool, ALT && q % 2 == 0>{}, std::integral_constant<int, q % PD>{}, s + q);
        WV_STEP(0) WV_STEP(1) WV_STEP(2) WV_STEP(3) WV_STEP(4) WV_STEP(5)
#undef WV_STEP
        s += UN;
    } while (s < nrow);
}

// One workgroup per tile: wave 0 the mean flow and wave 1 the k-omega equations (KIND 7), or one
// wave for one of them (KIND 5, 2).  ctr: the sweep's item counter; items are taken in the table's
// order (upstream tiles first), the backward sweep in the reverse.
template <typename R, bool FORWARD, int KIND, int PD, int WPE, bool ALT>
__global__ void __launch_bounds__(KIND == 7 ? 128 : 64, WPE)
    k_lusgs_wave(Fields f, const BlkInfo* __restrict__ blks, const WaveTile* __restrict__ tiles, int ntiles,
                 int* __restrict__ ctr, R* __restrict__ edge, int* __restrict__ err, int spin_limit)
{
    __shared__ R lds[(KIND == 7 ? 7 : KIND) * 80];
    __shared__ int s_item;
    if (threadIdx.x == 0) s_item = atomicAdd(ctr, 1);
    __syncthreads();
    const int q = __builtin_amdgcn_readfirstlane(s_item);
    const WaveTile tl = tiles[FORWARD ? q : ntiles - 1 - q];
    const BlkInfo b = blks[tl.blk];
    const bool kw = KIND == 2 || (KIND == 7 && __builtin_amdgcn_readfirstlane((int)threadIdx.x) >= 64);
    if (KIND != 2 && !kw)
        wave_sweep<R, FORWARD, 5, PD, ALT>(f, b, tl.ta, tl.tb, lds, edge, err, spin_limit);
    else if (KIND != 5)
        wave_sweep<R, FORWARD, 2, PD, ALT>(f, b, tl.ta, tl.tb, lds + (KIND == 7 ? 5 * 80 : 0), edge, err, spin_limit);
}
