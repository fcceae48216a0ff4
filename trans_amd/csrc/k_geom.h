// Geometry pre-processing on the device: the brute-force wall distance of
// Geom/CalcDst.F90:121-158 (every cell centre against every wall panel centre).
#pragma once
#include <hip/hip_runtime.h>

// Panels are staged through LDS in tiles; each thread keeps the running minimum of the
// squared distance of WD_CPT cells, so a panel read from LDS serves WD_CPT cells.  The
// squared distance is formed as the reference forms it, ((dx*dx + dy*dy) + dz*dz) with
// d = cell - panel, and the minimum is exact, so the result does not depend on the tiling.
constexpr int WD_TILE = 512;
constexpr int WD_CPT = 4;

__global__ void __launch_bounds__(256) k_wall_distance(const double* __restrict__ cell, long ncell,
                                                       const double* __restrict__ pan, long npan,
                                                       double* __restrict__ d2min)
{
    __shared__ double sx[WD_TILE], sy[WD_TILE], sz[WD_TILE];
    const long base = ((long)blockIdx.x * blockDim.x) * WD_CPT + threadIdx.x;
    double cx[WD_CPT], cy[WD_CPT], cz[WD_CPT], best[WD_CPT];
#pragma unroll
    for (int q = 0; q < WD_CPT; q++) {
        const long c = base + (long)q * blockDim.x;  // cells of one thread are blockDim apart: coalesced loads
        const bool ok = c < ncell;
        cx[q] = ok ? cell[c] : 0.0;
        cy[q] = ok ? cell[ncell + c] : 0.0;
        cz[q] = ok ? cell[2 * ncell + c] : 0.0;
        best[q] = 1.0e20;
    }
    for (long t0 = 0; t0 < npan; t0 += WD_TILE) {
        const int nt = (int)((npan - t0) < WD_TILE ? (npan - t0) : WD_TILE);
        __syncthreads();
        for (int q = threadIdx.x; q < nt; q += blockDim.x) {
            sx[q] = pan[t0 + q];
            sy[q] = pan[npan + t0 + q];
            sz[q] = pan[2 * npan + t0 + q];
        }
        __syncthreads();
        for (int p = 0; p < nt; p++) {
            const double px = sx[p], py = sy[p], pz = sz[p];
#pragma unroll
            for (int q = 0; q < WD_CPT; q++) {
                const double dx = cx[q] - px, dy = cy[q] - py, dz = cz[q] - pz;
                const double ddd = dx * dx + dy * dy + dz * dz;
                best[q] = ddd < best[q] ? ddd : best[q];
            }
        }
    }
#pragma unroll
    for (int q = 0; q < WD_CPT; q++) {
        const long c = base + (long)q * blockDim.x;
        if (c < ncell) d2min[c] = best[q];
    }
}

// ---------------------------------------------------------------------------------------
// O(N) metrics of one block (Geom/CalcDst.F90:170-632): cell centres and boundary face
// centres, face area vectors and areas, face-to-face lengths, neighbour distances, volumes
// and the first-ghost copies.  Arrays use the block's padded layout (bounds -2:N+2 on each
// axis, component first); every expression keeps the host restatement's operation order,
// so the results are bitwise equal to it (the angle thtc comes from the device atan2).
struct GeomGrid {
    int ni, nj, nk;  // points
    long nx, ny;     // padded extents ni+5, nj+5
    __host__ __device__ long at(int i, int j, int k) const { return (i + 2) + nx * ((j + 2) + ny * (long)(k + 2)); }
};

struct GeomOut {
    double *xc, *yc, *zc, *thtc, *rad, *aleng, *aseng, *vol;
    double* sd;     // 9 components first: (d-1) + 3*x
    double *grad, *alagm;  // 3 components first
};

// centres: interior cells and the boundary face centres at index 0 / N
__global__ void __launch_bounds__(256) k_geom_centres(GeomGrid g, const double* __restrict__ X,
                                                      const double* __restrict__ Y, const double* __restrict__ Z,
                                                      GeomOut o)
{
    const int ni = g.ni, nj = g.nj, nk = g.nk;
    const long n0 = ni + 1, n1 = nj + 1;
    const long lin = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (lin >= n0 * n1 * (nk + 1)) return;
    const int i = (int)(lin % n0), j = (int)((lin / n0) % n1), k = (int)(lin / (n0 * n1));
    const bool ii = i >= 1 && i <= ni - 1, ji = j >= 1 && j <= nj - 1, ki = k >= 1 && k <= nk - 1;
    const double* P[3] = {X, Y, Z};
    double* C[3] = {o.xc, o.yc, o.zc};
    const long c = g.at(i, j, k);
    if (ii && ji && ki) {
        for (int q = 0; q < 3; q++) {
            const double* A = P[q];
            C[q][c] = (A[g.at(i + 1, j + 1, k + 1)] + A[g.at(i + 1, j + 1, k)] + A[g.at(i + 1, j, k + 1)] +
                       A[g.at(i + 1, j, k)] + A[g.at(i, j + 1, k + 1)] + A[g.at(i, j + 1, k)] + A[g.at(i, j, k + 1)] +
                       A[g.at(i, j, k)]) /
                      8.0;
        }
        const double yc = o.yc[c], zc = o.zc[c];
        o.thtc[c] = atan2(zc, yc);
        o.rad[c] = sqrt(yc * yc + zc * zc);
        return;
    }
    if ((i == 0 || i == ni) && ji && ki) {
        const int f = i == 0 ? 1 : ni;
        for (int q = 0; q < 3; q++) {
            const double* A = P[q];
            C[q][c] = (A[g.at(f, j, k)] + A[g.at(f, j + 1, k)] + A[g.at(f, j, k + 1)] + A[g.at(f, j + 1, k + 1)]) / 4.0;
        }
    } else if ((j == 0 || j == nj) && ii && ki) {
        const int f = j == 0 ? 1 : nj;
        for (int q = 0; q < 3; q++) {
            const double* A = P[q];
            C[q][c] = (A[g.at(i, f, k)] + A[g.at(i + 1, f, k)] + A[g.at(i, f, k + 1)] + A[g.at(i + 1, f, k + 1)]) / 4.0;
        }
    } else if ((k == 0 || k == nk) && ii && ji) {
        const int f = k == 0 ? 1 : nk;
        for (int q = 0; q < 3; q++) {
            const double* A = P[q];
            C[q][c] = (A[g.at(i, j, f)] + A[g.at(i + 1, j, f)] + A[g.at(i, j + 1, f)] + A[g.at(i + 1, j + 1, f)]) / 4.0;
        }
    }
}

// face area vectors S = (R1 x R2) / 2 * dl and areas |S| (plus tiny under the root) of the
// faces of direction DIR; dl orients them by the first cell's i direction (:198-210)
template <int DIR>
__global__ void __launch_bounds__(256) k_geom_faces(GeomGrid g, const double* __restrict__ X,
                                                    const double* __restrict__ Y, const double* __restrict__ Z,
                                                    GeomOut o, double tiny)
{
    const int ni = g.ni, nj = g.nj, nk = g.nk;
    const int n0 = DIR == 1 ? ni : ni - 1, n1 = DIR == 2 ? nj : nj - 1, n2 = DIR == 3 ? nk : nk - 1;
    const long lin = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (lin >= (long)n0 * n1 * n2) return;
    const int i = (int)(lin % n0) + 1, j = (int)((lin / n0) % n1) + 1, k = (int)(lin / ((long)n0 * n1)) + 1;
    const double* P[3] = {X, Y, Z};
    double dl;
    {
        double xv[3], r1[3], r2[3];
        for (int q = 0; q < 3; q++) {
            const double* C = q == 0 ? o.xc : (q == 1 ? o.yc : o.zc);
            xv[q] = (C[g.at(1, 1, 1)] - C[g.at(2, 1, 1)]) * -1.0;
            r1[q] = P[q][g.at(1, 2, 2)] - P[q][g.at(1, 1, 1)];
            r2[q] = P[q][g.at(1, 1, 2)] - P[q][g.at(1, 2, 1)];
        }
        const double sv[3] = {(r1[1] * r2[2] - r1[2] * r2[1]) * 0.5, (r1[2] * r2[0] - r1[0] * r2[2]) * 0.5,
                              (r1[0] * r2[1] - r1[1] * r2[0]) * 0.5};
        dl = xv[0] * sv[0] + xv[1] * sv[1] + xv[2] * sv[2] < 0 ? -1.0 : 1.0;
    }
    double R1[3], R2[3];
    for (int q = 0; q < 3; q++) {
        const double* A = P[q];
        if (DIR == 1) {
            R1[q] = A[g.at(i, j + 1, k + 1)] - A[g.at(i, j, k)];
            R2[q] = A[g.at(i, j, k + 1)] - A[g.at(i, j + 1, k)];
        } else if (DIR == 2) {
            R1[q] = A[g.at(i, j, k + 1)] - A[g.at(i + 1, j, k)];
            R2[q] = A[g.at(i + 1, j, k + 1)] - A[g.at(i, j, k)];
        } else {
            R1[q] = A[g.at(i + 1, j, k)] - A[g.at(i, j + 1, k)];
            R2[q] = A[g.at(i + 1, j + 1, k)] - A[g.at(i, j, k)];
        }
    }
    const double S0 = (R1[1] * R2[2] - R1[2] * R2[1]) * 0.5 * dl;
    const double S1 = (R1[2] * R2[0] - R1[0] * R2[2]) * 0.5 * dl;
    const double S2 = (R1[0] * R2[1] - R1[1] * R2[0]) * 0.5 * dl;
    const long c = g.at(i, j, k);
    o.sd[(DIR - 1) + 9 * c] = S0;
    o.sd[(DIR - 1) + 3 + 9 * c] = S1;
    o.sd[(DIR - 1) + 6 + 9 * c] = S2;
    o.grad[(DIR - 1) + 3 * c] = sqrt(S0 * S0 + S1 * S1 + S2 * S2 + tiny);
}

__device__ __forceinline__ double geom_fc(const GeomGrid& g, const double* A, int i0, int i1, int j0, int j1, int k0,
                                          int k1)
{
    return 0.25 * (A[g.at(i0, j0, k0)] + A[g.at(i1, j1, k0)] + A[g.at(i0, j0, k1)] + A[g.at(i1, j1, k1)]);
}

// face-to-face lengths Alagm (:289-325), neighbour distances aleng/aseng (:430-476) and
// volumes (:481-515) of the interior cells
__global__ void __launch_bounds__(256) k_geom_cells(GeomGrid g, const double* __restrict__ X,
                                                    const double* __restrict__ Y, const double* __restrict__ Z,
                                                    GeomOut o)
{
    const int NI1 = g.ni - 1, NJ1 = g.nj - 1, NK1 = g.nk - 1;
    const long lin = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (lin >= (long)NI1 * NJ1 * NK1) return;
    const int i = (int)(lin % NI1) + 1, j = (int)((lin / NI1) % NJ1) + 1, k = (int)(lin / ((long)NI1 * NJ1)) + 1;
    const double* P[3] = {X, Y, Z};
    const long c = g.at(i, j, k);
    {
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        for (int q = 0; q < 3; q++) {
            const double* A = P[q];
            const double w = geom_fc(g, A, i, i, j, j + 1, k, k + 1), e = geom_fc(g, A, i + 1, i + 1, j, j + 1, k, k + 1);
            const double s = geom_fc(g, A, i, i + 1, j, j, k, k + 1), n = geom_fc(g, A, i, i + 1, j + 1, j + 1, k, k + 1);
            const double b = geom_fc(g, A, i, i + 1, j, j + 1, k, k), t = geom_fc(g, A, i, i + 1, j, j + 1, k + 1, k + 1);
            s0 = s0 + (w - e) * (w - e);
            s1 = s1 + (s - n) * (s - n);
            s2 = s2 + (b - t) * (b - t);
        }
        o.alagm[0 + 3 * c] = sqrt(s0);
        o.alagm[1 + 3 * c] = sqrt(s1);
        o.alagm[2 + 3 * c] = sqrt(s2);
    }
    {
        const double* C[3] = {o.xc, o.yc, o.zc};
        auto dd = [&](int di, int dj, int dk) {
            const long cn = g.at(i + di, j + dj, k + dk);
            const double a = C[0][cn] - C[0][c], b = C[1][cn] - C[1][c], e = C[2][cn] - C[2][c];
            return sqrt(a * a + b * b + e * e);
        };
        const double dw = dd(-1, 0, 0), de = dd(1, 0, 0), ds = dd(0, -1, 0), dn = dd(0, 1, 0), dlo = dd(0, 0, -1),
                     du = dd(0, 0, 1);
        double cand[6] = {dw, de, ds, dn, dlo, du};
        int nc = 6;
        if (NI1 == 2) {
            cand[0] = ds, cand[1] = dn, cand[2] = dlo, cand[3] = du;
            nc = 4;
        }
        if (NJ1 == 2) {
            cand[0] = dw, cand[1] = de, cand[2] = dlo, cand[3] = du;
            nc = 4;
        }
        if (NK1 == 2) {
            cand[0] = dw, cand[1] = de, cand[2] = ds, cand[3] = dn;
            nc = 4;
        }
        double mx = cand[0], mn = cand[0];
        for (int q = 1; q < nc; q++) {
            mx = fmax(mx, cand[q]);
            mn = fmin(mn, cand[q]);
        }
        o.aleng[c] = mx;
        o.aseng[c] = mn;
    }
    {
        const long p = g.at(i + 1, j + 1, k + 1);
        const long pi = g.at(i, j + 1, k + 1), pj = g.at(i + 1, j, k + 1), pk = g.at(i + 1, j + 1, k);
        double si = 0.0, sj = 0.0, sk = 0.0;
        for (int x = 0; x < 3; x++) {
            const double* A = P[x];
            si = si + (A[p] - A[pi]) * o.sd[0 + 3 * x + 9 * c];
            sj = sj + (A[p] - A[pj]) * o.sd[1 + 3 * x + 9 * c];
            sk = sk + (A[p] - A[pk]) * o.sd[2 + 3 * x + 9 * c];
        }
        double om = 0.0;
        om = om + si;
        om = om + sj;
        om = om + sk;
        o.vol[c] = (1.0 / 3.0) * om;
    }
}

// first-ghost copies of Vol and Alagm (:579-608), Grad's face-0 copy, and the SD extension
// to faces 0 and N+1 (:611-632); every read is of an interior entry no thread writes
__global__ void __launch_bounds__(256) k_geom_ghosts(GeomGrid g, GeomOut o)
{
    const int NI = g.ni, NJ = g.nj, NK = g.nk, NI1 = NI - 1, NJ1 = NJ - 1, NK1 = NK - 1;
    const long n0 = NI + 2, n1 = NJ + 2;
    const long lin = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (lin >= n0 * n1 * (NK + 2)) return;
    const int i = (int)(lin % n0), j = (int)((lin / n0) % n1), k = (int)(lin / (n0 * n1));
    const bool ii = i >= 1 && i <= NI1, ji = j >= 1 && j <= NJ1, ki = k >= 1 && k <= NK1;
    const long c = g.at(i, j, k);
    if (ji && ki && (i == 0 || i == NI)) {
        const long s = g.at(i == 0 ? 1 : NI1, j, k);
        o.vol[c] = o.vol[s];
        o.alagm[0 + 3 * c] = o.alagm[0 + 3 * s];
        if (i == 0) o.grad[0 + 3 * c] = o.grad[0 + 3 * s];
    }
    if (ii && ki && (j == 0 || j == NJ)) {
        const long s = g.at(i, j == 0 ? 1 : NJ1, k);
        o.vol[c] = o.vol[s];
        o.alagm[1 + 3 * c] = o.alagm[1 + 3 * s];
        if (j == 0) o.grad[1 + 3 * c] = o.grad[1 + 3 * s];
    }
    if (ii && ji && (k == 0 || k == NK)) {
        const long s = g.at(i, j, k == 0 ? 1 : NK1);
        o.vol[c] = o.vol[s];
        o.alagm[2 + 3 * c] = o.alagm[2 + 3 * s];
        if (k == 0) o.grad[2 + 3 * c] = o.grad[2 + 3 * s];
    }
    const bool jw = j >= 1 && j <= NJ, kw = k >= 1 && k <= NK, iw = i >= 1 && i <= NI;
    if (jw && kw && (i == 0 || i == NI + 1)) {
        const long s = g.at(i == 0 ? 2 : NI1, j, k);
        for (int x = 0; x < 3; x++) o.sd[0 + 3 * x + 9 * c] = o.sd[0 + 3 * x + 9 * s];
    }
    if (iw && kw && (j == 0 || j == NJ + 1)) {
        const long s = g.at(i, j == 0 ? 2 : NJ1, k);
        for (int x = 0; x < 3; x++) o.sd[1 + 3 * x + 9 * c] = o.sd[1 + 3 * x + 9 * s];
    }
    if (iw && jw && (k == 0 || k == NK + 1)) {
        const long s = g.at(i, j, k == 0 ? 2 : NK1);
        for (int x = 0; x < 3; x++) o.sd[2 + 3 * x + 9 * c] = o.sd[2 + 3 * x + 9 * s];
    }
}

// ---------------------------------------------------------------------------------------
// The same minimum over fewer pairs, for many points: cells and panels are put in Morton order
// (32^3 boxes, counting sort), panels in tiles of 64 with their bounding
// boxes.  A wave holds 64 consecutive cells; it evaluates the tile that is nearest to
// its cells' box, then every tile whose box is not farther than its largest minimum so far from its
// cells' box, and then not farther from some cell than that cell's minimum.  A
// skipped tile's pairs are all above the minima by more than their rounding (WB_SLACK), the pairs
// evaluated are formed as above, and a minimum does not depend on the order, so the result is the
// same bit for bit.  485 000 cells and 30 000 panels: 1.2 ms of kernels and 2.0 ms for the call, with
// every pair 6 ms and 7.9 ms.  With two and four cells per lane the last kernel took 1.3 and 1.6 ms
// instead of 1.1 ms (larger boxes).
//
// The boxes' faces are quantiles of the coordinates, taken from a sample, so that each slab holds
// about 1/32 of the points however they are spread.  Equal boxes of the bounding box put nearly all
// points into one where a single point was far away.  Calls with equal boxes, and now (with every
// pair): 485 000 x 30 000 with one far cell 18.5 ms, 2.0 ms (8.0 ms); 485 000 x 2 048 with a far cell
// and a far panel 12.6 ms, 1.1 ms (2.1 ms); an O-grid stretched to 100 chords, 512 000 x 20 480,
// 3.2 ms, 1.9 ms (6.4 ms); 100 000 x 10 000 coincident points 4.6 ms, 1.8 ms (2.0 ms).  What is still
// slower than every pair is a set none of whose panels is nearer than another: 485 000 cells on the
// axis of a cylinder of 30 000 panels 8.9 ms (7.6 ms).
constexpr int WB_BITS = 5, WB_SIDE = 1 << WB_BITS, WB_BINS = 1 << (3 * WB_BITS);
constexpr int WB_TILE = 64;
constexpr int WB_SAMPLE = 512;
constexpr double WB_SLACK = 1.0 + 1.0e-9;

// A set of points in sorted form, and its tables.
struct WbSet {
    const double* pt;  // x, then y, then z of all points
    long n;
    const double* faces;  // 3 x WB_SIDE
    int* bins;
    double4* out;  // x, y, z, 0 per point, in order
    int* from;     // where a point came from, or null
};

// The faces between the slabs, one workgroup per set of points and coordinate (0 to 5): entry k of
// the 32 is the lower face of slab k (entry 0 is not used).  The sample is one point of each of
// WB_SAMPLE equal runs of the points, at a scattered place, so that the strides of a grid do not
// show in it.  The other workgroups clear the tables.
__global__ void __launch_bounds__(WB_SAMPLE) k_wb_faces(WbSet cells, WbSet panels, double* __restrict__ faces)
{
    const int t = threadIdx.x;
    if (blockIdx.x >= 6) {
        int* const bins = cells.bins;  // (the panels' behind them)
        for (int k = (blockIdx.x - 6) * WB_SAMPLE + t; k < 2 * WB_BINS; k += (gridDim.x - 6) * WB_SAMPLE) bins[k] = 0;
        return;
    }
    __shared__ double x[WB_SAMPLE];
    const WbSet& s = blockIdx.x < 3 ? cells : panels;
    const long from = s.n * t / WB_SAMPLE, len = max(1L, s.n * (t + 1) / WB_SAMPLE - from);
    const double v = s.pt[blockIdx.x % 3 * s.n + from + (long)((unsigned)t * 2654435761u >> 8) % len];
    x[t] = v != v ? INFINITY : v;  // (a NaN has no place in an order)
    // bitonic sort
    for (int k = 2; k <= WB_SAMPLE; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            __syncthreads();
            const int o = t ^ j;
            if (o > t) {
                const double a = x[t], b = x[o];
                if ((a > b) == ((t & k) == 0)) {
                    x[t] = b;
                    x[o] = a;
                }
            }
        }
    __syncthreads();
    if (t < WB_SIDE) faces[blockIdx.x * WB_SIDE + t] = x[t * (WB_SAMPLE / WB_SIDE)];
}

// The set that a workgroup takes 256 points of, and the first of them: the cells, then the panels.
__device__ __forceinline__ const WbSet& wb_share(const WbSet& cells, const WbSet& panels, long& base)
{
    const long nc = (cells.n + 255) / 256;
    base = ((long)blockIdx.x < nc ? (long)blockIdx.x : (long)blockIdx.x - nc) * 256;
    return (long)blockIdx.x < nc ? cells : panels;
}

// Morton number of point q among the boxes; faces: of its set of points, in LDS.
__device__ __forceinline__ int wb_bin(const double* __restrict__ pt, long n, long q, const double* faces)
{
    int m = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double x = pt[d * n + q];
        int k = 0;  // (of a NaN too)
#pragma unroll
        for (int s = WB_SIDE / 2; s > 0; s >>= 1) k += x >= faces[d * WB_SIDE + k + s] ? s : 0;
#pragma unroll
        for (int b = 0; b < WB_BITS; b++) m |= ((k >> b) & 1) << (3 * b + d);
    }
    return m;
}

// Adds 1 to counter `m` for every active lane and returns the lane's place.  The lanes that share
// the first lane's counter, of which there are many where points coincide, add theirs together.
__device__ __forceinline__ int wb_add(int* __restrict__ bins, int m)
{
    const int lead = __builtin_amdgcn_readfirstlane(m);
    const unsigned long long same = __ballot(m == lead);
    if (m != lead) return atomicAdd(bins + m, 1);
    const int before = __popcll(same & ((1ull << (threadIdx.x & 63)) - 1));
    int at = 0;
    if (before == 0) at = atomicAdd(bins + m, __popcll(same));
    return __builtin_amdgcn_readfirstlane(at) + before;
}

__global__ void __launch_bounds__(256) k_wb_count(WbSet cells, WbSet panels)
{
    __shared__ double s_faces[3 * WB_SIDE];
    long base;
    const WbSet& s = wb_share(cells, panels, base);
    if (threadIdx.x < 3 * WB_SIDE) s_faces[threadIdx.x] = s.faces[threadIdx.x];
    __syncthreads();
    const long q = base + threadIdx.x;
    if (q < s.n) (void)wb_add(s.bins, wb_bin(s.pt, s.n, q, s_faces));
}

// Counts to first positions; one workgroup per table.
__global__ void __launch_bounds__(1024) k_wb_scan(int* __restrict__ tables)
{
    __shared__ int part[1024];
    int* const t = tables + (long)blockIdx.x * WB_BINS;
    constexpr int PER = WB_BINS / 1024;
    int sum = 0;
    for (int q = 0; q < PER; q++) sum += t[threadIdx.x * PER + q];
    part[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int v = (int)threadIdx.x >= off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    int at = part[threadIdx.x] - sum;
    for (int q = 0; q < PER; q++) {
        const int c = t[threadIdx.x * PER + q];
        t[threadIdx.x * PER + q] = at;
        at += c;
    }
}

// Points to their sorted places.
__global__ void __launch_bounds__(256) k_wb_scatter(WbSet cells, WbSet panels)
{
    __shared__ double s_faces[3 * WB_SIDE];
    long base;
    const WbSet& s = wb_share(cells, panels, base);
    if (threadIdx.x < 3 * WB_SIDE) s_faces[threadIdx.x] = s.faces[threadIdx.x];
    __syncthreads();
    const long q = base + threadIdx.x;
    if (q >= s.n) return;
    const int at = wb_add(s.bins, wb_bin(s.pt, s.n, q, s_faces));
    s.out[at] = make_double4(s.pt[q], s.pt[s.n + q], s.pt[2 * s.n + q], 0.0);
    if (s.from) s.from[at] = (int)q;
}

// Bounding boxes of the panel tiles: 3 lower, 3 upper bounds, each ntile values; one wave per tile.
__global__ void __launch_bounds__(64) k_wb_tiles(const double4* __restrict__ pan, int npan, int ntile,
                                                 double* __restrict__ tb)
{
    const int q = min((int)(blockIdx.x * WB_TILE + threadIdx.x), npan - 1);
    const double4 p = pan[q];
    double lo[3] = {p.x, p.y, p.z}, hi[3] = {p.x, p.y, p.z};
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], __shfl_xor(lo[d], off, 64));
            hi[d] = fmax(hi[d], __shfl_xor(hi[d], off, 64));
        }
    if (threadIdx.x == 0)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            tb[(long)d * ntile + blockIdx.x] = lo[d];
            tb[(long)(3 + d) * ntile + blockIdx.x] = hi[d];
        }
}

// One wave per workgroup: distances of 64 sorted cells.
__global__ void __launch_bounds__(64) k_wb_distance(const double4* __restrict__ cell, const int* __restrict__ from,
                                                    long ncell, const double4* __restrict__ pan, int npan,
                                                    const double* __restrict__ tb, int ntile, double* __restrict__ dst)
{
    const int lane = threadIdx.x;
    const long me = (long)blockIdx.x * 64 + lane;
    const double4 c4 = cell[min(me, ncell - 1)];  // past the end: the last cell again
    const double c[3] = {c4.x, c4.y, c4.z};
    double best = 1.0e20;
    double lo[3] = {c4.x, c4.y, c4.z}, hi[3] = {c4.x, c4.y, c4.z};
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], __shfl_xor(lo[d], off, 64));
            hi[d] = fmax(hi[d], __shfl_xor(hi[d], off, 64));
        }
    // squared distance between the box from a to b and that of tile t (a NaN counts as 0)
    auto bound = [&](const double* a, const double* b, int t) {
        double s = 0.0;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double x = fmax(fmax(tb[(long)d * ntile + t] - b[d], a[d] - tb[(long)(3 + d) * ntile + t]), 0.0);
            s += x * x;
        }
        return s;
    };
    auto tile = [&](int t) {
        const double4* const p = pan + (long)t * WB_TILE;
        const int n = min(WB_TILE, npan - t * WB_TILE);
#pragma unroll 4
        for (int k = 0; k < n; k++) {
            const double4 w = p[k];
            const double dx = c[0] - w.x, dy = c[1] - w.y, dz = c[2] - w.z;
            const double ddd = dx * dx + dy * dy + dz * dz;
            best = ddd < best ? ddd : best;
        }
    };
    auto worst = [&]() {
        double m = best;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
        return m * WB_SLACK;
    };
    // the nearest tile first
    double near = INFINITY;
    int first = 0;
    for (int t = lane; t < ntile; t += 64) {
        const double s = bound(lo, hi, t);
        if (s < near) {
            near = s;
            first = t;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double s = __shfl_xor(near, off, 64);
        const int t = __shfl_xor(first, off, 64);
        if (s < near || (s == near && t < first)) {
            near = s;
            first = t;
        }
    }
    first = __builtin_amdgcn_readfirstlane(first);
    tile(first);
    double lim = worst();
    for (int t0 = 0; t0 < ntile; t0 += 64) {
        const double s = t0 + lane < ntile ? bound(lo, hi, t0 + lane) : INFINITY;
        unsigned long long todo = __ballot(t0 + lane < ntile && t0 + lane != first && !(s > lim));
        while (todo) {
            const int b = __ffsll((long long)todo) - 1;
            todo &= ~(1ull << b);
            const int t = __builtin_amdgcn_readfirstlane(t0 + b);
            if (!__any(!(bound(c, c, t) > best * WB_SLACK))) continue;
            tile(t);
            lim = worst();
            todo &= __ballot(!(s > lim));  // what has come out of reach meanwhile
        }
    }
    // the root of the clamped minimum, as the host forms it for the other form
    if (me < ncell) dst[from[me]] = sqrt(fmax(best, 1.0e-20));
}
