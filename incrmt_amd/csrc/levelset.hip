// GPU narrow-band level set (see levelset.hh).
//
// Rebuild. The reference rebuilds the band serially: a sign-change scan, an
// exact closest-point distance for the two interface layers (Newton on a
// bicubic), then a heap-ordered second-order fast march out to the band
// limit (levelset.cc:199-335, heap.cc). Here the scan and the Newton solves
// are one thread per point, and the march is replaced by a Jacobi fixed-point
// iteration of the SAME local update (eikonal.hh) over the points near the
// interface: a neighbour counts as known when its current value is upwind of
// the point's own, which is exactly the set the heap has accepted when it
// accepts the point. Where the heap's order is monotone and free of exact
// ties the fixed point equals the heap's result bit for bit.
//
// Extension. The reference extends (nX,nY) outward in increasing-phi order,
// each point by a weighted least-squares fit over the neighbours with
// smaller phi (traverse.hh:169-260). The set a point reads depends on phi
// alone, so a point evaluated once, when all that it reads is final, has
// exactly the sequential result (extend_tile).
#include <algorithm>
#include <cstdio>
#include "levelset.hh"
#include "eikonal.hh"

namespace incrmt {

namespace {

constexpr int BX = 64, BY = 4;

// Rows a thread of the scan and of the finalisation takes: a workgroup of
// BX x BY threads covers BX x (BY kRowSeg) points, whose shared neighbour rows
// are read once, all loads in flight together.
constexpr int kRowSeg = 4;

// Workgroup-aggregated list append: bit r of `bits` puts ij0 + r stride on the
// list, with one atomic on `counter` per workgroup that has any (same-address
// atomics of a whole launch run one after another: an atomic per wavefront
// and row made the scan of a circle on 1024^2 take 21.6 us, now 7.5). Every
// thread of the workgroup calls it. The order inside a list carries no
// meaning: each entry is processed on its own.
__device__ inline void block_append(unsigned bits, int ij0, int stride, int *counter, int *list) {
    __shared__ int tot[BY], base;
    const int lane = __lane_id(), wave = threadIdx.y;
    const unsigned long long below = (1ull << lane) - 1;
    int pos[kRowSeg], n = 0;
#pragma unroll
    for (int r = 0; r < kRowSeg; r++) {
        const unsigned long long m = __ballot(bits >> r & 1);
        pos[r] = n + __popcll(m & below);
        n += __popcll(m);
    }
    if (lane == 0) tot[wave] = n;
    __syncthreads();
    if (lane == 0 && wave == 0) {
        int all = 0;
        for (int k = 0; k < BY; k++) all += tot[k];
        if (all) base = atomicAdd(counter, all);
    }
    __syncthreads();
    if (!n) return;
    int start = base;
    for (int k = 0; k < wave; k++) start += tot[k];
#pragma unroll
    for (int r = 0; r < kRowSeg; r++)
        if (bits >> r & 1) list[start + pos[r]] = ij0 + r * stride;
}
static_assert(BX == 64, "a row of a workgroup is a wavefront");
// Wavefront-aggregated flag set: one atomicOr per distinct tile index.
__device__ inline void wave_flag(bool pred, int *flags, int tile, int bit) {
    unsigned long long m = __ballot(pred);
    const int lane = __lane_id();
    while (m) {
        const int l = __ffsll((long long)m) - 1;
        const int t = __shfl(tile, l, 64);
        const unsigned long long same = __ballot(pred && tile == t);
        if (lane == l) atomicOr(&flags[t], bit);
        m &= ~same;
    }
}

inline dim3 grid_rows(const Win &v) {
    return dim3((v.I1 - v.I0 + BX - 1) / BX, (v.J1 - v.J0 + BY * kRowSeg - 1) / (BY * kRowSeg));
}
inline dim3 grid_win(const Win &v) { return dim3((v.I1 - v.I0 + BX - 1) / BX, (v.J1 - v.J0 + BY - 1) / BY); }
constexpr int kListBlocks = 1024;
constexpr int kNewtonThreads = 64;  // a wavefront a workgroup: the few there are spread over the chip
constexpr int kTileBlocks = 512;

__device__ inline void ls_coords(const Grid &g, int ij, int &I, int &J) {
    const int r = ij - (kOrigin - 2);
    J = r / g.P;
    I = r - J * g.P;
}

// ---- bicubic with gradient on the ghosted grid (levelset.cc:63-79,
// built/bicubic.cc); evaluation order as in the reference.
struct xrow { double v, d; };
__device__ inline xrow herm_mid(double pl, double f0, double f1, double pr, double e, double me) {
    xrow r;
    r.v = pl * e * me * me + f0 * me * me * (1 + 2 * e) + f1 * e * e * (3 - 2 * e) - pr * e * e * me;
    r.d = pl * me * (1 - 3 * e) - f0 * 6 * e * me + f1 * 6 * e * me + pr * e * (3 * e - 2);
    return r;
}
__device__ inline xrow herm_left(double f0, double f1, double pr, double e, double me) {
    xrow r;
    r.v = f0 * me * me + f1 * e * (2 - e) - pr * e * me;
    r.d = -f0 * 2 * me + f1 * 2 * me + pr * (2 * e - 1);
    return r;
}
__device__ inline xrow herm_right(double pl, double f0, double f1, double e, double me) {
    xrow r;
    r.v = pl * e * me + f0 * (1 - e * e) + f1 * e * e;
    r.d = pl * (1 - 2 * e) - f0 * 2 * e + f1 * 2 * e;
    return r;
}

struct LsGeom {
    int m, n, P;
    double ax, ay, dx, dy, xsp, ysp;
};

// The Hermite data of the cell of the last evaluation: its four values, x
// and y slopes and cross slopes, as the rows of the interpolant take them. A
// Newton solve evaluates the interpolant nine times or more, one after
// another, and mostly in one cell, on one wavefront's chain of dependent
// operations: the 16 values behind them are read together, and the slopes
// formed once, while the cell stays. Read where each is first needed they cost
// several dependent round trips per evaluation: 22.1 -> 14.2 us for a circle on 64^2,
// 26.4 -> 14.1 us on 1024^2, 64.4 -> 28.5 us for 64 circles on 2048^2.
struct Patch {
    int at = -1;
    double r0[4], r1[4], r2[4], r3[4];  // left slope, left value, right value, right slope
};

__device__ double bicubic(const LsGeom &g, const double *base, Patch &c, double x, double y, double &phix,
                          double &phiy) {
    const int m = g.m, n = g.n, P = g.P;
    const double dxf = 0.5, dyf = 0.5, d2f = 0.25;
    double e = (x - g.ax) * g.xsp, f = (y - g.ay) * g.ysp;
    int i = int(e), j = int(f);
    int xc, yc, ic, jc;
    if (i < 1) { xc = 0; ic = 0; }
    else if (i >= m - 2) { xc = 2; ic = m - 2; e -= double(m - 2); }
    else { xc = 1; ic = i; e -= double(i); }
    if (j < 1) { yc = 0; jc = 0; }
    else if (j >= n - 2) { yc = 2; jc = n - 2; f -= double(n - 2); }
    else { yc = 1; jc = j; f -= double(j); }
    const double me = 1 - e, mf = 1 - f;
    if (const int at = jc * P + ic; at != c.at) {
        c.at = at;
        // a column or row that an edge cell does not have repeats the nearest
        // one; its slope is not used
        const int col[4] = {xc == 0 ? 0 : -1, 0, 1, xc == 2 ? 1 : 2};
        const int rw[4] = {yc == 0 ? 0 : -P, 0, P, yc == 2 ? P : 2 * P};
        double v[4][4];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int q = 0; q < 4; q++) v[r][q] = base[at + rw[r] + col[q]];
        auto values = [&](double (&o)[4], int r) {
            o[0] = (v[r][2] - v[r][0]) * dxf;
            o[1] = v[r][1];
            o[2] = v[r][2];
            o[3] = (v[r][3] - v[r][1]) * dxf;
        };
        auto slopes = [&](double (&o)[4], int u, int d) {
            o[0] = (v[u][2] - v[d][2] - v[u][0] + v[d][0]) * d2f;
            o[1] = (v[u][1] - v[d][1]) * dyf;
            o[2] = (v[u][2] - v[d][2]) * dyf;
            o[3] = (v[u][3] - v[d][3] - v[u][1] + v[d][1]) * d2f;
        };
        slopes(c.r0, 2, 0);
        values(c.r1, 1);
        values(c.r2, 2);
        slopes(c.r3, 3, 1);
    }
    auto row = [&](const double (&o)[4]) -> xrow {
        return xc == 1 ? herm_mid(o[0], o[1], o[2], o[3], e, me) : xc == 0 ? herm_left(o[1], o[2], o[3], e, me)
                                                                       : herm_right(o[0], o[1], o[2], e, me);
    };
    const xrow r1 = row(c.r1), r2 = row(c.r2);
    xrow r0 = {0, 0}, r3 = {0, 0};
    if (yc != 0) r0 = row(c.r0);
    if (yc != 2) r3 = row(c.r3);
    if (yc == 1) {
        phix = g.xsp * (f * mf * mf * r0.d + mf * mf * (1 + 2 * f) * r1.d + f * f * (3 - 2 * f) * r2.d - f * f * mf * r3.d);
        phiy = g.ysp * (mf * (1 - 3 * f) * r0.v - 6 * f * mf * r1.v + 6 * f * mf * r2.v + f * (3 * f - 2) * r3.v);
        return f * mf * mf * r0.v + mf * mf * (1 + 2 * f) * r1.v + f * f * (3 - 2 * f) * r2.v - f * f * mf * r3.v;
    } else if (yc == 0) {
        phix = g.xsp * (mf * mf * r1.d + f * (2 - f) * r2.d - f * mf * r3.d);
        phiy = g.ysp * (-2 * mf * r1.v + 2 * mf * r2.v + (2 * f - 1) * r3.v);
        return mf * mf * r1.v + f * (2 - f) * r2.v - f * mf * r3.v;
    }
    phix = g.xsp * (f * mf * r0.d + (1 - f * f) * r1.d + f * f * r2.d);
    phiy = g.ysp * ((1 - 2 * f) * r0.v - 2 * f * r1.v + 2 * f * r2.v);
    return f * mf * r0.v + (1 - f * f) * r1.v + f * f * r2.v;
}

// The compiled reference truncates before abs (levelset.cc:124,126).
__device__ inline double int_abs(double v) { return double(abs(int(v))); }

// levelset::newton_failsafe (levelset.cc:137-195)
__device__ bool newton_failsafe(const LsGeom &g, const double *phi, const int *st, int I, int J, int ij, double x0,
                                double y0, double &x, double &y) {
    const int ts = 7 - st[ij], P = g.P;
    const double cphi = phi[ij];
    bool hf = false, vf = false;
    double fx = 0, fy = 0, t;
    if (I > 0 && st[ij - 1] == ts) {
        fx = cphi / (phi[ij - 1] - cphi);
        if (I < g.m - 1 && st[ij + 1] == ts) {
            t = cphi / (cphi - phi[ij + 1]);
            if (t < -fx) fx = t;
        }
        hf = true;
    } else if (I < g.m - 1 && st[ij + 1] == ts) {
        fx = cphi / (cphi - phi[ij + 1]);
        hf = true;
    }
    if (J > 0 && st[ij - P] == ts) {
        fy = cphi / (phi[ij - P] - cphi);
        if (J < g.n - 1 && st[ij + P] == ts) {
            t = cphi / (cphi - phi[ij + P]);
            if (t < -fy) fy = t;
        }
        vf = true;
    } else if (J < g.n - 1 && st[ij + P] == ts) {
        fy = cphi / (cphi - phi[ij + P]);
        vf = true;
    }
    if (hf && vf) {
        double yy = fy * g.dy, tx = fx * g.dx;
        double cc = tx * yy / (tx * tx + yy * yy);
        x = yy * cc + x0;
        y = tx * cc + y0;
        return true;
    }
    if (hf) { x = fx * g.dx + x0; y = y0; return true; }
    if (vf) { x = x0; y = fy * g.dy + y0; return true; }
    return false;
}

// levelset::newton (levelset.cc:107-127). b0 and st point at ghosted point
// (0,0) and ij = J*P + I indexes both; y0 is formed from the reference's own
// linear index J*m as (J*m)*(dy/m).
__device__ bool newton(const LsGeom &g, const double *b0, const int *st, int I, int J, int ij, double &x0,
                       double &y0, double &x, double &y) {
    const double dyy = g.dy / double(g.m), step_limit = sqrt(g.dx * g.dx + g.dy * g.dy);
    int iter = 0, cutoff = 0;
    double ph, px, py;
    x0 = x = g.ax + I * g.dx;
    y0 = y = g.ay + double(J * g.m) * dyy;
    Patch c;
    ph = bicubic(g, b0, c, x, y, px, py);
    do {
        double delx = x0 - x, dely = y0 - y;
        double m0 = delx * px + dely * py + ph;
        double m1 = px * px + py * py;
        iter++;
        m0 /= m1;
        if (iter > 100 || !isfinite(m0) || m0 > step_limit)
            return newton_failsafe(g, b0, st, I, J, ij, x0, y0, x, y);
        x += delx - m0 * px;
        y += dely - m0 * py;
        ph = bicubic(g, b0, c, x, y, px, py);
        if (int_abs(ph) < 1e-10) cutoff++; else cutoff = 0;
    } while (cutoff < 8);
    if (int_abs(x0 - x) < 3 * g.dx && int_abs(y0 - y) < 3 * g.dy) return true;
    return newton_failsafe(g, b0, st, I, J, ij, x0, y0, x, y);
}

LsGeom geom_of(const Grid &g) {
    LsGeom l;
    l.m = g.ml; l.n = g.nl; l.P = g.P;
    l.ax = g.lax; l.ay = g.lay;
    l.dx = g.dx; l.dy = g.dy; l.xsp = g.xsp; l.ysp = g.ysp;
    return l;
}

// ------------------------------------------------------------------ kernels
__device__ inline void bbox_clear(int *b) {
    if (threadIdx.x == 0) {
        b[0] = b[2] = 1 << 30;
        b[1] = b[3] = -1;
    }
}
// bbox, when given, starts a rebuild's band box
__global__ void k_zero_counts(int *cnt, int n, int *bbox = nullptr) {
    if (bbox) bbox_clear(bbox);
    for (int k = threadIdx.x; k < n; k += blockDim.x) cnt[k] = 0;
}

// obj_field::pin (obj_field.cc:92-97) over the ghosted grid
// (ix, iy), when given, stand in for (X, Y) on the interior cells: the
// reference map update_velocity will copy there (X = nX, Y = nY), so a
// rebuild can pin to the end-of-step map before that copy has run.
__device__ __forceinline__ void pin_body(const Grid &g, const ObjConst &c, const ObjArrays &a, const Win &wn,
                                         const double *ix, const double *iy) {
    const int I = wn.I0 + blockIdx.x * BX + threadIdx.x, J = wn.J0 + blockIdx.y * BY + threadIdx.y;
    if (I >= wn.I1 || J >= wn.J1) return;
    const int ij = g.ls(I, J);
    const bool inner = ix && I >= 2 && I < g.m + 2 && J >= 2 && J < g.n + 2;
    const double p = a.phi[ij];
    if (p < c.pinw && p > -c.pinw) a.phi[ij] = obj_phi(c, inner ? ix[ij] : a.X[ij], inner ? iy[ij] : a.Y[ij]);
}
__global__ void k_pin(Grid g, ObjConst c, ObjArrays a, Win wn, const double *ix, const double *iy) {
    pin_body(g, c, a, wn, ix, iy);
}

// Sign-change scan (levelset.cc:211-263): a point is on an interface layer
// when a 4-neighbour has the other sign. Interface points are listed for
// the Newton solves; the fixed-point buffers start at +-inf elsewhere.
__device__ __forceinline__ void scan_body(const Grid &g, const ObjArrays &a, const LsWork &w, const Win &wn) {
    const int I = wn.I0 + blockIdx.x * BX + threadIdx.x;
    const int J0 = wn.J0 + (blockIdx.y * BY + threadIdx.y) * kRowSeg, P = g.P;
    const int ij0 = g.ls(I, J0);
    unsigned im = 0;  // bit r: row J0 + r is on an interface layer
    if (I < wn.I1 && J0 < wn.J1) {
        const double *phi = a.phi;
        // the points, their neighbours' rows and columns read together (a
        // neighbour off the grid reads the point nearest to it, which in a row
        // or column of its own never differs in sign), then tested
        double pc[kRowSeg + 2], pl[kRowSeg], pr[kRowSeg];
#pragma unroll
        for (int r = 0; r < kRowSeg + 2; r++) {
            const int J = min(max(J0 + r - 1, 0), g.nl - 1);
            pc[r] = phi[g.ls(I, J)];
        }
#pragma unroll
        for (int r = 0; r < kRowSeg; r++) {
            const int q = g.ls(I, min(J0 + r, g.nl - 1));
            pl[r] = phi[I > 0 ? q - 1 : q];
            pr[r] = phi[I < g.ml - 1 ? q + 1 : q];
        }
#pragma unroll
        for (int r = 0; r < kRowSeg; r++) {
            if (J0 + r >= wn.J1) break;
            const int ij = ij0 + r * P;
            const bool pos = pc[r + 1] > 0;
            const bool iface = ((pl[r] > 0) != pos) | ((pr[r] > 0) != pos) | ((pc[r] > 0) != pos) |
                               ((pc[r + 2] > 0) != pos);
            a.st[ij] = pos ? (iface ? 4 : 7) : (iface ? 3 : 0);
            if (!iface) {
                const double inf = pos ? INFINITY : -INFINITY;
                w.va[ij] = inf;
                w.vb[ij] = inf;
            }
            im |= (unsigned)iface << r;
        }
    }
    block_append(im, ij0, P, &w.cnt[kCntIface], w.iface);
}
__global__ void k_scan(Grid g, ObjArrays a, LsWork w, Win wn) { scan_body(g, a, w, wn); }

// Exact closest-point distances of both interface layers, from the pinned
// phi (levelset.cc:266-291). The results go to the fixed-point buffers; phi
// itself keeps the pinned values until the band is finalised, since every
// Newton solve reads the pinned field.
__device__ __forceinline__ void newton_body(const Grid &g, const LsGeom &lg, const ObjArrays &a, const LsWork &w) {
    const int n = w.cnt[kCntIface];
    const double *b0 = a.phi + g.ls(0, 0);
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int ij = w.iface[k];
        int I, J;
        ls_coords(g, ij, I, J);
        double x0, y0, x, y;
        if (!newton(lg, b0, a.st + g.ls(0, 0), I, J, ij - g.ls(0, 0), x0, y0, x, y)) {
            atomicOr(&w.cnt[kCntErr], kErrNewton);
            continue;
        }
        x -= x0; y -= y0;
        const double d = sqrt(x * x + y * y);
        const double v = a.st[ij] == 4 ? d : -d;
        w.va[ij] = v;
        w.vb[ij] = v;
    }
}
__global__ __launch_bounds__(kNewtonThreads) void k_newton(Grid g, LsGeom lg, ObjArrays a, LsWork w) { newton_body(g, lg, a, w); }

// Candidate points: non-interface points within R cells (max norm) of an
// interface point, R covering the band cut-offs; separable dilation, rows
// then columns.
// A wavefront is 64 columns of a row: the interface flags of its columns and of
// the 64 on either side (more for R > 64) are three votes, and a point's window is
// a range of their bits, instead of 2R + 1 reads a point (5.7 -> 4.2 us for a
// circle on 1024^2, 26.7 -> 13.0 us for 2048^2 whole).
__device__ __forceinline__ void dilate_rows_body(const Grid &g, const ObjArrays &a, const LsWork &w, int R,
                                                 const Win &wn) {
    const int I = wn.I0 + blockIdx.x * BX + threadIdx.x, lane = threadIdx.x;
    const int J0 = wn.J0 + (blockIdx.y * BY + threadIdx.y) * kRowSeg;
    const int far = (R + 63) / 64;
    unsigned hit = 0;
    for (int k = -far; k <= far; k++) {
        const int Ik = I + 64 * k;
        const bool in = Ik >= 0 && Ik < g.ml;
        int st[kRowSeg];
#pragma unroll
        for (int r = 0; r < kRowSeg; r++) {
            const int s = a.st[g.ls(min(max(Ik, 0), g.ml - 1), min(J0 + r, g.nl - 1))];
            st[r] = in ? s : 0;
        }
        // the bits of this group within R of the lane's point
        const int lo = max(lane - R - 64 * k, 0), hi = min(lane + R - 64 * k, 63);
        const unsigned long long win = lo > hi ? 0 : (~0ull >> (63 - hi)) & (~0ull << lo);
#pragma unroll
        for (int r = 0; r < kRowSeg; r++) {
            const unsigned long long m = __ballot(st[r] == 3 || st[r] == 4);
            hit |= (unsigned)((m & win) != 0) << r;
        }
    }
    if (I >= wn.I1) return;
#pragma unroll
    for (int r = 0; r < kRowSeg; r++)
        if (J0 + r < wn.J1) w.mark[g.ls(I, J0 + r)] = hit >> r & 1;
}
__global__ void k_dilate_rows(Grid g, ObjArrays a, LsWork w, int R, Win wn) { dilate_rows_body(g, a, w, R, wn); }
// The column pass: a thread takes kColSeg consecutive rows of one column and
// keeps the count of marked points in the column window [J - R, J + R]
// (clipped to the grid) as it slides down, one point in and one out per row,
// instead of reading the 2R + 1 marks of every point. Bound by latency: the
// reads of the first window go out eight at a time, the sliding ones with them
// (13.1 -> 5.4 us for a circle on 1024^2).
constexpr int kColSeg = 8;
static_assert(kTileY >= kColSeg, "a thread's rows span at most two tile rows");
inline dim3 grid_win_cols(const Win &v) {
    return dim3((v.I1 - v.I0 + BX - 1) / BX, (v.J1 - v.J0 + BY * kColSeg - 1) / (BY * kColSeg));
}
__device__ __forceinline__ void dilate_cols_body(const Grid &g, const ObjArrays &a, const LsWork &w, int R,
                                                 const Win &wn) {
    const int I = wn.I0 + blockIdx.x * BX + threadIdx.x;
    const int J0 = wn.J0 + (blockIdx.y * BY + threadIdx.y) * kColSeg;
    const bool col = I < wn.I1 && J0 < wn.J1;
    const unsigned char *mk = w.mark + (col ? g.ls(I, 0) : 0);
    int cnt = 0;
    unsigned hm = 0;  // bit k: row J0 + k is a candidate
    if (col) {
        // the points' statuses and the marks entering and leaving the sliding
        // window are read ahead of the first window's count
        int st[kColSeg], in[kColSeg], out[kColSeg];
#pragma unroll
        for (int k = 0; k < kColSeg; k++) {
            const int J = min(J0 + k, g.nl - 1);
            st[k] = a.st[g.ls(I, J)];
            const int a1 = J0 + k + R, a0 = J0 + k - 1 - R;
            const int m1 = mk[min(a1, g.nl - 1) * g.P], m0 = mk[max(a0, 0) * g.P];
            in[k] = k > 0 && a1 < g.nl && m1 != 0;
            out[k] = k > 0 && a0 >= 0 && m0 != 0;
        }
        const int lo = J0 - R < 0 ? 0 : J0 - R, hi = J0 + R >= g.nl ? g.nl - 1 : J0 + R;
        for (int J = lo; J <= hi; J += 8) {
            int m[8];
#pragma unroll
            for (int k = 0; k < 8; k++) m[k] = mk[min(J + k, hi) * g.P];
#pragma unroll
            for (int k = 0; k < 8; k++) cnt += J + k <= hi && m[k] != 0;
        }
#pragma unroll
        for (int k = 0; k < kColSeg; k++) {
            const int J = J0 + k;
            if (J >= wn.J1) break;
            // the window moves from [J-1-R, J-1+R] to [J-R, J+R]
            cnt += in[k] - out[k];
            const bool hit = st[k] != 3 && st[k] != 4 && cnt > 0;
            w.cflag[g.ls(I, J)] = hit;
            hm |= (unsigned)hit << k;
        }
    }
    // the tile flags set once per wavefront and tile row: a thread's rows span
    // at most two tile rows
    const int ta = J0 / kTileY, tb = (J0 + kColSeg - 1) / kTileY;
    unsigned ma = 0;  // rows of tile row ta
#pragma unroll
    for (int k = 0; k < kColSeg; k++)
        if ((J0 + k) / kTileY == ta) ma |= 1u << k;
    wave_flag((hm & ma) != 0, w.tflag, ta * w.ntx + I / kTileX, 1);
    if (tb != ta) wave_flag((hm & ~ma) != 0, w.tflag, tb * w.ntx + I / kTileX, 1);
}
__global__ void k_dilate_cols(Grid g, ObjArrays a, LsWork w, int R, Win wn) { dilate_cols_body(g, a, w, R, wn); }

// Collect the tiles whose flag has `bit` set into a list, clearing the bit.
__device__ __forceinline__ void compact_tiles_body(const LsWork &w, int bit, int *list, int slot) {
    const int n = w.ntx * w.nty;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const int f = w.tflag[t];
        if (f & bit) {
            const int k = atomicAdd(&w.cnt[slot], 1);
            list[k] = t;
            w.tflag[t] = f & ~bit;
        }
    }
}
__global__ void k_compact_tiles(LsWork w, int bit, int *list, int slot) { compact_tiles_body(w, bit, list, slot); }

// One pass of the band march over the active tiles. A workgroup loads its
// tile and a 2-point halo (the reach of the local update) into LDS and
// repeats the Jacobi update on the tile until it stops changing, the halo
// held at the previous pass's values; passes repeat until no tile changes.
// Any order of such relaxations reaches the same fixed point.
// A pass is bound by the chain of local iterations of its slowest tile, one
// wavefront a SIMD: with the update's rules evaluated once each instead of
// branch by branch (Eik::calc_fast, RegAcc) an average launch takes 17.2 us
// instead of 38.7 at 64^2, 23.7 instead of 46.2 at 1024^2, and 93 instead of
// 166 for 64 circles at 2048^2.
constexpr int kFH = 2, kFW = kTileX + 2 * kFH, kFHt = kTileY + 2 * kFH, kFN = kFW * kFHt;

// The OR over a workgroup of one predicate per thread, with one barrier:
// the wavefronts post their votes to one of three LDS slots used in turn,
// and the slot two rounds ahead is cleared between this round's barrier and
// the next (its last readers have passed this barrier, its next writers
// have not passed the next one). The slots are zero before the first round,
// behind a barrier.
struct VoteOr {
    int *slot;
    int k;
    __device__ int operator()(int pred) {
        if (__any(pred) && (threadIdx.x & 63) == 0) slot[k] = 1;
        __syncthreads();
        const int r = slot[k];
        if (threadIdx.x == 0) slot[k == 0 ? 2 : k - 1] = 0;
        k = k == 2 ? 0 : k + 1;
        return r;
    }
};

// Known-neighbour test of the heap march (heap.hh:59-83) at the fixed point:
// the other side and the interface layer are always known; a same-side
// point is known when it has been reached, lies within the band, and is
// upwind of the point being updated. Here on one point's radius-2 cross
// stencil held in registers (slots: the point, x -1 +1 -2 +2, y -1 +1 -2 +2).
// The update's reads, taken one by one from LDS, form a chain of dependent
// round trips; here the statuses are read once per tile, as two bits a slot
// (known whatever its value; known once it is upwind), and the values once
// per iteration, all issued together. The offsets the update asks for are compile-time constants
// after inlining, so the slot lookups fold away. The values, pval and limit
// carry the inward march's sign flipped, so both marches run the outward
// update: negating every input of the inward update negates its result exactly
// (IEEE rounding is symmetric), which keeps one code path per wavefront.
struct RegAcc {
    double v[9];
    unsigned always, upwind;
    int base;
    double pval, limit;
    __device__ static int slot(int d) {
        return d == -1 ? 1 : d == 1 ? 2 : d == -2 ? 3 : d == 2 ? 4 : d == -kFW ? 5 : d == kFW ? 6
             : d == -2 * kFW ? 7 : d == 2 * kFW ? 8 : 0;
    }
    __device__ bool in(int q) const {
        const int k = slot(q - base);
        return (always >> k & 1) | ((upwind >> k & 1) & (v[k] < pval) & (v[k] < limit));
    }
    __device__ double val(int q) const { return v[slot(q - base)]; }
};
// v with its sign flipped where s (0 or the sign bit) says so
__device__ __forceinline__ double flip(double v, unsigned long long s) {
    return __longlong_as_double((long long)((unsigned long long)__double_as_longlong(v) ^ s));
}
__device__ constexpr int kStencil[9] = {0, -1, 1, -2, 2, -kFW, kFW, -2 * kFW, 2 * kFW};

__device__ __forceinline__ void fim_tiles(const Grid &g, const EikGeom &eg, const ObjConst &c, const ObjArrays &a,
                                          const LsWork &w, const double *src, double *dst, int slot, int max_local) {
    __shared__ double sv[2][kFN];
    __shared__ int sst[kFN];
    __shared__ int vslot[3];
    if (slot > 0 && w.cnt[kCntIter + slot - 1] == 0) return;  // fixed point already reached
    const int nt = w.cnt[kCntTileFim];
    if (threadIdx.x < 3) vslot[threadIdx.x] = 0;
    VoteOr vote{vslot, 0};
    int changed_any = 0;
    constexpr int kRounds = (kFN + kTileThreads - 1) / kTileThreads;
    for (int t = blockIdx.x; t < nt; t += gridDim.x) {
        const int tile = w.tiles_fim[t], tx = tile % w.ntx, ty = tile / w.ntx;
        const int I0 = tx * kTileX - kFH, J0 = ty * kTileY - kFH;
        // the tile and its halo: every global read issued before any wait
        double rv[kRounds];
        int rs[kRounds];
#pragma unroll
        for (int u = 0; u < kRounds; u++) {
            const int e = threadIdx.x + u * kTileThreads, I = I0 + e % kFW, J = J0 + e / kFW;
            rv[u] = 0;
            rs[u] = -1;
            if (e < kFN && I >= 0 && I < g.ml && J >= 0 && J < g.nl) {
                const int q = g.ls(I, J);
                rv[u] = src[q];
                rs[u] = a.st[q];
            }
        }
        const int li = threadIdx.x % kTileX + kFH, lj = threadIdx.x / kTileX + kFH, e = lj * kFW + li;
        const int I = I0 + li, J = J0 + lj;
        const bool mine = I < g.ml && J < g.nl && w.cflag[g.ls(I, J)];
#pragma unroll
        for (int u = 0; u < kRounds; u++) {
            const int f = threadIdx.x + u * kTileThreads;
            if (f < kFN) {
                sv[0][f] = sv[1][f] = rv[u];
                sst[f] = rs[u];
            }
        }
        __syncthreads();
        const bool pos = mine && sst[e] == 7;
        const unsigned long long sign = pos ? 0 : 1ull << 63;
        // every stencil point of a tile point lies in the tile's 2-point
        // halo; a point off the grid (status -1) is never known, so the
        // update needs no bounds of its own
        RegAcc acc;
        acc.base = e; acc.limit = pos ? c.phi_up : -c.phi_down;
        acc.always = acc.upwind = 0;
#pragma unroll
        for (int k = 0; k < 9; k++) {
            const int s = sst[e + kStencil[k]];
            if (pos ? s >= 0 && s <= 4 : s >= 3) acc.always |= 1u << k;
            else if (s >= 0) acc.upwind |= 1u << k;
        }
        int cur = 0;
        for (int it = 0; it < max_local; it++) {
            int changed = 0;
            if (mine) {
#pragma unroll
                for (int k = 0; k < 9; k++) acc.v[k] = flip(sv[cur][e + kStencil[k]], sign);
                acc.pval = acc.v[0];
                double r = INFINITY;
                if (acc.in(e - 1) | acc.in(e + 1) | acc.in(e - kFW) | acc.in(e + kFW)) {
                    const Eik<true, RegAcc> k{acc, eg, 1 << 30, 1 << 30, kFW};
                    r = k.calc_fast(2, 2, e);
                }
                changed = __double_as_longlong(r) != __double_as_longlong(acc.v[0]);
                sv[cur ^ 1][e] = flip(r, sign);
            }
            const int ch = vote(changed);
            cur ^= 1;
            if (!ch) break;
        }
        if (mine) {
            const int q = g.ls(I, J);
            const double v = sv[cur][e];
            dst[q] = v;
            if (__double_as_longlong(v) != __double_as_longlong(src[q])) changed_any = 1;
        }
        __syncthreads();
    }
    if (__any(changed_any) && (threadIdx.x & 63) == 0) atomicAdd(&w.cnt[kCntIter + slot], 1);
}
__global__ __launch_bounds__(kTileThreads) void k_fim_tiles(Grid g, EikGeom eg, ObjConst c, ObjArrays a, LsWork w,
                                                   const double *src, double *dst, int slot, int max_local) {
    fim_tiles(g, eg, c, a, w, src, dst, slot, max_local);
}
// The march passes of several solids in one launch: workgroup (x, y) runs
// the pass of solid y with x as its block index, on its own buffers and
// counters (pass p reads buf[p & 1], writes the other), so each solid's
// passes are exactly those it runs alone.
struct FimItem {
    ObjConst c;
    ObjArrays a;
    LsWork w;
    double *buf[2];
};
__global__ __launch_bounds__(kTileThreads) void k_fim_tiles_batch(Grid g, EikGeom eg, const FimItem *it, int p,
                                                         int slot, int max_local) {
    const FimItem &x = it[blockIdx.y];
    fim_tiles(g, eg, x.c, x.a, x.w, x.buf[p & 1], x.buf[(p + 1) & 1], slot, max_local);
}

// Final band (levelset.cc:300-335, 408-413): accepted points get their
// fixed-point values and status 5/2, points the heap would have left in its
// queue status 6/1, everything outside the band the cut-off value. Tiles with
// outside band points are flagged for the extension.
// Bound by latency: a thread's four points share their neighbours' rows, every
// load is issued before the first test (29.6 -> 12.7 us for a circle
// on 1024^2), the band's box is formed from votes, and an atomic goes out only
// where it widens the box that the launch has so far.
__device__ __forceinline__ void finalize_body(const Grid &g, const ObjConst &c, const ObjArrays &a, const LsWork &w,
                                              const double *v, const Win &wn) {
    __shared__ int box[4];
    const int t = threadIdx.y * BX + threadIdx.x, lane = threadIdx.x;
    if (t < 4) box[t] = t & 1 ? -1 : 1 << 30;
    const int I = wn.I0 + blockIdx.x * BX + threadIdx.x;
    const int J0 = wn.J0 + (blockIdx.y * BY + threadIdx.y) * kRowSeg;
    const double lim = c.phi_up, dlim = c.phi_down;
    unsigned nm = 0, pm = 0;  // bit r: row J0 + r in the band or its trial points; outside band
    if (I < wn.I1 && J0 < wn.J1) {
        // a point outside the band tests its four neighbours (one off the grid
        // counts as not accepted)
        int sc[kRowSeg + 2], sl[kRowSeg], sr[kRowSeg];
        double vc[kRowSeg + 2], vl[kRowSeg], vr[kRowSeg];
        const bool hl = I > 0, hr = I < g.ml - 1;
#pragma unroll
        for (int r = 0; r < kRowSeg + 2; r++) {
            const int q = g.ls(I, min(max(J0 + r - 1, 0), g.nl - 1));
            sc[r] = a.st[q];
            vc[r] = v[q];
        }
#pragma unroll
        for (int r = 0; r < kRowSeg; r++) {
            const int q = g.ls(I, min(J0 + r, g.nl - 1)), ql = hl ? q - 1 : q, qr = hr ? q + 1 : q;
            sl[r] = a.st[ql];
            vl[r] = v[ql];
            sr[r] = a.st[qr];
            vr[r] = v[qr];
        }
        auto acc_pos = [&](int s, double x) { return s == 4 || (s == 7 && x < lim); };
        auto acc_neg = [&](int s, double x) { return s == 3 || (s == 0 && x > dlim); };
#pragma unroll
        for (int r = 0; r < kRowSeg; r++) {
            const int J = J0 + r;
            if (J >= wn.J1) break;
            const bool hd = J > 0, hu = J < g.nl - 1;
            auto any_nb = [&](auto acc) {
                return (hl && acc(sl[r], vl[r])) | (hr && acc(sr[r], vr[r])) | (hd && acc(sc[r], vc[r])) |
                       (hu && acc(sc[r + 2], vc[r + 2]));
            };
            const int s = sc[r + 1], ij = g.ls(I, J);
            const double v0 = vc[r + 1];
            int ns = s;
            double phi;
            if (s == 3 || s == 4) {
                phi = v0;
            } else if (s == 7) {
                if (v0 < lim) { ns = 5; phi = v0; }
                else {
                    ns = any_nb(acc_pos) ? 6 : 7;
                    phi = lim;
                }
            } else {
                if (v0 > dlim) { ns = 2; phi = v0; }
                else {
                    ns = any_nb(acc_neg) ? 1 : 0;
                    phi = dlim;
                }
            }
            w.mark[ij] = (unsigned char)ns;  // statuses go to st after every thread read the old ones
            a.phi[ij] = phi;
            nm |= (unsigned)(ns >= 1 && ns <= 6) << r;
            pm |= (unsigned)(ns == 4 || ns == 5) << r;
        }
    }
    // outside band points mark their tile for the extension
    const int ta = J0 / kTileY, tb = (J0 + kRowSeg - 1) / kTileY;
    unsigned ma = 0;  // rows of tile row ta
#pragma unroll
    for (int r = 0; r < kRowSeg; r++)
        if ((J0 + r) / kTileY == ta) ma |= 1u << r;
    wave_flag((pm & ma) != 0, w.tflag, ta * w.ntx + I / kTileX, 2);
    if (tb != ta) wave_flag((pm & ~ma) != 0, w.tflag, tb * w.ntx + I / kTileX, 2);
    // bounding box of the band and its trial points, for the next window
    __syncthreads();
    const unsigned long long cols = __ballot(nm != 0);
    if (cols) {
        int lo = kRowSeg, hi = 0;
#pragma unroll
        for (int r = 0; r < kRowSeg; r++)
            if (__ballot(nm >> r & 1)) { lo = min(lo, r); hi = r; }
        if (lane == 0) {
            atomicMin(&box[0], I + __ffsll((long long)cols) - 1);
            atomicMax(&box[1], I + 63 - __clzll((long long)cols));
            atomicMin(&box[2], J0 + lo);
            atomicMax(&box[3], J0 + hi);
        }
    }
    __syncthreads();
    if (t < 4 && box[1] >= 0) {
        const int b = box[t], now = __hip_atomic_load(&w.bbox[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (t & 1) { if (b > now) atomicMax(&w.bbox[t], b); }
        else if (b < now) atomicMin(&w.bbox[t], b);
    }
}
__global__ void k_finalize(Grid g, ObjConst c, ObjArrays a, LsWork w, const double *v, Win wn) {
    finalize_body(g, c, a, w, v, wn);
}
// The new statuses, and the band's box to the host (work sets that keep a
// window): a copy command behind the kernels cost as much as a launch, one per
// solid.
__device__ __forceinline__ void commit_status_body(const Grid &g, const ObjArrays &a, const LsWork &w, const Win &wn) {
    const int I = wn.I0 + blockIdx.x * BX + threadIdx.x, J = wn.J0 + blockIdx.y * BY + threadIdx.y;
    if (w.hbbox && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.y == 0 && threadIdx.x < 4)
        w.hbbox[threadIdx.x] = w.bbox[threadIdx.x];
    if (I >= wn.I1 || J >= wn.J1) return;
    const int ij = g.ls(I, J);
    a.st[ij] = w.mark[ij];
}
__global__ void k_commit_status(Grid g, ObjArrays a, LsWork w, Win wn) { commit_status_body(g, a, w, wn); }

// The extension (traverse.hh:169-231) over the active tiles: outside band
// points take a weighted least-squares linear fit of (nX,nY) over band
// neighbours with smaller phi, in a (2r+1)^2 box, r = 3 growing to 7 while
// the fit is singular. A point's fit reads only neighbours of strictly
// smaller phi, so the fits form an acyclic system with one solution and a
// point needs to be evaluated once, when the last value it reads is final.
//
// What bounds it is the chain of dependent fits (60 to 90 long, along the
// band as well as across it), not bytes or arithmetic, so the kernel is
// built for the time of one link. A workgroup holds a tile and a 3-point
// halo in LDS with a bit per point that says whether its value is final. A
// point's wavefront evaluates it as soon as the bits of its neighbour mask
// are all set: 49 lanes form the six products of one window position each
// and leave them in LDS in mask order, six lanes add up one sum each in that
// order (the reference's order of additions, so the sums are the same bits).
// Values cross between workgroups through (ex, ey): an open point holds
// kExtOpen in both, its owner stores each value with one agent-scope atomic
// store, and one further wavefront per workgroup polls the halo points that
// its tile's open points read. A value is its own flag, so nothing is fenced.
// No barrier, launch or host check lies between two links.
//
// A tile whose halo brings nothing new for its patience is left: the workgroup
// takes or goes on to others and comes back (ext_next), and what is still open
// when nothing moves any more is counted for another pass, which takes up the
// values found so far. So the kernel ends whatever the other workgroups do,
// also when not all of them are on the GPU at once.
//
// Measured per extension: a rotor at 64^2 0.63 -> 0.09 ms and at 1024^2 0.44
// -> 0.12 ms against 14 to 20 launches that swept whole tiles to a local fixed
// point (25-31 us each); 64 circles at 2048^2 3.3 -> 0.75 ms. At 64^2 about 26
// of the 64 links cross between workgroups.
constexpr int kEH = 3;
// Its tiles are the march's, whole where a row with its halo fits one 32-bit word
// of flags and the points' wavefronts and one more a workgroup (the default
// 16 x 16 does), else in the fewest equal parts of whole wavefronts for which
// that holds.
struct ExtParts {
    int x = 0, y = 0;
};
constexpr ExtParts ext_parts(int tx, int ty) {
    ExtParts best;
    for (int x = 1; x <= tx; x++)
        for (int y = 1; y <= ty; y++) {
            const int ex = tx / x, ey = ty / y;
            if (tx % x || ty % y || ex + 2 * kEH > 32 || ex * ey % 64 || ex * ey + 64 > 1024) continue;
            if (!best.x || x * y < best.x * best.y) best = {x, y};
        }
    return best;
}
constexpr ExtParts kExtParts = ext_parts(kTileX, kTileY);
static_assert(kExtParts.x > 0, "the extension needs parts of whole wavefronts, at most 26 points wide");
constexpr int kExtPerTile = kExtParts.x * kExtParts.y;
constexpr int kExtX = kTileX / kExtParts.x, kExtY = kTileY / kExtParts.y;
constexpr int kEW = kExtX + 2 * kEH, kEHt = kExtY + 2 * kEH, kEN = kEW * kEHt;
constexpr int kExtWaves = kExtX * kExtY / 64, kExtThreads = kExtX * kExtY + 64;
// a signalling NaN, which no arithmetic returns
constexpr unsigned long long kExtOpen = 0x7ff4a5a5a5a5a5a5ull;
constexpr int kExtProd = 49;  // row of products: at most 48 neighbours; odd, so that six rows start in different banks

__device__ __forceinline__ unsigned long long ext_load(const double *p) {
    return __hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ext_store(double *p, double v) {
    unsigned long long b = (unsigned long long)__double_as_longlong(v);
    if (b == kExtOpen) b |= 1ull << 51;  // a value that stays (singular fit) may be any bits: never the open mark
    __hip_atomic_store((unsigned long long *)p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Lanes of one wavefront hand values to each other through LDS: its LDS
// operations run in order, so only the compiler has to keep theirs.
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }
// a word of LDS that other wavefronts of the workgroup change
template <class T>
__device__ __forceinline__ T lds_now(const T &v) {
    return __hip_atomic_load(&v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ double lane_double(double v, int l) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, l), hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), l);
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// Mark the outside band points of the active tiles open, clear the tiles' counters.
__device__ __forceinline__ void ext_open_body(const Grid &g, const ObjArrays &a, const LsWork &w) {
    const int nt = w.cnt[kCntTileExt];
    for (int t = blockIdx.x; t < nt; t += gridDim.x) {
        const int tile = w.tiles_ext[t];
        if (threadIdx.x == 0) w.tprog[tile] = 0;
        const int I = tile % w.ntx * kTileX + threadIdx.x % kTileX, J = tile / w.ntx * kTileY + threadIdx.x / kTileX;
        if (I >= g.ml || J >= g.nl) continue;
        const int q = g.ls(I, J), s = a.st[q];
        if (s == 4 || s == 5) {
            w.ex[q] = __longlong_as_double((long long)kExtOpen);
            w.ey[q] = __longlong_as_double((long long)kExtOpen);
        }
    }
}
__global__ __launch_bounds__(kTileThreads) void k_ext_open(Grid g, ObjArrays a, LsWork w) { ext_open_body(g, a, w); }

constexpr int kExtHeld = 32;  // tiles that a workgroup goes round between at the most
struct ExtLds {
    double phi[kEN], x[kEN], y[kEN];
    double prod[kExtWaves][6][kExtProd];
    unsigned char st[kEN];           // status + 1, 0 off the grid
    unsigned known[kEHt];            // bit c of row r: the value is final, or never computed
    unsigned need[kEHt];             // ... is read by an open point of the tile
    unsigned short halo[kEN];        // the halo points to poll
    int nhalo, left, stop;
    unsigned news;                   // counts values that have become final here
    unsigned quit;                   // what it was when the first wavefront gave up
    int was;                         // points open before the visit
    // ext_next's state: the visit (tile number, -1: none; its place in held,
    // ext_news before it), the tiles held and ext_news before their last
    // visits (-1: none yet)
    int t, k, heard, patience, nheld, open, idle, moved;
    bool fresh, more, take;
    bool wide;                       // a point's fit is of a larger radius
    int held[kExtHeld], seen[kExtHeld];
};

// Rounds of idle polling (0.2-1 us each) before a tile is left. kPatienceMany: by
// a workgroup that holds others too (the lattice of 6924 tiles 2.1, 2.1 and 3.0 ms for
// 8, 16 and 64). kPatienceTake: by one that holds this tile only and may take
// another, which workgroups that have finished should do first (32, 64, 128, 256, 512,
// 1024: a lattice of 1000 tiles 270, 250, 165, 175, 185, 180 us, that of 6924 2.2, 2.2,
// 2.2, 2.4, 2.7, 3.1 ms). kPatienceLast: where no other is to be had; then again
// while any of the solid's tiles has moved since, which a tile tells every
// kTellPoints points (without that 64 circles on 2048^2 took two launches with 200, one
// with 2000).
constexpr int kPatienceMany = 16, kPatienceTake = 256, kPatienceLast = 1000, kTellPoints = 32;
// Fruitless looks (1-2 us each) at the tiles of a workgroup that holds several
// before it asks the same, and leaves them to another pass
constexpr int kIdleMany = 256;
__device__ __forceinline__ void ext_tell(const LsWork &w) {
    (void)__hip_atomic_fetch_add(&w.cnt[kCntExtMoved], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int ext_moved(const LsWork &w) {
    return __hip_atomic_load(&w.cnt[kCntExtMoved], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One visit of a tile. fresh: every open mark of this extension is still as
// k_ext_open left it (the first visit of the first pass); many: the tile's counter
// is kept for ext_news. L.was and L.left: the points open before and after it.
__device__ __forceinline__ void extend_tile(const Grid &g, const ObjArrays &a, const LsWork &w, ExtLds &L, int tile,
                                           int part, bool fresh, bool many, int patience) {
    const int m = g.ml, nn = g.nl, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int I0 = tile % w.ntx * kTileX + part % kExtParts.x * kExtX - kEH,
              J0 = tile / w.ntx * kTileY + part / kExtParts.x * kExtY - kEH;
    // the tile and its halo, two rows a wavefront: every global read issued
    // before any wait, both rows' flags from one ballot
    constexpr int kRowsAtOnce = kExtThreads / 32, kRounds = (kEHt + kRowsAtOnce - 1) / kRowsAtOnce;
    double rph[kRounds], rnx[kRounds], rny[kRounds];
    int rst[kRounds];
    const int fc = tid & 31, fr = tid >> 5;
#pragma unroll
    for (int u = 0; u < kRounds; u++) {
        const int r = fr + u * kRowsAtOnce, I = I0 + fc, J = J0 + r;
        rst[u] = -1;
        rph[u] = rnx[u] = rny[u] = 0;
        if (fc < kEW && r < kEHt && I >= 0 && I < m && J >= 0 && J < nn) {
            const int q = g.ls(I, J);
            rst[u] = a.st[q];
            rph[u] = a.phi[q];
            rnx[u] = a.nX[q];
            rny[u] = a.nY[q];
        }
    }
    if (tid < kEHt) L.need[tid] = 0;
    if (tid == 0) {
        L.nhalo = L.left = L.stop = L.news = 0;
        L.quit = ~0u;
        L.wide = false;
    }
#pragma unroll
    for (int u = 0; u < kRounds; u++) {
        const int r = fr + u * kRowsAtOnce, s = rst[u];
        const unsigned long long k = __ballot(!(s == 4 || s == 5));
        if (r < kEHt) {
            if (fc < kEW) {
                const int e = r * kEW + fc;
                L.st[e] = (unsigned char)(s + 1);
                L.phi[e] = rph[u];
                L.x[e] = rnx[u];
                L.y[e] = rny[u];
            }
            if (fc == 0) L.known[r] = (unsigned)(lane < 32 ? k : k >> 32);
        }
    }
    __syncthreads();
    const int li = tid % kExtX + kEH, lj = tid / kExtX + kEH, e = lj * kEW + li;
    const int i = I0 + li, j = J0 + lj;
    const bool mine = wave < kExtWaves && i < m && j < nn && (L.st[e] == 5 || L.st[e] == 6);
    const int q = mine ? g.ls(i, j) : 0;
    bool todo = mine;
    if (mine && !fresh) {  // taken up again: values found by an earlier visit
        const unsigned long long bx = ext_load(w.ex + q), by = ext_load(w.ey + q);
        if (bx != kExtOpen && by != kExtOpen) {
            L.x[e] = __longlong_as_double((long long)bx);
            L.y[e] = __longlong_as_double((long long)by);
            atomicOr(&L.known[lj], 1u << li);
            todo = false;
        }
    }
    // The fit's weights and moments depend on phi and the status only: they
    // are formed once, the contributing neighbours of the usual radius 3 kept
    // as a 7x7 bit mask.
    unsigned long long mask = 0;
    double al = 0, be = 0, ga = 0;
    bool wide = false, singular = false;
    int rw = 3;  // the fit's radius
    const double pp = mine ? L.phi[e] : 0;
    auto window = [&](int r, int &ilo, int &ihi, int &jlo, int &jhi) {
        ilo = i <= r ? -i : -r; ihi = i + r >= m ? m - 1 - i : r;
        jlo = j <= r ? -j : -r; jhi = j + r >= nn ? nn - 1 - j : r;
    };
    // A fit of a larger radius (none in the usual shapes: the moments of a
    // radius-3 window are far from singular unless the spacing is below about
    // 1e-5) reaches past the halo and reads the grid itself. Its mask holds one of
    // the outside points that it reads: the last in phi, mostly the last to be
    // final, and so the one to wait for (looking at the whole window, up to 225
    // points, at every poll instead took 3.1 ms for 13 tiles at 61 x 66 and spacing
    // 8e-6, now 0.32, and 49 ms for a band 40 cells deep on 700 x 690, now 1.9).
    if (todo) {
        // the radius-3 window, unrolled a row at a time; window points
        // outside the grid hold status -1, which the status test rejects, so
        // the window is the clipped one of traverse.hh:180-203
        double S = 0, Sx = 0, Sy = 0, Sxx = 0, Sxy = 0, Syy = 0;
#pragma unroll
        for (int dj = -3; dj <= 3; dj++) {
            int rs[7];
            double rp[7];
#pragma unroll
            for (int di = -3; di <= 3; di++) {
                rs[di + 3] = (int)L.st[e + dj * kEW + di] - 1;
                rp[di + 3] = L.phi[e + dj * kEW + di];
            }
#pragma unroll
            for (int di = -3; di <= 3; di++) {
                const int s = rs[di + 3];
                if (s < 2 || s > 5) continue;
                double wgt = rp[di + 3];
                if (!(wgt < pp)) continue;
                wgt = pp - wgt;
                S += wgt; Sx += di * wgt; Sy += dj * wgt;
                Sxx += di * di * wgt; Sxy += di * dj * wgt; Syy += dj * dj * wgt;
                mask |= 1ull << ((dj + 3) * 7 + di + 3);
            }
        }
        double det = S * (Sxy * Sxy - Sxx * Syy) + Sx * Sx * Syy - 2 * Sx * Sxy * Sy + Sy * Sy * Sxx;
        if (fabs(det) < 1e-10) {
            // the radius grows (traverse.hh:179-207) while the fit is
            // singular, to 7 at most; the radius it stops at depends on phi
            // and the status only
            wide = true;
            int rr = 4;
            do {
                int ilo, ihi, jlo, jhi;
                window(rr, ilo, ihi, jlo, jhi);
                S = Sx = Sy = Sxx = Sxy = Syy = 0;
                int last = -1;
                double least = INFINITY;
                for (int dj = jlo; dj <= jhi; dj++) {
                    const int p0 = q + dj * g.P;
#pragma unroll 1  // unrolled, it costs the loop below its registers
                    for (int di = ilo; di <= ihi; di++) {
                        const int s = a.st[p0 + di];  // read with phi, whatever it is
                        const double ph = a.phi[p0 + di], wgt = pp - ph;
                        if (s < 2 || s > 5 || !(ph < pp)) continue;
                        S += wgt; Sx += di * wgt; Sy += dj * wgt;
                        Sxx += di * di * wgt; Sxy += di * dj * wgt; Syy += dj * dj * wgt;
                        if (s >= 4 && wgt < least) {
                            least = wgt;
                            last = p0 + di;
                        }
                    }
                }
                mask = (unsigned)last;
                det = S * (Sxy * Sxy - Sxx * Syy) + Sx * Sx * Syy - 2 * Sx * Sxy * Sy + Sy * Sy * Sxx;
                rr++;
            } while (fabs(det) < 1e-10 && rr <= 7);
            rw = rr - 1;
            if (fabs(det) < 1e-10) singular = true;
        }
        if (singular) {
            atomicOr(&w.cnt[kCntErr], kErrSingular);  // the value stays
            ext_store(w.ex + q, L.x[e]);
            ext_store(w.ey + q, L.y[e]);
            atomicOr(&L.known[lj], 1u << li);
            todo = false;
        } else {
            det = 1 / det;
            al = (Sxy * Sxy - Sxx * Syy) * det;
            be = (Sx * Syy - Sxy * Sy) * det;
            ga = (Sxx * Sy - Sxy * Sx) * det;
            if (!wide) {
#pragma unroll
                for (int dj = -3; dj <= 3; dj++)
                    atomicOr(&L.need[lj + dj], (unsigned)(mask >> (7 * (dj + 3)) & 127u) << (li - 3));
            }
        }
    }
    if (todo && wide) L.wide = true;
    const unsigned long long open = __ballot(todo);
    if (lane == 0 && open) atomicAdd(&L.left, __popcll(open));
    __syncthreads();
    if (tid == 0) L.was = L.left;
    if (tid < kEHt) {  // the halo points to poll, a row a thread
        const unsigned own = tid >= kEH && tid < kEH + kExtY ? ((1u << kExtX) - 1) << kEH : 0u;
        unsigned b = L.need[tid] & ~L.known[tid] & ~own;
        int at = b ? atomicAdd(&L.nhalo, __popc(b)) : 0;
        for (; b; b &= b - 1) L.halo[at++] = (unsigned short)(tid * kEW + __ffs(b) - 1);
    }
    __syncthreads();
    if (wave == kExtWaves) {
        // the watching wavefront: values of the neighbours' points as they
        // come, until the tile is done or nothing has moved for `patience`
        // rounds
        const int nh = L.nhalo;
        // each lane keeps its points of the list in registers: a poll is
        // their two loads (0.1 us where the line is in the L2 and nothing
        // has come; a value takes 0.6-0.8 us from store to here)
        constexpr int kOwn = (kEN - kExtX * kExtY + 63) / 64;
        int at[kOwn], hp[kOwn];
#pragma unroll
        for (int u = 0; u < kOwn; u++) {
            const int k = lane + 64 * u;
            hp[u] = k < nh ? L.halo[k] : -1;
            at[u] = hp[u] < 0 ? 0 : g.ls(I0 + hp[u] % kEW, J0 + hp[u] / kEW);
        }
        // (a visit of larger windows takes long to set up)
        const int enough = L.wide && patience < kPatienceTake ? kPatienceTake : patience;
        int seen = -1, idle = 0, moved = -1;
        while (true) {
            unsigned long long px[kOwn], py[kOwn];
#pragma unroll
            for (int u = 0; u < kOwn; u++)
                if (64 * u < nh && hp[u] >= 0) {
                    px[u] = ext_load(w.ex + at[u]);
                    py[u] = ext_load(w.ey + at[u]);
                }
            bool got = false;
#pragma unroll
            for (int u = 0; u < kOwn; u++)
                if (64 * u < nh && hp[u] >= 0 && px[u] != kExtOpen && py[u] != kExtOpen) {
                    L.x[hp[u]] = __longlong_as_double((long long)px[u]);
                    L.y[hp[u]] = __longlong_as_double((long long)py[u]);
                    lds_order();
                    atomicOr(&L.known[hp[u] / kEW], 1u << (hp[u] % kEW));
                    hp[u] = -1;
                    got = true;
                }
            const bool any = __any(got);
            if (any && lane == 0) atomicAdd(&L.news, 1u);
            const int lf = lds_now(L.left);
            if (lf == 0) break;
            if (lf != seen || any) {
                if (((lf ^ seen) & -kTellPoints) && lane == 0) ext_tell(w);
                seen = lf;
                idle = 0;
            } else if (++idle > enough) {
                const int now = patience == kPatienceLast ? ext_moved(w) : moved;
                if (now == moved) {
                    if (lane == 0) atomicOr(&L.stop, 1);
                    break;
                }
                moved = now;
                idle = 0;
            }
            if (!nh) __builtin_amdgcn_s_sleep(8);
        }
    } else {
        const int dk = lane < 49 ? lane : 0, dj = dk / 7 - 3, di = dk % 7 - 3, off = dj * kEW + di;
        const double xx = di, yy = dj;
        double *pr = &L.prod[wave][0][0];
        const bool store = mine && (w.mark[q] == 4 || w.mark[q] == 5);  // a point of the band as it was built
        // The products of the lanes with `in` set (weight wgt, window
        // position (cx, cy), values (fa, fb)) added to the sums that lanes
        // 0 to 5 hold, one each, in lane order.
        auto add_up = [&](bool in, double wgt, double cx, double cy, double fa, double fb, double &sum) {
            const unsigned long long bits = __ballot(in);
            const int n = __popcll(bits);
            const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(bits >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bits, 0));
            const double wx = wgt * cx, wy = wgt * cy;
            // the other lanes fill the row up with -0.0, which leaves any
            // sum as it is
            const int at = in ? rank : n + lane - rank;
            if (at < kExtProd) {
                pr[at] = in ? wgt * fa : -0.0;
                pr[kExtProd + at] = in ? wx * fa : -0.0;
                pr[2 * kExtProd + at] = in ? wy * fa : -0.0;
                pr[3 * kExtProd + at] = in ? wgt * fb : -0.0;
                pr[4 * kExtProd + at] = in ? wx * fb : -0.0;
                pr[5 * kExtProd + at] = in ? wy * fb : -0.0;
            }
            lds_order();
            if (lane < 6) {
                const double *row = pr + lane * kExtProd;
                for (int k = 0; k < n; k += 8) {
                    double v[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) v[u] = row[k + u];
#pragma unroll
                    for (int u = 0; u < 8; u++) sum += v[u];
                }
            }
            lds_order();
        };
        // The grid points of lane l's larger window that its fit reads, up
        // to `most` at a time in window order, one a lane:
        // f(read, point, status, weight, x, y).
        auto each_wide = [&](int l, int most, auto f) {
            const int ql = __builtin_amdgcn_readlane(q, l), rl = __builtin_amdgcn_readlane(rw, l),
                      il = __builtin_amdgcn_readlane(i, l), jl = __builtin_amdgcn_readlane(j, l), wd = 2 * rl + 1;
            const double pe = lane_double(pp, l);
            for (int k0 = 0; k0 < wd * wd; k0 += most) {
                const int k = k0 + lane, cy = k / wd - rl, cx = k % wd - rl, p = ql + cy * g.P + cx;
                bool in = lane < most && k < wd * wd && il + cx >= 0 && il + cx < m && jl + cy >= 0 && jl + cy < nn;
                const int st = in ? a.st[p] : 0;
                in = in && st >= 2 && st <= 5;
                const double ph = in ? a.phi[p] : 0;
                f(in && ph < pe, p, st, pe - ph, cx, cy);
            }
            // the loads end here: a wait further on, in code that the usual
            // path shares, would also wait for that path's last stores
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        };
        // the points of this wavefront; by itself where none has a larger window,
        // whose code would cost that loop registers
        auto work = [&](auto larger) {
            constexpr bool WIDE = decltype(larger)::value;
            while (__any(todo)) {
                const unsigned news = lds_now(L.news);
                lds_order();
                bool ready = false;
                if (todo && !(WIDE && wide)) {
                    // (plain reads, issued together: one after the other they
                    // took half of a link's time)
                    unsigned k[7], miss = 0;
#pragma unroll
                    for (int b = 0; b < 7; b++) k[b] = L.known[lj + b - 3];
#pragma unroll
                    for (int b = 0; b < 7; b++) miss |= (unsigned)(mask >> (7 * b)) & 127u & ~(k[b] >> (li - 3));
                    ready = !miss;
                }
                const unsigned long long far = WIDE ? __ballot(todo && wide) : 0;
                if (WIDE && todo && wide) {
                    const int p = (int)(unsigned)mask;
                    ready = p < 0 || (ext_load(w.ex + p) != kExtOpen && ext_load(w.ey + p) != kExtOpen);
                }
                const unsigned long long rd = __ballot(ready);
                if (!rd) {
                    // nothing to do until another value is final: a spin on one
                    // word leaves the SIMD to the wavefronts that work (a larger
                    // window waits for values outside the tile too)
                    int end = 0;
                    do {
                        __builtin_amdgcn_s_sleep(1);
                        end = lds_now(L.stop);
                    } while (!end && !far && lds_now(L.news) == news);
                    if (end) {
                        if (lane == 0) atomicMin(&L.quit, news);
                        break;
                    }
                    continue;
                }
                lds_order();
                unsigned long long done = rd;
                for (unsigned long long b = rd; b; b &= b - 1) {
                    const int l = __ffsll((long long)b) - 1;
                    double sum = 0;
                    if (!WIDE || !(far >> l & 1)) {
                        const int el = __builtin_amdgcn_readlane(e, l);
                        const unsigned mlo = __builtin_amdgcn_readlane((unsigned)mask, l),
                                       mhi = __builtin_amdgcn_readlane((unsigned)(mask >> 32), l);
                        add_up(lane < 49 && ((lane < 32 ? mlo >> lane : mhi >> (lane - 32)) & 1), L.phi[el] - L.phi[el + off],
                               xx, yy, L.x[el + off], L.y[el + off], sum);
                    } else {
                        int last = -1;  // a point that is open still: the next to wait for
                        double least = INFINITY;
                        each_wide(l, 48, [&](bool in, int p, int st, double wgt, int cx, int cy) {
                            double fa = 0, fb = 0;
                            if (in && st >= 4) {
                                const unsigned long long bx = ext_load(w.ex + p), by = ext_load(w.ey + p);
                                fa = __longlong_as_double((long long)bx);
                                fb = __longlong_as_double((long long)by);
                                if ((bx == kExtOpen || by == kExtOpen) && wgt < least) {
                                    least = wgt;
                                    last = p;
                                }
                            } else if (in) {
                                fa = a.nX[p];
                                fb = a.nY[p];
                            }
                            add_up(in, wgt, cx, cy, fa, fb, sum);
                        });
                        if (__any(last >= 0)) {
                            for (int h = 32; h > 0; h /= 2) {
                                const double o = __shfl_xor(least, h, 64);
                                const int po = __shfl_xor(last, h, 64);
                                if (o < least) {
                                    least = o;
                                    last = po;
                                }
                            }
                            if (lane == l) mask = (unsigned)last;
                            done &= ~(1ull << l);
                            continue;
                        }
                    }
                    const double p0 = lane_double(sum, 0), p1 = lane_double(sum, 1), p2 = lane_double(sum, 2),
                                 p3 = lane_double(sum, 3), p4 = lane_double(sum, 4), p5 = lane_double(sum, 5);
                    if (lane == l) {
                        const double vx = p0 * al + p1 * be + p2 * ga, vy = p3 * al + p4 * be + p5 * ga;
                        L.x[e] = vx;
                        L.y[e] = vy;
                        lds_order();
                        atomicOr(&L.known[lj], 1u << li);
                        atomicAdd(&L.news, 1u);
                        ext_store(w.ex + q, vx);
                        ext_store(w.ey + q, vy);
                        if (store) {
                            a.nX[q] = vx;
                            a.nY[q] = vy;
                        }
                        todo = false;
                    }
                }
                if (lane == 0) atomicSub(&L.left, __popcll(done));
                if (many && lane == 0 && done) (void)__hip_atomic_fetch_add(&w.tprog[tile], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        };
        if (__any(todo && wide)) work(std::true_type());
        else work(std::false_type());
    }
    __syncthreads();
}

// Tiles that hold what a part of a tile reads, to either side (fits reach 7 points)
constexpr int kNewsX = (7 + kTileX - 1) / kTileX, kNewsY = (7 + kTileY - 1) / kTileY;
static_assert((2 * kNewsX + 1) * (2 * kNewsY + 1) <= 64, "a lane a tile");
// The sum of those tiles' counters of evaluated batches (its own tile's only where
// that has other parts): where it stays, a visit would find what the last one left.
// For a whole wavefront.
__device__ __forceinline__ int ext_news(const LsWork &w, int tile) {
    const int lane = __lane_id(), dx = lane % (2 * kNewsX + 1) - kNewsX, dy = lane / (2 * kNewsX + 1) - kNewsY;
    const int X = tile % w.ntx + dx, Y = tile / w.ntx + dy;
    int n = 0;
    if (dy <= kNewsY && X >= 0 && X < w.ntx && Y >= 0 && Y < w.nty && (kExtPerTile > 1 || dx || dy))
        n = __hip_atomic_load(&w.tprog[tile + dy * w.ntx + dx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int h = 32; h > 0; h /= 2) n += __shfl_xor(n, h, 64);
    return n;
}

// The workgroup's next visit, by its first wavefront. A workgroup takes one tile
// and, while there are others that nobody has, a further one whenever a look at
// all it holds brought nothing: so a tile that others wait for is held by a
// workgroup that runs, however many there are. It visits a tile again when
// ext_news has changed. (With the tiles dealt out beforehand and visited in turn,
// news or not, a band 200 cells wide on 1400^2, 2963 tiles, took 700 to 1040 ms, now
// 9; a lattice of blobs, 6924 tiles, 12.5 to 14, now 2.4.)
__device__ __forceinline__ void ext_next(const LsWork &w, ExtLds &L, int nt, int p, int slot) {
    const bool first = __lane_id() == 0;
    int k = L.k, held = L.nheld, idle = L.idle;
    bool more = L.more, take = L.take;
    auto go = [&](int t, int news, bool fresh, int patience) {
        if (!first) return;
        L.t = t; L.k = k; L.heard = news; L.fresh = fresh; L.patience = patience;
        L.nheld = held; L.idle = idle; L.more = more; L.take = take;
    };
    auto end = [&]() {
        if (L.open + held && first) atomicAdd(&w.cnt[kCntIter + slot], L.open + held);
        go(-1, 0, false, 0);
    };
    // the visit that has ended
    const int left = L.left;
    if (left < L.was) {
        idle = 0;
        take = false;
        if (first) ext_tell(w);
    } else {
        idle += kPatienceMany;
    }
    if (left) {
        // (a wavefront that gave up before the last values came here may have
        // points that are ready now)
        if (first) L.seen[k] = L.quit == L.news ? L.heard : -2;
        k++;
    } else {  // the last one takes its place
        held--;
        if (first) {
            L.held[k] = L.held[held];
            L.seen[k] = L.seen[held];
        }
    }
    lds_order();
    // the last of all was waited for as long as anything moved
    if (L.patience == kPatienceLast) return end();
    while (true) {
        const bool one = held == 1 && !more;
        for (; k < held; k++) {
            const int t = L.held[k], seen = L.seen[k];
            const int news = ext_news(w, w.tiles_ext[t / kExtPerTile]);
            if (seen != news || one)
                return go(t, news, p == 0 && seen == -1, one ? kPatienceLast : held == 1 ? kPatienceTake : kPatienceMany);
            idle++;
        }
        // all looked at
        if (idle > kIdleMany) {  // nothing for long: stay while any of the solid's tiles moves
            const int now = ext_moved(w);
            if (now == L.moved) {
                if (first) L.open += held;
                held = 0;
            } else if (first) {
                L.moved = now;
            }
            lds_order();
            idle = 0;
        }
        if (more && (take || !held) && held < kExtHeld) {
            int t = 0;
            if (first) t = gridDim.x + atomicAdd(&w.cnt[kCntTicket + slot], 1);
            t = __builtin_amdgcn_readfirstlane(t);
            more = t < nt;
            if (more) {
                if (first) {
                    L.held[held] = t;
                    L.seen[held] = -1;
                }
                held++;
                lds_order();
            }
        }
        if (!held && !more) return end();
        k = 0;
        take = true;
    }
}

__device__ __forceinline__ void extend_tiles(const Grid &g, const ObjArrays &a, const LsWork &w, int p, int slot) {
    __shared__ ExtLds L;
    if (slot > 0 && w.cnt[kCntIter + slot - 1] == 0) return;  // nothing left open
    const int nt = w.cnt[kCntTileExt] * kExtPerTile;
    if ((int)blockIdx.x >= nt) return;
    const bool many = __builtin_amdgcn_readfirstlane(nt > (int)gridDim.x);
    // the first tile is the workgroup's own, the others go by ticket
    if (threadIdx.x == 0) {
        L.held[0] = blockIdx.x;
        L.patience = many ? kPatienceTake : kPatienceLast;
        L.t = L.k = L.idle = L.open = 0;
        L.heard = -2;  // not asked
        L.nheld = 1;
        L.moved = -1;
        L.fresh = p == 0;
        L.more = L.take = many;
    }
    int t = blockIdx.x;
    bool fresh = p == 0;
    int patience = many ? kPatienceTake : kPatienceLast;
    while (true) {
        extend_tile(g, a, w, L, w.tiles_ext[t / kExtPerTile], t % kExtPerTile, fresh, many, patience);
        if (!many) {
            if (L.left && threadIdx.x == 0) atomicAdd(&w.cnt[kCntIter + slot], 1);
            break;
        }
        if (threadIdx.x < 64) ext_next(w, L, nt, p, slot);
        __syncthreads();
        t = L.t;
        if (t < 0) break;
        fresh = L.fresh;
        patience = L.patience;
    }
}
__global__ __launch_bounds__(kExtThreads, 5) void k_extend_tiles(Grid g, ObjArrays a, LsWork w, int p, int slot) {
    extend_tiles(g, a, w, p, slot);
}
// The extension of several solids in one launch: workgroup (x, y) takes
// solid y's tiles as workgroup x of its own launch would.
struct ExtItem {
    ObjArrays a;
    LsWork w;
};
// (6 wavefronts a SIMD, a few spilled registers: many solids want more
// workgroups at once, 0.87 -> 0.75 ms for 64 circles; a lone solid's do not
// fill the chip and are faster without the spills, 91 against 95 us.)
__global__ __launch_bounds__(kExtThreads, 6) void k_extend_tiles_batch(Grid g, const ExtItem *it, int p, int slot) {
    const ExtItem &x = it[blockIdx.y];
    extend_tiles(g, x.a, x.w, p, slot);
}
__global__ __launch_bounds__(kTileThreads) void k_ext_open_b(Grid g, const ExtItem *it) {
    const ExtItem &x = it[blockIdx.y];
    ext_open_body(g, x.a, x.w);
}
// Counters of a batch of solids: clear the passes' tickets and slots of every solid, or
// gather its error flags and the first `batch` slots into out (batch + 1
// ints per solid)
template <class Item>
__global__ void k_batch_zero(const Item *it, int n) {
    for (int k = blockIdx.x; k < n; k += gridDim.x)
        for (int e = threadIdx.x; e < 2 * kIterSlots; e += blockDim.x) it[k].w.cnt[kCntTicket + e] = 0;
}
template <class Item>
__global__ void k_batch_gather(const Item *it, int n, int batch, int *out) {
    for (int k = blockIdx.x; k < n; k += gridDim.x)
        for (int e = threadIdx.x; e <= batch; e += blockDim.x)
            out[k * (batch + 1) + e] = e == 0 ? it[k].w.cnt[kCntErr] : it[k].w.cnt[kCntIter + e - 1];
}

// ---- the set-up and finish of several solids' rebuilds in shared launches: workgroup (x, y, z) does
// what workgroup (x, y) of the single-solid launch does for solid z, whose
// windows and parameters are item z (grids sized for the largest window;
// workgroups past a solid's window do nothing). The solids' arrays and
// counters are their own, so each gets exactly what its own launches give.
struct SetupItem {
    ObjConst c;
    ObjArrays a;
    LsWork w;
    Win wn, wr;                   // the rebuild's window, the row dilation's
    int R;                        // dilation radius
    int pin;                      // pin before the rebuild
    const double *pin_x, *pin_y;  // (nX, nY) standing in for (X, Y) inside, or null
    const double *v;              // finish: the fixed-point buffer of the last pass
};
__global__ void k_pin_b(Grid g, const SetupItem *it) {
    const SetupItem &x = it[blockIdx.z];
    if (x.pin) pin_body(g, x.c, x.a, x.wn, x.pin_x, x.pin_y);
}
// starts a rebuild's counters and band box
__global__ void k_counts_b(const SetupItem *it, int n) {
    int *cnt = it[blockIdx.z].w.cnt;
    bbox_clear(it[blockIdx.z].w.bbox);
    for (int k = threadIdx.x; k < n; k += blockDim.x) cnt[k] = 0;
}
__global__ void k_scan_b(Grid g, const SetupItem *it) {
    const SetupItem &x = it[blockIdx.z];
    scan_body(g, x.a, x.w, x.wn);
}
__global__ __launch_bounds__(kNewtonThreads) void k_newton_b(Grid g, LsGeom lg, const SetupItem *it) {
    const SetupItem &x = it[blockIdx.z];
    newton_body(g, lg, x.a, x.w);
}
__global__ void k_dilate_rows_b(Grid g, const SetupItem *it) {
    const SetupItem &x = it[blockIdx.z];
    dilate_rows_body(g, x.a, x.w, x.R < g.ml ? x.R : g.ml, x.wr);
}
__global__ void k_dilate_cols_b(Grid g, const SetupItem *it) {
    const SetupItem &x = it[blockIdx.z];
    dilate_cols_body(g, x.a, x.w, x.R < g.nl ? x.R : g.nl, x.wn);
}
__global__ void k_compact_tiles_b(const SetupItem *it, int ext) {
    const LsWork &w = it[blockIdx.z].w;
    if (ext) compact_tiles_body(w, 2, w.tiles_ext, kCntTileExt);
    else compact_tiles_body(w, 1, w.tiles_fim, kCntTileFim);
}
__global__ void k_finalize_b(Grid g, const SetupItem *it) {
    const SetupItem &x = it[blockIdx.z];
    finalize_body(g, x.c, x.a, x.w, x.v, x.wn);
}
__global__ void k_commit_status_b(Grid g, const SetupItem *it) {
    const SetupItem &x = it[blockIdx.z];
    commit_status_body(g, x.a, x.w, x.wn);
}

#define KCHECK() HIP_CHECK(hipGetLastError())

// Run a fixed-point iteration in batches of passes, reading the change
// counts back once per batch. A pass whose predecessor in the batch changed
// nothing returns at once (the fixed point is reached and both ping-pong
// buffers hold it), so a batch may safely run past convergence; its length
// is the number of passes the previous iteration needed, which usually
// makes one host round trip per iteration. *passes_out: passes up to and
// including the first one that changed nothing. Returns 0, 7 when
// max_passes pass without convergence, or a HIP error.
// Its two halves: enqueue one batch of passes (starting at pass `passes`)
// with the read-back of its counters, and, once the stream has run them,
// decide from the counters whether the iteration has ended. zeroed: the
// first batch's counters are zero already (a rebuild's set-up cleared them).
template <class F>
int iter_enqueue(hipStream_t s, LsWork &w, int predict, int passes, F pass, int &batch, int least = 2,
                 bool zeroed = false) {
    batch = predict < least ? least : predict;
    if (batch > kIterSlots) batch = kIterSlots;
    if (passes || !zeroed) {
        k_zero_counts<<<1, 64, 0, s>>>(w.cnt + kCntTicket, 2 * kIterSlots);
        KCHECK();
    }
    for (int b = 0; b < batch; b++)
        if (int rc = pass(passes + b, b)) return rc;
    HIP_CHECK(hipMemcpyAsync(w.hcnt, w.cnt, (kCntIter + kIterSlots) * sizeof(int), hipMemcpyDeviceToHost, s));
    return 0;
}
bool iter_done(LsWork &w, int &predict, int &passes, int batch, int *passes_out) {
    if (w.hcnt[kCntErr]) {
        *passes_out = passes + batch;
        return true;
    }
    for (int b = 0; b < batch; b++)
        if (w.hcnt[kCntIter + b] == 0) {
            *passes_out = passes + b + 1;
            predict = passes + b + 1;
            return true;
        }
    passes += batch;
    predict = passes + 2;
    return false;
}
template <class F>
int iterate(hipStream_t s, LsWork &w, int &predict, int max_passes, F pass, int *passes_out, int least = 2,
            bool zeroed = false) {
    int passes = 0;
    while (passes < max_passes) {
        int batch;
        if (int rc = iter_enqueue(s, w, predict, passes, pass, batch, least, zeroed)) return rc;
        HIP_CHECK(hipStreamSynchronize(s));
        if (iter_done(w, predict, passes, batch, passes_out)) return 0;
    }
    *passes_out = passes;
    return 7;
}

// The same iteration for several solids at once: every pass is one launch
// for all solids not yet at their fixed point (launch(p, slot, items, n)),
// one gather of their counters per batch. Each solid's passes, results,
// pass count and prediction are those of iterate on it alone; its error
// flags go to its host mirror (hcnt[kCntErr]).
// Its state between the halves (enqueue one batch of passes with the
// gather and read-back of the counters; once the stream has run them,
// decide per solid), so that a caller can overlap the first batch with other
// work.
template <class Item>
struct BatchIter {
    std::vector<Item> items;
    std::vector<int *> predict;
    std::vector<size_t> idx;  // solids still going
    std::vector<int> passes_out;
    int passes = 0, batch = 0, least = 2;  // least: passes a batch has at least
    void start(std::vector<Item> it, std::vector<int *> pr) {
        items = std::move(it);
        predict = std::move(pr);
        idx.resize(items.size());
        for (size_t k = 0; k < idx.size(); k++) idx[k] = k;
        passes_out.assign(items.size(), 0);
        passes = batch = 0;
    }
};
template <class Item, class F>
int batch_enqueue(hipStream_t s, LsBatch &bt, BatchIter<Item> &it, F launch) {
    Item *d_items = (Item *)bt.d_items, *h_items = (Item *)bt.h_items;
    const int n = (int)it.idx.size();
    int batch = it.least;
    for (size_t k : it.idx) batch = std::max(batch, *it.predict[k]);
    if (batch > kIterSlots) batch = kIterSlots;
    it.batch = batch;
    for (int k = 0; k < n; k++) h_items[k] = it.items[it.idx[k]];
    HIP_CHECK(hipMemcpyAsync(d_items, h_items, n * sizeof(Item), hipMemcpyHostToDevice, s));
    k_batch_zero<Item><<<n < 256 ? n : 256, 64, 0, s>>>(d_items, n);
    KCHECK();
    for (int b = 0; b < batch; b++)
        if (int rc = launch(it.passes + b, b, d_items, n)) return rc;
    k_batch_gather<Item><<<n < 256 ? n : 256, 64, 0, s>>>(d_items, n, batch, bt.d_cnt);
    KCHECK();
    HIP_CHECK(hipMemcpyAsync(bt.h_cnt, bt.d_cnt, (size_t)n * (batch + 1) * sizeof(int), hipMemcpyDeviceToHost, s));
    return 0;
}
template <class Item>
void batch_check(LsBatch &bt, BatchIter<Item> &it) {
    const int n = (int)it.idx.size(), batch = it.batch;
    std::vector<size_t> rest;
    for (int k = 0; k < n; k++) {
        const int *c = bt.h_cnt + (size_t)k * (batch + 1);
        const size_t id = it.idx[k];
        it.items[id].w.hcnt[kCntErr] = c[0];
        if (c[0]) {
            it.passes_out[id] = it.passes + batch;
            continue;
        }
        int done = -1;
        for (int b = 0; b < batch && done < 0; b++)
            if (c[1 + b] == 0) done = b;
        if (done >= 0) {
            it.passes_out[id] = it.passes + done + 1;
            *it.predict[id] = it.passes + done + 1;
        } else {
            rest.push_back(id);
        }
    }
    it.passes += batch;
    for (size_t id : rest) *it.predict[id] = it.passes + 2;
    it.idx.swap(rest);
}
// the loop from the state left by batch_enqueue's first batch, or from the start
template <class Item, class F>
int batch_finish(hipStream_t s, LsBatch &bt, BatchIter<Item> &it, int max_passes, F launch, bool pending) {
    if (pending) {
        HIP_CHECK(hipStreamSynchronize(s));
        batch_check(bt, it);
    }
    while (!it.idx.empty()) {
        if (it.passes >= max_passes) {
            for (size_t k : it.idx) it.passes_out[k] = it.passes;
            return 7;
        }
        if (int rc = batch_enqueue(s, bt, it, launch)) return rc;
        HIP_CHECK(hipStreamSynchronize(s));
        batch_check(bt, it);
    }
    return 0;
}
template <class Item, class F>
int iterate_batch(hipStream_t s, LsBatch &bt, std::vector<Item> items, std::vector<int *> predict, int max_passes,
                  F launch, std::vector<int> &passes_out, int least = 2) {
    BatchIter<Item> it;
    it.least = least;
    it.start(std::move(items), std::move(predict));
    const int rc = batch_finish(s, bt, it, max_passes, launch, false);
    passes_out = it.passes_out;
    return rc;
}

}  // namespace

int ls_batch_alloc(int cap, LsBatch &bt) {
    const size_t bytes = (size_t)cap * std::max(sizeof(FimItem), sizeof(ExtItem));
    HIP_CHECK(hipMalloc(&bt.d_items, bytes));
    HIP_CHECK(hipHostMalloc(&bt.h_items, bytes, hipHostMallocDefault));
    HIP_CHECK(hipMalloc((void **)&bt.d_cnt, (size_t)cap * (kIterSlots + 1) * sizeof(int)));
    HIP_CHECK(hipHostMalloc((void **)&bt.h_cnt, (size_t)cap * (kIterSlots + 1) * sizeof(int), hipHostMallocDefault));
    bt.setup_stride = ((size_t)cap * sizeof(SetupItem) + 255) / 256 * 256;
    HIP_CHECK(hipMalloc(&bt.d_setup, 2 * bt.setup_stride));
    HIP_CHECK(hipHostMalloc(&bt.h_setup, 2 * bt.setup_stride, hipHostMallocDefault));
    for (hipEvent_t &e : bt.ev_setup) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    bt.cap = cap;
    return 0;
}

void ls_batch_free(LsBatch &bt) {
    if (bt.d_items) (void)hipFree(bt.d_items);
    if (bt.h_items) (void)hipHostFree(bt.h_items);
    if (bt.d_cnt) (void)hipFree(bt.d_cnt);
    if (bt.h_cnt) (void)hipHostFree(bt.h_cnt);
    if (bt.d_setup) (void)hipFree(bt.d_setup);
    if (bt.h_setup) (void)hipHostFree(bt.h_setup);
    for (hipEvent_t e : bt.ev_setup)
        if (e) (void)hipEventDestroy(e);
    bt = LsBatch{};
}

int ls_alloc(const Grid &g, LsWork &w, hipStream_t s) {
    const size_t N = (size_t)g.N;
    double **d[] = {&w.va, &w.vb, &w.ex, &w.ey};
    for (auto p : d) {
        HIP_CHECK(hipMalloc((void **)p, N * sizeof(double)));
        HIP_CHECK(memset_sync(*p, 0, N * sizeof(double), s));
    }
    const size_t L = (size_t)g.ml * g.nl + 64;
    HIP_CHECK(hipMalloc((void **)&w.iface, L * sizeof(int)));
    HIP_CHECK(hipMalloc((void **)&w.mark, N));
    HIP_CHECK(memset_sync(w.mark, 0, N, s));
    HIP_CHECK(hipMalloc((void **)&w.cflag, N));
    HIP_CHECK(memset_sync(w.cflag, 0, N, s));
    w.ntx = (g.ml + kTileX - 1) / kTileX;
    w.nty = (g.nl + kTileY - 1) / kTileY;
    const size_t T = (size_t)w.ntx * w.nty + 64;
    HIP_CHECK(hipMalloc((void **)&w.tflag, T * sizeof(int)));
    HIP_CHECK(memset_sync(w.tflag, 0, T * sizeof(int), s));
    HIP_CHECK(hipMalloc((void **)&w.tiles_fim, T * sizeof(int)));
    HIP_CHECK(hipMalloc((void **)&w.tiles_ext, T * sizeof(int)));
    HIP_CHECK(hipMalloc((void **)&w.tprog, T * sizeof(int)));
    HIP_CHECK(memset_sync(w.tprog, 0, T * sizeof(int), s));
    HIP_CHECK(hipMalloc((void **)&w.cnt, (kCntIter + kIterSlots) * sizeof(int)));
    HIP_CHECK(hipHostMalloc((void **)&w.hcnt, (kCntIter + kIterSlots) * sizeof(int), hipHostMallocDefault));
    HIP_CHECK(hipMalloc((void **)&w.bbox, 4 * sizeof(int)));
    HIP_CHECK(hipHostMalloc((void **)&w.hbbox, 4 * sizeof(int), hipHostMallocDefault));
    HIP_CHECK(hipEventCreateWithFlags(&w.ev_bbox, hipEventDisableTiming));
    return 0;
}

void ls_free(LsWork &w) {
    void *p[] = {w.va, w.vb, w.ex, w.ey, w.iface, w.mark, w.cflag, w.tflag,
                 w.tiles_fim, w.tiles_ext, w.tprog, w.cnt, w.bbox};
    for (auto q : p)
        if (q) (void)hipFree(q);
    if (w.hcnt) (void)hipHostFree(w.hcnt);
    if (w.hbbox) (void)hipHostFree(w.hbbox);
    if (w.ev_bbox) (void)hipEventDestroy(w.ev_bbox);
    w = LsWork{};
}

// The points a rebuild may change lie within the reach of the march from
// the previous band. The window is the union of every earlier window and
// the previous band's bounding box (statuses 1..6) widened by that reach
// plus two, aligned outward to whole tiles; it never shrinks, so every
// point outside it still holds what the first, whole-grid rebuild left
// there (status 0 or 7, phi at the cut-off, +-inf in the march buffers).
static Win next_window(const Grid &g, LsWork &w, int R) {
    const Win full{0, g.ml, 0, g.nl};
    if (!w.have_win) return full;
    Win v{w.win[0], w.win[1], w.win[2], w.win[3]};
    if (w.bbox_pending) {
        (void)hipEventSynchronize(w.ev_bbox);
        w.bbox_pending = false;
        const int *b = w.hbbox;
        if (b[1] >= 0) {
            const int m = R + 2;
            int I0 = (b[0] - m) / kTileX * kTileX, I1 = ((b[1] + 1 + m + kTileX - 1) / kTileX) * kTileX;
            int J0 = (b[2] - m) / kTileY * kTileY, J1 = ((b[3] + 1 + m + kTileY - 1) / kTileY) * kTileY;
            if (b[0] - m < 0) I0 = 0;
            if (b[2] - m < 0) J0 = 0;
            if (I1 > g.ml) I1 = g.ml;
            if (J1 > g.nl) J1 = g.nl;
            if (v.I1 <= v.I0) v = Win{I0, I1, J0, J1};
            else v = Win{I0 < v.I0 ? I0 : v.I0, I1 > v.I1 ? I1 : v.I1, J0 < v.J0 ? J0 : v.J0, J1 > v.J1 ? J1 : v.J1};
        }
    }
    return v;
}

// A rebuild in three parts: the set-up (pinning, interface list, Newton
// closest points, dilation to the march region, active tiles), the march
// passes, and the finish (final band and statuses, the extension's tiles).
// *live = false: nothing of the solid is left on the grid (nothing to do).
// The host side of a rebuild's set-up: its window wn, the row dilation's
// window wr, the dilation radius R; false when the window is empty.
static bool rebuild_window(const Grid &g, const ObjConst &c, LsWork &w, Win &wn, Win &wr, bool &whole, int &R) {
    // the march cannot accept a point further than limit/h + 2 cells (max
    // norm) from the interface layer: beyond it every path is longer
    const double reach = fmax(-c.phi_down, c.phi_up) / fmin(g.dx, g.dy) + 3;
    R = reach > g.ml + g.nl ? g.ml + g.nl : (int)reach;
    whole = !w.have_win;
    wn = next_window(g, w, R);
    if (wn.I1 <= wn.I0 || wn.J1 <= wn.J0) return false;
    // the row dilation also covers R rows either side, which the column pass reads
    wr = Win{wn.I0, wn.I1, wn.J0 - R < 0 ? 0 : wn.J0 - R, wn.J1 + R > g.nl ? g.nl : wn.J1 + R};
    return true;
}

static int rebuild_setup(hipStream_t s, const Grid &g, const ObjConst &c, const ObjArrays &a, LsWork &w, Win &wn,
                         bool &whole, bool *live, const double *pin_x = nullptr, const double *pin_y = nullptr) {
    const dim3 bb(BX, BY);
    Win wr;
    int R;
    *live = rebuild_window(g, c, w, wn, wr, whole, R);
    if (!*live) return 0;
    if (w.pin_first) {
        k_pin<<<grid_win(wn), bb, 0, s>>>(g, c, a, wn, pin_x, pin_y);
        KCHECK();
    }
    k_zero_counts<<<1, 64, 0, s>>>(w.cnt, kCntIter + kIterSlots, w.bbox);
    KCHECK();
    k_scan<<<grid_rows(wn), bb, 0, s>>>(g, a, w, wn);
    KCHECK();
    k_newton<<<kListBlocks, kNewtonThreads, 0, s>>>(g, geom_of(g), a, w);
    KCHECK();
    k_dilate_rows<<<grid_rows(wr), bb, 0, s>>>(g, a, w, R < g.ml ? R : g.ml, wr);
    KCHECK();
    k_dilate_cols<<<grid_win_cols(wn), bb, 0, s>>>(g, a, w, R < g.nl ? R : g.nl, wn);
    KCHECK();
    k_compact_tiles<<<64, 256, 0, s>>>(w, 1, w.tiles_fim, kCntTileFim);
    KCHECK();
    return 0;
}

// The host side of a rebuild's finish (after its last kernel, which writes the
// band's box to the host): the event to wait for and the window the next rebuild grows from.
static int finish_window(hipStream_t s, LsWork &w, const Win &wn, bool whole) {
    if (w.ev_bbox) {  // a work set without the event keeps no window (one-off rebuilds)
        HIP_CHECK(hipEventRecord(w.ev_bbox, s));
        w.bbox_pending = true;
    }
    w.have_win = true;
    if (whole) {  // windows grow from the band's box, not from the whole grid
        w.win[0] = w.win[1] = w.win[2] = w.win[3] = 0;
    } else {
        w.win[0] = wn.I0; w.win[1] = wn.I1; w.win[2] = wn.J0; w.win[3] = wn.J1;
    }
    return 0;
}

static int rebuild_finish(hipStream_t s, const Grid &g, const ObjConst &c, const ObjArrays &a, LsWork &w,
                          const Win &wn, bool whole, int passes) {
    const dim3 bb(BX, BY);
    double *bufs[2] = {w.va, w.vb};
    k_finalize<<<grid_rows(wn), bb, 0, s>>>(g, c, a, w, bufs[passes & 1], wn);
    KCHECK();
    k_compact_tiles<<<64, 256, 0, s>>>(w, 2, w.tiles_ext, kCntTileExt);
    KCHECK();
    k_commit_status<<<grid_win(wn), bb, 0, s>>>(g, a, w, wn);
    KCHECK();
    return finish_window(s, w, wn, whole);
}

constexpr int kMaxFimPasses = 4096;

// One march pass of a single solid
static int fim_pass(hipStream_t s, const Grid &g, const EikGeom &eg, const ObjConst &c, const ObjArrays &a,
                    const LsWork &w, int p, int slot) {
    double *bufs[2] = {w.va, w.vb};
    k_fim_tiles<<<kTileBlocks, kTileThreads, 0, s>>>(g, eg, c, a, w, bufs[p & 1], bufs[(p + 1) & 1], slot, 64);
    KCHECK();
    return 0;
}

static int rebuild_common(hipStream_t s, const Grid &g, const ObjConst &c, const ObjArrays &a, LsWork &w,
                          int *fim_iters) {
    Win wn;
    bool whole, live;
    if (int rc = rebuild_setup(s, g, c, a, w, wn, whole, &live)) return rc;
    if (!live) return 0;
    EikGeom eg;
    eg.init(g.dx, g.dy);
    int passes = 0;
    int rc = iterate(s, w, w.pred_fim, kMaxFimPasses,
                     [&](int p, int slot) { return fim_pass(s, g, eg, c, a, w, p, slot); }, &passes, 2, true);
    if (rc) return rc;
    if (w.hcnt[kCntErr] & kErrNewton) return 3;
    if (fim_iters) *fim_iters = passes;
    return rebuild_finish(s, g, c, a, w, wn, whole, passes);
}

// Workgroups per solid of a batched pass: the single-solid count shared out,
// at least 64
static int batch_blocks(int n) { return std::max(64, kTileBlocks / std::max(1, (n + 3) / 4)); }

// Upload the items of one region (0 set-up, 1 finish) after its last upload
// has run; the device copy of the items.
static const SetupItem *upload_items(hipStream_t s, LsBatch &bt, int region, const std::vector<SetupItem> &v,
                                     int *rc) {
    *rc = 0;
    if (bt.setup_used[region]) {
        const hipError_t e = hipEventSynchronize(bt.ev_setup[region]);
        if (e != hipSuccess) {
            *rc = hip_fail(e, "hipEventSynchronize", __FILE__, __LINE__);
            return nullptr;
        }
    }
    SetupItem *h = (SetupItem *)((char *)bt.h_setup + region * bt.setup_stride);
    SetupItem *d = (SetupItem *)((char *)bt.d_setup + region * bt.setup_stride);
    std::copy(v.begin(), v.end(), h);
    hipError_t e = hipMemcpyAsync(d, h, v.size() * sizeof(SetupItem), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipEventRecord(bt.ev_setup[region], s);
    if (e != hipSuccess) {
        *rc = hip_fail(e, "upload of batch items", __FILE__, __LINE__);
        return nullptr;
    }
    bt.setup_used[region] = true;
    return d;
}
// a grid covering the largest of the items' windows (rows: their row windows)
template <class F>
static dim3 grid_items(const std::vector<SetupItem> &v, F grid) {
    unsigned gx = 1, gy = 1;
    for (const SetupItem &x : v) {
        const dim3 d = grid(x);
        gx = std::max(gx, d.x);
        gy = std::max(gy, d.y);
    }
    return dim3(gx, gy, (unsigned)v.size());
}
static int list_blocks(size_t n) { return std::max(16, kListBlocks / (int)std::max<size_t>(1, n)); }

// A batched rebuild between its halves.
struct LsBatchPending {
    std::vector<Win> wn;
    std::vector<char> whole;
    std::vector<SetupItem> su;
    std::vector<size_t> who;
    BatchIter<FimItem> it;
    EikGeom eg;
    bool live = false;
};
void ls_batch_pending_free(LsBatchPending *p) { delete p; }

int ls_pin_rebuild_batch_begin(hipStream_t s, const Grid &g, const std::vector<LsJob> &jobs, LsBatch &bt,
                               bool pin_new, LsBatchPending **out) {
    *out = nullptr;
    const size_t n = jobs.size();
    if (n > (size_t)bt.cap) return 7;
    LsBatchPending *p = new LsBatchPending;
    *out = p;
    p->wn.resize(n);
    p->whole.resize(n);
    std::vector<FimItem> items;
    std::vector<int *> pred;
    for (size_t k = 0; k < n; k++) {
        LsWork &w = *jobs[k].w;
        w.pin_first = true;
        Win wr;
        int R;
        bool wh;
        const bool lv = rebuild_window(g, *jobs[k].c, w, p->wn[k], wr, wh, R);
        p->whole[k] = wh;
        if (!lv) continue;
        const ObjArrays &a = *jobs[k].a;
        p->su.push_back(SetupItem{*jobs[k].c, a, w, p->wn[k], wr, R, 1, pin_new ? a.nX : nullptr,
                                  pin_new ? a.nY : nullptr, nullptr});
        items.push_back(FimItem{*jobs[k].c, a, w, {w.va, w.vb}});
        pred.push_back(&w.pred_fim);
        p->who.push_back(k);
    }
    if (items.empty()) return 0;
    p->live = true;
    // the set-up of every live solid (the single-solid rebuild_setup's
    // launches, one per kernel for all of them)
    int rc = 0;
    const SetupItem *d = upload_items(s, bt, 0, p->su, &rc);
    if (rc) return rc;
    const dim3 bb(BX, BY), gw = grid_items(p->su, [](const SetupItem &x) { return grid_win(x.wn); }),
               gs = grid_items(p->su, [](const SetupItem &x) { return grid_rows(x.wn); }),
               gr = grid_items(p->su, [](const SetupItem &x) { return grid_rows(x.wr); }),
               gc = grid_items(p->su, [](const SetupItem &x) { return grid_win_cols(x.wn); });
    const unsigned m = (unsigned)p->su.size();
    k_pin_b<<<gw, bb, 0, s>>>(g, d);
    KCHECK();
    k_counts_b<<<dim3(1, 1, m), 64, 0, s>>>(d, kCntIter + kIterSlots);
    KCHECK();
    k_scan_b<<<gs, bb, 0, s>>>(g, d);
    KCHECK();
    k_newton_b<<<dim3(list_blocks(m), 1, m), kNewtonThreads, 0, s>>>(g, geom_of(g), d);
    KCHECK();
    k_dilate_rows_b<<<gr, bb, 0, s>>>(g, d);
    KCHECK();
    k_dilate_cols_b<<<gc, bb, 0, s>>>(g, d);
    KCHECK();
    k_compact_tiles_b<<<dim3(64, 1, m), 256, 0, s>>>(d, 0);
    KCHECK();
    // the predicted batch of march passes, its counters read back later
    p->eg.init(g.dx, g.dy);
    p->it.start(std::move(items), std::move(pred));
    const int nb = batch_blocks((int)p->it.items.size());
    const EikGeom eg = p->eg;
    return batch_enqueue(s, bt, p->it, [&](int q, int slot, const FimItem *dd, int mm) -> int {
        k_fim_tiles_batch<<<dim3(nb, mm), kTileThreads, 0, s>>>(g, eg, dd, q, slot, 64);
        KCHECK();
        return 0;
    });
}

int ls_pin_rebuild_batch_end(hipStream_t s, const Grid &g, const std::vector<LsJob> &jobs, LsBatch &bt,
                             LsBatchPending *p, int *fim_iters) {
    if (!p->live) {
        delete p;
        return 0;
    }
    const int nb = batch_blocks((int)p->it.items.size());
    const EikGeom eg = p->eg;
    int rc = batch_finish(s, bt, p->it, kMaxFimPasses, [&](int q, int slot, const FimItem *dd, int mm) -> int {
        k_fim_tiles_batch<<<dim3(nb, mm), kTileThreads, 0, s>>>(g, eg, dd, q, slot, 64);
        KCHECK();
        return 0;
    }, true);
    if (!rc) rc = [&]() -> int {
        int most = 0;
        for (size_t t = 0; t < p->who.size(); t++) {
            LsWork &w = *jobs[p->who[t]].w;
            if (w.hcnt[kCntErr] & kErrNewton) return 3;
            most = std::max(most, p->it.passes_out[t]);
            p->su[t].v = p->it.passes_out[t] & 1 ? w.vb : w.va;
        }
        // the finish of every live solid (rebuild_finish's launches, shared)
        int e = 0;
        const SetupItem *d = upload_items(s, bt, 1, p->su, &e);
        if (e) return e;
        const dim3 bb(BX, BY), gw = grid_items(p->su, [](const SetupItem &x) { return grid_win(x.wn); }),
                   gs = grid_items(p->su, [](const SetupItem &x) { return grid_rows(x.wn); });
        const unsigned m = (unsigned)p->su.size();
        k_finalize_b<<<gs, bb, 0, s>>>(g, d);
        KCHECK();
        k_compact_tiles_b<<<dim3(64, 1, m), 256, 0, s>>>(d, 1);
        KCHECK();
        k_commit_status_b<<<gw, bb, 0, s>>>(g, d);
        KCHECK();
        for (size_t t = 0; t < p->who.size(); t++)
            if ((e = finish_window(s, *jobs[p->who[t]].w, p->wn[p->who[t]], p->whole[p->who[t]]))) return e;
        if (fim_iters) *fim_iters = most;
        return 0;
    }();
    delete p;
    return rc;
}

int ls_pin_rebuild_batch(hipStream_t s, const Grid &g, const std::vector<LsJob> &jobs, LsBatch &bt,
                         int *fim_iters) {
    LsBatchPending *p = nullptr;
    if (int rc = ls_pin_rebuild_batch_begin(s, g, jobs, bt, false, &p)) {
        if (p) (void)hipStreamSynchronize(s);
        delete p;
        return rc;
    }
    return ls_pin_rebuild_batch_end(s, g, jobs, bt, p, fim_iters);
}

int ls_rebuild(hipStream_t s, const Grid &g, const ObjConst &c, const ObjArrays &a, LsWork &w, int *fim_iters) {
    ls_reset_window(w);  // a new field: the whole grid
    w.pin_first = false;
    return rebuild_common(s, g, c, a, w, fim_iters);
}

int ls_pin_rebuild(hipStream_t s, const Grid &g, const ObjConst &c, const ObjArrays &a, LsWork &w,
                   int *fim_iters) {
    w.pin_first = true;
    return rebuild_common(s, g, c, a, w, fim_iters);
}

int ls_pin_rebuild_begin(hipStream_t s, const Grid &g, const ObjConst &c, const ObjArrays &a, LsWork &w,
                         const double *pin_x, const double *pin_y, LsRebuild &r) {
    w.pin_first = true;
    r = LsRebuild{};
    if (int rc = rebuild_setup(s, g, c, a, w, r.wn, r.whole, &r.live, pin_x, pin_y)) return rc;
    if (!r.live) return 0;
    r.eg.init(g.dx, g.dy);
    return iter_enqueue(s, w, w.pred_fim, 0,
                        [&](int p, int slot) { return fim_pass(s, g, r.eg, c, a, w, p, slot); }, r.batch, 2, true);
}

int ls_pin_rebuild_end(hipStream_t s, const Grid &g, const ObjConst &c, const ObjArrays &a, LsWork &w, LsRebuild &r,
                       int *fim_iters) {
    if (!r.live) return 0;
    HIP_CHECK(hipStreamSynchronize(s));
    int passes = 0;
    // the rest of iterate from the batch begin enqueued
    bool done = iter_done(w, w.pred_fim, r.passes, r.batch, &passes);
    while (!done && r.passes < kMaxFimPasses) {
        if (int rc = iter_enqueue(s, w, w.pred_fim, r.passes,
                                  [&](int p, int slot) { return fim_pass(s, g, r.eg, c, a, w, p, slot); }, r.batch))
            return rc;
        HIP_CHECK(hipStreamSynchronize(s));
        done = iter_done(w, w.pred_fim, r.passes, r.batch, &passes);
    }
    if (!done) return 7;
    if (w.hcnt[kCntErr] & kErrNewton) return 3;
    if (fim_iters) *fim_iters = passes;
    return rebuild_finish(s, g, c, a, w, r.wn, r.whole, passes);
}

void ls_reset_window(LsWork &w) {
    if (w.bbox_pending) (void)hipEventSynchronize(w.ev_bbox);
    w.bbox_pending = false;
    w.have_win = false;
}

// Workgroups per solid of an extension. A lone solid gets as many as run on the
// GPU at once (three of these workgroups fit a CU): every one holds its tiles
// from the start, none waits for one that has not been dispatched (with 1024
// a band 60 cells wide, 917 tiles, takes 2 to 8 ms in up to 10 launches, now 1.6).
// Of several solids the first ones' workgroups are dispatched first, so a
// solid whose tiles are all held is always among them.
constexpr int kExtBlocks = 768, kExtBlocksBatch = 1024;
static int ext_blocks_batch(size_t n) { return std::max(128, kExtBlocksBatch / std::max(1, (int)(n + 3) / 4)); }
constexpr int kMaxExtPasses = 4096;

int ls_extend(hipStream_t s, const Grid &g, const ObjArrays &a, LsWork &w, int *ext_iters) {
    const int nb = kExtBlocks;
    k_ext_open<<<nb, kTileThreads, 0, s>>>(g, a, w);
    KCHECK();
    int passes = 0;
    int rc = iterate(s, w, w.pred_ext, kMaxExtPasses, [&](int p, int slot) -> int {
        k_extend_tiles<<<nb, kExtThreads, 0, s>>>(g, a, w, p, slot);
        KCHECK();
        return 0;
    }, &passes, 1);
    if (rc) return rc;
    if (w.hcnt[kCntErr] & kErrSingular) return 5;
    if (ext_iters) *ext_iters = passes;
    return 0;
}

int ls_extend_batch(hipStream_t s, const Grid &g, const std::vector<LsJob> &jobs, LsBatch &bt, int *ext_iters) {
    const size_t n = jobs.size();
    if (n > (size_t)bt.cap) return 7;
    if (!n) return 0;
    std::vector<ExtItem> items;
    std::vector<int *> pred;
    for (size_t k = 0; k < n; k++) {
        items.push_back(ExtItem{*jobs[k].a, *jobs[k].w});
        pred.push_back(&jobs[k].w->pred_ext);
    }
    const int nb = ext_blocks_batch(n);
    std::vector<int> passes;
    const int rc = iterate_batch(s, bt, items, pred, kMaxExtPasses, [&](int p, int slot, const ExtItem *dd, int m) -> int {
        if (p == 0) {
            k_ext_open_b<<<dim3(nb, m), kTileThreads, 0, s>>>(g, dd);
            KCHECK();
        }
        k_extend_tiles_batch<<<dim3(nb, m), kExtThreads, 0, s>>>(g, dd, p, slot);
        KCHECK();
        return 0;
    }, passes, 1);
    if (rc) return rc;
    int most = 0;
    for (size_t k = 0; k < n; k++) {
        if (jobs[k].w->hcnt[kCntErr] & kErrSingular) return 5;
        most = std::max(most, passes[k]);
    }
    if (ext_iters) *ext_iters = most;
    return 0;
}

}  // namespace incrmt
