// pb_kernels.hip -- Poisson-Boltzmann boundary from ion radii.
//
// Maps (library/src/grid_general.c:138-301).  With the smooth step
//   H(s) = -(1/(4 w^3)) s^3 + (3/(4 w^2)) s^2,  s = |x - x_ion| - r + w,
// each ion multiplies the solvent fraction of the points and faces of its box
// (+-(floor((r+w)/h)+1) points around its cell) by 0 inside r - w and by H in
// the shell up to r + w; eps_x/y/z = eps_int + (eps_s - eps_int) * product on
// the +x/+y/+z face of each point, k2 = kbar2 * product on the point.  The
// reference scatters ion by ion; here each point gathers: a work-group owns an
// 8^3 tile, collects the ions that can reach it from the bins around it, sorts
// them by ion id in LDS and applies their factors in that order, so every
// product is formed in the reference's order.
//
// Forces (library/src/particles.c:420-775).  One work-group per ion walks the
// ion's box (+-(floor((r+w)/h)+2) points) and sums the ionic-boundary term at
// the shell points and the dielectric-boundary and non-polar terms at the
// shell faces; the sums are reduced in a fixed tree (deterministic, ordered
// differently from the reference's serial loop).
#include "pb.hpp"

namespace maze {

namespace {

struct StepCoef {
    double c3, c2;   // H(s) = c3 s^3 + c2 s^2
    double d2, d1;   // H'(s) = d2 s^2 + d1 s
};

inline StepCoef step_coef(double w) {
    const double w2 = w * w, w3 = w2 * w;
    return {-(1 / (4 * w3)), 3 / (4 * w2), -(3 / (4 * w3)), 3 / (2 * w2)};
}

__device__ __forceinline__ double step_h(const StepCoef& c, double s) {
    return c.c3 * cube(s) + c.c2 * (s * s);
}

// H'(s) / H(s) (library/src/particles.c:407-417).
__device__ __forceinline__ double step_dlog(const StepCoef& c, double s) {
    return (c.d2 * (s * s) + c.d1 * s) / (c.c3 * cube(s) + c.c2 * (s * s));
}

__device__ __forceinline__ int cell_of(double x, double h) { return (int)floor(x / h); }

__device__ __forceinline__ int wrap1(int i, int n) {
    return i < 0 ? i + n : (i >= n ? i - n : i);
}

// i mod n in [0, n) for any i (cells of positions outside the box included).
__device__ __forceinline__ int pmod(int i, int n) {
    const int r = i % n;
    return r < 0 ? r + n : r;
}

}  // namespace

// ---- binning ---------------------------------------------------------------------
// A list of ions per 8^3 bin, in no order (the maps sort the few ions that reach a
// tile).  Clearing and linking take 5 us at 8000 ions and 20^3 bins, against 60 us
// for a radix sort of the ions by bin.
__global__ void k_pb_clear(int bins, int* __restrict__ head) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < bins) head[i] = -1;
}

__global__ void k_pb_bin(int np, int n, double h, int nb, const double* __restrict__ pos,
                         int* __restrict__ head, int* __restrict__ next) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    int b[3];
    for (int a = 0; a < 3; a++) {
        b[a] = pmod(cell_of(pos[3 * i + a], h), n) / kPbTile;
    }
    next[i] = atomicExch(&head[(b[0] * nb + b[1]) * nb + b[2]], i);
}

void launch_pb_bin(hipStream_t s, PBDev& b, const double* pos) {
    if (b.np == 0) return;
    const int bins = b.nb * b.nb * b.nb;
    MAZE_LAUNCH(k_pb_clear, dim3((bins + kBlock - 1) / kBlock), dim3(kBlock), 0, s, bins, b.head);
    MAZE_LAUNCH(k_pb_bin, dim3((b.np + kBlock - 1) / kBlock), dim3(kBlock), 0, s, b.np, b.n, b.h,
                b.nb, pos, b.head, b.next);
}

// ---- maps --------------------------------------------------------------------------
// Bins along one axis whose ions can reach the tile's points [t0, t0 + kPbTile):
// those holding cells in [t0 - R, t0 + kPbTile - 1 + R] (periodic).
struct AxisBins {
    int first, count;
};

__device__ __forceinline__ AxisBins axis_bins(int t0, int R, int n, int nb) {
    const int len = kPbTile + 2 * R;
    if (len + kPbTile > n) return {0, nb};
    int v0 = (t0 - R) % n;
    if (v0 < 0) v0 += n;
    const int v1 = (v0 + len - 1) % n;
    const int b0 = v0 / kPbTile, b1 = v1 / kPbTile;
    return {b0, (b1 - b0 + nb) % nb + 1};
}

// Offset d = g - c (mod n) of grid index g from an ion's cell c, as the one
// value in [-R, R] (the ion's box), or a value beyond R when g is outside it.
__device__ __forceinline__ int box_offset(int g, int c, int n, int R) {
    int d = g - c;
    if (d < 0) d += n;
    else if (d >= n) d -= n;
    if (d > R) d = (d >= n - R) ? d - n : R + 1;
    return d;
}

// Whether an ion whose points lie within R of cell c (at f = its distance from the
// cell's point) comes within `dist` of the tile's points [t0, t0 + len) along one
// axis, faces included.
__device__ __forceinline__ bool axis_reach(int t0, int len, int c, int n, int R, double f,
                                           double h, double& dist) {
    int o = t0 - c;
    if (o < 0) o += n;
    else if (o >= n) o -= n;
    dist = 1e300;
#pragma unroll
    for (int u = 0; u < 2; u++, o -= n) {  // offsets o + [0, len) and one period below
        const int lo = max(o, -R), hi = min(o + len - 1, R);
        if (lo <= hi) dist = fmin(dist, fmax(fmax(lo * h - f, f - hi * h) - h / 2.0, 0.0));
    }
    return dist < 1e300;
}

// Which of a point's coefficients give boundary forces: bit 0 k2, bits 1 to 3 the
// +x, +y, +z faces.  The forces look at all points of all shells: their marks (a byte
// each, 4 MB at 160^3) stay in the L2 caches, which the maps (131 MB) do not.
__device__ __forceinline__ unsigned char pb_mark(double ex, double ey, double ez, double k2,
                                                 double eps_int) {
    return (k2 != 0.0 ? 1 : 0) | (ex != eps_int ? 2 : 0) | (ey != eps_int ? 4 : 0) |
           (ez != eps_int ? 8 : 0);
}

struct PBMapArgs {
    int n, nb, rmax, np;
    double h, w, eps_s, eps_int, kbar2;
    StepCoef c;
    const double* pos;
    const double* radii;
    const double* rp2;
    const double* rm2;
    const int* rmap;
    const int* head;
    const int* next;
    double *ex, *ey, *ez, *k2;
    unsigned char* mark;
    int* flag;
};

// One ion that can reach the tile.  An entry is inside it if not beyond `core`.
struct alignas(16) PBReach {
    double p[3], r, rp2, core;
    int cell[3], R;
    int g0[3];  // the tile's first point, as the image nearest the ion
    int split;  // two images are in the box: g0 does not tell
};

// One work-group per 8^3 tile; wave v owns planes i = 2 v and 2 v + 1 of the tile,
// a thread points (i, j, k) and (i + 1, j, k) with k = t % 8, j = t / 8 % 8.
//
// The reference's mask of an array entry: unchanged beyond r + w of an ion, times
// H in the shell, 0 inside r - w, ion after ion.  The zeros need no order, so a
// first pass over the ions whose core reaches the wave's planes finds the
// entries inside any of them; only what is left gets the shell factors, in the
// order of the ions.  Bounded by the FP64 distances (30 operations per ion and
// pair of points): in an 8000-ion melt on 160^3, where 0.4 % of the entries are
// not 0, 163 us (beside the pair kernel 280) where one ordered
// pass with the factors of all took 372 (417).
static_assert(kPbTile == 8 && kBlock == 256, "tile-to-thread map assumes 8^3 tiles, 256 threads");
__global__ __launch_bounds__(kBlock) void k_pb_maps(PBMapArgs a) {
    __shared__ int list[kPbCap];
    __shared__ PBReach ions[kPbChunk];
    __shared__ int s_total, s_kept;
    const int nb = a.nb, n = a.n, t = threadIdx.x;
    const int b = blockIdx.x;
    const int tb[3] = {b / (nb * nb), (b / nb) % nb, b % nb};
    const double h = a.h, hd2 = h / 2.0, w = a.w;
    AxisBins ab[3];
    for (int d = 0; d < 3; d++) ab[d] = axis_bins(tb[d] * kPbTile, a.rmax, n, nb);
    // Rows of bins, in two parts where the z range wraps.
    const int rows = ab[0].count * ab[1].count * (ab[2].first + ab[2].count > nb ? 2 : 1);
    if (rows > kPbMaxSeg) {
        if (t == 0) a.flag[0] = 1;
        return;
    }
    if (t == 0) s_total = s_kept = 0;
    __syncthreads();
    // The ions of the bins around whose sphere r + w can reach a point or face of
    // the tile.
    const int bins = a.np > 0 ? ab[0].count * ab[1].count * ab[2].count : 0;
    for (int q = t; q < bins; q += kBlock) {
        const int qz = q % ab[2].count, qxy = q / ab[2].count;
        int bin[3] = {ab[0].first + qxy / ab[1].count, ab[1].first + qxy % ab[1].count,
                      ab[2].first + qz};
        for (int d = 0; d < 3; d++) bin[d] = bin[d] >= nb ? bin[d] - nb : bin[d];
        int found = 0;
        for (int id = a.head[(bin[0] * nb + bin[1]) * nb + bin[2]]; id >= 0; id = a.next[id]) {
            found++;
            bool keep = true;
            double d2 = 0.0;
            const int R = a.rmap[id];
            for (int d = 0; d < 3; d++) {
                const double x = a.pos[3 * id + d];
                const int c = cell_of(x, h), t0 = tb[d] * kPbTile;
                double dist;
                keep = axis_reach(t0, min(kPbTile, n - t0), c, n, R, x - c * h, h, dist) && keep;
                d2 += dist * dist;
            }
            if (keep && d2 < a.rp2[id] * (1.0 + 1e-9) + 1e-300) {
                const int slot = atomicAdd(&s_kept, 1);
                if (slot < kPbCap) list[slot] = id;
            }
        }
        if (found) atomicAdd(&s_total, found);
    }
    __syncthreads();
    if (s_total > kPbCap) {
        if (t == 0) a.flag[0] = 1;
        return;
    }
    // Ascending ids, by rank.
    const int kept = s_kept;
    int id[kPbCap / kBlock], rank[kPbCap / kBlock];
#pragma unroll
    for (int u = 0; u < kPbCap / kBlock; u++) {
        if (u * kBlock >= kept) break;
        id[u] = t + u * kBlock < kept ? list[t + u * kBlock] : 0;
        rank[u] = 0;
        for (int q = 0; q < kept; q++) rank[u] += list[q] < id[u];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPbCap / kBlock; u++)
        if (t + u * kBlock < kept) list[rank[u]] = id[u];
    auto stage = [&](int c0) {
        __syncthreads();
        if (t < kPbChunk && c0 + t < kept) {
            const int i = list[c0 + t];
            PBReach v;
            v.split = 0;
            v.R = a.rmap[i];
            for (int d = 0; d < 3; d++) {
                const int t0 = tb[d] * kPbTile, len = min(kPbTile, n - t0);
                v.p[d] = a.pos[3 * i + d];
                v.cell[d] = cell_of(v.p[d], h);
                int o = t0 - v.cell[d];
                if (o < 0) o += n;
                else if (o >= n) o -= n;
                const bool above = o <= v.R, below = o - n + len - 1 >= -v.R;
                if (above && below) v.split = 1;
                v.g0[d] = v.cell[d] + (above ? o : o - n);
            }
            v.r = a.radii[i];
            v.rp2 = a.rp2[i];
            // r2 < rp2 and r2 <= rm2, as one bound.
            const double rm2 = a.rm2[i];
            v.core = rm2 < v.rp2 ? rm2
                     : v.rp2 > 0.0 ? __longlong_as_double(__double_as_longlong(v.rp2) - 1) : -1.0;
            ions[t] = v;
        }
        __syncthreads();
    };

    const int lane = t & (kWave - 1), wave = t / kWave;
    const int tk = t & 7, tj = (t >> 3) & 7, ti = 2 * wave;
    const int gk = tb[2] * kPbTile + tk, gj = tb[1] * kPbTile + tj, gi = tb[0] * kPbTile + ti;
    const bool ok0 = gj < n && gk < n && gi < n, ok1 = ok0 && gi + 1 < n;
    // The staged ions from c0 on whose sphere of squared radius rp2 (core) can reach the
    // wave's points and faces, 64 at a time, as a mask.
    auto reaching = [&](int c0, int q0, bool core) {
        bool hit = false;
        if (c0 + q0 + lane < kept && q0 + lane < kPbChunk && gi < n) {
            const PBReach& v = ions[q0 + lane];
            double d2 = 0.0;
            hit = true;
            for (int d = 0; d < 3; d++) {
                const int t0 = d == 0 ? gi : tb[d] * kPbTile;
                double dist;
                hit = axis_reach(t0, min(d == 0 ? 2 : kPbTile, n - t0), v.cell[d], n, v.R,
                                 v.p[d] - v.cell[d] * h, h, dist) && hit;
                d2 += dist * dist;
            }
            hit = hit && d2 < (core ? v.core : v.rp2) * (1.0 + 1e-9) + 1e-300;
        }
        return __ballot(hit);
    };
    // Squared distances of the two points and their +x, +y, +z faces from an ion, and
    // whether the points are in its box.
    const double x0 = gi * h, x1 = (gi + 1) * h, y0 = gj * h, z0 = gk * h;
    auto distances = [&](const PBReach& v, double (&r2)[2][4], bool (&in)[2]) {
        int oi, oi1, oj, ok;
        double X0 = x0, X1 = x1, Y = y0, Z = z0;
        if (!v.split) {
            const int mi = v.g0[0] + ti, mj = v.g0[1] + tj, mk = v.g0[2] + tk;
            oi = mi - v.cell[0];
            oi1 = oi + 1;
            oj = mj - v.cell[1];
            ok = mk - v.cell[2];
            if (v.g0[0] != tb[0] * kPbTile) {
                X0 = mi * h;
                X1 = (mi + 1) * h;
            }
            if (v.g0[1] != tb[1] * kPbTile) Y = mj * h;
            if (v.g0[2] != tb[2] * kPbTile) Z = mk * h;
        } else {
            oi = box_offset(gi, v.cell[0], n, v.R);
            oi1 = box_offset(gi + 1, v.cell[0], n, v.R);
            oj = box_offset(gj, v.cell[1], n, v.R);
            ok = box_offset(gk, v.cell[2], n, v.R);
            X0 = (v.cell[0] + oi) * h;
            X1 = (v.cell[0] + oi1) * h;
            Y = (v.cell[1] + oj) * h;
            Z = (v.cell[2] + ok) * h;
        }
        const unsigned int R = v.R, D = 2 * R;
        const bool jk = oj + R <= D && ok + R <= D;
        in[0] = jk && oi + R <= D;
        in[1] = jk && oi1 + R <= D;
        const double dy = v.p[1] - Y, dy2 = dy * dy, ty = dy - hd2, ty2 = ty * ty;
        const double dz = v.p[2] - Z, dz2 = dz * dz, tz = dz - hd2, tz2 = tz * tz;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const double dx = v.p[0] - (u == 0 ? X0 : X1), dx2 = dx * dx;
            const double tx = dx - hd2;
            r2[u][0] = dx2 + dy2 + dz2;
            r2[u][1] = tx * tx + dy2 + dz2;
            r2[u][2] = dx2 + ty2 + dz2;
            r2[u][3] = dx2 + dy2 + tz2;
        }
    };
    // Entries that are 0: inside an ion, or no entries at all.
    bool zero[2][4];
#pragma unroll
    for (int e = 0; e < 8; e++) zero[e / 4][e % 4] = !(e / 4 == 0 ? ok0 : ok1);
    auto finished = [&]() {
        bool all = true;
#pragma unroll
        for (int e = 0; e < 8; e++) all = all && zero[e / 4][e % 4];
        return __all(all);
    };
    for (int c0 = 0; c0 < kept; c0 += kPbChunk) {
        stage(c0);
        for (int q0 = 0; q0 < kPbChunk; q0 += kWave) {
            for (unsigned long long m = reaching(c0, q0, true); m && !finished(); m &= m - 1) {
                const PBReach& v = ions[q0 + __builtin_ctzll(m)];
                double r2[2][4];
                bool in[2];
                distances(v, r2, in);
#pragma unroll
                for (int e = 0; e < 8; e++)
                    zero[e / 4][e % 4] |= in[e / 4] & !(r2[e / 4][e % 4] > v.core);
            }
        }
    }
    const double e0 = a.eps_s - a.eps_int;
    double f[2][4];
#pragma unroll
    for (int e = 0; e < 8; e++)
        f[e / 4][e % 4] = zero[e / 4][e % 4] ? 0.0 : e % 4 == 0 ? a.kbar2 : e0;
    for (int c0 = 0; c0 < kept; c0 += kPbChunk) {
        if (kept > kPbChunk) stage(c0);
        if (finished()) continue;
        for (int q0 = 0; q0 < kPbChunk; q0 += kWave) {
            for (unsigned long long m = reaching(c0, q0, false); m; m &= m - 1) {
                const PBReach& v = ions[q0 + __builtin_ctzll(m)];
                double r2[2][4];
                bool in[2];
                distances(v, r2, in);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const double d2 = r2[e / 4][e % 4];
                    if (in[e / 4] && !zero[e / 4][e % 4] && !(d2 >= v.rp2))
                        f[e / 4][e % 4] *= step_h(a.c, sqrt(d2) - v.r + w);
                }
            }
        }
    }
    const long n2 = (long)n * n;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        if (!(u == 0 ? ok0 : ok1)) continue;
        const long idx = (gi + u) * n2 + (long)gj * n + gk;
        const double k2 = f[u][0], ex = f[u][1] + a.eps_int;
        const double ey = f[u][2] + a.eps_int, ez = f[u][3] + a.eps_int;
        a.k2[idx] = k2;
        a.ex[idx] = ex;
        a.ey[idx] = ey;
        a.ez[idx] = ez;
        a.mark[idx] = pb_mark(ex, ey, ez, k2, a.eps_int);
    }
}

// The marks of given maps.
__global__ __launch_bounds__(kBlock) void k_pb_mark(long G, double eps_int,
                                                    const double* __restrict__ ex,
                                                    const double* __restrict__ ey,
                                                    const double* __restrict__ ez,
                                                    const double* __restrict__ k2,
                                                    unsigned char* __restrict__ mark) {
    const long c = (long)blockIdx.x * kBlock + threadIdx.x;
    if (c < G) mark[c] = pb_mark(ex[c], ey[c], ez[c], k2[c], eps_int);
}

void launch_pb_maps(hipStream_t s, PBDev& b, const double* pos, double* ex, double* ey,
                    double* ez, double* k2) {
    PBMapArgs a{};
    a.n = b.n; a.nb = b.nb; a.rmax = b.rmax; a.np = b.np;
    a.h = b.h; a.w = b.w; a.eps_s = b.eps_s; a.eps_int = b.eps_int; a.kbar2 = b.kbar2;
    a.c = step_coef(b.w);
    a.pos = pos; a.radii = b.radii; a.rp2 = b.rp2; a.rm2 = b.rm2; a.rmap = b.rmap;
    a.head = b.head; a.next = b.next;
    a.ex = ex; a.ey = ey; a.ez = ez; a.k2 = k2; a.mark = b.mark;
    a.flag = b.flag;
    b.marked = 1;
    MAZE_LAUNCH(k_pb_maps, dim3(b.nb * b.nb * b.nb), dim3(kBlock), 0, s, a);
}

// ---- forces ------------------------------------------------------------------------
struct PBForceArgs {
    int n, nonpolar;
    double h, w, eps_int, sdb, snp;
    StepCoef c;
    const double* pos;
    const double* radii;
    const double* rp2;
    const double* rm2;
    const int* rfrc;
    const double *phi, *ex, *ey, *ez, *k2;
    const unsigned long long* any;
    int words;  // of any, per row
    double *fdb, *fib, *fnp;
};

__device__ __forceinline__ bool in_shell(double r2, double rp2, double rm2) {
    return r2 < rp2 && r2 > rm2;
}

// One face term (library/src/particles.c:585-764): the face at (fx, fy, fz)
// from the ion, eps_f its dielectric, dphi the potential step across it, g the
// normalised dielectric gradient component; sgn -1 below the point, +1 above.
__device__ __forceinline__ void face_term(double fx, double fy, double fz, double r2, double r,
                                          double w, const StepCoef& c, double eps_f,
                                          double eps_int, double dphi, double phic, double g,
                                          int sgn, int nonpolar, double* acc) {
    const double r1 = sqrt(r2) + 1E-12;
    const double ux = fx / r1, uy = fy / r1, uz = fz / r1;
    const double k = (eps_f - eps_int) * step_dlog(c, r1 - r + w);
    acc[0] -= k * dphi * phic * ux;
    acc[1] -= k * dphi * phic * uy;
    acc[2] -= k * dphi * phic * uz;
    if (nonpolar) {
        const double s = sgn < 0 ? -1.0 : 1.0;
        acc[6] += s * (k * g * ux);
        acc[7] += s * (k * g * uy);
        acc[8] += s * (k * g * uz);
    }
}

// A bit per point whether it or one of its faces is marked, rows in 64-bit words.
__global__ __launch_bounds__(kBlock) void k_pb_any(int n, int words,
                                                   const unsigned char* __restrict__ mark,
                                                   unsigned long long* __restrict__ any) {
    const long w = ((long)blockIdx.x * kBlock + threadIdx.x) / kWave;
    const int n2 = n * n;
    const long row = w / words;
    if (row >= n2) return;
    const int k = (int)(w - row * words) * kWave + (threadIdx.x & (kWave - 1));
    bool hit = false;
    if (k < n) {
        const int i = (int)row / n, j = (int)row - i * n;
        const long c = row * n + k;
        hit = mark[c] | (mark[c + (i == 0 ? (long)n2 * (n - 1) : -n2)] & 2) |
              (mark[c + (j == 0 ? n2 - n : -n)] & 4) | (mark[c + (k == 0 ? n - 1 : -1)] & 8);
    }
    const unsigned long long m = __ballot(hit);
    if ((threadIdx.x & (kWave - 1)) == 0) any[w] = m;
}

// (128 registers at most: 4 waves per SIMD hide more of the listed points' loads than the
// spill of a few costs; 3 waves 217 us, 5 waves with 48 spilled 265.)
__global__ __launch_bounds__(kBlock, 4) void k_pb_forces(PBForceArgs a) {
    __shared__ double sh[kBlock / kWave];
    const int ion = blockIdx.x;
    const int n = a.n;
    const long n2 = (long)n * n;
    const double h = a.h, hd2 = h / 2.0, w = a.w;
    const double px = a.pos[3 * ion], py = a.pos[3 * ion + 1], pz = a.pos[3 * ion + 2];
    const double r = a.radii[ion], rp2 = a.rp2[ion], rm2 = a.rm2[ion];
    const int R = a.rfrc[ion], S = 2 * R + 1;
    const int cx = cell_of(px, h), cy = cell_of(py, h), cz = cell_of(pz, h);
    double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // db xyz, ib xyz, np xyz
    // Only points whose centre lies within h/2 of the shell (rm2, rp2) can have a
    // shell point or face: per box row (qi, qj) the k ranges of centre distances in
    // (sqrt(rm2) - h/2, sqrt(rp2) + h/2), widened by a point on each side, are listed
    // (up to two per row) and their points spread over the threads.  In a dense system
    // nearly all of their coefficients vanish, so a row takes a bit per point (k_pb_any),
    // and only points with any get their distances: at 8000 ions on 160^3 187 us for
    // 24 million points, against 546 with the distances of all.
    __shared__ int e_off[2 * kBlock + 1], e_k[2 * kBlock];
    __shared__ int2 e_row[2 * kBlock];
    __shared__ unsigned long long bits[kBlock];
    __shared__ unsigned long long w_tot[kBlock / kWave];
    const double band_hi = (sqrt(rp2) + hd2) * (1.0 + 1e-12);
    double band_lo = (sqrt(rm2) - hd2) * (1.0 - 1e-12);
    band_lo = band_lo > 0.0 ? band_lo : 0.0;
    const double hi2 = band_hi * band_hi, lo2 = band_lo * band_lo;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int gx0 = pmod(cx, n), gy0 = pmod(cy, n), gz0 = pmod(cz, n);
    const int rows = S * S;
    for (int row0 = 0; row0 < rows; row0 += kBlock) {
        int st[2] = {0, 0}, cnt[2] = {0, 0};
        const int row = row0 + threadIdx.x;
        const int qi = row / S, qj = row - qi * S;
        if (row < rows) {
            const double dx = px - (cx + qi - R) * h, dy = py - (cy + qj - R) * h;
            const double rho2 = dx * dx + dy * dy;
            if (rho2 < hi2) {
                const double b = sqrt(hi2 - rho2);
                const double c = rho2 < lo2 ? sqrt(lo2 - rho2) : 0.0;
                // dz = pz - (cz + qk - R) h in [c, b] or [-b, -c].
                const double base = pz / h - cz + R;
                int a0 = (int)floor(base - b / h) - 1, a1 = (int)ceil(base - c / h) + 1;
                int b0 = (int)floor(base + c / h) - 1, b1 = (int)ceil(base + b / h) + 1;
                a0 = max(a0, 0); a1 = min(a1, S - 1);
                b0 = max(b0, 0); b1 = min(b1, S - 1);
                if (a1 >= b0 - 1) {  // the two ranges touch: one range
                    a1 = max(a1, b1);
                    b0 = 1; b1 = 0;
                }
                if (a1 >= a0) { st[0] = a0; cnt[0] = a1 - a0 + 1; }
                if (b1 >= b0) { st[1] = b0; cnt[1] = b1 - b0 + 1; }
            }
        }
        // Exclusive scan of the points (low word) and the ranges that hold any.
        auto entry = [](int c) { return c > 0 ? (1ull << 32) + (unsigned int)c : 0ull; };
        const unsigned long long mine = entry(cnt[0]) + entry(cnt[1]);
        unsigned long long incl = mine;
        for (int o = 1; o < kWave; o <<= 1) {
            const unsigned long long v = __shfl_up(incl, o);
            if (lane >= o) incl += v;
        }
        if (lane == kWave - 1) w_tot[wave] = incl;
        __syncthreads();
        unsigned long long before = incl - mine, all = 0;
        for (int q = 0; q < kBlock / kWave; q++) {
            if (q < wave) before += w_tot[q];
            all += w_tot[q];
        }
        const int total = (int)(all & 0xffffffffull), ranges = (int)(all >> 32);
        int off[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            off[u] = (int)(before & 0xffffffffull);
            if (cnt[u] > 0) {
                const int e = (int)(before >> 32);
                e_off[e] = off[u];
                e_k[e] = st[u];
                e_row[e] = make_int2(qi, qj);
            }
            before += entry(cnt[u]);
        }
        if (threadIdx.x == 0) e_off[ranges] = total;
        __syncthreads();
        // The points of up to 64 rounds (of one per thread) that may give a term, as bits.
        for (int base = 0; base < total; base += kWave * kBlock) {
            if (base > 0) __syncthreads();
            bits[threadIdx.x] = 0;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const unsigned long long* any = a.any;
                if (cnt[u] > 0)
                    any += ((long)wrap1(gx0 + qi - R, n) * n + wrap1(gy0 + qj - R, n)) * a.words;
                for (int pos = 0; pos < cnt[u];) {
                    const int k = wrap1(gz0 + st[u] + pos - R, n), left = kWave - (k & (kWave - 1));
                    const int len = min(min(cnt[u] - pos, n - k), left), f = off[u] + pos - base;
                    unsigned long long m = any[k / kWave] >> (k & (kWave - 1));
                    if (len < kWave) m &= (1ull << len) - 1ull;
                    if (m) {
                        // (Bits of other segments fall outside.)
                        const int w = f >> 6, sh = f & 63;
                        if (w >= 0 && w < kBlock) atomicOr(&bits[w], m << sh);
                        if (sh && w + 1 >= 0 && w + 1 < kBlock) atomicOr(&bits[w + 1], m >> (64 - sh));
                    }
                    pos += len;
                }
            }
            __syncthreads();
            const int rounds = min((total - base + kBlock - 1) / kBlock, kWave);
            unsigned long long todo = 0;
            for (int it = 0; it < rounds; it++)
                todo |= (bits[it * (kBlock / kWave) + wave] >> lane & 1ull) << it;
            for (; todo; todo &= todo - 1) {
                const int f = base + __builtin_ctzll(todo) * kBlock + threadIdx.x;
                int lo = 0, hi = ranges - 1;  // the last range that starts at or before f
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (e_off[mid] <= f) lo = mid;
                    else hi = mid - 1;
                }
                const int2 q = e_row[lo];
                const int qk = e_k[lo] + (f - e_off[lo]);
                const int i = wrap1(gx0 + q.x - R, n), j = wrap1(gy0 + q.y - R, n);
                const int k = wrap1(gz0 + qk - R, n);
                const long c = i * n2 + (long)j * n + k;
                const long im = c + (i == 0 ? n2 * (n - 1) : -n2);
                const long ip = c + (i == n - 1 ? -n2 * (n - 1) : n2);
                const long jm = c + (j == 0 ? n2 - n : -n), jp = c + (j == n - 1 ? n - n2 : n);
                const long km = c + (k == 0 ? n - 1 : -1), kp = c + (k == n - 1 ? 1 - n : 1);
                const double ei = a.eps_int, phic = a.phi[c];
                const double k2c = a.k2[c], exc = a.ex[c], eyc = a.ey[c], ezc = a.ez[c];
                const double exb = a.ex[im], eyb = a.ey[jm], ezb = a.ez[km];
                const int ii = cx + q.x - R, jj = cy + q.y - R, kk = cz + qk - R;
                const double dx = px - ii * h, dy = py - jj * h, dz = pz - kk * h;
                const double dx2 = dx * dx, dy2 = dy * dy, dz2 = dz * dz;
                const double xm = dx + hd2, xp = dx - hd2, ym = dy + hd2, yp = dy - hd2;
                const double zm = dz + hd2, zp = dz - hd2;
                const double r2c = dx2 + dy2 + dz2;
                const double r2xm = xm * xm + dy2 + dz2, r2xp = xp * xp + dy2 + dz2;
                const double r2ym = dx2 + ym * ym + dz2, r2yp = dx2 + yp * yp + dz2;
                const double r2zm = dx2 + dy2 + zm * zm, r2zp = dx2 + dy2 + zp * zp;
                const bool tc = in_shell(r2c, rp2, rm2) && k2c != 0.0;
                const bool txm = in_shell(r2xm, rp2, rm2) && exb != ei;
                const bool txp = in_shell(r2xp, rp2, rm2) && exc != ei;
                const bool tym = in_shell(r2ym, rp2, rm2) && eyb != ei;
                const bool typ = in_shell(r2yp, rp2, rm2) && eyc != ei;
                const bool tzm = in_shell(r2zm, rp2, rm2) && ezb != ei;
                const bool tzp = in_shell(r2zp, rp2, rm2) && ezc != ei;
                if (!(tc | txm | txp | tym | typ | tzm | tzp)) continue;
                if (tc) {
                    const double r1 = sqrt(r2c) + 1E-12;
                    const double g = k2c * phic * phic * step_dlog(a.c, r1 - r + w);
                    acc[3] += g * (dx / r1);
                    acc[4] += g * (dy / r1);
                    acc[5] += g * (dz / r1);
                }
                double gxn = 0.0, gyn = 0.0, gzn = 0.0;
                if (a.nonpolar) {
                    const double gx = exc - exb, gy = eyc - eyb, gz = ezc - ezb;
                    const double gn = sqrt(gx * gx + gy * gy + gz * gz) / h;
                    const double ig = (gn > 0.0) ? 1.0 / gn : 0.0;
                    gxn = ig * gx;
                    gyn = ig * gy;
                    gzn = ig * gz;
                }
                auto face = [&](bool in, double fx, double fy, double fz, double r2f, double eps_f,
                                long nbr, double g, int sgn) {
                    if (in)
                        face_term(fx, fy, fz, r2f, r, w, a.c, eps_f, ei, a.phi[nbr] - phic, phic, g,
                                  sgn, a.nonpolar, acc);
                };
                face(txm, xm, dy, dz, r2xm, exb, im, gxn, -1);
                face(txp, xp, dy, dz, r2xp, exc, ip, gxn, +1);
                face(tym, dx, ym, dz, r2ym, eyb, jm, gyn, -1);
                face(typ, dx, yp, dz, r2yp, eyc, jp, gyn, +1);
                face(tzm, dx, dy, zm, r2zm, ezb, km, gzn, -1);
                face(tzp, dx, dy, zp, r2zp, ezc, kp, gzn, +1);
            }
        }
        __syncthreads();
    }
    double tot[9];
#pragma unroll
    for (int q = 0; q < 9; q++) tot[q] = block_sum(acc[q], sh);
    if (threadIdx.x == 0) {
        for (int d = 0; d < 3; d++) {
            a.fdb[3 * ion + d] = tot[d] * a.sdb;
            a.fib[3 * ion + d] = tot[3 + d] * a.sdb;
            a.fnp[3 * ion + d] = tot[6 + d] * a.snp;
        }
    }
}

void launch_pb_any(hipStream_t s, PBDev& b, const double* ex, const double* ey, const double* ez,
                   const double* k2) {
    if (!b.marked) {
        const long G = (long)b.n * b.n * b.n;
        MAZE_LAUNCH(k_pb_mark, dim3((unsigned int)((G + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                    G, b.eps_int, ex, ey, ez, k2, b.mark);
        b.marked = 1;
    }
    const long waves = (long)b.n * b.n * b.words;
    MAZE_LAUNCH(k_pb_any, dim3((unsigned int)((waves * kWave + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                s, b.n, b.words, b.mark, b.any);
}

void launch_pb_forces(hipStream_t s, const PBDev& b, const double* pos, const double* phi,
                      const double* ex, const double* ey, const double* ez, const double* k2) {
    if (b.np == 0) return;
    PBForceArgs a{};
    a.n = b.n; a.nonpolar = b.nonpolar;
    a.h = b.h; a.w = b.w; a.eps_int = b.eps_int;
    a.sdb = b.h / (8.0 * kPi);
    a.snp = -b.gamma_np * b.h / (b.eps_s - b.eps_int);
    a.c = step_coef(b.w);
    a.pos = pos; a.radii = b.radii; a.rp2 = b.rp2; a.rm2 = b.rm2; a.rfrc = b.rfrc;
    a.phi = phi; a.ex = ex; a.ey = ey; a.ez = ez; a.k2 = k2;
    a.any = b.any; a.words = b.words;
    a.fdb = b.fdb; a.fib = b.fib; a.fnp = b.fnp;
    MAZE_LAUNCH(k_pb_forces, dim3(b.np), dim3(kBlock), 0, s, a);
}

}  // namespace maze
