// spectral.hip -- direct FP64 solve of the periodic 7-point Poisson operator.
//
// A = T (+) T (+) T with T the periodic second difference on n points, so A is
// diagonal in the tensor basis of T's real eigenvectors: A^-1 is a transform of
// the three axes, a division by the eigenvalue sums and the inverse transform.
// n is even: T's eigenvectors of even frequency repeat after h = n / 2 points
// and those of odd frequency change sign, so an axis transform of x is two
// h x h products, of x[j] + x[j + h] and of x[j] - x[j + h] (half the work of
// one n x n product).  The products run on the FP64 matrix cores.
//
// Five passes over the grid (z, y, x forward and back, y, z), each reading and
// writing it once, 33.5 MB at 128^3: memory and matrix cores (1.6 GFLOP over
// the five) both take some 30 us there.  A work-group stages 32 lines of one axis
// in LDS (lines along z are contiguous; of y and x lines, 32 neighbours in k are
// taken together, 256-byte runs), and each wave forms 16-wide column tiles of
// the product for both 16-line halves, so that a basis value, read from L2, is
// used twice.
#include <cmath>
#include <vector>

#include "grid.hpp"

namespace maze {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int kLines = 32;
constexpr int kSpecThreads = 256;
constexpr int kStage = 8;  // line-pair values a thread loads at once

enum Axis { kZ, kY, kX };

struct SpecArgs {
    int n, h, hp;      // hp: h rounded up to whole tiles; rows and columns past h are zero
    const double* mf;  // forward: [block][m][t], t-th eigenvector's value at m
    const double* mi;  // inverse: [block][t][m]
    const double* lam; // eigenvalues, even-frequency ones first
};

// LDS pitch of a line (even and odd part, hp values each): 4 more than a
// multiple of 32 doubles, so that the 16 lines x 4 values of an operand read
// use every bank twice, the least there is.
__host__ __device__ inline int spec_pitch(int hp) { return ((2 * hp + 31) & ~31) + 4; }

// acc[b] += basis (columns t0.., from global memory) x lines (16 b.., from LDS):
// D[t][line].  16x16x4 operands: lane i + 16 k holds row / column i of step k,
// result register r of lane j + 16 q is D[q + 4 r][j].
__device__ __forceinline__ void tile_product(const double* __restrict__ m, const double* lines,
                                             int hp, int P, int t0, v4d (&acc)[kLines / 16]) {
    const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
    const double* a = m + lk * hp + t0 + lr;
    const double* b = lines + lr * P + lk;
    double av[4];
#pragma unroll
    for (int u = 0; u < 4; u++) av[u] = a[4 * u * hp];
    for (int m0 = 0; m0 < hp; m0 += 16) {
        double nx[4];
        const int nm = m0 + 16 < hp ? m0 + 16 : m0;
#pragma unroll
        for (int u = 0; u < 4; u++) nx[u] = a[(nm + 4 * u) * hp];
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int q = 0; q < kLines / 16; q++)
                acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], b[16 * q * P + m0 + 4 * u],
                                                              acc[q], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 4; u++) av[u] = nx[u];
    }
}

// Line l's value m: its index in the grid, for this work-group's lines.
template <Axis AX>
struct LineMap {
    int base, lines, stride, n;
    __device__ LineMap(int n_, int wg) : n(n_) {
        const int n2 = n * n;
        if (AX == kZ) {  // 32 rows
            base = wg * kLines * n;
            lines = min(kLines, n2 - wg * kLines);
            stride = 1;
        } else if (AX == kY) {  // 32 neighbours in k of one plane
            const int per = (n + kLines - 1) / kLines;
            const int i = wg / per, k0 = (wg - i * per) * kLines;
            base = i * n2 + k0;
            lines = min(kLines, n - k0);
            stride = n;
        } else {  // 32 neighbours in the (j, k) plane
            base = wg * kLines;
            lines = min(kLines, n2 - base);
            stride = n2;
        }
    }
    __device__ int at(int l, int m) const { return AX == kZ ? base + l * n + m : base + l + m * stride; }
};

template <Axis AX>
int spec_groups(int n) {
    return AX == kY ? n * ((n + kLines - 1) / kLines) : (n * n + kLines - 1) / kLines;
}

// Fwd: transform; Inv: inverse transform; both: with the division by the
// eigenvalue sums between (the last forward axis).  In place where in == out
// (a work-group reads its lines whole before it writes them).
template <Axis AX, bool Fwd, bool Inv>
__global__ __launch_bounds__(kSpecThreads) void k_spec(SpecArgs A, const double* in, double* out) {
    extern __shared__ double L[];
    __shared__ double lsum[kLines];
    const int n = A.n, h = A.h, hp = A.hp, P = spec_pitch(hp), t = threadIdx.x;
    const LineMap<AX> map(n, blockIdx.x);
    if (Fwd && Inv && t < kLines) {
        const int c = min(map.base + t, n * n - 1);
        lsum[t] = A.lam[c / n] + A.lam[c % n];
    }
    // Stage the lines: entry (l, m) of both parts; z lines: neighbouring threads
    // take neighbouring m, else neighbouring l.  Values past h and lines past the
    // last are zero.
    const int count = kLines * hp;
    for (int x0 = t; x0 < count; x0 += kStage * kSpecThreads) {
        double a[kStage], b[kStage];
#pragma unroll
        for (int u = 0; u < kStage; u++) {
            const int x = min(x0 + u * kSpecThreads, count - 1);
            const int l = AX == kZ ? x / hp : x % kLines, m = AX == kZ ? x % hp : x / kLines;
            const bool ok = l < map.lines && m < h;
            const int lc = ok ? l : 0, mc = ok ? m : 0;
            a[u] = in[map.at(lc, mc)];
            b[u] = in[map.at(lc, mc + h)];
            if (!ok) a[u] = b[u] = 0.0;
        }
#pragma unroll
        for (int u = 0; u < kStage; u++) {
            const int x = x0 + u * kSpecThreads;
            if (x < count) {
                const int l = AX == kZ ? x / hp : x % kLines, m = AX == kZ ? x % hp : x / kLines;
                L[l * P + m] = Fwd ? a[u] + b[u] : a[u];
                L[l * P + hp + m] = Fwd ? a[u] - b[u] : b[u];
            }
        }
    }
    __syncthreads();
    const int wave = t >> 6, lane = t & 63, lr = lane & 15, lq = lane >> 4;
    const int tiles = hp / 16;
    constexpr int NW = kSpecThreads / 64, NB = kLines / 16;
    if (Fwd) {
        // Column tiles of both parts; a wave's results stay in registers until
        // every wave has read the lines (up to 16 tiles: n <= 256).
        constexpr int TW = 4;
        v4d acc[TW][NB];
#pragma unroll
        for (int v = 0; v < TW; v++) {
#pragma unroll
            for (int q = 0; q < NB; q++) acc[v][q] = v4d{0.0, 0.0, 0.0, 0.0};
            const int tt = wave + v * NW;
            if (tt < 2 * tiles) {
                const int part = tt >= tiles, t0 = (tt - part * tiles) * 16;
                tile_product(A.mf + (long)part * hp * hp, L + part * hp, hp, P, t0, acc[v]);
            }
        }
        if (Inv) __syncthreads();
#pragma unroll
        for (int v = 0; v < TW; v++) {
            const int tt = wave + v * NW;
            if (tt < 2 * tiles) {
                const int part = tt >= tiles, t0 = (tt - part * tiles) * 16;
#pragma unroll
                for (int q = 0; q < NB; q++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int tc = t0 + lq + 4 * r, l = 16 * q + lr;
                        if (Inv) {
                            const double s = lsum[l] + A.lam[part * h + min(tc, h - 1)];
                            L[l * P + part * hp + tc] =
                                tc < h && s != 0.0 ? acc[v][q][r] / s : 0.0;
                        } else if (tc < h && l < map.lines) {
                            out[map.at(l, part * h + tc)] = acc[v][q][r];
                        }
                    }
            }
        }
        if (Inv) __syncthreads();
    }
    if (Inv) {
        // Values j and j + h from the two parts' tiles.
        for (int tt = wave; tt < tiles; tt += NW) {
            v4d e[NB], o[NB];
#pragma unroll
            for (int q = 0; q < NB; q++) e[q] = o[q] = v4d{0.0, 0.0, 0.0, 0.0};
            tile_product(A.mi, L, hp, P, tt * 16, e);
            tile_product(A.mi + (long)hp * hp, L + hp, hp, P, tt * 16, o);
#pragma unroll
            for (int q = 0; q < NB; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = tt * 16 + lq + 4 * r, l = 16 * q + lr;
                    if (m < h && l < map.lines) {
                        out[map.at(l, m)] = e[q][r] + o[q][r];
                        out[map.at(l, m + h)] = e[q][r] - o[q][r];
                    }
                }
        }
    }
}

template <Axis AX, bool Fwd, bool Inv>
void launch_axis(hipStream_t s, const SpecArgs& a, const double* in, double* out) {
    const size_t lds = sizeof(double) * kLines * (size_t)spec_pitch(a.hp);
    MAZE_LAUNCH((k_spec<AX, Fwd, Inv>), dim3(spec_groups<AX>(a.n)), dim3(kSpecThreads), lds, s, a,
                in, out);
}

int padded(int n) { return (n / 2 + 15) & ~15; }

}  // namespace

bool spectral_ok(int n) { return n % 2 == 0 && n >= 4 && n <= 256; }

long spectral_doubles(int n) { return 4L * padded(n) * padded(n) + n; }

// The eigenbasis on h = n / 2 points and the eigenvalues 2 cos(2 pi k / n) - 2,
// even frequencies k, then odd ones: constant, cosine and sine of each pair, the
// alternating vector (of k = h, in the part of h's parity).
void spectral_tables(int n, double* tab) {
    const int h = n / 2, hp = padded(n);
    const double pi = 3.14159265358979323846;
    double* mf = tab;
    double* mi = tab + 2L * hp * hp;
    double* lam = tab + 4L * hp * hp;
    for (long i = 0; i < 4L * hp * hp; i++) tab[i] = 0.0;
    for (int part = 0; part < 2; part++) {
        int t = 0;
        for (int k = part; k <= h; k += 2)
            for (int sine = 0; sine < 2; sine++) {
                const bool single = k == 0 || k == h;
                if (single && sine) continue;
                const double scale = std::sqrt((single ? 1.0 : 2.0) / n);
                for (int m = 0; m < h; m++) {
                    // The angle reduced in integers.
                    const double ang = 2.0 * pi * (double)((long)k * m % n) / n;
                    const double v = scale * (sine ? std::sin(ang) : std::cos(ang));
                    mf[((long)part * hp + m) * hp + t] = v;
                    mi[((long)part * hp + t) * hp + m] = v;
                }
                lam[part * h + t] = k == 0 ? 0.0 : -4.0 * std::pow(std::sin(pi * k / n), 2);
                t++;
            }
    }
}

// x = A^-1 b without the constant mode; w: a scratch grid (b, x and w may not
// overlap).
void launch_spectral_solve(hipStream_t s, int n, const double* tab, const double* b, double* x,
                           double* w) {
    SpecArgs a;
    a.n = n;
    a.h = n / 2;
    a.hp = padded(n);
    a.mf = tab;
    a.mi = tab + 2L * a.hp * a.hp;
    a.lam = tab + 4L * a.hp * a.hp;
    launch_axis<kZ, true, false>(s, a, b, w);
    launch_axis<kY, true, false>(s, a, w, w);
    launch_axis<kX, true, true>(s, a, w, w);
    launch_axis<kY, false, true>(s, a, w, w);
    launch_axis<kZ, false, true>(s, a, w, x);
}

}  // namespace maze
