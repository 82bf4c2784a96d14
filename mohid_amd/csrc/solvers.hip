// The stand-alone tridiagonal solvers on caller-held rows:
// THOMASZ_NewType2 (Software/MOHIDBase1/ModuleFunctions.F90:4026-4123) and
// THOMAS_3D (MF:3667-3870) = MF.
//
// All three sweeps are bound by memory: a row needs D, E, F and TI once and
// the solution once (40 bytes), and the forward sweep's W and G go out and
// back for the rows that do not stay on chip.  The recurrence itself is
// serial along a line (two operations, then two divisions by the same
// pivot), so a lane keeps whole batches of rows in flight ahead of it.
#include "mgpu_internal.h"

namespace {

// Orders a wave's LDS writes before its later LDS reads.  The kernels here run
// one wave per block, whose LDS instructions execute in order: it is enough
// to keep the compiler from reordering them.  __syncthreads would also wait
// for the loads in flight ahead and the W and G stores (lines along i: 276
// us with it at 512 x 512 x 50, 269 without).
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// One forward-sweep row (MF:4090-4099): W and G from the carried ones.
__device__ __forceinline__ void sweep_row(double D, double E, double F, double TI, double &W,
                                          double &G, bool &pivot) {
    const double aux = E + D * W;
    double w = 0.0, g = 0.0;
    if (fabs(aux) > 0.0) {
        w = -F / aux;
        g = (TI - D * G) / aux;
    } else {
        pivot = true;
    }
    W = w;
    G = g;
}

// ---------------------------------------------------------------------------
// THOMAS_3D along j (THOMAS_3D_i0_j1_NewType, MF:3756-3810): neighbouring
// lanes take neighbouring i, so every row is one contiguous run of the wave.
// One wave per block, so that the few waves there are (a line per lane: 400
// waves at 512 x 50 lines) spread over all CUs; JB rows of the four arrays
// are loaded while the JB before them are swept.  W and G go to the scratch
// as pairs, [block][row][lane].  512 x 512 x 50: 850 us as one load at a time
// in blocks of 256, 197 us now, 4.8 TB/s for the 72 bytes a row moves.
constexpr int JB = 8;

struct RowBatch {
    double d[JB], e[JB], f[JB], t[JB];
};

__device__ __forceinline__ void load_batch(RowBatch &b, int r0, int nrow, long base, long st,
                                           const double *__restrict__ D,
                                           const double *__restrict__ E,
                                           const double *__restrict__ F,
                                           const double *__restrict__ TI) {
#pragma unroll
    for (int q = 0; q < JB; ++q) {
        const int r = r0 + q < nrow ? r0 + q : nrow - 1;   // past the end: the last row again
        const long x = base + r * st;
        b.d[q] = D[x];
        b.e[q] = E[x];
        b.f[q] = F[x];
        b.t[q] = TI[x];
    }
}

__device__ __forceinline__ void sweep_batch(const RowBatch &b, int r0, int nrow, double &W,
                                            double &G, bool &pivot, double2 *__restrict__ wg) {
#pragma unroll
    for (int q = 0; q < JB; ++q) {
        if (r0 + q >= nrow) break;
        if (r0 + q == 0) {
            W = -b.f[q] / b.e[q];
            G = b.t[q] / b.e[q];
        } else {
            sweep_row(b.d[q], b.e[q], b.f[q], b.t[q], W, G, pivot);
        }
        wg[(long)(r0 + q) * 64] = make_double2(W, G);
    }
}

__global__ void __launch_bounds__(64)
lines_j_kernel(long base0, long sIJ, long sJI, long sK, int nIJ, long nl, int nrow,
               const double *__restrict__ D, const double *__restrict__ E,
               const double *__restrict__ F, const double *__restrict__ TI,
               double *__restrict__ res, double2 *__restrict__ scr,
               unsigned long long *__restrict__ pivots) {
    const long line = blockIdx.x * 64L + threadIdx.x;
    if (line >= nl) return;
    const long b = base0 + (line % nIJ) * sIJ + (line / nIJ) * sK;
    double2 *wg = scr + (long)blockIdx.x * nrow * 64 + threadIdx.x;
    double W = 0.0, G = 0.0;
    bool pivot = false;
    RowBatch A, B;
    load_batch(A, 0, nrow, b, sJI, D, E, F, TI);
    for (int r0 = 0; r0 < nrow; r0 += 2 * JB) {
        load_batch(B, r0 + JB, nrow, b, sJI, D, E, F, TI);
        sweep_batch(A, r0, nrow, W, G, pivot, wg);
        load_batch(A, r0 + 2 * JB, nrow, b, sJI, D, E, F, TI);
        sweep_batch(B, r0 + JB, nrow, W, G, pivot, wg);
    }
    // back substitution, 2 JB pairs a batch, the next one in flight
    double xs = G;
    res[b + (nrow - 1) * sJI] = xs;
    constexpr int BB = 2 * JB;
    double2 cur[BB], nxt[BB];
    auto pairs = [&](double2 (&v)[BB], int r0) {
#pragma unroll
        for (int q = 0; q < BB; ++q) v[q] = wg[(long)(r0 - q > 0 ? r0 - q : 0) * 64];
    };
    auto back = [&](const double2 (&v)[BB], int r0) {
#pragma unroll
        for (int q = 0; q < BB; ++q) {
            if (r0 - q < 0) break;
            xs = v[q].x * xs + v[q].y;
            res[b + (r0 - q) * sJI] = xs;
        }
    };
    pairs(cur, nrow - 2);
    for (int r0 = nrow - 2; r0 >= 0; r0 -= 2 * BB) {
        pairs(nxt, r0 - BB);
        back(cur, r0);
        pairs(cur, r0 - 2 * BB);
        back(nxt, r0 - BB);
    }
    if (pivot) atomicAdd(pivots, 1ull);
}

// ---------------------------------------------------------------------------
// THOMAS_3D along i (THOMAS_3D_i1_j0_NewType, MF:3814-3870): a line is
// contiguous in memory and neighbouring lanes' lines lie a column apart, so
// a lane reading its own line would touch 64 cache lines per load.  A wave
// takes 64 lines in tiles of IT rows: it loads a tile so that 16 lanes read
// one line's 128 bytes, turns it in LDS, and every lane then sweeps its own
// line; the next tile's loads are in flight meanwhile.  The solution goes
// back the same way.  W and G go to the scratch as pairs [block][row][lane].
// 512 x 512 x 50: 1722 us with every lane on its own line, 269 us now.
constexpr int IT = 16;
constexpr int ITP = IT + 1;   // LDS row pitch: no two lanes of a half wave on one bank

__global__ void __launch_bounds__(64)
lines_i_kernel(long base0, long sIJ, long sK, int nIJ, long nl, int nrow,
               const double *__restrict__ D, const double *__restrict__ E,
               const double *__restrict__ F, const double *__restrict__ TI,
               double *__restrict__ res, double2 *__restrict__ scr,
               unsigned long long *__restrict__ pivots) {
    __shared__ double tile[4][64 * ITP];
    const int lane = threadIdx.x;
    const long line0 = blockIdx.x * 64L;
    // the lines this lane helps to load: 4 q + lane / IT, its row in the tile
    const int lr = lane % IT, ll = lane / IT;
    constexpr int LPL = 64 / IT;       // lines of one load instruction
    constexpr int NL = 64 / LPL;       // load instructions a tile and array
    long lb[NL];
#pragma unroll
    for (int q = 0; q < NL; ++q) {
        long l = line0 + q * LPL + ll;
        if (l >= nl) l = nl - 1;       // past the end: the last line again (never stored)
        lb[q] = base0 + (l % nIJ) * sIJ + (l / nIJ) * sK;
    }
    double2 *wg = scr + (long)blockIdx.x * nrow * 64 + lane;
    double v[4][NL];
    auto fetch = [&](int r0) {
        const int r = r0 + lr < nrow ? r0 + lr : nrow - 1;
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            v[0][q] = D[lb[q] + r];
            v[1][q] = E[lb[q] + r];
            v[2][q] = F[lb[q] + r];
            v[3][q] = TI[lb[q] + r];
        }
    };
    double W = 0.0, G = 0.0;
    bool pivot = false;
    fetch(0);
    for (int r0 = 0; r0 < nrow; r0 += IT) {
#pragma unroll
        for (int q = 0; q < NL; ++q)
#pragma unroll
            for (int a = 0; a < 4; ++a) tile[a][(q * LPL + ll) * ITP + lr] = v[a][q];
        lds_order();
        if (r0 + IT < nrow) fetch(r0 + IT);
        const int n = nrow - r0 < IT ? nrow - r0 : IT;
#pragma unroll 8
        for (int q = 0; q < n; ++q) {
            const int at = lane * ITP + q;
            const double d = tile[0][at], e = tile[1][at], f = tile[2][at], t = tile[3][at];
            if (r0 + q == 0) {
                W = -f / e;
                G = t / e;
            } else {
                sweep_row(d, e, f, t, W, G, pivot);
            }
            wg[(long)(r0 + q) * 64] = make_double2(W, G);
        }
        lds_order();
    }
    // back substitution, a tile of rows at a time from the top, the next
    // tile's pairs in flight
    double xs = G;
    double2 cur[IT], nxt[IT];
    auto pairs = [&](double2 (&p)[IT], int r0) {
#pragma unroll
        for (int q = 0; q < IT; ++q) {
            const int r = r0 + q < nrow ? r0 + q : nrow - 1;
            p[q] = wg[(long)(r > 0 ? r : 0) * 64];
        }
    };
    const int last = (nrow - 1) / IT * IT;
    pairs(cur, last);
    for (int r0 = last; r0 >= 0; r0 -= IT) {
        if (r0 > 0) pairs(nxt, r0 - IT);
#pragma unroll
        for (int q = IT - 1; q >= 0; --q) {
            if (r0 + q < nrow) {
                if (r0 + q < nrow - 1) xs = cur[q].x * xs + cur[q].y;
                tile[0][lane * ITP + q] = xs;
            }
        }
        lds_order();
        if (r0 + lr < nrow) {
#pragma unroll
            for (int q = 0; q < NL; ++q)
                if (line0 + q * LPL + ll < nl)
                    res[lb[q] + r0 + lr] = tile[0][(q * LPL + ll) * ITP + lr];
        }
        lds_order();
#pragma unroll
        for (int q = 0; q < IT; ++q) cur[q] = nxt[q];
    }
    if (pivot && line0 + lane < nl) atomicAdd(pivots, 1ull);
}

// ---------------------------------------------------------------------------
// THOMASZ_NewType2 on caller-held rows: one lane per water column, KB levels
// loaded while the KB before them are swept.  W and G of the top `win` rows
// stay in LDS (one wave per block: win KB); the rows below them keep W in
// Wscr and G in res, as the reference keeps them in VEC.
//
// Solving 512 x 512 x 50 (262k columns): 209 us with every row's W and G in
// memory and no loads ahead, 219 / 195 / 186 / 154 / 140 us with the loads
// ahead and 0 / 16 / 24 / 40 / 51 rows in LDS: the traffic saved is worth
// more than the waves lost.  52 rows still leave 3 blocks per CU (156 of
// 160 KB); beyond that a third of the loads in flight would go.
constexpr int KB = 4;
constexpr int TZ_WIN = 52;

struct LevelBatch {
    double d[KB], e[KB], f[KB], t[KB];
};

__global__ void __launch_bounds__(64)
thomasz_kernel(Dims d, int win, const double *__restrict__ D, const double *__restrict__ E,
               const double *__restrict__ F, const double *__restrict__ TI,
               const int32_t *__restrict__ wp, double *__restrict__ res,
               double *__restrict__ Wscr) {
    extern __shared__ double2 lwg[];     // [win][64]
    // columns in memory order (i fastest), 64 per block
    const int ni = d.wIUB - d.wILB + 1;
    const long col = blockIdx.x * 64L + threadIdx.x;
    const int i = d.wILB + (int)(col % ni);
    const long jj = d.wJLB + col / ni;
    if (jj > d.wJUB) return;
    const int j = (int)jj;
    const int KLB = d.wKLB, KUB = d.wKUB;
    if (wp[d.idx(i, j, KUB)] != 1) return;
    const int nrow = KUB + 1 - KLB + 1;          // rows KLB .. KUB + 1
    const long b = d.idx(i, j, KLB), st = d.sk;
    const int low = nrow - win;                  // rows below `low` go to memory
    LevelBatch A, B;
    auto load = [&](LevelBatch &v, int r0) {
#pragma unroll
        for (int q = 0; q < KB; ++q) {
            const int r = r0 + q < nrow ? r0 + q : nrow - 1;
            const long x = b + r * st;
            v.d[q] = D[x];
            v.e[q] = E[x];
            v.f[q] = F[x];
            v.t[q] = TI[x];
        }
    };
    double W = 0.0, G = 0.0;
    auto sweep = [&](const LevelBatch &v, int r0) {
#pragma unroll
        for (int q = 0; q < KB; ++q) {
            if (r0 + q >= nrow) break;
            bool zero = false;                   // a zero pivot leaves W = G = 0
            if (r0 + q == 0) {
                // the literal row 1 (MF:4087-4088): KLB is 1
                W = -v.f[q] / v.e[q];
                G = v.t[q] / v.e[q];
            } else {
                sweep_row(v.d[q], v.e[q], v.f[q], v.t[q], W, G, zero);
            }
            if (r0 + q >= low) {
                lwg[(r0 + q - low) * 64 + threadIdx.x] = make_double2(W, G);
            } else {
                const long x = b + (r0 + q) * st;
                Wscr[x] = W;
                res[x] = G;
            }
        }
    };
    load(A, 0);
    for (int r0 = 0; r0 < nrow; r0 += 2 * KB) {
        load(B, r0 + KB);
        sweep(A, r0);
        load(A, r0 + 2 * KB);
        sweep(B, r0 + KB);
    }
    double x1 = G;
    res[b + (nrow - 1) * st] = x1;
    int r = nrow - 2;
    for (; r >= 0 && r >= low; --r) {
        const double2 p = lwg[(r - low) * 64 + threadIdx.x];
        x1 = p.x * x1 + p.y;
        res[b + r * st] = x1;
    }
    for (; r >= 0; r -= 2 * KB) {
        double w[2 * KB], g[2 * KB];
#pragma unroll
        for (int q = 0; q < 2 * KB; ++q) {
            const long x = b + (r - q > 0 ? r - q : 0) * st;
            w[q] = Wscr[x];
            g[q] = res[x];
        }
#pragma unroll
        for (int q = 0; q < 2 * KB; ++q) {
            if (r - q < 0) break;
            x1 = w[q] * x1 + g[q];
            res[b + (r - q) * st] = x1;
        }
    }
}

}  // namespace

long thomas3d_scratch(long nl, int nrow) { return 2 * ((nl + 63) / 64 * 64) * nrow; }

int launch_thomas3d(const mgpu_size3d &sz, int IJmin, int IJmax, int JImin, int JImax, int Kmin,
                    int Kmax, int di, const double *D, const double *E, const double *F,
                    const double *TI, double *res, double *scr, unsigned long long *pivots,
                    hipStream_t s) {
    const long nI = sz.IUB - sz.ILB + 1, nJ = sz.JUB - sz.JLB + 1;
    const long sj = nI, sk = nI * nJ;
    const int nIJ = IJmax - IJmin + 1;
    const long nl = (long)nIJ * (Kmax - Kmin + 1);
    const int nrow = JImax - JImin + 2;
    if (nl <= 0 || nrow <= 0) return MGPU_SUCCESS;
    const dim3 g((unsigned)((nl + 63) / 64)), b(64);
    double2 *wg = reinterpret_cast<double2 *>(scr);
    if (di == 0) {
        const long base0 = (IJmin - sz.ILB) + (JImin - sz.JLB) * sj + (Kmin - sz.KLB) * sk;
        hipLaunchKernelGGL(lines_j_kernel, g, b, 0, s, base0, 1L, sj, sk, nIJ, nl, nrow, D, E, F,
                           TI, res, wg, pivots);
    } else {
        const long base0 = (JImin - sz.ILB) + (IJmin - sz.JLB) * sj + (Kmin - sz.KLB) * sk;
        hipLaunchKernelGGL(lines_i_kernel, g, b, 0, s, base0, sj, sk, nIJ, nl, nrow, D, E, F, TI,
                           res, wg, pivots);
    }
    HIPCHK(hipGetLastError());
    return MGPU_SUCCESS;
}

int launch_thomasz(const Dims &d, const double *D, const double *E, const double *F,
                   const double *TI, const int32_t *wp, double *res, double *Wscr,
                   hipStream_t s) {
    const int ni = d.wIUB - d.wILB + 1, nj = d.wJUB - d.wJLB + 1;
    const int nrow = d.wKUB - d.wKLB + 2;
    const int win = nrow < TZ_WIN ? nrow : TZ_WIN;
    hipLaunchKernelGGL(thomasz_kernel, dim3((unsigned)(((long)ni * nj + 63) / 64)), dim3(64),
                       (size_t)win * 64 * sizeof(double2), s, d, win, D, E, F, TI, wp, res, Wscr);
    HIPCHK(hipGetLastError());
    return MGPU_SUCCESS;
}
