// The step's column pass: everything between the stress and advection
// transforms and the next step's velocity spectra, one (kx, ky) column of
// all levels at a time: the stress divergence, the RHS assembly and AB2
// update (main.f90:211-296), the pressure solve (press_stag_array.f90:
// 149-250, tridag_array.f90:165-246), and the projection with its boundary
// rows (forcing.f90:149-244), in one launch.
//
// A block takes CT neighbouring columns of one member and cuts the levels
// 1..nz into chunks of L, one thread per (column, chunk).  A thread reads its
// L levels of the sixteen input spectra, writes the RHS, keeps u* in its own
// slots of LDS and forms its rows' right-hand sides, pivots and reciprocal
// pivots; then the two Thomas sweeps pass from chunk to chunk (shuffles inside
// a wave, which holds 64 / CT chunks of its columns, LDS between waves), five
// dependent operations a row.  The elimination ratio at a chunk's first level
// comes from the case's table (k_tridag_gam), the others from the same
// recurrence.  All in FP64 and with k_tridag's roundings.  (Combining the
// chunks by a scan over their end values and factors takes 4 us less at 64^3
// and 20 us less at 256 x 256 x 192, FP32, but rounds differently.)
//
// Bound by HBM: sixteen spectra in and seven out.  The AB2, tridiagonal,
// projection and boundary kernels it replaces moved 21 + 4 (and the FP64
// Thomas scratch) + 13 and ran the tridiagonal with one thread per column, a
// chain of 2 nz divisions on half the chip's SIMDs.  Measured, those four
// kernels and this one: 256 x 256 x 192 FP32 454 -> 291 us (4.0 TB/s), FP64
// 826 -> 540 us (4.3 TB/s); 128^3 FP32 128 -> 45 to 50 us; 64^3 FP32 52 -> 14
// us; 32^3 FP64 34 -> 9.0 us.  The HBM counters give 1.03 (FP32) and 1.04 (FP64)
// times those volumes.  What holds the largest back: u* takes a block to 152
// (FP32) or 153 KB of LDS, so one is on a CU, and its loads, its two sweeps and
// its stores follow one another with nothing else in flight.  In FP64 one in
// ten requests also misses the CU's first-level TLB (4.1 M of 39.8 M a launch;
// FP32 0.07 M of 38.7 M): a thread's levels lie a plane apart in every array.
#pragma once

#include "pressure.hpp"
#include "spectral.hpp"
#include "timer.hpp"

namespace lg {

// Arguments of the pressure solve alone (press_stag_array's spectra).
template <typename T>
struct ColPress {
    const cplx<T> *hx, *hy, *hz;       // levels 1..nz-1 (hz: 1..nz)
    const cplx<T> *rb, *rt;            // Neumann planes, bottom and top
};

// LDS of a block of nthr threads: row 0 and the solution passed from wave to
// wave (one value per column each), the levels that waves hand to their
// neighbours (one per wave and column) and the u* slots (STEP).
template <typename T>
constexpr size_t column_lds(int L, int CT, int nthr, bool step) {
    return (size_t)2 * CT * sizeof(double2) + (size_t)(nthr / 64) * CT * sizeof(cplx<T>) +
           (size_t)nthr * (step ? 3 * L * sizeof(cplx<T>) : 0);
}

template <typename T>
__device__ __forceinline__ cplx<T> shfl_up_c(cplx<T> v, int d) {
    return cplx<T>{__shfl_up(v.x, d, 64), __shfl_up(v.y, d, 64)};
}
template <typename T>
__device__ __forceinline__ cplx<T> shfl_down_c(cplx<T> v, int d) {
    return cplx<T>{__shfl_down(v.x, d, 64), __shfl_down(v.y, d, 64)};
}

// v is formed here and kept (not sunk to its uses with its operands).
__device__ __forceinline__ void pin(double& v) { asm volatile("" : "+v"(v)); }

// Grid (column tiles, members); whole waves covering CT * ceil(nz / L) threads.
// STEP: the whole column pass on a and g; else the solve alone on q.
// (FP32: 128 registers, sixteen waves a CU; FP64 needs 168, twelve.)
template <typename T>
constexpr int column_max_threads() {
    return sizeof(T) == 4 ? 1024 : 768;
}

template <typename T, int L, int CT, bool STEP>
__global__ void __launch_bounds__(column_max_threads<T>(), sizeof(T) == 4 ? 4 : 3)
    k_column(SpecAb2<T> a, ColPress<T> q, SpecGeo<T> g, TriGeo tg, cplx<T>* ph, const double* gam,
             T dzv, int* err) {
    extern __shared__ __align__(16) unsigned char smem_col[];
    const int nthr = blockDim.x;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6, NW = nthr >> 6;
    double2* x0 = reinterpret_cast<double2*>(smem_col);          // [CT] row 0
    double2* xe = x0 + CT;                                       // [CT] a wave's last value
    cplx<T>* xn = reinterpret_cast<cplx<T>*>(xe + CT);           // [wave][CT] neighbour level
    cplx<T>* Ul = xn + NW * CT;                                  // [3 L][threads] u*
    const int zc = tid / CT, c0 = tid - zc * CT;
    const bool wlo = lane < CT, whi = lane >= 64 - CT;           // a wave's end chunks
    const int ncol = g.ny * g.NK;
    const int cidx = blockIdx.x * CT + c0;
    const bool act = cidx < ncol;
    const int idx = act ? cidx : ncol - 1;
    const int m = blockIdx.y;
    const int nz = g.nz;
    const int k0 = 1 + zc * L;
    const int j = idx / g.NK, cc = idx - j * g.NK;
    const bool nyq = j == g.ny / 2;
    const bool zero = idx == 0;
    const long S = g.splane;
    const long mb = (long)m * g.msp;
    // a member's spectrum is addressed by 32-bit byte offsets from its base
    // (the launcher checks that it is under 4 GiB)
    constexpr unsigned CB = (unsigned)sizeof(cplx<T>);
    const unsigned SB = (unsigned)S * CB;
    unsigned ib = (unsigned)idx * CB;
    auto ld = [&](const cplx<T>* p, int k) -> cplx<T> {
        return *reinterpret_cast<const cplx<T>*>(reinterpret_cast<const char*>(p + mb) +
                                                 ((unsigned)k * SB + ib));
    };
    auto st = [&](cplx<T>* p, int k, cplx<T> v) {
        *reinterpret_cast<cplx<T>*>(reinterpret_cast<char*>(p + mb) + ((unsigned)k * SB + ib)) = v;
    };
    cplx<T> rbt{}, rtt{};              // Neumann rows, in the chunks that hold level 1 and nz
    T kx = (T)0, ky = (T)0;
    const double gk0 = gam[(long)min(k0, nz) * S + idx];
    const double kxd = tg.kxs * (double)cc;
    const double kyd = tg.kys * (double)(j < g.ny / 2 ? j : j - g.ny);
    const double hs = tg.hsc;
    // the right-hand side of the solve's row m, (i kx Hx + i ky Hy) +
    // (Hz(m+1) - Hz(m)) / dz; the (0,0) mode's increments Hz dz.  No
    // contraction here or in the solve: k_tridag's roundings.
    double2 V[L];
    double2 zl{0.0, 0.0};              // Hz of the level before
    cplx<T> uz0{};                     // the chunk's first w
    auto rhs = [&](int l, cplx<T> hx, cplx<T> hy, cplx<T> hz) {
#pragma clang fp contract(off)
        const double2 z{(double)hz.x * hs, (double)hz.y * hs};
        if (l == 0) {
            uz0 = hz;
        } else if (!zero) {
            V[l - 1].x = V[l - 1].x + (z.x - zl.x) * tg.const4;
            V[l - 1].y = V[l - 1].y + (z.y - zl.y) * tg.const4;
        }
        zl = z;
        const double2 x{(double)hx.x * hs, (double)hx.y * hs};
        const double2 y{(double)hy.x * hs, (double)hy.y * hs};
        V[l].x = -x.y * kxd + -y.y * kyd;
        V[l].y = x.x * kxd + y.x * kyd;
        if (zero) V[l] = make_double2(z.x * tg.dz, z.y * tg.dz);
        pin(V[l].x);
        pin(V[l].y);
    };
    if constexpr (STEP) {
        spec_k(g, j, cc, kx, ky);
        const bool eu = a.euler[m] != 0;
        const T mpx = (zero && a.use_mpf) ? (T)a.mpf[2 * m] : (T)0;
        const T mpy = (zero && a.use_mpf) ? (T)a.mpf[2 * m + 1] : (T)0;
        // level indices are clamped to the last level, so every load is in
        // bounds and unconditional; what a clamped level gives is not stored
        cplx<T> xz0 = ld(a.ts.txz, min(k0, nz)), yz0 = ld(a.ts.tyz, min(k0, nz));
        cplx<T> zzm = ld(a.ts.tzz, min(k0 - 1, nz)), pfm = ld(a.pf, min(k0 - 1, nz));
#pragma unroll
        for (int l = 0; l < L; ++l) {
            const int k = k0 + l;
            const int kk = min(k, nz), kp = min(k + 1, nz);
            const cplx<T> cvx = ld(a.cx, kk), cvy = ld(a.cy, kk), cvz = ld(a.cz, kk);
            const cplx<T> xx = ld(a.ts.txx, kk), xy = ld(a.ts.txy, kk), yy = ld(a.ts.tyy, kk);
            const cplx<T> xz1 = ld(a.ts.txz, kp), yz1 = ld(a.ts.tyz, kp);
            const cplx<T> zz = ld(a.ts.tzz, kk);
            const cplx<T> u0 = ld(a.ux, kk), v0 = ld(a.uy, kk), w0 = ld(a.uz, kk);
            const cplx<T> fx = ld(a.rfx, kk), fy = ld(a.rfy, kk), fz = ld(a.rfz, kk);
            const cplx<T> pf = ld(a.pf, kk);
            // (kx = ky = 0 on the Nyquist row)
            cplx<T> dvz = div_ik(xz0, yz0, kx, ky);
            const cplx<T> dvx = add_dz(div_ik(xx, xy, kx, ky), xz1, xz0, a.rdz);
            const cplx<T> dvy = add_dz(div_ik(xy, yy, kx, ky), yz1, yz0, a.rdz);
            if (k >= 2 && k <= nz - 1) dvz = add_dz(dvz, zz, zzm, a.rdz);
            if (k == 1) rbt = dvz;
            if (k == nz) rtt = dvz;
            cplx<T> Rx{-cvx.x - dvx.x, -cvx.y - dvx.y};
            cplx<T> Ry{-cvy.x - dvy.x, -cvy.y - dvy.y};
            cplx<T> Rz{-cvz.x - dvz.x, -cvz.y - dvz.y};
            Rx.x = Rx.x + mpx;
            Ry.x = Ry.x + mpy;
            if (a.fx && k >= a.kf0 && k <= a.kf1 && k <= nz - 1) {
                const cplx<T> p = ld(a.fx, k), r = ld(a.fy, k), s = ld(a.fz, k);
                Rx = cadd(Rx, p);
                Ry = cadd(Ry, r);
                Rz = cadd(Rz, s);
            }
            // RHS_f = its stored part - grad of its pressure; a member's
            // first step is an Euler step: RHS_f = RHS
            const cplx<T> Fx = eu ? Rx : sub_ik(fx, pf, kx);
            const cplx<T> Fy = eu ? Ry : sub_ik(fy, pf, ky);
            const cplx<T> Fz = eu ? Rz : csub(fz, dz_p(pf, pfm, dzv));
            const cplx<T> us = ab2_of(u0, Rx, Fx, a.dt, a.t1, a.t2);
            const cplx<T> vs = ab2_of(v0, Ry, Fy, a.dt, a.t1, a.t2);
            const cplx<T> ws = ab2_of(w0, Rz, Fz, a.dt, a.t1, a.t2);
            Ul[(3 * l + 0) * nthr + tid] = us;
            Ul[(3 * l + 1) * nthr + tid] = vs;
            Ul[(3 * l + 2) * nthr + tid] = ws;
            rhs(l, us, vs, ws);
            if (act && k <= nz) {
                if (k <= nz - 1) {
                    st(a.rx, k, Rx);
                    st(a.ry, k, Ry);
                }
                st(a.rz, k, Rz);
                if (eu) {
                    if (k <= nz - 1) {
                        st(a.rfx, k, Rx);
                        st(a.rfy, k, Ry);
                    }
                    st(a.rfz, k, Rz);
                }
            }
            xz0 = xz1;
            yz0 = yz1;
            zzm = zz;
            pfm = pf;
            // one level's loads at a time: hoisting the next levels' costs
            // the registers of a second block on the CU
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll
        for (int l = 0; l < L; ++l) {
            const int kk = min(k0 + l, nz);
            rhs(l, ld(q.hx, kk), ld(q.hy, kk), ld(q.hz, kk));
        }
        rbt = ld(q.rb, 0);
        rtt = ld(q.rt, 0);
    }
    // row 0: u(0) = dz rb (its -b, -r); the (0,0) mode starts from p(0) = 0
    if (zc == 0)
        x0[c0] = zero ? double2{0.0, 0.0}
                      : double2{tg.dz * (double)rbt.x, tg.dz * (double)rbt.y};
    if (wlo) xn[wave * CT + c0] = uz0;
    __syncthreads();
    {
#pragma clang fp contract(off)
        cplx<T> zn = shfl_down_c(uz0, CT);
        if (whi) zn = wave + 1 < NW ? xn[(wave + 1) * CT + c0] : cplx<T>{(T)0, (T)0};
        if (!zero) {
            V[L - 1].x = V[L - 1].x + ((double)zn.x * hs - zl.x) * tg.const4;
            V[L - 1].y = V[L - 1].y + ((double)zn.y * hs - zl.y) * tg.const4;
        }
    }
    double G[L];                       // gam(m + 1)
    double2 xin{0.0, 0.0};             // the solution one level above the chunk
    {
#pragma clang fp contract(off)
        // The plain recurrences, one chunk after another, so that the solution
        // is k_tridag's to the bit (the dynamic model's clips make a run's
        // 1e-16 roundings visible at 1e-8 within some 100 steps).  The chain is
        // short: the pivots and their reciprocals are formed by every chunk at
        // once, and a quotient t / bet is q = t rb corrected by its remainder,
        // fma(fma(-q, bet, t), rb, q) (Markstein).  With rb = 1 / bet correctly
        // rounded q is within 1.5 ulp and the result is t / bet rounded unless
        // t / bet lies within some 2^-52 ulp of the middle between two doubles;
        // below about 1e-290 the remainder can underflow and the correction with
        // it, and an infinite t gives NaN where a division gives infinity (a
        // run that has diverged).  tests/test_gpu_column_bits.py
        // compares whole steps with k_tridag's divisions.
        const double c3 = tg.const3;
        const double b_in = -(kxd * kxd + kyd * kyd + 2.0 * c3);
        auto quot = [](double t, double bet, double rb) {
            const double q = t * rb;
            return __builtin_fma(__builtin_fma(-q, bet, t), rb, q);
        };
        // row m: u(m) = (V - A u(m-1)) / BT.  The (0,0) mode's p(m) = p(m-1) +
        // V and the rows past the lid (u unchanged) take A = -1, BT = 1, for
        // which the quotient is exact.
        double A[L], BT[L], RB[L];
        {
            double gk = gk0;
            bool bad = false;
#pragma unroll
            for (int l = 0; l < L; ++l) {
                const int k = k0 + l;
                const bool top = k == nz, run = zero || k > nz;
                double bet = (top ? 1.0 : b_in) - (top ? -1.0 : c3) * gk;
                bad |= bet == 0.0 && !run;
                if (run) bet = 1.0;
                A[l] = (top || run) ? -1.0 : c3;
                BT[l] = bet;
                RB[l] = 1.0 / bet;
                G[l] = (top || run) ? 0.0 : quot(c3, bet, RB[l]);
                if (top && !zero) V[l] = make_double2(-tg.dz * (double)rtt.x, -tg.dz * (double)rtt.y);
                if (k == 1 && zero)
                    V[l] = make_double2(-tg.dz * (double)rbt.x, -tg.dz * (double)rbt.y);
                if (k > nz) V[l] = make_double2(0.0, 0.0);
                pin(A[l]);
                pin(BT[l]);
                pin(RB[l]);
                pin(G[l]);
                gk = G[l];
            }
            if (bad && act && !nyq) atomicExch(err, 1);
        }
        // one chunk upward from u (the value below it)
        auto up = [&](double2 u, auto&& keep) {
#pragma unroll
            for (int l = 0; l < L; ++l) {
                const double tx = V[l].x - A[l] * u.x, ty = V[l].y - A[l] * u.y;
                u = make_double2(quot(tx, BT[l], RB[l]), quot(ty, BT[l], RB[l]));
                keep(l, u);
            }
            return u;
        };
        auto down = [&](double2 u) {
#pragma unroll
            for (int l = L - 1; l >= 0; --l)
                u = make_double2(V[l].x - G[l] * u.x, V[l].y - G[l] * u.y);
            return u;
        };
        constexpr int SUB = 64 / CT;   // chunks of a wave
        for (int w = 0; w < NW; ++w) {
            if (wave == w) {
                const double2 u0 = w ? xe[c0] : x0[c0];
                double2 u = u0;
                for (int q = 1; q < SUB; ++q) {
                    const double2 e = up(u, [](int, double2) {});
                    const double2 s{__shfl_up(e.x, CT, 64), __shfl_up(e.y, CT, 64)};
                    u = wlo ? u0 : s;
                }
                u = up(u, [&](int l, double2 v) { V[l] = v; });
                if (whi) xe[c0] = u;
            }
            __syncthreads();
        }
        for (int w = NW - 1; w >= 0; --w) {
            if (wave == w) {
                double2 u0{0.0, 0.0};
                if (w < NW - 1) u0 = xe[c0];
                xin = u0;
                for (int q = 1; q < SUB; ++q) {
                    const double2 e = down(xin);
                    const double2 s{__shfl_down(e.x, CT, 64), __shfl_down(e.y, CT, 64)};
                    xin = whi ? u0 : s;
                }
                const double2 e = down(xin);
                if (wlo) xe[c0] = e;
            }
            __syncthreads();
        }
    }
    cplx<T> p[L];
    cplx<T> pm{(T)0, (T)0};            // the pressure one level below the chunk
    {
#pragma clang fp contract(off)
        double2 u = xin;
#pragma unroll
        for (int l = L - 1; l >= 0; --l) {
            u = make_double2(V[l].x - G[l] * u.x, V[l].y - G[l] * u.y);
            p[l] = nyq ? cplx<T>{(T)0, (T)0} : cplx<T>{(T)u.x, (T)u.y};
        }
        if (zc == 0) {
            // row 0: gam(1) = -1, so p(0) = u(0) + p(1); 0 for the (0,0) mode
            const double2 r0 = x0[c0];
            if (!nyq && !zero) pm = cplx<T>{(T)(r0.x + u.x), (T)(r0.y + u.y)};
            if (act) st(ph, 0, pm);
        }
    }
    // (the levels' offsets are formed again, not kept across the solve)
    int rt = tid;
    asm volatile("" : "+v"(ib), "+v"(rt));
    if constexpr (STEP) {
        __syncthreads();
        if (whi) xn[wave * CT + c0] = p[L - 1];
        __syncthreads();
        const cplx<T> pb = shfl_up_c(p[L - 1], CT);
        if (zc) pm = wlo ? xn[(wave - 1) * CT + c0] : pb;
        if (!act) return;
        const T dt = a.dt, t1 = a.t1;
        const bool eu = a.euler[m] != 0;
#pragma unroll
        for (int l = 0; l < L; ++l) {
            const int k = k0 + l;
            if (k <= nz) {
                const cplx<T> pk = p[l];
                st(ph, k, pk);
                if (eu) st(a.pf, k, cplx<T>{(T)0, (T)0});
                if (k <= nz - 1) {
                    const cplx<T> u1 = proj_ik(Ul[(3 * l + 0) * nthr + rt], pk, kx, dt, t1);
                    const cplx<T> v1 = proj_ik(Ul[(3 * l + 1) * nthr + rt], pk, ky, dt, t1);
                    st(a.ux, k, u1);
                    st(a.uy, k, v1);
                    if (k == nz - 1) {
                        st(a.ux, nz, u1);
                        st(a.uy, nz, v1);
                    }
                }
                cplx<T> w1{(T)0, (T)0};
                if (k >= 2 && k <= nz - 1)
                    w1 = proj_dz(Ul[(3 * l + 2) * nthr + rt], dz_p(pk, pm, dzv), dt, t1);
                st(a.uz, k, w1);
                pm = pk;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (zc == 0) {
            // level 0 BOGUS: the spectrum of a constant plane
            const cplx<T> b = zero ? cplx<T>{(T)BOGUS, (T)0} : cplx<T>{(T)0, (T)0};
            st(a.ux, 0, b);
            st(a.uy, 0, b);
            st(a.uz, 0, b);
            if (eu) st(a.pf, 0, cplx<T>{(T)0, (T)0});
        }
    } else {
        if (!act) return;
#pragma unroll
        for (int l = 0; l < L; ++l)
            if (k0 + l <= nz) st(ph, k0 + l, p[l]);
    }
}

// Chunk length, columns and threads per block (L = 0: no instance, the
// separate kernels run).  It depends on the grid alone, so a member's bits do
// not depend on the batch.
struct ColumnPlan {
    int L = 0, CT = 0, threads = 0;
};

constexpr size_t COLUMN_LDS_MAX = 160 * 1024;

// Columns per block: 256 bytes a level where that leaves 128 blocks or more
// (256 x 256 x 96 FP32: 119 against 135 us with 128 bytes; 128^3: 45 against
// 49; 96 x 48 x 64 FP64, 144 blocks: 17 against 19), else 128 bytes (64^3
// FP32, 64 blocks of 256: 16.9 against 14.9 us).  Chunk length: the shortest
// that needs at most `want` threads, since a short chunk has more loads in
// flight (32^3 FP64: 2, 3, 4 levels 9.2, 10.7, 11.4 us), but a block wider
// than that gains nothing (256 x 256 x 96 FP32, 448, 640, 800 threads: 119,
// 142, 141 us; 96 x 96 x 64 FP64, 256 and 384: 31, 37), else the longest, up to
// the kernel's registers and LDS; taller grids (about 400 levels) have no plan.
template <typename T>
inline ColumnPlan column_plan(int nz, int ncol, long splane) {
    ColumnPlan p;
    if ((unsigned long long)(nz + 1) * (unsigned long long)splane * sizeof(cplx<T>) >=
        (1ull << 32))
        return p;
    constexpr bool f32 = sizeof(T) == 4;
    const int narrow = f32 ? 16 : 8;
    const bool wide_ok = ncol >= 128 * 2 * narrow;
    const int lmax = f32 ? 7 : 5;
    for (int w = wide_ok ? 1 : 0; w >= 0; --w) {
        const int CT = narrow << w;
        const int want = f32 ? (w ? 512 : 384) : 256;
        for (int L : {2, 3, 4, 5, 7}) {
            if (L > lmax) break;
            const int n = (((nz + L - 1) / L) * CT + 63) / 64 * 64;
            if (n > (L == lmax ? column_max_threads<T>() : want)) continue;
            if (column_lds<T>(L, CT, n, true) > COLUMN_LDS_MAX) continue;
            p.L = L;
            p.CT = CT;
            p.threads = n;
            return p;
        }
    }
    return p;
}

// Launches the column pass (STEP) or the solve alone for every member;
// false when the grid has no instance.
template <typename T, bool STEP>
bool launch_column(const SpecAb2<T>& a, const ColPress<T>& q, const SpecGeo<T>& g,
                   const TriGeo& tg, cplx<T>* ph, const double* gam, T dzv, int* err, int M,
                   hipStream_t s) {
    const ColumnPlan p = column_plan<T>(g.nz, g.ny * g.NK, g.splane);
    if (!p.L) return false;
    const dim3 grid((unsigned)((g.ny * g.NK + p.CT - 1) / p.CT), (unsigned)M);
    const dim3 blk((unsigned)p.threads);
    const size_t lds = column_lds<T>(p.L, p.CT, p.threads, STEP);
    constexpr int N = sizeof(T) == 4 ? 16 : 8;
#define LG_COLUMN(LL, CC)                                                                     \
    if (p.L == LL && p.CT == CC) {                                                            \
        LG_LAUNCH((k_column<T, LL, CC, STEP>), grid, blk, lds, s, a, q, g, tg, ph, gam, dzv,  \
                  err);                                                                       \
        return true;                                                                          \
    }
    LG_COLUMN(2, N) LG_COLUMN(3, N) LG_COLUMN(4, N) LG_COLUMN(5, N)
    LG_COLUMN(2, 2 * N) LG_COLUMN(3, 2 * N) LG_COLUMN(4, 2 * N) LG_COLUMN(5, 2 * N)
    if constexpr (sizeof(T) == 4) {
        LG_COLUMN(7, N) LG_COLUMN(7, 2 * N)
    }
#undef LG_COLUMN
    return false;
}

}  // namespace lg
