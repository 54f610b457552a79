// biofvm_fused_kernels.h -- gfx950 device code of the fused x + y sweep.
//
// The x rows of a k-plane are contiguous and its y lines stay inside it, so a
// block that holds a whole plane in LDS solves both axes with one read and
// one write of the field, and one launch takes the place of three (x sweep,
// face pass, y sweep).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "biofvm_kernels.h"

namespace bfa {

// Division by a launch constant: a uniform integer division costs about 30
// scalar instructions, and the block's index arithmetic stands before its
// first load, so the host passes 1/D and the quotient is corrected by one
// where the product rounds across it.  Exact for 0 <= n < 2^22.
struct Divisor {
    int d;
    float r;
};
__device__ __forceinline__ int div_by(int n, const Divisor& D) {
    int q = (int)((float)n * D.r);
    const int rem = n - q * D.d;
    q += rem >= D.d ? 1 : 0;
    q -= rem < 0 ? 1 : 0;
    return __builtin_amdgcn_readfirstlane(q);
}

// A value of another lane, `from` = 4 * lane (taken modulo the wavefront).
__device__ __forceinline__ float lane_get(float v, int from) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(v)));
}
__device__ __forceinline__ double lane_get(double v, int from) {
    const int lo = __builtin_amdgcn_ds_bpermute(from, __double2loint(v));
    const int hi = __builtin_amdgcn_ds_bpermute(from, __double2hiint(v));
    return __hiloint2double(hi, lo);
}

// ---- rows in LDS -----------------------------------------------------------------
// Rows of nx values at a pitch S >= P*L (P = ceil(nx/L) chunks of L nodes, L
// odd, S rounded up to 16 bytes): lane l of a wavefront owns chunk l % P of its
// row l / P, so its node m sits about L*l + m past the wave's first row, and
// with L odd the lanes of an access fall into (nearly) distinct banks, for the
// row's coefficients too.  The padding of a row is zero.

// One row per P lanes of a wavefront, solved in place in LDS: the recurrences
// of x_row_compute with coefficients and scan multipliers in LDS.  No node is
// tested for its place in the row: the Dirichlet ends are set in LDS first,
// coefficients past the row end are zero (so the padding solves to zero), and
// the first padded node repeats the last one, which makes the FP32 form's link
// past the row end vanish.  Lanes without a row (on false) solve the row that
// `row` points to and do not store.
template <typename T, int L, bool DEV>
__device__ __forceinline__ void lds_row_solve(T* __restrict__ row, bool on, int nx, int p, int P, bool dact, T v_lo,
                                              T v_hi, const T* __restrict__ s_xi, const T* __restrict__ s_xc,
                                              const T* __restrict__ s_sm, T k, T lam, T bt) {
    if (dact && on) {
        if (p == 0) row[0] = v_lo;
        if (p == P - 1) row[nx - 1] = v_hi;
    }
    if (DEV && on && p == P - 1 && nx < P * L) row[nx] = row[nx - 1];
    __builtin_amdgcn_wave_barrier();
    const int s = p * L;
    const int self = (threadIdx.x & 63) << 2;
    T* c = row + s;
    T x[L];
#pragma unroll
    for (int m = 0; m < L; ++m) x[m] = c[m];
    if (DEV) {
        T vl = lane_get(x[L - 1], self - 4);
        T vr = lane_get(x[0], self + 4);
        if (p == 0) vl = x[0];
        if (p == P - 1) vr = x[L - 1];
        T dprev = x[0] - vl;
#pragma unroll
        for (int m = 0; m < L; ++m) {
            const T dnext = (m == L - 1 ? vr : x[m + 1 < L ? m + 1 : m]) - x[m];
            x[m] = fma(k, dnext - dprev, fma(-lam, x[m], -bt));
            dprev = dnext;
        }
    }
    const T* inv = s_xi + s;
    const T* cp = s_xc + s;
    const T* sm = s_sm + p;
    T z = T(0);
#pragma unroll
    for (int m = 0; m < L; ++m) z = fma(k, z, x[m]) * inv[m];
#pragma unroll
    for (int j = 0; j < 6; ++j)
        if ((1 << j) < P) z = fma(sm[j * P], lane_get(z, self - (4 << j)), z);
    T y = lane_get(z, self - 4);
    if (p == 0) y = T(0);
#pragma unroll
    for (int m = 0; m < L; ++m) {
        y = fma(k, y, x[m]) * inv[m];
        x[m] = y;
    }
    T w = T(0);
#pragma unroll
    for (int m = L - 1; m >= 0; --m) w = fma(-cp[m], w, x[m]);
#pragma unroll
    for (int j = 0; j < 6; ++j)
        if ((1 << j) < P) w = fma(sm[(6 + j) * P], lane_get(w, self + (4 << j)), w);
    T xn = lane_get(w, self + 4);
    if (p == P - 1) xn = T(0);
#pragma unroll
    for (int m = L - 1; m >= 0; --m) {
        xn = fma(-cp[m], xn, x[m]);
        x[m] = xn;
    }
    if (on) {
#pragma unroll
        for (int m = 0; m < L; ++m) c[m] = DEV ? c[m] + x[m] : x[m];
    }
}

// The multipliers of lds_row_solve's scans (XCoef::fm and ::bm): sm[d][step][p],
// the forward steps 0..5, then the backward ones.  One wavefront per substrate.
template <typename T>
__global__ __launch_bounds__(64) void k_scan_multipliers(int nx, int L, const T* __restrict__ inv,
                                                         const T* __restrict__ cp, const T* __restrict__ k,
                                                         T* __restrict__ sm) {
    const int d = blockIdx.x, p = threadIdx.x, P = (nx + L - 1) / L;
    T za = T(1), wa = T(1);
    for (int m = 0; m < L; ++m) {
        const int f = p * L + m, b = p * L + L - 1 - m;
        za = za * (k[d] * (f < nx ? inv[(long long)d * nx + f] : T(0)));
        wa = wa * (b < nx ? -cp[(long long)d * nx + b] : T(0));
    }
    T* o = sm + (long long)d * 12 * P;
    for (int j = 0; j < 6; ++j) {
        const int off = 1 << j;
        const T pa = shfl_up_t(za, off), na = shfl_down_t(wa, off);
        const bool fo = p >= off, bo = p + off < P;
        if (p < P) {
            o[j * P + p] = fo ? za : T(0);
            o[(6 + j) * P + p] = bo ? wa : T(0);
        }
        if (fo) za = za * pa;
        if (bo) wa = wa * na;
    }
}

// Rows of nx values from memory into LDS rows of pitch S without passing
// through registers (global_load_lds), B bytes per lane and load; the rows are
// dealt to the wavefronts.  Complete after this thread's s_waitcnt vmcnt(0)
// and a barrier.  16 bytes per lane need rows of whole 16-byte vectors (a
// longer load would write into the padding).
template <typename T, int B>
__device__ __forceinline__ void rows_to_lds(T* tile, int S, const T* src, int nx, int rows, int wave, int nw, int lane) {
    const int bytes = nx * (int)sizeof(T);
    for (int r = wave; r < rows; r += nw) {
        const char* g = reinterpret_cast<const char*>(src + (long long)r * nx);
        char* l = reinterpret_cast<char*>(tile + r * S);
        for (int o = 0; o < bytes; o += 64 * B)
            if (o + lane * B < bytes) {
                const auto from = (const __attribute__((address_space(1))) void*)(g + o + lane * B);
                const auto to = (__attribute__((address_space(3))) void*)(l + o);
                if constexpr (B == 16)
                    __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
                else
                    __builtin_amdgcn_global_load_lds(from, to, 4, 0, 0);
            }
    }
}

// ---- one plane per block -----------------------------------------------------------
template <typename T>
struct PlaneArgs {
    SweepArgs<T> x;      // field, x coefficients, constants, Dirichlet table, window d0
    const T* yinv;       // [ns][ny] 1/den and c' of the y lines
    const T* ycp;
    const T* sm;         // [ns][12][P] multipliers of the x scans
    int k0;              // planes k0 .. k0 + nk.d of every substrate of the window
    Divisor nk;
    int P, S;            // x chunks of a row, LDS row pitch
    int PY;              // chunks of a y column
    int W;               // columns per pass of the y phase (W * PY <= blockDim.x)
    int vec;             // rows are whole 16-byte vectors
};

// The x sweep with the Dirichlet passes around it and the y sweep with the one
// after it, of one plane (BioFVM/BioFVM_solvers.cpp:345-731).  x: RW = 64/P rows
// per wavefront (lds_row_solve).  y: PY threads per column, W columns at a
// time, chunk_solve as the separate sweep.  What bounds it on small and middle
// grids is the chain load - x - y - store of one block per CU, so the block
// takes as many threads as both phases can use (plan_fused).  Measured (step,
// separate sweeps -> this): 50^3 FP64 23.2 -> 20.0 us, 75^3 x 2 FP32 28.7 ->
// 22.7, 100^3 x 2 FP64 50.2 -> 39.1, FP32 39.4 -> 29.0, 203x157x121 x 3 FP32
// 89.4 -> 78.9 us.
// Dynamic LDS, of T: ny*S tile | 2*roundup4(PY*LY) y coefficients | 2*P*L x
// coefficients | 12*P scan multipliers | PY*W carries | PY products.
template <typename T, int L, int LY, bool DEV>
__global__ __launch_bounds__(1024) void k_sweep_xy_plane(PlaneArgs<T> g) {
    extern __shared__ __align__(16) unsigned char smem[];
    const SweepArgs<T>& a = g.x;
    const int nx = a.nx, ny = a.ny, nz = a.nz, S = g.S, P = g.P, PY = g.PY, W = g.W;
    T* tile = reinterpret_cast<T*>(smem);
    T* s_inv = tile + ny * S;
    T* s_cp = s_inv + (PY * LY + 3) / 4 * 4;
    T* s_xi = s_cp + (PY * LY + 3) / 4 * 4;
    T* s_xc = s_xi + P * L;
    T* s_sm = s_xc + P * L;
    T* s_z = s_sm + 12 * P;
    T* s_g = s_z + PY * W;
    const int t = threadIdx.x, nthr = blockDim.x, lane = t & 63, nw = nthr >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int b = __builtin_amdgcn_readfirstlane(xcd_block(blockIdx.x, gridDim.x));
    const int dd = div_by(b, g.nk);
    const int d = a.d0 + dd, k = g.k0 + b - dd * g.nk.d;
    T* plane = a.u + (long long)d * a.N + (long long)k * ny * nx;
    if (g.vec)
        rows_to_lds<T, 16>(tile, S, plane, nx, ny, wave, nw, lane);
    else
        rows_to_lds<T, 4>(tile, S, plane, nx, ny, wave, nw, lane);
    for (int e = t; e < P * L; e += nthr) {
        s_xi[e] = e < nx ? a.inv[(long long)d * nx + e] : T(0);
        s_xc[e] = e < nx ? a.cp[(long long)d * nx + e] : T(0);
    }
    for (int e = t; e < 12 * P; e += nthr) s_sm[e] = g.sm[(long long)d * 12 * P + e];
    stage_coefs<T>(s_inv, s_cp, g.yinv + (long long)d * ny, g.ycp + (long long)d * ny, ny, PY * LY, t, nthr);
    if (S > nx) {  // zero padding
        const int pad = S - nx;
        for (int e = t; e < ny * pad; e += nthr) {
            const int r = e / pad;
            tile[r * S + nx + e - r * pad] = T(0);
        }
    }
    const bool dact = (a.active >> d) & 1ull;
    const T kd = a.k[d], lam = DEV ? a.k[a.ns + d] : T(0), bt = DEV ? a.beta[d] : T(0);
    const T v_lo = a.dval[dir_slot_xonly(0, nx, a.reg) * a.ns + d];
    const T v_hi = a.dval[dir_slot_xonly(nx - 1, nx, a.reg) * a.ns + d];
    const int RW = 64 / P, rw = lane / P, p = rw < RW ? lane - rw * P : 0;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's rows are in LDS
    __syncthreads();
    // x phase.  Rows on a y or z face are solved too and overwritten below.
    for (int r = wave * RW; r < ny; r += nw * RW) {
        const bool on = rw < RW && r + rw < ny;
        lds_row_solve<T, L, DEV>(tile + (on ? r + rw : r) * S, on, nx, p, P, dact, v_lo, v_hi, s_xi, s_xc, s_sm, kd, lam,
                                 bt);
    }
    __syncthreads();
    // y phase: thread (yi, py) owns rows [py*LY, py*LY + LY) of column c0 + yi
    const bool kface = k == 0 || k == nz - 1;
    const int py = t / W, yi = t - py * W, sy = py * LY;
    for (int c0 = 0; c0 < nx; c0 += W) {
        const int i = c0 + yi;
        const bool act = py < PY && yi < W && i < nx;
        const int cnt = act ? ny - sy : 0;
        const T* col = tile + sy * S + i;
        T x[LY];
        load_line_chunk<T, LY>(x, col, (size_t)S, cnt);
        // the Dirichlet pass between the sweeps: the end nodes of lines on no
        // face (lines on a face are overwritten whole after the solve)
        const bool ends = act && dact && !kface && i > 0 && i < nx - 1;
        T vlast = T(0);
        if (ends) {
            vlast = a.dval[dir_slot(i, ny - 1, k, nx, ny, nz, a.reg) * a.ns + d];
            if (sy == 0) x[0] = a.dval[dir_slot(i, 0, k, nx, ny, nz, a.reg) * a.ns + d];
            if (cnt <= LY) {
#pragma unroll
                for (int m = 0; m < LY; ++m)
                    if (m == cnt - 1) x[m] = vlast;
            }
        }
        if (DEV) {
            const T vl = cnt > 0 && sy > 0 ? col[-S] : T(0);
            T vr = cnt > LY ? col[LY * S] : T(0);
            if (ends && cnt == LY + 1) vr = vlast;
            delta_residual<T, LY>(x, vl, vr, sy, act ? ny : 0, kd, lam, bt);
        }
        __syncthreads();  // the previous pass's fold readers are done
        chunk_solve<T, LY>(x, act, py, PY, yi, W, s_inv, s_cp, kd, s_z, s_g);
        if (DEV && cnt > 0) {
#pragma unroll
            for (int m = 0; m < LY; ++m) x[m] = (m < cnt ? col[m * S] : T(0)) + x[m];
        }
        if (act && dact) col_dirichlet<T, LY, 1>(x, a, d, i, k, sy, ny, py, PY);
        if (cnt > 0) store_line_chunk<T, LY>(x, plane + (long long)sy * nx + i, (size_t)nx, cnt);
    }
}

}  // namespace bfa
