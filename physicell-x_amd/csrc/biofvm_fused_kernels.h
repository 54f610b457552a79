// biofvm_fused_kernels.h -- gfx950 device code of the fused x + y sweep.
//
// The x rows of a k-plane are contiguous and its y lines stay inside it, so a
// block that holds rows of a plane in LDS solves both axes with one read and
// one write of the field.
//
//  * Planes that fit LDS (k_sweep_xy_plane): a block per plane, y lines whole;
//    one launch takes the place of three (x sweep, face pass, y sweep).
//  * Fields larger than the last-level cache (k_sweep_xy_brick): a block per
//    brick of consecutive rows.  Three separate sweeps move such a field six
//    times; with y lines cut at the brick borders it moves four times.  (The
//    cut is that of the SPIKE method of Polizzi and Sameh, Parallel Computing
//    32, 2006: block diagonal solves, a reduced system of the border values,
//    and spikes that carry them back.)  With T_c the rows of brick c of the
//    line's matrix and k = D*dt/dx^2 the coupling across a border,
//      x_c = T_c^-1 r_c + SL_c * E_(c-1) + SR_c * F_(c+1),
//      SL_c = k T_c^-1 e_first,  SR_c = k T_c^-1 e_last,
//    where F and E are the line's values at a brick's first and last row.  The
//    fused sweep writes T_c^-1 r_c; k_brick_link solves for the border values
//    of every line; the z sweep adds the two spike terms to each node as it
//    loads it (k_sweep_z_fix), so the correction costs no pass of its own.
//    The spikes depend on the row and the substrate only.
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
// longer load would write into the padding).  AUX: cache policy of the loads
// (kStream where the field is larger than the caches).  Returns the wavefront's
// last row (negative if it has none).
constexpr int kStream = 2;
template <typename T, int B, int AUX>
__device__ __forceinline__ int rows_to_lds(T* tile, int S, const T* src, int nx, int rows, int wave, int nw, int lane) {
    const int bytes = nx * (int)sizeof(T);
    int r = wave;
    for (; r < rows; r += nw) {
        const char* g = reinterpret_cast<const char*>(src + (long long)r * nx);
        char* l = reinterpret_cast<char*>(tile + r * S);
        for (int o = 0; o < bytes; o += 64 * B)
            if (o + lane * B < bytes) {
                const auto from = (const __attribute__((address_space(1))) void*)(g + o + lane * B);
                const auto to = (__attribute__((address_space(3))) void*)(l + o);
                if constexpr (B == 16)
                    __builtin_amdgcn_global_load_lds(from, to, 16, 0, AUX);
                else
                    __builtin_amdgcn_global_load_lds(from, to, 4, 0, AUX);
            }
    }
    return r - nw;
}

// ---- one plane per block -----------------------------------------------------------
// Shape and tables of a plane's solve.
template <typename T>
struct PlaneShape {
    const T* yinv;  // [ns][ny] 1/den and c' of the y lines
    const T* ycp;
    const T* sm;    // [ns][12][P] multipliers of the x scans
    int P, S;       // x chunks of a row, LDS row pitch
    int PY;         // chunks of a y column
    int W;          // columns per pass of the y phase (W * PY <= blockDim.x)
    int vec;        // rows are whole 16-byte vectors
};

// The x sweep with the Dirichlet passes around it and the y sweep with the one
// after it, of one plane (BioFVM/BioFVM_solvers.cpp:345-731).  x: RW = 64/P rows
// per wavefront (lds_row_solve).  y: PY threads per column, W columns at a
// time, chunk_solve as the separate sweep.  What bounds it on small and middle
// grids is the chain load - x - y - store of one block per CU, so the block
// takes as many threads as both phases can use (plan_planes).  Measured (step,
// separate sweeps -> this): 50^3 FP64 22.7 -> 14.3 us, 75^3 x 2 FP32 24.8 ->
// 18.8, 100^3 x 2 FP64 45.8 -> 34.4, FP32 35.0 -> 24.3, 203x157x121 x 3 FP32
// 89.4 -> 74.9 us.
// Dynamic LDS, of T: ny*S tile | 2*roundup4(PY*LY) y coefficients | 2*P*L x
// coefficients | 12*P scan multipliers | PY*W carries | PY products.
template <typename T, int L, int LY, bool DEV, bool PV>
__device__ __forceinline__ void sweep_xy_plane(const PlaneShape<T>& g, const SweepArgs<T>& a, int d, int k, T* smem) {
    const int nx = a.nx, ny = a.ny, nz = a.nz, S = g.S, P = g.P, PY = g.PY, W = g.W;
    T* tile = smem;
    T* s_inv = tile + ny * S;
    T* s_cp = s_inv + (PY * LY + 3) / 4 * 4;
    T* s_xi = s_cp + (PY * LY + 3) / 4 * 4;
    T* s_xc = s_xi + P * L;
    T* s_sm = s_xc + P * L;
    T* s_z = s_sm + 12 * P;
    T* s_g = s_z + PY * W;
    const int t = threadIdx.x, nthr = blockDim.x, lane = t & 63, nw = nthr >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    T* plane = a.u + (long long)d * a.N + (long long)k * ny * nx;
    // Held rows on a y face start from zero: the Dirichlet passes set them below
    // whatever they hold, and a NaN or infinity there would reach the rows that
    // share the wavefront (a scan step that is off multiplies another row's value
    // by zero).  Not loading them costs nothing; leaving them out of the x phase
    // cost 1 to 5 % of this kernel (64^3 x 2 FP64 12.2 -> 12.9 us).
    const bool dact = (a.active >> d) & 1ull;
    const int jlo = dact ? 1 : 0, jhi = dact ? ny - 1 : ny;
    if (g.vec)
        rows_to_lds<T, 16, 0>(tile + jlo * S, S, plane + jlo * nx, nx, jhi - jlo, wave, nw, lane);
    else
        rows_to_lds<T, 4, 0>(tile + jlo * S, S, plane + jlo * nx, nx, jhi - jlo, wave, nw, lane);
    if (dact)
        for (int e = t; e < nx; e += nthr) tile[e] = tile[(ny - 1) * S + e] = T(0);
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
    const T kd = a.k[d], lam = DEV ? a.k[a.ns + d] : T(0), bt = DEV ? a.beta[d] : T(0);
    const T v_lo = PV ? T(0) : a.dval[dir_slot_xonly(0, nx, a.reg) * a.ns + d];
    const T v_hi = PV ? T(0) : a.dval[dir_slot_xonly(nx - 1, nx, a.reg) * a.ns + d];
    // Dirichlet value of a boundary voxel of this plane
    auto value = [&](int i, int j) {
        return PV ? dir_value(a, d, i, j, k) : a.dval[dir_slot(i, j, k, nx, ny, nz, a.reg) * a.ns + d];
    };
    const int RW = 64 / P, rw = lane / P, p = rw < RW ? lane - rw * P : 0;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's rows are in LDS
    __syncthreads();
    if (PV && dact) {  // the row ends differ from row to row
        for (int e = t; e < 2 * ny; e += nthr) {
            const int r = e >> 1, i = e & 1 ? nx - 1 : 0;
            tile[r * S + i] = value(i, r);
        }
        __syncthreads();
    }
    // x phase.  Rows on a y or z face are solved too and overwritten below.
    for (int r = wave * RW; r < ny; r += nw * RW) {
        const bool on = rw < RW && r + rw < ny;
        lds_row_solve<T, L, DEV>(tile + (on ? r + rw : r) * S, on, nx, p, P, dact && !PV, v_lo, v_hi, s_xi, s_xc,
                                 s_sm, kd, lam, bt);
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
            vlast = value(i, ny - 1);
            if (sy == 0) x[0] = value(i, 0);
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
        if (PV && act && dact) {
            const bool whole = kface || i == 0 || i == nx - 1;
#pragma unroll
            for (int m = 0; m < LY; ++m)
                if (m < cnt && (whole || sy + m == 0 || m == cnt - 1)) x[m] = value(i, sy + m);
        } else if (act && dact) {
            col_dirichlet<T, LY, 1>(x, a, d, i, k, sy, ny, py, PY);
        }
        if (cnt > 0) store_line_chunk<T, LY>(x, plane + (long long)sy * nx + i, (size_t)nx, cnt);
    }
}

template <typename T>
struct PlaneArgs {
    SweepArgs<T> x;  // field, x coefficients, constants, Dirichlet table, window d0
    PlaneShape<T> s;
    int k0;          // planes k0 .. k0 + nk.d of every substrate of the window
    Divisor nk;
};

// PV: the Dirichlet values are per-voxel planes (SweepArgs::plane), which the
// separate sweeps need four face passes of their own for.
template <typename T, int L, int LY, bool DEV, bool PV>
__global__ __launch_bounds__(1024) void k_sweep_xy_plane(PlaneArgs<T> g) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int b = __builtin_amdgcn_readfirstlane(xcd_block(blockIdx.x, gridDim.x));
    const int dd = div_by(b, g.nk);
    sweep_xy_plane<T, L, LY, DEV, PV>(g.s, g.x, g.x.d0 + dd, g.k0 + b - dd * g.nk.d, reinterpret_cast<T*>(smem));
}

// ---- bricks of rows ------------------------------------------------------------------
// ny rows cut into C bricks: brick c starts at row floor(c*ny / C), so bricks
// differ by at most one row.
constexpr int brick_row_host(int c, int C, int ny) { return (int)((long long)c * ny / C); }
__device__ __forceinline__ int brick_row(int c, const Divisor& C, int ny) { return div_by(c * ny, C); }

template <typename T>
struct BrickArgs {
    SweepArgs<T> x;  // field read, x coefficients, constants, Dirichlet table, window d0
    const T* yinv;   // [ns][C][LY] 1/den and c' of the y lines, restarted at every
    const T* ycp;    //   brick and zero past its rows
    const T* sm;     // [ns][12][P] multipliers of the x scans
    T* out;          // field written (FP64: x.u)
    T* f;            // [ns][nz][C][nx] FP32: increments at the bricks' first and
    T* e;            //   last rows
    Divisor C;       // bricks per plane
    int k0;          // planes k0 .. k0 + nk.d of every substrate of the window
    Divisor nk;
    int P, S;        // x chunks of a row, LDS row pitch
    int vec;         // rows are whole 16-byte vectors
};

// Border system of the bricked y lines.
template <typename T>
struct LinkArgs {
    const T* rc;  // [ns][C][kLinkConsts]
    const T* f;   // first-row values (FP32: increments) of brick c of line (d, k, i)
    const T* e;   // last-row values
    long long fd, fk;  // strides of f and e over d and k (elements)
    T* A;         // [ns][nz][C][nx] out: coupling of brick c to the row before it
    T* B;         //   ... and to the row after it (0 at the ends of the line)
    int C, nx, ny, nz, d0, nd, k0, nk;
    int rows_of_field;  // f and e index the field's rows (else the [C] planes)
};
constexpr int kLinkConsts = 5;  // SL at the first row, 1/(1 - SL_first*q_prev), gamma, SL at the last row, q_prev

// Thomas pivots of every brick's rows, their spikes and the elimination
// constants of the border system, in FP64, rounded once to T.  One block per
// substrate, one thread per brick.  The rows at a brick border keep the full
// diagonal 1 + 2k + lam (their outer neighbour is a known term); the line's
// two end rows keep the Neumann diagonal, as k_thomas.
template <typename T>
__global__ __launch_bounds__(1024) void k_thomas_bricks(int ny, int ns, int C, int LY,
                                                        const double* __restrict__ params,
                                                        double dt, double dx, double* __restrict__ w64,
                                                        T* __restrict__ yinv, T* __restrict__ ycp,
                                                        T* __restrict__ sl, T* __restrict__ sr,
                                                        T* __restrict__ rc) {
    __shared__ double s_end[4 * 1024];  // SL first, SL last, SR first, SR last per brick
    const int d = blockIdx.x, c = threadIdx.x;
    double c1 = params[d];
    c1 *= dt;
    c1 /= dx;
    c1 /= dx;
    double c2 = params[ns + d];
    c2 *= dt;
    c2 /= 3.0;
    const double c3 = 1.0 + c1 + c1 + c2, c3a = 1.0 + c1 + c2;
    if (c < C) {
        const int j0 = brick_row_host(c, C, ny), j1 = brick_row_host(c + 1, C, ny);
        double* inv = w64 + (size_t)d * 3 * ny;  // 1/den, c', forward values of a spike
        double* cp = inv + ny;
        double* y = cp + ny;
        double prev = 0.0;
        for (int j = j0; j < j1; ++j) {
            const double den = fma(c1, prev, (j == 0 || j == ny - 1) ? c3a : c3);
            inv[j] = 1.0 / den;
            prev = cp[j] = (-c1) / den;
        }
        for (int m = 0; m < LY; ++m) {
            yinv[((size_t)d * C + c) * LY + m] = j0 + m < j1 ? (T)inv[j0 + m] : T(0);
            ycp[((size_t)d * C + c) * LY + m] = j0 + m < j1 ? (T)cp[j0 + m] : T(0);
        }
        double z = 0.0, x = 0.0, xl = 0.0;
        for (int j = j0; j < j1; ++j) y[j] = z = ((j == j0 ? c1 : 0.0) + c1 * z) * inv[j];
        for (int j = j1 - 1; j >= j0; --j) {
            x = y[j] - cp[j] * x;  // x = 0 past the brick
            if (j == j1 - 1) xl = x;
            sl[(size_t)d * ny + j] = (T)x;
        }
        s_end[4 * c] = x;
        s_end[4 * c + 1] = xl;
        xl = c1 * inv[j1 - 1];
        x = xl;
        for (int j = j1 - 1; j >= j0; --j) {
            if (j < j1 - 1) x = -cp[j] * x;
            sr[(size_t)d * ny + j] = (T)x;
        }
        s_end[4 * c + 2] = x;
        s_end[4 * c + 3] = xl;
    }
    __syncthreads();
    if (c == 0) {
        double q = s_end[3];
        T* r = rc + (size_t)d * C * kLinkConsts;
        for (int i = 0; i < kLinkConsts; ++i) r[i] = T(0);
        for (int b = 1; b < C; ++b) {
            const double* se = s_end + 4 * b;
            const double rd = 1.0 / (1.0 - se[0] * q);
            const double ga = se[2] * rd;
            r = rc + ((size_t)d * C + b) * kLinkConsts;
            r[0] = (T)se[0];
            r[1] = (T)rd;
            r[2] = (T)ga;
            r[3] = (T)se[1];
            r[4] = (T)q;
            q = fma(se[1] * q, ga, se[3]);
        }
    }
}

// The border values of every bricked y line (d, k, i), one thread each:
// forward, E_c = p_c + q_c F_(c+1) by elimination of F_c; backward, F and E
// from the last brick on.  Writes A_c = E_(c-1) and B_c = F_(c+1).  With the
// FP32 increments the same recurrence gives the increments at the borders.
// Traffic: 2 reads and 2 writes per brick and line.  CM >= C bounds the
// registers that hold the forward values.  400^3 x 4: 89 us in FP64.
template <typename T, int CM>
__global__ __launch_bounds__(256) void k_brick_link(LinkArgs<T> a) {
    const long long lines = (long long)a.nd * a.nk * a.nx;
    const long long g = (long long)blockIdx.x * 256 + threadIdx.x;
    if (g >= lines) return;
    const int i = (int)(g % a.nx);
    const long long dk = g / a.nx;
    const int k = a.k0 + (int)(dk % a.nk), d = a.d0 + (int)(dk / a.nk);
    const T* fp = a.f + d * a.fd + k * a.fk + i;
    const T* ep = a.e + d * a.fd + k * a.fk + i;
    const size_t o = ((size_t)d * a.nz + k) * a.C * a.nx + i;
    const T* rc = a.rc + (size_t)d * a.C * kLinkConsts;
    T f[CM], e[CM];
#pragma unroll
    for (int c = 0; c < CM; ++c)
        if (c < a.C) {
            const int rf = a.rows_of_field ? c * a.ny / a.C : c;
            const int re = a.rows_of_field ? (c + 1) * a.ny / a.C - 1 : c;
            f[c] = fp[(size_t)rf * a.nx];
            e[c] = ep[(size_t)re * a.nx];
        }
    // f[c] becomes alpha_c (F_c = alpha_c + gamma_c F_(c+1)), e[c] becomes p_c
    T p = e[0];
#pragma unroll
    for (int c = 1; c < CM; ++c)
        if (c < a.C) {
            const T* r = rc + c * kLinkConsts;
            const T al = fma(r[0], p, f[c]) * r[1];
            p = fma(r[3], fma(r[4], al, p), e[c]);
            f[c] = al;
            e[c] = p;
        }
    T b = T(0);
#pragma unroll
    for (int c = CM - 1; c >= 0; --c)
        if (c < a.C) {
            const T* r = rc + c * kLinkConsts;
            const size_t at = o + (size_t)c * a.nx;
            a.B[at] = b;
            if (c > 0) {
                const T F = fma(r[2], b, f[c]);
                a.A[at] = fma(r[4], F, e[c - 1]);
                b = F;
            } else {
                a.A[at] = T(0);
            }
        }
}

// Bounded accesses past which nothing is read (0 comes back) or written:
// byte offsets from a uniform base.
template <typename T>
struct Span {
    __amdgpu_buffer_rsrc_t r;
    // base and bytes are uniform; read from the first lane they are known to be
    __device__ __forceinline__ Span(const T* base, unsigned bytes) {
        const uintptr_t b = (uintptr_t)base;
        const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
        const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
        r = __builtin_amdgcn_make_buffer_rsrc((void*)(((uintptr_t)hi << 32) | lo), 0,
                                              __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
    }
    __device__ __forceinline__ T load(unsigned at, unsigned uniform = 0) const;
    __device__ __forceinline__ T load_nt(unsigned at, unsigned uniform = 0) const;
    __device__ __forceinline__ void store(T v, unsigned at, unsigned uniform = 0) const;
    __device__ __forceinline__ void store_nt(T v, unsigned at, unsigned uniform = 0) const;
};
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
template <>
__device__ __forceinline__ float Span<float>::load(unsigned at, unsigned uniform) const {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, at, uniform, 0));
}
template <>
__device__ __forceinline__ double Span<double>::load(unsigned at, unsigned uniform) const {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, at, uniform, 0);
    return __hiloint2double((int)v.y, (int)v.x);
}
template <>
__device__ __forceinline__ float Span<float>::load_nt(unsigned at, unsigned uniform) const {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, at, uniform, kStream));
}
template <>
__device__ __forceinline__ double Span<double>::load_nt(unsigned at, unsigned uniform) const {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, at, uniform, kStream);
    return __hiloint2double((int)v.y, (int)v.x);
}

template <>
__device__ __forceinline__ void Span<float>::store(float v, unsigned at, unsigned uniform) const {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, at, uniform, 0);
}
template <>
__device__ __forceinline__ void Span<double>::store(double v, unsigned at, unsigned uniform) const {
    u32x2 w;
    w.x = (unsigned)__double2loint(v);
    w.y = (unsigned)__double2hiint(v);
    __builtin_amdgcn_raw_buffer_store_b64(w, r, at, uniform, 0);
}
template <>
__device__ __forceinline__ void Span<float>::store_nt(float v, unsigned at, unsigned uniform) const {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, at, uniform, kStream);
}
template <>
__device__ __forceinline__ void Span<double>::store_nt(double v, unsigned at, unsigned uniform) const {
    u32x2 w;
    w.x = (unsigned)__double2loint(v);
    w.y = (unsigned)__double2hiint(v);
    __builtin_amdgcn_raw_buffer_store_b64(w, r, at, uniform, kStream);
}

// Products of the multipliers of a line's chunks of L nodes, as fwd_local and
// bwd_local form them: g[d][0][p] forward, g[d][1][p] backward.
template <typename T>
__global__ __launch_bounds__(64) void k_chunk_products(int n, int L, const T* __restrict__ inv, const T* __restrict__ cp,
                                                       const T* __restrict__ k, T* __restrict__ g) {
    const int d = blockIdx.x, p = threadIdx.x, P = (n + L - 1) / L;
    if (p >= P) return;
    T f = T(1), h = T(1);
    for (int m = 0; m < L; ++m) {
        const int i = p * L + m, j = p * L + L - 1 - m;
        f = f * (k[d] * (i < n ? inv[(long long)d * n + i] : T(0)));
        h = h * (j < n ? -cp[(long long)d * n + j] : T(0));
    }
    g[((long long)d * 2) * P + p] = f;
    g[((long long)d * 2 + 1) * P + p] = h;
}

// One brick per block: rows to LDS (nontemporal: nothing reads the field again
// before it has left the caches), the x lines as in k_sweep_xy_plane, then the
// local y solve, one thread per column, and nontemporal stores.  FP32 solves
// for increments, so it needs the rows next to the brick after their x solve:
// it loads and solves up to two halo rows (8 % of the x work) and writes to a
// second field, since a neighbour may not have read them yet.  FP64 solves for
// values, needs no halo and works in place.
// Bound by HBM with the x phase of one block under the loads of the other (two
// 512-thread blocks per CU).  400^3 x 4: 830 us FP64 (4.9 TB/s; x and y sweep:
// 1700), 465 us FP32 (4.4 TB/s; 870).
// Dynamic LDS, of T: (LY, FP32 LY + 2)*S tile | 2*roundup4(LY) y coefficients |
// 2*P*L x coefficients | 12*P scan multipliers.
template <typename T, int L, int LY, bool DEV>
__global__ __launch_bounds__(1024) void k_sweep_xy_brick(BrickArgs<T> g) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int kRows = DEV ? LY + 2 : LY, kCoefs = (LY + 3) / 4 * 4;
    const SweepArgs<T>& a = g.x;
    const int nx = a.nx, ny = a.ny, nz = a.nz, C = g.C.d, S = g.S, P = g.P;
    T* tile = reinterpret_cast<T*>(smem);
    T* s_inv = tile + kRows * S;
    T* s_cp = s_inv + kCoefs;
    T* s_xi = s_cp + kCoefs;
    T* s_xc = s_xi + P * L;
    T* s_sm = s_xc + P * L;
    const int t = threadIdx.x, nthr = blockDim.x, lane = t & 63, nw = nthr >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // neighbouring bricks, which share halo rows, in one XCD
    const int b = __builtin_amdgcn_readfirstlane(xcd_block(blockIdx.x, gridDim.x));
    const int dk = div_by(b, g.C), cb = b - dk * C, dd = div_by(dk, g.nk);
    const int d = a.d0 + dd, k = g.k0 + dk - dd * g.nk.d;
    const int j0 = brick_row(cb, g.C, ny), j1 = brick_row(cb + 1, g.C, ny), nr = j1 - j0;
    const int hl = DEV && j0 > 0 ? 1 : 0, hr = DEV && j1 < ny ? 1 : 0;
    const int nrx = nr + hl + hr;
    const T* src = a.u + (long long)d * a.N + (long long)(k * ny + j0 - hl) * nx;
    const int last = g.vec ? rows_to_lds<T, 16, kStream>(tile, S, src, nx, nrx, wave, nw, lane)
                           : rows_to_lds<T, 4, kStream>(tile, S, src, nx, nrx, wave, nw, lane);
    for (int e = t; e < P * L; e += nthr) {
        s_xi[e] = e < nx ? a.inv[(long long)d * nx + e] : T(0);
        s_xc[e] = e < nx ? a.cp[(long long)d * nx + e] : T(0);
    }
    for (int e = t; e < 12 * P; e += nthr) s_sm[e] = g.sm[(long long)d * 12 * P + e];
    if (S > nx) {  // zero padding
        const int pad = S - nx;
        for (int e = t; e < nrx * pad; e += nthr) {
            const int r = e / pad;
            tile[r * S + nx + e - r * pad] = T(0);
        }
    }
    // rows past the brick (their y coefficients are zero)
    for (int e = nrx * S + t; e < kRows * S; e += nthr) tile[e] = T(0);
    const bool dact = (a.active >> d) & 1ull;
    const T kd = a.k[d], lam = DEV ? a.k[a.ns + d] : T(0), bt = DEV ? a.beta[d] : T(0);
    const T v_lo = a.dval[dir_slot_xonly(0, nx, a.reg) * a.ns + d];
    const T v_hi = a.dval[dir_slot_xonly(nx - 1, nx, a.reg) * a.ns + d];
    const int RW = 64 / P, rw = lane / P, p = rw < RW ? lane - rw * P : 0;
    if (t < LY) {
        s_inv[t] = g.yinv[((long long)d * C + cb) * LY + t];
        s_cp[t] = g.ycp[((long long)d * C + cb) * LY + t];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's rows are in LDS
    // held rows are cleared, as in sweep_xy_plane, by the wavefront that loaded
    // them (not loading them took 950 us where this takes 929, 400^3 x 4 FP64)
    if (dact && j0 == 0 && wave == 0)
        for (int e = lane; e < nx; e += 64) tile[e] = T(0);
    if (dact && j1 == ny && last == nrx - 1)
        for (int e = lane; e < nx; e += 64) tile[last * S + e] = T(0);
    __syncthreads();
    // x phase: RW rows per wavefront
    for (int r = wave * RW; r < nrx; r += nw * RW) {
        const bool on = rw < RW && r + rw < nrx;
        lds_row_solve<T, L, DEV>(tile + (on ? r + rw : r) * S, on, nx, p, P, dact, v_lo, v_hi, s_xi, s_xc, s_sm, kd, lam,
                                 bt);
    }
    __syncthreads();
    // y phase
    T* ub = g.out + (long long)d * a.N + ((long long)k * ny + j0) * nx;
    const bool kface = k == 0 || k == nz - 1;
    // thread i owns column i of the brick
    const Span<T> out(ub, (unsigned)(nr * nx) * sizeof(T));
    const unsigned rowb = nx * sizeof(T);
    for (int i = t; i < nx; i += nthr) {
        T* col = tile + hl * S + i;
        // Dirichlet before the y solve: the end nodes of lines on no face
        // (lines on a face are overwritten whole by the z sweep)
        if (dact && !kface && i > 0 && i < nx - 1) {
            if (j0 == 0) col[0] = a.dval[dir_slot(i, 0, k, nx, ny, nz, a.reg) * a.ns + d];
            if (j1 == ny) col[(nr - 1) * S] = a.dval[dir_slot(i, ny - 1, k, nx, ny, nz, a.reg) * a.ns + d];
        }
        // no link past the line's end
        if (DEV && !hr) col[nr * S] = col[(nr - 1) * S];
        T x[LY + 1];
#pragma unroll
        for (int m = 0; m < (DEV ? LY + 1 : LY); ++m) x[m] = col[m * S];
        if (DEV) {
            // links to the halo rows are known terms of the local solve
            T dprev = hl ? x[0] - col[-S] : T(0);
#pragma unroll
            for (int m = 0; m < LY; ++m) {
                const T dnext = x[m + 1] - x[m];
                x[m] = fma(kd, dnext - dprev, fma(-lam, x[m], -bt));
                dprev = dnext;
            }
        }
        T y = T(0);
#pragma unroll
        for (int m = 0; m < LY; ++m) {
            y = fma(kd, y, x[m]) * s_inv[m];
            x[m] = y;
        }
        y = T(0);
#pragma unroll
        for (int m = LY - 1; m >= 0; --m) {
            y = fma(-s_cp[m], y, x[m]);
            x[m] = y;
            if (!DEV) {
                // stored as it is found: issued in one burst behind the solve
                // the stores took 10 % longer (400^3) to 20 % (300^3)
                out.store_nt(y, i * sizeof(T) + m * rowb);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (DEV) {  // the increments at the brick's borders
            const size_t o = (((size_t)d * nz + k) * C + cb) * nx + i;
            g.f[o] = x[0];
            T* e = g.e + o;
            *e = x[LY - 1];
            if (nr < LY) {  // uniform
                T last = x[0];
#pragma unroll
                for (int m = 1; m < LY - 1; ++m)
                    if (m == nr - 1) last = x[m];
                *e = last;
            }
        }
        if (DEV) {
#pragma unroll
            for (int m = 0; m < LY; ++m) out.store_nt(col[m * S] + x[m], i * sizeof(T) + m * rowb);
        }
    }
}

// ---- z sweep of a bricked field ------------------------------------------------
// The z sweep on the field that the fused sweep left: each node's value is
// w + (SL*A + SR*B) with the spikes of its row and the border values of its
// line, and the Dirichlet pass before the z sweep follows.  FP64 forms the
// value first; FP32 keeps w and the correction apart up to the end
// (x = w + (correction + increment)), so the field is rounded once per sweep
// as in the separate sweeps.
//
// FP64 blocks solve TX columns of several rows of one brick, one row after the
// other: A and B belong to the brick, so they are read once and stay in
// registers, and the next row's values are in flight while a row is solved.
// The kernel is bound by HBM; 25 nodes per thread with their A and B take the
// registers of two 256-thread blocks per CU, which the loop over rows makes
// up for.  FP32 also keeps the corrections of 25 nodes until the end and has
// no registers left for a loop: one row per block, more blocks, A and B from
// L2.  Loads of the field are nontemporal; stores are not (rows that are no
// multiple of 128 bytes share lines with their neighbours: nontemporal stores
// took 780 us where these take 580, 300^3 x 4 FP64).  400^3 x 4: 905 us FP64
// (4.5 TB/s; plain z sweep 1150), 555 us FP32 (443: the x + y sweep gains more).
template <typename T>
struct FixArgs {
    const T* in;  // the fused sweep's field
    const T* sl;
    const T* sr;
    const T* A;
    const T* B;
    const T* g;   // [ns][2][P] products of the z chunks' multipliers, forward and backward
    unsigned long long active;  // Dirichlet before the z sweep
    Divisor C;
    Divisor parts;  // row groups per brick (FP32: one row each)
    Divisor IT;     // tiles per row, ceil(nx / TX)
    Divisor tiles;  // tiles per substrate: IT * parts * C
};

// chunk_solve for a block that solves several lines in turn: the chunks'
// multiplier products gf / gb are in LDS already, and the two carry buffers
// leave two barriers per line.
template <typename T, int L>
__device__ __forceinline__ void chunk_solve_again(T (&x)[L], int p, int P, int line, int lines,
                                                  const T* __restrict__ s_inv, const T* __restrict__ s_cp, T k,
                                                  T* s_zf, T* s_zb, const T* __restrict__ s_gf,
                                                  const T* __restrict__ s_gb) {
    const int s = p * L;
    T z = T(0);
#pragma unroll
    for (int m = 0; m < L; ++m) z = fma(k, z, x[m]) * s_inv[s + m];
    s_zf[p * lines + line] = z;
    __syncthreads();
    T y = T(0);
#pragma unroll 8
    for (int q = 0; q < p; ++q) y = fma(s_gf[q], y, s_zf[q * lines + line]);
    fwd_apply<T, L>(x, s, s_inv, k, y);
    T w = T(0);
#pragma unroll
    for (int m = L - 1; m >= 0; --m) w = fma(-s_cp[s + m], w, x[m]);
    s_zb[p * lines + line] = w;
    __syncthreads();
    T xn = T(0);
#pragma unroll 8
    for (int q = P - 1; q > p; --q) xn = fma(s_gb[q], xn, s_zb[q * lines + line]);
    bwd_apply<T, L>(x, s, s_cp, xn);
}

// blockDim.x = TX*P; grid = (C*parts*ceil(nx/TX), nd).  Dynamic LDS, of T:
// 2*P*L coefficients | 2*TX*P carries | 2*P products, FP32: | TX*P*L values.
template <typename T, int L, bool DEV, int TX, int NT, int WPE>
__global__ __launch_bounds__(NT, WPE) void k_sweep_z_fix(SweepArgs<T> a, FixArgs<T> fx) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int nx = a.nx, ny = a.ny, n = a.nz, C = fx.C.d;
    const int P = (n + L - 1) / L;
    T* s_inv = reinterpret_cast<T*>(smem);
    T* s_cp = s_inv + P * L;
    T* s_zf = s_cp + P * L;
    T* s_zb = s_zf + (size_t)TX * P;
    T* s_gf = s_zb + (size_t)TX * P;
    T* s_gb = s_gf + P;
    T* s_v = s_gb + P;

    const int t = threadIdx.x;
    const int lane = t % TX;
    const int p = t / TX;
    const int lb = __builtin_amdgcn_readfirstlane(a.runs == 1 ? xcd_block(blockIdx.x, gridDim.x)
                                                              : xcd_runs(blockIdx.x, gridDim.x, a.runs));
    const int dd = div_by(lb, fx.tiles), d = a.d0 + dd;
    const int tb = lb - dd * fx.tiles.d, bp = div_by(tb, fx.IT), cb = div_by(bp, fx.parts), part = bp - cb * fx.parts.d;
    const int jb = brick_row(cb, fx.C, ny), nrb = brick_row(cb + 1, fx.C, ny) - jb;
    const int ja = jb + div_by(part * nrb, fx.parts), je = jb + div_by((part + 1) * nrb, fx.parts);
    if (ja >= je) return;  // uniform over the block
    const int ci = (tb - bp * fx.IT.d) * TX + lane;
    const bool act = ci < nx;
    const int s = p * L;
    int cnt = n - s;  // nodes of the chunk and past it
    // byte offsets of the chunk's first node in the substrate's field and in
    // the brick's border planes; past the line's end and for lanes without a
    // column they lie outside the spans (reads give 0, writes are dropped)
    const unsigned sb = (unsigned)nx * ny * sizeof(T), bb = (unsigned)C * nx * sizeof(T);
    unsigned vo = act ? (unsigned)(s * ny * nx + ci) * (unsigned)sizeof(T) : (unsigned)a.N * (unsigned)sizeof(T);
    const Span<T> in(fx.in + (long long)d * a.N, (unsigned)a.N * (unsigned)sizeof(T));
    const Span<T> out(a.u + (long long)d * a.N, (unsigned)a.N * (unsigned)sizeof(T));
    const bool dpre = (fx.active >> d) & 1ull, dpost = (a.active >> d) & 1ull;
    const T k = a.k[d], lam = DEV ? a.k[a.ns + d] : T(0), beta = DEV ? a.beta[d] : T(0);
    // end values of lines on no other face
    const T d_lo = a.dval[dir_slot(-1, -1, 0, nx, ny, n, a.reg) * a.ns + d];
    const T d_hi = a.dval[dir_slot(-1, -1, n - 1, nx, ny, n, a.reg) * a.ns + d];
    const bool lo = s == 0, hi = cnt <= L, next_last = cnt == L + 1;
    // the border values of this chunk's nodes, and (FP32) those of the nodes next to it
    T A[L], B[L];
    T Al = T(0), Bl = T(0), Ar = T(0), Br = T(0);
    const unsigned bytes = ((unsigned)(n - 1) * C * nx + nx) * (unsigned)sizeof(T);
    const long long bo = ((long long)d * n * C + cb) * nx;
    const Span<T> sA(fx.A + bo, bytes), sB(fx.B + bo, bytes);
    unsigned at = act ? (unsigned)(s * C * nx + ci) * (unsigned)sizeof(T) : bytes;
    auto borders = [&](unsigned at) {
#pragma unroll
        for (int m = 0; m < L; ++m) {
            A[m] = sA.load(at + m * bb);
            B[m] = sB.load(at + m * bb);
        }
        if (DEV) {
            if (!lo) {
                Al = sA.load(at - bb);
                Bl = sB.load(at - bb);
            }
            Ar = sA.load(at + L * bb);
            Br = sB.load(at + L * bb);
        }
    };
    constexpr bool LOOP = !DEV;
    if (LOOP) borders(at);
    T nxt[L], nl = T(0), nr = T(0);
    auto fetch = [&](int j, unsigned vo) {
        const unsigned ju = __builtin_amdgcn_readfirstlane(j * nx * (int)sizeof(T));
#pragma unroll
        for (int m = 0; m < L; ++m) nxt[m] = in.load_nt(vo + m * sb, ju);
        if (DEV) {
            if (!lo) nl = in.load(vo - sb, ju);
            nr = in.load(vo + L * sb, ju);
        }
    };
    fetch(ja, vo);
    stage_coefs<T>(s_inv, s_cp, a.inv + (long long)d * n, a.cp + (long long)d * n, n, P * L, t, blockDim.x);
    if (t < 2 * P) s_gf[t] = fx.g[(long long)d * 2 * P + t];
    __syncthreads();  // coefficient staging complete
    T* sv = s_v + p * L * TX + lane;
    for (int j = ja; j < (LOOP ? je : ja + 1); ++j) {
        T x[L];
#pragma unroll
        for (int m = 0; m < L; ++m) x[m] = nxt[m];
        T vl = nl, vr = nr;
        // the thread's place is invariant over the rows; laundering it keeps
        // the offsets and tests formed from it from being hoisted out of the
        // row loop, where they would take a register each
        asm volatile("" : "+v"(vo), "+v"(cnt), "+v"(at));
        if (!LOOP) borders(at);
        if (LOOP && j + 1 < je) fetch(j + 1, vo);
        T ml = fx.sl[(long long)d * ny + j], mr = fx.sr[(long long)d * ny + j];
        const bool lineb = ci == 0 || ci == nx - 1 || j == 0 || j == ny - 1;
        if constexpr (!DEV) {
#pragma unroll
            for (int m = 0; m < L; ++m) x[m] = fma(mr, B[m], fma(ml, A[m], x[m]));
            if (dpre && (lineb || lo || hi)) {
                if (lineb) {
                    col_dirichlet<T, L, 2>(x, a, d, ci, j, s, n, p, P);
                } else {
                    if (lo) x[0] = d_lo;
#pragma unroll
                    for (int m = 0; m < L; ++m)
                        if (m == cnt - 1) x[m] = d_hi;
                }
            }
            if (hi) {
#pragma unroll
                for (int m = 0; m < L; ++m)
                    if (m >= cnt) x[m] = T(0);
            }
            chunk_solve_again<T, L>(x, p, P, lane, TX, s_inv, s_cp, k, s_zf, s_zb, s_gf, s_gb);
        } else {
            T cr[L];
#pragma unroll
            for (int m = 0; m < L; ++m) cr[m] = fma(ml, A[m], mr * B[m]);
            T cl = fma(ml, Al, mr * Bl), cn = fma(ml, Ar, mr * Br);
            // no correction where the Dirichlet pass sets the node, and past
            // the line's end the last node again (no link there)
            if (dpre && lineb) {
                col_dirichlet<T, L, 2>(x, a, d, ci, j, s, n, p, P);
#pragma unroll
                for (int m = 0; m < L; ++m) cr[m] = T(0);
                cl = cn = T(0);
                if (s > 0) vl = a.dval[dir_slot(ci, j, s - 1, nx, ny, n, a.reg) * a.ns + d];
                if (cnt > L) vr = a.dval[dir_slot(ci, j, s + L, nx, ny, n, a.reg) * a.ns + d];
            } else if (dpre) {
                if (lo) {
                    x[0] = d_lo;
                    cr[0] = T(0);
                }
                if (next_last) {
                    vr = d_hi;
                    cn = T(0);
                }
            }
            if (hi) {
#pragma unroll
                for (int m = 0; m < L; ++m) {
                    if (dpre && !lineb && m == cnt - 1) {
                        x[m] = d_hi;
                        cr[m] = T(0);
                    }
                    if (m > 0 && m == cnt) {
                        x[m] = x[m > 0 ? m - 1 : 0];
                        cr[m] = cr[m > 0 ? m - 1 : 0];
                    }
                }
                if (cnt == L) {
                    vr = x[L - 1];
                    cn = cr[L - 1];
                }
            }
#pragma unroll
            for (int m = 0; m < L; ++m) sv[m * TX] = x[m];
            T dprev = lo ? T(0) : (x[0] - vl) + (cr[0] - cl);
#pragma unroll
            for (int m = 0; m < L; ++m) {
                const T v = x[m], e = cr[m];
                const T right = m == L - 1 ? vr : x[m + 1 < L ? m + 1 : m];
                const T en = m == L - 1 ? cn : cr[m + 1 < L ? m + 1 : m];
                const T dnext = (right - v) + (en - e);
                x[m] = fma(k, dnext - dprev, fma(-lam, v + e, -beta));
                dprev = dnext;
            }
            chunk_solve_again<T, L>(x, p, P, lane, TX, s_inv, s_cp, k, s_zf, s_zb, s_gf, s_gb);
#pragma unroll
            for (int m = 0; m < L; ++m) x[m] = sv[m * TX] + (cr[m] + x[m]);
        }
        if (dpost && (lineb || lo || hi)) {
            if (lineb) {
                col_dirichlet<T, L, 2>(x, a, d, ci, j, s, n, p, P);
            } else {
                if (lo) x[0] = d_lo;
#pragma unroll
                for (int m = 0; m < L; ++m)
                    if (m == cnt - 1) x[m] = d_hi;
            }
        }
        const unsigned ju = __builtin_amdgcn_readfirstlane(j * nx * (int)sizeof(T));
#pragma unroll
        for (int m = 0; m < L; ++m) out.store(x[m], vo + m * sb, ju);
    }
}

}  // namespace bfa
