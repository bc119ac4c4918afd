// Element-local passes of hexahedra with line operators in LDS.
//
// With Gauss-Legendre solution points and flux points at the ends of their
// lines (HexShape, pyfr/shapes.py:378-432) every FR operator is a set of 1-D
// operators along the three lines through a point.  A column-per-thread
// kernel (gen_ops.py) cannot couple an element's five variables, so tgradf,
// tflux, gradcoru_fpts and tdivf each read and write whole (3 Nu, 5, E)
// arrays between them.  Here a block owns EB elements and all their
// variables, and those arrays stay on the chip:
//
//  * thread (i, j, e) owns the pencil of N = p + 1 points (i, j, 0..N-1) of
//    element e: the z operators act in its registers;
//  * the block sweeps the N layers of constant z; each layer's x and y line
//    data go through LDS ([component][N*N][EB], so a wavefront's lanes are
//    consecutive elements: coalesced global access, conflict-free LDS);
//  * EB (16 to 64) elements give each (row, variable) access 64 to 512
//    contiguous bytes.
//
// k_hex_div: Euler tdisf + tdivtpcorf + tdivtconf + negdivconf (FLUX), or
// the correction of a stored volume divergence (Navier-Stokes, after
// k_hex_nsvol), each with the RK stage epilogues of frhip_mul2 and,
// optionally, the next stage's disu (M0 of the stage input it has just
// formed, written over the common fluxes it has just read).
// k_hex_nsvol: Navier-Stokes tgradpcoru + tgradcoru + tdisf + tdivtpcorf +
// gradcoru_fpts; writes the volume divergence and, at the flux points, the
// gradients or only the normal viscous flux each side contributes.
//
// k_hex_div is bound by HBM (4.2-4.8 TB/s).  k_hex_nsvol moves 301 x 40 B of
// an FP64 p = 3 element (1.33 GB on 48^3, by counters as by count; the four
// kernels replaced moved 1600 x 40 B) and is bound by issue: 1,107 vector
// and 180 LDS instructions a wavefront, 44 % and 34 % of its cycles.
#include "frhip_common.h"
#include "frhip_physics.h"

#include <algorithm>
#include <type_traits>

namespace frhip {

// Elements per block of k_hex_div.  64 make a wavefront one pencil: its
// addresses and operator rows are scalar, its accesses whole 512 B (FP64)
// row segments.  RK4 steps, FP64 unless said, elements per block 64 / 32 /
// 16: 48^3 p = 2 1.29 / 1.53 / 1.43 ms, 40^3 p = 3 FP32 0.73 / 0.76 / 0.94.
// From p = 3 in FP64 and p = 4 in FP32 such a block leaves a CU too few
// registers: 40^3 p = 3 - / 1.92 / 1.66 ms, 27^3 p = 4 FP32 - / 0.50 / 0.60.
template <typename T, int N>
constexpr int hex_eb()
{
    return N + (sizeof(T) == 8) <= 4 ? 64 : sizeof(T) == 8 ? 16 : 32;
}

// A grid that leaves CUs without a block takes 16-element blocks (8^3 p = 2:
// 86 against 109 us a step), but not at p = 1 in FP32: such a block is one
// wavefront, whose rows are half a line (RK4 steps with 64 / 16 elements,
// 11^3: 69 / 80 us, 28^3: 107 / 131; in FP64 14^3: 76 / 72).
template <typename T, int N>
constexpr int hex_eb_short()
{
    return N > 2 || sizeof(T) == 8 ? 16 : hex_eb<T, N>();
}

// 1-D operators, on the device: d[i][m] the derivative corrected for the
// interior traces (the line block of M1 - M3 M2, which is also that of
// M4 - M6 M0), hl / hr the correction functions, ll / lr the traces, x the
// points.
template <typename T, int N>
struct HexLine {
    T d[N][N], hl[N], hr[N], ll[N], lr[N], x[N];
};

struct HexPlan {
    int n, dtype;
    void *line;
};

// Barrier for LDS traffic only: global loads stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Ends a layer: x is computed here and no later load is issued before.
// Uncontrolled, the compiler issues every layer's loads first and sums them
// at the end, and spills.
template <typename T, int M>
__device__ __forceinline__ void layer_end(T (&x)[M])
{
#pragma unroll
    for (int v = 0; v < M; ++v) asm volatile("" : "+v"(x[v]) : : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// The thread's pencil; uniform (scalar registers) where a wavefront is one
// pencil of 64 elements.
template <int EB>
__device__ __forceinline__ int hex_pencil()
{
    const int ij = threadIdx.x/EB;
    return EB == 64 ? __builtin_amdgcn_readfirstlane(ij) : ij;
}

// Metric terms along a pencil of a linear hex: dX/dx and dX/dy are linear in
// z, dX/dz is constant (hex_smats of frhip_pointwise.hip, with the vertex
// differences formed first).
template <typename T>
struct PencilGeo {
    T p0[3], p1[3], q0[3], q1[3], r[3];

    __device__ __forceinline__ void load(const T *geo, long ldg,
                                         unsigned lane, T x, T y)
    {
        const T fx[2] = {T(1) - x, T(1) + x}, fy[2] = {T(1) - y, T(1) + y};
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            T v[8];
#pragma unroll
            for (int w = 0; w < 8; ++w) v[w] = at(geo, w*ldg + b*SOA, lane);
            // vertex w: x side w & 1, y side w & 2, z side w & 4
            const T xa = fy[0]*(v[1] - v[0]) + fy[1]*(v[3] - v[2]);
            const T xb = fy[0]*(v[5] - v[4]) + fy[1]*(v[7] - v[6]);
            const T ya = fx[0]*(v[2] - v[0]) + fx[1]*(v[3] - v[1]);
            const T yb = fx[0]*(v[6] - v[4]) + fx[1]*(v[7] - v[5]);
            p0[b] = T(0.125)*(xb + xa);
            p1[b] = T(0.125)*(xb - xa);
            q0[b] = T(0.125)*(yb + ya);
            q1[b] = T(0.125)*(yb - ya);
            r[b] = T(0.125)*(fy[0]*(fx[0]*(v[4] - v[0]) + fx[1]*(v[5] - v[1]))
                           + fy[1]*(fx[0]*(v[6] - v[2]) +
                                    fx[1]*(v[7] - v[3])));
        }
    }

    // S (rows: reference directions) and |J| at height z
    __device__ __forceinline__ void smats(T z, T s[3][3], T &d) const
    {
        T a[3], b[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            a[c] = p0[c] + z*p1[c];
            b[c] = q0[c] + z*q1[c];
        }
        cross(b, r, s[0]);
        cross(r, a, s[1]);
        cross(a, b, s[2]);
        d = a[0]*s[0][0] + a[1]*s[0][1] + a[2]*s[0][2];
    }

    static __device__ __forceinline__ void cross(const T a[3], const T b[3],
                                                 T c[3])
    {
        c[0] = a[1]*b[2] - a[2]*b[1];
        c[1] = a[2]*b[0] - a[0]*b[2];
        c[2] = a[0]*b[1] - a[1]*b[0];
    }
};

template <typename T>
struct HexDivArgs {
    int neles;
    const T *u;         // solution (FLUX) or volume divergence
    long ldu;
    const T *geo;
    long ldg;
    T *f;               // common normal fluxes; next stage's traces
    long ldf;
    T *c;
    long ldc;
    const T *rcp;
    long ldr;
    void *xa;
    double dta, dtb;
    int ep, disu;
    T gm1;
    BaseState<T> bs;
};

// Epilogue families: the epilogues of frhip_mul2 that one instantiation
// serves (the stage is a uniform run-time branch).
enum { HEX_STORE, HEX_RK45, HEX_RK45M, HEX_RK4, HEX_RK4M };

static int hex_family(int ep)
{
    return ep <= 1 ? HEX_STORE : ep == 2 || ep == 4 ? HEX_RK45
         : ep <= 5 ? HEX_RK45M : ep <= 13 ? HEX_RK4 : HEX_RK4M;
}

// Stage update of five values (one point's variables, SOA apart) at row
// offset u and lane element offset off; t holds the stage's RHS and receives
// the next stage's input.
template <typename T, int FAM>
__device__ __forceinline__ void hex_stage(const HexDivArgs<T> &a, long u,
                                          unsigned off, double dta, T t[5],
                                          bool ok)
{
    const unsigned oc = off*(unsigned)sizeof(T), od = off*8u;
    (void)od;
    if constexpr (FAM == HEX_STORE) {
        if (ok)
#pragma unroll
            for (int v = 0; v < 5; ++v) at(a.c, u + v*SOA, oc) = t[v];
    }
    else if constexpr (FAM == HEX_RK45) {
        T *r1 = static_cast<T *>(a.xa);
        T x[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) x[v] = at(r1, u + v*SOA, oc);
        if (a.ep == 4) {
            if (ok)
#pragma unroll
                for (int v = 0; v < 5; ++v)
                    at(r1, u + v*SOA, oc) = x[v] + T(a.dtb)*t[v];
        }
        else
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                // the two registers swap roles: r1 is the next input
                const T nc = x[v] + T(a.dtb)*t[v];
                t[v] = x[v] + T(a.dta)*t[v];
                if (ok) {
                    at(r1, u + v*SOA, oc) = t[v];
                    at(a.c, u + v*SOA, oc) = nc;
                }
            }
    }
    else if constexpr (FAM == HEX_RK45M) {
        double *r1 = static_cast<double *>(a.xa);
        double x[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) x[v] = at(r1, u + v*SOA, od);
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            const double td = (double)t[v], na = x[v] + a.dtb*td;
            t[v] = a.ep == 5 ? (T)na : (T)(x[v] + a.dta*td);
            if (ok) {
                at(r1, u + v*SOA, od) = na;
                at(a.c, u + v*SOA, oc) = t[v];
            }
        }
    }
    else {
        // RK4 (steppers.py:67-108), in T or, for the precision form, FP64
        using R = typename std::conditional<FAM == HEX_RK4, T, double>::type;
        R *const *pp = static_cast<R *const *>(a.xa);
        R *r1 = global_ptr(pp[0]);
        const R *r0 = global_ptr(pp[1]);
        const unsigned orr = off*(unsigned)sizeof(R);
        const int stage = FAM == HEX_RK4 ? a.ep - 9 : a.ep - 13;
        R x[5], y[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            x[v] = stage > 1 ? at(r1, u + v*SOA, orr) : R(0);
            y[v] = stage < 4 ? at(r0, u + v*SOA, orr) : R(0);
        }
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            const R k = (R)t[v];
            R n1, nc;
            if (stage == 1) {
                n1 = k;
                nc = R(1)*y[v];
                nc = nc + R(dta/2.0)*k;
            }
            else if (stage == 2) {
                n1 = R(dta/6.0)*x[v];
                n1 = n1 + R(1)*y[v];
                n1 = n1 + R(dta/3.0)*k;
                nc = R(dta/2.0)*k;
                nc = nc + R(1)*y[v];
            }
            else if (stage == 3) {
                n1 = x[v] + R(dta/3.0)*k;
                nc = R(dta)*k;
                nc = nc + R(1)*y[v];
            }
            else {
                n1 = x[v] + R(dta/6.0)*k;
                nc = n1;
            }
            t[v] = (T)nc;
            if (ok) {
                at(r1, u + v*SOA, orr) = n1;
                if (FAM == HEX_RK4M || stage < 4) at(a.c, u + v*SOA, oc) = t[v];
            }
        }
    }
}

// Flux points at the ends of the lines: faces in HEX_FACES order, first
// face coordinate fastest (pyfr/shapes.py:378-385).  Side s of the x line at
// (j, k) is row FX(s) + j + N k, of the y line at (i, k) FY(s) + i + N k, of
// the z line at (i, j) FZ(s) + i + N j.
template <int N>
struct HexRows {
    static constexpr int x(int s) { return (s ? 2 : 4)*N*N; }
    static constexpr int y(int s) { return (s ? 3 : 1)*N*N; }
    static constexpr int z(int s) { return (s ? 5 : 0)*N*N; }
};

// GEO: the FRHIP_GEO_* mode of the metric terms, or -1: u holds the volume
// part of the transformed divergence and only the correction is added.
template <typename T, int N, int GEO, int FAM, int EB>
__global__ __launch_bounds__(N*N*EB)
__attribute__((amdgpu_waves_per_eu(
    sizeof(T) == 8 && GEO >= 0 ? (N <= 4 ? 3 : 2) : 4))) void k_hex_div(
    const HexLine<T, N> *__restrict__ line, HexDivArgs<T> a)
{
    constexpr int NN = N*N, NU = N*NN;
    constexpr bool FLUX = GEO >= 0;
    // flux lines of two layers, or all layers of the next stage's input
    constexpr int SZ = (FLUX && 20 > 5*N) ? 20 : 5*N;
    __shared__ T sh[SZ*NN*EB];
    using Rows = HexRows<N>;

    const int el = threadIdx.x % EB, ij = hex_pencil<EB>();
    const int i = ij % N, j = ij/N;
    const int e = blockIdx.x*EB + el;
    const bool ok = e < a.neles;
    // lane offsets; everything else in an address is uniform
    const unsigned col = (unsigned)soa_ix(e, 0, 5);
    constexpr unsigned TS = sizeof(T);
    const unsigned ou = ((unsigned)(ij*a.ldu) + col)*TS;
    const unsigned ofi = ((unsigned)(i*a.ldf) + col)*TS;
    const unsigned ofj = ((unsigned)(j*a.ldf) + col)*TS;
    const unsigned ofz = ((unsigned)(ij*a.ldf) + col)*TS;
    const unsigned oc = (unsigned)(ij*a.ldc) + col;
    const unsigned orc = ((unsigned)(ij*a.ldr) + e)*TS;
    [[maybe_unused]] const unsigned og =
        ((unsigned)(ij*a.ldg) + (unsigned)soa_ix(e, 0, 3))*TS;
    double dta = a.dta;
    if constexpr (FAM == HEX_RK4 || FAM == HEX_RK4M)
        dta = *static_cast<const double *>(
            static_cast<void *const *>(a.xa)[2]);

    T wn[5];
    if constexpr (FLUX)
#pragma unroll
        for (int v = 0; v < 5; ++v) wn[v] = at(a.u, v*SOA, ou);

    T dx[N], dy[N];
    if constexpr (FLUX)
#pragma unroll
        for (int m = 0; m < N; ++m) {
            dx[m] = line->d[i][m];
            dy[m] = line->d[j][m];
        }
    const T hx[2] = {line->hl[i], line->hr[i]};
    const T hy[2] = {line->hl[j], line->hr[j]};

    PencilGeo<T> pg;
    if constexpr (GEO == FRHIP_GEO_HEX_LINEAR)
        pg.load(a.geo, a.ldg, (unsigned)soa_ix(e, 0, 3)*TS, line->x[i],
                line->x[j]);

    T acc[N][5];
    if constexpr (!FLUX)
#pragma unroll
        for (int k = 0; k < N; ++k)
#pragma unroll
            for (int v = 0; v < 5; ++v)
                acc[k][v] = at(a.u, NN*k*a.ldu + v*SOA, ou);

#pragma unroll
    for (int k = 0; k < N; ++k) {
        T w[5];
        if constexpr (FLUX)
#pragma unroll
            for (int v = 0; v < 5; ++v) w[v] = wn[v];
        if constexpr (FLUX) {
            T s[3][3], f[3][5], p, vel[3], d;
            if constexpr (GEO == FRHIP_GEO_HEX_LINEAR)
                pg.smats(line->x[k], s, d);
            else
#pragma unroll
                for (int q = 0; q < 3; ++q)
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        s[q][c] = at(a.geo, (q*NU + NN*k)*a.ldg + c*SOA, og);
            inviscid_flux_base(w, f, p, vel, a.gm1, a.bs);
            T *sb = sh + (k & 1)*10*NN*EB + ij*EB + el;
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                sb[v*NN*EB] = s[0][0]*f[0][v] + s[0][1]*f[1][v] +
                              s[0][2]*f[2][v];
                sb[(5 + v)*NN*EB] = s[1][0]*f[0][v] + s[1][1]*f[1][v] +
                                    s[1][2]*f[2][v];
                const T t = s[2][0]*f[0][v] + s[2][1]*f[1][v] +
                            s[2][2]*f[2][v];
#pragma unroll
                for (int m = 0; m < N; ++m)
                    acc[m][v] = k == 0 ? line->d[m][k]*t
                                       : fma(line->d[m][k], t, acc[m][v]);
            }
#pragma unroll
            for (int m = 0; m < N; ++m) layer_end(acc[m]);
        }
        // this layer's common fluxes and the next one's solution are in
        // flight across the barrier (issued earlier, they would live beside
        // the flux's temporaries and cost a wavefront per SIMD)
        T fx[2][5], fy[2][5];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                fx[s][v] = at(a.f, (Rows::x(s) + N*k)*a.ldf + v*SOA, ofj);
                fy[s][v] = at(a.f, (Rows::y(s) + N*k)*a.ldf + v*SOA, ofi);
            }
        if constexpr (FLUX) {
            if (k + 1 < N)
#pragma unroll
                for (int v = 0; v < 5; ++v)
                    wn[v] = at(a.u, NN*(k + 1)*a.ldu + v*SOA, ou);
            // the other buffer was last read before this barrier's
            // predecessor, so one barrier a layer orders both
            lds_barrier();
            const T *sx = sh + (k & 1)*10*NN*EB + j*N*EB + el;
            const T *sy = sh + ((k & 1)*10 + 5)*NN*EB + i*EB + el;
#pragma unroll
            for (int v = 0; v < 5; ++v)
#pragma unroll
                for (int m = 0; m < N; ++m) {
                    acc[k][v] = fma(dx[m], sx[v*NN*EB + m*EB], acc[k][v]);
                    acc[k][v] = fma(dy[m], sy[v*NN*EB + m*N*EB], acc[k][v]);
                }
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                acc[k][v] = fma(hx[s], fx[s][v], acc[k][v]);
                acc[k][v] = fma(hy[s], fy[s][v], acc[k][v]);
            }
        if constexpr (FLUX)
#pragma unroll
            for (int m = 0; m < N; ++m) layer_end(acc[m]);
        else
            layer_end(acc[k]);
    }

    // z corrections, 1/|J| and the stage update, point by point
    T fz[2][5];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int v = 0; v < 5; ++v)
            fz[s][v] = at(a.f, Rows::z(s)*a.ldf + v*SOA, ofz);
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const T nr = -at(a.rcp, NN*k*a.ldr, orc);
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            acc[k][v] = fma(line->hl[k], fz[0][v], acc[k][v]);
            acc[k][v] = fma(line->hr[k], fz[1][v], acc[k][v]);
            acc[k][v] = nr*acc[k][v];
        }
        hex_stage<T, FAM>(a, NN*k*a.ldc, oc, dta, acc[k], ok);
        layer_end(acc[k]);
    }

    if constexpr (FAM != HEX_STORE)
        if (a.disu) {
            // traces of the next stage's input; its values depend on every
            // common flux read above, so those reads are done by the barrier
            T *sb = sh + ij*EB + el;
            lds_barrier();
#pragma unroll
            for (int k = 0; k < N; ++k)
#pragma unroll
                for (int v = 0; v < 5; ++v)
                    sb[(k*5 + v)*NN*EB] = acc[k][v];
            // rows of the lines at (i, j) on the faces: i + N j
            T tz[2][5] = {};
#pragma unroll
            for (int k = 0; k < N; ++k)
#pragma unroll
                for (int v = 0; v < 5; ++v) {
                    tz[0][v] = fma(line->ll[k], acc[k][v], tz[0][v]);
                    tz[1][v] = fma(line->lr[k], acc[k][v], tz[1][v]);
                }
            lds_barrier();
            // thread (i, j) takes the x line and the y line at (i, j) of
            // the faces: points (., i, j) and (i, ., j)
            const T *sx = sh + (j*5*NN + i*N)*EB + el;
            const T *sy = sh + (j*5*NN + i)*EB + el;
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                T t[4] = {};
#pragma unroll
                for (int m = 0; m < N; ++m) {
                    const T px = sx[v*NN*EB + m*EB];
                    const T py = sy[v*NN*EB + m*N*EB];
                    t[0] = fma(line->ll[m], px, t[0]);
                    t[1] = fma(line->lr[m], px, t[1]);
                    t[2] = fma(line->ll[m], py, t[2]);
                    t[3] = fma(line->lr[m], py, t[3]);
                }
                if (ok) {
                    at(a.f, Rows::x(0)*a.ldf + v*SOA, ofz) = t[0];
                    at(a.f, Rows::x(1)*a.ldf + v*SOA, ofz) = t[1];
                    at(a.f, Rows::y(0)*a.ldf + v*SOA, ofz) = t[2];
                    at(a.f, Rows::y(1)*a.ldf + v*SOA, ofz) = t[3];
                    at(a.f, Rows::z(0)*a.ldf + v*SOA, ofz) = tz[0][v];
                    at(a.f, Rows::z(1)*a.ldf + v*SOA, ofz) = tz[1][v];
                }
            }
        }
}

// ---------------------------------------------------------------------------
// Navier-Stokes volume pass
// ---------------------------------------------------------------------------

template <typename T>
struct HexNsArgs {
    int neles;
    const T *u;
    long ldu;
    const T *cm;        // common solution at the flux points
    long ldcm;
    const T *geo;
    long ldg;
    const T *rcp;
    long ldr;
    const T *fn;        // NFV in FP32: the faces' normals, rows of ldg
    T *dv;              // volume part of the transformed divergence
    long ldd;
    T *g;               // gradients (3, nfpts, 5, E) or normal viscous flux
    long ldgr;
    NSConsts<T> c;
    BaseState<T> bs;
};

// Five variables at NP points of EB elements in LDS, as many of them side by
// side as 16 B hold, so that most accesses are ds_read_b128: an 8 B read
// takes as many LDS cycles as a 16 B one (k_hex_nsvol, FP64 p = 3, 48^3:
// 596 us with a plane per variable).
template <typename T, int NP, int EB>
struct Lds5 {
    static constexpr int W = 16/sizeof(T), G = 5/W, R = 5 - G*W;
    typedef T V __attribute__((ext_vector_type(W)));

    static __device__ __forceinline__ void load(const T *b, int p, int el,
                                                T (&x)[5])
    {
        const int q = p*EB + el;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const V v = *reinterpret_cast<const V *>(b + (g*NP*EB + q)*W);
#pragma unroll
            for (int w = 0; w < W; ++w) x[g*W + w] = v[w];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) x[G*W + r] = b[(G*W + r)*NP*EB + q];
    }

    static __device__ __forceinline__ void store(T *b, int p, int el,
                                                 const T (&x)[5])
    {
        const int q = p*EB + el;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            V v;
#pragma unroll
            for (int w = 0; w < W; ++w) v[w] = x[g*W + w];
            *reinterpret_cast<V *>(b + (g*NP*EB + q)*W) = v;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) b[(G*W + r)*NP*EB + q] = x[G*W + r];
    }
};

// y += l x
template <typename T>
__device__ __forceinline__ void fma5(T l, const T (&x)[5], T (&y)[5])
{
#pragma unroll
    for (int v = 0; v < 5; ++v) y[v] = fma(l, x[v], y[v]);
}

// The two in-plane axes of face axis a and the faces of its sides
// (HEX_FACES, pyfr/shapes.py:378-385)
struct HexFace {
    int axis, side, a, b;       // flux point (a, b), first coordinate first

    template <int N>
    static __device__ __forceinline__ HexFace of(int q)
    {
        const int f = q/(N*N), r = q - f*N*N;
        HexFace h;
        h.axis = f == 0 || f == 5 ? 2 : f == 1 || f == 3 ? 1 : 0;
        h.side = f == 2 || f == 3 || f == 5;
        h.b = r/N;
        h.a = r - h.b*N;
        return h;
    }

    // first solution point of the line that ends here, and its step
    template <int N>
    __device__ __forceinline__ void line(int &p0, int &step) const
    {
        p0 = axis == 0 ? N*(a + N*b) : axis == 1 ? a + N*N*b : a + N*b;
        step = axis == 0 ? 1 : axis == 1 ? N : N*N;
    }
};

// One thread per (solution point, element).  The element's u and common
// solution, then the transformed flux, then the gradients pass through one
// LDS buffer; all of the (3, Nu, 5) and (3, Nf, 5) intermediates of the
// kernels replaced stay in registers and LDS.  NFV: at the flux points only
// the normal viscous flux of this side (4 values) instead of the gradients
// (15), for meshes whose interface kernel needs no more.  In FP32 the normal
// comes from coefficients formed in FP64 and rounded once: rebuilt from FP32
// vertices it was off by 4e-6 of its length on 48^3 elements of [0, 2 pi],
// 8e-5 with the box at 100 (48^3 p = 3 steps of the precision form 3.97
// against 4.03 ms: 54 values an element).  FP64 vertices lose nothing, and
// the coefficients cost 3 % of the kernel (64^3 p = 3: 1,271 against 1,307
// us).
template <typename T, int N, int GEO, bool NFV, int EB>
__global__ __launch_bounds__(N*N*N*EB)
__attribute__((amdgpu_waves_per_eu(4))) void k_hex_nsvol(
    const HexLine<T, N> *__restrict__ line, HexNsArgs<T> a)
{
    constexpr int NN = N*N, NU = N*NN, NF = 6*NN;
    constexpr int SLOTS = (NF + NU - 1)/NU;
    // u, and one buffer for the common solution (5 NF), then the flux, then
    // the gradients (15 NU each)
    static_assert(5*NF <= 15*NU, "LDS layout");
    __shared__ __attribute__((aligned(16))) T sh[20*NU*EB];

    const int el = threadIdx.x % EB, pt = threadIdx.x/EB;
    const int i = pt % N, j = pt/N % N;
    // uniform where a layer of constant z is whole wavefronts
    const int k = NN*EB % 64 ? pt/NN
                             : __builtin_amdgcn_readfirstlane(pt/NN);
    const int e = xcd_block()*EB + el;
    const bool ok = e < a.neles;
    const long col = soa_ix(e, 0, 5);

    T u[5];
    const T *pu = a.u + pt*a.ldu + col;
#pragma unroll
    for (int v = 0; v < 5; ++v) u[v] = pu[v*SOA];
    T cm[SLOTS][5];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        const int q = pt + s*NU;
        if (q < NF)
#pragma unroll
            for (int v = 0; v < 5; ++v)
                cm[s][v] = a.cm[q*a.ldcm + col + v*SOA];
    }

    using Lu = Lds5<T, NU, EB>;
    using Lf = Lds5<T, NF, EB>;
    T *su = sh, *sb = sh + 5*NU*EB;
    Lu::store(su, pt, el, u);
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        const int q = pt + s*NU;
        if (q < NF) Lf::store(sb, q, el, cm[s]);
    }
    layer_end(u);

    // metric terms at this point
    T S[3][3], rj[1];
    if constexpr (GEO == FRHIP_GEO_HEX_LINEAR) {
        PencilGeo<T> pg;
        T d;
        pg.load(a.geo, a.ldg, (unsigned)soa_ix(e, 0, 3)*(unsigned)sizeof(T),
                line->x[i], line->x[j]);
        pg.smats(line->x[k], S, d);
        rj[0] = T(1)/d;
    }
    else {
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                S[q][c] = a.geo[((long)q*NU + pt)*a.ldg + soa_ix(e, c, 3)];
        rj[0] = a.rcp[pt*a.ldr + e];
    }

    lds_barrier();

    // corrected gradient, made physical (transform_grad.mako:3-10)
    T g[3][5];
    {
        T cx[N], cy[N], cz[N];
#pragma unroll
        for (int m = 0; m < N; ++m) {
            cx[m] = line->d[i][m];
            cy[m] = line->d[j][m];
            cz[m] = line->d[k][m];
        }
        const T hx[2] = {-line->hl[i], line->hr[i]};
        const T hy[2] = {-line->hl[j], line->hr[j]};
        const T hz[2] = {-line->hl[k], line->hr[k]};
        const int px = N*(j + N*k), py = i + NN*k, pz = i + N*j;
        const int qx = j + N*k, qy = i + N*k, qz = i + N*j;
        using Rows = HexRows<N>;
        T r[3][5] = {}, w[5];
#pragma unroll
        for (int m = 0; m < N; ++m) {
            Lu::load(su, px + m, el, w);
            fma5(cx[m], w, r[0]);
            Lu::load(su, py + N*m, el, w);
            fma5(cy[m], w, r[1]);
            Lu::load(su, pz + NN*m, el, w);
            fma5(cz[m], w, r[2]);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            Lf::load(sb, Rows::x(s) + qx, el, w);
            fma5(hx[s], w, r[0]);
            Lf::load(sb, Rows::y(s) + qy, el, w);
            fma5(hy[s], w, r[1]);
            Lf::load(sb, Rows::z(s) + qz, el, w);
            fma5(hz[s], w, r[2]);
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
#pragma unroll
            for (int v = 0; v < 5; ++v)
                g[d][v] = rj[0]*(S[0][d]*r[0][v] + S[1][d]*r[1][v] +
                                 S[2][d]*r[2][v]);
            layer_end(g[d]);
        }
    }

    lds_barrier();              // the common solution has been read
#pragma unroll
    for (int d = 0; d < 3; ++d) Lu::store(sb + 5*d*NU*EB, pt, el, g[d]);
    lds_barrier();
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        const int q = pt + s*NU;
        if (q >= NF) continue;
        const HexFace h = HexFace::of<N>(q);
        int p0, st;
        h.line<N>(p0, st);
        // this side's normal and state
        T nf[3] = {}, uf[5] = {};
        if constexpr (NFV) {
            const T x = line->x[h.a], y = line->x[h.b];
            if constexpr (sizeof(T) == 4) {
                // linear in each of the face's coordinates: their product's
                // coefficient vanishes
                const T *gn = a.fn + 3*(q/NN)*a.ldg + soa_ix(e, 0, 3);
#pragma unroll
                for (int b = 0; b < 3; ++b)
                    nf[b] = fma(y, gn[2*a.ldg + b*SOA],
                                fma(x, gn[a.ldg + b*SOA], gn[b*SOA]));
            }
            else {
                // the tangents along the face's axes, from its four vertices
                T ts[3], tt[3];
                const int sa = h.axis == 0 ? 1 : 0, ta = h.axis == 2 ? 1 : 2;
                const int v0 = h.side << h.axis;
                const T *gv = a.geo + soa_ix(e, 0, 3);
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    const T w00 = gv[v0*a.ldg + b*SOA];
                    const T w10 = gv[(v0 | 1 << sa)*a.ldg + b*SOA];
                    const T w01 = gv[(v0 | 1 << ta)*a.ldg + b*SOA];
                    const T w11 = gv[(v0 | 1 << sa | 1 << ta)*a.ldg + b*SOA];
                    ts[b] = T(0.25)*((T(1) - y)*(w10 - w00) +
                                     (T(1) + y)*(w11 - w01));
                    tt[b] = T(0.25)*((T(1) - x)*(w01 - w00) +
                                     (T(1) + x)*(w11 - w10));
                }
                PencilGeo<T>::cross(ts, tt, nf);
                // axes (y, z), (x, z), (x, y): the middle one is left-handed
                const T sg = (h.axis == 1) != (h.side == 0) ? T(-1) : T(1);
#pragma unroll
                for (int b = 0; b < 3; ++b) nf[b] *= sg;
            }
            layer_end(nf);
#pragma unroll
            for (int m = 0; m < N; ++m) {
                T w[5];
                Lu::load(su, p0 + st*m, el, w);
                fma5(h.side ? line->lr[m] : line->ll[m], w, uf);
            }
            layer_end(uf);
        }
        T gf[3][5] = {};
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const T l = h.side ? line->lr[m] : line->ll[m];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                T w[5];
                Lu::load(sb + 5*d*NU*EB, p0 + st*m, el, w);
                fma5(l, w, gf[d]);
            }
        }
        T *pg = a.g + q*a.ldgr + col;
        if constexpr (NFV) {
#pragma unroll
            for (int d = 0; d < 3; ++d) layer_end(gf[d]);
            T w[5], f[3][5] = {};
            base_full(uf, w, a.bs);
            viscous_flux_add(w, gf, f, a.c);
            if (ok)
#pragma unroll
                for (int v = 1; v < 5; ++v)
                    pg[v*SOA] = nf[0]*f[0][v] + nf[1]*f[1][v] +
                                nf[2]*f[2][v];
        }
        else if (ok)
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int v = 0; v < 5; ++v)
                    pg[(long)d*NF*a.ldgr + v*SOA] = gf[d][v];
        layer_end(rj);
    }

    // the transformed flux
    {
        T w[5], f[3][5], p, vel[3];
        Lu::load(su, pt, el, u);
#pragma unroll
        for (int d = 0; d < 3; ++d) Lu::load(sb + 5*d*NU*EB, pt, el, g[d]);
        base_full(u, w, a.bs);
        inviscid_flux_base(u, f, p, vel, a.c.gm1, a.bs);
        viscous_flux_add(w, g, f, a.c);
        lds_barrier();                      // the gradients have been read
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            T t[5];
#pragma unroll
            for (int v = 0; v < 5; ++v)
                t[v] = S[d][0]*f[0][v] + S[d][1]*f[1][v] + S[d][2]*f[2][v];
            Lu::store(sb + 5*d*NU*EB, pt, el, t);
        }
    }
    lds_barrier();
    {
        T r[5] = {}, w[5];
#pragma unroll
        for (int m = 0; m < N; ++m) {
            Lu::load(sb, N*(j + N*k) + m, el, w);
            fma5(line->d[i][m], w, r);
            Lu::load(sb + 5*NU*EB, i + NN*k + N*m, el, w);
            fma5(line->d[j][m], w, r);
            Lu::load(sb + 10*NU*EB, i + N*j + NN*m, el, w);
            fma5(line->d[k][m], w, r);
        }
        T *pd = a.dv + pt*a.ldd + col;
        if (ok)
#pragma unroll
            for (int v = 0; v < 5; ++v) pd[v*SOA] = r[v];
    }
}

// ---------------------------------------------------------------------------
// Dispatch
// ---------------------------------------------------------------------------

template <typename T, int N>
static int hex_line_upload(HexPlan *p, const double *d, const double *hl,
                           const double *hr, const double *ll,
                           const double *lr, const double *x)
{
    HexLine<T, N> h;
    for (int i = 0; i < N; ++i) {
        for (int m = 0; m < N; ++m) h.d[i][m] = (T)d[i*N + m];
        h.hl[i] = (T)hl[i];
        h.hr[i] = (T)hr[i];
        h.ll[i] = (T)ll[i];
        h.lr[i] = (T)lr[i];
        h.x[i] = (T)x[i];
    }
    FR_HIP(hipMalloc(&p->line, sizeof(h)));
    FR_HIP(hipMemcpy(p->line, &h, sizeof(h), hipMemcpyHostToDevice));
    return 0;
}

template <typename T, int N, int GEO>
static int hex_div_launch(const HexPlan *p, const HexDivArgs<T> &a,
                          hipStream_t s)
{
    constexpr int EB = hex_eb<T, N>(), EBS = hex_eb_short<T, N>();
    const int eb = cdiv(a.neles, EB) < 256 ? EBS : EB;
    const dim3 grid(cdiv(a.neles, eb)), block(N*N*eb);
    const auto *line = static_cast<const HexLine<T, N> *>(p->line);
#define FR_FAM(F)                                                           \
    case F: {                                                               \
        auto k = eb == EB ? k_hex_div<T, N, GEO, F, EB>                     \
                          : k_hex_div<T, N, GEO, F, EBS>;                   \
        hipLaunchKernelGGL(k, grid, block, 0, s, line, a);                  \
        break;                                                              \
    }
    switch (hex_family(a.ep)) {
        FR_FAM(HEX_STORE) FR_FAM(HEX_RK45) FR_FAM(HEX_RK4)
        default:
            if constexpr (sizeof(T) == 4)
                switch (hex_family(a.ep)) {
                    FR_FAM(HEX_RK45M) FR_FAM(HEX_RK4M)
                }
    }
#undef FR_FAM
    FR_LAUNCHED();
    return 0;
}

template <typename T, int N>
static int hex_div_n(const HexPlan *p, int geo, const HexDivArgs<T> &a,
                     hipStream_t s)
{
    if constexpr (N > 2)
        if (geo == FRHIP_GEO_HEX_LINEAR)
            return hex_div_launch<T, N, FRHIP_GEO_HEX_LINEAR>(p, a, s);
    return geo < 0 ? hex_div_launch<T, N, -1>(p, a, s)
                   : hex_div_launch<T, N, FRHIP_GEO_CURVED>(p, a, s);
}

template <typename T>
static int hex_div_t(const HexPlan *p, int geo, int neles, const void *u,
                     long ldu, const void *gm, long ldg, void *f, long ldf,
                     void *c, long ldc, int ep, const void *rcp, long ldr,
                     void *xa, double dta, double dtb, int disu, double gamma,
                     const double *base, hipStream_t s)
{
    const HexDivArgs<T> a{neles, (const T *)u, ldu, (const T *)gm, ldg,
                          (T *)f, ldf, (T *)c, ldc, (const T *)rcp, ldr, xa,
                          dta, dtb, ep, disu, (T)(gamma - 1),
                          base ? base_state<T>(base, gamma) : BaseState<T>{}};
    switch (p->n) {
        case 2: return hex_div_n<T, 2>(p, geo, a, s);
        case 3: return hex_div_n<T, 3>(p, geo, a, s);
        case 4: return hex_div_n<T, 4>(p, geo, a, s);
        default: return hex_div_n<T, 5>(p, geo, a, s);
    }
}

// Elements per block of k_hex_nsvol: about 512 threads, so that two blocks
// share a CU and one computes while the other loads (a wavefront holds 128
// registers, a block 80 KB of LDS at p = 3 in FP64).  RK45 steps, 48^3 p = 3
// FP64 with 8 / 4 elements 7.01 / 7.52 ms; 30^3 p = 4 FP64 3.66 / 3.38.
template <typename T, int N>
constexpr int hex_ns_eb()
{
    return N == 2 ? 64 : N == 3 ? 16 : N == 4 ? (sizeof(T) == 8 ? 8 : 16)
                                              : (sizeof(T) == 8 ? 4 : 8);
}

template <typename T, int N>
static int hex_ns_n(const HexPlan *p, int geo, int nfv, const HexNsArgs<T> &a,
                    hipStream_t s)
{
    constexpr int EB = hex_ns_eb<T, N>();
    const dim3 grid(cdiv(a.neles, EB)), block(N*N*N*EB);
    const auto *line = static_cast<const HexLine<T, N> *>(p->line);
    auto k = k_hex_nsvol<T, N, FRHIP_GEO_CURVED, false, EB>;
    if constexpr (N > 2)
        if (geo == FRHIP_GEO_HEX_LINEAR)
            k = nfv ? k_hex_nsvol<T, N, FRHIP_GEO_HEX_LINEAR, true, EB>
                    : k_hex_nsvol<T, N, FRHIP_GEO_HEX_LINEAR, false, EB>;
    hipLaunchKernelGGL(k, grid, block, 0, s, line, a);
    FR_LAUNCHED();
    return 0;
}

template <typename T>
static int hex_ns_t(const HexPlan *p, int geo, int nfv, int neles,
                    const void *u, long ldu, const void *cm, long ldcm,
                    const void *gm, long ldg, const void *rcp, long ldr,
                    void *dv, long ldd, void *g, long ldgr, const void *fn,
                    const double *consts, const double *base, hipStream_t s)
{
    const HexNsArgs<T> a{neles, (const T *)u, ldu, (const T *)cm, ldcm,
                         (const T *)gm, ldg, (const T *)rcp, ldr,
                         (const T *)fn, (T *)dv, ldd, (T *)g, ldgr,
                         ns_consts<T>(consts, -1.0),
                         base ? base_state<T>(base, consts[0])
                              : BaseState<T>{}};
    switch (p->n) {
        case 2: return hex_ns_n<T, 2>(p, geo, nfv, a, s);
        case 3: return hex_ns_n<T, 3>(p, geo, nfv, a, s);
        case 4: return hex_ns_n<T, 4>(p, geo, nfv, a, s);
        default: return hex_ns_n<T, 5>(p, geo, nfv, a, s);
    }
}

}  // namespace frhip

using namespace frhip;

extern "C" {

int frhip_hex_plan_create(void **plan, int n, const double *d,
                          const double *hl, const double *hr,
                          const double *ll, const double *lr,
                          const double *x, int dtype)
{
    FR_API_BEGIN
    FR_CHECK(plan && d && hl && hr && ll && lr && x, "null argument");
    FR_CHECK(n >= 2 && n <= 5, "line operators of 2..5 points");
    FR_DTYPE_OK(dtype);
    HexPlan *p = new HexPlan{n, dtype, nullptr};
    int rc = 0;
#define FR_N(NV)                                                            \
    case NV:                                                                \
        rc = dtype == FRHIP_F64                                             \
            ? hex_line_upload<double, NV>(p, d, hl, hr, ll, lr, x)          \
            : hex_line_upload<float, NV>(p, d, hl, hr, ll, lr, x);          \
        break;
    switch (n) { FR_N(2) FR_N(3) FR_N(4) FR_N(5) }
#undef FR_N
    if (rc) {
        frhip_hex_plan_destroy(p);
        return rc;
    }
    *plan = p;
    return 0;
    FR_API_END
}

int frhip_hex_plan_destroy(void *plan)
{
    FR_API_BEGIN
    HexPlan *p = static_cast<HexPlan *>(plan);
    if (p) {
        if (p->line) (void)hipFree(p->line);
        delete p;
    }
    return 0;
    FR_API_END
}

int frhip_hex_div(void *plan, int geo, int neles, const void *u, long ldu,
                  const void *gm, long ldg, void *f, long ldf, void *c,
                  long ldc, int ep, const void *rcp, long ldr, void *xa,
                  double dta, double dtb, int last, int disu, double gamma,
                  const double *base, void *stream)
{
    FR_API_BEGIN
    HexPlan *p = static_cast<HexPlan *>(plan);
    FR_CHECK(p && u && f && c && rcp, "null argument");
    // p = 1 hexes take their stored metric, as in the reference (pyfr/
    // solvers/base/elements.py:224-227)
    FR_CHECK(geo >= -1 && geo <= (p->n > 2) && (geo < 0 || gm),
             "invalid geometry mode");
    FR_CHECK((ep >= 1 && ep <= 3) || (ep >= 10 && ep <= 17),
             "invalid epilogue");
    FR_CHECK(p->dtype == FRHIP_F32 || (ep != 3 && ep < 14),
             "the precision form's epilogues need FP32 operands");
    FR_CHECK(ep < 2 || xa, "RK epilogue needs the r1 / accumulator array");
    FR_CHECK(neles >= 0, "invalid extents");
    // the last block's lanes past neles read (and drop) whole blocks of 64
    const long ncol = 320L*((neles + 63L)/64);
    FR_CHECK(ldu >= ncol && ldf >= ncol && ldc >= ncol &&
             (geo < 0 || ldg*5 >= ncol*3) && ldr*5 >= ncol,
             "invalid leading dimensions");
    // lane offsets are 32-bit byte offsets of up to n^2 rows
    const size_t esz = p->dtype == FRHIP_F64 ? 8 : 4;
    const long ldmax = std::max({ldu, ldf, ldc, ldg, ldr});
    FR_CHECK((size_t)(p->n*p->n*ldmax)*(ep == 3 || ep >= 14 ? 8 : esz) <
                 (size_t)1 << 32, "leading dimension too large");
    FR_CHECK(!disu || (ep >= 2 && !(last && ep <= 3)),
             "no next stage to take the traces of");
    if (neles == 0) return 0;
    const int epi = (ep >= 2 && ep <= 3 && last) ? ep + 2 : ep;
    hipStream_t s = as_stream(stream);
    return p->dtype == FRHIP_F64
        ? hex_div_t<double>(p, geo, neles, u, ldu, gm, ldg, f, ldf, c, ldc,
                            epi, rcp, ldr, xa, dta, dtb, disu, gamma, base, s)
        : hex_div_t<float>(p, geo, neles, u, ldu, gm, ldg, f, ldf, c, ldc,
                           epi, rcp, ldr, xa, dta, dtb, disu, gamma, base, s);
    FR_API_END
}

int frhip_hex_nsvol(void *plan, int geo, int neles, const void *u, long ldu,
                    const void *cm, long ldcm, const void *gm, long ldg,
                    const void *rcp, long ldr, void *dv, long ldd, void *g,
                    long ldgr, int nfv, const void *fn, const double *consts,
                    const double *base, void *stream)
{
    FR_API_BEGIN
    HexPlan *p = static_cast<HexPlan *>(plan);
    FR_CHECK(p && u && cm && gm && dv && g && consts, "null argument");
    FR_CHECK((geo == FRHIP_GEO_HEX_LINEAR && p->n > 2) ||
             (geo == FRHIP_GEO_CURVED && rcp && !nfv),
             "invalid geometry mode");
    FR_CHECK(!nfv || fn || p->dtype == FRHIP_F64,
             "normal viscous fluxes in FP32 need the faces' normals");
    FR_CHECK(neles >= 0, "invalid extents");
    const long ncol = 320L*((neles + 63L)/64);
    FR_CHECK(ldu >= ncol && ldcm >= ncol && ldd >= ncol && ldgr >= ncol &&
             ldg*5 >= ncol*3 && (geo != FRHIP_GEO_CURVED || ldr*5 >= ncol),
             "invalid leading dimensions");
    // the vertices of a lane are addressed by 32-bit byte offsets
    FR_CHECK((size_t)(neles + 63)*24 < (size_t)1 << 32, "too many elements");
    if (neles == 0) return 0;
    hipStream_t s = as_stream(stream);
    return p->dtype == FRHIP_F64
        ? hex_ns_t<double>(p, geo, nfv, neles, u, ldu, cm, ldcm, gm, ldg, rcp,
                           ldr, dv, ldd, g, ldgr, fn, consts, base, s)
        : hex_ns_t<float>(p, geo, nfv, neles, u, ldu, cm, ldcm, gm, ldg, rcp,
                          ldr, dv, ldd, g, ldgr, fn, consts, base, s);
    FR_API_END
}

}  // extern "C"
