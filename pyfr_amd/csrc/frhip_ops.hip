// Operator application (the `mul` provider of the C ABI).
//
// Replaces HIPGiMMiKKernels.mul (pyfr/backends/hip/gimmik.py:24-117) and
// HIPRocBLASKernels.mul (pyfr/backends/hip/rocblas.py:93-192):
//   C(m, ncol) = alpha * A(m, k) @ B(k, ncol) + beta * C.
// Plans match A's nonzero pattern and values (bit for bit) against the
// structured kernels generated by gen_ops.py; anything else is a dense plan
// (frhip_dense.hip: matrix-core or scalar kernel, picked by the tuner).
#include "frhip_dense.h"
#include "frhip_opk.h"

#include <cstring>
#include <vector>

namespace frhip {

struct MulPlan {
    int m, k, dtype, kind;          // kind: 1 structured, 2 dense, 3 bf16
    const OpKernelEntry *ent;
    void *dvals;                    // nonzeros (structured)
    DensePlan *dense;
    Bf16Plan *bf16;
};

static int bmode_of(double alpha, double beta)
{
    if (alpha == 1.0 && beta == 0.0) return 0;
    if (alpha == 1.0 && beta == 1.0) return 1;
    if (beta == 0.0) return 3;
    return 2;
}

}  // namespace frhip

using namespace frhip;

extern "C" {

int frhip_mul_plan_create(void **plan, int m, int k, const double *a_host,
                          int dtype, int *kind)
{
    FR_API_BEGIN
    FR_CHECK(plan && a_host, "null argument");
    FR_CHECK(m > 0 && k > 0, "invalid operator shape");
    FR_CHECK(dtype == FRHIP_F64 || dtype == FRHIP_F32 ||
             dtype == FRHIP_F32_BF16OPS, "invalid dtype");
    if (dtype == FRHIP_F32_BF16OPS) {
        Bf16Plan *b = nullptr;
        if (int rc = bf16_plan_create(&b, m, k, 0, a_host, nullptr))
            return rc;
        *plan = new MulPlan{m, k, FRHIP_F32, 3, nullptr, nullptr, nullptr, b};
        if (kind) *kind = 3;
        return 0;
    }

    std::vector<int32_t> lin;
    for (long i = 0; i < (long)m*k; ++i)
        if (a_host[i] != 0.0) lin.push_back((int32_t)i);

    const OpKernelEntry *ent = nullptr;
    for (int t = 0; t < g_opk_count; ++t) {
        const OpKernelEntry &e = g_opk_table[t];
        if (e.m == m && e.k == k && e.nnz == (int)lin.size() &&
            std::memcmp(e.lin, lin.data(), lin.size()*sizeof(int32_t)) == 0) {
            bool same = true;
            for (size_t i = 0; i < lin.size() && same; ++i)
                same = e.vals[i] == a_host[lin[i]];
            if (same) {
                ent = &e;
                break;
            }
        }
    }

    if (!ent) {
        DensePlan *d = nullptr;
        if (int rc = dense_plan_create(&d, m, k, 0, a_host, nullptr, dtype))
            return rc;
        *plan = new MulPlan{m, k, dtype, 2, nullptr, nullptr, d, nullptr};
        if (kind) *kind = 2;
        return 0;
    }

    const size_t esz = dtype == FRHIP_F64 ? 8 : 4;
    const size_t nv = lin.size();
    std::vector<char> hv(nv*esz);
    for (size_t i = 0; i < nv; ++i) {
        double v = a_host[lin[i]];
        if (dtype == FRHIP_F64) std::memcpy(&hv[i*8], &v, 8);
        else { float f = (float)v; std::memcpy(&hv[i*4], &f, 4); }
    }

    void *dv = nullptr;
    FR_HIP(hipMalloc(&dv, hv.size() ? hv.size() : 8));
    hipError_t e = hipMemcpy(dv, hv.data(), hv.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(dv);
        FR_HIP(e);
    }

    *plan = new MulPlan{m, k, dtype, 1, ent, dv, nullptr, nullptr};
    if (kind) *kind = 1;
    return 0;
    FR_API_END
}

int frhip_mul_plan_tune(void *plan, int ncol, const void *b, long ldb,
                        int reps, int *variant)
{
    FR_API_BEGIN
    MulPlan *p = static_cast<MulPlan *>(plan);
    FR_CHECK(p, "null plan");
    if (p->kind != 2) {
        if (variant) *variant = -1;
        return 0;
    }
    return dense_tune(p->dense, ncol, b, ldb, nullptr, 0, reps, variant);
    FR_API_END
}

int frhip_mul_plan_destroy(void *plan)
{
    FR_API_BEGIN
    MulPlan *p = static_cast<MulPlan *>(plan);
    if (p) {
        if (p->dvals) (void)hipFree(p->dvals);
        dense_plan_destroy(p->dense);
        bf16_plan_destroy(p->bf16);
        delete p;
    }
    return 0;
    FR_API_END
}

int frhip_mul_slabs(void *plan, int n, int ncol, const void *b, long ldb,
                    long sb, void *c, long ldc, long sc, void *stream)
{
    FR_API_BEGIN
    MulPlan *p = static_cast<MulPlan *>(plan);
    FR_CHECK(p, "null plan");
    FR_CHECK(n >= 0 && n <= 65535 && sb >= 0 && sc >= 0,
             "invalid mul slabs");
    FR_CHECK(ncol >= 0 && ldb >= ncol && ldc >= ncol, "invalid mul extents");
    if (ncol == 0 || n == 0) return 0;
    if (p->kind == 2)
        return dense_launch(p->dense, 0, ncol, b, ldb, nullptr, 0, c, ldc,
                            nullptr, 0, 1, nullptr, 0, 0, 1.0, 0.0,
                            as_stream(stream), {n, sb, sc});
    const long esz = p->dtype == FRHIP_F64 ? 8 : 4;
    for (int i = 0; i < n; ++i) {
        const int rc = frhip_mul(p, ncol, (const char *)b + i*sb*esz, ldb,
                                 (char *)c + i*sc*esz, ldc, 1.0, 0.0,
                                 stream);
        if (rc) return rc;
    }
    return 0;
    FR_API_END
}

int frhip_mul(void *plan, int ncol, const void *b, long ldb, void *c,
              long ldc, double alpha, double beta, void *stream)
{
    FR_API_BEGIN
    MulPlan *p = static_cast<MulPlan *>(plan);
    FR_CHECK(p, "null plan");
    FR_CHECK(ncol >= 0 && ldb >= ncol && ldc >= ncol, "invalid mul extents");
    if (ncol == 0) return 0;
    const int bm = bmode_of(alpha, beta);
    hipStream_t s = as_stream(stream);
    static const int ep_of_bm[4] = {0, 6, 7, 8};
    if (p->kind == 2)
        return dense_launch(p->dense, ep_of_bm[bm], ncol, b, ldb, nullptr, 0,
                            c, ldc, nullptr, 0, 1, nullptr, 0, 0, alpha,
                            beta, s);
    if (p->kind == 3)
        return bf16_launch(p->bf16, ep_of_bm[bm], ncol, b, ldb, nullptr, 0,
                           c, ldc, nullptr, 0, 1, nullptr, 0, 0, alpha, beta,
                           s);
    dim3 grid(cdiv(ncol, 256)), block(256);
    if (p->dtype == FRHIP_F64)
        hipLaunchKernelGGL(p->ent->fd[bm], grid, block, 0, s, ncol,
                           (const double *)b, ldb, (double *)c, ldc,
                           (const double *)p->dvals, alpha, beta);
    else
        hipLaunchKernelGGL(p->ent->ff[bm], grid, block, 0, s, ncol,
                           (const float *)b, ldb, (float *)c, ldc,
                           (const float *)p->dvals, (float)alpha,
                           (float)beta);
    FR_LAUNCHED();
    return 0;
    FR_API_END
}

// ---- fused two-input operator kernels ------------------------------------

namespace frhip {
struct Mul2Plan {
    int m, k0, k1, dtype;
    const FusedKernelEntry *ent;   // structured, or
    DensePlan *dense;              // dense, or
    Bf16Plan *bf16;                // BF16 operands
};
}

int frhip_mul2_plan_create(void **plan, int m, int k0, int k1,
                           const double *a0, const double *a1, int dtype,
                           int *kind)
{
    FR_API_BEGIN
    FR_CHECK(plan && a0 && a1 && kind, "null argument");
    FR_CHECK(m > 0 && k0 > 0 && k1 > 0, "invalid operator shape");
    FR_CHECK(dtype == FRHIP_F64 || dtype == FRHIP_F32 ||
             dtype == FRHIP_F32_BF16OPS, "invalid dtype");
    if (dtype == FRHIP_F32_BF16OPS) {
        Bf16Plan *b = nullptr;
        if (int rc = bf16_plan_create(&b, m, k0, k1, a0, a1)) return rc;
        *plan = new Mul2Plan{m, k0, k1, FRHIP_F32, nullptr, nullptr, b};
        *kind = 3;
        return 0;
    }
    const int k = k0 + k1;
    std::vector<int32_t> lin;
    std::vector<double> val;
    for (int r = 0; r < m; ++r)
        for (int q = 0; q < k; ++q) {
            const double v = q < k0 ? a0[(long)r*k0 + q]
                                    : a1[(long)r*k1 + q - k0];
            if (v != 0.0) {
                lin.push_back(r*k + q);
                val.push_back(v);
            }
        }
    const FusedKernelEntry *ent = nullptr;
    for (int t = 0; t < g_fk_count && !ent; ++t) {
        const FusedKernelEntry &e = g_fk_table[t];
        if (e.m != m || e.k0 != k0 || e.k1 != k1 || e.nnz != (int)lin.size())
            continue;
        if (std::memcmp(e.lin, lin.data(), lin.size()*sizeof(int32_t)))
            continue;
        bool same = true;
        for (size_t i = 0; i < val.size() && same; ++i)
            same = e.vals[i] == val[i];
        if (same) ent = &e;
    }
    DensePlan *d = nullptr;
    if (!ent)
        if (int rc = dense_plan_create(&d, m, k0, k1, a0, a1, dtype))
            return rc;
    *plan = new Mul2Plan{m, k0, k1, dtype, ent, d, nullptr};
    *kind = ent ? 1 : 2;
    return 0;
    FR_API_END
}

int frhip_mul2_plan_tune(void *plan, int ncol, const void *b0, long ld0,
                         const void *b1, long ld1, int reps, int *variant)
{
    FR_API_BEGIN
    Mul2Plan *p = static_cast<Mul2Plan *>(plan);
    FR_CHECK(p, "null plan");
    if (!p->dense) {
        if (variant) *variant = -1;
        return 0;
    }
    return dense_tune(p->dense, ncol, b0, ld0, b1, ld1, reps, variant);
    FR_API_END
}

int frhip_mul_plan_set_variant(void *plan, int variant)
{
    FR_API_BEGIN
    MulPlan *p = static_cast<MulPlan *>(plan);
    FR_CHECK(p && p->kind == 2, "not a dense plan");
    FR_CHECK(dense_variant_ok(p->dense, variant), "invalid variant");
    p->dense->variant = variant;
    return 0;
    FR_API_END
}

int frhip_mul2_plan_set_variant(void *plan, int variant)
{
    FR_API_BEGIN
    Mul2Plan *p = static_cast<Mul2Plan *>(plan);
    FR_CHECK(p && p->dense, "not a dense plan");
    FR_CHECK(dense_variant_ok(p->dense, variant), "invalid variant");
    p->dense->variant = variant;
    return 0;
    FR_API_END
}

int frhip_mul2_plan_destroy(void *plan)
{
    FR_API_BEGIN
    Mul2Plan *p = static_cast<Mul2Plan *>(plan);
    if (p) {
        dense_plan_destroy(p->dense);
        bf16_plan_destroy(p->bf16);
        delete p;
    }
    return 0;
    FR_API_END
}

int frhip_mul2(void *plan, int ncol, const void *b0, long ld0, const void *b1,
               long ld1, void *c, long ldc, int ep, const void *rcp, long ldr,
               void *xa, double dta, double dtb, int last, void *stream)
{
    FR_API_BEGIN
    Mul2Plan *p = static_cast<Mul2Plan *>(plan);
    FR_CHECK(p && (p->ent || p->dense || p->bf16), "null plan");
    FR_CHECK((ep >= 0 && ep <= 3) || (ep >= 10 && ep <= 17) ||
             (ep >= 20 && ep <= 23), "invalid epilogue");
    FR_CHECK(ep < 10 || p->ent,
             "RK4 stage epilogues need a structured (generated) plan");
    FR_CHECK(ep < 14 || ep > 17 || p->dtype == FRHIP_F32,
             "the mixed RK4 epilogues need FP32 operands");
    FR_CHECK(ep < 20 || p->dtype == FRHIP_F64,
             "the per-element RK4 epilogues are built for FP64");
    FR_CHECK(ep == 0 || rcp, "epilogue needs 1/|J|");
    FR_CHECK(ep < 2 || xa, "RK epilogue needs the r1 / accumulator array");
    FR_CHECK(ep != 3 || p->dtype == FRHIP_F32,
             "the mixed RK epilogue needs FP32 operands");
    FR_CHECK(ncol >= 0 && ncol % (64*5) == 0,
             "ncol must cover whole 64-element SoA blocks of 5 variables");
    FR_CHECK(ld0 >= ncol && ld1 >= ncol && ldc >= ncol,
             "invalid leading dimensions");
    if (ncol == 0) return 0;
    // the last RK45 stage is its own instantiation
    const int epi = (ep >= 2 && ep <= 3 && last) ? ep + 2 : ep;
    hipStream_t s = as_stream(stream);
    if (p->dense)
        return dense_launch(p->dense, epi, ncol, b0, ld0, b1, ld1, c, ldc,
                            rcp, ldr, 5, xa, dta, dtb, 1, 0, s);
    if (p->bf16)
        return bf16_launch(p->bf16, epi, ncol, b0, ld0, b1, ld1, c, ldc, rcp,
                           ldr, 5, xa, dta, dtb, 1, 0, s);
    dim3 grid(cdiv(ncol, 256)), block(256);
    const int slot = epi >= 20 ? epi - 6 : epi >= 10 ? epi - 4 : epi;
    FR_CHECK(p->dtype == FRHIP_F64 ? p->ent->fd[slot] != nullptr
                                   : p->ent->ff[slot] != nullptr,
             "epilogue not built for this kernel");
    if (p->dtype == FRHIP_F64)
        hipLaunchKernelGGL(p->ent->fd[slot], grid, block, 0, s, ncol,
                           (const double *)b0, ld0, (const double *)b1, ld1,
                           (double *)c, ldc, (const double *)rcp, ldr, xa,
                           dta, dtb, last);
    else
        hipLaunchKernelGGL(p->ent->ff[slot], grid, block, 0, s, ncol,
                           (const float *)b0, ld0, (const float *)b1, ld1,
                           (float *)c, ldc, (const float *)rcp, ldr, xa, dta,
                           dtb, last);
    FR_LAUNCHED();
    return 0;
    FR_API_END
}

}  // extern "C"
