// plain.hip -- the plain FP64 method: element kernels that write the values of
// the COO stream in Elfel's order, and the matrix built from it by row buckets
// (bucket.hip), or by the stable sort and in-order segmented reduce (sort.hip)
// where those do not apply.  Compiled with -ffp-contract=off so every product
// and sum rounds exactly like the reference's unfused Julia arithmetic.
//
// COO stream order (what SysmatAssemblerSparse's append! produces):
//   per element, in element order (for el in elit, src/FEIterators.jl:92-98),
//   the element block column-major (LocalMatrixAssembler init!,
//   src/LocalAssemblers.jl:68-83; assemble!, src/Assemblers.jl:97-102);
//   Stokes adds kup column-major and transpose(kup) row-major of kup
//   (src/Assemblers.jl:109-114), as test/test_stokes.jl:654-656 does.
#include <string.h>

#include "elem.h"

// ---- element kernel: the values of the COO stream, in stream order ----------
// A workgroup takes EB elements.  First a work-item per (element, point) leaves
// the spatial gradients and JxW in LDS; then a work-item per (element, column of
// the block) forms the column's ND values and stores them side by side, so that
// a wavefront writes one contiguous range and the L2 lines are full before they
// leave it.  (One work-item per element, its whole block and the sort keys
// stored a value at a time 1152 bytes apart: elasticity T6 200^2 199 us, 0.9 TB/s
// written; this kernel writes no keys and takes 41 us, 2.2 TB/s.)  The last items of an
// element are the load vector (heat) or the coupling block and its transpose
// (Stokes, ND values each).
template <int KIND, int NEN, int NC, int NQ>
struct ElemVals {
    static constexpr int ND = NEN * NC;
    static constexpr bool STOKES = KIND == ELFEL_STOKES_GEN || KIND == ELFEL_STOKES_VECLAP;
    static constexpr bool HEAT = KIND == ELFEL_HEAT;
    static constexpr int NBLK = ND * ND + (STOKES ? 2 * ND * 3 : 0);
    static constexpr int ITEMS = ND + (STOKES ? 6 : 0) + (HEAT ? 1 : 0);
    static constexpr int EB = NQ == 1 ? 256 : 64;
    static constexpr int GS = (2 * NEN * NQ + NQ) | 1;  // words an element, odd against bank conflicts
};

template <int KIND, int NEN, int NC, int NQ>
__global__ __launch_bounds__(256) void k_elem_vals(int64_t E, const int32_t *__restrict__ conn,
                                                   const double2 *__restrict__ xy, Coef cf, QTable tab,
                                                   double *__restrict__ vals, double *__restrict__ fvals)
{
    using V = ElemVals<KIND, NEN, NC, NQ>;
    constexpr int ND = V::ND, EB = V::EB, GS = V::GS;
    __shared__ double sg[EB * GS];  // per element: gx[q][k], gy[q][k], jxw[q]
    const int64_t e0 = (int64_t)blockIdx.x * EB;
    for (int x = threadIdx.x; x < EB * NQ; x += 256) {
        const int el = x % EB, q = __builtin_amdgcn_readfirstlane(x / EB);  // EB is a multiple of the wave
        const int64_t e = e0 + el;
        if (e >= E) continue;
        double X[NEN], Y[NEN], gx[NEN], gy[NEN], jxw, det;
#pragma unroll
        for (int k = 0; k < NEN; k++) {
            const double2 p = xy[conn[e * NEN + k]];
            X[k] = p.x; Y[k] = p.y;
        }
        geometry_at<double, NEN>(tab, q, X, Y, gx, gy, jxw, det);
        double *g = sg + el * GS;
#pragma unroll
        for (int k = 0; k < NEN; k++) {
            g[q * NEN + k] = gx[k];
            g[(NQ + q) * NEN + k] = gy[k];
        }
        g[2 * NQ * NEN + q] = jxw;
    }
    __syncthreads();
    for (int x = threadIdx.x; x < EB * V::ITEMS; x += 256) {
        const int el = x / V::ITEMS, it = x - el * V::ITEMS;
        const int64_t e = e0 + el;
        if (e >= E) break;
        const double *sge = sg + el * GS;
        Geo<double, NEN, NQ> g;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
#pragma unroll
            for (int k = 0; k < NEN; k++) {
                g.gx[q][k] = sge[q * NEN + k];
                g.gy[q][k] = sge[(NQ + q) * NEN + k];
            }
            g.jxw[q] = sge[2 * NQ * NEN + q];
        }
        double v[ND];
        double *dst = vals + e * V::NBLK + it * ND;
        if (it < ND) {
            const int bj = it / NC, cj = it - bj * NC;
            double gxj[NQ], gyj[NQ];
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                gxj[q] = sge[q * NEN + bj];
                gyj[q] = sge[(NQ + q) * NEN + bj];
            }
            if constexpr (KIND == ELFEL_HEAT) {
                const double kap = cf.kappa_e ? cf.kappa_e[padded(e, cf.cgap)] : cf.kappa;
#pragma unroll
                for (int i = 0; i < ND; i++) {
                    double acc = 0.0;
#pragma unroll
                    for (int q = 0; q < NQ; q++)
                        acc += (g.gx[q][i] * gxj[q] + g.gy[q][i] * gyj[q]) * (kap * g.jxw[q]);
                    v[i] = acc;
                }
            } else if constexpr (KIND == ELFEL_ELAST || KIND == ELFEL_STOKES_GEN) {
                const double sc = cf.scale_e ? cf.scale_e[padded(e, cf.cgap)] : 1.0;
                double D[9], db[NQ][3];
#pragma unroll
                for (int i = 0; i < 9; i++) D[i] = cf.scale_e ? sc * cf.D[i] : cf.D[i];
#pragma unroll
                for (int q = 0; q < NQ; q++) dmul_b<double>(D, gxj[q], gyj[q], cj, db[q]);
#pragma unroll
                for (int i = 0; i < ND; i++) {
                    double acc = 0.0;
#pragma unroll
                    for (int q = 0; q < NQ; q++)
                        acc += dot_b<double>(db[q], g.gx[q][i / NC], g.gy[q][i / NC], i % NC) * g.jxw[q];
                    v[i] = acc;
                }
            } else {
#pragma unroll
                for (int i = 0; i < ND; i++) {
                    double acc = 0.0;
#pragma unroll
                    for (int q = 0; q < NQ; q++)
                        acc += (cf.mu * g.jxw[q]) * (g.gx[q][i / NC] * gxj[q] + g.gy[q][i / NC] * gyj[q]);
                    v[i] = (i % NC) == cj ? acc : 0.0;
                }
            }
        } else if constexpr (V::HEAT) {
            if (!fvals) continue;
            const double Qe = cf.Q_e ? cf.Q_e[padded(e, cf.cgap)] : cf.Q;
#pragma unroll
            for (int j = 0; j < ND; j++) v[j] = fe_value<double, NEN, NQ>(tab, g, Qe, j);
            dst = fvals + e * ND;
        } else if constexpr (V::STOKES) {
            if (it < ND + 3) {  // kup, column jp
                const int jp = it - ND;
                double np[NQ];
#pragma unroll
                for (int q = 0; q < NQ; q++) np[q] = jp == 0 ? tab.Np[q][0] : jp == 1 ? tab.Np[q][1] : tab.Np[q][2];
#pragma unroll
                for (int i = 0; i < ND; i++) {
                    double acc = 0.0;
#pragma unroll
                    for (int q = 0; q < NQ; q++) {
                        const double gi = (i % NC) == 0 ? g.gx[q][i / NC] : g.gy[q][i / NC];
                        acc += (-g.jxw[q] * np[q]) * gi;
                    }
                    v[i] = acc;
                }
            } else {  // its transpose: rows b of kup, ND / 3 of them
                const int b0 = (it - ND - 3) * (ND / 3);
#pragma unroll
                for (int bb = 0; bb < ND / 3; bb++) {
                    const int b = b0 + bb;
#pragma unroll
                    for (int a = 0; a < 3; a++) {
                        double acc = 0.0;
#pragma unroll
                        for (int q = 0; q < NQ; q++) {
                            const double gi = (b % NC) == 0 ? sge[q * NEN + b / NC] : sge[(NQ + q) * NEN + b / NC];
                            acc += (-g.jxw[q] * tab.Np[q][a]) * gi;
                        }
                        v[bb * 3 + a] = acc;
                    }
                }
            }
        }
        if constexpr (ND % 2 == 0) {
#pragma unroll
            for (int i = 0; i < ND; i += 2) *(double2 *)(dst + i) = make_double2(v[i], v[i + 1]);
        } else {
#pragma unroll
            for (int i = 0; i < ND; i++) dst[i] = v[i];
        }
    }
}

// ---- generic COO (host stream) -> keys with range check --------------------
__global__ void k_coo_keys(const int64_t *__restrict__ I, const int64_t *__restrict__ J, int64_t n, int64_t nrow,
                           int64_t ncol, int minor_bits, int csc, uint64_t *__restrict__ keys, int *__restrict__ err)
{
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int64_t r = I[k], cc = J[k];
    if (r < 1 || r > nrow || cc < 1 || cc > ncol) {
        atomicOr(err, DERR_RANGE);
        r = 1; cc = 1;
    }
    const uint64_t mj = (uint64_t)(csc ? cc - 1 : r - 1), mn = (uint64_t)(csc ? r - 1 : cc - 1);
    keys[k] = (mj << minor_bits) | mn;
}

// the same for checked 0-based indices
__global__ void k_coo_keys32(const int32_t *__restrict__ I, const int32_t *__restrict__ J, int64_t n, int minor_bits, int csc,
                             uint64_t *__restrict__ keys)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint64_t r = (uint64_t)I[k], cc = (uint64_t)J[k];
    keys[k] = csc ? (cc << minor_bits) | r : (r << minor_bits) | cc;
}

__global__ void k_vec_keys(const int32_t *__restrict__ I, int64_t n, uint64_t *__restrict__ keys)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) keys[k] = (uint64_t)I[k];
}

// Host wrappers used for the generic drop-in.
int plain_coo_keys(elfel_hip_ctx *c, const int64_t *I, const int64_t *J, int64_t n, int64_t nrow, int64_t ncol,
                   int minor_bits, int csc, uint64_t *keys)
{
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_coo_keys, dim3(ceil_div(n, 256)), dim3(256), 0, c->stream, I, J, n, nrow, ncol, minor_bits,
                       csc, keys, (int *)c->dscal.p + 1);
    HIPCHK(c, hipGetLastError());
    return 0;
}

int plain_coo_keys32(elfel_hip_ctx *c, const int32_t *I, const int32_t *J, int64_t n, int minor_bits, int csc, uint64_t *keys)
{
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_coo_keys32, dim3(ceil_div(n, 256)), dim3(256), 0, c->stream, I, J, n, minor_bits, csc, keys);
    HIPCHK(c, hipGetLastError());
    return 0;
}

int plain_vec_keys(elfel_hip_ctx *c, const int32_t *I, int64_t n, uint64_t *keys)
{
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_vec_keys, dim3(ceil_div(n, 256)), dim3(256), 0, c->stream, I, n, keys);
    HIPCHK(c, hipGetLastError());
    return 0;
}

// ---- orchestration --------------------------------------------------------
template <int KIND, int NEN, int NC, int NQ>
static int launch_plain(elfel_hip_ctx *c, const QTable &tab, const Coef &cf, double *vals, double *fvals)
{
    const Field &F = c->f[0];
    const int64_t E = F.E;
    if (E == 0) return 0;  // no elements: an empty stream
    hipEvent_t ev = nullptr;
    tm_begin(c, ELFEL_PH_ELEMENT, &ev);
    hipLaunchKernelGGL((k_elem_vals<KIND, NEN, NC, NQ>), dim3(ceil_div(E, ElemVals<KIND, NEN, NC, NQ>::EB)), dim3(256), 0,
                       c->stream, E, (const int32_t *)F.conn.p, (const double2 *)F.xy.p, cf, tab, vals, fvals);
    HIPCHK(c, hipGetLastError());
    tm_end(c, ELFEL_PH_ELEMENT, ev);
    return 0;
}

typedef int (*plain_fn)(elfel_hip_ctx *, const QTable &, const Coef &, double *, double *);

static plain_fn pick_plain(int kind, int fe, int nq)
{
#define P(K, N, C, Q) return launch_plain<K, N, C, Q>
    if (kind == ELFEL_HEAT) {
        if (fe == ELFEL_T3 && nq == 1) P(ELFEL_HEAT, 3, 1, 1);
        if (fe == ELFEL_T3 && nq == 3) P(ELFEL_HEAT, 3, 1, 3);
        if (fe == ELFEL_T6 && nq == 3) P(ELFEL_HEAT, 6, 1, 3);
        if (fe == ELFEL_Q4 && nq == 1) P(ELFEL_HEAT, 4, 1, 1);
        if (fe == ELFEL_Q4 && nq == 4) P(ELFEL_HEAT, 4, 1, 4);
    } else if (kind == ELFEL_ELAST) {
        if (fe == ELFEL_T3 && nq == 1) P(ELFEL_ELAST, 3, 2, 1);
        if (fe == ELFEL_T3 && nq == 3) P(ELFEL_ELAST, 3, 2, 3);
        if (fe == ELFEL_T6 && nq == 3) P(ELFEL_ELAST, 6, 2, 3);
        if (fe == ELFEL_Q4 && nq == 4) P(ELFEL_ELAST, 4, 2, 4);
    } else if (kind == ELFEL_STOKES_GEN) {
        if (fe == ELFEL_T6 && nq == 3) P(ELFEL_STOKES_GEN, 6, 2, 3);
    } else if (kind == ELFEL_STOKES_VECLAP) {
        if (fe == ELFEL_T6 && nq == 3) P(ELFEL_STOKES_VECLAP, 6, 2, 3);
    }
#undef P
    return nullptr;
}

int sort_buffers(elfel_hip_ctx *c, int64_t n, int64_t nv, bool vec)
{
    int rc;
    if ((rc = ensure(c, c->keys[0], sizeof(uint64_t) * n)) || (rc = ensure(c, c->keys[1], sizeof(uint64_t) * n)) ||
        (rc = ensure(c, c->vals[0], sizeof(double) * n)) || (rc = ensure(c, c->vals[1], sizeof(double) * n)))
        return rc;
    if (vec) {
        if ((rc = ensure(c, c->fkeys[0], sizeof(uint64_t) * nv)) || (rc = ensure(c, c->fkeys[1], sizeof(uint64_t) * nv)) ||
            (rc = ensure(c, c->fvals[0], sizeof(double) * nv)) || (rc = ensure(c, c->fvals[1], sizeof(double) * nv)))
            return rc;
    }
    return 0;
}

// The sort of the stream whose values are in vals[0] (and fvals[0]).
static int build_by_sort(elfel_hip_ctx *c, const FormMap &m, int64_t E, const int32_t *edof, int64_t ndofs)
{
    const int64_t n = E * m.nmat, nv = E * m.nvec;
    const int minor_bits = bits_for(ndofs);
    const bool vec = m.nvec > 0;
    int rc = sort_buffers(c, n, nv, vec);
    if (rc) return rc;
    uint64_t *k0 = (uint64_t *)c->keys[0].p, *k1 = (uint64_t *)c->keys[1].p;
    uint64_t *v0 = (uint64_t *)c->vals[0].p, *v1 = (uint64_t *)c->vals[1].p;
    uint64_t *fk0 = vec ? (uint64_t *)c->fkeys[0].p : nullptr, *fk1 = vec ? (uint64_t *)c->fkeys[1].p : nullptr;
    uint64_t *fv0 = vec ? (uint64_t *)c->fvals[0].p : nullptr, *fv1 = vec ? (uint64_t *)c->fvals[1].p : nullptr;
    hipEvent_t ev = nullptr;
    tm_begin(c, ELFEL_PH_SORT, &ev);
    if ((rc = form_keys(c, m, E, edof, minor_bits, k0, fk0))) return rc;
    if ((rc = radix_sort_pairs(c, k0, v0, k1, v1, n, bits_for(ndofs) + minor_bits))) return rc;
    if (vec && (rc = radix_sort_pairs(c, fk0, fv0, fk1, fv1, nv, bits_for(ndofs)))) return rc;
    tm_end(c, ELFEL_PH_SORT, ev);
    tm_begin(c, ELFEL_PH_REDUCE, &ev);
    rc = build_csr_from_sorted(c, k0, (const double *)v0, n, minor_bits, ndofs, (int32_t *)c->ptr.p,
                               (int32_t *)c->ind.p, (double *)c->val.p, (int32_t *)c->dscal.p, true);
    if (rc) return rc;
    if (vec && (rc = build_dense_from_sorted(c, fk0, (const double *)fv0, nv, ndofs, (double *)c->F.p))) return rc;
    tm_end(c, ELFEL_PH_REDUCE, ev);
    return 0;
}

// Whether the rows of this problem's matrix fit the buckets' tiles depends on
// the mesh, the dof map and the weak form alone.  The first assembly on them
// waits for the answer and keeps it; later ones take the one way or the other
// without a wait.
int plain_build(elfel_hip_ctx *c, const elfel_hip_problem *pb, const FormMap &m, int64_t E, int64_t ndofs,
                const StreamElements &elements)
{
    const int64_t n = E * m.nmat, nv = E * m.nvec;
    const bool vec = m.nvec > 0;
    const uint64_t key[6] = {c->f[0].mesh_version, c->f[0].dof_version, c->f[0].edof_version,
                             c->f[1].mesh_version, c->f[1].dof_version, c->f[1].edof_version};
    auto &R = c->rows;
    const bool known = R.valid && R.kind == pb->kind && R.fe == pb->fe && R.fe_p == pb->fe_p && R.ndofs == ndofs &&
                       memcmp(R.key, key, sizeof key) == 0;
    bool buckets = bucket_form_takes(m, E, ndofs) && !(known && R.toolong);
    int rc;
    if ((rc = ensure(c, c->vals[0], 8 * n)) || (vec && (rc = ensure(c, c->fvals[0], 8 * nv))) ||
        (vec && (rc = ensure(c, c->F, 8 * ndofs))) || (rc = ensure(c, c->ptr, 4 * (ndofs + 1))) ||
        (rc = ensure(c, c->ind, 4 * n)) || (rc = ensure(c, c->val, 8 * n)) || (rc = ensure(c, c->geom, 4 * E * m.nd)) ||
        (buckets && (rc = ensure(c, c->keys[0], bucket_form_bytes(m, E, ndofs)))))
        return rc;
    int32_t *edof = (int32_t *)c->geom.p;
    hipEvent_t ev = nullptr;
    tm_begin(c, ELFEL_PH_GATHER, &ev);
    if ((rc = form_dofs(c, m, edof))) return rc;
    tm_end(c, ELFEL_PH_GATHER, ev);
    const StreamOut so{c->vals[0].p, vec ? c->fvals[0].p : nullptr};
    if ((rc = elements(so, false))) return rc;
    if (buckets) {
        const BucketOut o{(int32_t *)c->ptr.p, (int32_t *)c->ind.p, (double *)c->val.p, vec ? (double *)c->F.p : nullptr,
                          nullptr, nullptr, nullptr, nullptr};
        if ((rc = bucket_form(c, c->keys[0].p, m, E, edof, ndofs, (const double *)so.vals, (const double *)so.fvals, o)))
            return rc;
        if (!known) {
            HIPCHK(c, hipStreamSynchronize(c->stream));
            R.toolong = ((const int32_t *)c->told)[2] != 0;
            R.kind = pb->kind; R.fe = pb->fe; R.fe_p = pb->fe_p; R.ndofs = ndofs;
            memcpy(R.key, key, sizeof key);
            R.valid = true;
            buckets = !R.toolong;
        }
        c->nnz_told = buckets;
    }
    if (!buckets && (rc = build_by_sort(c, m, E, edof, ndofs))) return rc;
    c->has_F = vec;
    c->nF = vec ? ndofs : 0;
    c->nmaj = ndofs;
    c->nmin = ndofs;
    c->layout = pb->layout;
    c->result_src = RES_PLAIN;
    return 0;
}

// The stream of a 2D weak form: the block column-major; Stokes then kup
// column-major and transpose(kup) row-major of kup.
static void plain_map(const Field &F, const elfel_hip_problem *pb, FormMap &m)
{
    const bool stokes = pb->kind == ELFEL_STOKES_GEN || pb->kind == ELFEL_STOKES_VECLAP;
    const int csc = pb->layout == ELFEL_CSC ? 1 : 0;
    const int nu = F.nen * F.ncomp;
    if (!stokes) {
        form_square(m, nu, csc);
        m.nvec = pb->kind == ELFEL_HEAT ? nu : 0;
    } else {
        const int nd = nu + 3;
        m.nd = nd;
        m.nmat = nu * nu + 6 * nu;
        // entry (row i, column j) of the element block in stream order, -1: none
        auto at = [&](int i, int j) {
            if (i < nu && j < nu) return i + nu * j;
            if (i < nu) return nu * nu + (j - nu) * nu + i;
            if (j < nu) return nu * nu + 3 * nu + j * 3 + (i - nu);
            return -1;
        };
        for (int a = 0; a < nd; a++) {
            m.ncol[a] = (uint8_t)(a < nu ? nd : nu);
            for (int b = 0; b < nd; b++) m.pos[a * nd + b] = (int16_t)(csc ? at(b, a) : at(a, b));
        }
        for (int k = 0; k < 3; k++) m.src[nu + k] = {1, 0, (uint8_t)k, 0};
    }
    for (int i = 0; i < nu; i++) m.src[i] = {0, 0, (uint8_t)(i / F.ncomp), (uint8_t)(i % F.ncomp)};
}

// The 2D weak forms on the stream REUSE method (FP64): every entry is the sum
// of its run in the cached sort order.
int plain_stream_reuse(elfel_hip_ctx *c, const elfel_hip_problem *pb, const QTable &tab, const Coef &cf)
{
    const Field &F = c->f[0];
    plain_fn fn = pick_plain(pb->kind, pb->fe, tab.nq);
    if (!fn) return set_err(c, ELFEL_ENOTSUP, "unsupported (kind, element, rule) for the plain method");
    FormMap m;
    plain_map(F, pb, m);
    elfel_hip_problem p = *pb;
    p.precision = ELFEL_FP64;
    if (F.E * m.nmat >= INT32_MAX || F.E * m.nvec >= INT32_MAX) {  // the cached permutation is int32
        p.method = ELFEL_SORT;
        c->used_method = ELFEL_SORT;
        c->used_note += " (a COO stream of 2^31 entries or more: the plain FP64 method)";
        c->nnz = -1;
        return plain_assemble(c, &p, tab, cf);
    }
    return stream_reuse(c, &p, m, F.E, c->nrow, false, [&](const StreamOut &o, bool) {
        return fn(c, tab, cf, (double *)o.vals, (double *)o.fvals);
    });
}

int plain_assemble(elfel_hip_ctx *c, const elfel_hip_problem *pb, const QTable &tab, const Coef &cf)
{
    plain_fn fn = pick_plain(pb->kind, pb->fe, tab.nq);
    if (!fn) return set_err(c, ELFEL_ENOTSUP, "unsupported (kind, element, rule) for the plain method");
    FormMap m;
    plain_map(c->f[0], pb, m);
    return plain_build(c, pb, m, c->f[0].E, c->nrow, [&](const StreamOut &o, bool) {
        return fn(c, tab, cf, (double *)o.vals, (double *)o.fvals);
    });
}
