// HRZ-lumped mass: bilform_dot (src/FEMMBaseModule.jl:1335-1366) into a
// SysmatAssemblerSparseHRZLumpingSymm (src/AssemblyModule.jl:943-1141): each
// element's diagonal, scaled by (sum of its entries) / (sum of its diagonal),
// summed per DOF in ascending element order; the diagonal CSC of the DOFs that
// some element touches.
//
// The numbers are nodal sums (vector.hip).  The pattern belongs to the mesh's
// numbering: it is made with the first lumped mass of it, and kept.
#include "common.hpp"

namespace feasm {

namespace {

__global__ __launch_bounds__(256) void k_diag_flag(const int64_t *__restrict__ n2e_ptr, int64_t nnodes, int ndn,
                                                   const int32_t *__restrict__ dofs, int32_t *__restrict__ flag) {
    for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n < nnodes; n += (int64_t)gridDim.x * blockDim.x)
        if (n2e_ptr[n] != n2e_ptr[n + 1])  // a node of no element has no stored entry
            for (int k = 0; k < ndn; k++) flag[dofs[n * ndn + k]] = 1;
}

__global__ __launch_bounds__(256) void k_diag_rows(const int32_t *__restrict__ flag, const int64_t *__restrict__ pos,
                                                   int64_t n, int32_t *__restrict__ rowval) {
    for (int64_t d = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; d < n; d += (int64_t)gridDim.x * blockDim.x)
        if (flag[d]) rowval[pos[d]] = (int32_t)d;
}

std::shared_ptr<DiagPattern> diag_pattern(feasm_ctx *ctx, const feasm_mesh *m) {
    auto D = std::make_shared<DiagPattern>();
    const int64_t n = m->nalldofs;
    DevPtr flag = dev_alloc((n + 1) * sizeof(int32_t));
    FEASM_HIP(hipMemsetAsync(flag->p, 0, (n + 1) * sizeof(int32_t), ctx->stream));
    hipLaunchKernelGGL(k_diag_flag, dim3(grid_for(m->nnodes, 256)), dim3(256), 0, ctx->stream, dp<int64_t>(m->n2e_ptr),
                       m->nnodes, m->ndn, dp<int32_t>(m->dofs), dp<int32_t>(flag));
    FEASM_HIP(hipGetLastError());
    D->colptr = dev_alloc((n + 1) * sizeof(int64_t));
    exclusive_scan_i32_to_i64(ctx, dp<int32_t>(flag), dp<int64_t>(D->colptr), n + 1);
    read_back(ctx->stream, &D->nnz, dp<int64_t>(D->colptr) + n, sizeof(int64_t));
    D->rowval = dev_alloc(std::max<int64_t>(D->nnz, 1) * sizeof(int32_t));
    hipLaunchKernelGGL(k_diag_rows, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, dp<int32_t>(flag),
                       dp<int64_t>(D->colptr), n, dp<int32_t>(D->rowval));
    FEASM_HIP(hipGetLastError());
    return D;
}

}  // namespace

feasm_matrix *hrz_lumped(feasm_ctx *ctx, feasm_mesh *m, const DevQTable &qt, const double *coef) {
    const int ndn = m->ndn;
    const int64_t n = m->nalldofs;
    FEASM_REQUIRE(m->conn && m->xyz && m->n2e_ptr && m->n2e && m->dofs, FEASM_ESTATE, "lumped mass: mesh arrays missing");
    FEASM_REQUIRE(qt.nqp <= 64, FEASM_EUNSUPPORTED, "lumped mass: rules of at most 64 points");
    FEASM_REQUIRE(ndn >= 1 && ndn <= 3, FEASM_EUNSUPPORTED, "lumped mass: 1 to 3 DOFs per node");
    if (!m->diag) m->diag = diag_pattern(ctx, m);
    std::unique_ptr<feasm_matrix> M(new feasm_matrix);
    M->ctx = ctx;
    M->m = M->n = n;
    M->nnz = m->diag->nnz;
    M->colptr = m->diag->colptr;
    M->rowval = m->diag->rowval;
    M->nzval = dev_alloc(std::max<int64_t>(M->nnz, 1) * sizeof(double));
    double sums[2] = {0.0, 0.0}, f[3] = {0.0, 0.0, 0.0};  // of all entries of c, of its diagonal; its diagonal
    for (int p = 0; p < ndn; p++) {
        for (int k = 0; k < ndn; k++) sums[0] += coef[ndn * p + k];
        f[p] = coef[ndn * p + p];
        sums[1] += f[p];
    }
    double *stage = static_cast<double *>(ctx->scratch_get((size_t)m->nelem * m->npe * sizeof(double)));
    launch_nodal_sums(ctx, m, qt, sums, f, m->nodemajor && M->nnz == n, dp<int64_t>(m->diag->colptr), stage,
                      dp<double>(M->nzval));
    FEASM_HIP(hipStreamSynchronize(ctx->stream));
    return M.release();
}

}  // namespace feasm
