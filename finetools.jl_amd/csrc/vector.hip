// Nodal sums over the elements: the load vector of a constant force
// (linform_dot on solid elements, m = 3, with the SysvecAssembler;
// src/FEMMBaseModule.jl:1207-1241, src/AssemblyModule.jl:853-917) and the
// diagonal of the HRZ-lumped mass (lumped.hip).
//
// Both are one number per (element, local node) times constants:
//   load    s_a = sum_q N_a J w            F[(n, k)] = sum_e s_a f_k
//   lumped  s_a = (em2 / dem2) sum_q N_a^2 J w, with em2 the sum of the element
//           mass matrix's entries, (sum_a N_a)^2 J w summed over the points times
//           the sum of c, and dem2 the sum of its diagonal;
//           M[(n, k), (n, k)] = c_kk sum_e s_a
// k_nodal_elem: one thread per element stages s_a in npe planes, so that a
// wavefront's stores, and the reads of neighbouring nodes, fill whole lines;
// k_nodal_gather: one thread per node adds its elements' numbers in ascending
// element order (the node -> element lists are sorted), the order of
// assemble!.
//
// What bounds them is the gathers (24-byte node records, then 8-byte staged
// numbers), so few wide loads per thread: a connectivity row as 16- or 8-byte
// loads, a node as one 16- and one 8-byte load.  H8 87x79x61 load vector, 40 MB
// compulsory: staging the points' J w (64 B read per list entry) 54 us, the
// nodal numbers (8 B) 31 us; HRZ mass of H8 73x61x59: forming the 24 x 24
// entries 208 us with its scan, this 46 us.
#include "common.hpp"

namespace feasm {

namespace {

constexpr int kBlock = 128;

// three doubles from an 8-byte aligned address (16- and 8-byte loads)
struct __attribute__((packed, aligned(8))) Node3 {
    double x, y, z;
};

template <int NPE>
__device__ __forceinline__ void load_row(const int32_t *__restrict__ conn, int64_t e, int32_t (&c)[NPE]) {
    if constexpr (NPE == 8) {  // 32-byte rows
        const int4 *r = reinterpret_cast<const int4 *>(conn + e * NPE);
        const int4 a = r[0], b = r[1];
        c[0] = a.x; c[1] = a.y; c[2] = a.z; c[3] = a.w;
        c[4] = b.x; c[5] = b.y; c[6] = b.z; c[7] = b.w;
    } else {  // 40-byte rows
        const int2 *r = reinterpret_cast<const int2 *>(conn + e * NPE);
#pragma unroll
        for (int i = 0; i < NPE / 2; i++) {
            const int2 a = r[i];
            c[2 * i] = a.x;
            c[2 * i + 1] = a.y;
        }
    }
}

// The points are a loop: unrolled, their tables (33 doubles a point) spill the
// scalar registers.
template <int NPE, bool LUMPED>
__global__ __launch_bounds__(kBlock) void k_nodal_elem(const int32_t *__restrict__ conn, const double *__restrict__ xyz,
                                                    int64_t nelem, int nqp, const double *__restrict__ N,
                                                    const double *__restrict__ dN, const double *__restrict__ w,
                                                    double csum, double ctrace, double *__restrict__ stage) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nelem;
         e += (int64_t)gridDim.x * blockDim.x) {
        int32_t c[NPE];
        load_row<NPE>(conn, e, c);
        Node3 X[NPE];
#pragma unroll
        for (int a = 0; a < NPE; a++) X[a] = reinterpret_cast<const Node3 *>(xyz)[c[a]];
        double s[NPE], total = 0.0;
#pragma unroll
        for (int a = 0; a < NPE; a++) s[a] = 0.0;
#pragma unroll 1
        for (int q = 0; q < nqp; q++) {
            double J[9];
#pragma unroll
            for (int i = 0; i < 9; i++) J[i] = 0.0;
#pragma unroll
            for (int a = 0; a < NPE; a++) {
                const double d0 = dN[(q * NPE + a) * 3], d1 = dN[(q * NPE + a) * 3 + 1], d2 = dN[(q * NPE + a) * 3 + 2];
                J[0] += X[a].x * d0; J[1] += X[a].x * d1; J[2] += X[a].x * d2;
                J[3] += X[a].y * d0; J[4] += X[a].y * d1; J[5] += X[a].y * d2;
                J[6] += X[a].z * d0; J[7] += X[a].z * d1; J[8] += X[a].z * d2;
            }
            const double det = J[0] * (J[4] * J[8] - J[7] * J[5]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
                               J[2] * (J[3] * J[7] - J[4] * J[6]);
            const double jw = det * w[q];
            double ns = 0.0;
#pragma unroll
            for (int a = 0; a < NPE; a++) {
                const double na = N[q * NPE + a];
                if (LUMPED) ns += na;
                s[a] += LUMPED ? na * na * jw : na * jw;
            }
            if (LUMPED) total += ns * ns * jw;
        }
        double f = 1.0;
        if (LUMPED) {
            double d = 0.0;
#pragma unroll
            for (int a = 0; a < NPE; a++) d += s[a];
            f = (total * csum) / (d * ctrace);
        }
#pragma unroll
        for (int a = 0; a < NPE; a++) stage[a * nelem + e] = LUMPED ? s[a] * f : s[a];
    }
}

// The node's list entries, then their numbers, are loaded eight at a time (all
// of an interior H8 node's) before any is added.  DIRECT: the DOFs are
// node-major and out[d] is DOF d's, so that a node of no element gets its
// zeros here.  Otherwise DOF d goes to out[place[d]] (place null: out[d]),
// and the DOFs of a node of no element are left alone.
template <int NDN, bool DIRECT>
__global__ __launch_bounds__(kBlock) void k_nodal_gather(const int64_t *__restrict__ n2e_ptr,
                                                      const uint32_t *__restrict__ n2e, int64_t nnodes,
                                                      int64_t nelem, const double *__restrict__ stage, double f0, double f1,
                                                      double f2, const int32_t *__restrict__ dofs,
                                                      const int64_t *__restrict__ place, double *__restrict__ out) {
    for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n < nnodes;
         n += (int64_t)gridDim.x * blockDim.x) {
        const int64_t s0 = n2e_ptr[n], s1 = n2e_ptr[n + 1];
        if (!DIRECT && s0 == s1) continue;
        double a0 = 0.0, a1 = 0.0, a2 = 0.0;
        constexpr int U = 8;
        for (int64_t s = s0; s < s1; s += U) {
            uint32_t v[U];
            double x[U];
#pragma unroll
            for (int j = 0; j < U; j++) v[j] = s + j < s1 ? n2e[s + j] : 0u;
#pragma unroll
            for (int j = 0; j < U; j++) x[j] = stage[(int64_t)(v[j] & 15u) * nelem + (v[j] >> 4)];
#pragma unroll
            for (int j = 0; j < U; j++) {
                if (s + j >= s1) break;
                a0 += x[j] * f0;
                if (NDN > 1) a1 += x[j] * f1;
                if (NDN > 2) a2 += x[j] * f2;
            }
        }
        const double a[3] = {a0, a1, a2};
#pragma unroll
        for (int k = 0; k < NDN; k++) {
            if (DIRECT) {
                out[n * NDN + k] = a[k];
            } else {
                const int32_t d = dofs[n * NDN + k];
                out[place ? place[d] : d] = a[k];
            }
        }
    }
}

template <int NPE, bool LUMPED>
void launch_elem(feasm_ctx *ctx, const feasm_mesh *m, const DevQTable &qt, double csum, double ctrace, double *stage) {
    if (m->nelem == 0) return;
    hipLaunchKernelGGL((k_nodal_elem<NPE, LUMPED>), dim3(grid_for(m->nelem, kBlock)), dim3(kBlock), 0, ctx->stream,
                       dp<int32_t>(m->conn), dp<double>(m->xyz), m->nelem, qt.nqp, qt.N(), qt.dN(), qt.w(), csum,
                       ctrace, stage);
    FEASM_HIP(hipGetLastError());
}

template <int NDN>
void launch_gather_t(feasm_ctx *ctx, const feasm_mesh *m, const double *stage, const double *f, bool direct,
                     const int64_t *place, double *out) {
    if (m->nnodes == 0) return;
    const auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(grid_for(m->nnodes, kBlock)), dim3(kBlock), 0, ctx->stream, dp<int64_t>(m->n2e_ptr),
                           dp<uint32_t>(m->n2e), m->nnodes, m->nelem, stage, f[0], f[1], f[2], dp<int32_t>(m->dofs), place, out);
    };
    direct ? go(k_nodal_gather<NDN, true>) : go(k_nodal_gather<NDN, false>);
    FEASM_HIP(hipGetLastError());
}

void launch_gather_n(feasm_ctx *ctx, const feasm_mesh *m, const double *stage, const double *f, bool direct,
                     const int64_t *place, double *out) {
    if (m->ndn == 1) return launch_gather_t<1>(ctx, m, stage, f, direct, place, out);
    if (m->ndn == 2) return launch_gather_t<2>(ctx, m, stage, f, direct, place, out);
    return launch_gather_t<3>(ctx, m, stage, f, direct, place, out);
}

}  // namespace

void launch_nodal_sums(feasm_ctx *ctx, const feasm_mesh *m, const DevQTable &qt, const double *lumped_sums,
                       const double *f, bool direct, const int64_t *place, double *stage, double *out) {
    FEASM_REQUIRE(m->conn && m->xyz && m->n2e_ptr && m->n2e && m->dofs && stage && out, FEASM_ESTATE,
                  "nodal sums: mesh arrays missing");
    FEASM_REQUIRE(m->npe == 8 || m->npe == 10, FEASM_EUNSUPPORTED, "nodal sums cover H8 and T10 meshes");
    const double csum = lumped_sums ? lumped_sums[0] : 0.0, ctrace = lumped_sums ? lumped_sums[1] : 0.0;
    if (m->npe == 8) {
        lumped_sums ? launch_elem<8, true>(ctx, m, qt, csum, ctrace, stage)
                    : launch_elem<8, false>(ctx, m, qt, csum, ctrace, stage);
        launch_gather_n(ctx, m, stage, f, direct, place, out);
    } else {
        lumped_sums ? launch_elem<10, true>(ctx, m, qt, csum, ctrace, stage)
                    : launch_elem<10, false>(ctx, m, qt, csum, ctrace, stage);
        launch_gather_n(ctx, m, stage, f, direct, place, out);
    }
}

void launch_linform_dot(feasm_ctx *ctx, const feasm_mesh *m, const DevQTable &qt, const double *force,
                        double *stage, double *F) {
    const double f[3] = {force[0], m->ndn > 1 ? force[1] : 0.0, m->ndn > 2 ? force[2] : 0.0};
    // node-major: every entry of F is some node's; otherwise F may hold
    // numbers of no DOF
    if (!m->nodemajor) FEASM_HIP(hipMemsetAsync(F, 0, (size_t)m->nalldofs * sizeof(double), ctx->stream));
    launch_nodal_sums(ctx, m, qt, nullptr, f, m->nodemajor, nullptr, stage, F);
}

}  // namespace feasm
