// Fused numeric assembly: element integration and the global summation in
// one kernel, nothing staged in HBM.
//
// Each workgroup walks tiles of its XCD's contiguous range (a tile: a compact
// set of owned column nodes plus the halo of elements incident to them, with
// the tile's node blocks listed as tasks; see tiles.cpp).  Per tile:
//   0  the tile's LDS image (column pointers, task and item lists, halo
//      connectivity; one contiguous blob laid out by TileShape::layout) and
//      the coordinates of its halo nodes go to LDS.  These global loads are
//      issued while the previous tile is in phase 2 and held in registers;
//   1  one thread per (halo element, quadrature point): J = X' dN (in FP64
//      kernels by exchanges between the element's points, point_fp64), det J
//      and the adjugate inverse (src/FESetModule.jl:479-544) in FP64; the spatial gradients g_a = inv(J)' dN_a are stored scaled by
//      sqrt(|J w|) (u_a = sqrt(|Jw|) g_a, with the sign of J w kept apart), so
//      that an element's node-pair matrix is M_ab = sum_q s_q u_a u_b^T;
//   2  one thread per CSC node block (m, c) of the tile's columns forms the
//      element matrices M^e_{m c} of the elements holding both nodes and adds
//      them in ascending element number -- the order in which
//      SparseArrays.sparse folds the duplicates of the reference's
//      element-major COO (src/AssemblyModule.jl:319-325) -- applies the
//      material (K = D : M for elasticity, src/DeforModelRedModule.jl:447-472
//      with src/MatrixUtilityModule.jl:189-216) and writes the block once.
// The products u_m[k] u_c[l] are formed symmetrically (a sign flip is exact,
// the product commutes) and every block is contracted in the orientation of
// its lower node number, so the assembled matrix is exactly symmetric, as the
// reference's is (test/test_forms.jl:442).
#include "fused.hpp"

namespace feasm {

namespace {

constexpr int kMaxThreads = 1024;

__device__ constexpr int voigt(int i, int k) {
    return (i == k) ? i : ((i + k == 1) ? 3 : ((i + k == 2) ? 4 : 5));
}

// Linear elasticity with a material matrix of cubic symmetry (isotropic
// materials among them): D00 = D11 = D22, D01 = D02 = D12, D33 = D44 = D55,
// every other entry zero.  Then K = D01 M + D33 M^T off the diagonal and
// K_ii = D00 M_ii + D33 (tr M - M_ii), three coefficients instead of 36.
constexpr int kFormElasticCubic = 16;

}  // namespace

bool cubic_symmetry(const double *D) {
    for (int i = 0; i < 6; i++)
        for (int j = 0; j < 6; j++) {
            const double v = D[6 * i + j];
            if (i < 3 && j < 3) {
                if (v != (i == j ? D[0] : D[1])) return false;
            } else if (i == j) {
                if (v != D[21]) return false;
            } else if (v != 0.0) {
                return false;
            }
        }
    return true;
}

namespace {

struct FusedParams {
    FormParams fp;
    int cubic;         // elasticity with a cubic-symmetry D (see kFormElasticCubic)
    const double *N;   // [nqp][npe]
    const double *dN;  // [nqp][npe][3]
    const double *w;   // [nqp]
};

// Everything one workgroup needs to process the tiles of one mesh.
struct TileJob {
    const TileHdr *hdr;
    const unsigned char *blob;
    const int32_t *hnodes;
    const double *xyz;
    double *nzval;
};

// signs of J w at the points of one element (nonzero byte = negative)
template <int NQP>
__device__ __forceinline__ uint64_t neg_mask(const uint8_t *s) {
    if constexpr (NQP == 8) return *reinterpret_cast<const uint64_t *>(s);
    else if constexpr (NQP == 4) return *reinterpret_cast<const uint32_t *>(s);
    else {
        uint64_t m = 0;
        for (int q = 0; q < NQP; q++) m |= (uint64_t)s[q] << (8 * q);
        return m;
    }
}

// Adds M^e for the node pair (row ar, column ac) of halo element h to M: the
// sum over the points of s_q u_ar u_ac^T (grad forms; 9 values, or its trace
// for SWP 1) or of N_ar N_ac J w (DOT).  DIAG: a diagonal block (ar == ac),
// whose M^e is symmetric: one vector per point is read and, for SWP 9, only
// the upper triangle (M[0..2], M[4], M[5], M[8]) is formed.
template <int FORM>
constexpr int form_swp() {
    return (FORM == FEASM_FORM_LIN_ELASTIC || FORM == kFormElasticCubic || FORM == FEASM_FORM_DIFFUSION_MAT) ? 9 : 1;
}

// The 16-byte chunk type of the scaled-gradient records (see
// TileShape::uchunks): two doubles or four floats.
template <typename R>
struct Chunk;
template <>
struct Chunk<double> {
    using T = double2;
};
template <>
struct Chunk<float> {
    using T = float4;
};

// s_q r c^T (SWP 9: the 9 products; DIAG: the upper triangle) or its trace
template <int SWP, bool SIGNED, bool DIAG, typename R, typename A>
__device__ __forceinline__ void point_product(bool negative, R c0, R c1, R c2, R r0, R r1, R r2, A *M) {
    if (SIGNED && negative) {
        r0 = -r0;
        r1 = -r1;
        r2 = -r2;
    }
    if (SWP == 9) {
        M[0] = fma(r0, c0, M[0]); M[1] = fma(r0, c1, M[1]); M[2] = fma(r0, c2, M[2]);
        if (!DIAG) M[3] = fma(r1, c0, M[3]);
        M[4] = fma(r1, c1, M[4]); M[5] = fma(r1, c2, M[5]);
        if (!DIAG) { M[6] = fma(r2, c0, M[6]); M[7] = fma(r2, c1, M[7]); }
        M[8] = fma(r2, c2, M[8]);
    } else {
        M[0] = fma(r0, c0, M[0]);
        M[0] = fma(r1, c1, M[0]);
        M[0] = fma(r2, c2, M[0]);
    }
}

template <int NPE, int NQP, int FORM, typename R, bool SIGNED, bool DIAG, typename A>
__device__ __forceinline__ void elem_block(uint32_t it, const R *__restrict__ sU, const uint8_t *__restrict__ sSg,
                                           const double *__restrict__ sN, const R *__restrict__ sW, A *M) {
    constexpr int SWP = form_swp<FORM>();
    const int h = (int)(it >> 8), ac = (int)((it >> 4) & 15u), ar = (int)(it & 15u);
    if constexpr (FORM != FEASM_FORM_DOT) {
        using C = typename Chunk<R>::T;
        constexpr int PX = (sizeof(R) == 8) ? 1 : 2;  // points per xy chunk
        constexpr int PZ = 2 * PX;                    // points per z chunk
        constexpr int US = (NQP * NPE * 3 * (int)sizeof(R) / 16 + 1) * 16 / (int)sizeof(R);  // TileShape::ustride()
        static_assert(NQP % PZ == 0, "points per element must fill the z chunks");
        const C *U = reinterpret_cast<const C *>(sU + h * US);
        const C *UZ = U + (NQP / PX) * NPE;
        uint64_t neg = 0;
        if (SIGNED) neg = neg_mask<NQP>(sSg + h * NQP);
#pragma unroll
        for (int g = 0; g < NQP / PZ; g++) {
            const C cz = UZ[g * NPE + ac];
            const C rz = DIAG ? cz : UZ[g * NPE + ar];
#pragma unroll
            for (int x = 0; x < PZ / PX; x++) {
                const C cxy = U[(g * (PZ / PX) + x) * NPE + ac];
                const C rxy = DIAG ? cxy : U[(g * (PZ / PX) + x) * NPE + ar];
                if constexpr (sizeof(R) == 8) {  // one point: (u0, u1), u2 in cz.x / cz.y
                    const int q = g * 2 + x;
                    const R c2 = x ? cz.y : cz.x, r2 = x ? rz.y : rz.x;
                    point_product<SWP, SIGNED, DIAG>(((neg >> (8 * q)) & 255u) != 0, (R)cxy.x, (R)cxy.y, c2,
                                                     (R)rxy.x, (R)rxy.y, r2, M);
                } else {  // two points: (u0, u1, u0', u1'), u2 of four points in cz
                    const int q = g * 4 + x * 2;
                    const R c2a = x ? cz.z : cz.x, c2b = x ? cz.w : cz.y;
                    const R r2a = x ? rz.z : rz.x, r2b = x ? rz.w : rz.y;
                    point_product<SWP, SIGNED, DIAG>(((neg >> (8 * q)) & 255u) != 0, (R)cxy.x, (R)cxy.y, c2a,
                                                     (R)rxy.x, (R)rxy.y, r2a, M);
                    point_product<SWP, SIGNED, DIAG>(((neg >> (8 * (q + 1))) & 255u) != 0, (R)cxy.z, (R)cxy.w,
                                                     c2b, (R)rxy.z, (R)rxy.w, r2b, M);
                }
            }
        }
    } else {
#pragma unroll
        for (int q = 0; q < NQP; q++) {
            const R nn = (R)(sN[q * NPE + ar] * sN[q * NPE + ac]);
            M[0] = fma(nn, sW[h * NQP + q], M[0]);
        }
    }
}

// The element matrices of one block's shared elements, added in ascending
// element order (items j = 0..k-1); ILP elements (1 or 2) in flight at a
// time.  In FP64 the products go straight into the FP64 sums (element after
// element, point after point); in mixed precision each element's matrix is
// formed in FP32 and added in FP64.
template <int NPE, int NQP, int FORM, typename R, bool SIGNED, bool DIAG, int SWP, int ILP>
__device__ __forceinline__ void block_sum(int k, const uint16_t *__restrict__ items, const R *__restrict__ sU,
                                          const uint8_t *__restrict__ sSg, const double *__restrict__ sN,
                                          const R *__restrict__ sW, double *acc) {
    // the next item's index is read while the current one is summed
    if constexpr (sizeof(R) == 8) {
        uint32_t it = items[0];  // k >= 1: every block of the pattern has an element
        for (int j = 0; j < k; j++) {
            const uint32_t nx = items[min(j + 1, k - 1)];
            elem_block<NPE, NQP, FORM, R, SIGNED, DIAG>(it, sU, sSg, sN, sW, acc);
            it = nx;
        }
    } else {
        int j = 0;
        for (; ILP == 2 && j + 1 < k; j += 2) {
            const uint32_t i0 = items[j], i1 = items[j + 1];
            R M0[SWP], M1[SWP];
#pragma unroll
            for (int i = 0; i < SWP; i++) M0[i] = M1[i] = (R)0;
            elem_block<NPE, NQP, FORM, R, SIGNED, DIAG>(i0, sU, sSg, sN, sW, M0);
            elem_block<NPE, NQP, FORM, R, SIGNED, DIAG>(i1, sU, sSg, sN, sW, M1);
#pragma unroll
            for (int i = 0; i < SWP; i++) acc[i] = (acc[i] + (double)M0[i]) + (double)M1[i];
        }
        for (; j < k; j++) {
            R M0[SWP];
#pragma unroll
            for (int i = 0; i < SWP; i++) M0[i] = (R)0;
            elem_block<NPE, NQP, FORM, R, SIGNED, DIAG>(items[j], sU, sSg, sN, sW, M0);
#pragma unroll
            for (int i = 0; i < SWP; i++) acc[i] = acc[i] + (double)M0[i];
        }
    }
}

// Global loads of one tile's LDS image, issued ahead and held in registers:
// NC 16-byte chunks per thread (chunks tid, tid + threads, ...; the rest of a
// larger blob is copied at store time).  COEF: the tile also brings its
// mesh's material coefficients (batched launches); otherwise the launch's
// coefficients are loaded once.
template <bool COEF, int NC>
struct Staged {
    uint4 c[NC];
    double d;  // material coefficient tid (COEF)
    // waits for the loads here: called before the wavefront's global stores,
    // so that the wait does not include them (the vector memory counter
    // counts loads and stores in issue order)
    __device__ __forceinline__ void ready() const {
#pragma unroll
        for (int i = 0; i < NC; i++) asm volatile("" ::"v"(c[i].x), "v"(c[i].y), "v"(c[i].z), "v"(c[i].w));
        if constexpr (COEF) asm volatile("" ::"v"(d));
    }
};
// chunks prefetched per thread (measured: the FP64 and DOT kernels gain from
// a second chunk on the larger T10 blobs and nothing from a third; the
// mixed-precision gradient kernels are faster with one; T10 FP64 scalar
// diffusion, 197k elements 150.6 us with two, 154.5 with one)
template <typename R, int FORM>
constexpr int staged_chunks() {
    return (sizeof(R) == 4 && FORM != FEASM_FORM_DOT) ? 1 : 2;
}

// A tile header.  With `hdr` a __restrict__ kernel argument (nothing the
// kernel stores aliases it) and t the same in every lane, the compiler reads
// it with scalar loads, so that it sits in scalar registers and no vector
// memory wait is needed for it.
__device__ __forceinline__ TileHdr load_hdr(const TileHdr *__restrict__ hdr, int64_t t) { return hdr[t]; }

// A tile header (and in a batched launch the tile's entry) on its way, as words
// in the lanes of each wavefront: a vector load like the blob's, waited for
// together with it.  (A scalar load still pending makes every wait for an LDS
// read wait for it too, and the walk's next header is a new cache line each
// time.)
struct StagedHdr {
    static constexpr int kWords = sizeof(TileHdr) / 4;
    uint32_t w;
    __device__ __forceinline__ void issue(const TileHdr *__restrict__ hdr, const int32_t *__restrict__ entry,
                                          int64_t t) {
        const int lane = threadIdx.x & 63;
        const uint32_t *p = reinterpret_cast<const uint32_t *>(hdr + t) + min(lane, kWords - 1);
        if (entry && lane >= kWords) p = reinterpret_cast<const uint32_t *>(entry + t);
        w = *p;
    }
    __device__ __forceinline__ void ready() const { asm volatile("" ::"v"(w)); }
    __device__ __forceinline__ uint32_t word(int i) const { return (uint32_t)__builtin_amdgcn_readlane((int)w, i); }
    __device__ __forceinline__ int32_t entry() const { return (int32_t)word(kWords); }
    __device__ __forceinline__ TileHdr get() const {
        TileHdr h;
        h.P = (int32_t)word(0);
        h.H = (int32_t)word(1);
        h.NH = (int32_t)word(2);
        h.NT = (int32_t)word(3);
        h.K = (int32_t)word(4);
        h.NI = (int32_t)word(5);
        h.x0 = (int32_t)word(6);
        h.nbytes = (int32_t)word(7);
        h.blob = (int64_t)((uint64_t)word(8) | ((uint64_t)word(9) << 32));
        return h;
    }
};

template <bool COEF, int NC>
__device__ __forceinline__ void stage_issue(const TileJob &job, const TileHdr &hd, const double *coef,
                                            Staged<COEF, NC> &st) {
    const int tid = threadIdx.x, nt = blockDim.x;
    const int nch = hd.nbytes >> 4;  // at least one chunk: every tile owns a column
    const uint4 *src = reinterpret_cast<const uint4 *>(job.blob + hd.blob);
#pragma unroll
    for (int i = 0; i < NC; i++) st.c[i] = src[min(tid + i * nt, nch - 1)];
    if constexpr (COEF) st.d = coef[min(tid, 35)];
}

// The staged image into LDS (blob with the halo coordinates, material
// coefficients); clears the tile's sign flag.
template <bool COEF, int NC>
__device__ __forceinline__ void stage_store(const TileJob &job, const TileHdr &hd, const Staged<COEF, NC> &st,
                                            const TileShape::Layout &L, unsigned char *smem, double *sD,
                                            int *sNeg) {
    const int tid = threadIdx.x, nt = blockDim.x;
    const int nch = hd.nbytes >> 4;
    uint4 *dst = reinterpret_cast<uint4 *>(smem + L.cbase);
#pragma unroll
    for (int i = 0; i < NC; i++)
        if (tid + i * nt < nch) dst[tid + i * nt] = st.c[i];
    const uint4 *src = reinterpret_cast<const uint4 *>(job.blob + hd.blob);
    for (int i = tid + NC * nt; i < nch; i += nt) dst[i] = src[i];
    if constexpr (COEF)
        if (tid < 36) sD[tid] = st.d;
    if (tid == 0) *sNeg = 0;
}

// Phase 1 in FP64: the lanes of an element's points share its coordinates.
// The 8 points of the H8 Gauss rule and the 4 of the T10 rule lie each beside a
// corner of their own, so the element looks the same from every point once its
// corners are named from there: corner m of point q is corner q ^ m (H8:
// reflected, one bit per direction; T10: permuted, always evenly).  Lane q reads
// its own corner (T10: and that corner's edges), the sums over the others are
// lane exchanges, and the basis values are the same constants in every lane.
// Phase 1 waits for LDS: a thread that sums over all nodes makes 48 (H8) or 40
// (T10) reads, half of them of scattered coordinates; this one makes 2 or 8.  It
// takes 3500 instead of 7200 of an H8 tile's cycles (T10: 3400 for 8500); H8
// elasticity, 1M elements 985 -> 936 us, T10, 178k elements 217 -> 212.  The
// FP32 kernels read the tables: their values would not stay the same.

// the value of lane (lane ^ M), M < 8, in a group of 8 whose lanes all run
template <int M>
__device__ __forceinline__ double lane_swap(double v) {
    const auto word = [](int x) {
        if constexpr (M >= 4) x = __builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, false);  // row_half_mirror: lane ^ 7
        constexpr int q = M >= 4 ? M ^ 7 : M;
        if constexpr (q == 1) x = __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
        if constexpr (q == 2) x = __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
        if constexpr (q == 3) x = __builtin_amdgcn_mov_dpp(x, 0x1B, 0xF, 0xF, false);  // quad_perm [3,2,1,0]
        return x;
    };
    return __hiloint2double(word(__double2hiint(v)), word(__double2loint(v)));
}

__device__ __forceinline__ double det3(const double (&a)[3], const double (&b)[3], const double (&c)[3]) {
    return a[0] * (b[1] * c[2] - b[2] * c[1]) + a[1] * (b[2] * c[0] - b[0] * c[2]) + a[2] * (b[0] * c[1] - b[1] * c[0]);
}

struct H8Point {
    static constexpr int kNodes = 8, kPoints = 8;
    static constexpr double lo = 0.5 * (1.0 - kGauss2), hi = 0.5 * (1.0 + kGauss2);
    int q;
    // local node of corner c = 4 i + 2 j + k (bit 1: the + side)
    __device__ __forceinline__ static int node(int c) { return (int)(0x62517340u >> (4 * c)) & 7; }
    // columns of the Jacobian along each direction, from this corner towards
    // the other (2 J times -1 on the + side); returns det J
    __device__ __forceinline__ double jacobian(const uint16_t *cn, const double2 *sXY, const double *sZ,
                                               double (&j1)[3], double (&j2)[3], double (&j3)[3], double &det) {
        const int n = (int)cn[node(q)];
        const double2 xy = sXY[n];
        const double x[3] = {xy.x, xy.y, sZ[n]};
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double xi = lane_swap<4>(x[c]);
            const double d = xi - x[c], v = hi * x[c] + lo * xi;  // derivative and value along xi
            const double dj = lane_swap<2>(d), vj = lane_swap<2>(v);
            const double dv = hi * d + lo * dj, vd = vj - v, vv = hi * v + lo * vj;  // and along eta
            j1[c] = hi * dv + lo * lane_swap<1>(dv);
            j2[c] = hi * vd + lo * lane_swap<1>(vd);
            j3[c] = lane_swap<1>(vv) - vv;
        }
        det = det3(j1, j2, j3);
        return (__popc(q) & 1) ? -0.125 * det : 0.125 * det;
    }
    // put(a, u) for every node a: its gradient in terms of the inverse's rows
    template <typename Put>
    __device__ __forceinline__ void gradients(const double (&r1)[3], const double (&r2)[3], const double (&r3)[3],
                                              const Put &put) const {
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const double n1 = (m & 4) ? lo : hi, n2 = (m & 2) ? lo : hi, n3 = (m & 1) ? lo : hi;
            const double d1 = (m & 4) ? n2 * n3 : -n2 * n3, d2 = (m & 2) ? n1 * n3 : -n1 * n3,
                         d3 = (m & 1) ? n1 * n2 : -n1 * n2;
            double u[3];
#pragma unroll
            for (int c = 0; c < 3; c++) u[c] = d1 * r1[c] + d2 * r2[c] + d3 * r3[c];
            put(node(q ^ m), u);
        }
    }
};

struct T10Point {
    static constexpr int kNodes = 10, kPoints = 4;
    static constexpr double lo = kTet4Lo, hi = kTet4Hi;
    int q, e[3];  // e: the edges from corner q to the corners q ^ 1, q ^ 2, q ^ 3
    // columns of the Jacobian: the derivatives along the barycentric
    // coordinates of the corners q ^ 1, q ^ 2, q ^ 3, less corner q's
    __device__ __forceinline__ double jacobian(const uint16_t *cn, const double2 *sXY, const double *sZ,
                                               double (&j1)[3], double (&j2)[3], double (&j3)[3], double &det) {
        e[0] = (q & 2) ? 9 : 4;
        e[1] = (q & 1) ? 8 : 6;
        e[2] = (q == 1 || q == 2) ? 5 : 7;
        const int n = (int)cn[q], n1 = (int)cn[e[0]], n2 = (int)cn[e[1]], n3 = (int)cn[e[2]];
        const double2 p = sXY[n], p1 = sXY[n1], p2 = sXY[n2], p3 = sXY[n3];
        const double x[3] = {p.x, p.y, sZ[n]}, x1[3] = {p1.x, p1.y, sZ[n1]}, x2[3] = {p2.x, p2.y, sZ[n2]},
                     x3[3] = {p3.x, p3.y, sZ[n3]};
        // along corner c: E_c + 4 (hi - lo) x(edge c q), E_c the lane's own
        // corner at lo; along q itself E_q + 4 (hi - lo) x_q
        constexpr double g = 4.0 * (hi - lo);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double E = (4.0 * lo - 1.0) * x[c] + 4.0 * lo * ((x1[c] + x2[c]) + x3[c]);
            j1[c] = (lane_swap<1>(E) - E) + g * (x1[c] - x[c]);
            j2[c] = (lane_swap<2>(E) - E) + g * (x2[c] - x[c]);
            j3[c] = (lane_swap<3>(E) - E) + g * (x3[c] - x[c]);
        }
        det = det3(j1, j2, j3);
        return det;
    }
    template <typename Put>
    __device__ __forceinline__ void gradients(const double (&r1)[3], const double (&r2)[3], const double (&r3)[3],
                                              const Put &put) const {
        double t[3];
#pragma unroll
        for (int c = 0; c < 3; c++) t[c] = -((r1[c] + r2[c]) + r3[c]);  // corner q's own coordinate
        const auto corner = [&](int a, double s, const double (&v)[3]) {
            const double u[3] = {s * v[0], s * v[1], s * v[2]};
            put(a, u);
        };
        const auto edge = [&](int a, double s, const double (&v)[3], const double (&w)[3]) {
            const double u[3] = {s * v[0] + 4.0 * lo * w[0], s * v[1] + 4.0 * lo * w[1], s * v[2] + 4.0 * lo * w[2]};
            put(a, u);
        };
        corner(q, 4.0 * hi - 1.0, t);
        corner(q ^ 1, 4.0 * lo - 1.0, r1);
        corner(q ^ 2, 4.0 * lo - 1.0, r2);
        corner(q ^ 3, 4.0 * lo - 1.0, r3);
        edge(e[0], 4.0 * hi, r1, t);
        edge(e[1], 4.0 * hi, r2, t);
        edge(e[2], 4.0 * hi, r3, t);
        // the edges that do not meet corner q, each opposite one that does
        edge(13 - e[0], 4.0 * lo, r2, r3);
        edge(14 - e[1], 4.0 * lo, r1, r3);
        edge(12 - e[2], 4.0 * lo, r1, r2);
    }
};

template <typename P, int FORM>
__device__ __forceinline__ void point_fp64(int h, int q, const uint16_t *sLc, const double *sX, int NH,
                                           const double *sWq, const double *coef, double *sU, uint8_t *sSg, double *sW,
                                           int *sNeg) {
    constexpr int NPE = P::kNodes, NQP = P::kPoints;
    P pt;
    pt.q = q;
    double j1[3], j2[3], j3[3], det;
    const double detJ = pt.jacobian(sLc + h * NPE, reinterpret_cast<const double2 *>(sX), sX + 2 * NH, j1, j2, j3, det);
    const double wj = (FORM == FEASM_FORM_DIFFUSION_ISO) ? (coef[0] * detJ) * sWq[q] : detJ * sWq[q];
    if constexpr (FORM == FEASM_FORM_DOT) {
        sW[h * NQP + q] = wj;
    } else {
        sSg[h * NQP + q] = (wj < 0.0) ? 1 : 0;
        if (wj < 0.0) atomicOr(sNeg, 1);
        // the inverse scaled by sqrt(|J w|) once: its rows are the cross
        // products of the columns
        const double s = (1.0 / det) * sqrt(fabs(wj));
        const double r1[3] = {(j2[1] * j3[2] - j2[2] * j3[1]) * s, (j2[2] * j3[0] - j2[0] * j3[2]) * s,
                              (j2[0] * j3[1] - j2[1] * j3[0]) * s};
        const double r2[3] = {(j3[1] * j1[2] - j3[2] * j1[1]) * s, (j3[2] * j1[0] - j3[0] * j1[2]) * s,
                              (j3[0] * j1[1] - j3[1] * j1[0]) * s};
        const double r3[3] = {(j1[1] * j2[2] - j1[2] * j2[1]) * s, (j1[2] * j2[0] - j1[0] * j2[2]) * s,
                              (j1[0] * j2[1] - j1[1] * j2[0]) * s};
        // the element's record of 16-byte chunks (TileShape::uchunks): (u0, u1)
        // of point q in xy chunk q, u2 in z chunk q / 2
        double2 *const rec = reinterpret_cast<double2 *>(sU) + (size_t)h * (NPE * NQP * 3 / 2 + 1);
        double2 *const xy = rec + q * NPE;
        double *const zz = reinterpret_cast<double *>(rec + NQP * NPE + (q >> 1) * NPE) + (q & 1);
        pt.gradients(r1, r2, r3, [&](int a, const double (&u)[3]) {
            xy[a] = make_double2(u[0], u[1]);
            zz[2 * a] = u[2];
        });
    }
}

// One tile, phases 1 and 2, with its image already in LDS.  `after_phase1`
// runs between the phases; `before_stores` in phase 2, before the first
// global store of every thread.  LDSCOEF: the scalar material coefficients
// are read from LDS (batched launches, where each tile brings its own)
// rather than from the launch's parameters.
template <int NPE, int NQP, int FORM, int NDN, typename R, bool LDSCOEF, typename AfterPhase1,
          typename BeforeStores>
__device__ __forceinline__ void tile_compute(const TileShape &shape, const TileJob &job, const FusedParams &kp,
                                             const TileHdr &hd, unsigned char *smem, const AfterPhase1 &after_phase1,
                                             const BeforeStores &before_stores) {
    constexpr bool GRAD = (FORM != FEASM_FORM_DOT);
    constexpr int SWP = form_swp<FORM>();
    const int tid = threadIdx.x;
    const int kThreads = blockDim.x;
    const int P = hd.P, H = hd.H, NH = hd.NH, NT = hd.NT, K = hd.K, NI = hd.NI;
    constexpr int US = (NQP * NPE * 3 * (int)sizeof(R) / 16 + 1) * 16 / (int)sizeof(R);  // TileShape::ustride()
    // two elements in flight where the registers allow it under 1024 threads
    constexpr int ILP = 2;
    constexpr int DS = NPE * 3;  // TileShape::dstride()
    const TileShape::Layout L = shape.layout(H, P, NH, K, NT, NI);
    double *sN = reinterpret_cast<double *>(smem + L.tab);
    double *sDN = sN + NQP * NPE;
    double *sD = sDN + NQP * DS;  // material coefficients (read as broadcasts)
    int *sNeg = reinterpret_cast<int *>(sD + 36);  // set when J w < 0 somewhere in the tile
    const double *sWq = sD + 37;                   // quadrature weights
    const double *coef = LDSCOEF ? sD : kp.fp.coef;
    const uint64_t *sTask = reinterpret_cast<const uint64_t *>(smem + L.task);
    uint16_t *sItem = reinterpret_cast<uint16_t *>(smem + L.item);
    double *sX = reinterpret_cast<double *>(smem + L.X);
    uint16_t *sLc = reinterpret_cast<uint16_t *>(smem + L.lconn);
    int64_t *sCb = reinterpret_cast<int64_t *>(smem + L.cbase);
    int32_t *sCd = reinterpret_cast<int32_t *>(smem + L.cdeg);
    R *sU = reinterpret_cast<R *>(smem + L.U);
    uint8_t *sSg = reinterpret_cast<uint8_t *>(smem + L.sgn);
    R *sW = reinterpret_cast<R *>(smem + L.sgn);

    // ---- phase 1: Jacobians, inverses and scaled gradients
    for (int task = tid; task < H * NQP; task += kThreads) {
        const int h = task / NQP, q = task % NQP;
        if constexpr (sizeof(R) == 8) {
            using P = typename std::conditional<NPE == 8, H8Point, T10Point>::type;
            static_assert(P::kNodes == NPE && P::kPoints == NQP, "one lane per corner");
            point_fp64<P, FORM>(h, q, sLc, sX, NH, sWq, coef, reinterpret_cast<double *>(sU), sSg,
                                reinterpret_cast<double *>(sW), sNeg);
            continue;
        }
        const uint16_t *cn = sLc + h * NPE;
        // coordinates: (x, y) pairs then z values; gradient table: (d0, d1)
        // pairs then d2 values; nodes visited in an order rotated by the
        // point, so that the reads are single 16- and 8-byte loads and the
        // lanes of one element fall into different banks
        const double2 *sXY = reinterpret_cast<const double2 *>(sX);
        const double *sZ = sX + 2 * NH;
        const double2 *dxy = reinterpret_cast<const double2 *>(sDN) + q * NPE;
        const double *dz = sDN + 2 * NQP * NPE + q * NPE;
        double J[9];
#pragma unroll
        for (int i = 0; i < 9; i++) J[i] = 0.0;
#pragma unroll
        for (int i = 0; i < NPE; i++) {
            const int a = (i + q) % NPE;
            const int n = (int)cn[a];
            const double2 xy = sXY[n];
            const double x0 = xy.x, x1 = xy.y, x2 = sZ[n];
            const double2 dd = dxy[a];
            const double d0 = dd.x, d1 = dd.y, d2 = dz[a];
            J[0] += x0 * d0; J[1] += x0 * d1; J[2] += x0 * d2;
            J[3] += x1 * d0; J[4] += x1 * d1; J[5] += x1 * d2;
            J[6] += x2 * d0; J[7] += x2 * d1; J[8] += x2 * d2;
        }
#define RJ(i, j) J[3 * ((i)-1) + ((j)-1)]
        const double det = RJ(1, 1) * (RJ(2, 2) * RJ(3, 3) - RJ(3, 2) * RJ(2, 3)) -
                           RJ(1, 2) * (RJ(2, 1) * RJ(3, 3) - RJ(2, 3) * RJ(3, 1)) +
                           RJ(1, 3) * (RJ(2, 1) * RJ(3, 2) - RJ(2, 2) * RJ(3, 1));
        double wj = (FORM == FEASM_FORM_DIFFUSION_ISO) ? (coef[0] * det) * sWq[q] : det * sWq[q];
        if (GRAD) {
            // the inverse scaled by sqrt(|J w|) once: g_a scaled is inv(J)' dN_a times it
            const double invdet = (1.0 / det) * sqrt(fabs(wj));
            const double iv[9] = {(RJ(2, 2) * RJ(3, 3) - RJ(3, 2) * RJ(2, 3)) * invdet,
                                  -(RJ(1, 2) * RJ(3, 3) - RJ(1, 3) * RJ(3, 2)) * invdet,
                                  (RJ(1, 2) * RJ(2, 3) - RJ(1, 3) * RJ(2, 2)) * invdet,
                                  -(RJ(2, 1) * RJ(3, 3) - RJ(2, 3) * RJ(3, 1)) * invdet,
                                  (RJ(1, 1) * RJ(3, 3) - RJ(1, 3) * RJ(3, 1)) * invdet,
                                  -(RJ(1, 1) * RJ(2, 3) - RJ(2, 1) * RJ(1, 3)) * invdet,
                                  (RJ(2, 1) * RJ(3, 2) - RJ(3, 1) * RJ(2, 2)) * invdet,
                                  -(RJ(1, 1) * RJ(3, 2) - RJ(3, 1) * RJ(1, 2)) * invdet,
                                  (RJ(1, 1) * RJ(2, 2) - RJ(2, 1) * RJ(1, 2)) * invdet};
            sSg[h * NQP + q] = (wj < 0.0) ? 1 : 0;
            if (wj < 0.0) atomicOr(sNeg, 1);
            R ivr[9];
#pragma unroll
            for (int i = 0; i < 9; i++) ivr[i] = (R)iv[i];
            // the element's record of 16-byte chunks (TileShape::uchunks):
            // (u0, u1) of point q in xy chunk q / PX, u2 in z chunk q / PZ
            constexpr int PX = (sizeof(R) == 8) ? 1 : 2, PZ = 2 * PX, CR = 16 / (int)sizeof(R);
            R *urec = sU + (size_t)h * US;
            // node order rotated by the point, so that the lanes of one
            // element store into different LDS banks
#pragma unroll
            for (int i = 0; i < NPE; i++) {
                const int a = (i + q) % NPE;
                const double2 dd = dxy[a];
                const R d0 = (R)dd.x, d1 = (R)dd.y, d2 = (R)dz[a];
                const R u0 = d0 * ivr[0] + d1 * ivr[3] + d2 * ivr[6];
                const R u1 = d0 * ivr[1] + d1 * ivr[4] + d2 * ivr[7];
                const R u2 = d0 * ivr[2] + d1 * ivr[5] + d2 * ivr[8];
                const int cxy = (q / PX) * NPE + a, cz = (NQP / PX) * NPE + (q / PZ) * NPE + a;
                if constexpr (sizeof(R) == 8)
                    reinterpret_cast<double2 *>(urec)[cxy] = make_double2(u0, u1);
                else
                    reinterpret_cast<float2 *>(urec)[cxy * 2 + (q % PX)] = make_float2(u0, u1);
                urec[cz * CR + (q % PZ)] = u2;
            }
        } else {
            sW[h * NQP + q] = (R)wj;
        }
#undef RJ
    }
    // one flag for the tile: J w < 0 somewhere (inverted elements) selects
    // the path that applies the signs
    __syncthreads();
    const bool tile_neg = *sNeg != 0;
    after_phase1();


    // ---- phase 2: one thread per node block: element matrices of the shared
    // elements, ordered sum, material, one write
    double *__restrict__ nzval = job.nzval;
    // one block task: its values and where they go
    struct BlockOut {
        double out[NDN * NDN];
        int64_t base, base2;
        int deg, deg2;
        bool valid, pair;
    };
    const auto compute = [&](int t, BlockOut &b) {
        b.valid = false;
        const uint64_t rec = sTask[t];
        const uint32_t th = (uint32_t)rec;
        if (th == kNullTask) return;
        const int c = (int)(th & 255u), r = (int)((th >> 8) & 255u), k = (int)((th >> 16) & 255u);
        const bool sw = (th >> 24) & 1u, diag = (th >> 25) & 1u, sym = (th >> 26) & 1u;
        double acc[SWP];
#pragma unroll
        for (int i = 0; i < SWP; i++) acc[i] = 0.0;
        const uint16_t *items = sItem + (uint32_t)((rec >> 32) & 0xffffu);
        if (GRAD && sym) {  // symmetric diagonal blocks sit in wavefronts of their own
            if (tile_neg)
                block_sum<NPE, NQP, FORM, R, true, true, SWP, ILP>(k, items, sU, sSg, sN, sW, acc);
            else
                block_sum<NPE, NQP, FORM, R, false, true, SWP, ILP>(k, items, sU, sSg, sN, sW, acc);
            if constexpr (SWP == 9) {  // the lower triangle of the symmetric sum
                acc[3] = acc[1];
                acc[6] = acc[2];
                acc[7] = acc[5];
            }
        } else {
            if (tile_neg)
                block_sum<NPE, NQP, FORM, R, true, false, SWP, ILP>(k, items, sU, sSg, sN, sW, acc);
            else
                block_sum<NPE, NQP, FORM, R, false, false, SWP, ILP>(k, items, sU, sSg, sN, sW, acc);
        }
        double *out = b.out;
        if constexpr (SWP == 9) {
            // contract in the orientation of the lower node number
            double Mc[9];
#pragma unroll
            for (int a = 0; a < 3; a++)
#pragma unroll
                for (int b = 0; b < 3; b++) Mc[3 * a + b] = sw ? acc[3 * b + a] : acc[3 * a + b];
            if constexpr (FORM == FEASM_FORM_DIFFUSION_MAT) {
                // the address depends on the task, which keeps the compiler
                // from holding every coefficient in registers across tasks
                const double *D = sD + (th >> 31);
                double s = 0.0;
#pragma unroll
                for (int a = 0; a < 3; a++)
#pragma unroll
                    for (int b = 0; b < 3; b++) s += D[3 * a + b] * Mc[3 * a + b];
                out[0] = s;
            } else {
                double Kc[9];
                if constexpr (FORM == kFormElasticCubic) {
                    const double d00 = coef[0], d01 = coef[1], d33 = coef[21];
                    const double tr = (Mc[0] + Mc[4]) + Mc[8];
#pragma unroll
                    for (int i = 0; i < 3; i++)
#pragma unroll
                        for (int jj = 0; jj < 3; jj++)
                            Kc[3 * i + jj] = (i == jj) ? d00 * Mc[4 * i] + d33 * (tr - Mc[4 * i])
                                                       : d01 * Mc[3 * i + jj] + d33 * Mc[3 * jj + i];
                } else {
                    const double *D = sD + (th >> 31);  // see above
#pragma unroll
                    for (int i = 0; i < 3; i++)
#pragma unroll
                        for (int jj = 0; jj < 3; jj++) {
                            double s = 0.0;
#pragma unroll
                            for (int a = 0; a < 3; a++)
#pragma unroll
                                for (int b = 0; b < 3; b++) s += D[6 * voigt(i, a) + voigt(jj, b)] * Mc[3 * a + b];
                            Kc[3 * i + jj] = s;
                        }
                }
                if (diag) {  // diagonal block: upper triangle mirrored, as complete_lt! does
                    Kc[3] = Kc[1];
                    Kc[6] = Kc[2];
                    Kc[7] = Kc[5];
                }
#pragma unroll
                for (int a = 0; a < 3; a++)
#pragma unroll
                    for (int b = 0; b < 3; b++) out[(NDN * a + b) % (NDN * NDN)] = sw ? Kc[3 * b + a] : Kc[3 * a + b];
            }
        } else if constexpr (FORM == FEASM_FORM_DOT) {
            const double *D = sD + (th >> 31);  // see above
#pragma unroll
            for (int a = 0; a < NDN; a++)
#pragma unroll
                for (int b = 0; b < NDN; b++) out[NDN * a + b] = acc[0] * D[NDN * a + b];
        } else {
            out[0] = acc[0];
        }
        b.deg = sCd[c];
        b.base = (int64_t)NDN * NDN * sCb[c] + (int64_t)r * NDN;
        const uint32_t pr = (uint32_t)(rec >> 48);
        b.pair = pr != kNoPair;
        if (b.pair) {  // the transposed block (row c, column m), in its own column
            const int c2 = (int)(pr & 255u), r2 = (int)(pr >> 8);
            b.deg2 = sCd[c2];
            b.base2 = (int64_t)NDN * NDN * sCb[c2] + (int64_t)r2 * NDN;
        }
        b.valid = true;
    };
    const auto store = [&](const BlockOut &b) {
        if (!b.valid) return;
#pragma unroll
        for (int l = 0; l < NDN; l++)
#pragma unroll
            for (int a = 0; a < NDN; a++) nzval[b.base + (int64_t)l * NDN * b.deg + a] = b.out[NDN * a + l];
        if (b.pair) {
            // K_cm = K_mc^T; the DOT forms scale a scalar by the same matrix
            // in both blocks
#pragma unroll
            for (int l = 0; l < NDN; l++)
#pragma unroll
                for (int a = 0; a < NDN; a++)
                    nzval[b.base2 + (int64_t)l * NDN * b.deg2 + a] =
                        (FORM == FEASM_FORM_DOT) ? b.out[NDN * a + l] : b.out[NDN * l + a];
        }
    };
    // The first task of every thread is computed before `before_stores`
    // runs and stored after it: the wait there (for loads issued before
    // phase 1) then comes as late as it can without including any store.
    {
        BlockOut b;
        b.valid = false;
        if (tid < NT) compute(tid, b);
        before_stores();
        store(b);
    }
    for (int t = tid + kThreads; t < NT; t += kThreads) {
        BlockOut b;
        compute(t, b);
        store(b);
    }
    __syncthreads();  // LDS is reused by the workgroup's next tile
}

// The tables of the element family, once per workgroup.
template <int NPE, int NQP>
__device__ __forceinline__ void load_tables(const FusedParams &kp, unsigned char *smem) {
    double *sN = reinterpret_cast<double *>(smem);  // the layout's tab region starts at 0
    double *sDN = sN + NQP * NPE;  // (d0, d1) pairs [q][a], then d2 [q][a]
    double *sWq = sDN + NQP * NPE * 3 + 37;  // after the material coefficients and the flag
    for (int i = threadIdx.x; i < NQP; i += blockDim.x) sWq[i] = kp.w[i];
    for (int i = threadIdx.x; i < NQP * NPE; i += blockDim.x) sN[i] = kp.N[i];
    for (int i = threadIdx.x; i < NQP * NPE; i += blockDim.x) {
        sDN[2 * i] = kp.dN[3 * i];
        sDN[2 * i + 1] = kp.dN[3 * i + 1];
        sDN[2 * NQP * NPE + i] = kp.dN[3 * i + 2];
    }
}

// XCD-aware persistent walk: consecutive workgroups land on different XCDs,
// so each XCD takes a contiguous range of the (Morton-ordered) tile list.  The
// workgroups stride through the first kAhead tiles each; the rest of a range
// (QUEUE: queue_tiles() per workgroup at least) is handed out one tile at a
// time, and a workgroup whose range has run out goes on with the next one's:
// tiles differ in time (T10: by a quarter of the mean), and with a fixed stride
// the last workgroup ended 20 % (T10), 5 % (H8) after the mean.  Measured: H8
// elasticity, 1M elements 1010 -> 984 us, T10 elasticity, 178k elements 233 ->
// 216.
//
// A workgroup runs tile t, loads the blob of t1, reads the header of t2 and
// claims the tile after it.  One lane claims: the atomic is issued before phase
// 1 and its result goes to the other wavefronts through LDS.
constexpr int kAhead = 3;
// Tiles per workgroup from which a launch hands its tiles out, 0 for never.
// The claim costs a tile of 4 to 15 us up to 0.3 us, and what it evens out is a
// part of the last tile.  Times with the queue against the stride's, at these
// tiles per workgroup:
//   FP64 gradient records   H8 3.7 1.05, 8.6 .99, 45 .98; T10 6 .97, 12 .95, 26 .87
//   packed                  4.3 1.11, 11 .99, 24 .94
//   DOT of 2 or 3           H8 4 1.10, 9 1.01, 17 .98; T10 5 1.08, 9 1.01, 18 .97
//   FP32 gradient records   H8 4.5 1.04, 9 1.00, 48 .98; T10 5 1.04, 9 1.05, 18 .97
//   DOT of 1                H8 (4 us a tile) 4 1.24, 17 1.05, 99 1.00 (FP32 1.36, 1.25, 1.25);
//                           T10 9 1.03, 18 1.01, 38 .98
// and in a batch of 24 uneven meshes, whose tiles differ more:
//   FP32 gradient records   H8 5 .94, 13 .97, 22 .91; T10 5 .97, 9 1.00, 37 .93
//   FP64 ones and packed    H8 7 1.02, 11 1.00, 19 .97, 34 .93; T10 5 1.01, 9 .99, 42 .95
//   DOT of 2 or 3           H8 6 1.07, 11 .94, 47 .97; T10 10 1.02, 18 .99, 76 .91
//   DOT of 1                H8 11 1.03, 47 1.02, 157 .99; T10 18 1.00, 40 .99, 76 .94
constexpr int queue_tiles(int npe, int form, int ndn, size_t rbytes, bool batch) {
    if (form == FEASM_FORM_DOT && ndn == 1) return npe == 10 ? 32 : batch ? 128 : 0;
    if (form == FEASM_FORM_DOT) return batch ? 10 : 12;
    const bool packed =
        npe == 8 && rbytes == 8 && (form == FEASM_FORM_DIFFUSION_ISO || form == FEASM_FORM_DIFFUSION_MAT);
    if (batch) return rbytes == 8 ? 8 : 4;
    return rbytes == 8 && !packed ? 6 : 12;
}
constexpr int kQueuePad = 32;  // words between counters: a cache line each
template <bool QUEUE>
struct TileWalk {
    uint32_t *queue;  // 8 counters, one per XCD's range, and the finished workgroups
    int64_t ntiles;
    int xcd, slot, slots;
    int32_t v = 0;         // claiming wavefront: ranges found empty
    uint32_t claimed = 0;  // claiming lane: the atomic's result
    __device__ __forceinline__ TileWalk(uint32_t *q, int64_t n)
        : queue(q), ntiles(n), xcd(blockIdx.x % 8), slot(blockIdx.x / 8), slots(gridDim.x / 8) {}
    __device__ __forceinline__ static bool claimer() { return threadIdx.x == blockDim.x - 64; }
    __device__ __forceinline__ int64_t range(int x) const { return ntiles * x / 8; }
    // the workgroup's i-th tile by the stride, -1 if its range has no such tile
    __device__ __forceinline__ int32_t strided(int i) const {
        const int64_t t = range(xcd) + slot + (int64_t)i * slots;
        return t < range(xcd + 1) ? (int32_t)t : -1;
    }
    // the tile after t by the stride, -1 after the last
    __device__ __forceinline__ int32_t after(int32_t t) const {
        return t >= 0 && (int64_t)t + slots < range(xcd + 1) ? t + slots : -1;
    }
    __device__ __forceinline__ void start(int *next) const {
        if (QUEUE && claimer()) *next = strided(kAhead - 1);
    }
    __device__ __forceinline__ void claim() {
        if (claimer() && v < 8) claimed = atomicAdd(queue + kQueuePad * ((xcd + v) & 7), 1u);
    }
    // by the claiming wavefront together, so that only `claimed` takes a vector
    // register (between the two calls)
    __device__ __forceinline__ void resolve(int *next) {
        if ((threadIdx.x >> 6) != (blockDim.x >> 6) - 1) return;
        const auto add = [&](int k) {
            uint32_t old = 0;
            if (claimer()) old = atomicAdd(queue + kQueuePad * k, 1u);
            return (uint32_t)__builtin_amdgcn_readfirstlane(old);
        };
        int32_t t = -1;
        uint32_t c = __builtin_amdgcn_readfirstlane(claimed);
        while (v < 8) {
            const int x = (xcd + v) & 7;
            const int64_t i = range(x) + (int64_t)kAhead * slots + c;
            if (i < range(x + 1)) {
                t = (int32_t)i;
                break;
            }
            if (++v < 8) {
                c = add((xcd + v) & 7);
            } else if (add(8) == gridDim.x - 1 && claimer()) {
                // every workgroup has made its last claim: ready for the next launch
                for (int k = 0; k <= 8; k++) atomicExch(queue + kQueuePad * k, 0u);
            }
        }
        if (claimer()) *next = t;
    }
};

template <int NPE, int NQP, int FORM, int NDN, typename R, bool QUEUE>
__global__ __launch_bounds__(kMaxThreads) void k_fused(TileShape shape_, TileJob job,
                                                    const TileHdr *__restrict__ hdr, int64_t ntiles,
                                                    FusedParams kp, uint32_t *queue) {
    extern __shared__ __align__(16) unsigned char smem[];
    TileShape shape = shape_;
    shape.packed = false;  // known here, so that the layout has no branch for it
    TileWalk<QUEUE> walk(queue, ntiles);
    const int32_t t0 = walk.strided(0);
    if (t0 < 0) return;
    constexpr int DS = NPE * 3;  // TileShape::dstride()
    double *sD = reinterpret_cast<double *>(smem) + NQP * NPE + NQP * DS;
    int *sNeg = reinterpret_cast<int *>(sD + 36), *sNext = sNeg + 1;
    walk.start(sNext);
    load_tables<NPE, NQP>(kp, smem);
    for (int i = threadIdx.x; i < 36; i += blockDim.x) sD[i] = kp.fp.coef[i];  // one material per launch
    // Tile t runs while the blob of tile t1 (the next one) is loaded and
    // the header of tile t2 is read.  For the gradient forms the blob load is
    // issued before phase 1 and waited for before phase 2's global stores:
    // the vector memory counter counts loads and stores together, in issue
    // order, so a load waited for after the stores would wait for every
    // store too.  The DOT forms have too short a phase 1 to hide the load:
    // they issue it after phase 1 and wait for it (and the stores) at the
    // next tile (measured faster for them).
    constexpr bool EARLY = (FORM != FEASM_FORM_DOT);
    int32_t t1 = walk.strided(1);
    TileHdr hd = load_hdr(hdr, t0);
    TileHdr hn = load_hdr(hdr, max(t1, 0));
    // (the loads are unconditional, from valid tiles, so that no register
    // copy of a pending load forces an early wait)
    Staged<false, staged_chunks<R, FORM>()> st;
    stage_issue(job, hd, nullptr, st);
    st.ready();
    for (;;) {
        const bool more = t1 >= 0;
        int32_t t2 = QUEUE ? -1 : walk.after(t1);
        TileHdr h2;    // the header of tile t2
        StagedHdr sh;  // (QUEUE: on its way)
        // without the queue the gradient forms read it while the blob goes to
        // LDS: the barrier's wait covers it, and no scalar load is left
        // pending in the phases; the store-bound DOT forms measured faster
        // with the read after the barrier
        if constexpr (!QUEUE && EARLY) h2 = load_hdr(hdr, t2 >= 0 ? t2 : t0);
        stage_store(job, hd, st, shape.layout(hd.H, hd.P, hd.NH, hd.K, hd.NT, hd.NI), smem, sD, sNeg);
        __syncthreads();
        if constexpr (!QUEUE && !EARLY) h2 = load_hdr(hdr, t2 >= 0 ? t2 : t0);
        if constexpr (QUEUE) {
            t2 = __builtin_amdgcn_readfirstlane(*sNext);
            walk.claim();
        }
        const TileHdr &hb = more ? hn : hd;
        const auto issue = [&]() {
            if constexpr (QUEUE) sh.issue(hdr, nullptr, max(t2, 0));
            stage_issue(job, hb, nullptr, st);
        };
        if constexpr (EARLY) issue();
        tile_compute<NPE, NQP, FORM, NDN, R, false>(
            shape, job, kp, hd, smem,
            [&]() {
                if constexpr (QUEUE && EARLY) {
                    // done with before phase 2: the claim and the header held
                    // in vector registers across it cost spills (H8 elasticity
                    // with a general D, 64k elements: 97.6 us, so 87.8)
                    walk.resolve(sNext);
                    sh.ready();
                    h2 = sh.get();
                }
                if constexpr (!EARLY) issue();
            },
            [&]() {
                if constexpr (EARLY) {
                    st.ready();
                } else if constexpr (QUEUE) {
                    walk.resolve(sNext);  // (phase 1 is too short for the claim)
                }
            });
        if (!more) break;
        t1 = t2;
        hd = hn;
        if constexpr (QUEUE && !EARLY)
            hn = sh.get();
        else
            hn = h2;
    }
}

// ---- H8 FP64 diffusion (scalar or 3 x 3 coefficient): packed element matrices
//
// One number per node pair, so a halo element's whole symmetric matrix (36
// doubles) takes less LDS than its gradients (192) and a block's sum reads one
// double per element instead of two nodes' gradients at every point.
// Phase 1: two lanes per halo element form the matrix in registers, half of the
// points each, and add their halves.  Phase 2: as in the general kernel, the sums in ascending
// element order.  Two workgroups of 256 threads per CU, so that one's phase 1
// (vector arithmetic) runs beside the other's loads, sums and stores.  H8
// 71x53x47: the general kernel, bound by its LDS reads, 152 us; this one 61 us.

constexpr int kPackedThreads = 256, kPackedKiB = 80, kPackedChunks = 4;

// The metric of one point for diffusion, G = J w inv(J) (coefficient) inv(J)',
// as G11 G12 G13 G22 G23 G33, from the columns of the Jacobian (derivatives of
// x along the three directions).
template <int FORM>
__device__ __forceinline__ void point_metric(const double (&j1)[3], const double (&j2)[3], const double (&j3)[3],
                                             double w, const double *coef, double (&G)[6]) {
    // the rows of the adjugate: cross products of the columns
    const double r1[3] = {j2[1] * j3[2] - j2[2] * j3[1], j2[2] * j3[0] - j2[0] * j3[2], j2[0] * j3[1] - j2[1] * j3[0]};
    const double r2[3] = {j3[1] * j1[2] - j3[2] * j1[1], j3[2] * j1[0] - j3[0] * j1[2], j3[0] * j1[1] - j3[1] * j1[0]};
    const double r3[3] = {j1[1] * j2[2] - j1[2] * j2[1], j1[2] * j2[0] - j1[0] * j2[2], j1[0] * j2[1] - j1[1] * j2[0]};
    const double det = j1[0] * r1[0] + j1[1] * r1[1] + j1[2] * r1[2];
    double s = w / det;  // det w / det^2
    double f1[3], f2[3], f3[3];
    if constexpr (FORM == FEASM_FORM_DIFFUSION_ISO) {
        s *= coef[0];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            f1[k] = s * r1[k];
            f2[k] = s * r2[k];
            f3[k] = s * r3[k];
        }
    } else {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            f1[k] = s * (coef[3 * k] * r1[0] + coef[3 * k + 1] * r1[1] + coef[3 * k + 2] * r1[2]);
            f2[k] = s * (coef[3 * k] * r2[0] + coef[3 * k + 1] * r2[1] + coef[3 * k + 2] * r2[2]);
            f3[k] = s * (coef[3 * k] * r3[0] + coef[3 * k + 1] * r3[1] + coef[3 * k + 2] * r3[2]);
        }
    }
    G[0] = r1[0] * f1[0] + r1[1] * f1[1] + r1[2] * f1[2];
    G[1] = r1[0] * f2[0] + r1[1] * f2[1] + r1[2] * f2[2];
    G[2] = r1[0] * f3[0] + r1[1] * f3[1] + r1[2] * f3[2];
    G[3] = r2[0] * f2[0] + r2[1] * f2[1] + r2[2] * f2[2];
    G[4] = r2[0] * f3[0] + r2[1] * f3[1] + r2[2] * f3[2];
    G[5] = r3[0] * f3[0] + r3[1] * f3[1] + r3[2] * f3[2];
}

// H8 with GaussRule(3, 2): the four points of one xi half (point number 4 xi +
// 2 eta + zeta), summed over the points direction by direction.  With n(c, p)
// the 1D basis value of corner side c at point p (lo or hi below), node a =
// (i, j, k) has dN_a = (s_i n_j n_k, s_j n_i n_k, s_k n_i n_j) / 2 (s = -1 or
// 1), so the metric's six components are contracted with products of 1D values
// one direction at a time and each pair adds a few of the results: about 700
// operations for the 36 pairs, against 1250 for gradients and their dot
// products.  S: packed upper triangle in the local node order.
template <int FORM>
__device__ __forceinline__ void h8_half(const double2 *__restrict__ sXY, const double *__restrict__ sZ,
                                        const int (&n)[8], bool odd, double w, const double *coef, double (&S)[36]) {
    // local node of corner (i, j, k)
    constexpr int node[2][2][2] = {{{0, 4}, {3, 7}}, {{1, 5}, {2, 6}}};
    constexpr double lo = 0.5 * (1.0 - kGauss2), hi = 0.5 * (1.0 + kGauss2);
    // n[c][p]: side c at point p
    constexpr double nb[2][2] = {{hi, lo}, {lo, hi}};
    const double x0 = odd ? lo : hi, x1 = odd ? hi : lo;  // n_0, n_1 at this half's xi
    // differences of the coordinates first (exact to rounding; a point far
    // from the origin costs no digits): D along xi on the (eta, zeta) corners,
    // E along eta at this xi on the zeta sides, F along zeta on the eta sides
    // (all halved)
    double X[2][2][2][3];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const int a = n[node[i][j][k]];
                const double2 p = sXY[a];
                X[i][j][k][0] = p.x;
                X[i][j][k][1] = p.y;
                X[i][j][k][2] = sZ[a];
            }
    const double w0 = 0.5 * x0, w1 = 0.5 * x1;
    double D[2][2][3], E[2][3], F[2][3];
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            D[j][0][c] = 0.5 * (X[1][j][0][c] - X[0][j][0][c]);
            D[j][1][c] = 0.5 * (X[1][j][1][c] - X[0][j][1][c]);
            E[j][c] = w0 * (X[0][1][j][c] - X[0][0][j][c]) + w1 * (X[1][1][j][c] - X[1][0][j][c]);
            F[j][c] = w0 * (X[0][j][1][c] - X[0][j][0][c]) + w1 * (X[1][j][1][c] - X[1][j][0][c]);
        }
    double J2[2][3], J3[2][3];  // d/deta at zeta point z, d/dzeta at eta point e
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            J2[p][c] = nb[0][p] * E[0][c] + nb[1][p] * E[1][c];
            J3[p][c] = nb[0][p] * F[0][c] + nb[1][p] * F[1][c];
        }
    // contractions: over eta (e) inside, then zeta (z)
    double A11[3][3], A22[3], A33[3], A12[2][3], A13[3][2], A23[2][2];  // [eta index][zeta index]; pairs 00 01 11
    constexpr double pp[3][2] = {{hi * hi, lo * lo}, {hi * lo, hi * lo}, {lo * lo, hi * hi}};  // n_c n_c' at point p
#pragma unroll
    for (int i = 0; i < 3; i++) {
        A22[i] = A33[i] = 0.0;
#pragma unroll
        for (int j = 0; j < 3; j++) A11[i][j] = 0.0;
#pragma unroll
        for (int j = 0; j < 2; j++) A12[j][i] = A13[i][j] = 0.0;
    }
    A23[0][0] = A23[0][1] = A23[1][0] = A23[1][1] = 0.0;
#pragma unroll
    for (int z = 0; z < 2; z++) {
        double G[2][6];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            double J1[3];
#pragma unroll
            for (int c = 0; c < 3; c++)
                J1[c] = nb[0][e] * (nb[0][z] * D[0][0][c] + nb[1][z] * D[0][1][c]) +
                        nb[1][e] * (nb[0][z] * D[1][0][c] + nb[1][z] * D[1][1][c]);
            point_metric<FORM>(J1, J2[z], J3[e], w, coef, G[e]);
        }
        const double t22 = G[0][3] + G[1][3];
        double t11[3], t13[3], t33[3], t12[2], t23[2];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            t11[i] = pp[i][0] * G[0][0] + pp[i][1] * G[1][0];
            t13[i] = pp[i][0] * G[0][2] + pp[i][1] * G[1][2];
            t33[i] = pp[i][0] * G[0][5] + pp[i][1] * G[1][5];
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            t12[j] = nb[j][0] * G[0][1] + nb[j][1] * G[1][1];
            t23[j] = nb[j][0] * G[0][4] + nb[j][1] * G[1][4];
        }
#pragma unroll
        for (int i = 0; i < 3; i++) {
            A22[i] += pp[i][z] * t22;
            A33[i] += t33[i];
#pragma unroll
            for (int j = 0; j < 3; j++) A11[i][j] += pp[j][z] * t11[i];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                A12[j][i] += pp[i][z] * t12[j];
                A13[i][j] += nb[j][z] * t13[i];
            }
        }
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 2; k++) A23[j][k] += nb[k][z] * t23[j];
    }
    // pairs of (eta, zeta) corners (j, k), (l, m): T the xi xi part, B the eta and
    // zeta parts, U[jk][lm] the cross part with xi derived on the jk side
    double U[4][4];
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int j = p >> 1, k = p & 1, l = q >> 1, m = q & 1;
            const double a = A12[j][k + m], b = A13[j + l][k];
            U[p][q] = (l ? a : -a) + (m ? b : -b);
        }
    const double q0 = 0.25 * x0 * x0, q1 = 0.25 * x1 * x1, q01 = 0.25 * x0 * x1, h0 = 0.25 * x0, h1 = 0.25 * x1;
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int q = p; q < 4; q++) {
            const int j = p >> 1, k = p & 1, l = q >> 1, m = q & 1;
            const double T = 0.25 * A11[j + l][k + m];
            const double a22 = A22[k + m], a33 = A33[j + l];
            const double c1 = A23[l][k], c2 = A23[j][m];  // d/deta on jk with d/dzeta on lm, and the other way
            const double B = (j == l ? a22 : -a22) + (k == m ? a33 : -a33) + (j == m ? c1 : -c1) + (k == l ? c2 : -c2);
            const double V = U[p][q] + U[q][p];
            const auto put = [&](int x, int y, double v) { S[x > y ? x * (x + 1) / 2 + y : y * (y + 1) / 2 + x] = v; };
            put(node[0][j][k], node[0][l][m], T + q0 * B - h0 * V);
            put(node[1][j][k], node[1][l][m], T + q1 * B + h1 * V);
            put(node[0][j][k], node[1][l][m], q01 * B - T + (h0 * U[q][p] - h1 * U[p][q]));
            if (p != q) put(node[1][j][k], node[0][l][m], q01 * B - T + (h0 * U[p][q] - h1 * U[q][p]));
        }
}

template <int FORM, bool LDSCOEF, typename BeforeStores>
__device__ __forceinline__ void packed_tile(const TileShape &shape, const TileJob &job, const FusedParams &kp,
                                            const TileHdr &hd, unsigned char *smem, const BeforeStores &before_stores) {
    constexpr int NPE = 8, NP = 36, PS = NP | 1;  // TileShape::packed_stride()
    const int tid = threadIdx.x;
    const TileShape::Layout L = shape.layout(hd.H, hd.P, hd.NH, hd.K, hd.NT, hd.NI);
    const double *coef = LDSCOEF ? reinterpret_cast<const double *>(smem) + 8 * 8 * 4 : kp.fp.coef;
    const uint64_t *sTask = reinterpret_cast<const uint64_t *>(smem + L.task);
    const uint16_t *sItem = reinterpret_cast<const uint16_t *>(smem + L.item);
    const double2 *sXY = reinterpret_cast<const double2 *>(smem + L.X);
    const double *sZ = reinterpret_cast<const double *>(smem + L.X) + 2 * hd.NH;
    const int64_t *sCb = reinterpret_cast<const int64_t *>(smem + L.cbase);
    double *sS = reinterpret_cast<double *>(smem + L.U);

    // two lanes per element, each half of the points; i < 2 H for both or none
    const bool odd = tid & 1;
    for (int i = tid; i < 2 * hd.H; i += kPackedThreads) {
        const int h = i >> 1;
        const uint16_t *cn = reinterpret_cast<const uint16_t *>(smem + L.lconn) + h * NPE;
        int n[NPE];
#pragma unroll
        for (int a = 0; a < NPE; a++) n[a] = cn[a];
        double S[NP];
        h8_half<FORM>(sXY, sZ, n, odd, 1.0, coef, S);  // every weight of the rule is 1
        // each lane adds the other's half of the points for its half of the
        // pairs (quad_perm 1,0,3,2: the neighbour's value)
        constexpr int HALF = NP / 2;
#pragma unroll
        for (int p = 0; p < HALF; p++) {
            const double keep = odd ? S[p + HALF] : S[p], send = odd ? S[p] : S[p + HALF];
            const int2 w = __builtin_bit_cast(int2, send);
            const int2 x = make_int2(__builtin_amdgcn_mov_dpp(w.x, 0xB1, 0xf, 0xf, false),
                                     __builtin_amdgcn_mov_dpp(w.y, 0xB1, 0xf, 0xf, false));
            const double sum = keep + __builtin_bit_cast(double, x);
            sS[h * PS + p + (odd ? HALF : 0)] = sum;
        }
    }
    __syncthreads();
    before_stores();

    double *__restrict__ nzval = job.nzval;
    for (int t = tid; t < hd.NT; t += kPackedThreads) {
        const uint64_t rec = sTask[t];
        if ((uint32_t)rec == kNullTask) continue;
        const int k = (int)((rec >> 16) & 255u);
        const uint16_t *items = sItem + (uint32_t)((rec >> 32) & 0xffffu);
        // items, then their numbers, four at a time; summed in item order
        double acc = 0.0;
        for (int j = 0; j < k; j += 4) {
            uint32_t it[4];
            double x[4];
#pragma unroll
            for (int u = 0; u < 4; u++) it[u] = items[min(j + u, k - 1)];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t ac = (it[u] >> 4) & 15u, ar = it[u] & 15u, lo = min(ac, ar), hi = max(ac, ar);
                x[u] = sS[(it[u] >> 8) * PS + (__umul24(hi, hi + 1) >> 1) + lo];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) acc = j + u < k ? acc + x[u] : acc;
        }
        nzval[sCb[rec & 255u] + ((rec >> 8) & 255u)] = acc;
        const uint32_t pr = (uint32_t)(rec >> 48);
        if (pr != kNoPair) nzval[sCb[pr & 255u] + (pr >> 8)] = acc;  // the transposed block
    }
}

template <int NPE, int NQP, int FORM, int NDN, typename R, bool QUEUE>
__global__ __launch_bounds__(kPackedThreads, 2) void k_packed(TileShape shape_, TileJob job,
                                                           const TileHdr *__restrict__ hdr, int64_t ntiles,
                                                           FusedParams kp, uint32_t *queue) {
    static_assert(NPE == 8 && NQP == 8 && NDN == 1 && sizeof(R) == 8);
    extern __shared__ __align__(16) unsigned char smem[];
    TileShape shape = shape_;
    shape.packed = true;
    TileWalk<QUEUE> walk(queue, ntiles);
    const int32_t t0 = walk.strided(0);
    if (t0 < 0) return;
    double *sD = reinterpret_cast<double *>(smem) + NQP * NPE * 4;
    int *sNeg = reinterpret_cast<int *>(sD + 36), *sNext = sNeg + 1;
    walk.start(sNext);
    int32_t t1 = walk.strided(1);
    TileHdr hd = load_hdr(hdr, t0);
    TileHdr hn = load_hdr(hdr, max(t1, 0));
    Staged<false, kPackedChunks> st;
    stage_issue(job, hd, nullptr, st);
    st.ready();
    for (;;) {
        const bool more = t1 >= 0;
        int32_t t2 = QUEUE ? -1 : walk.after(t1);
        TileHdr h2;  // the header of tile t2, as in k_fused
        StagedHdr sh;
        if constexpr (!QUEUE) h2 = load_hdr(hdr, t2 >= 0 ? t2 : t0);
        stage_store(job, hd, st, shape.layout(hd.H, hd.P, hd.NH, hd.K, hd.NT, hd.NI), smem, sD, sNeg);
        __syncthreads();
        if constexpr (QUEUE) {
            t2 = __builtin_amdgcn_readfirstlane(*sNext);
            walk.claim();
            sh.issue(hdr, nullptr, max(t2, 0));
        }
        stage_issue(job, more ? hn : hd, nullptr, st);  // waited for before this tile's stores
        packed_tile<FORM, false>(shape, job, kp, hd, smem, [&]() {
            if constexpr (QUEUE) sh.ready();
            st.ready();
            if constexpr (QUEUE) walk.resolve(sNext);
        });
        if (!more) break;
        __syncthreads();
        t1 = t2;
        hd = hn;
        if constexpr (QUEUE)
            hn = sh.get();
        else
            hn = h2;
    }
}

// One entry per mesh of a batched launch.
struct BatchEntry {
    TileJob job;
    FusedParams kp;
    TileShape shape;
    int64_t tile0;
};

// Persistent batched launch: as k_fused over the global tile list (all
// meshes' tiles, mesh after mesh); every tile carries its mesh's
// coefficients and arrays.  One launch covers the meshes of one element
// type, rule, arithmetic and form.
template <int NPE, int NQP, int FORM, int NDN, typename R, bool QUEUE>
__global__ __launch_bounds__(kMaxThreads) void k_fused_batch(const BatchEntry *__restrict__ entries,
                                                          const int32_t *__restrict__ tile_entry,
                                                          const TileHdr *__restrict__ hdr, int64_t ntiles,
                                                          TileShape shape_, uint32_t *queue) {
    extern __shared__ __align__(16) unsigned char smem[];
    TileShape shape = shape_;
    shape.packed = false;  // known here, so that the layout has no branch for it
    TileWalk<QUEUE> walk(queue, ntiles);
    const int32_t t0 = walk.strided(0);
    if (t0 < 0) return;
    constexpr int DS = NPE * 3;  // TileShape::dstride()
    double *sD = reinterpret_cast<double *>(smem) + NQP * NPE + NQP * DS;
    int *sNeg = reinterpret_cast<int *>(sD + 36), *sNext = sNeg + 1;
    walk.start(sNext);
    load_tables<NPE, NQP>(entries[tile_entry[t0]].kp, smem);
    // the tile walk and its loads as in k_fused; every tile also brings its
    // mesh's coefficients
    constexpr bool EARLY = (FORM != FEASM_FORM_DOT);
    int32_t t1 = walk.strided(1);
    TileHdr hd = load_hdr(hdr, t0);
    const BatchEntry *E = entries + tile_entry[t0];
    TileHdr hn = load_hdr(hdr, max(t1, 0));
    const BatchEntry *En = entries + tile_entry[max(t1, 0)];
    Staged<true, staged_chunks<R, FORM>()> st;
    stage_issue(E->job, hd, E->kp.fp.coef, st);
    st.ready();
    for (;;) {
        const bool more = t1 >= 0;
        int32_t t2 = QUEUE ? -1 : walk.after(t1);
        TileHdr h2;  // the header and entry of tile t2, as in k_fused
        const BatchEntry *E2 = nullptr;
        StagedHdr sh;
        if constexpr (!QUEUE && EARLY) {
            h2 = load_hdr(hdr, t2 >= 0 ? t2 : t0);
            E2 = entries + tile_entry[t2 >= 0 ? t2 : t0];
        }
        stage_store(E->job, hd, st, shape.layout(hd.H, hd.P, hd.NH, hd.K, hd.NT, hd.NI), smem, sD, sNeg);
        __syncthreads();
        if constexpr (!QUEUE && !EARLY) {
            h2 = load_hdr(hdr, t2 >= 0 ? t2 : t0);
            E2 = entries + tile_entry[t2 >= 0 ? t2 : t0];
        }
        if constexpr (QUEUE) {
            t2 = __builtin_amdgcn_readfirstlane(*sNext);
            walk.claim();
        }
        const TileHdr &hb = more ? hn : hd;
        const BatchEntry *Eb = more ? En : E;
        const auto issue = [&]() {
            if constexpr (QUEUE) sh.issue(hdr, tile_entry, max(t2, 0));
            stage_issue(Eb->job, hb, Eb->kp.fp.coef, st);
        };
        if constexpr (EARLY) issue();
        tile_compute<NPE, NQP, FORM, NDN, R, true>(
            shape, E->job, E->kp, hd, smem,
            [&]() {
                if constexpr (QUEUE && EARLY) walk.resolve(sNext);
                if constexpr (!EARLY) issue();
            },
            [&]() {
                if constexpr (EARLY) {
                    if constexpr (QUEUE) sh.ready();
                    st.ready();
                } else if constexpr (QUEUE) {
                    walk.resolve(sNext);  // (phase 1 is too short for the claim)
                }
            });
        if (!more) break;
        t1 = t2;
        hd = hn;
        E = En;
        if constexpr (QUEUE) {
            hn = sh.get();
            En = entries + sh.entry();
        } else {
            hn = h2;
            En = E2;
        }
    }
}

// k_packed over the global tile list of a batched launch.
template <int NPE, int NQP, int FORM, int NDN, typename R, bool QUEUE>
__global__ __launch_bounds__(kPackedThreads, 2) void k_packed_batch(const BatchEntry *__restrict__ entries,
                                                                 const int32_t *__restrict__ tile_entry,
                                                                 const TileHdr *__restrict__ hdr, int64_t ntiles,
                                                                 TileShape shape_, uint32_t *queue) {
    static_assert(NPE == 8 && NQP == 8 && NDN == 1 && sizeof(R) == 8);
    extern __shared__ __align__(16) unsigned char smem[];
    TileShape shape = shape_;
    shape.packed = true;
    TileWalk<QUEUE> walk(queue, ntiles);
    const int32_t t0 = walk.strided(0);
    if (t0 < 0) return;
    double *sD = reinterpret_cast<double *>(smem) + NQP * NPE * 4;
    int *sNeg = reinterpret_cast<int *>(sD + 36), *sNext = sNeg + 1;
    walk.start(sNext);
    int32_t t1 = walk.strided(1);
    TileHdr hd = load_hdr(hdr, t0);
    const BatchEntry *E = entries + tile_entry[t0];
    TileHdr hn = load_hdr(hdr, max(t1, 0));
    const BatchEntry *En = entries + tile_entry[max(t1, 0)];
    Staged<true, kPackedChunks> st;
    stage_issue(E->job, hd, E->kp.fp.coef, st);
    st.ready();
    for (;;) {
        const bool more = t1 >= 0;
        int32_t t2 = QUEUE ? -1 : walk.after(t1);
        TileHdr h2;  // the header and entry of tile t2, as in k_fused
        const BatchEntry *E2 = nullptr;
        StagedHdr sh;
        if constexpr (!QUEUE) {
            h2 = load_hdr(hdr, t2 >= 0 ? t2 : t0);
            E2 = entries + tile_entry[t2 >= 0 ? t2 : t0];
        }
        stage_store(E->job, hd, st, shape.layout(hd.H, hd.P, hd.NH, hd.K, hd.NT, hd.NI), smem, sD, sNeg);
        __syncthreads();
        const TileHdr &hb = more ? hn : hd;
        const BatchEntry *Eb = more ? En : E;
        if constexpr (QUEUE) {
            t2 = __builtin_amdgcn_readfirstlane(*sNext);
            walk.claim();
            sh.issue(hdr, tile_entry, max(t2, 0));
        }
        stage_issue(Eb->job, hb, Eb->kp.fp.coef, st);
        packed_tile<FORM, true>(shape, E->job, E->kp, hd, smem, [&]() {
            if constexpr (QUEUE) sh.ready();
            st.ready();
            if constexpr (QUEUE) walk.resolve(sNext);
        });
        if (!more) break;
        __syncthreads();
        t1 = t2;
        hd = hn;
        E = En;
        if constexpr (QUEUE) {
            hn = sh.get();
            En = entries + sh.entry();
        } else {
            hn = h2;
            En = E2;
        }
    }
}

TileJob make_job(const feasm_mesh *m, const TileSet &t, double *nzval) {
    TileJob j;
    j.hdr = static_cast<const TileHdr *>(t.hdr->p);
    j.blob = static_cast<const unsigned char *>(t.blob->p);
    j.hnodes = dp<int32_t>(t.hnodes);
    j.xyz = dp<double>(m->xyz);
    j.nzval = nzval;
    return j;
}

// workgroups of a persistent launch: as many as stay resident (LDS-bound),
// a multiple of the 8 XCDs, and no more than the tiles need
unsigned persistent_grid(feasm_ctx *ctx, size_t budget, int64_t ntiles) {
    int cus = 0;
    FEASM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
    const size_t lds_cu = 160 * 1024;
    const int per_cu = (int)std::max<size_t>(1, lds_cu / std::max<size_t>(budget, 1));
    int64_t grid = (int64_t)cus * per_cu;
    grid = std::max<int64_t>(8, (grid / 8) * 8);
    const int64_t need = 8 * ((ntiles + 7) / 8);
    return (unsigned)std::min(grid, std::max<int64_t>(need, 8));
}

// A launch leaves its queue cleared for the next one, so launches that share
// one must run one after the other: those on the context's stream do.  A launch
// recorded into a graph may be replayed on another stream, beside the next
// one: it gets none and walks with the fixed stride.
constexpr size_t kQueueBytes = sizeof(uint32_t) * kQueuePad * 9;
uint32_t *ctx_tile_queue(feasm_ctx *ctx) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    FEASM_HIP(hipStreamIsCapturing(ctx->stream, &cs));
    if (cs != hipStreamCaptureStatusNone) return nullptr;
    if (!ctx->tile_queue) {
        ctx->tile_queue = dev_alloc(kQueueBytes);
        FEASM_HIP(hipMemsetAsync(ctx->tile_queue->p, 0, kQueueBytes, ctx->stream));
    }
    return dp<uint32_t>(ctx->tile_queue);
}

template <int NPE, int NQP, int FORM, int NDN, typename R>
void go(feasm_ctx *ctx, const feasm_mesh *m, const Pattern &p, const TileSet &t, const FusedParams &kp,
        double *nzval) {
    constexpr bool PACKED = NPE == 8 && sizeof(R) == 8 && (FORM == FEASM_FORM_DIFFUSION_ISO || FORM == FEASM_FORM_DIFFUSION_MAT);
    constexpr int QT = queue_tiles(NPE, FORM, NDN, sizeof(R), false);
    static_assert(QT == 0 || QT >= kAhead, "a workgroup strides through its first tiles");
    const unsigned grid = persistent_grid(ctx, t.shape.budget, t.ntiles);
    uint32_t *queue = QT > 0 && t.ntiles >= (int64_t)QT * grid ? ctx_tile_queue(ctx) : nullptr;
    auto kern = [&] {
        if constexpr (PACKED)
            return queue ? k_packed<NPE, NQP, FORM, NDN, R, true> : k_packed<NPE, NQP, FORM, NDN, R, false>;
        else
            return queue ? k_fused<NPE, NQP, FORM, NDN, R, QT != 0> : k_fused<NPE, NQP, FORM, NDN, R, false>;
    }();
    const int budget = (int)t.shape.budget;
    FEASM_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, budget));
    TileJob job = make_job(m, t, nzval);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(t.shape.threads), budget, ctx->stream, t.shape, job, job.hdr, t.ntiles,
                       kp, queue);
    FEASM_HIP(hipGetLastError());
}

template <int NPE, int NQP, typename R>
void by_form(feasm_ctx *ctx, const feasm_mesh *m, const Pattern &p, const TileSet &t, const FusedParams &kp,
             double *nzval) {
    switch (kp.fp.form) {
        case FEASM_FORM_LIN_ELASTIC:
            if (kp.cubic) return go<NPE, NQP, kFormElasticCubic, 3, R>(ctx, m, p, t, kp, nzval);
            return go<NPE, NQP, FEASM_FORM_LIN_ELASTIC, 3, R>(ctx, m, p, t, kp, nzval);
        case FEASM_FORM_DIFFUSION_ISO: return go<NPE, NQP, FEASM_FORM_DIFFUSION_ISO, 1, R>(ctx, m, p, t, kp, nzval);
        case FEASM_FORM_DIFFUSION_MAT: return go<NPE, NQP, FEASM_FORM_DIFFUSION_MAT, 1, R>(ctx, m, p, t, kp, nzval);
        case FEASM_FORM_DOT:
            if (kp.fp.ndn == 1) return go<NPE, NQP, FEASM_FORM_DOT, 1, R>(ctx, m, p, t, kp, nzval);
            if (kp.fp.ndn == 2) return go<NPE, NQP, FEASM_FORM_DOT, 2, R>(ctx, m, p, t, kp, nzval);
            if (kp.fp.ndn == 3) return go<NPE, NQP, FEASM_FORM_DOT, 3, R>(ctx, m, p, t, kp, nzval);
            break;
    }
    throw Error(FEASM_EUNSUPPORTED, "unsupported form in the fused kernel");
}

template <typename R>
void dispatch(feasm_ctx *ctx, const feasm_mesh *m, const Pattern &p, const TileSet &t, const FusedParams &kp,
              double *nzval) {
    if (t.shape.npe == 8 && t.shape.nqp == 8) return by_form<8, 8, R>(ctx, m, p, t, kp, nzval);
    if (t.shape.npe == 10 && t.shape.nqp == 4) return by_form<10, 4, R>(ctx, m, p, t, kp, nzval);
    throw Error(FEASM_EUNSUPPORTED, "the fused kernel covers H8 with 2x2x2 Gauss and T10 with 4-point rules");
}

template <int NPE, int NQP, int FORM, int NDN, typename R>
void go_batch(feasm_ctx *ctx, const BatchLaunch &b) {
    constexpr bool PACKED = NPE == 8 && sizeof(R) == 8 && (FORM == FEASM_FORM_DIFFUSION_ISO || FORM == FEASM_FORM_DIFFUSION_MAT);
    auto kern = [&] {
        if constexpr (PACKED)
            return b.queue ? k_packed_batch<NPE, NQP, FORM, NDN, R, true> : k_packed_batch<NPE, NQP, FORM, NDN, R, false>;
        else
            return b.queue ? k_fused_batch<NPE, NQP, FORM, NDN, R, true> : k_fused_batch<NPE, NQP, FORM, NDN, R, false>;
    }();
    FEASM_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)b.budget));
    hipLaunchKernelGGL(kern, dim3(b.grid), dim3(b.threads), b.budget, ctx->stream,
                       static_cast<const BatchEntry *>(b.entries->p), dp<int32_t>(b.tile_entry),
                       static_cast<const TileHdr *>(b.hdr->p), b.ntiles, b.shape,
                       b.queue ? dp<uint32_t>(b.queue) : nullptr);
    FEASM_HIP(hipGetLastError());
}

}  // namespace

void prepare_batch_launch(feasm_ctx *ctx, BatchLaunch &b, const std::vector<BatchMesh> &items) {
    std::vector<BatchEntry> host;
    std::vector<int32_t> tile_entry;
    b.ntiles = 0;
    b.budget = 0;
    for (size_t i = 0; i < items.size(); i++) {
        const BatchMesh &it = items[i];
        BatchEntry E;
        E.job = make_job(it.mesh, *it.tiles, it.nzval);
        E.kp.fp = it.fp;
        E.kp.cubic = (it.fp.form == FEASM_FORM_LIN_ELASTIC && cubic_symmetry(it.fp.coef)) ? 1 : 0;
        const DevQTable &qt = device_qtable(ctx, it.mesh->etype, it.rule, it.order);
        E.kp.N = qt.N();
        E.kp.dN = qt.dN();
        E.kp.w = qt.w();
        E.shape = it.tiles->shape;
        E.tile0 = b.ntiles;
        for (int64_t t = 0; t < it.tiles->ntiles; t++) tile_entry.push_back((int32_t)i);
        b.ntiles += it.tiles->ntiles;
        b.budget = std::max(b.budget, it.tiles->shape.budget);
        b.threads = it.tiles->shape.threads;
        if (i == 0) b.shape = it.tiles->shape;
        const TileShape &s0 = b.shape, &si = it.tiles->shape;
        FEASM_REQUIRE(si.npe == s0.npe && si.nqp == s0.nqp && si.rbytes == s0.rbytes && si.grad == s0.grad,
                      FEASM_ESTATE, "meshes of one batched launch differ in their tile layout");
        host.push_back(E);
    }
    b.entries = dev_alloc(std::max<size_t>(host.size() * sizeof(BatchEntry), 16));
    b.tile_entry = dev_alloc(std::max<size_t>(tile_entry.size() * 4, 4));
    b.hdr = dev_alloc(std::max<size_t>((size_t)b.ntiles * sizeof(TileHdr), 16));
    FEASM_HIP(hipMemcpy(b.entries->p, host.data(), host.size() * sizeof(BatchEntry), hipMemcpyHostToDevice));
    FEASM_HIP(hipMemcpy(b.tile_entry->p, tile_entry.data(), tile_entry.size() * 4, hipMemcpyHostToDevice));
    // on the launches' own stream: device work on the null stream need not be
    // done when the call returns, and the context's stream does not wait for it
    for (size_t i = 0; i < items.size(); i++)  // the meshes' headers, one after the other
        FEASM_HIP(hipMemcpyAsync(static_cast<TileHdr *>(b.hdr->p) + host[i].tile0, items[i].tiles->hdr->p,
                                 (size_t)items[i].tiles->ntiles * sizeof(TileHdr), hipMemcpyDeviceToDevice,
                                 ctx->stream));
    b.grid = persistent_grid(ctx, b.budget, b.ntiles);
    if (b.ntiles >= (int64_t)queue_tiles(b.npe, b.kform, b.ndn, (size_t)b.rbytes, true) * b.grid) {
        b.queue = dev_alloc(kQueueBytes);
        FEASM_HIP(hipMemsetAsync(b.queue->p, 0, kQueueBytes, ctx->stream));
    }
}

namespace {

template <int NPE, int NQP, typename R>
void batch_by_form(feasm_ctx *ctx, const BatchLaunch &b) {
    switch (b.kform) {
        case FEASM_FORM_LIN_ELASTIC: return go_batch<NPE, NQP, FEASM_FORM_LIN_ELASTIC, 3, R>(ctx, b);
        case kFormElasticCubic: return go_batch<NPE, NQP, kFormElasticCubic, 3, R>(ctx, b);
        case FEASM_FORM_DIFFUSION_ISO: return go_batch<NPE, NQP, FEASM_FORM_DIFFUSION_ISO, 1, R>(ctx, b);
        case FEASM_FORM_DIFFUSION_MAT: return go_batch<NPE, NQP, FEASM_FORM_DIFFUSION_MAT, 1, R>(ctx, b);
        case FEASM_FORM_DOT:
            if (b.ndn == 1) return go_batch<NPE, NQP, FEASM_FORM_DOT, 1, R>(ctx, b);
            if (b.ndn == 2) return go_batch<NPE, NQP, FEASM_FORM_DOT, 2, R>(ctx, b);
            if (b.ndn == 3) return go_batch<NPE, NQP, FEASM_FORM_DOT, 3, R>(ctx, b);
            break;
    }
    throw Error(FEASM_EUNSUPPORTED, "unsupported form in the batched launch");
}

}  // namespace

int fused_kernel_form(const FormParams &fp) {
    if (fp.form == FEASM_FORM_LIN_ELASTIC && cubic_symmetry(fp.coef)) return kFormElasticCubic;
    return fp.form;
}

void launch_batch(feasm_ctx *ctx, const BatchLaunch &b) {
    if (b.ntiles == 0) return;
    if (b.npe == 8 && b.nqp == 8) {
        if (b.rbytes == 4) return batch_by_form<8, 8, float>(ctx, b);
        return batch_by_form<8, 8, double>(ctx, b);
    }
    if (b.npe == 10 && b.nqp == 4) {
        if (b.rbytes == 4) return batch_by_form<10, 4, float>(ctx, b);
        return batch_by_form<10, 4, double>(ctx, b);
    }
    throw Error(FEASM_EUNSUPPORTED, "batched launch covers H8 2x2x2 Gauss and T10 4-point rules");
}

namespace {

// one workgroup per tile: the tile's halo coordinates into its blob
__global__ __launch_bounds__(256) void k_tile_coords(TileShape shape, const TileHdr *__restrict__ hdr,
                                                     int64_t ntiles, const int32_t *__restrict__ hnodes,
                                                     const double *__restrict__ xyz, unsigned char *__restrict__ blob) {
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const TileHdr hd = hdr[t];
        const TileShape::Layout L = shape.layout(hd.H, hd.P, hd.NH, hd.K, hd.NT, hd.NI);
        double *X = reinterpret_cast<double *>(blob + hd.blob + (L.X - L.cbase));
        for (int i = threadIdx.x; i < hd.NH; i += blockDim.x) {  // (x, y) pairs, then the z values
            const int64_t n = hnodes[hd.x0 + i];
            X[2 * i] = xyz[3 * n];
            X[2 * i + 1] = xyz[3 * n + 1];
            X[2 * hd.NH + i] = xyz[3 * n + 2];
        }
    }
}

}  // namespace

void refresh_tile_coords(feasm_mesh *m, TileSet &t) {
    if (t.ntiles == 0) return;
    feasm_ctx *ctx = m->ctx;
    hipLaunchKernelGGL(k_tile_coords, dim3((unsigned)std::min<int64_t>(t.ntiles, 1 << 16)), dim3(256), 0,
                       ctx->stream, t.shape, static_cast<const TileHdr *>(t.hdr->p), t.ntiles, dp<int32_t>(t.hnodes),
                       dp<double>(m->xyz), static_cast<unsigned char *>(t.blob->p));
    FEASM_HIP(hipGetLastError());
}

bool fused_supported(int npe, int nqp) { return (npe == 8 && nqp == 8) || (npe == 10 && nqp == 4); }

TileShape tile_shape_for(feasm_ctx *ctx, int npe, int nqp, int form, int precision, int nodes, int kib, int threads) {
    TileShape s;
    s.npe = npe;
    s.nqp = nqp;
    s.rbytes = (precision == FEASM_MIXED) ? 4 : 8;
    // H8 only: a T10's 55 pairs leave too few registers (measured 50 -> 65 us on 20x21x19)
    s.packed = npe == 8 && precision == FEASM_FP64 && (form == FEASM_FORM_DIFFUSION_ISO || form == FEASM_FORM_DIFFUSION_MAT);
    s.grad = (form != FEASM_FORM_DOT) && !s.packed;
    int lds = 0;
    FEASM_HIP(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, ctx->device));
    s.budget = (size_t)std::min(lds, (s.packed ? kPackedKiB : 160) * 1024);
    // measured best on MI355X: DOT tiles (tiny records, not bound by LDS)
    // with 64 nodes list more block tasks than the workgroup has threads
    s.max_nodes = (form == FEASM_FORM_DOT) ? 32 : 64;
    s.max_halo = 255;
    s.threads = 1024;
    if (nodes > 0) s.max_nodes = std::min(255, nodes);
    if (kib > 0) s.budget = std::min(s.budget, (size_t)kib * 1024);
    if (threads == 256 || threads == 512 || threads == 1024) s.threads = threads;
    if (s.packed) s.threads = kPackedThreads;  // two workgroups a CU, two lanes an element
    return s;
}

void launch_fused(feasm_ctx *ctx, const feasm_mesh *m, const Pattern &p, const TileSet &t, const DevQTable &qt,
                  const FormParams &fp, int precision, double *nzval) {
    if (t.ntiles == 0) return;
    FusedParams kp;
    kp.fp = fp;
    kp.cubic = (fp.form == FEASM_FORM_LIN_ELASTIC && cubic_symmetry(fp.coef)) ? 1 : 0;
    kp.N = qt.N();
    kp.dN = qt.dN();
    kp.w = qt.w();
    if (precision == FEASM_MIXED)
        dispatch<float>(ctx, m, p, t, kp, nzval);
    else
        dispatch<double>(ctx, m, p, t, kp, nzval);
}

}  // namespace feasm
