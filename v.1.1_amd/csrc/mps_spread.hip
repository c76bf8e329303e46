// mps_spread.hip -- the spread form of the explicit step, for meshes that leave most of the chip idle.
//
// A small mesh is bound by latency, not by throughput: in the patch form (mps_kernels.hip) a step of 1,000 hex8 elements
// takes as long as one of 30,000, about 19 us, of which 14 us is one wavefront walking through 2,700 instructions per
// element and 5 us the node kernel's chain of dependent loads.  Here a step is ONE launch (a launch in a replayed graph
// costs 1.6 us, no more than a grid barrier among as many workgroups), and the element work is spread over idle lanes:
//   - workgroup b first brings the distinct nodes of its elements to step k: it sums the element forces of step k-1 at
//     each node, solves step k-1 and predicts u_k, for every node it needs (a node shared by several workgroups is
//     updated by each of them, with the same bits; its owner writes it back).  u and the half-step velocity w are
//     double-buffered, since neighbours still read the old ones;
//   - then it computes the forces of its elements from the nodes in LDS -- eight lanes per hex8 element, one Gauss point
//     each -- and writes every nodal force to its place in node order, so that the next step reads each node's forces as
//     one contiguous run.  A second wave takes the stable dt meanwhile, exact for every element: no skip, no certificate.
// Two dependent global loads are left (tables and control; state and forces), about 1 us each, then 1.4 us of element
// work.  Every sum keeps the patch form's order -- the forces of a node are added per patch of MPS_PATCH elements and then
// over the patches -- and an element's arithmetic is the same function by function, so both forms give the same bits.
//
// Measured, us per step, patch form / here.  hex8 FP64: 1,000 elements 17.7 / 5.6, 8,000 18.4 / 7.4, 15,600 19.1 / 10.2,
// 29,800 19.2 / 16.8, 46,700 19.4 / 23.2; tet4 FP64: 750 12.3 / 6.6, 10,400 12.2 / 6.7, 48,000 12.2 / 10.2, 93,800 13.6 /
// 16.8; FP32 form: 10,400 9.7 / 6.4, 48,000 10.0 / 10.3.  Hex8 meshes in the FP32 form keep the patch kernels, whose FMAs the
// compiler chooses (cof3_c in mps_device.h).
// Every node is updated by all the workgroups that hold it (4.5 per 8 hex8 elements where the patch form has 1.03 per
// element), so past the size where the lanes are no longer idle the patch form is the better one.
// With energies every step and loads (hex8 FP64): 512 elements 29.3 / 7.3, 12,200 30.2 / 12.1, 35,800 30.9 / 24.5; tet4 750
// 22.0 / 7.2, 55,600 21.6 / 13.4, FP32 form 55,600 22.6 / 12.9; with viscosity and loads (FP64 Belytschko): 512 23.4 / 6.6,
// 12,200 25.2 / 11.6, 31,700 29.2 / 22.8.  The patch form takes three launches for these steps; here the external forces
// and the energy sums are extra workgroups of the step's launch, on a path of their own from the first instruction, and
// without the pressure loads' code: sharing the element workgroups' prologue, with that code, cost 48 registers, two of
// five waves per SIMD, and 18.7 instead of 16.8 us at 29,800 elements.
// Tried: one wave per workgroup, which takes the dt and the forces in turn (half the waves): 2 us more at 1,000 elements and
// the same above 30,000, where the issue of 1,380 vector instructions per 8 elements is the bound, not the waves in flight.
// Tried: 16 and 32 hex8 elements per workgroup: fewer shared nodes, but 0.4 to 1.8 us more up to 2,000 elements and
// nothing gained above.
#include "../../include/mps_gpu.h"
#include "mps_device.h"
#include "mps_kernels.h"

using namespace mpsd;

namespace {

// LDS of the hex8 element phase, in values per element: butterfly coefficients of X and u (42), later the moment
// sums (21); stress columns of the eight points (72); face triangle areas (12).  Coefficients
// and columns are read in 16-byte pieces; with these strides the eight elements of a wave fall into different banks.
constexpr int kCoef = 44, kCol = 76, kArea = 12;

// LDS exchange between the lanes of one wavefront: LDS operations of a wave stay in order, so only the compiler has to
// be kept from moving them.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Buffers of u and w: index 0 the solve's own arrays (u, v holding w), 1 the alternate ones.  The step with index ci in
// its launch sequence reads buffer ci & 1 and writes the other; index 0 finds v and a.
__device__ __forceinline__ void uw_buffers(const MpsInst& I, int which, double** u, double** w) {
    *u = which ? I.sp_uw : I.u;
    *w = which ? I.sp_uw + 3 * (size_t)I.N : I.v;
}

// Element forces of the step with index ci in its launch sequence.
template <typename T>
__device__ __forceinline__ T* spread_forces(const MpsInst& I, int ci) {
    return reinterpret_cast<T*>(I.sp_f) + (ci & 1 ? 3 * (size_t)I.nen * I.Ne : 0);
}

// Entry E of sp_node: count, Dirichlet bits and record of the node.
__device__ __forceinline__ int entry_count(const int4& E) { return E.z & 63; }
__device__ __forceinline__ bool entry_fixed(const int4& E, int d) { return ((uint32_t)E.z >> (6 + d)) & 1u; }
__device__ __forceinline__ uint32_t entry_record(const int4& E) { return (uint32_t)E.z >> 9; }

// What the update of one node in one direction reads, loaded before any of it is used (the Dirichlet value and the load
// index among it: read when needed they were a third dependent load, in the workgroups of every supported face).  At index
// 0 of a sequence w and m are v and a, and the forces are not used.
template <typename T, int FLIGHT>
struct NodeLoads {
    double X, u, w, m, bc, fg;
    int li;       // index of the node's external force, -1: none
    T c[FLIGHT];  // the first element forces
    __device__ __forceinline__ void load(const MpsInst& I, const int4& E, int d, bool first, const double* __restrict__ ur,
                                         const double* __restrict__ wr, const T* __restrict__ f) {
        const int n = E.x & 0x7FFFFFFF, last = entry_count(E) - 1;
        const size_t i = (size_t)d * I.N + n;
        li = -1;
        fg = 0.0;
        if (I.n_lnode > 0) li = I.lidx[n];  // uniform branches; the others load in every lane, used or not
        if (I.fgrav) {
            const double g = I.fgrav[n];
            fg = d == 2 ? g : 0.0;
        }
        bc = I.bcval[3 * (size_t)entry_record(E) + d];
        X = I.X[i];
        u = ur[i];
        w = wr[i];  // (at index 0 the buffer is v)
        m = *(first ? I.a + i : I.mass + n);
        const T* p = f + 3 * (size_t)E.y + d;
#pragma unroll
        for (int q = 0; q < FLIGHT; q++) c[q] = p[3 * min(q, last)];
    }
    __device__ __forceinline__ double fext(const double* __restrict__ lf, int d) const {
        return li >= 0 ? lf[3 * (size_t)li + d] : fg;
    }
    // Internal force of the node in direction d: its entries added per patch (end bits E.w), then over the patches --
    // the order and the roundings of patch_sums and node_partial_sum.  Without branches: entries past the end add 0.0 to
    // sums that are never -0.0.
    __device__ __forceinline__ double force(const int4& E, const T* __restrict__ f, int d) {
#pragma clang fp contract(off)
        const int count = entry_count(E);
        double fi = 0.0, s = 0.0;
        for (int q0 = 0; q0 < count; q0 += FLIGHT) {
            if (q0 > 0) {
                const T* p = f + 3 * (size_t)E.y + d;
#pragma unroll
                for (int q = 0; q < FLIGHT; q++) c[q] = p[3 * min(q0 + q, count - 1)];
            }
#pragma unroll
            for (int q = 0; q < FLIGHT; q++) {
                s += q0 + q < count ? (double)c[q] : 0.0;
                const bool end = ((uint32_t)E.w >> (q0 + q)) & 1u;  // q0 + q <= 31
                fi += end ? (sizeof(T) == 4 ? (double)(float)s : s) : 0.0;
                s = end ? 0.0 : s;
            }
        }
        return fi;
    }
};

// Min over the 16 lanes of a row, in every lane of it, by DPP rotations (a shuffle goes through LDS and takes several
// times as long).
template <int ROT>
__device__ __forceinline__ unsigned long long row_min_step(unsigned long long v) {
    const int lo = __builtin_amdgcn_update_dpp(0, (int)v, 0x120 + ROT, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), 0x120 + ROT, 0xf, 0xf, false);
    return umin64(v, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ unsigned long long row_min(unsigned long long v) {
    static_assert(MPS_DT_SLOTS == 16, "one slot per lane of a row");
    return row_min_step<1>(row_min_step<2>(row_min_step<4>(row_min_step<8>(v))));
}
__device__ __forceinline__ void spread_reset(const MpsInst& I, int q) {
#pragma unroll
    for (int s = 0; s < MPS_DT_SLOTS; s++) *dt_spread(I, q, s) = 0x7FF0000000000000ull;
}

__device__ __forceinline__ void check_finite(const MpsInst& I, int n, int d, long long k, double u) {
    if (n == I.dof1_node && d == I.dof1_dir && !isfinite(u)) {
        I.ctl->nonfinite = 1;
        atomicMin((unsigned long long*)&I.ctl->nan_step, (unsigned long long)k);
    }
}

// Vertices of the face triangles of hex_char_length: triangle t = (p, q, r), three bits each.
__device__ __forceinline__ int hex_triangle(int t) {
    constexpr int fc[6][4] = {{0, 1, 2, 3}, {4, 5, 6, 7}, {0, 1, 5, 4}, {1, 2, 6, 5}, {2, 3, 7, 6}, {0, 3, 7, 4}};
    unsigned long long lo = 0, hi = 0;
#pragma unroll
    for (int f = 0; f < 6; f++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const unsigned long long c = fc[f][0] | fc[f][1 + h] << 3 | fc[f][2 + h] << 6;
            if (f < 3) lo |= c << (9 * (2 * f + h));
            else hi |= c << (9 * (2 * (f - 3) + h));
        }
    return (int)((t < 6 ? lo >> (9 * t) : hi >> (9 * (t - 6))) & 511u);
}

// The unscaled inverse butterfly of coefficient vectors R for node a alone (hex_unbutterfly, same operations).
template <typename T>
__device__ __forceinline__ void unbutterfly_node(int a, const T* tss, const T* tsd, const T* tds, const T* tdd, T* f) {
#pragma clang fp contract(off)
    const T ys = unit_signed(T(), ((a >> 1) & 1) ^ 1), xs = unit_signed(T(), ((a ^ (a >> 1)) & 1) ^ 1);
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const T us = fma_t(ys, tsd[d], tss[d]), ud = fma_t(ys, tdd[d], tds[d]);
        f[d] = fma_t(xs, ud, us);
    }
}

// n values of T (a multiple of 16 bytes) from LDS in 16-byte pieces.
template <int N, typename T>
__device__ __forceinline__ void lds_read(const T* __restrict__ p, T* v) {
    constexpr int V = 16 / sizeof(T);
    struct alignas(16) Piece { T x[V]; };
    const Piece* q = reinterpret_cast<const Piece*>(p);
#pragma unroll
    for (int i = 0; i < N / V; i++) {
        const Piece t = q[i];
#pragma unroll
        for (int k = 0; k < V; k++) v[i * V + k] = t.x[k];
    }
}

// Forces of a hex8 element by its eight lanes: lane j takes component j of the butterflies (j < 6), Gauss point j, its
// share of the moment sums and node j.  sn: staged node values [9][ss] (X, u, X + u); lx: the element's local node indices.
template <typename T>
__device__ __forceinline__ void hex_coefficients1(const double* __restrict__ s, const uint16_t* __restrict__ lx, T* __restrict__ c) {
#pragma clang fp contract(off)
    {
        double x[8], A[7];
#pragma unroll
        for (int a = 0; a < 8; a++) x[a] = s[lx[a]];
        hex_butterfly1(x, A);
        const double g = MPS_GP;
        c[0] = (T)(0.125 * A[0]);
        c[3] = (T)(0.125 * A[1]);
        c[6] = (T)(0.125 * A[2]);
        c[9] = (T)((0.125 * g) * A[3]);
        c[12] = (T)((0.125 * g) * A[4]);
        c[15] = (T)((0.125 * g) * A[5]);
        c[18] = (T)((0.125 * g * g) * A[6]);
    }
}
template <typename T>
__device__ __forceinline__ void hex_coefficients(const double* __restrict__ sn, int ss, const uint16_t* __restrict__ lx,
                                                 T* __restrict__ sc, int j) {
    if (j < 6) hex_coefficients1<T>(sn + j * ss, lx, sc + (j < 3 ? j : 18 + j));
}

// What the element phase adds to the forces (step modes): bulk viscosity from the displacement increments of the step
// (coefficients sv of the element, qa and qb of visc_coeffs, rdt = 1/dt), or the step's energies (en: W(F), det F and wJ
// of the lane's Gauss point).
enum { kPlain = 0, kVisc = 1, kEnergy = 2 };
template <typename T>
struct StepExtra {
    const T* sv;
    T qa, qb, rdt;
    double en[3];
};
template <typename T, int LAW, int MODE>
__device__ __forceinline__ void hex_spread_force(T* __restrict__ sc, T* __restrict__ sq, int j, double pa, double pb, T* f,
                                                 StepExtra<T>& ex) {
#pragma clang fp contract(off)
    {  // Gauss point j
        T A[44];
        lds_read<44>(sc, A);
        const T(*Ax)[3] = reinterpret_cast<const T(*)[3]>(A);
        const T(*Au)[3] = reinterpret_cast<const T(*)[3]>(A + 21);
        const GpSigns<T> s = gp_signs<T>(j);
        T Jm[9], Du[9], cJ[9], H[9], Fd[3], P[9], Q[3][3], dJ, rJ;
        hex_jac<T>(Ax, s, Jm);
        hex_jac<T>(Au, s, Du);
        hex_grad(Jm, Du, cJ, H, Fd, &dJ, &rJ);
        if constexpr (MODE == kEnergy) {  // weight 1: wJ = |det J|
            double Wg, Jg;
            hex_pk1<LAW>(H, Fd, pa, pb, P, &Wg, &Jg);
            ex.en[0] = Wg;
            ex.en[1] = Jg;
            ex.en[2] = fabs(dJ);
        } else {
            hex_pk1<LAW>(H, Fd, (T)pa, (T)pb, P);
        }
        if constexpr (MODE == kVisc) {
            T tr = T(0);
#pragma unroll
            for (int i = 0; i < 3; i++) {
                T a[7];
#pragma unroll
                for (int m = 0; m < 7; m++) a[m] = ex.sv[m * 3 + i];
                tr += hex_visc_trace(a, s, cJ + 3 * i);
            }
            add_bulk_visc(H, tr * rJ * ex.rdt, ex.qa, ex.qb, P);
        }
        hex_stress_columns<T>(P, cJ, dJ, Q);
#pragma unroll
        for (int k = 0; k < 3; k++)
#pragma unroll
            for (int i = 0; i < 3; i++) sq[i * 24 + j * 3 + k] = Q[k][i];
    }
    wave_sync();
    // Moment sums over the points in order, with the roundings of hex8_element (its products with +-1 are exact, so
    // that its FMAs add and subtract): lanes 0-2 the sums 0, 1, 2, 6 of their component, lanes 3-5 the sums 3, 4, 5.
    if (j < 6) {
        const int i = j < 3 ? j : j - 3;
        T q[24];
        lds_read<24>(sq + 24 * i, q);
        T G[4] = {T(0), T(0), T(0), T(0)};
        if (j < 3) {
#pragma unroll
            for (int gp = 0; gp < 8; gp++) {
                const T x = T(sxi(gp)), y = T(seta(gp)), z = T(szeta(gp));
                G[0] += q[3 * gp];
                G[1] += q[3 * gp + 1];
                G[2] += q[3 * gp + 2];
                G[3] = fma_t(x * y, q[3 * gp + 2], fma_t(x * z, q[3 * gp + 1], fma_t(y * z, q[3 * gp], G[3])));
            }
        } else {
#pragma unroll
            for (int gp = 0; gp < 8; gp++) {
                const T x = T(sxi(gp)), y = T(seta(gp)), z = T(szeta(gp));
                G[0] = fma_t(x, q[3 * gp + 1], fma_t(y, q[3 * gp], G[0]));
                G[1] = fma_t(y, q[3 * gp + 2], fma_t(z, q[3 * gp + 1], G[1]));
                G[2] = fma_t(x, q[3 * gp + 2], fma_t(z, q[3 * gp], G[2]));
            }
        }
        T* g = sc + i + (j < 3 ? 0 : 9);
        g[0] = G[0];
        g[3] = G[1];
        g[6] = G[2];
        if (j < 3) g[18] = G[3];
    }
    wave_sync();
    {  // force at node j: hex_unbutterfly_scaled for one node
        T g[24];
        lds_read<24>(sc, g);
        const T s1 = (T)0.125, s2 = (T)(0.125 * MPS_GP), s3 = (T)(0.125 * MPS_GP * MPS_GP);
        const T zs = unit_signed(T(), (j >> 2) ^ 1);
        T tss[3], tsd[3], tds[3], tdd[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            tss[d] = zs * (g[6 + d] * s1);
            tsd[d] = fma_t(g[3 + d], s1, zs * (g[12 + d] * s2));
            tds[d] = fma_t(g[d], s1, zs * (g[15 + d] * s2));
            tdd[d] = fma_t(g[9 + d], s2, zs * (g[18 + d] * s3));
        }
        unbutterfly_node<T>(j, tss, tsd, tds, tdd, f);
    }
}

// Stable dt of the eight elements of a force wave, by a wave of their own: the 96 face triangles over its lanes, then one
// lane per element.  Returns the element's dt in lanes 0-7.
__device__ __forceinline__ double hex_spread_dt(const double* __restrict__ sn, int ss, const uint16_t* __restrict__ slx,
                                                double* __restrict__ sa, int lane, double c, double l0) {
#pragma clang fp contract(off)
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int it = lane + 64 * r;
        if (it < 96) {
            const int el = it / 12, t = it - 12 * el, code = hex_triangle(t);
            double p[3][3];
#pragma unroll
            for (int v = 0; v < 3; v++) {
                const int a = (code >> (3 * v)) & 7;
#pragma unroll
                for (int d = 0; d < 3; d++) p[v][d] = sn[(6 + d) * ss + slx[el * 8 + a]];
            }
            double n2 = tri_norm2(p[0], p[1], p[2]);
            sqrt_n<1>(&n2);
            sa[it] = 0.5 * n2;
        }
    }
    wave_sync();
    if (lane >= 8) return 0.0;
    double a[12], A = 0.0;
    lds_read<12>(sa + lane * kArea, a);
#pragma unroll
    for (int q = 0; q < 6; q++) {
        const double s = a[2 * q] + a[2 * q + 1];
        A = q == 0 ? fabs(s) : A + fabs(s);
    }
    double x[5][3];
    const int nd[4] = {0, 1, 3, 4};
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
        for (int d = 0; d < 3; d++) x[nd[v]][d] = sn[(6 + d) * ss + slx[lane * 8 + nd[v]]];
    return elem_dt(length_of(hex_corner_volume((const double(*)[3])x), A), l0, c);
}

// Threads of a workgroup: hex8 eight lanes per element for the forces and as many for the stable dt; tet4 a wave for the
// forces, one for the dt and one more for the nodes.
template <int NEN>
constexpr int spread_threads() {
    return NEN == 8 ? 16 * MPS_SPREAD_HEX : 3 * MPS_SPREAD_TET;
}
template <typename T, int NEN>
constexpr size_t fixed_lds() {
    return NEN == 8 ? sizeof(T) * MPS_SPREAD_HEX * (kCol + kCoef + kArea) : 0;
}
// Bytes of dynamic LDS: staged node values (hex8 X, u, X + u; tet4 X, u; with viscosity the increments, with energies the
// velocities), then the element phase's arrays.
template <int NEN, int MODE>
__host__ __device__ size_t stage_lds(int ss) {
    return ((size_t)((NEN == 8 ? 9 : 6) + (MODE != kPlain ? 3 : 0)) * ss * 8 + 15) / 16 * 16;
}
constexpr int kVisc21 = 22, kKin = 26;  // per element: viscosity coefficients; velocity sums and coefficients
template <typename T, int NEN, int MODE>
size_t spread_lds(const MpsInst& I) {
    size_t b = stage_lds<NEN, MODE>(I.sp_stride) + fixed_lds<T, NEN>() + (MODE == kVisc ? sizeof(T) * MPS_SPREAD_HEX * kVisc21 : 0) +
               (MODE == kEnergy && NEN == 8 ? 8 * MPS_SPREAD_HEX * kKin : 0);
    const size_t loads = I.n_lnode > 0 ? 3 * 8 * (size_t)spread_threads<NEN>() : 0;
    return b > loads ? b : loads;
}

// ---------------------------------------------------------------------------
// Energies.  A step's sums are added up while later steps run: the kernel with index ci leaves the energies of each element
// (DEFO_ENERGY and VOLUME of step k, KIN_ENERGY of step k-1) and the node sums of each of its waves (step k-1); a few
// workgroups of the next kernel add the elements of a patch or 256 workgroups' node sums, and one of the kernel after that
// adds those and writes the history.  One workgroup for all of them took as long as the step itself.  The elements are
// added in the patch form's order (block_sum of a patch, reduce_parts of the patches), the node sums in one of their own;
// neither depends on where the launch sequences end.
// ---------------------------------------------------------------------------
constexpr int kRows = 256;
__host__ __device__ __forceinline__ int ep_groups(int nb) { return (nb + kRows - 1) / kRows; }
template <int NEN>
constexpr int ep_width() {  // node sums of a workgroup
    return MPS_NODE_PARTS * (spread_threads<NEN>() / 64);
}
// Sets 0 and 1 by the parity of the kernel's index; set 2 of the node sums: the end of a sequence (its last step).
template <int NEN>
__device__ __forceinline__ double* ep_rows(const MpsInst& I, int set) {
    return I.sp_ep + (size_t)set * I.sp_nb * ep_width<NEN>();
}
template <int NEN>
__device__ __forceinline__ double* ep_sums(const MpsInst& I, int set) {  // of the groups
    return ep_rows<NEN>(I, 3) + (size_t)set * ep_groups(I.sp_nb) * MPS_NODE_PARTS;
}
template <int NEN>
__device__ __forceinline__ double* ep_patches(const MpsInst& I, int set) {  // element sums of the patches
    return ep_sums<NEN>(I, 3) + (size_t)set * 3 * I.n_patch;
}
template <int NEN>
__device__ __forceinline__ double* ep_elems(const MpsInst& I, int set) {  // [3][Ne]
    return ep_patches<NEN>(I, 2) + (size_t)set * 3 * I.Ne;
}

// Sum over the lanes of a wave of NV values, in every lane.
template <int NV>
__device__ __forceinline__ void wave_sum(double* v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int j = 0; j < NV; j++) v[j] += __shfl_xor(v[j], off, 64);
}
// block_sum of 256 work-items by a workgroup of fewer waves: get(i, v) gives the values of work-item i.
template <int NV, typename F>
__device__ __forceinline__ void sum256(F get, double* out, double* sh) {
    const int lane = threadIdx.x & 63;
    __syncthreads();  // an earlier call may still be reading sh
    for (int w = threadIdx.x >> 6; w < 4; w += blockDim.x >> 6) {
        double v[NV];
        get(w * 64 + lane, v);
        wave_sum<NV>(v);
        if (lane == 0)
#pragma unroll
            for (int j = 0; j < NV; j++) sh[w * NV + j] = v[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NV; j++) out[j] = ((sh[j] + sh[NV + j]) + sh[2 * NV + j]) + sh[3 * NV + j];
}
// The nb entries of NV values at part: work-item i takes i, i + 256, ... (reduce_parts of a workgroup of 256).
template <int NV>
__device__ __forceinline__ void sum_parts(const double* __restrict__ part, int nb, double* out, double* sh) {
    sum256<NV>([&](int i, double* v) {
#pragma unroll
        for (int j = 0; j < NV; j++) v[j] = 0.0;
        for (int b = i; b < nb; b += 256)
#pragma unroll
            for (int j = 0; j < NV; j++) v[j] += part[(size_t)b * NV + j];
    }, out, sh);
}
// Element sums of entry x (the patch that workgroup x of the patch form computes), and node sums of group x, of a set, by
// the calling workgroup.
template <int NEN>
__device__ __forceinline__ void ep_add_patch(const MpsInst& I, int set, int x, double* sh) {
    const double* ee = ep_elems<NEN>(I, set);
    const int p = xcd_tile(x, I.n_patch);
    double t[3];
    sum256<3>([&](int i, double* v) {
        const int e = p * MPS_PATCH + i;
#pragma unroll
        for (int j = 0; j < 3; j++) v[j] = e < I.Ne ? ee[(size_t)j * I.Ne + e] : 0.0;
    }, t, sh);
    if (threadIdx.x == 0)
#pragma unroll
        for (int j = 0; j < 3; j++) ep_patches<NEN>(I, set)[3 * x + j] = t[j];
}
template <int NEN>
__device__ __forceinline__ void ep_add_group(const MpsInst& I, int set, int x, double* sh) {
    constexpr int NW = spread_threads<NEN>() / 64;
    const double* rows = ep_rows<NEN>(I, set);
    double t[MPS_NODE_PARTS];
    sum256<MPS_NODE_PARTS>([&](int i, double* v) {
        const int b = x * kRows + i;
#pragma unroll
        for (int j = 0; j < MPS_NODE_PARTS; j++) {
            v[j] = 0.0;
#pragma unroll
            for (int w = 0; w < NW; w++) v[j] += b < I.sp_nb ? rows[(size_t)b * ep_width<NEN>() + w * MPS_NODE_PARTS + j] : 0.0;
        }
    }, t, sh);
    if (threadIdx.x == 0)
#pragma unroll
        for (int j = 0; j < MPS_NODE_PARTS; j++) ep_sums<NEN>(I, set)[x * MPS_NODE_PARTS + j] = t[j];
}
// Node sums t of step j into the running works and the history (by one work-item).
__device__ __forceinline__ void node_history(const MpsInst& I, long long j, const double* t) {
    MpsCtl* ctl = I.ctl;
    ctl->w_ext += t[0];
    ctl->w_react += t[1];
    *hist_at(I, MPS_H_WEXT, j) = ctl->w_ext;
    *hist_at(I, MPS_H_WREACT, j) = ctl->w_react;
    if (j % I.energy_every == 0) {
        *hist_at(I, MPS_H_EKL, j) = t[2];
        *hist_at(I, MPS_H_EEXT, j) = t[3];
    }
    ctl->wred = j;
}
// Sums of the kernel with index s of the sequence that starts at step A into the history, by the calling workgroup.
template <int NEN>
__device__ __forceinline__ void spread_history(const MpsInst& I, long long A, int s, double* sh) {
    double el[3], nd[MPS_NODE_PARTS];
    sum_parts<3>(ep_patches<NEN>(I, s & 1), I.n_patch, el, sh);
    sum_parts<MPS_NODE_PARTS>(ep_sums<NEN>(I, s & 1), ep_groups(I.sp_nb), nd, sh);
    if (threadIdx.x != 0 || I.hist_cap <= 0) return;
    const long long k = A + s;
    if (k % I.energy_every == 0) {
        *hist_at(I, MPS_H_EDEF, k) = el[0];
        *hist_at(I, MPS_H_VOL, k) = el[1];
    }
    if (s == 0) return;
    if ((k - 1) % I.energy_every == 0) *hist_at(I, MPS_H_EKIN, k - 1) = el[2];
    node_history(I, k - 1, nd);
}
// Energy terms of DOF d of a node (entry E, load index li) at step k, by the node's owner (node_energy_forces and node_energy_motion for one
// direction): u the step's displacement, incr its increment, fi and fe the forces, m, v and wkin as the update leaves them.
__device__ __forceinline__ void dof_energy(const MpsInst& I, const int4& E, int li, int d, long long k, double u, double incr,
                                           double fi, double fe, double m, double v, double wkin, double* red) {
    double fp = fe;
    if (li >= 0) {
        double* lp = I.lfprev + 3 * (size_t)li + d;
        fp = *lp;
        *lp = fe;
    }
    double wr = wkin;
    if (entry_fixed(E, d)) {
        double* rp = I.rprev + 3 * (size_t)entry_record(E) + d;
        const double r = fi - fe;
        wr += 0.5 * (*rp + r) * incr;
        *rp = r;
    }
    if (k >= 2) {
        red[0] += 0.5 * (fp + fe) * incr;
        red[1] += wr;
    }
    red[2] += 0.5 * m * v * v;
    red[3] += u * fe;
}

// External force of the step with index ci (its flagged nodes, two sets by parity).
__device__ __forceinline__ double* spread_lf(const MpsInst& I, int ci) {
    return I.lf + (ci & 1 ? 3 * (size_t)I.n_lnode : 0);
}

// The workgroups of a step kernel before its element workgroups: with energies the patches, the groups and the history,
// then the external forces of the step.
template <int NEN, int MODE>
__device__ __forceinline__ void spread_side(const MpsInst& I, int ci, int x, long long A, double time, double* sh) {
    if constexpr (MODE == kEnergy) {
        const int G = ep_groups(I.sp_nb), P = I.n_patch;
        if (x <= P + G) {
            if (x < P + G && ci >= 1) {
                if (x < P) ep_add_patch<NEN>(I, (ci - 1) & 1, x, sh);
                else ep_add_group<NEN>(I, (ci - 1) & 1, x - P, sh);
            } else if (x == P + G && ci >= 2) {
                spread_history<NEN>(I, A, ci - 2, sh);
            }
            return;
        }
        x -= P + G + 1;
    }
    loads_block<false>(I, x, time, sh, spread_lf(I, ci));
}
template <int NEN, int MODE>
unsigned side_blocks(const MpsInst& I) {
    constexpr int per = spread_threads<NEN>() / 32;
    return (MODE == kEnergy ? (unsigned)(I.n_patch + ep_groups(I.sp_nb)) + 1 : 0u) + (unsigned)((I.n_lnode + per - 1) / per);
}

}  // namespace

// Step control of the kernel with index ci, the same in every workgroup: requested by load (the lane's dt slot with it),
// evaluated by begin.
struct StepControl {
    long long A, k;
    MpsStepSlot prev, nx;
    unsigned long long m16;
    __device__ __forceinline__ void load(const MpsInst& I, int ci) {
        const MpsCtl* ctl = I.ctl;
        A = ctl->A;
        k = A + ci;
        const MpsStepSlot* pp = ci == 0 ? ctl->slot + ((A - 1) & 1) : ctl->sslot + ((ci - 1) & 1);
        prev.time = pp->time;
        prev.dt = pp->dt;
        prev.go = pp->go;
        const int row = threadIdx.x & (MPS_DT_SLOTS - 1);
        m16 = *(ci == 0 ? dt_slot(I, dt_parity(A), row) : dt_spread(I, ci % 3, row));
    }
    __device__ __forceinline__ int begin(const MpsInst& I) { return begin_scalars(I, k, prev, row_min(m16), &nx); }
};

// Step k = A + ci, ci its index in the launch sequence: solve of step k-1 (ci > 0), begin of step k, its element forces
// and the stable dt for step k+1 (the file's head).  eflags (energies): MPS_E_KIN.
template <typename T, int NEN, int LAW, int MODE>
__global__ __launch_bounds__(spread_threads<NEN>()) __attribute__((amdgpu_waves_per_eu(NEN == 8 ? 4 : MODE == kPlain && sizeof(T) == 4 ? 4 : 3))) void k_spread(MpsInst I, int ci, unsigned eflags) {
    extern __shared__ __align__(16) double smem[];
    constexpr int EB = NEN == 8 ? MPS_SPREAD_HEX : MPS_SPREAD_TET;  // elements of a workgroup
    __shared__ uint16_t slx[NEN == 8 ? EB * 8 : 1];
    constexpr int NT = spread_threads<NEN>(), FLIGHT = NEN == 8 ? 8 : 16;
    const int nside = (int)gridDim.x - I.sp_nb, bx = (int)blockIdx.x - nside;  // workgroups of spread_side come first
    if (bx < 0) {
        StepControl c;
        c.load(I, ci);
        (void)c.begin(I);
        if (c.nx.go) spread_side<NEN, MODE>(I, ci, (int)blockIdx.x, c.A, c.nx.time, smem);
        return;
    }
    const int b = xcd_tile(bx, I.sp_nb), t = threadIdx.x, ss = I.sp_stride;
    // tables first: their addresses depend on nothing.  Work item it: direction it % 3 of the workgroup's node it / 3.
    const int4* tab = I.sp_node + (size_t)b * ss;
    int4 E = make_int4(-1, 0, 0, 0);
    if (t < 3 * ss) E = tab[t / 3];
    // role in the element phase: wave of forces or of stable dt
    const bool force = t < 64;
    const int lane = t & 63, j = t & 7;
    const int el = NEN == 8 ? (force ? lane >> 3 : j) : lane;  // a dt wave's lanes 0-7: its elements
    const int e = b * EB + el;
    const bool mine = e < I.Ne && (NEN == 8 || t < 128);
    const int ec = min(e, I.Ne - 1);
    int pos[NEN == 8 ? 1 : 4];
    uint2 l4 = make_uint2(0u, 0u);
    if constexpr (NEN == 8) {
        pos[0] = I.sp_pos[(size_t)ec * 8 + j];
        if (force) slx[t] = I.sp_lx[(size_t)ec * 8 + j];
    } else {
        const int4 q = *reinterpret_cast<const int4*>(I.sp_pos + (size_t)ec * 4);
        pos[0] = q.x;
        pos[1] = q.y;
        pos[2] = q.z;
        pos[3] = q.w;
        l4 = *reinterpret_cast<const uint2*>(I.sp_lx + (size_t)ec * 4);
    }
    const TetConsts kc = tet_consts(I, ec, true);
    StepControl sc0;  // read now, used once the nodes' loads are on their way
    sc0.load(I, ci);
    const long long k = sc0.k;
    MpsCtl* ctl = I.ctl;
    const MpsStepSlot prev = sc0.prev;
    const size_t N = (size_t)I.N;
    double *ur, *wr, *uo, *wo;
    uw_buffers(I, ci & 1, &ur, &wr);
    uw_buffers(I, (ci & 1) ^ 1, &uo, &wo);
    const T* fr = spread_forces<T>(I, ci + 1);  // step k-1
    NodeLoads<T, FLIGHT> L;
    if (E.x != -1) L.load(I, E, t - 3 * (t / 3), ci == 0, ur, wr, fr);
    const int st = sc0.begin(I);
    const MpsStepSlot nx = sc0.nx;
    if (bx == 0 && t == 0) {
        ctl->sslot[ci & 1] = nx;
        if (st != MPSD_RUNNING) ctl->status = st;
        if (nx.go) {
            ctl->B = k;
            if (I.hist_cap > 0) {
                const size_t idx = (size_t)((k - 1) % I.hist_cap);
                I.hist[idx] = nx.time;
                I.hist[(size_t)I.hist_cap + idx] = nx.dt;
            }
        }
        spread_reset(I, (ci + 2) % 3);
    }
    if (!nx.go) return;
    const double* lf = spread_lf(I, ci + 1);  // step k-1
    double red[MPS_NODE_PARTS] = {0.0, 0.0, 0.0, 0.0};
    double* se = smem + (NEN == 8 ? 9 : 6) * ss;  // staged increments or velocities: se[d*ss + q]
    for (int it = t; it < 3 * ss; it += NT) {
        const int q = it / 3, d = it - 3 * q;
        if (it != t) {
            E = tab[q];
            if (E.x != -1) L.load(I, E, d, ci == 0, ur, wr, fr);
        }
        if (E.x == -1) break;  // the rest is padding
        const int n = E.x & 0x7FFFFFFF;
        const bool fixed = entry_fixed(E, d);
        double u = L.u, w;
        if (ci == 0) {
            w = half_velocity(nx.dt, L.w, L.m);
        } else {
            double v, acc, wkin = 0.0;
            const double fi = L.force(E, fr, d), fe = L.fext(lf, d);
            dof_update(I, fixed, L.bc, k - 1, prev.dt, L.m, -fi + fe, L.w, &v, &acc, MODE == kEnergy ? &wkin : nullptr);
            if (E.x < 0) check_finite(I, n, d, k - 1, u);
            if constexpr (MODE == kEnergy) {
                se[d * ss + q] = v;
                if (E.x < 0)
                    dof_energy(I, E, L.li, d, k - 1, u, dof_increment(I, fixed, L.bc, k - 1, prev.dt, L.w), fi, fe, L.m, v, wkin,
                               red);
            }
            w = half_velocity(nx.dt, v, acc);
        }
        u += dof_increment(I, fixed, L.bc, k, nx.dt, w);
        if constexpr (MODE == kVisc) se[d * ss + q] = u - L.u;
        if (E.x < 0) {
            uo[d * N + n] = u;
            wo[d * N + n] = w;
        }
        if constexpr (NEN == 8) {
            smem[d * ss + q] = L.X;
            smem[(3 + d) * ss + q] = u;
            smem[(6 + d) * ss + q] = L.X + u;
        } else {
            smem[6 * q + d] = L.X;
            smem[6 * q + 3 + d] = u;
        }
    }
    __syncthreads();
    StepExtra<T> ex;
    double* sums = ep_rows<NEN>(I, ci & 1) + (size_t)b * ep_width<NEN>();
    const auto node_row = [&]() {  // the wave's node sums of step k-1
        wave_sum<MPS_NODE_PARTS>(red);
        if (lane == 0)
#pragma unroll
            for (int j = 0; j < MPS_NODE_PARTS; j++) sums[(t >> 6) * MPS_NODE_PARTS + j] = red[j];
    };
    double* ee = ep_elems<NEN>(I, ci & 1);  // the elements' energies
    T* fo = spread_forces<T>(I, ci);
    unsigned long long dmin = 0x7FF0000000000000ull;
    if constexpr (NEN == 8) {
        T* base = reinterpret_cast<T*>(reinterpret_cast<char*>(smem) + stage_lds<8, MODE>(ss));
        T* sc = base + EB * kCol;  // the elements' coefficients
        if (force) hex_coefficients<T>(smem, ss, slx + el * 8, sc + el * kCoef, j);
        double* sk = reinterpret_cast<double*>(reinterpret_cast<char*>(base) + fixed_lds<T, 8>());
        if constexpr (MODE == kEnergy) {  // sums and coefficients of the nodal velocities (hex_kinetic)
            if ((eflags & MPS_E_KIN) && force && j < 3) {
                double x[8], A[7], sum = 0.0;
#pragma unroll
                for (int a = 0; a < 8; a++) {
                    x[a] = se[j * ss + slx[el * 8 + a]];
                    sum += x[a];
                }
                hex_butterfly1(x, A);
                double* c = sk + el * kKin + j;
                c[0] = sum;
#pragma unroll
                for (int m = 0; m < 7; m++) c[3 * (m + 1)] = A[m];
            }
        }
        if constexpr (MODE == kVisc) {
            T* sv = reinterpret_cast<T*>(reinterpret_cast<char*>(base) + fixed_lds<T, 8>()) + el * kVisc21;
            if (force && j < 3) hex_coefficients1<T>(se + j * ss, slx + el * 8, sv + j);
            double da, db;
            visc_coeffs(I, ec, kc.c, &da, &db);
            ex.sv = sv;
            ex.qa = (T)da;
            ex.qb = (T)db;
            ex.rdt = (T)(nx.dt == 0.0 ? 0.0 : 1 / nx.dt);
        }
        wave_sync();
        if (force) {
            T f[3];
            hex_spread_force<T, LAW, MODE>(sc + el * kCoef, base + el * kCol, j, kc.pa, kc.pb, f, ex);
            if (mine) {
                T* dst = fo + 3 * (size_t)pos[0];
#pragma unroll
                for (int i = 0; i < 3; i++) dst[i] = f[i];
            }
            if constexpr (MODE == kEnergy) {
                // the points' values to LDS (over the columns), where three lanes of an element add them in order
                double* sp = reinterpret_cast<double*>(base + el * kCol);
                double kv = 0.0;
                if (eflags & MPS_E_KIN) {
                    const double* c = sk + el * kKin;
                    double vc[24];
                    lds_read<24>(c, vc);
                    kv = hex_point_kinetic(vc, reinterpret_cast<const double(*)[3]>(vc + 3), gp_signs<double>(j),
                                           I.rho ? I.rho[ec] : I.rho0);
                }
                sp[j * 4] = ex.en[0];
                sp[j * 4 + 1] = ex.en[1];
                sp[j * 4 + 2] = kv;
                sp[j * 4 + 3] = ex.en[2];
                wave_sync();
                if (j < 3 && mine) {
                    double sum = 0.0;
#pragma unroll
                    for (int gp = 0; gp < 8; gp++) sum = fma(sp[gp * 4 + j], sp[gp * 4 + 3], sum);
                    ee[(size_t)j * I.Ne + e] = sum;
                }
                node_row();
            }
            return;
        }
        const double dte = hex_spread_dt(smem, ss, slx, base + EB * (kCol + kCoef), lane, kc.c, kc.l0);
        if (lane < 8 && mine) dmin = d2bits(dte);
    } else {
        if (t >= 128) {
            if constexpr (MODE == kEnergy) node_row();
            return;
        }
        const int l[4] = {(int)(l4.x & 0xffffu), (int)(l4.x >> 16), (int)(l4.y & 0xffffu), (int)(l4.y >> 16)};
        double x[4][3], uu[4][3];
#pragma unroll
        for (int a = 0; a < 4; a++) staged_node(smem, l[a], x[a], uu[a]);
        if (force) {
            T f[4][3];
            double r[4];
            tet4_core<T, LAW, false, MODE == kEnergy && sizeof(T) == 8>(I, e, nullptr, x, uu, kc, f, false, 0.0, r);
            if constexpr (MODE == kEnergy && sizeof(T) == 4) {  // the energies in FP64
                double f64[4][3];
                tet4_core<double, LAW, false, true>(I, e, nullptr, x, uu, kc, f64, false, 0.0, r);
            }
            if (mine) {
#pragma unroll
                for (int a = 0; a < 4; a++) {
                    T* dst = fo + 3 * (size_t)pos[a];
#pragma unroll
                    for (int i = 0; i < 3; i++) dst[i] = f[a][i];
                }
            }
            if constexpr (MODE == kEnergy) {
                if (mine) {
                    ee[e] = r[0];
                    ee[(size_t)I.Ne + e] = r[1];
                    if (eflags & MPS_E_KIN) {
                        double v[4][3];
#pragma unroll
                        for (int a = 0; a < 4; a++)
#pragma unroll
                            for (int d = 0; d < 3; d++) v[a][d] = se[d * ss + l[a]];
                        ee[2 * (size_t)I.Ne + e] = tet_point_kinetic(v, I.rho ? I.rho[e] : I.rho0, r[3]);
                    }
                }
                node_row();
            }
            return;
        }
        const double dte = tet_dt<T>(x, uu, kc);
        if (mine) dmin = d2bits(dte);
    }
    // one atomic per workgroup; all lanes of its dt wave are here
#pragma unroll
    for (int off = NEN == 8 ? 4 : 32; off > 0; off >>= 1) dmin = umin64(dmin, (unsigned long long)__shfl_xor((long long)dmin, off, 64));
    if (lane == 0) atomicMin(dt_spread(I, (ci + 1) % 3, b & (MPS_DT_SLOTS - 1)), dmin);
    if constexpr (MODE == kEnergy) node_row();
}

// After a launch sequence: solve of its last step (B), from the buffer that step wrote, into u, v and a.
template <typename T, int NEN, int MODE>
__global__ __launch_bounds__(spread_threads<NEN>()) void k_spread_end(MpsInst I) {
    constexpr int NT = spread_threads<NEN>();
    const MpsCtl* ctl = I.ctl;
    const long long A = ctl->A, k = ctl->B;
    if (k < A) return;  // no step was begun
    const int ss = I.sp_stride;
    const double dt = ctl->sslot[(k - A) & 1].dt;
    const size_t N = (size_t)I.N;
    double *ur, *wr;
    uw_buffers(I, (int)((k - A) & 1) ^ 1, &ur, &wr);
    const T* fr = spread_forces<T>(I, (int)(k - A));
    const double* lf = spread_lf(I, (int)(k - A));
    double red[MPS_NODE_PARTS] = {0.0, 0.0, 0.0, 0.0};
    const int b = xcd_tile(blockIdx.x, gridDim.x);
    for (int it = threadIdx.x; it < 3 * ss; it += NT) {
        const int q = it / 3, d = it - 3 * q;
        const int4 E = I.sp_node[(size_t)b * ss + q];
        if (E.x == -1) break;
        if (E.x >= 0) continue;  // another workgroup owns the node
        const int n = E.x & 0x7FFFFFFF;
        const size_t i = d * N + n;
        NodeLoads<T, 8> L;
        L.load(I, E, d, false, ur, wr, fr);
        double v, a, wkin = 0.0;
        const double u = L.u, fi = L.force(E, fr, d), fe = L.fext(lf, d);
        const bool fixed = entry_fixed(E, d);
        dof_update(I, fixed, L.bc, k, dt, L.m, -fi + fe, L.w, &v, &a, MODE == kEnergy ? &wkin : nullptr);
        check_finite(I, n, d, k, u);
        if constexpr (MODE == kEnergy)
            dof_energy(I, E, L.li, d, k, u, dof_increment(I, fixed, L.bc, k, dt, L.w), fi, fe, L.m, v, wkin, red);
        I.u[i] = u;
        I.v[i] = v;
        I.a[i] = a;
    }
    if constexpr (MODE == kEnergy) {
        wave_sum<MPS_NODE_PARTS>(red);
        double* sums = ep_rows<NEN>(I, 2) + (size_t)b * ep_width<NEN>();
        if ((threadIdx.x & 63) == 0)
#pragma unroll
            for (int j = 0; j < MPS_NODE_PARTS; j++) sums[(threadIdx.x >> 6) * MPS_NODE_PARTS + j] = red[j];
    }
}

// Sums that no step kernel has added up yet: the patches and groups of the last step kernel, the groups of the end.
template <int NEN>
__global__ __launch_bounds__(spread_threads<NEN>()) void k_spread_groups(MpsInst I) {
    __shared__ double sh[MPS_NODE_PARTS * 4];
    const long long A = I.ctl->A, k = I.ctl->B;
    if (k < A) return;
    const int G = ep_groups(I.sp_nb), P = I.n_patch, x = blockIdx.x, set = (int)(k - A) & 1;
    if (x < P) ep_add_patch<NEN>(I, set, x, sh);
    else if (x < P + G) ep_add_group<NEN>(I, set, x - P, sh);
    else ep_add_group<NEN>(I, 2, x - P - G, sh);
}

// Closes a launch sequence: its steps count as done, and the scalars and the pending min go where the patch form and the
// next sequence find them.  Energies: KIN_ENERGY of the last step is left to the standalone pass.
template <int NEN, int MODE>
__global__ __launch_bounds__(MODE == kEnergy ? spread_threads<NEN>() : 64) void k_spread_close(MpsInst I) {
    MpsCtl* ctl = I.ctl;
    const long long A = ctl->A, k = ctl->B;
    if (k < A) return;
    const int ci = (int)(k - A);
    if constexpr (MODE == kEnergy) {  // the sums that no step kernel has added up yet, in order
        __shared__ double sh[MPS_NODE_PARTS * 4];
        if (ci >= 1) spread_history<NEN>(I, A, ci - 1, sh);
        spread_history<NEN>(I, A, ci, sh);
        double t[MPS_NODE_PARTS];
        sum_parts<MPS_NODE_PARTS>(ep_sums<NEN>(I, 2), ep_groups(I.sp_nb), t, sh);
        if (threadIdx.x == 0 && I.hist_cap > 0) node_history(I, k, t);
        __syncthreads();  // every thread has read the control block
    }
    const unsigned long long mb = row_min(*dt_spread(I, (ci + 1) % 3, threadIdx.x & (MPS_DT_SLOTS - 1)));
    if (threadIdx.x != 0) return;
    MpsStepSlot s = ctl->sslot[ci & 1];
    s.go = 1;
    ctl->slot[k & 1] = s;
    dt_reset(I, 0);
    dt_reset(I, 1);
    *dt_slot(I, dt_parity(k + 1), 0) = mb;
    for (int q = 0; q < 3; q++) spread_reset(I, q);
    ctl->spread_last = ci & 1;
    ctl->A = k + 1;
}

// Internal force at DOF idx[i] = node + N*dir of the last step, from its element forces.
template <typename T>
__global__ void k_spread_pick(MpsInst I, const int32_t* __restrict__ idx, int64_t n, double* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 E = I.sp_node[I.sp_own[idx[i] % I.N]];
    const int d = idx[i] / I.N;
    const T* f = spread_forces<T>(I, I.ctl->spread_last);
    NodeLoads<T, 8> L;
#pragma unroll
    for (int q = 0; q < 8; q++) L.c[q] = f[3 * ((size_t)E.y + min(q, entry_count(E) - 1)) + d];
    out[i] = L.force(E, f, d);
}

namespace mpsk {

static int spread_mode(const MpsInst& I) { return I.energy_every > 0 ? kEnergy : I.uprev != nullptr ? kVisc : kPlain; }

size_t spread_energy_doubles(const MpsInst& I) {
    const size_t nb = (size_t)I.sp_nb, w = (size_t)(I.nen == 8 ? ep_width<8>() : ep_width<4>());
    return 3 * (nb * w + (size_t)ep_groups(I.sp_nb) * MPS_NODE_PARTS) + 2 * 3 * ((size_t)I.n_patch + (size_t)I.Ne);
}

hipError_t launch_spread(const MpsInst& I, int ci, unsigned eflags, hipStream_t st) {
    const unsigned nb = (unsigned)I.sp_nb;
#define MPS_SPREAD(T, NEN, LAW, M) \
    k_spread<T, NEN, LAW, M><<<nb + side_blocks<NEN, M>(I), spread_threads<NEN>(), spread_lds<T, NEN, M>(I), st>>>(I, ci, eflags)
#define MPS_SPREAD_LAW(T, NEN, M)                       \
    switch (I.law) {                                    \
        case 0: MPS_SPREAD(T, NEN, 0, M); break;        \
        case 1: MPS_SPREAD(T, NEN, 1, M); break;        \
        case 2: MPS_SPREAD(T, NEN, 2, M); break;        \
        default: MPS_SPREAD(T, NEN, 3, M); break;       \
    }
    const int mode = spread_mode(I);
    const bool f32 = I.precision == 1;
    if (I.nen == 8) {
        if (mode == kVisc) { MPS_SPREAD_LAW(double, 8, kVisc) }
        else if (mode == kEnergy) { MPS_SPREAD_LAW(double, 8, kEnergy) }
        else { MPS_SPREAD_LAW(double, 8, kPlain) }
    } else if (mode == kEnergy) {
        if (f32) { MPS_SPREAD_LAW(float, 4, kEnergy) } else { MPS_SPREAD_LAW(double, 4, kEnergy) }
    } else {
        if (f32) { MPS_SPREAD_LAW(float, 4, kPlain) } else { MPS_SPREAD_LAW(double, 4, kPlain) }
    }
#undef MPS_SPREAD_LAW
#undef MPS_SPREAD
    return hipGetLastError();
}

hipError_t launch_spread_end(const MpsInst& I, hipStream_t st) {
    const unsigned nb = (unsigned)I.sp_nb;
    const bool en = spread_mode(I) == kEnergy;
#define MPS_SPREAD_END(T, NEN, M) k_spread_end<T, NEN, M><<<nb, spread_threads<NEN>(), 0, st>>>(I)
#define MPS_SPREAD_END_T(NEN, M)                         \
    if (I.precision == 1) MPS_SPREAD_END(float, NEN, M); \
    else MPS_SPREAD_END(double, NEN, M)
    if (I.nen == 8) {
        if (en) MPS_SPREAD_END(double, 8, kEnergy);
        else MPS_SPREAD_END(double, 8, kPlain);
    } else {
        if (en) { MPS_SPREAD_END_T(4, kEnergy); } else { MPS_SPREAD_END_T(4, kPlain); }
    }
#undef MPS_SPREAD_END_T
#undef MPS_SPREAD_END
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const unsigned groups = (unsigned)I.n_patch + 2 * (unsigned)ep_groups(I.sp_nb);
    if (!en) {
        k_spread_close<8, kPlain><<<1, 64, 0, st>>>(I);
    } else if (I.nen == 8) {
        k_spread_groups<8><<<groups, spread_threads<8>(), 0, st>>>(I);
        k_spread_close<8, kEnergy><<<1, spread_threads<8>(), 0, st>>>(I);
    } else {
        k_spread_groups<4><<<groups, spread_threads<4>(), 0, st>>>(I);
        k_spread_close<4, kEnergy><<<1, spread_threads<4>(), 0, st>>>(I);
    }
    return hipGetLastError();
}

hipError_t launch_spread_pick(const MpsInst& I, const int32_t* idx, int64_t n, double* out, hipStream_t st) {
    const unsigned nb = (unsigned)((n + 255) / 256);
    if (I.precision == 1) k_spread_pick<float><<<nb, 256, 0, st>>>(I, idx, n, out);
    else k_spread_pick<double><<<nb, 256, 0, st>>>(I, idx, n, out);
    return hipGetLastError();
}

}  // namespace mpsk
