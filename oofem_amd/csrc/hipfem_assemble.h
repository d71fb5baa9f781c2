// Stiffness assembly by rows, each written once, in ascending element order:
// for LSpace and LTRSpace the wave that writes a node's rows forms the blocks
// B_a^T D B_b of its elements on the spot, for QSpace it sums stored element
// matrices.
// Included by hipfem_model.hip (after the element rules).
#pragma once

namespace hipfem {

// a double from another lane of the quad
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

constexpr int ASM_LMAX = 512;   // longest row (columns) of the row form: up to 8 KiB of column codes per wave

typedef double d2_t __attribute__((ext_vector_type(2)));

// what the row kernels read of the mesh and the Gauss-point state
struct AsmArgs {
    int nnode, nelem;
    const int *nptr, *nadj;      // node -> element * NEN + local node, ascending element
    const int *conn, *eqn, *emat;
    const double *coords, *mat;
    const uint16_t *eoff;
    const double *state;
    int ngp_total;
    const int8_t *sflag;         // SUR kernels: 1 where the point's tangent is the surrogate's (dsur)
    const float *dsur;
    const int32_t *rowptr;
    double *val;
    int *bad;
};

// Tangent of a point in the form the blocks need,
// dV B_a^T D B_b = cd ((g_a.g_b) I + g_b g_a^T) + kd g_a g_b^T - (M g_a)(M g_b)^T
// with cd = dV c / 2, kd = dV (K - c / 3) and M = sqrt(dV) times the tensor of
// m, from D = c I_dev + K 1x1 - m m^T (mises_tangent_parts)
struct PointState {
    double s[6], kn, kt;   // trial deviator, committed and temp kappa
};

__device__ __forceinline__ PointState load_point(const double *__restrict__ state, size_t ngp_total, size_t gp)
{
    PointState p;
#pragma unroll
    for (int i = 0; i < 6; i++) p.s[i] = state[(14 + i) * ngp_total + gp];
    p.kn = state[6 * ngp_total + gp];
    p.kt = state[13 * ngp_total + gp];
    return p;
}

__device__ __forceinline__ void point_parts(const double *mp, double dV, const PointState &ps, double &cd, double &kd,
                                            double m[6])
{
    const double E = mp[1], nu = mp[2];
    const double G = E / (2.0 * (1. + nu));
    const double K = E / (3.0 * (1. - 2. * nu));
    double c = 2. * G;
#pragma unroll
    for (int i = 0; i < 6; i++) m[i] = 0.0;
    if ((int)mp[0] == HIPFEM_MAT_MISES) {
        const double *s = ps.s, kn = ps.kn, dk = ps.kt - kn;
        if (dk > 0.0) {
            const double t2 = s[0] * s[0] + s[1] * s[1] + s[2] * s[2] + 2. * s[3] * s[3] + 2. * s[4] * s[4] +
                              2. * s[5] * s[5];
            // factor = -2 sqrt(6) G^2 / |s|, factor1 = factor sigma_Y / ((H + 3G) |s|^2) (misesmat.C:530-540)
            const double factor = 2. * sqrt(6.) * G * G / sqrt(t2);
            c -= factor * dk;
            const double sc = sqrt(factor * (mp[3] + mp[4] * kn) / ((mp[4] + 3. * G) * t2) * dV);
#pragma unroll
            for (int i = 0; i < 6; i++) m[i] = sc * s[i];
        }
    }
    cd = 0.5 * c * dV;
    kd = (K - c / 3.0) * dV;
}

// (M g) with M the symmetric tensor of the Voigt m
__device__ __forceinline__ void tensor_times(const double m[6], const double g[3], double v[3])
{
    v[0] = m[0] * g[0] + m[5] * g[1] + m[4] * g[2];
    v[1] = m[5] * g[0] + m[1] * g[1] + m[3] * g[2];
    v[2] = m[4] * g[0] + m[3] * g[1] + m[2] * g[2];
}

// block += cd ((n.m) I + m n^T) + kd n m^T - va vb^T (n = g_a, m = g_b).  The
// products n_i m_j are shared by the entries (i, j) and (j, i), and the block
// (b, a) of another wave gets the same bits transposed (the gradient of a node
// is the same expression as row and as column): a tangent without surrogate
// points is exactly symmetric.  Each point's contribution is formed apart and added once: with
// its terms chained into the block by FMAs, the roundings of the larger
// partial sums leave a rigid translation five times as far from force-free
// (displacements of the 10x10x40 cantilever 5e-12 off instead of 5e-13).
__device__ __forceinline__ void add_parts(const double n[3], const double m[3], double cd, double kd,
                                          const double va[3], const double vb[3], double K[9])
{
    double P[9];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) P[3 * i + j] = n[i] * m[j];
    const double nm = P[0] + P[4] + P[8];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            K[3 * i + j] +=
                fma(-va[i], vb[j], fma(kd, P[3 * i + j], cd * (i == j ? P[4 * i] + nm : P[3 * j + i])));
}

// block += dV (lambda n m^T + G (m n^T + (n.m) I)), the isotropic elastic D.
// ln lm = lambda: lambda goes to the gradient of the lower local node and 1 to
// the other, so that the blocks (a, b) and (b, a), formed by different waves,
// are transposes bit for bit (a block (a, a) is symmetric to rounding only).
__device__ __forceinline__ void add_elastic(const double n[3], const double m[3], double ln, double lm, double G,
                                            double dV, double K[9])
{
    const double nm = n[0] * m[0] + n[1] * m[1] + n[2] * m[2];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            K[3 * i + j] += dV * (ln * n[i] * (lm * m[j]) + G * (n[j] * m[i] + (i == j ? nm : 0.0)));
}

// block += dV B_a^T D B_b with the general symmetric D of a surrogate point;
// lower: a <= b.  The product is formed with the lower local node on the left
// and transposed for b < a, so that (a, b) and (b, a) are transposes bit for bit.
__device__ __forceinline__ void add_general(const double ga[3], const double gb[3], bool lower, double dV,
                                            const float *__restrict__ dsur, size_t ngp_total, size_t gp, double K[9])
{
    double D[36], n[3], m[3];
    int k = 0;
#pragma unroll
    for (int r = 0; r < 6; r++)
#pragma unroll
        for (int c = r; c < 6; c++, k++) D[6 * r + c] = D[6 * c + r] = (double)dsur[(size_t)k * ngp_total + gp];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        n[i] = lower ? ga[i] : gb[i];
        m[i] = lower ? gb[i] : ga[i];
    }
    // columns of B_b: x (m0,0,0,0,m2,m1), y (0,m1,0,m2,0,m0), z (0,0,m2,m1,m0,0)
    double DB[6][3], V[9];
#pragma unroll
    for (int r = 0; r < 6; r++) {
        DB[r][0] = D[6 * r + 0] * m[0] + D[6 * r + 4] * m[2] + D[6 * r + 5] * m[1];
        DB[r][1] = D[6 * r + 1] * m[1] + D[6 * r + 3] * m[2] + D[6 * r + 5] * m[0];
        DB[r][2] = D[6 * r + 2] * m[2] + D[6 * r + 3] * m[1] + D[6 * r + 4] * m[0];
    }
#pragma unroll
    for (int j = 0; j < 3; j++) {
        V[0 + j] = n[0] * DB[0][j] + n[2] * DB[4][j] + n[1] * DB[5][j];
        V[3 + j] = n[1] * DB[1][j] + n[2] * DB[3][j] + n[0] * DB[5][j];
        V[6 + j] = n[2] * DB[2][j] + n[1] * DB[3][j] + n[0] * DB[4][j];
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) K[3 * i + j] += dV * (lower ? V[3 * i + j] : V[3 * j + i]);
}

// The sources of a node's columns in one pass of SLOTS elements: byte slot of
// column p's SLOTS-byte code is 3 b + j, the column of the slot's element
// rows that adds there, or 255.
template <int SLOTS>
__device__ __forceinline__ void clear_codes(int t, int L, uint64_t *codes)
{
    wave_lds_fence();   // the pass before has read them
    for (int p = t; p < L * (SLOTS / 8); p += 64) codes[p] = ~0ull;
    wave_lds_fence();
}

// One pass's element rows (sV: SLOTS x 3 x NC doubles) summed into the node's
// rows, in slot order.  Passes after the first go on from what the lane itself
// has written: one running sum per entry in ascending element order, the same
// for (i, j) and (j, i).  (Adding slot after slot into LDS rows instead moves 8 of 64
// lanes at a time: 1.9 ms for the 1,085,825 nodes of the 64x64x256 block.)
//
// Hexahedra, 81 columns of up to 8 sources: each lane owns entries t, t + 64,
// ... of the three rows, and a slot without a source reads a zero (sV[zero]),
// so that all of an entry's reads are in flight together.
template <int NC>
__device__ __forceinline__ void rows_sum_entries(int t, int q0, int q1, int q2, int L, const double *sV, int zero,
                                                 const uint64_t *codes, const int32_t *__restrict__ rowptr,
                                                 double *__restrict__ val, bool first)
{
    for (int x = t; x < 3 * L; x += 64) {
        const int i = (x >= L) + (x >= 2 * L), p = x - i * L;
        const int qi = i == 0 ? q0 : i == 1 ? q1 : q2;
        const uint64_t w = codes[p];
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int c = (int)(w >> (8 * k)) & 255;
            v[k] = sV[c != 255 ? (k * 3 + i) * NC + c : zero];
        }
        if (qi > 0) {
            double *o = val + rowptr[qi - 1] + p;
            double s = first ? 0.0 : *o;
#pragma unroll
            for (int k = 0; k < 8; k++) s += v[k];
            *o = s;
        }
    }
}

// Tetrahedra, 45 columns with few of 16 slots each: a lane owns a column of
// all three rows and reads the sources it has (1.06 against 1.19 ms for the
// 412,000 nodes of the 70x70x82 block with one entry a lane).  The lane's first
// column stays in acc over the passes: 0.96 ms.
template <int NC>
__device__ __forceinline__ void rows_sum_columns(int t, const int q[3], int L, const double *sV,
                                                 const uint64_t *codes, const int32_t *__restrict__ rowptr,
                                                 double *__restrict__ val, bool first, bool last, double acc[3])
{
    for (int p = t; p < L; p += 64) {
        double s[3] = {acc[0], acc[1], acc[2]};
        if (p != t) {
#pragma unroll
            for (int i = 0; i < 3; i++) s[i] = !first && q[i] > 0 ? val[rowptr[q[i] - 1] + p] : 0.0;
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint64_t w = codes[2 * p + h];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int c = (int)(w >> (8 * k)) & 255;
                if (c != 255) {
#pragma unroll
                    for (int i = 0; i < 3; i++) s[i] += sV[((8 * h + k) * 3 + i) * NC + c];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 3; i++) {
            if (p == t) acc[i] = s[i];
            if ((p != t || last) && q[i] > 0) val[rowptr[q[i] - 1] + p] = s[i];
        }
    }
}

// LSpace rows, two nodes a wave.  Slot k = t / 4 of 16 is an element of the
// first (k < 8) or second node; lane (k, q) owns the element's nodes q and
// q + 4, which differ in the sign of zeta only.  For each sign of xi the four
// lanes of a slot form J^-1 and the tangent parts of its four Gauss points
// into LDS, and every lane then runs over those points, forming the gradients
// g (and M g) of its two nodes and of the row's node a: one read of a point
// serves two blocks.  Elastic: J^-1 (nine divisions), the gradients and the
// blocks are formed by the operations of gp_geometry and k_assemble in their
// order, and the rows summed in ascending element order, so that K keeps the
// bits of stored element matrices.  A mixed-precision solve to 1e-8 determines
// its solution to about 1e-9, and one rounding of K moves it by as much.
//
// Bound, by counters on the plastic 1,048,576-element block: FP64 issue, 66 %
// of the cycles, and what two waves a SIMD leave uncovered (40 % of the waves'
// time is waiting; 206 VGPRs with the tangent, 172 without; bounding it to
// three or four waves spills and is slower); 4.9 GB of traffic are 1.1 TB/s.
// Tangent 4.0 ms, elastic 3.4 ms.  Before, storing every element's matrix (4.8
// GB) and summing the rows from them: 4.90 and 3.8 ms; with eight elements a
// wave in that form 1.87 + 2.03 ms, and no buffer to hold here.  One node a
// wave: 4.2 ms for the tangent.  With one reciprocal for the nine divisions the
// elastic form takes 2.6 ms, in other bits.
template <bool TAN, bool SUR>
__global__ __launch_bounds__(64) void k_assemble_rows_hex(AsmArgs A)
{
    constexpr int NP = TAN ? 18 : 10;   // doubles per point: J^-1 (9), [M (6), cd, kd,] dV (< 0: surrogate D)
    __shared__ __align__(16) double sV[16 * 72 + 2];   // points; the element rows after
    __shared__ double sX[3][8][16];                    // coordinates of the slots' nodes
    extern __shared__ __align__(16) unsigned char sDyn[];
    static_assert(64 * NP <= 16 * 72, "shared buffer");
    const int t = threadIdx.x, k = t >> 2, q = t & 3;
    const int n0 = 2 * blockIdx.x, nk = min(n0 + (k >> 3), A.nnode - 1);
    if (t == 0) sV[16 * 72] = 0.0;
    // this slot's node and the two nodes' element counts (0: no rows)
    int cnt[2], L[2], qn[2][3];
#pragma unroll
    for (int w = 0; w < 2; w++) {
        const int n = n0 + w;
        cnt[w] = L[w] = 0;
        qn[w][0] = qn[w][1] = qn[w][2] = 0;
        if (n >= A.nnode) continue;
#pragma unroll
        for (int i = 0; i < 3; i++) qn[w][i] = A.eqn[3 * (size_t)n + i];
        const int r0 = qn[w][0] > 0 ? qn[w][0] : qn[w][1] > 0 ? qn[w][1] : qn[w][2];
        if (r0 <= 0) continue;
        L[w] = A.rowptr[r0] - A.rowptr[r0 - 1];
        cnt[w] = A.nptr[n + 1] - A.nptr[n];
    }
    const int cmax = max(cnt[0], cnt[1]), ck = k < 8 ? cnt[0] : cnt[1];
    const int j0 = A.nptr[nk];
    uint64_t *codes[2] = {reinterpret_cast<uint64_t *>(sDyn), reinterpret_cast<uint64_t *>(sDyn) + L[0]};
    const double ga = 0.577350269189626;   // gauss_point
    for (int base = 0; base < cmax; base += 8) {
        const int slot = base + (k & 7);
        const bool valid = slot < ck;
        // spare slots repeat an element of the pair and add nothing
        const int ea = valid ? A.nadj[j0 + slot] : A.nadj[A.nptr[cnt[0] ? n0 : n0 + 1]], e = ea >> 3, a = ea & 7;
        const double *mp = A.mat + (size_t)HIPFEM_MATP * A.emat[e];
        clear_codes<8>(t, L[0] + L[1], codes[0]);
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const int b = q + 4 * w, nb = A.conn[(size_t)e * 8 + b];
            const int off = A.eoff[(size_t)ea * 8 + b];
            int r = 0;
#pragma unroll
            for (int d = 0; d < 3; d++) {
                sX[d][b][k] = A.coords[3 * (size_t)nb + d];
                if (A.eqn[3 * (size_t)nb + d] > 0 && off != 0xFFFF && valid)
                    reinterpret_cast<uint8_t *>(codes[k >> 3] + off + r++)[k & 7] = (uint8_t)(3 * b + d);
            }
        }
        wave_lds_fence();
        const double G = mp[1] / (2.0 * (1. + mp[2]));
        const double lam = mp[1] / (3.0 * (1. - 2. * mp[2])) - 2.0 * G / 3.0;
        // local signs: nodes q (zeta +) and q + 4 (zeta -), and the row's node
        const double sx = q >= 2 ? 1.0 : -1.0, sy = (q == 1 || q == 2) ? 1.0 : -1.0;
        const double ax = (a & 3) >= 2 ? 1.0 : -1.0, ay = ((a & 3) == 1 || (a & 3) == 2) ? 1.0 : -1.0,
                     az = a < 4 ? 1.0 : -1.0;
        double K0[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, K1[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 1
        for (int hx = 0; hx < 2; hx++) {
            const double xi = hx ? ga : -ga;
            {
                PointState ps;   // in flight while J is formed
                if constexpr (TAN) ps = load_point(A.state, A.ngp_total, (size_t)e * 8 + 4 * hx + q);
                // point (xi, eta, zeta) of lane q: bits 2 and 1 of the point number
                const double eta = (q & 2) ? ga : -ga, ze = (q & 1) ? ga : -ga;
                const double xm = 1. - xi, xp = 1. + xi, ym = 1. - eta, yp = 1. + eta, zm = 1. - ze, zp = 1. + ze;
                const double yz[4] = {0.125 * ym * zm, 0.125 * ym * zp, 0.125 * yp * zm, 0.125 * yp * zp};
                const double xz[4] = {0.125 * xm * zm, 0.125 * xm * zp, 0.125 * xp * zm, 0.125 * xp * zp};
                const double xy[4] = {0.125 * xm * ym, 0.125 * xm * yp, 0.125 * xp * ym, 0.125 * xp * yp};
                double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int c = 0; c < 8; c++) {   // the signs of dndxi_hexlin
                    const int bx = (c & 3) >= 2, by = (c & 3) == 1 || (c & 3) == 2, bz = c < 4;
                    const double dN[3] = {bx ? yz[2 * by + bz] : -yz[2 * by + bz],
                                          by ? xz[2 * bx + bz] : -xz[2 * bx + bz],
                                          bz ? xy[2 * bx + by] : -xy[2 * bx + by]};
#pragma unroll
                    for (int i = 0; i < 3; i++) {
                        const double X = sX[i][c][k];
#pragma unroll
                        for (int j = 0; j < 3; j++) J[3 * i + j] += X * dN[j];
                    }
                    if (c & 1) __builtin_amdgcn_sched_barrier(0);   // keeps two nodes' loads in flight
                }
                double P[NP] = {}, dV = 0.0;
                if (!(TAN ? hex_inverse_rcp(J, P, dV) : hex_inverse(J, P, dV))) atomicMin(A.bad, e);
                dV = fabs(dV);   // the rule's weights are 1
                if constexpr (TAN) {
                    const size_t gp = (size_t)e * 8 + 4 * hx + q;
                    point_parts(mp, dV, ps, P[15], P[16], P + 9);
                    P[17] = (SUR && A.sflag[gp]) ? -dV : dV;
                } else {
                    P[9] = dV;
                }
                wave_lds_fence();   // the other sign's points have been read
#pragma unroll
                for (int i = 0; i < NP; i += 2)
                    *reinterpret_cast<d2_t *>(&sV[(q * 16 + k) * NP + i]) = d2_t{P[i], P[i + 1]};
                wave_lds_fence();
            }
            const double x = 1. + sx * xi, xa = 1. + ax * xi;
#pragma unroll 1
            for (int hy = 0; hy < 2; hy++) {
                const double eta = hy ? ga : -ga, y = 1. + sy * eta, ya = 1. + ay * eta;
                const double bx = 0.125 * sx * y, by = 0.125 * sy * x, bz = 0.125 * x * y;
                const double cx = 0.125 * ax * ya, cy = 0.125 * ay * xa, cz = 0.125 * az * xa * ya;
#pragma unroll
                for (int hz = 0; hz < 2; hz++) {
                    const double ze = hz ? ga : -ga, zp = 1. + ze, zm = 1. - ze, za = 1. + az * ze;
                    double R[NP];
#pragma unroll
                    for (int i = 0; i < NP; i += 2) {
                        const d2_t w = *reinterpret_cast<const d2_t *>(&sV[((2 * hy + hz) * 16 + k) * NP + i]);
                        R[i] = w.x;
                        R[i + 1] = w.y;
                    }
                    double n[3], m0[3], m1[3];
#pragma unroll
                    for (int j = 0; j < 3; j++) {
                        n[j] = cx * za * R[j] + cy * za * R[3 + j] + cz * R[6 + j];
                        m0[j] = bx * zp * R[j] + by * zp * R[3 + j] + bz * R[6 + j];
                        m1[j] = bx * zm * R[j] + by * zm * R[3 + j] + -bz * R[6 + j];
                    }
                    if constexpr (TAN) {
                        if (SUR && R[17] < 0.0) {
                            const size_t gp = (size_t)e * 8 + 4 * hx + 2 * hy + hz;
                            add_general(n, m0, a <= q, -R[17], A.dsur, A.ngp_total, gp, K0);
                            add_general(n, m1, a <= q + 4, -R[17], A.dsur, A.ngp_total, gp, K1);
                        } else {
                            double va[3], vb[3];
                            tensor_times(R + 9, n, va);
                            tensor_times(R + 9, m0, vb);
                            add_parts(n, m0, R[15], R[16], va, vb, K0);
                            tensor_times(R + 9, m1, vb);
                            add_parts(n, m1, R[15], R[16], va, vb, K1);
                        }
                    } else {
                        add_elastic(n, m0, a <= q ? lam : 1.0, a <= q ? 1.0 : lam, G, R[9], K0);
                        add_elastic(n, m1, a <= q + 4 ? lam : 1.0, a <= q + 4 ? 1.0 : lam, G, R[9], K1);
                    }
                }
            }
        }
        wave_lds_fence();
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) {
                sV[(k * 3 + i) * 24 + 3 * q + j] = K0[3 * i + j];
                sV[(k * 3 + i) * 24 + 3 * q + 12 + j] = K1[3 * i + j];
            }
        wave_lds_fence();
#pragma unroll
        for (int w = 0; w < 2; w++)
            if (base < cnt[w])
                rows_sum_entries<24>(t, qn[w][0], qn[w][1], qn[w][2], L[w], sV + w * 8 * 72, (16 - 8 * w) * 72,
                                     codes[w], A.rowptr, A.val, base == 0);
    }
}

// LTRSpace rows.  Lane (slot k, b): element k of the pass (16 a wave), its
// node b.  The four lanes of an element exchange the coordinates by quad
// permutes; each forms its own node's gradient g_b = +-(x_j - x_i) x (x_k -
// x_i) / det J of the opposite face (the cofactor form of
// fei3dtetlin.C:116-168), the row's node a shares g_a and M g_a through LDS.
//
// Bound, by counters on the plastic 2,410,800-element block: VALU issue, 69 % of
// the cycles, with 60 % of the waves' time spent waiting for the gathers and
// LDS.  Tangent 0.96 ms; 31 color launches adding 24-byte pieces into the
// zeroed values took 5.8 ms.
template <bool TAN, bool SUR>
__global__ __launch_bounds__(64) void k_assemble_rows_tet(AsmArgs A)
{
    __shared__ __align__(16) double sV[16 * 3 * 12];
    __shared__ __align__(16) double sA[16][6];
    extern __shared__ __align__(16) unsigned char sDyn[];
    uint64_t *sCodes = reinterpret_cast<uint64_t *>(sDyn);
    const int n = blockIdx.x;
    if (n >= A.nnode) return;
    const int t = threadIdx.x, k = t >> 2, b = t & 3;
    int q[3];
#pragma unroll
    for (int i = 0; i < 3; i++) q[i] = A.eqn[3 * (size_t)n + i];
    const int r0 = q[0] > 0 ? q[0] : q[1] > 0 ? q[1] : q[2];
    if (r0 <= 0) return;
    const int L = A.rowptr[r0] - A.rowptr[r0 - 1];
    const int j0 = A.nptr[n], cnt = A.nptr[n + 1] - j0;
    double acc[3] = {0.0, 0.0, 0.0};
    for (int base = 0; base < cnt; base += 16) {
        const int slot = base + k;
        const bool valid = slot < cnt;
        const int ea = A.nadj[j0 + (valid ? slot : cnt - 1)], e = ea >> 2, a = ea & 3;
        const int nb = A.conn[(size_t)e * 4 + b];
        const int off = A.eoff[((size_t)e * 4 + a) * 4 + b];
        const double *mp = A.mat + (size_t)HIPFEM_MATP * A.emat[e];
        PointState ps;
        if constexpr (TAN) ps = load_point(A.state, A.ngp_total, e);
        int qb[3];
        double v[3], p[3], r[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            v[d] = A.coords[3 * (size_t)nb + d];
            qb[d] = A.eqn[3 * (size_t)nb + d];
        }
        double w[3];   // x_b - x_i
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double xi = dpp_d<0x39>(v[d]);            // node b + 1 (mod 4)
            p[d] = dpp_d<0x4E>(v[d]) - xi;                  // node b + 2
            r[d] = dpp_d<0x93>(v[d]) - xi;                  // node b + 3
            w[d] = v[d] - xi;
        }
        const double sg = (b & 1) ? 1.0 : -1.0;
        double m[3] = {sg * (p[1] * r[2] - r[1] * p[2]), sg * (p[2] * r[0] - r[2] * p[0]),
                       sg * (p[0] * r[1] - r[0] * p[1])};
        // one det J for the four lanes (node 4's: exact symmetry of K)
        const double det = dpp_d<0xFF>(m[0] * w[0] + m[1] * w[1] + m[2] * w[2]);
        if (!(det > 0.0)) atomicMin(A.bad, e);
        const double id = 1.0 / det, dV = fabs(det) * (1.0 / 6.0);
        double vb[3] = {0, 0, 0}, cd, kd, mm[6];
#pragma unroll
        for (int j = 0; j < 3; j++) m[j] *= id;
        if constexpr (TAN) {
            point_parts(mp, dV, ps, cd, kd, mm);
            tensor_times(mm, m, vb);
        }
        wave_lds_fence();
        if (b == a) {
#pragma unroll
            for (int j = 0; j < 3; j++) {
                sA[k][j] = m[j];
                if constexpr (TAN) sA[k][3 + j] = vb[j];
            }
        }
        wave_lds_fence();
        double na[3], va[3] = {0, 0, 0}, K[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 3; j++) {
            na[j] = sA[k][j];
            if constexpr (TAN) va[j] = sA[k][3 + j];
        }
        if constexpr (TAN) {
            if (SUR && A.sflag[e])
                add_general(na, m, a <= b, dV, A.dsur, A.ngp_total, e, K);
            else
                add_parts(na, m, cd, kd, va, vb, K);
        } else {
            const double G = mp[1] / (2.0 * (1. + mp[2]));
            const double lam = mp[1] / (3.0 * (1. - 2. * mp[2])) - 2.0 * G / 3.0;
            add_elastic(na, m, a <= b ? lam : 1.0, a <= b ? 1.0 : lam, G, dV, K);
        }
        clear_codes<16>(t, L, sCodes);
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) sV[(k * 3 + i) * 12 + 3 * b + j] = K[3 * i + j];
        if (valid && off != 0xFFFF) {
            uint8_t *bytes = reinterpret_cast<uint8_t *>(sCodes);
            int rk = 0;
#pragma unroll
            for (int j = 0; j < 3; j++)
                if (qb[j] > 0) bytes[(off + rk++) * 16 + k] = (uint8_t)(3 * b + j);
        }
        wave_lds_fence();
        rows_sum_columns<12>(t, q, L, sV, sCodes, A.rowptr, A.val, base == 0, base + 16 >= cnt, acc);
    }
}

// K_e of the QSpace elements from e0 on, 60 x 60 row-major: 256 threads an element.
// The (point, node) pairs, the 9 entries of every point's J and the 210 node
// pairs a <= b are each shared out over the threads; a block is stored with
// its transpose.
//
// Bound, by counters on 9,261 elements: VALU issue, 84 % of the cycles: 0.153
// ms.  The rows summed from the matrices (267 MB each way) wait for their
// loads, 69 % of the waves' time: 0.150 ms.  Eight color launches of one wave an
// element, which leave a SIMD one wave, took 0.78 ms.
template <bool TAN, bool SUR>
__global__ __launch_bounds__(256) void k_element_matrices_quad(AsmArgs A, double *__restrict__ kbuf, int e0)
{
    constexpr int NGP = 27, NEN = 20;
    __shared__ double sX[60];
    __shared__ double sN[NGP][60];    // dN/dxi, then dN/dx
    __shared__ double sJ[NGP][9];     // J, then J^-1
    __shared__ double sQ[NGP][TAN ? 10 : 2];   // dV (< 0: surrogate D), [cd, kd, M (6)]
    const int e = e0 + blockIdx.x, t = threadIdx.x;
    for (int k = t; k < 60; k += 256) sX[k] = A.coords[3 * (size_t)A.conn[(size_t)e * NEN + k / 3] + k % 3];
    for (int k = t; k < NGP * NEN; k += 256) {
        double xi[3], w, d[3];
        gauss_point(HIPFEM_QSPACE, k / NEN, xi, w);
        dndxi_hexquad(k % NEN, xi, d);
#pragma unroll
        for (int j = 0; j < 3; j++) sN[k / NEN][3 * (k % NEN) + j] = d[j];
    }
    __syncthreads();
    if (t < NGP * 9) {
        const int g = t / 9, i = t % 9 / 3, j = t % 3;
        double v = 0.0;
#pragma unroll 4
        for (int a = 0; a < NEN; a++) v += sX[3 * a + i] * sN[g][3 * a + j];
        sJ[g][3 * i + j] = v;
    }
    __syncthreads();
    const double *mp = A.mat + (size_t)HIPFEM_MATP * A.emat[e];
    if (t < NGP) {
        double J[9], I[9], xi[3], w, det;
        gauss_point(HIPFEM_QSPACE, t, xi, w);
#pragma unroll
        for (int i = 0; i < 9; i++) J[i] = sJ[t][i];
        if (!hex_inverse_rcp(J, I, det)) atomicMin(A.bad, e);
        const double dV = fabs(det) * w;
#pragma unroll
        for (int i = 0; i < 9; i++) sJ[t][i] = I[i];
        sQ[t][0] = dV;
        if constexpr (TAN) {
            const size_t gp = (size_t)e * NGP + t;
            double cd, kd, m[6];
            point_parts(mp, dV, load_point(A.state, A.ngp_total, gp), cd, kd, m);
            sQ[t][1] = cd;
            sQ[t][2] = kd;
#pragma unroll
            for (int i = 0; i < 6; i++) sQ[t][3 + i] = m[i];
            if (SUR && A.sflag[gp]) sQ[t][0] = -dV;
        }
    }
    __syncthreads();
    for (int k = t; k < NGP * NEN; k += 256) {
        const int g = k / NEN, a = k % NEN;
        const double d0 = sN[g][3 * a], d1 = sN[g][3 * a + 1], d2 = sN[g][3 * a + 2];
#pragma unroll
        for (int j = 0; j < 3; j++) sN[g][3 * a + j] = d0 * sJ[g][j] + d1 * sJ[g][3 + j] + d2 * sJ[g][6 + j];
    }
    __syncthreads();
    if (t >= NEN * (NEN + 1) / 2) return;
    int a = 0, rem = t;
    while (rem >= NEN - a) rem -= NEN - a++;
    const int b = a + rem;
    const double G = mp[1] / (2.0 * (1. + mp[2]));
    const double lam = mp[1] / (3.0 * (1. - 2. * mp[2])) - 2.0 * G / 3.0;
    double K[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 3
    for (int g = 0; g < NGP; g++) {
        const double n[3] = {sN[g][3 * a], sN[g][3 * a + 1], sN[g][3 * a + 2]};
        const double m[3] = {sN[g][3 * b], sN[g][3 * b + 1], sN[g][3 * b + 2]};
        if constexpr (TAN) {
            if (SUR && sQ[g][0] < 0.0) {
                add_general(n, m, true, -sQ[g][0], A.dsur, A.ngp_total, (size_t)e * NGP + g, K);
            } else {
                double va[3], vb[3];
                tensor_times(&sQ[g][3], n, va);
                tensor_times(&sQ[g][3], m, vb);
                add_parts(n, m, sQ[g][1], sQ[g][2], va, vb, K);
            }
        } else {
            add_elastic(n, m, lam, 1.0, G, sQ[g][0], K);
        }
    }
    double *o = kbuf + (size_t)blockIdx.x * 3600;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) o[(3 * a + i) * 60 + 3 * b + j] = K[3 * i + j];
    if (a != b) {
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int i = 0; i < 3; i++) o[(3 * b + j) * 60 + 3 * a + i] = K[3 * i + j];
    }
}

// The rows of node n from the stored matrices of elements [e0, e1): eight
// elements a pass, whose three rows (3 x 3 NEN contiguous doubles) go to LDS as
// they lie; the columns are then summed and written.  One wave per node.  The
// running sums of a node whose elements lie in several ranges go on from val,
// so the ranges do not change the result.
template <int NEN>
__global__ __launch_bounds__(64) void k_assemble_gather(AsmArgs A, const double *__restrict__ kbuf, int e0, int e1)
{
    constexpr int NC = 3 * NEN, ROW2 = 3 * NC / 2;   // 16-byte words of an element's three rows
    __shared__ __align__(16) double sV[8 * 3 * NC + 2];
    extern __shared__ __align__(16) unsigned char sDyn[];
    uint64_t *sCodes = reinterpret_cast<uint64_t *>(sDyn);
    const int n = blockIdx.x;
    if (n >= A.nnode) return;
    const int t = threadIdx.x;
    if (t == 0) sV[8 * 3 * NC] = 0.0;
    int q[3];
#pragma unroll
    for (int i = 0; i < 3; i++) q[i] = A.eqn[3 * (size_t)n + i];
    const int r0 = q[0] > 0 ? q[0] : q[1] > 0 ? q[1] : q[2];
    if (r0 <= 0) return;   // no free dof: no rows
    const int L = A.rowptr[r0] - A.rowptr[r0 - 1];
    const int jn = A.nptr[n];
    int j0 = jn, j1 = A.nptr[n + 1];
    if (e0 > 0 || e1 < A.nelem) {   // the list ascends: its part in [e0, e1)
        for (int hi = j1; j0 < hi;) {
            const int mid = (j0 + hi) / 2;
            if (A.nadj[mid] < (int64_t)e0 * NEN) j0 = mid + 1;
            else hi = mid;
        }
        for (int lo = j0; lo < j1;) {
            const int mid = (lo + j1) / 2;
            if (A.nadj[mid] < (int64_t)e1 * NEN) lo = mid + 1;
            else j1 = mid;
        }
    }
    const int cnt = j1 - j0;
    for (int base = 0; base < cnt; base += 8) {
        const int ns = min(8, cnt - base);
        d2_t v[(8 * ROW2 + 63) / 64];
#pragma unroll
        for (int u = 0; u < (8 * ROW2 + 63) / 64; u++) {
            const int idx = u * 64 + t, s = min(idx / ROW2, ns - 1);
            const size_t ea = (size_t)A.nadj[j0 + base + s] - (size_t)e0 * NEN;
            v[u] = reinterpret_cast<const d2_t *>(kbuf + ea * (3 * NC))[idx % ROW2];
        }
        clear_codes<8>(t, L, sCodes);
        uint8_t *bytes = reinterpret_cast<uint8_t *>(sCodes);
        for (int i = t; i < ns * NEN; i += 64) {
            const int s = i / NEN, b = i % NEN, ea = A.nadj[j0 + base + s];
            const int off = A.eoff[(size_t)ea * NEN + b];
            const int nb = A.conn[(size_t)(ea / NEN) * NEN + b];
            int r = 0;
#pragma unroll
            for (int j = 0; j < 3; j++)
                if (A.eqn[3 * (size_t)nb + j] > 0 && off != 0xFFFF) bytes[(off + r++) * 8 + s] = (uint8_t)(3 * b + j);
        }
#pragma unroll
        for (int u = 0; u < (8 * ROW2 + 63) / 64; u++) {
            const int idx = u * 64 + t;
            if (idx / ROW2 < ns) reinterpret_cast<d2_t *>(sV)[idx] = v[u];
        }
        wave_lds_fence();
        rows_sum_entries<NC>(t, q[0], q[1], q[2], L, sV, 8 * 3 * NC, sCodes, A.rowptr, A.val, j0 + base == jn);
    }
}

}  // namespace hipfem
