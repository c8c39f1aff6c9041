// Linear-algebra kernels of the coupled solve:
//   block SpMV        coupledMatrix::matrixMul -> blockFvMatrix::Amul
//                     (coupledMatrix.C:66-123, blockFvMatrix.C:331-381)
//   LU-SGS            lusgs::precondition (lusgs.C:220-382), level-scheduled
//   block-Jacobi      Jacobi::precondition / JacobiSmoother (Jacobi.C:55-132)
//   GMRES pieces      gmres::solveDelta (gmres.C:772-1108): reductions,
//                     orthogonalisation, Givens, back-substitution, update.
//
// Vectors are SoA [5][nC] in [rho, rhoE, rhoUx, rhoUy, rhoUz] order.
// Off-diagonal 5x5 blocks live in a sliced-ELL layout (64-row slices, one
// wavefront per slice, entry-major inside a slot) so every block load of a
// wavefront is one contiguous 64-element run.
#include "icsf_flux.h"
#include "icsf_kernels.h"
#include "icsf_math.h"
#include "icsf_views.h"

namespace icsf {

namespace {

// ---------------------------------------------------------- reductions ----
__device__ __forceinline__ double waveSum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// Wave sums of NA values per lane (NA a power of two up to 64): every lane
// keeps half of its values and hands the other half to its partner, so the
// values thin out as the lanes combine: 17 exchanges for 16 values instead of
// 96.  Lane `lane` returns the sum of value `id` (the lanes of one value all
// hold it); the pairs added are those of waveSum, whatever NA.
template <int HALF, int D, int NA>
__device__ __forceinline__ void waveFold(double (&v)[NA], int lane, int& id) {
    if constexpr (HALF >= 1) {
        const bool hi = lane & D;
#pragma unroll
        for (int k = 0; k < HALF; ++k) {
            const double give = hi ? v[k] : v[k + HALF], keep = hi ? v[k + HALF] : v[k];
            v[k] = keep + __shfl_xor(give, D, 64);
        }
        if (hi) id += HALF;
        waveFold<HALF / 2, D / 2>(v, lane, id);
    } else if constexpr (D >= 1) {
        v[0] += __shfl_xor(v[0], D, 64);
        waveFold<0, D / 2>(v, lane, id);
    }
}
template <int NA>
__device__ __forceinline__ double waveSums(double (&v)[NA], int lane, int& id) {
    id = 0;
    waveFold<NA / 2, 32>(v, lane, id);
    return v[0];
}

// The norm whose partials (nb of them) are at part, by one wavefront; every
// lane returns it.
__device__ __forceinline__ double waveNorm(const double* __restrict__ part, int nb) {
    const int lane = threadIdx.x & 63;
    double v = 0;
    for (int b = lane; b < nb; b += 64) v += part[b];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return sqrt(v);
}

template <typename T>
__device__ __forceinline__ double ld(const T* p, size_t i) { return (double)p[i]; }

// ---------------------------------------------------------------- SpMV ----
// Per output component three partial sums are kept (scalar-scalar,
// scalar-scalar', scalar/vector-vector parts) and combined in the order
// coupledMatrix::matrixMul adds its sub-block products.
// One block row of y = A (x/scal): the diagonal block, then the
// off-diagonal slots in column order, three partial sums per row (scalar
// rho column, scalar rhoE column, vector rhoU columns) combined as the
// blockFvMatrix sub-block sums (coupledMatrix.C:66-123).
// Off-diagonal block of sliced-ELL slot sk for the row in lane `lane`, in
// arithmetic type A: read from full storage, or generated from the slot's
// NGEN generators in the storage precision (the same bits as the block the
// Jacobian kernel would have stored, for FP64).
// NT: non-temporal loads (the SpMV rows: each slot is read once per pass
// and a full L2 pass lies between reads; keeping these lines out of L2
// leaves it to the gathered vectors).
template <typename TB, typename A, bool GEN, bool NT = false>
__device__ __forceinline__ void slotBlock(const MeshView& m, const TB* __restrict__ blk, size_t sk, int lane,
                                          A b[NB]) {
    if (GEN) {
        const size_t gb = sk * NGEN * 64 + lane;
        TB g[NGEN], t[NB];
#pragma unroll
        for (int e = 0; e < NGEN; ++e)
            g[e] = NT ? __builtin_nontemporal_load(blk + gb + (size_t)e * 64) : blk[gb + (size_t)e * 64];
        const TB* gm = (const TB*)m.genMo;
        TB mo = (TB)0;
        if (gm) mo = NT ? __builtin_nontemporal_load(gm + sk * 64 + lane) : gm[sk * 64 + lane];
        blockFromGen<TB>(g, (TB)m.gamma, t, mo, gm != nullptr);
#pragma unroll
        for (int e = 0; e < NB; ++e) b[e] = (A)t[e];
    } else {
        const size_t bb = sk * NB * 64 + lane;
#pragma unroll
        for (int e = 0; e < NB; ++e) b[e] = (A)blk[bb + (size_t)e * 64];
    }
}

// Cyclic faces of row c: interfacesUpper & (x_far with its momentum part
// transformed by forwardT), added to the three partial sums after the
// internal faces (blockFvMatrix::Amul, blockFvMatrix.C:398-420).  Not part
// of the LU-SGS sweeps (lusgs.C:143-186 visits internal faces only).
template <typename TB, typename A, typename XF>
__device__ __forceinline__ void spmvCyclic(const MeshView& m, const TB* __restrict__ blk, int c, XF X,
                                           A acc[5][3]) {
    const int q1 = m.cycRowOff[c + 1];
    for (int q = m.cycRowOff[c]; q < q1; ++q) {
        const int kc = m.cycRowK[q];
        const int j = m.cycCell[kc];
        const double* R = m.cycR + 9 * (size_t)kc;
        const A x0 = X(0, j), x1 = X(1, j), x2 = X(2, j), x3 = X(3, j), x4 = X(4, j);
        const A v2 = (A)R[0] * x2 + (A)R[1] * x3 + (A)R[2] * x4;
        const A v3 = (A)R[3] * x2 + (A)R[4] * x3 + (A)R[5] * x4;
        const A v4 = (A)R[6] * x2 + (A)R[7] * x3 + (A)R[8] * x4;
        const TB* ib = blk + m.cycBase + (size_t)kc * NB;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const A b0 = (A)ib[5 * i], b1 = (A)ib[5 * i + 1], b2 = (A)ib[5 * i + 2], b3 = (A)ib[5 * i + 3],
                    b4 = (A)ib[5 * i + 4];
            acc[i][0] += b0 * x0;
            acc[i][1] += b1 * x1;
            const A dd = b2 * v2 + b3 * v3 + b4 * v4;
            acc[i][2] += dd;
        }
    }
}

template <typename TB, typename TV, bool GEN>
__device__ __forceinline__ void spmvRow(const MeshView& m, const TB* __restrict__ blk, const TB* __restrict__ dg,
                                        const TV* __restrict__ x, const double* __restrict__ scal,
                                        TV* __restrict__ vout, TV* __restrict__ y, int c) {
    const size_t nC = m.nC;
    typedef TV A;
    const A beta = scal ? (A)(*scal) : (A)1;
    auto X = [&](int k, int j) -> A {
        const A v = x[(size_t)k * nC + j];
        return scal ? v / beta : v;
    };
    A xc[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) xc[k] = X(k, c);
    if (vout)
#pragma unroll
        for (int k = 0; k < 5; ++k) stnt(vout + (size_t)k * nC + c, xc[k]);
    A acc[5][3];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const A b0 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i)),
                b1 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i + 1));
        const A b2 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i + 2)),
                b3 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i + 3)),
                b4 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i + 4));
        acc[i][0] = b0 * xc[0];
        acc[i][1] = b1 * xc[1];
        acc[i][2] = b2 * xc[2] + b3 * xc[3] + b4 * xc[4];
    }
    const int sl = c >> 6, lane = c & 63;
    const int len = m.rowLen[c];
    const size_t base = (size_t)m.slicePtr[sl];
    for (int k = 0; k < len; ++k) {
        const size_t slot = (base + k) * 64 + lane;
        const int j = ldnt(m.col + slot);
        A xj[5];
#pragma unroll
        for (int q = 0; q < 5; ++q) xj[q] = X(q, j);
        A bk[NB];
        slotBlock<TB, A, GEN, true>(m, blk, base + k, lane, bk);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const A b0 = bk[5 * i], b1 = bk[5 * i + 1];
            const A b2 = bk[5 * i + 2], b3 = bk[5 * i + 3], b4 = bk[5 * i + 4];
            acc[i][0] += b0 * xj[0];
            acc[i][1] += b1 * xj[1];
            const A dd = b2 * xj[2] + b3 * xj[3] + b4 * xj[4];
            acc[i][2] += dd;
        }
    }
    if (m.nCyc > 0) spmvCyclic<TB, A>(m, blk, c, X, acc);
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        A r = (A)0 + acc[i][0];
        r = r + acc[i][1];
        r = r + acc[i][2];
        y[(size_t)i * nC + c] = r;
    }
}

template <typename TB, typename TV, bool GEN, int W = 1>
__global__ void __launch_bounds__(256, W) k_spmv(MeshView m, const TB* __restrict__ blk, const TB* __restrict__ dg,
                                              const TV* __restrict__ x, const double* __restrict__ scal,
                                              TV* __restrict__ vout, TV* __restrict__ y) {
    const int c = xcdBlock() * blockDim.x + threadIdx.x;
    if (c >= m.nC) return;
    spmvRow<TB, TV, GEN>(m, blk, dg, x, scal, vout, y, c);
}

// Harmonic-balance SpMV: row cell c of instance J = blockIdx.y.  The own
// instance's partial sums are those of k_spmv; the cross-instance terms
// (V_c D_JK) x_K are added in coupledMatrix::matrixMul order
// (coupledMatrix.C:66-123): scalar rows add the scalar columns of
// instances 0..nO-1 (own rho, rhoE blocks at K = J) and then the own
// vector column; vector rows add the own scalar columns and then the vector
// columns of instances 0..nO-1 (own block at K = J).
template <typename TB, typename TV, bool GEN>
__device__ __forceinline__ void spmvRowHB(const MeshView& m, const HBBlocks& hb, int J, const TV* __restrict__ x,
                                          const double* __restrict__ scal, TV* __restrict__ vout,
                                          TV* __restrict__ y, int c) {
    typedef TV A;
    const size_t nC = m.nC;
    const size_t vs = 5 * nC;
    const TB* blk = (const TB*)hb.blk[J];
    const TB* dg = (const TB*)hb.dg[J];
    const A beta = scal ? (A)(*scal) : (A)1;
    auto X = [&](int K, int k, int j) -> A {
        const A v = x[(size_t)K * vs + (size_t)k * nC + j];
        return scal ? v / beta : v;
    };
    A xc[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) xc[k] = X(J, k, c);
    if (vout)
#pragma unroll
        for (int k = 0; k < 5; ++k) vout[(size_t)J * vs + (size_t)k * nC + c] = xc[k];
    A acc[5][3];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const A b0 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i)),
                b1 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i + 1));
        const A b2 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i + 2)),
                b3 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i + 3)),
                b4 = (A)__builtin_nontemporal_load(dg + diagOff(c, 5 * i + 4));
        acc[i][0] = b0 * xc[0];
        acc[i][1] = b1 * xc[1];
        acc[i][2] = b2 * xc[2] + b3 * xc[3] + b4 * xc[4];
    }
    const int sl = c >> 6, lane = c & 63;
    const int len = m.rowLen[c];
    const size_t base = (size_t)m.slicePtr[sl];
    for (int k = 0; k < len; ++k) {
        const size_t slot = (base + k) * 64 + lane;
        const int j = ldnt(m.col + slot);
        A xj[5];
#pragma unroll
        for (int q = 0; q < 5; ++q) xj[q] = X(J, q, j);
        A bk[NB];
        slotBlock<TB, A, GEN, true>(m, blk, base + k, lane, bk);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const A b0 = bk[5 * i], b1 = bk[5 * i + 1];
            const A b2 = bk[5 * i + 2], b3 = bk[5 * i + 3], b4 = bk[5 * i + 4];
            acc[i][0] += b0 * xj[0];
            acc[i][1] += b1 * xj[1];
            const A dd = b2 * xj[2] + b3 * xj[3] + b4 * xj[4];
            acc[i][2] += dd;
        }
    }
    if (m.nCyc > 0) spmvCyclic<TB, A>(m, blk, c, [&](int k, int j) { return X(J, k, j); }, acc);
    const double Vc = m.V[c];
    const int nO = hb.nO;
    A out[5];
    // scalar rows
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        A r = (A)0;
        for (int K = 0; K < nO; ++K) {
            if (K == J) {
                r = r + acc[i][0];
                r = r + acc[i][1];
            } else {
                r = r + (A)(Vc * hb.D[J * nO + K]) * X(K, i, c);
            }
        }
        out[i] = r + acc[i][2];
    }
    // vector rows
#pragma unroll
    for (int i = 2; i < 5; ++i) {
        A r = (A)0 + acc[i][0];
        r = r + acc[i][1];
        for (int K = 0; K < nO; ++K) {
            if (K == J) r = r + acc[i][2];
            else r = r + (A)(Vc * hb.D[J * nO + K]) * X(K, i, c);
        }
        out[i] = r;
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) y[(size_t)J * vs + (size_t)i * nC + c] = out[i];
}

template <typename TB, typename TV, bool GEN>
__global__ void __launch_bounds__(256) k_spmv_hb(MeshView m, HBBlocks hb, const TV* __restrict__ x,
                                                 const double* __restrict__ scal, TV* __restrict__ vout,
                                                 TV* __restrict__ y) {
    const int c = xcdBlock() * blockDim.x + threadIdx.x;
    if (c >= m.nC) return;
    spmvRowHB<TB, TV, GEN>(m, hb, blockIdx.y, x, scal, vout, y, c);
}

// ------------------------------------ Arnoldi operator, two colours -------
// y = LU-SGS(A x), x = w/beta, on a two-level dependency graph: colour-0 rows
// have upper neighbours only (all colour 1), colour-1 rows lower ones only.
// With A = [D0 U; L D1] and the preconditioner ((1/rD + L) rD (1/rD + U))^-1:
//   phase 0 (colour-0 rows): z0 = D0 x0 + U x1,  t0 = x0 - rD0 z0
//   phase 1 (colour-1 rows): y1 = rD1 (D1 x1 + L x0 - L rD0 z0)
//                               = rD1 (D1 x1 + L t0)
//   phase 2 (colour-0 rows): y0 = rD0 (z0 - U y1)
// What bounds it: the generators or blocks streamed once per phase and the
// neighbour gathers beside them.  t0 (its own buffer) makes the product and
// the forward sweep of phase 1 one block product of one gathered vector: 5
// gathers per slot instead of 11 (x, y and rD) and half of its arithmetic;
// the 1/beta scaling is applied to row sums, 5 divisions per row instead of
// 5 per slot.  Phases 0 / 1 / 2 at 104x96x96, FP32 generators: 35 / 41 / 33
// us (36 / 52 / 38 us with x, y and rD gathered and the blocks formed);
// 64^3, FP64: 20 / 22 / 18 us (20 / 27 / 20 us).

// acc += B x of slot sk.  FP32 generators: the flux Jacobian is applied
// without forming its 25 entries (h A(U, E, n) x - (v + sv + mo) x, about 70
// operations instead of 190, and 15 registers less); FP64 forms the block,
// so that generator and block storage give the same bits.
template <typename TB, bool GEN>
__device__ __forceinline__ void slotApply(const MeshView& m, const TB (&g)[GEN ? NGEN : NB], TB mo, const TB x[5],
                                          TB acc[5]) {
    if constexpr (GEN && sizeof(TB) == 4) {
        const TB ux = g[0], uy = g[1], uz = g[2], E = g[3], nx = g[4], ny = g[5], nz = g[6], h = g[7];
        const TB gm = (TB)m.gamma, a2 = gm - (TB)1;
        const TB th = (TB)0.5 * a2 * fmaf(ux, ux, fmaf(uy, uy, uz * uz));
        const TB a1 = gm * E - th;
        const TB pu = fmaf(ux, nx, fmaf(uy, ny, uz * nz));
        const TB mn = fmaf(nx, x[2], fmaf(ny, x[3], nz * x[4]));
        const TB um = fmaf(ux, x[2], fmaf(uy, x[3], uz * x[4]));
        const TB k = fmaf(th, x[0], a2 * (x[1] - um));
        const TB s = fmaf(-pu, x[0], mn);
        const TB d = g[8] + g[9] + mo;
        acc[0] = fmaf(h, mn, fmaf(-d, x[0], acc[0]));
        acc[1] = fmaf(h, fmaf(a1, s, pu * (k + x[1])), fmaf(-d, x[1], acc[1]));
        acc[2] = fmaf(h, fmaf(nx, k, fmaf(ux, s, pu * x[2])), fmaf(-d, x[2], acc[2]));
        acc[3] = fmaf(h, fmaf(ny, k, fmaf(uy, s, pu * x[3])), fmaf(-d, x[3], acc[3]));
        acc[4] = fmaf(h, fmaf(nz, k, fmaf(uz, s, pu * x[4])), fmaf(-d, x[4], acc[4]));
    } else {
        TB t[NB];
        if constexpr (GEN) blockFromGen<TB>(g, (TB)m.gamma, t, mo, m.genMo != nullptr);
        else
#pragma unroll
            for (int e = 0; e < NB; ++e) t[e] = g[e];
#pragma unroll
        for (int i = 0; i < 5; ++i)
#pragma unroll
            for (int q = 0; q < 5; ++q) acc[i] = __builtin_fma(t[5 * i + q], x[q], acc[i]);
    }
}

// acc += sum over the row's slots of B_k v[col_k] (v: [5][nC]).  UN slots'
// columns, generators and gathers are in flight together.  NT: the slot data
// loaded non-temporally.
template <typename TB, bool GEN, bool NT, int UN>
__device__ __forceinline__ void rowApply(const MeshView& m, const TB* __restrict__ blk, const TB* __restrict__ v,
                                         int c, TB acc[5]) {
    constexpr int NE = GEN ? NGEN : NB;
    const size_t nC = m.nC;
    const int lane = c & 63, len = m.rowLen[c];
    const size_t base = (size_t)m.slicePtr[c >> 6];
    const TB* gm = (const TB*)m.genMo;
    for (int k = 0; k < len; k += UN) {
        int j[UN];
        TB g[UN][NE], mo[UN], x[UN][5];
#pragma unroll
        for (int u = 0; u < UN; ++u) j[u] = k + u < len ? ldnt(m.col + (base + k + u) * 64 + lane) : -1;
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const size_t sk = base + (k + u < len ? k + u : k);
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                const TB* q = blk + (sk * NE + e) * 64 + lane;
                g[u][e] = NT ? ldnt(q) : *q;
            }
            mo[u] = (TB)0;
            if (GEN && gm) mo[u] = NT ? ldnt(gm + sk * 64 + lane) : gm[sk * 64 + lane];
        }
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int q = 0; q < 5; ++q) x[u][q] = v[(size_t)q * nC + (j[u] < 0 ? c : j[u])];
#pragma unroll
        for (int u = 0; u < UN; ++u)
            if (j[u] >= 0) slotApply<TB, GEN>(m, g[u], mo[u], x[u], acc);
    }
}

// One phase of the operator for a row per thread: rows c0 + [0, n), or a
// cell list.  HB: instance blockIdx.y, with its cross-instance terms
// (V_c D_JK) x_K of the other instances.  W: waves per SIMD the registers
// must allow.
template <typename TB, bool GEN, int PH, bool HB, int UN, int W>
__global__ void __launch_bounds__(256, W) k_op(MeshView m, HBBlocks hb, const TB* __restrict__ blk_,
                                               const TB* __restrict__ dg_, const TB* __restrict__ w_,
                                               const double* __restrict__ scal, TB* __restrict__ vout,
                                               TB* __restrict__ t_, TB* __restrict__ y_,
                                               const double* __restrict__ rD, const int* __restrict__ cells, int c0,
                                               int n, NormIn norm) {
    const int i0 = xcdBlock() * blockDim.x + threadIdx.x;
    double bn = 1.0;
    if constexpr (PH == 0) {
        // beta from the norm's partials, by every block; the first one keeps
        // it for phase 1 and the cycle's end
        __shared__ double sb;
        if (norm.part) {
            if (threadIdx.x < 64) {
                const double v = waveNorm(norm.part, norm.nb);
                if (threadIdx.x == 0) {
                    sb = v;
                    if (blockIdx.x == 0 && blockIdx.y == 0) {
                        *norm.beta = v;
                        *norm.hn = v;
                    }
                }
            }
            __syncthreads();
            bn = sb;
        } else if (scal) bn = *scal;
    } else if (PH == 1 && scal) bn = *scal;
    const bool scaled = scal || (PH == 0 && norm.part);
    if (i0 >= n) return;
    const int c = cells ? ldnt(cells + i0) : c0 + i0;
    const size_t nC = m.nC;
    const int J = HB ? blockIdx.y : 0;
    const size_t off = HB ? (size_t)J * 5 * nC : 0;
    const TB* blk = HB ? (const TB*)hb.blk[J] : blk_;
    const TB* dg = HB ? (const TB*)hb.dg[J] : dg_;
    TB* y = y_ + off;
    TB* t = t_ + off;
    const TB rd = (TB)rD[c];
    TB acc[5];
    if constexpr (PH == 2) {
        TB z[5];
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            z[q] = y[(size_t)q * nC + c];
            acc[q] = (TB)0;
        }
        rowApply<TB, GEN, false, UN>(m, blk, y, c, acc);
#pragma unroll
        for (int q = 0; q < 5; ++q) y[(size_t)q * nC + c] = rd * (z[q] - acc[q]);
        return;
    }
    const TB* w = w_ + off;
    const TB beta = (TB)bn;
    TB x[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) x[q] = w[(size_t)q * nC + c];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        acc[i] = (TB)0;
#pragma unroll
        for (int q = 0; q < 5; ++q) acc[i] = __builtin_fma(ldnt(dg + diagOff(c, 5 * i + q)), x[q], acc[i]);
    }
    if (m.nCyc > 0) {
        // interface blocks on the far cells' rows of w, forwardT applied
        TB a3[5][3];
#pragma unroll
        for (int i = 0; i < 5; ++i) a3[i][0] = a3[i][1] = a3[i][2] = (TB)0;
        spmvCyclic<TB, TB>(m, blk, c, [&](int k, int j) { return w[(size_t)k * nC + j]; }, a3);
#pragma unroll
        for (int i = 0; i < 5; ++i) acc[i] += a3[i][0] + a3[i][1] + a3[i][2];
    }
    if (HB) {
        const double Vc = m.V[c];
        for (int K = 0; K < hb.nO; ++K) {
            if (K == J) continue;
            const TB d = (TB)(Vc * hb.D[J * hb.nO + K]);
#pragma unroll
            for (int q = 0; q < 5; ++q) acc[q] = __builtin_fma(d, w_[((size_t)K * 5 + q) * nC + c], acc[q]);
        }
    }
    if constexpr (PH == 0) {
        // sums of w, then scaled
        rowApply<TB, GEN, true, UN>(m, blk, w, c, acc);
        if (scaled)
#pragma unroll
            for (int q = 0; q < 5; ++q) {
                acc[q] /= beta;
                x[q] /= beta;
            }
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            y[(size_t)q * nC + c] = acc[q];
            t[(size_t)q * nC + c] = x[q] - rd * acc[q];
        }
    } else {
        if (scaled)
#pragma unroll
            for (int q = 0; q < 5; ++q) {
                acc[q] /= beta;
                x[q] /= beta;
            }
        rowApply<TB, GEN, true, UN>(m, blk, t, c, acc);
#pragma unroll
        for (int q = 0; q < 5; ++q) y[(size_t)q * nC + c] = rd * acc[q];
    }
    if (vout)
#pragma unroll
        for (int q = 0; q < 5; ++q) stnt(vout + off + (size_t)q * nC + c, x[q]);
}

// ------------------------------------------------------------- LU-SGS -----
// Forward sweep of one level: r[c] -= sum over lower neighbours p (in
// increasing p) of L_cp * (rD[p] r[p]).
template <typename TB, typename TV, bool GEN>
__device__ __forceinline__ void lusgsFwdRow(const MeshView& m, const TB* __restrict__ blk,
                                            const double* __restrict__ rD, TV* __restrict__ r, int c) {
    const int nl = m.nLower[c];
    if (nl == 0) return;
    const size_t nC = m.nC;
    typedef TV A;
    A acc[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) acc[i] = r[(size_t)i * nC + c];
    const int sl = c >> 6, lane = c & 63;
    const size_t base = (size_t)m.slicePtr[sl];
    for (int k = 0; k < nl; ++k) {
        const size_t slot = (base + k) * 64 + lane;
        const int p = m.col[slot];
        const A rd = (A)rD[p];
        A d[5];
#pragma unroll
        for (int q = 0; q < 5; ++q) d[q] = rd * r[(size_t)q * nC + p];
        A bk[NB];
        slotBlock<TB, A, GEN>(m, blk, base + k, lane, bk);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const A b0 = bk[5 * i], b1 = bk[5 * i + 1];
            const A b2 = bk[5 * i + 2], b3 = bk[5 * i + 3], b4 = bk[5 * i + 4];
            acc[i] -= b0 * d[0];
            acc[i] -= b1 * d[1];
            const A dd = b2 * d[2] + b3 * d[3] + b4 * d[4];
            acc[i] -= dd;
        }
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) r[(size_t)i * nC + c] = acc[i];
}

// Backward sweep of one level: r[c] = rD[c] (r[c] - sum over upper
// neighbours q (decreasing q) of U_cq r[q]), r[q] already final.
template <typename TB, typename TV, bool GEN>
__device__ __forceinline__ void lusgsBwdRow(const MeshView& m, const TB* __restrict__ blk,
                                            const double* __restrict__ rD, TV* __restrict__ r, int c) {
    const size_t nC = m.nC;
    typedef TV A;
    A acc[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) acc[i] = r[(size_t)i * nC + c];
    const int sl = c >> 6, lane = c & 63;
    const size_t base = (size_t)m.slicePtr[sl];
    const int nl = m.nLower[c], len = m.rowLen[c];
    for (int k = len - 1; k >= nl; --k) {
        const size_t slot = (base + k) * 64 + lane;
        const int q = m.col[slot];
        A d[5];
#pragma unroll
        for (int z = 0; z < 5; ++z) d[z] = r[(size_t)z * nC + q];
        A bk[NB];
        slotBlock<TB, A, GEN>(m, blk, base + k, lane, bk);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const A b0 = bk[5 * i], b1 = bk[5 * i + 1];
            const A b2 = bk[5 * i + 2], b3 = bk[5 * i + 3], b4 = bk[5 * i + 4];
            acc[i] -= b0 * d[0];
            acc[i] -= b1 * d[1];
            const A dd = b2 * d[2] + b3 * d[3] + b4 * d[4];
            acc[i] -= dd;
        }
    }
    const A rd = (A)rD[c];
#pragma unroll
    for (int i = 0; i < 5; ++i) r[(size_t)i * nC + c] = rd * acc[i];
}

template <typename TB, typename TV, bool GEN, int W = 1>
__global__ void __launch_bounds__(256, W) k_lusgs_fwd(MeshView m, const TB* __restrict__ blk,
                                                   const double* __restrict__ rD, TV* __restrict__ r,
                                                   const int* __restrict__ cells, int n) {
    const int t = xcdBlock() * blockDim.x + threadIdx.x;
    if (t >= n) return;
    lusgsFwdRow<TB, TV, GEN>(m, blk, rD, r, cells[t]);
}

template <typename TB, typename TV, bool GEN, int W = 1>
__global__ void __launch_bounds__(256, W) k_lusgs_bwd(MeshView m, const TB* __restrict__ blk,
                                                   const double* __restrict__ rD, TV* __restrict__ r,
                                                   const int* __restrict__ cells, int n) {
    const int t = xcdBlock() * blockDim.x + threadIdx.x;
    if (t >= n) return;
    lusgsBwdRow<TB, TV, GEN>(m, blk, rD, r, cells[t]);
}

// Harmonic balance: one launch per level for all instances (blockIdx.y =
// instance; the cross-instance blocks have no faces, so the sweeps are
// independent per instance and share the diagonal rD).
template <typename TB, typename TV, bool FWD, bool GEN>
__global__ void __launch_bounds__(256) k_lusgs_hb(MeshView m, HBBlocks hb, const double* __restrict__ rD,
                                                  TV* __restrict__ r, const int* __restrict__ cells, int n) {
    const int t = xcdBlock() * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int J = blockIdx.y;
    TV* rJ = r + (size_t)J * 5 * m.nC;
    if (FWD) lusgsFwdRow<TB, TV, GEN>(m, (const TB*)hb.blk[J], rD, rJ, cells[t]);
    else lusgsBwdRow<TB, TV, GEN>(m, (const TB*)hb.blk[J], rD, rJ, cells[t]);
}

// LU-SGS of a numbering with many dependency levels (RCM or file order: a
// hundred and more each way) in one launch.  A launch per level costs 5 to 7
// us whatever the level holds; here a level costs one store-to-load round
// trip between wavefronts, about 2 us.  The cells of a level form chunks of
// one wavefront; the wavefronts draw the chunks in level order, forward
// levels first, from one counter, and wait for the values their rows read:
//   - forward results f and final results o start as a sentinel (a signalling
//     NaN pattern, which arithmetic does not return), are stored once with
//     agent-scope relaxed atomics and read with the same until they differ
//     from it: each value is its own flag, so nothing depends on the order in
//     which different values become visible;
//   - before that, a wavefront waits on the finished-chunk count of the level
//     two before its own, one load at a time, so that wavefronts far from the
//     front do not load the rows' values over and over.  The counts only pace
//     the loads.
// A row reads only rows of earlier levels, i.e. of lower chunks.  A chunk is
// drawn by a running wavefront, which finishes the chunks it drew in order,
// so the lowest unfinished chunk always runs, however few of the wavefronts
// the GPU has room for.  Each wait counts the polls that found it incomplete
// and gives up past `limit` of them (kSweepPolls: seconds, while a wait is
// for at most the grid's chunks ahead of it, milliseconds, however many
// levels the sweep has); the wavefront then sets ERR_FLAG_SWEEP and ends, and
// so does every wavefront that waits for its chunk.
// Same operations and order per row as lusgsFwdRow / lusgsBwdRow.

__device__ __forceinline__ unsigned long long sweepSentinel(double) { return 0x7FF4DEADBEEF5A5Aull; }
__device__ __forceinline__ unsigned sweepSentinel(float) { return 0x7FA5A5A5u; }
__device__ __forceinline__ unsigned long long sweepBits(double v) { return __double_as_longlong(v); }
__device__ __forceinline__ unsigned sweepBits(float v) { return __float_as_uint(v); }
template <typename TV>
__device__ __forceinline__ TV sweepLoad(const TV* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename TV>
__device__ __forceinline__ void sweepStore(TV* p, TV v) {
    if (sweepBits(v) == sweepSentinel(v)) v = (TV)__builtin_nan("");
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// done: the finished chunks of each level, then the next chunk to draw
template <typename TV>
__global__ void k_sweep_init(size_t n, int nLev, TV* __restrict__ f, TV* __restrict__ o, int* __restrict__ done) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    TV v;
    const auto s = sweepSentinel((TV)0);
    __builtin_memcpy(&v, &s, sizeof(TV));
    if (i < n) f[i] = o[i] = v;
    if (i <= (size_t)nLev) done[i] = 0;
}

template <typename TB, typename TV, bool GEN>
__global__ void __launch_bounds__(64) k_sweep(MeshView m, const TB* __restrict__ blk, const double* __restrict__ rD,
                                               TV* r, TV* f, TV* o, const int* __restrict__ chunkCells,
                                               const int* __restrict__ chunkLevel,
                                               const int* __restrict__ levelChunks, int nFwd, int nChunks,
                                               int nFwdLevels, int limit, int* done, int* next, int* err) {
    constexpr int UN = 3;  // slots whose blocks and values are in flight together
    typedef TV A;
    const size_t nC = m.nC;
    const int lane = threadIdx.x & 63;
    const auto sent = sweepSentinel((TV)0);
    // the values at q (5 of them nC apart) of every lane with on set
    auto wait5 = [&](const TV* q, bool on, A (&v)[5]) {
        bool ready = !on;
        for (int polls = 0;;) {
            if (!ready) {
                ready = true;
#pragma unroll
                for (int z = 0; z < 5; ++z) {
                    const TV x = sweepLoad(q + (size_t)z * nC);
                    v[z] = (A)x;
                    ready = ready && sweepBits(x) != sent;
                }
            }
            if (__all(ready)) return true;
            if (++polls > limit) return false;
        }
    };
    auto draw = [&]() {
        int i = 0;
        if (lane == 0) i = __hip_atomic_fetch_add(next, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return __builtin_amdgcn_readfirstlane(i);
    };
    for (int ch = draw(); ch < nChunks; ch = draw()) {
        const bool bwd = ch >= nFwd;
        const int lev = chunkLevel[ch];                        // within its sweep
        const int lg = bwd ? nFwdLevels + lev : lev;           // over both
        const int c = chunkCells[(size_t)ch * 64 + lane];
        const bool on = c >= 0;
        const int cc = on ? c : 0;
        const int sl = cc >> 6, ln = cc & 63;
        const size_t base = (size_t)m.slicePtr[sl];
        const int nl = m.nLower[cc], len = m.rowLen[cc];
        const int n = on ? (bwd ? len - nl : nl) : 0;
        const A rdc = (A)rD[cc];
        bool ok = true, begun = false;
        A acc[5];
        // the pacing wait, then the row's own value (forward: r; backward: f)
        auto begin = [&]() {
            begun = true;
            if (lev >= 2) {
                const int want = levelChunks[lg - 2];
                int polls = 0;
                while (__builtin_amdgcn_readfirstlane(
                           __hip_atomic_load(done + lg - 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) < want) {
                    if (++polls > limit) { ok = false; return; }
                    __builtin_amdgcn_s_sleep(8);
                }
            }
            if (bwd) ok = wait5(f + cc, on, acc);
            else
#pragma unroll
                for (int q = 0; q < 5; ++q) acc[q] = (A)r[(size_t)q * nC + cc];
        };
        const TV* src = bwd ? o : f;
        for (int k = 0; ok && __any(k < n); k += UN) {
            // forward: lower slots upwards; backward: upper slots downwards.
            // The blocks are formed before the wait (the empty asm keeps
            // them from being moved behind it): after it a slot costs its
            // product only
            constexpr int NE = GEN ? NGEN : NB;
            TB b[UN][NB];
            A rd[UN];
            int p[UN];
            A d[UN][5];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const bool has = k + u < n;
                const size_t sk = base + (has ? (bwd ? len - 1 - (k + u) : k + u) : 0);
                p[u] = has ? m.col[sk * 64 + ln] : cc;
                rd[u] = bwd ? (A)1 : (A)rD[p[u]];
                TB g[NE];
#pragma unroll
                for (int e = 0; e < NE; ++e) g[e] = has ? blk[(sk * NE + e) * 64 + ln] : (TB)0;
                const TB mo = GEN && m.genMo && has ? ((const TB*)m.genMo)[sk * 64 + ln] : (TB)0;
                if constexpr (GEN) blockFromGen<TB>(g, (TB)m.gamma, b[u], mo, m.genMo != nullptr);
                else
#pragma unroll
                    for (int e = 0; e < NB; ++e) b[u][e] = g[e];
#pragma unroll
                for (int e = 0; e < NB; ++e) asm volatile("" : "+v"(b[u][e]));
            }
            if (!begun) begin();
            // the slots' values, those not there yet loaded again
            unsigned miss = 0;
#pragma unroll
            for (int u = 0; u < UN; ++u) miss |= ok && k + u < n ? 1u << u : 0u;
            for (int polls = 0; ok;) {
#pragma unroll
                for (int u = 0; u < UN; ++u)
                    if (miss & (1u << u)) {
                        bool got = true;
#pragma unroll
                        for (int z = 0; z < 5; ++z) {
                            const TV x = sweepLoad(src + (size_t)z * nC + p[u]);
                            d[u][z] = (A)x;
                            got = got && sweepBits(x) != sent;
                        }
                        if (got) miss &= ~(1u << u);
                    }
                if (!__any(miss)) break;
                ok = ++polls <= limit;
            }
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                if (k + u >= n) continue;
                if (!bwd)
#pragma unroll
                    for (int z = 0; z < 5; ++z) d[u][z] = rd[u] * d[u][z];
#pragma unroll
                for (int i = 0; i < 5; ++i) {
                    const A b0 = (A)b[u][5 * i], b1 = (A)b[u][5 * i + 1];
                    const A b2 = (A)b[u][5 * i + 2], b3 = (A)b[u][5 * i + 3], b4 = (A)b[u][5 * i + 4];
                    acc[i] -= b0 * d[u][0];
                    acc[i] -= b1 * d[u][1];
                    const A dd = b2 * d[u][2] + b3 * d[u][3] + b4 * d[u][4];
                    acc[i] -= dd;
                }
            }
        }
        if (!begun) begin();
        if (!ok) {
            if (lane == 0) atomicOr(err, ERR_FLAG_SWEEP);
            return;
        }
        if (on)
#pragma unroll
            for (int q = 0; q < 5; ++q) {
                const A v = bwd ? rdc * acc[q] : acc[q];
                sweepStore((bwd ? o : f) + (size_t)q * nC + c, (TV)v);
                // r[c] was read by the forward chunk whose f[c] this wave has
                if (bwd) r[(size_t)q * nC + c] = (TV)v;
            }
        if (lane == 0) __hip_atomic_fetch_add(done + lg, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ------------------------------------------------------- block-Jacobi -----
// 5x5 inverse of each diagonal block by LU with partial pivoting.
template <typename TB>
__global__ void k_jacobi_setup(int nC, const TB* __restrict__ dg, TB* __restrict__ dinv) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nC) return;
    double a[5][5];
    int piv[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        piv[i] = i;
#pragma unroll
        for (int j = 0; j < 5; ++j) a[i][j] = (double)dg[diagOff(c, 5 * i + j)];
    }
    for (int col = 0; col < 5; ++col) {
        int p = col;
        for (int r = col + 1; r < 5; ++r)
            if (fabs(a[r][col]) > fabs(a[p][col])) p = r;
        if (p != col) {
            for (int q = 0; q < 5; ++q) { double t = a[p][q]; a[p][q] = a[col][q]; a[col][q] = t; }
            int t = piv[p]; piv[p] = piv[col]; piv[col] = t;
        }
        for (int r = col + 1; r < 5; ++r) {
            a[r][col] /= a[col][col];
            for (int q = col + 1; q < 5; ++q) a[r][q] -= a[r][col] * a[col][q];
        }
    }
    for (int e = 0; e < 5; ++e) {
        double yv[5];
        for (int i = 0; i < 5; ++i) {
            double s = piv[i] == e ? 1.0 : 0.0;
            for (int q = 0; q < i; ++q) s -= a[i][q] * yv[q];
            yv[i] = s;
        }
        for (int i = 4; i >= 0; --i) {
            double s = yv[i];
            for (int q = i + 1; q < 5; ++q) s -= a[i][q] * yv[q];
            yv[i] = s / a[i][i];
        }
        for (int i = 0; i < 5; ++i) dinv[diagOff(c, 5 * i + e)] = (TB)yv[i];
    }
}

template <typename TB, typename TV>
__global__ void k_jacobi_apply(int nC, const TB* __restrict__ dinv, TV* __restrict__ r) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nC) return;
    typedef TV A;
    A v[5], o[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) { v[i] = r[(size_t)i * nC + c]; o[i] = 0; }
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int j = 0; j < 5; ++j) o[i] += (A)dinv[diagOff(c, 5 * i + j)] * v[j];
#pragma unroll
    for (int i = 0; i < 5; ++i) r[(size_t)i * nC + c] = o[i];
}

// Block-level sum of NV values per thread -> out[blockIdx.x*NV + k].
template <int NV>
__device__ __forceinline__ void blockReduceStore(double (&v)[NV], double* out) {
    __shared__ double sh[4][NV > 0 ? NV : 1];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double s = waveSum(v[k]);
        if (lane == 0) sh[wv][k] = s;
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        const int k = threadIdx.x;
        out[(size_t)blockIdx.x * NV + k] = ((sh[0][k] + sh[1][k]) + sh[2][k]) + sh[3][k];
    }
}

// Sum of value k over nb partial rows of `stride` values, in a fixed order
// (thread t adds rows t, t+256, ...; then the wave sums; then the four
// waves in order).  Called by all threads of a 256-thread block; every
// thread gets the sum.
__device__ __forceinline__ double sumPartials(const double* __restrict__ part, int nb, int stride, int k) {
    __shared__ double sh[4];
    double v = 0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) v += part[(size_t)b * stride + k];
    v = waveSum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    const double s = ((sh[0] + sh[1]) + sh[2]) + sh[3];
    __syncthreads();
    return s;
}

// Sum of value k over nb partial rows of `stride` values by one wavefront, in
// a fixed order (lane t adds rows t, t+64, ...; then the lanes).
__device__ __forceinline__ double waveSumPartials(const double* __restrict__ part, int nb, int stride, int k) {
    double v = 0;
    for (int b = threadIdx.x & 63; b < nb; b += 64) v += part[(size_t)b * stride + k];
    return waveSum(v);
}

// Final reduction of an instance's [nb][nv] partials (instance blockIdx.y):
// value k = blockIdx.x (grid nv, 256 threads); out[8 instance + k].
__global__ void __launch_bounds__(256) k_reduce_final(const double* __restrict__ part, int nb, int nv,
                                                      double* __restrict__ out) {
    const int k = blockIdx.x;
    const double s = sumPartials(part + (size_t)blockIdx.y * nb * 8, nb, nv, k);
    if (threadIdx.x == 0) out[8 * blockIdx.y + k] = s;
}

// The reductions of a solve's start and end run over blockIdx.y = instance of
// a harmonic-balance system (vectors [nO][5][nC]; one otherwise), partials
// [instance][block][value] with 8 rows' room per block.

// sums of the 5 components of x (for the average) -> partials
template <typename TV>
__global__ void __launch_bounds__(256) k_sum5(int nC, const TV* __restrict__ x, double* __restrict__ part) {
    x += (size_t)blockIdx.y * 5 * nC;
    part += (size_t)blockIdx.y * gridDim.x * 8;
    double v[5] = {0, 0, 0, 0, 0};
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nC; c += gridDim.x * blockDim.x)
#pragma unroll
        for (int k = 0; k < 5; ++k) v[k] += (double)x[(size_t)k * nC + c];
    blockReduceStore<5>(v, part);
}

// norm-factor partials (gmres.C:839-850):
// [0..1] sum |t_s|+|b_s|, [2] sum |t_v|+|b_v|, [3..4] sum |b_s|, [5..7] sum |b_v,d|
template <typename TV>
__global__ void __launch_bounds__(256) k_normfactor(int nC, const TV* __restrict__ t, const TV* __restrict__ b,
                                                    double* __restrict__ part) {
    t += (size_t)blockIdx.y * 5 * nC;
    b += (size_t)blockIdx.y * 5 * nC;
    part += (size_t)blockIdx.y * gridDim.x * 8;
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nC; c += gridDim.x * blockDim.x) {
        double tv[5], bv[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) { tv[k] = (double)t[(size_t)k * nC + c]; bv[k] = (double)b[(size_t)k * nC + c]; }
        v[0] += fabs(tv[0]) + fabs(bv[0]);
        v[1] += fabs(tv[1]) + fabs(bv[1]);
        v[2] += sqrt(tv[2] * tv[2] + tv[3] * tv[3] + tv[4] * tv[4]) + sqrt(bv[2] * bv[2] + bv[3] * bv[3] + bv[4] * bv[4]);
        v[3] += fabs(bv[0]);
        v[4] += fabs(bv[1]);
        v[5] += fabs(bv[2]);
        v[6] += fabs(bv[3]);
        v[7] += fabs(bv[4]);
    }
    blockReduceStore<8>(v, part);
}

// final residual partials of r = b - A dW: [0..4] sum |r_k|
template <typename TV>
__global__ void __launch_bounds__(256) k_resid_l1(int nC, const TV* __restrict__ b, TV* __restrict__ Ax,
                                                  double* __restrict__ part) {
    b += (size_t)blockIdx.y * 5 * nC;
    Ax += (size_t)blockIdx.y * 5 * nC;
    part += (size_t)blockIdx.y * gridDim.x * 8;
    double v[5] = {0, 0, 0, 0, 0};
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nC; c += gridDim.x * blockDim.x)
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const TV r = b[(size_t)k * nC + c] - Ax[(size_t)k * nC + c];
            Ax[(size_t)k * nC + c] = r;
            v[k] += fabs((double)r);
        }
    blockReduceStore<5>(v, part);
}

template <typename TV>
__global__ void __launch_bounds__(256) k_norm2(int nC, const TV* __restrict__ x, double* __restrict__ part) {
    double v[1] = {0};
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nC; c += gridDim.x * blockDim.x)
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const double q = (double)x[(size_t)k * nC + c];
            v[0] += q * q;
        }
    blockReduceStore<1>(v, part);
}

// Projection partials of one Arnoldi step: <w, V_j> for j < nv = i + 1, and
// with WY (modified Gram-Schmidt) <v_i, V_k> for k < i from the same loads,
// blockIdx.y = a chunk of CH basis vectors.  Value q's partials are
// contiguous (part + q * gridDim.x): projections q = j, Gram values
// q = KMAX + k.  The basis vectors are streamed with non-temporal loads here
// and in the update and combine kernels: each is read once per pass and the
// passes between two reads of one vector move far more than L2 holds.
template <typename TV, int CH, bool WY>
__global__ void __launch_bounds__(256) k_project(int nC, const TV* __restrict__ w, const TV* __restrict__ Vb,
                                                 size_t vstride, int nv, double* __restrict__ part) {
    constexpr int NA = WY ? 2 * CH : CH;
    const int j0 = blockIdx.y * CH;
    const TV* vi = Vb + (size_t)(nv - 1) * vstride;
    double v[NA];
#pragma unroll
    for (int k = 0; k < NA; ++k) v[k] = 0;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nC; c += gridDim.x * blockDim.x) {
        TV wv[5], vv[5];
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            wv[q] = w[(size_t)q * nC + c];
            if (WY) vv[q] = vi[(size_t)q * nC + c];
        }
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            if (j0 + k < nv) {
                const TV* vj = Vb + (size_t)(j0 + k) * vstride;
                double s = 0, g = 0;
#pragma unroll
                for (int q = 0; q < 5; ++q) {
                    const TV x = __builtin_nontemporal_load(vj + (size_t)q * nC + c);
                    s += (double)(wv[q] * x);
                    if (WY) g += (double)(vv[q] * x);
                }
                v[k] += s;
                if (WY) v[CH + k] += g;
            }
        }
    }
    __shared__ double sh[4][NA];
    int id;
    const double t = waveSums<NA>(v, threadIdx.x & 63, id);
    sh[threadIdx.x >> 6][id] = t;  // every lane of a value stores the same
    __syncthreads();
    if (threadIdx.x < NA) {
        const int k = threadIdx.x, j = j0 + (k < CH ? k : k - CH);
        if (j < nv)
            part[(size_t)(k < CH ? j : KMAX + j) * gridDim.x + blockIdx.x] =
                ((sh[0][k] + sh[1][k]) + sh[2][k]) + sh[3][k];
    }
}

// All projections of one Arnoldi step, ch (8, 16 or 32) basis vectors per
// workgroup.
template <typename TV, bool WY>
void launchProject(int ch, int nbk, int nC, const TV* w, const TV* V, size_t vs, int nv, double* part,
                   hipStream_t st) {
    const dim3 g(nbk, (nv + ch - 1) / ch);
    if (ch == 8) k_project<TV, 8, WY><<<g, 256, 0, st>>>(nC, w, V, vs, nv, part);
    else if (ch == 32) k_project<TV, 32, WY><<<g, 256, 0, st>>>(nC, w, V, vs, nv, part);
    else k_project<TV, 16, WY><<<g, 256, 0, st>>>(nC, w, V, vs, nv, part);
}

// x = y - avg (component-wise), instance blockIdx.y.  The sums are those of
// k_reduce_final, or (part, nb partial rows) are formed here by every block.
template <typename TV>
__global__ void __launch_bounds__(256) k_sub_avg(int nC, const TV* __restrict__ W, const double* __restrict__ sums,
                                                 const double* __restrict__ part, int nb, TV* __restrict__ out) {
    __shared__ double sh[5];
    if (part) {
        for (int k = threadIdx.x >> 6; k < 5; k += 4) {
            const double a = waveSumPartials(part + (size_t)blockIdx.y * nb * 8, nb, 5, k);
            if ((threadIdx.x & 63) == 0) sh[k] = a;
        }
    } else if (threadIdx.x < 5) sh[threadIdx.x] = sums[8 * blockIdx.y + threadIdx.x];
    __syncthreads();
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nC) return;
    W += (size_t)blockIdx.y * 5 * nC;
    out += (size_t)blockIdx.y * 5 * nC;
#pragma unroll
    for (int k = 0; k < 5; ++k) out[(size_t)k * nC + c] = W[(size_t)k * nC + c] - (TV)(sh[k] / nC);
}

// a GMRES solve's start: r = b, dW = 0
__global__ void __launch_bounds__(256) k_start(size_t n, const double* __restrict__ b, double* __restrict__ r,
                                               double* __restrict__ dW) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    r[i] = b[i];
    dW[i] = 0.0;
}

template <typename TV>
__global__ void k_copy(size_t n, const TV* __restrict__ a, TV* __restrict__ b) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = a[i];
}

template <typename TA, typename TB2>
__global__ void k_convert(size_t n, const TA* __restrict__ a, TB2* __restrict__ b) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (TB2)a[i];
}

// dW += sum_i y_i V_i (gmres.C:1050-1059), sequential in i per entry
template <typename TV, typename TX>
__global__ void __launch_bounds__(256) k_update_sol(int nC, TX* __restrict__ dW, const TV* __restrict__ Vb,
                                                    size_t vstride, int nv, const double* __restrict__ yh) {
    const size_t n = (size_t)5 * nC;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    TX a = dW[i];
    // four basis vectors' loads in flight, added in order j = 0..nv-1
    int j = 0;
    for (; j + 4 <= nv; j += 4) {
        TV x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = __builtin_nontemporal_load(Vb + (size_t)(j + u) * vstride + i);
#pragma unroll
        for (int u = 0; u < 4; ++u) a += (TX)yh[j + u] * (TX)x[u];
    }
    for (; j < nv; ++j) a += (TX)yh[j] * (TX)Vb[(size_t)j * vstride + i];
    dW[i] = a;
}

}  // namespace

// ------------------------------------------------------------ GMRES state --
// Scalars of one GMRES(m) cycle kept on the device (no host round trips).
struct GmresScalars {
    double H[KMAX][KMAX];   // projections of column i: H[j][i], j <= i
    double hn[KMAX + 1];    // ||r|| of the cycle's start, then ||w_i|| after the orthogonalisation
    double T[KMAX][KMAX];   // modified Gram-Schmidt: unit lower triangular, (I + L)^-1 (orthCoeffs)
    double s[2 * KMAX];     // reduced projections (and Gram values) of the current step
    double yh[KMAX];
    double beta;
    double sNF[2], vNF;
    double res[10];   // sInit[2] vInit[3] sFinal[2] vFinal[3]
    double red[8 * HB_MAXO];  // component sums of the state, 8 per instance
};

namespace {

__device__ void givensRot(double h, double beta, double& c, double& s) {
    if (beta == 0) { c = 1; s = 0; }
    else if (fabs(beta) > fabs(h)) {
        const double tau = -h / beta;
        s = 1.0 / sqrt(1.0 + tau * tau);
        c = s * tau;
    } else {
        const double tau = -beta / h;
        c = 1.0 / sqrt(1.0 + tau * tau);
        s = c * tau;
    }
}

// Norm factors and initial residuals from the k_normfactor partials, one
// block per instance, one wavefront per value (512 threads).
__global__ void __launch_bounds__(512) k_gm_init(GmresPtrs gp, const double* __restrict__ part, int nb) {
    GmresScalars* g = gp.g[blockIdx.x];
    __shared__ double r[8];
    const int k = threadIdx.x >> 6;
    const double a = waveSumPartials(part + (size_t)blockIdx.x * nb * 8, nb, 8, k);
    if ((threadIdx.x & 63) == 0) r[k] = a;
    __syncthreads();
    if (threadIdx.x != 0) return;
    g->sNF[0] = r[0] + kVSMALL;
    g->sNF[1] = r[1] + kVSMALL;
    g->vNF = r[2] + kVSMALL;
    g->res[0] = r[3] / g->sNF[0];
    g->res[1] = r[4] / g->sNF[1];
    for (int d = 0; d < 3; ++d) g->res[2 + d] = r[5 + d] / g->vNF;
    for (int q = 0; q < 5; ++q) g->res[5 + q] = g->res[q];
}

// beta = ||r|| (a cycle's start) or ||w_i|| from the norm's partials.
__global__ void __launch_bounds__(64) k_reduce_norm(NormIn n) {
    const double beta = waveNorm(n.part, n.nb);
    if (threadIdx.x == 0) *n.beta = *n.hn = beta;
}

// Sums of the projection partials, one block per value: projections
// (blockIdx.x < nv), then the Gram values.
__global__ void __launch_bounds__(256) k_reduce_proj(const double* __restrict__ part, int nb, GmresScalars* g,
                                                     int nv) {
    const int q = (int)blockIdx.x < nv ? (int)blockIdx.x : KMAX + (int)blockIdx.x - nv;
    const double s = sumPartials(part + (size_t)q * nb, nb, 1, 0);
    if (threadIdx.x == 0) g->s[q] = s;
}

// Coefficients h (LDS, KMAX) with which w loses its projections on v_0..v_i,
// from the reduced sums s_j = <w, V_j>; called by all threads of a block.
// Classical Gram-Schmidt: h = s.  Modified Gram-Schmidt subtracts h_j v_j one
// after the other, h_j = <w - sum_{k<j} h_k v_k, v_j>, which is the forward
// substitution (I + L) h = s with L_jk = <v_j, v_k>, k < j (the inverse
// compact WY form of the product of the projectors): one pass over the
// basis instead of i + 1, and one reduction.  T = (I + L)^-1 of the earlier
// rows is kept, so the substitution is a product without a serial chain;
// row i of T follows from L_i, the Gram values that came with s.  Block 0
// stores column i of H and row i of T.
// part (few workgroups): the projection partials, nb <= 64 per value, summed
// here by every block instead of by a launch of its own.
template <bool WY>
__device__ void orthCoeffs(GmresScalars* g, int i, double* h, const double* __restrict__ part, int nb) {
    __shared__ double s[KMAX], l[KMAX];
    const int t = threadIdx.x;
    if (part) {
        const int lane = t & 63;
        for (int q0 = 16 * (t >> 6); q0 < (WY ? KMAX + i : i + 1); q0 += 64) {
            double v[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int q = q0 + k;
                const bool has = lane < nb && (q < KMAX ? q <= i : q < KMAX + i);
                v[k] = has ? part[(size_t)q * nb + lane] : 0.0;
            }
            int id;
            const double a = waveSums<16>(v, lane, id);
            if (q0 < KMAX) s[q0 + id] = a;
            else l[q0 - KMAX + id] = a;
        }
    } else {
        if (t <= i) s[t] = g->s[t];
        if (WY && t < i) l[t] = g->s[KMAX + t];
    }
    __syncthreads();
    if (WY) {
        double a = 0;
        if (t < i)
            for (int k = 0; k <= t; ++k) a += g->T[t][k] * s[k];
        if (t < i) h[t] = a;
        __syncthreads();
        if (t == i) {
            a = s[i];
            for (int k = 0; k < i; ++k) a -= l[k] * h[k];
            h[i] = a;
        }
        if (blockIdx.x == 0 && t <= i) {
            double r = t == i ? 1.0 : 0.0;
            for (int k = t; k < i; ++k) r -= l[k] * g->T[k][t];
            g->T[i][t] = r;
        }
    } else if (t <= i) h[t] = s[t];
    __syncthreads();
    if (blockIdx.x == 0 && t <= i) g->H[t][i] = h[t];
}

// w -= sum_j h_j V_j (j <= i), then ||w||^2 partials.  A thread takes single
// entries, 16 basis vectors' loads in flight, added in order j = 0..i
// (104x96x96 FP32, 16 vectors on average: 58 us with four vectors of five
// entries in flight -> 55 us).
template <typename TV, bool WY>
__global__ void __launch_bounds__(1024) k_orth_update(size_t n, TV* __restrict__ w, const TV* __restrict__ Vb,
                                                     GmresScalars* g, int i, const double* __restrict__ proj, int nb,
                                                     double* __restrict__ part) {
    __shared__ double h[KMAX];
    orthCoeffs<WY>(g, i, h, proj, nb);
    const int nv = i + 1;
    double v = 0;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
        TV a = w[e];
        const TV* q = Vb + e;
        int j = 0;
        for (; j + 16 <= nv; j += 16, q += 16 * n) {
            TV x[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) x[u] = __builtin_nontemporal_load(q + u * n);
#pragma unroll
            for (int u = 0; u < 16; ++u) a -= (TV)h[j + u] * x[u];
        }
        if (j < nv) {
            TV x[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) x[u] = j + u < nv ? __builtin_nontemporal_load(q + u * n) : (TV)0;
#pragma unroll
            for (int u = 0; u < 16; ++u)
                if (j + u < nv) a -= (TV)h[j + u] * x[u];
        }
        w[e] = a;
        v += (double)a * (double)a;
    }
    __shared__ double sh[16];
    v = waveSum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = sh[0];
        for (int k = 1; k < (int)(blockDim.x >> 6); ++k) t += sh[k];
        part[blockIdx.x] = t;
    }
}

// End of a cycle (one wavefront, lane = column): the Givens rotations of the
// n columns of H with sub-diagonal hn (gmres.C:999-1027) and the back
// substitution into yh.  Step k's rotation is formed by lane k and applied
// to all later columns at once, from LDS: 30 directions take 30 short steps
// instead of the 435 dependent column updates of one thread.
// part: the last norm's partials (null: hn[n] is there).
__global__ void __launch_bounds__(64) k_gm_finish(GmresScalars* g, int n, const double* __restrict__ part, int nb) {
    __shared__ double Hs[KMAX + 1][KMAX];
    __shared__ double bh[KMAX + 1], rot[2];
    const int t = threadIdx.x;
    if (t < n) {
        for (int j = 0; j <= t; ++j) Hs[j][t] = g->H[j][t];
        Hs[t + 1][t] = g->hn[t + 1];
        bh[t + 1] = 0;
    }
    if (t == 0) bh[0] = g->hn[0];
    __syncthreads();
    if (part) {
        const double beta = waveNorm(part, nb);
        if (t == 0) Hs[n][n - 1] = beta;
        __syncthreads();
    }
    for (int k = 0; k < n; ++k) {
        if (t == k) {
            double c, s;
            const double beta = Hs[k + 1][k];
            givensRot(Hs[k][k], beta, c, s);
            Hs[k][k] = c * Hs[k][k] - s * beta;
            const double b0 = bh[k], b1 = bh[k + 1];
            bh[k] = c * b0 - s * b1;
            bh[k + 1] = s * b0 + c * b1;
            rot[0] = c;
            rot[1] = s;
        }
        __syncthreads();
        if (t > k && t < n) {
            const double a = Hs[k][t], b = Hs[k + 1][t];
            Hs[k][t] = rot[0] * a - rot[1] * b;
            Hs[k + 1][t] = rot[1] * a + rot[0] * b;
        }
        __syncthreads();
    }
    for (int i = n - 1; i >= 0; --i) {
        if (t == i) {
            double hd = Hs[i][i];
            hd = hd >= 0 ? hd + kVSMALL : hd - kVSMALL;
            rot[0] = bh[i] / hd;
            g->yh[i] = rot[0];
        }
        __syncthreads();
        if (t < i) bh[t] -= Hs[t][i] * rot[0];
        __syncthreads();
    }
}

__global__ void __launch_bounds__(320) k_gm_final(GmresPtrs gp, const double* __restrict__ part, int nb,
                                                  int emptyDir) {
    GmresScalars* g = gp.g[blockIdx.x];
    __shared__ double r[5];
    const int k = threadIdx.x >> 6;
    const double a = waveSumPartials(part + (size_t)blockIdx.x * nb * 8, nb, 5, k);
    if ((threadIdx.x & 63) == 0) r[k] = a;
    __syncthreads();
    if (threadIdx.x != 0) return;
    g->res[5] = r[0] / g->sNF[0];
    g->res[6] = r[1] / g->sNF[1];
    for (int d = 0; d < 3; ++d) g->res[7 + d] = (d == emptyDir) ? 0.0 : r[2 + d] / g->vNF;
}

}  // namespace

// --------------------------------------------------------------- host side --
static inline int nb(size_t n, int b) { return (int)((n + b - 1) / b); }

// The projection pass of one Arnoldi step against nv basis vectors, ch
// vectors per workgroup (autotuner timing).
void launchProjectionPasses(const MeshView& m, int vecFp32, int ch, int mgs, const void* w, const void* V, int nv,
                            double* part, hipStream_t st) {
    const int nC = m.nC, nbk = reduceBlocks(nC);
    const size_t vs = (size_t)5 * nC;
    if (vecFp32) {
        if (mgs) launchProject<float, true>(ch, nbk, nC, (const float*)w, (const float*)V, vs, nv, part, st);
        else launchProject<float, false>(ch, nbk, nC, (const float*)w, (const float*)V, vs, nv, part, st);
    } else {
        if (mgs) launchProject<double, true>(ch, nbk, nC, (const double*)w, (const double*)V, vs, nv, part, st);
        else launchProject<double, false>(ch, nbk, nC, (const double*)w, (const double*)V, vs, nv, part, st);
    }
}

int reduceBlocks(int nC) {
    int n = nb(nC, 256);
    return n < 1024 ? (n < 1 ? 1 : n) : 1024;
}

// Full off-diagonal blocks from generator storage (read-back of the
// assembled matrix; padding slots are left untouched).
template <typename TB>
__global__ void k_expand_blocks(MeshView m, const TB* __restrict__ gen, TB* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= m.nC) return;
    const int sl = c >> 6, lane = c & 63;
    const size_t base = (size_t)m.slicePtr[sl];
    for (int k = 0; k < m.rowLen[c]; ++k) {
        TB b[NB];
        slotBlock<TB, TB, true>(m, gen, base + k, lane, b);
#pragma unroll
        for (int e = 0; e < NB; ++e) out[((base + k) * NB + e) * 64 + lane] = b[e];
    }
}

void launchExpandBlocks(const MeshView& m, int fp32, const void* gen, void* out, hipStream_t st) {
    if (fp32) k_expand_blocks<float><<<nb(m.nC, 256), 256, 0, st>>>(m, (const float*)gen, (float*)out);
    else k_expand_blocks<double><<<nb(m.nC, 256), 256, 0, st>>>(m, (const double*)gen, (double*)out);
}

template <typename TB, typename TV>
void spmv(const MeshView& m, const void* blk, const void* dg, const void* x, const double* scal, void* vout, void* y,
          hipStream_t st) {
    const dim3 g(xcdGrid(m.nC, m.bsOp));
    const TB *B = (const TB*)blk, *G = (const TB*)dg;
    if (m.blkGen && m.occOp)
        k_spmv<TB, TV, true, 4><<<g, m.bsOp, 0, st>>>(m, B, G, (const TV*)x, scal, (TV*)vout, (TV*)y);
    else if (m.blkGen)
        k_spmv<TB, TV, true><<<g, m.bsOp, 0, st>>>(m, B, G, (const TV*)x, scal, (TV*)vout, (TV*)y);
    else
        k_spmv<TB, TV, false><<<g, m.bsOp, 0, st>>>(m, B, G, (const TV*)x, scal, (TV*)vout, (TV*)y);
}

void launchSpmv(const MeshView& m, int blkFp32, int vecFp32, const void* blk, const void* dg, const void* x,
                const double* scal, void* vout, void* y, hipStream_t st) {
    if (blkFp32 && vecFp32) spmv<float, float>(m, blk, dg, x, scal, vout, y, st);
    else if (blkFp32) spmv<float, double>(m, blk, dg, x, scal, vout, y, st);
    else if (vecFp32) spmv<double, float>(m, blk, dg, x, scal, vout, y, st);
    else spmv<double, double>(m, blk, dg, x, scal, vout, y, st);
}

// The three phases on a two-colour level structure.  Below kOpLatencyRows
// rows per launch (about one wavefront per SIMD) a launch lasts as long as
// one row's chain of dependent loads, and the loads of two slots (FP64) or six
// (FP32, a third of the registers) are issued together; above, more
// registers cost waves.  Pseudo-step, one slot / together: FP64 36^3 1.745 /
// 1.643 ms, 64^3 4.43 / 4.48 ms; mixed 48^3 1.90 / 1.74 ms, 64^3 3.08 /
// 3.12 ms.
constexpr size_t kOpLatencyRows = 65536;
// Cells (instances included) from which a norm is summed by a launch of its
// own (and the update takes its large form, updateBlocks).  Pseudo-step, own
// launch / merged: 125 000 cells FP64 2.79 / 2.66 ms, mixed 1.99 / 1.86 ms;
// 195 000 3.78 / 3.70, 2.70 / 2.58; 262 000 4.44 / 4.43, 2.97 / 2.95; 512 000
// 8.18 / 8.10, 4.98 / 4.97; 1 000 000 15.15 / 15.09, 8.86 / 8.80: the line lies
// where the gain has fallen to a percent, and above it the first phase grows
// by what the launch saves (gmresCycleT).
constexpr int kNormMergeCells = 200000;

template <typename TB, bool GEN, bool HB, int UN, int W>
static void opPhases(const MeshView& m, const Levels& L, const HBBlocks& hb, const void* blk, const void* dg,
                     const double* rD, const void* x, const double* scal, const NormIn& norm, void* vout, void* t,
                     void* y, int bs, hipStream_t st) {
    const int n0 = L.fwdPtrHost[1], n1 = L.fwdPtrHost[2] - n0;
    const int s0 = L.bwdPtrHost[1], nbw = L.bwdPtrHost[2] - s0;
    const int nO = HB ? hb.nO : 1;
    // colour-major numberings: the levels are cell ranges, no list
    const int *l0 = L.colourMajor ? nullptr : L.fwdCells, *l1 = L.colourMajor ? nullptr : L.fwdCells + n0;
    const int* l2 = L.colourMajor ? nullptr : L.bwdCells + s0;
    const TB *B = (const TB*)blk, *G = (const TB*)dg, *X = (const TB*)x;
    TB *V = (TB*)vout, *T = (TB*)t, *Y = (TB*)y;
    k_op<TB, GEN, 0, HB, UN, W><<<dim3(xcdGrid(n0, bs), nO), bs, 0, st>>>(m, hb, B, G, X, scal, V, T, Y, rD, l0, 0, n0, norm);
    k_op<TB, GEN, 1, HB, UN, W><<<dim3(xcdGrid(n1, bs), nO), bs, 0, st>>>(m, hb, B, G, X, scal, V, T, Y, rD, l1, n0, n1, norm);
    k_op<TB, GEN, 2, HB, UN, W><<<dim3(xcdGrid(nbw, bs), nO), bs, 0, st>>>(m, hb, B, G, X, scal, V, T, Y, rD, l2, 0, nbw, norm);
}

template <typename TB, bool HB>
static void opLaunch(const MeshView& m, const Levels& L, const HBBlocks& hb, const void* blk, const void* dg,
                     const double* rD, const void* x, const double* scal, const NormIn& norm, void* vout, void* t,
                     void* y, int bs, hipStream_t st) {
    const bool few = (size_t)L.fwdPtrHost[1] * (HB ? hb.nO : 1) <= kOpLatencyRows;
    if (!m.blkGen) opPhases<TB, false, HB, 1, 1>(m, L, hb, blk, dg, rD, x, scal, norm, vout, t, y, bs, st);
    else if (few) opPhases<TB, true, HB, sizeof(TB) == 4 ? 6 : 2, 1>(m, L, hb, blk, dg, rD, x, scal, norm, vout, t, y, bs, st);
    else {
        // register budgets: FP32 fits 8 waves per SIMD (64 VGPRs), FP64 4
        if constexpr (!HB)
            if (m.occOp)
                return opPhases<TB, true, HB, 1, sizeof(TB) == 4 ? 8 : 4>(m, L, hb, blk, dg, rD, x, scal, norm, vout,
                                                                         t, y, bs, st);
        opPhases<TB, true, HB, 1, 1>(m, L, hb, blk, dg, rD, x, scal, norm, vout, t, y, bs, st);
    }
}

bool launchSpmvLusgs(const MeshView& m, const Levels& L, int blkFp32, int vecFp32, const void* blk, const void* dg,
                     const double* rD, const void* x, const double* scal, const NormIn& norm, void* vout, void* t,
                     void* y, hipStream_t st) {
    if (!fusedOperator(L, blkFp32, vecFp32)) return false;
    const HBBlocks none{};
    if (vecFp32) opLaunch<float, false>(m, L, none, blk, dg, rD, x, scal, norm, vout, t, y, m.bsOp, st);
    else opLaunch<double, false>(m, L, none, blk, dg, rD, x, scal, norm, vout, t, y, m.bsOp, st);
    return true;
}

template <typename TB, typename TV, bool GEN, int W>
static void lusgsG(const MeshView& m, const Levels& L, const void* blk, const double* rD, void* r, hipStream_t st) {
    const int bs = m.bsOp;
    for (int l = 0; l < L.nFwd; ++l) {
        const int s0 = L.fwdPtrHost[l], n = L.fwdPtrHost[l + 1] - s0;
        if (L.fwdSkip && l == 0) continue;  // first level has no lower neighbours
        k_lusgs_fwd<TB, TV, GEN, W><<<xcdGrid(n, bs), bs, 0, st>>>(m, (const TB*)blk, rD, (TV*)r, L.fwdCells + s0,
                                                                   n);
    }
    for (int l = 0; l < L.nBwd; ++l) {
        const int s0 = L.bwdPtrHost[l], n = L.bwdPtrHost[l + 1] - s0;
        k_lusgs_bwd<TB, TV, GEN, W><<<xcdGrid(n, bs), bs, 0, st>>>(m, (const TB*)blk, rD, (TV*)r, L.bwdCells + s0,
                                                                   n);
    }
}

// The dataflow sweep, one wavefront per workgroup.  Per application, forward
// and backward: 48x24x24 in RCM order (82 levels each way) 1110 us as 164
// launches -> 540 us; 200x50x1 in file order (249 levels) 3200 -> 1010 us;
// 128x64x64 in RCM order (201 levels) 3200 -> 1850 us.  256 wavefronts: with 512
// the 72x64x56 and 128x64x64 boxes take 7 and 12 % longer (their loads
// queue behind each other's), smaller ones the same; chunks of 32 rows 10 to
// 25 % longer (more counts and draws).
constexpr int kSweepWaves = 256;
template <typename TB, typename TV, bool GEN>
static void sweepG(const MeshView& m, const Levels& L, const Work& wk, const void* blk, const double* rD, void* r,
                   hipStream_t st) {
    const int nCh = L.nFwdChunks + L.nBwdChunks, nLev = L.nFwd + L.nBwd;
    const size_t n = (size_t)5 * m.nC;
    k_sweep_init<TV><<<nb(n, 256), 256, 0, st>>>(n, nLev, (TV*)wk.swF, (TV*)wk.swO, wk.swDone);
    const int nWg = nCh < kSweepWaves ? nCh : kSweepWaves;
    k_sweep<TB, TV, GEN><<<nWg, 64, 0, st>>>(m, (const TB*)blk, rD, (TV*)r, (TV*)wk.swF, (TV*)wk.swO, L.chunkCells,
                                             L.chunkLevel, L.levelChunks, L.nFwdChunks, nCh, L.nFwd, wk.swLimit,
                                             wk.swDone, wk.swDone + nLev, wk.err);
}

template <typename TB, typename TV>
static void lusgsT(const MeshView& m, const Levels& L, const Work& wk, const void* blk, const double* rD, void* r,
                   hipStream_t st) {
    if (wk.swF && m.blkGen) sweepG<TB, TV, true>(m, L, wk, blk, rD, r, st);
    else if (wk.swF) sweepG<TB, TV, false>(m, L, wk, blk, rD, r, st);
    else if (m.blkGen && m.occOp) lusgsG<TB, TV, true, 4>(m, L, blk, rD, r, st);
    else if (m.blkGen) lusgsG<TB, TV, true, 1>(m, L, blk, rD, r, st);
    else lusgsG<TB, TV, false, 1>(m, L, blk, rD, r, st);
}

void launchLusgs(const MeshView& m, const Levels& L, const Work& wk, int blkFp32, int vecFp32, const void* blk,
                 const double* rD, void* r, hipStream_t st) {
    if (blkFp32 && vecFp32) lusgsT<float, float>(m, L, wk, blk, rD, r, st);
    else if (blkFp32) lusgsT<float, double>(m, L, wk, blk, rD, r, st);
    else if (vecFp32) lusgsT<double, float>(m, L, wk, blk, rD, r, st);
    else lusgsT<double, double>(m, L, wk, blk, rD, r, st);
}

void launchJacobiSetup(int nC, int blkFp32, const void* dg, void* dinv, hipStream_t st) {
    if (blkFp32) k_jacobi_setup<float><<<nb(nC, 256), 256, 0, st>>>(nC, (const float*)dg, (float*)dinv);
    else k_jacobi_setup<double><<<nb(nC, 256), 256, 0, st>>>(nC, (const double*)dg, (double*)dinv);
}

void launchJacobiApply(int nC, int blkFp32, int vecFp32, const void* dinv, void* r, hipStream_t st) {
    if (blkFp32 && vecFp32) k_jacobi_apply<float, float><<<nb(nC, 256), 256, 0, st>>>(nC, (const float*)dinv, (float*)r);
    else if (blkFp32) k_jacobi_apply<float, double><<<nb(nC, 256), 256, 0, st>>>(nC, (const float*)dinv, (double*)r);
    else if (vecFp32) k_jacobi_apply<double, float><<<nb(nC, 256), 256, 0, st>>>(nC, (const double*)dinv, (float*)r);
    else k_jacobi_apply<double, double><<<nb(nC, 256), 256, 0, st>>>(nC, (const double*)dinv, (double*)r);
}

// Workgroup size and workgroups of the update of 5 nC entries: at most 256
// where every workgroup of the operator's first phase sums their partials
// (53x42x39 FP64: 16 + 11 us, with up to 1024 of 256 threads 16 + 15), else up
// to 1024 small ones (104x96x96 FP32: 55 us against 60, 64^3 FP64 31 against 36).
static int updateThreads(int nC) { return nC < kNormMergeCells && (size_t)5 * nC > 65536 ? 1024 : 256; }
static int updateBlocks(int nC) {
    const int n = nb((size_t)5 * nC, updateThreads(nC)), most = nC < kNormMergeCells ? 256 : 1024;
    return n < most ? n : most;
}

// Orthogonalisation of w against v_0..v_i (V): projections, their reduction,
// the update with ||w||'s partials.  Three launches for both Gram-Schmidt
// forms, two with at most 64 workgroups (16 384 cells), whose update sums the
// projection partials itself; modified Gram-Schmidt step by step took
// 2 (i + 2) launches and 4 (i + 1) vector passes where this takes 2 i + 6
// (200x50x1 cells, GMRES(30): 990 of the cycle's 1110 launches).  The norm's
// partials are summed by whoever needs it next: the operator's first phase,
// the cycle's end, or k_reduce_norm.  Pseudo-steps with modified
// Gram-Schmidt, FP64: 200x50x1 3.83 -> 1.34 ms, 53x42x39 viscous 5.69 -> 2.86
// ms; classical, 64^3: 5.89 -> 5.39 ms (one projection launch for all chunks,
// the Givens chain once per cycle).
template <typename TV, bool WY>
static void orthStepT(const MeshView& m, int nC, TV* w, const TV* V, int i, GmresScalars* g, double* part,
                      hipStream_t st) {
    const int nbk = reduceBlocks(nC);
    const size_t vs = (size_t)5 * nC;
    const bool few = nbk <= 64;
    launchProject<TV, WY>(m.mdCh, nbk, nC, w, V, vs, i + 1, part, st);
    if (!few) k_reduce_proj<<<WY ? 2 * i + 1 : i + 1, 256, 0, st>>>(part, nbk, g, i + 1);
    k_orth_update<TV, WY><<<updateBlocks(nC), updateThreads(nC), 0, st>>>(vs, w, V, g, i, few ? part : nullptr, nbk,
                                                           part + kNormPart);
}
template <typename TV>
static void orthStep(const MeshView& m, int orth, int nC, TV* w, const TV* V, int i, GmresScalars* g, double* part,
                     hipStream_t st) {
    if (orth == 0) orthStepT<TV, true>(m, nC, w, V, i, g, part, st);
    else orthStepT<TV, false>(m, nC, w, V, i, g, part, st);
}

// --------------------------------------------------------- GMRES driver --
template <typename TV>
void gmresCycleT(const GmresArgs& a, hipStream_t st) {
    const MeshView& m = *a.m;
    const int nC = a.nVec > 0 ? a.nVec : m.nC;
    const int nbk = reduceBlocks(nC);
    const size_t vs = (size_t)5 * nC;
    TV* r = (TV*)a.r;    // current w
    TV* r2 = (TV*)a.r2;  // SpMV output (ping-pong with r)
    TV* V = (TV*)a.V;
    GmresScalars* g = a.g;
    auto mark = [&](int k, int b) {
        if (a.mark) a.mark(k, b);
    };
    auto precond = [&](TV* v) {
        mark(TK_PRECOND, 1);
        if (a.pre) a.pre(v);
        else if (a.precond == 0) launchLusgs(m, *a.lev, *a.wk, a.blkFp32, sizeof(TV) == 4, a.blk, a.rD, v, st);
        else if (a.precond == 1) launchJacobiApply(nC, a.blkFp32, sizeof(TV) == 4, a.dinv, v, st);
        mark(TK_PRECOND, 0);
    };
    // r <- P^-1 r; ||r||
    precond(r);
    double* pn = a.wk->part + kNormPart;
    k_norm2<TV><<<nbk, 256, 0, st>>>(nC, r, pn);
    // fused SpMV + LU-SGS on two-colour level structures (the colour-1
    // blocks are read once for both; the SPMV timing class then covers the
    // sweeps too), which sums the norm's partials as well; otherwise the
    // norm, the SpMV, then the preconditioner
    const bool fused = a.opPre || (!a.op && !a.pre && a.precond == 0 && a.fuse &&
                                   fusedOperator(*a.lev, a.blkFp32, sizeof(TV) == 4));
    for (int i = 0; i < a.nDirs; ++i) {
        TV* vi = V + (size_t)i * vs;
        // v_i = r / ||r|| ; w = A v_i (into the other buffer: the SpMV gathers
        // neighbour entries of its input, so it never runs in place)
        const NormIn all{pn, i == 0 ? nbk : updateBlocks(nC), &g->beta, &g->hn[i]};
        // many partials are summed once instead of by every block of the
        // operator's first phase (104x96x96, 1024 partials: 43 us against
        // 35 + 5; 53x42x39, 340: 11.9 against 11.1 + 4.7)
        const bool own = !fused || nC >= kNormMergeCells;
        if (own) k_reduce_norm<<<1, 64, 0, st>>>(all);
        NormIn norm = all;
        if (own) norm.part = nullptr;
        mark(TK_SPMV, 1);
        if (a.opPre) a.opPre(r, norm, vi, r2);
        else if (fused)
            launchSpmvLusgs(m, *a.lev, a.blkFp32, sizeof(TV) == 4, a.blk, a.dg, a.rD, r, &g->beta, norm, vi, a.t, r2,
                            st);
        else if (a.op) a.op(r, &g->beta, vi, r2);
        else launchSpmv(m, a.blkFp32, sizeof(TV) == 4, a.blk, a.dg, r, &g->beta, vi, r2, st);
        mark(TK_SPMV, 0);
        {
            TV* t = r;
            r = r2;
            r2 = t;
        }
        if (!fused) precond(r);
        mark(TK_ORTH, 1);
        orthStep<TV>(m, a.orth, nC, r, V, i, g, a.wk->part, st);
        mark(TK_ORTH, 0);
    }
    k_gm_finish<<<1, 64, 0, st>>>(g, a.nDirs, pn, updateBlocks(nC));
}

}  // namespace icsf

namespace icsf {

namespace {
template <typename TV>
__global__ void k_zero_comp(int nC, int comp, TV* x) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < nC) x[(size_t)comp * nC + c] = (TV)0;
}
}  // namespace

size_t gmresScalarsBytes() { return sizeof(GmresScalars); }

void gmresCycle(const GmresArgs& a, int vecFp32, hipStream_t st) {
    if (vecFp32) gmresCycleT<float>(a, st);
    else gmresCycleT<double>(a, st);
}

// Up to this many workgroups of partial sums (32 768 cells) the average is
// formed by k_sub_avg's blocks instead of by a launch of its own.
constexpr int kSubAvgMerge = 128;

template <typename TV>
static void subAverage(int nC, int nO, Work& wk, GmresScalars* g, const TV* W, TV* out, hipStream_t st) {
    const int nbk = reduceBlocks(nC);
    const bool merge = nbk <= kSubAvgMerge;
    k_sum5<TV><<<dim3(nbk, nO), 256, 0, st>>>(nC, W, wk.part);
    if (!merge) k_reduce_final<<<dim3(5, nO), 256, 0, st>>>(wk.part, nbk, 5, g->red);
    k_sub_avg<TV><<<dim3(nb(nC, 256), nO), 256, 0, st>>>(nC, W, g->red, merge ? wk.part : nullptr, nbk, out);
}

template <typename TV>
static void normFactors(int nC, int nO, Work& wk, const GmresPtrs& gp, const TV* t, const TV* b, hipStream_t st) {
    const int nbk = reduceBlocks(nC);
    k_normfactor<TV><<<dim3(nbk, nO), 256, 0, st>>>(nC, t, b, wk.part);
    k_gm_init<<<nO, 512, 0, st>>>(gp, wk.part, nbk);
}

template <typename TV>
static void finalResidual(int nC, int nO, int emptyDir, Work& wk, const GmresPtrs& gp, const TV* b, TV* r,
                          hipStream_t st) {
    const int nbk = reduceBlocks(nC);
    k_resid_l1<TV><<<dim3(nbk, nO), 256, 0, st>>>(nC, b, r, wk.part);
    k_gm_final<<<nO, 320, 0, st>>>(gp, wk.part, nbk, emptyDir);
}

template <typename TV>
static void prepareT(const MeshView& m, Work& wk, GmresScalars* g, const void* W, const void* b, void* tmp1,
                     void* tmp2, int blkFp32, const void* blk, const void* dg, hipStream_t st) {
    subAverage<TV>(m.nC, 1, wk, g, (const TV*)W, (TV*)tmp1, st);
    launchSpmv(m, blkFp32, sizeof(TV) == 4, blk, dg, tmp1, nullptr, nullptr, tmp2, st);
    normFactors<TV>(m.nC, 1, wk, GmresPtrs{{g}}, (const TV*)tmp2, (const TV*)b, st);
}

void gmresPrepare(const MeshView& m, Work& wk, GmresScalars* g, int vecFp32, const void* W, const void* b,
                  void* tmp1, void* tmp2, int blkFp32, const void* blk, const void* dg, hipStream_t st) {
    if (vecFp32) prepareT<float>(m, wk, g, W, b, tmp1, tmp2, blkFp32, blk, dg, st);
    else prepareT<double>(m, wk, g, W, b, tmp1, tmp2, blkFp32, blk, dg, st);
}

template <typename TV>
static void updResT(const MeshView& m, Work& wk, GmresScalars* g, int blkFp32, const void* blk, const void* dg,
                    int nDirs, const void* V, void* dW, const void* b, void* r, hipStream_t st) {
    const int nC = m.nC;
    const size_t vs = (size_t)5 * nC;
    k_update_sol<TV, TV><<<nb(vs, 256), 256, 0, st>>>(nC, (TV*)dW, (const TV*)V, vs, nDirs, g->yh);
    launchSpmv(m, blkFp32, sizeof(TV) == 4, blk, dg, dW, nullptr, nullptr, r, st);
    finalResidual<TV>(nC, 1, m.emptyDir, wk, GmresPtrs{{g}}, (const TV*)b, (TV*)r, st);
}

void gmresUpdateAndResidual(const MeshView& m, Work& wk, GmresScalars* g, int vecFp32, int blkFp32,
                            const void* blk, const void* dg, int nDirs, const void* V, void* dW, const void* b,
                            void* r, hipStream_t st) {
    if (vecFp32) updResT<float>(m, wk, g, blkFp32, blk, dg, nDirs, V, dW, b, r, st);
    else updResT<double>(m, wk, g, blkFp32, blk, dg, nDirs, V, dW, b, r, st);
}

void gmresReadResiduals(const GmresScalars* g, double* res10, hipStream_t st) {
    (void)hipMemcpyAsync(res10, g->res, sizeof(double) * 10, hipMemcpyDeviceToHost, st);
    (void)hipStreamSynchronize(st);
}

const double* gmresResidualsDevice(const GmresScalars* g) { return g->res; }

void launchCopy(size_t n, int fp32, const void* a, void* b, hipStream_t st) {
    if (fp32) k_copy<float><<<nb(n, 256), 256, 0, st>>>(n, (const float*)a, (float*)b);
    else k_copy<double><<<nb(n, 256), 256, 0, st>>>(n, (const double*)a, (double*)b);
}

void launchConvert(size_t n, int fromFp32, const void* a, void* b, hipStream_t st) {
    if (fromFp32) k_convert<float, double><<<nb(n, 256), 256, 0, st>>>(n, (const float*)a, (double*)b);
    else k_convert<double, float><<<nb(n, 256), 256, 0, st>>>(n, (const double*)a, (float*)b);
}

namespace {
template <typename T>
__global__ void k_zero(size_t n, T* x) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = (T)0;
}
}  // namespace

// Zero fill by a kernel (no memset nodes, so the sequence can be captured).
void launchZero(size_t n, int fp32, void* x, hipStream_t st) {
    if (fp32) k_zero<float><<<nb(n, 256), 256, 0, st>>>(n, (float*)x);
    else k_zero<double><<<nb(n, 256), 256, 0, st>>>(n, (double*)x);
}

void launchZeroComponent(int nC, int comp, int fp32, void* x, hipStream_t st) {
    if (fp32) k_zero_comp<float><<<nb(nC, 256), 256, 0, st>>>(nC, comp, (float*)x);
    else k_zero_comp<double><<<nb(nC, 256), 256, 0, st>>>(nC, comp, (double*)x);
}

}  // namespace icsf

// ------------------------------------------------- harmonic balance -----
namespace icsf {

template <typename TB, typename TV>
void spmvHBT(const MeshView& m, const HBBlocks& hb, const void* x, const double* scal, void* vout, void* y,
             hipStream_t st) {
    dim3 grid(xcdGrid(m.nC, 256), hb.nO);
    if (m.blkGen) k_spmv_hb<TB, TV, true><<<grid, 256, 0, st>>>(m, hb, (const TV*)x, scal, (TV*)vout, (TV*)y);
    else k_spmv_hb<TB, TV, false><<<grid, 256, 0, st>>>(m, hb, (const TV*)x, scal, (TV*)vout, (TV*)y);
}

void launchSpmvHB(const MeshView& m, const HBBlocks& hb, int vecFp32, const void* x, const double* scal, void* vout,
                  void* y, hipStream_t st) {
    if (hb.fp32 && vecFp32) spmvHBT<float, float>(m, hb, x, scal, vout, y, st);
    else if (hb.fp32) spmvHBT<float, double>(m, hb, x, scal, vout, y, st);
    else if (vecFp32) spmvHBT<double, float>(m, hb, x, scal, vout, y, st);
    else spmvHBT<double, double>(m, hb, x, scal, vout, y, st);
}

template <typename TB, typename TV, bool GEN>
void lusgsHBG(const MeshView& m, const Levels& L, const HBBlocks& hb, const double* rD, void* r, hipStream_t st) {
    for (int l = 0; l < L.nFwd; ++l) {
        const int s0 = L.fwdPtrHost[l], n = L.fwdPtrHost[l + 1] - s0;
        if (L.fwdSkip && l == 0) continue;
        dim3 grid(xcdGrid(n, 256), hb.nO);
        k_lusgs_hb<TB, TV, true, GEN><<<grid, 256, 0, st>>>(m, hb, rD, (TV*)r, L.fwdCells + s0, n);
    }
    for (int l = 0; l < L.nBwd; ++l) {
        const int s0 = L.bwdPtrHost[l], n = L.bwdPtrHost[l + 1] - s0;
        dim3 grid(xcdGrid(n, 256), hb.nO);
        k_lusgs_hb<TB, TV, false, GEN><<<grid, 256, 0, st>>>(m, hb, rD, (TV*)r, L.bwdCells + s0, n);
    }
}

template <typename TB, typename TV>
void lusgsHBT(const MeshView& m, const Levels& L, const HBBlocks& hb, const double* rD, void* r, hipStream_t st) {
    if (m.blkGen) lusgsHBG<TB, TV, true>(m, L, hb, rD, r, st);
    else lusgsHBG<TB, TV, false>(m, L, hb, rD, r, st);
}

void launchLusgsHB(const MeshView& m, const Levels& L, const HBBlocks& hb, int vecFp32, const double* rD, void* r,
                   hipStream_t st) {
    if (hb.fp32 && vecFp32) lusgsHBT<float, float>(m, L, hb, rD, r, st);
    else if (hb.fp32) lusgsHBT<float, double>(m, L, hb, rD, r, st);
    else if (vecFp32) lusgsHBT<double, float>(m, L, hb, rD, r, st);
    else lusgsHBT<double, double>(m, L, hb, rD, r, st);
}

bool launchSpmvLusgsHB(const MeshView& m, const Levels& L, const HBBlocks& hb, int vecFp32, const double* rD,
                       const void* x, const double* scal, const NormIn& norm, void* vout, void* t, void* y,
                       hipStream_t st) {
    if (!fusedOperator(L, hb.fp32, vecFp32)) return false;
    if (vecFp32) opLaunch<float, true>(m, L, hb, nullptr, nullptr, rD, x, scal, norm, vout, t, y, 256, st);
    else opLaunch<double, true>(m, L, hb, nullptr, nullptr, rD, x, scal, norm, vout, t, y, 256, st);
    return true;
}

void hbSubAverage(const MeshView& m, int nO, Work& wk, GmresScalars* g, const double* W, double* out,
                  hipStream_t st) {
    subAverage<double>(m.nC, nO, wk, g, W, out, st);
}

void hbNormFactors(const MeshView& m, int nO, Work& wk, const GmresPtrs& gp, const double* t, const double* b,
                   hipStream_t st) {
    normFactors<double>(m.nC, nO, wk, gp, t, b, st);
}

void hbFinalResidual(const MeshView& m, int nO, Work& wk, const GmresPtrs& gp, const double* b, double* r,
                     hipStream_t st) {
    finalResidual<double>(m.nC, nO, m.emptyDir, wk, gp, b, r, st);
}

void launchStart(size_t n, const double* b, double* r, double* dW, hipStream_t st) {
    k_start<<<nb(n, 256), 256, 0, st>>>(n, b, r, dW);
}

void launchUpdateSolution(size_t nVec, double* dW, const double* V, size_t vstride, int nv, const GmresScalars* g,
                          hipStream_t st) {
    k_update_sol<double, double><<<nb(5 * nVec, 256), 256, 0, st>>>((int)nVec, dW, V, vstride, nv, g->yh);
}

}  // namespace icsf

// ------------------------------------------------------- flexible GMRES ---
namespace icsf {

namespace {
template <typename TV>
__global__ void k_scale_by(size_t n, const TV* __restrict__ a, const double* __restrict__ beta, TV* __restrict__ b) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = a[i] / (TV)(*beta);
}
}  // namespace

// One FGMRES(m) cycle in FP64 (Saad's right-preconditioned flexible GMRES):
// v_0 = r/||r||; z_j = M_j^-1 v_j (callback); w = A z_j; Gram-Schmidt
// against v_0..v_j; Givens; back-substitution into g->yh.  Z holds z_j.
void fgmresCycle(const FgmresArgs& a, hipStream_t st) {
    const MeshView& m = *a.m;
    const int nC = a.nVec ? a.nVec : m.nC;
    const int nbk = reduceBlocks(nC);
    const size_t vs = (size_t)5 * nC;
    double* r = (double*)a.r;
    double* V = (double*)a.V;
    double* Z = (double*)a.Z;
    GmresScalars* g = a.g;
    double* pn = a.wk->part + kNormPart;
    k_norm2<double><<<nbk, 256, 0, st>>>(nC, r, pn);
    for (int i = 0; i < a.nDirs; ++i) {
        double* vi = V + (size_t)i * vs;
        double* zi = Z + (size_t)i * vs;
        k_reduce_norm<<<1, 64, 0, st>>>(NormIn{pn, i == 0 ? nbk : updateBlocks(nC), &g->beta, &g->hn[i]});
        k_scale_by<double><<<nb(vs, 256), 256, 0, st>>>(vs, r, &g->beta, vi);
        a.precond(vi, zi);
        // the outer product is timed with the other work, so that the
        // operator class holds the Arnoldi operator groups only
        if (a.mark) a.mark(TK_OTHER, 1);
        if (a.op) a.op(zi, r);
        else launchSpmv(m, a.blkFp32, 0, a.blk, a.dg, zi, nullptr, nullptr, r, st);
        if (a.mark) a.mark(TK_OTHER, 0);
        if (a.mark) a.mark(TK_ORTH, 1);
        orthStep<double>(m, a.orth, nC, r, V, i, g, a.wk->part, st);
        if (a.mark) a.mark(TK_ORTH, 0);
    }
    k_reduce_norm<<<1, 64, 0, st>>>(NormIn{pn, updateBlocks(nC), &g->beta, &g->hn[a.nDirs]});
    k_gm_finish<<<1, 64, 0, st>>>(g, a.nDirs, nullptr, 0);
}

// z = sum_i y_i V_i from zero (inner solve result), FP32 or FP64 vectors.
void launchCombine(int nC, int vecFp32, const void* V, int nv, const GmresScalars* g, void* z, hipStream_t st) {
    const size_t vs = (size_t)5 * nC;
    launchZero(vs, vecFp32, z, st);
    if (vecFp32)
        k_update_sol<float, float><<<nb(vs, 256), 256, 0, st>>>(nC, (float*)z, (const float*)V, vs, nv, g->yh);
    else
        k_update_sol<double, double><<<nb(vs, 256), 256, 0, st>>>(nC, (double*)z, (const double*)V, vs, nv, g->yh);
}

void fgmresUpdateAndResidual(const MeshView& m, Work& wk, GmresScalars* g, int blkFp32, const void* blk,
                             const void* dg, int nDirs, const void* Z, void* dW, const void* b, void* r,
                             hipStream_t st) {
    updResT<double>(m, wk, g, blkFp32, blk, dg, nDirs, Z, dW, b, r, st);
}

}  // namespace icsf
