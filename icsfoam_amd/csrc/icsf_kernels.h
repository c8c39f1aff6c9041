// Launch interfaces of the HIP kernels (host side).
#pragma once
#include <hip/hip_runtime.h>
#include <functional>
#include <vector>

#include "icsf_views.h"

namespace icsf {

constexpr int KMAX = 64;  // largest nDirections supported by the device GMRES

// Sweep levels of the LU-SGS dependency graph (cells grouped by level).
struct Levels {
    int nFwd = 0, nBwd = 0;
    std::vector<int> fwdPtrHost, bwdPtrHost;  // [n+1] offsets into the cell lists
    int* fwdCells = nullptr;                  // device, [nC]
    int* bwdCells = nullptr;                  // device, [nC]
    bool fwdSkip = true;                      // level 0 has no lower neighbours
    // two levels each way, forward level 1 == backward level 0 (a two-colour
    // numbering: every neighbour of a level-1 cell is a level-0 cell)
    bool twoColour = false;
    // two-colour levels that are the cell ranges [0, n0) and [n0, nC)
    bool colourMajor = false;
    // dataflow sweep (null when the levels are swept by a launch each): the
    // cells of each level in chunks of a wavefront (-1 pads a level's last
    // chunk), the level of each chunk, the chunks of each level (forward,
    // then backward levels), all on the device
    int nFwdChunks = 0, nBwdChunks = 0;
    int *chunkCells = nullptr, *chunkLevel = nullptr, *levelChunks = nullptr;
};
// Largest average number of cells per level swept in one dataflow launch: a
// launch per level costs the same up to there (its latency), while the
// dataflow's uncached loads add up.  Boxes in random order (34 to 42 levels),
// pseudo-step with a launch per level / in one launch: 3770 cells per level
// FP64 14.1 / 10.5 ms, mixed 11.7 / 10.0; 8270 17.0 / 13.6, 14.1 / 12.5; 9760
// 19.5 / 16.6, 15.9 / 14.8; 12700 21.8 / 20.0, 17.3 / 17.8; 13800 25.5 / 23.7,
// 19.8 / 20.6; 17800 34.4 / 32.8, 26.5 / 28.5.  One line for both precisions,
// on the side of mixed, which crosses near 11000.
constexpr int kSweepLevelCells = 8192;
// Fewest levels (forward and backward together) for it: the 28 059-cell LS89
// mesh coloured (4 + 4 levels) steps in 2.36 ms with its 7 launches per
// application and 2.43 ms in one, 17 + 17 levels are well ahead (above).
constexpr int kSweepMinLevels = 24;

// Incomplete polls after which one wait of the dataflow sweep gives up.
constexpr int kSweepPolls = 1 << 21;

// Scratch for two-stage reductions, and of the dataflow sweep: the forward
// and the final values [5][nC], the levels' finished chunks and the next chunk
// to draw, the case's error flags (swF null: none).
struct Work {
    double* part = nullptr;  // [kPartSize]
    void *swF = nullptr, *swO = nullptr;
    int *swDone = nullptr, *err = nullptr;
    int swLimit = kSweepPolls;
};

// 1024 workgroups' partials of the 2 KMAX projection values of one step, then
// those of a norm (from kNormPart)
constexpr size_t kNormPart = (size_t)1024 * 2 * KMAX, kPartSize = kNormPart + 1024;

// A norm still in partials: nb sums of squares at part; whoever reduces them
// stores the norm at beta and hn.
struct NormIn {
    const double* part = nullptr;
    int nb = 0;
    double *beta = nullptr, *hn = nullptr;
};

struct GmresScalars;

struct GmresArgs {
    const MeshView* m;
    const Levels* lev;
    Work* wk;
    GmresScalars* g;  // device
    int nDirs;
    int precond;      // 0 LUSGS, 1 Jacobi, 2 none
    int orth;         // 0 MGS (reference order), 1 CGS
    int blkFp32;
    const void* blk;
    const void* dg;
    const double* rD;
    const void* dinv;
    void* r;          // residual / work vector, [5][nC]
    void* r2;         // second work vector (SpMV output), [5][nC]
    void* V;          // Krylov basis, nDirs vectors of [5][nC]
    void* t;          // work vector of the fused operator, [5][nC]
    // optional timing marks: mark(kernelClass, begin?1:0)
    std::function<void(int, int)> mark;
    // Batched (harmonic-balance) systems: vectors of 5*nVec entries and
    // caller-supplied operator y = A (x/scal) (vout = x/scal when given)
    // and preconditioner v <- M^-1 v.  nVec 0 / empty hooks: the single
    // mesh SpMV and LU-SGS/Jacobi above.
    int nVec = 0;
    std::function<void(const void*, const double*, void*, void*)> op;
    std::function<void(void*)> pre;
    // fuse the Arnoldi SpMV with the LU-SGS sweeps when the level structure
    // allows it (same algorithm; a row's terms summed in another order)
    bool fuse = false;
    // batched systems: fused operator + preconditioner on x / norm (empty: op
    // and pre are used)
    std::function<void(const void*, const NormIn&, void*, void*)> opPre;
};

// Harmonic balance, one launch per stage for all instances
// (blockIdx.y = instance): each instance's mesh view (its own boundary
// conditions), state and FP64 Jacobian storage, in device memory.
struct HBInst {
    MeshView m;
    StateView s;
    void* blk;    // FP64, or FP32 with mixed precision
    void* dg;
    double* rD;
    int* err;
};
// The harmonic-balance terms formed in the instances' Jacobian launch
// (HBZone.C:359-518): with the residual cell sums, the spectral source into
// the coupled right-hand side; V D_JJ on each instance's diagonal blocks;
// then (one small launch) the shared LU-SGS diagonal over all instances.
struct HBCouple {
    int nO;
    const double* D;  // [nO][nO] spectral operator
    double* Wall;     // [nO][5][nC] coupled state (written with the source)
    double* ball;     // [nO][5][nC] coupled right-hand side b + source
    double* rD;       // [nC] shared LU-SGS reciprocal diagonal
    int* err;         // zero-diagonal flag of the coupled system
};
// cellSums: as launchResidual / launchCellSumsJacobian, for all instances
void launchResidualHB(const HBInst* inst, int nO, const MeshView& m, const Phys& ph, hipStream_t st,
                      bool cellSums = true);
// Fourier reconstruction of the instances' fields at one time, out [nC][6]
void launchHBReconstruct(int nC, int nO, const HBInst* inst, const double* w, double* out, hipStream_t st);
void launchJacobianHB(const HBInst* inst, int nO, int fp32, const MeshView& m, const Phys& ph, hipStream_t st,
                      bool cellSums, const HBCouple& hc);

// Harmonic-balance coupling: per-instance block storage (FP64) and the
// spectral operator D [nO][nO] (device).
constexpr int HB_MAXO = 16;
struct HBBlocks {
    int nO;
    int fp32;                     // blocks stored in FP32 (mixed precision)
    const void* blk[HB_MAXO];
    const void* dg[HB_MAXO];
    const double* D;
};

// kernel classes of the timing marks
enum { TK_RESIDUAL = 0, TK_JACOBIAN = 1, TK_SPMV = 2, TK_PRECOND = 3, TK_ORTH = 4, TK_OTHER = 5 };

// Flexible GMRES (FP64 outer); precond(v, z) writes z = M^-1 v.
struct FgmresArgs {
    const MeshView* m;
    Work* wk;
    GmresScalars* g;
    int nDirs;
    int orth;
    int blkFp32;
    const void* blk;
    const void* dg;
    void* r;  // [5][nC] FP64
    void* V;  // nDirs+1 FP64 vectors
    void* Z;  // nDirs FP64 vectors
    std::function<void(const double*, double*)> precond;
    std::function<void(int, int)> mark;
    // batched (harmonic-balance) systems: 5*nVec entries per vector and a
    // caller-supplied y = A z (FP64 vectors); nVec 0 / empty: the mesh SpMV
    int nVec = 0;
    std::function<void(const double*, double*)> op;
};

int reduceBlocks(int nC);
// Full 5x5 off-diagonal blocks (sliced layout) from generator storage.
void launchExpandBlocks(const MeshView& m, int fp32, const void* gen, void* out, hipStream_t st);
void launchProjectionPasses(const MeshView& m, int vecFp32, int ch, int mgs, const void* w, const void* V, int nv,
                            double* part, hipStream_t st);

// State update from Wsrc (null: the state's W) plus dW (null: none); W0 (optional)
// keeps a copy of Wsrc.
void launchUpdate(const MeshView& m, const Phys& ph, const StateView& s, const double* dW, int mode,
                  const double* rho0, const double* U0, const double* T0, hipStream_t st,
                  const double* Wsrc = nullptr, double* W0 = nullptr);
// the same for instances J0 .. J0 + n - 1 of a harmonic-balance system, each
// with its own view, dW [nO][5][nC]
void launchUpdateHB(const HBInst* inst, int J0, int n, const MeshView& m, const Phys& ph, const double* dW,
                    hipStream_t st);
// Forward part of the residual adjoint: boundary values and gradients,
// keeping the unlimited gradients and limiter values.
void launchAdjointForward(const MeshView& m, const Phys& ph, const StateView& s, double* gun, double* limo,
                          hipStream_t st);
// Reverse pass: gW = (db/dW)^T v, gS = (db/dSf)^T v, gC = (db/dCf)^T v
// (geom false: gS and gC are work space only, and the Roe reverse skips
// its Sf passes).
void launchResidualVjp(const MeshView& m, const Phys& ph, const StateView& s, const AdjView& a, const double* v,
                       double* gW, double* gS, double* gC, bool geom, hipStream_t st);
// cellSums false: everything up to the face terms; the cell sums (b,
// rPseudoDeltaT) are then formed by launchCellSumsJacobian.  bOut: b is written
// there too, and the face records are short ones that the Jacobian cannot read
// (launchFaceTerms makes the full ones).
void launchResidual(const MeshView& m, const Phys& ph, const StateView& s, hipStream_t st, bool cellSums = true,
                    double* bOut = nullptr);
void launchFaceTerms(const MeshView& m, const Phys& ph, const StateView& s, hipStream_t st);
void launchFaceFlux(const MeshView& m, const Phys& ph, const StateView& s, double* phi, double* phiU, double* phiE,
                    hipStream_t st);
void launchJacobian(const MeshView& m, const Phys& ph, const StateView& s, void* blk, void* dg, int fp32,
                    double* rD, int* err, hipStream_t st);
// Cell sums of the residual (b, rPseudoDeltaT) and the Jacobian rows in one
// kernel, after launchResidual(..., cellSums = false); same results as
// k_cell_residual followed by launchJacobian.
void launchCellSumsJacobian(const MeshView& m, const Phys& ph, const StateView& s, void* blk, void* dg, int fp32,
                            double* rD, int* err, hipStream_t st);

void launchSpmv(const MeshView& m, int blkFp32, int vecFp32, const void* blk, const void* dg, const void* x,
                const double* scal, void* vout, void* y, hipStream_t st);
void launchLusgs(const MeshView& m, const Levels& L, const Work& wk, int blkFp32, int vecFp32, const void* blk,
                 const double* rD, void* r, hipStream_t st);
// Whether the fused operator applies: two-colour levels, blocks and vectors of
// one precision.
inline bool fusedOperator(const Levels& L, int blkFp32, int vecFp32) { return L.twoColour && blkFp32 == vecFp32; }
// y = LU-SGS(A (x/scal)) in three passes on a two-colour level structure, t
// a work vector (false: not applicable, nothing launched).  norm.part: the
// scale is that norm, reduced in the first pass; scal is then where it stores
// it (norm.beta).
bool launchSpmvLusgs(const MeshView& m, const Levels& L, int blkFp32, int vecFp32, const void* blk, const void* dg,
                     const double* rD, const void* x, const double* scal, const NormIn& norm, void* vout, void* t,
                     void* y, hipStream_t st);
void launchJacobiSetup(int nC, int blkFp32, const void* dg, void* dinv, hipStream_t st);
void launchJacobiApply(int nC, int blkFp32, int vecFp32, const void* dinv, void* r, hipStream_t st);

// GMRES building blocks (icsf_krylov.hip)
size_t gmresScalarsBytes();
void gmresPrepare(const MeshView& m, Work& wk, GmresScalars* g, int vecFp32, const void* W, const void* b,
                  void* tmp1, void* tmp2, int blkFp32, const void* blk, const void* dg, hipStream_t st);
void gmresCycle(const GmresArgs& a, int vecFp32, hipStream_t st);
void gmresUpdateAndResidual(const MeshView& m, Work& wk, GmresScalars* g, int vecFp32, int blkFp32,
                            const void* blk, const void* dg, int nDirs, const void* V, void* dW, const void* b,
                            void* r, hipStream_t st);
void fgmresCycle(const FgmresArgs& a, hipStream_t st);
void fgmresUpdateAndResidual(const MeshView& m, Work& wk, GmresScalars* g, int blkFp32, const void* blk,
                             const void* dg, int nDirs, const void* Z, void* dW, const void* b, void* r,
                             hipStream_t st);
void launchCombine(int nC, int vecFp32, const void* V, int nv, const GmresScalars* g, void* z, hipStream_t st);

// Harmonic balance (icsf_krylov.hip): y = A_HB (x/scal) over [nO][5][nC]
// vectors in coupledMatrix order, with vout = x/scal when given.
void launchSpmvHB(const MeshView& m, const HBBlocks& hb, int vecFp32, const void* x, const double* scal, void* vout,
                  void* y, hipStream_t st);
// Per-variable bookkeeping of one instance slice ([5][nC]) into g: W minus
// its per-component average; norm factors and initial residuals from
// t = A (W - avg) and b; final residuals from r = b - A dW (r holds A dW on
// entry).
// y = LU-SGS(A_HB (x/scal)) in three passes on a two-colour level
// structure, t a work vector (false: not applicable, nothing launched).
bool launchSpmvLusgsHB(const MeshView& m, const Levels& L, const HBBlocks& hb, int vecFp32, const double* rD,
                       const void* x, const double* scal, const NormIn& norm, void* vout, void* t, void* y,
                       hipStream_t st);
// LU-SGS of all HB instances (per-instance sweeps, shared diagonal rD).
void launchLusgsHB(const MeshView& m, const Levels& L, const HBBlocks& hb, int vecFp32, const double* rD, void* r,
                   hipStream_t st);
// The pieces of gmresPrepare / gmresUpdateAndResidual for nO instances' vectors
// [nO][5][nC], one launch over all; g: the solver's scalars (scratch sums),
// gp: each instance's residuals.
struct GmresPtrs {
    GmresScalars* g[HB_MAXO];
};
void hbSubAverage(const MeshView& m, int nO, Work& wk, GmresScalars* g, const double* W, double* out,
                  hipStream_t st);
void hbNormFactors(const MeshView& m, int nO, Work& wk, const GmresPtrs& gp, const double* t, const double* b,
                   hipStream_t st);
void hbFinalResidual(const MeshView& m, int nO, Work& wk, const GmresPtrs& gp, const double* b, double* r,
                     hipStream_t st);
// a solve's start over n entries: r = b, dW = 0
void launchStart(size_t n, const double* b, double* r, double* dW, hipStream_t st);
// dW += sum_i y_i V_i over 5*nVec entries
void launchUpdateSolution(size_t nVec, double* dW, const double* V, size_t vstride, int nv, const GmresScalars* g,
                          hipStream_t st);
void gmresReadResiduals(const GmresScalars* g, double* res10, hipStream_t st);
const double* gmresResidualsDevice(const GmresScalars* g);

void launchCopy(size_t n, int fp32, const void* a, void* b, hipStream_t st);
void launchConvert(size_t n, int fromFp32, const void* a, void* b, hipStream_t st);
void launchZero(size_t n, int fp32, void* x, hipStream_t st);
void launchZeroComponent(int nC, int comp, int fp32, void* x, hipStream_t st);

}  // namespace icsf
