// Kernels of the device Davidson iteration (solver_step.hip) and what they share with the host.
#pragma once

#include "context.hpp"

namespace xatu_dev {

constexpr int kStepMaxBlock = 32;  // columns of a Ritz or correction block

// Device clock values: start of the Rayleigh-Ritz kernel, of the Ritz block, of the whitening, of the
// operator's product (left by its first kernel: the host waits for the iteration's report before it
// launches the product) and of the projections after it.
enum { kStampEigen, kStampRitz, kStampWhiten, kStampProduct, kStampExtend, kStamps };

// Report of an iteration in mapped host memory: Ritz values, squared residual norms, stamps, whether
// the block was whitened. Each value comes with its exclusive or with the report's sequence
// number. Words of 8 bytes arrive whole, in any order; a value that matches its check with the
// sequence asked for is the new one: with the new check that is plain, with an older check o
// the match would make the value another than the one that o was written with.
constexpr int kReportEntries = 2 * kStepMaxBlock + kStamps + 1;
struct StepReport {
    ulonglong2 entry[kReportEntries];
};

struct RitzBlockArgs {
    double2 *V, *W;         // N x m
    const double2* Y;       // m x b
    const double *theta, *diag;
    int64_t N;
    int m, b, nb, restart;
    double2 *X, *AX, *T;    // N x b, N x b, N x nb
    double* partial;        // ritz_block_partials(N) per column
    double2* Tm;            // projected matrix, ld ldt (restart)
    int ldt;
    unsigned long long* stamps;
};
int ritz_block_partials(int64_t N);
void launch_ritz_block(const RitzBlockArgs& a, hipStream_t s);

struct WhitenArgs {
    const double2* P;   // the block's rows of its Gram matrix
    int ldp, nb, b;
    double2* T;         // N x nb, the block
    int64_t N;
    double2* S;         // nb x nb
    int* flag;
    const double *theta, *norm2;
    unsigned long long* stamps;
    StepReport* host;
    unsigned long long sequence;
};
// Whitening of the block and its application; the report to the host.
void launch_whiten(const WhitenArgs& a, hipStream_t s);

// P = A^H B (m x n), and norm2[j] = the sum of column j's residual partials (n = 0: these only)
void launch_gram_norms(Context& c, const double2* A, int lda, const double2* B, int ldb, int m, int n, double2* P, int ldp,
                       const double* partial, int npartial, int ncols, double* norm2, hipStream_t s);
// The rows and columns m0 .. m0 + nb of the projected matrix from V^H W, V of m0 + nb columns
// and W the last nb products; leaves its start in stamps.
void launch_gram_extend(Context& c, const double2* V, const double2* W, int64_t N, int m0, int nb, double2* Tm, int ldt,
                        unsigned long long* stamps, hipStream_t s);

}  // namespace xatu_dev
