// Block GMRES with one shared block Krylov basis and rank-drop deflation:
// block_gmres_preconditioned_with_guess → block_gmres_inner
// (crates/sonium-solvers/crates/sonium-solvers-iterative/src/block_gmres.rs:
// 163-215, 666-1120), the reference's solve_many path
// (BemSolver::solve_many → solve_compressed_many → block_gmres_preconditioned,
// crates/sonium-bem/src/core/bem_solver.rs:2032, 2175-2181).
//
// Device: the basis (column-major, vector i at V + i*n), the block products,
// the block Gram matrices V^H W and the projections W -= V G and X += V Y on
// FP64 MFMA, and the per-column CGS2 QR of each new block with the
// reference's rank-drop test (block_krylov_kernels.hip).  The block-Hessenberg
// least-squares problem (solve_block_ls, :614-664) is on the device too, as a
// Householder QR that grows with the basis: the reference refactors the whole
// (p + s') x p matrix with Givens rotations after every block step, but a step
// adds columns whose new rows are zero in every older column, so the older
// columns' factors hold and only the new ones are formed.  Host: the control
// flow of block_gmres_inner, from the residual norms each step leaves in pinned
// memory; it waits once a step.  The minimiser Y is formed only where the
// reference uses it (an exact residual check, the end of a cycle).

#include <algorithm>
#include <cmath>
#include <vector>

#include "block_krylov.hpp"
#include "internal.hpp"

namespace sbh {

// block_krylov_kernels.hip
int64_t bk_gram_partial_elems(int64_t n, int max_basis, int s);
void bk_gram(sbh_context* ctx, const double2* V, int64_t ldv, int p, const double2* W, int64_t ldw, int sj,
             int64_t n, double* part, double2* gram, double2* hacc, int hmode, const int* flag);
void bk_combine(sbh_context* ctx, const double2* V, int64_t ldv, int p, const double2* C, int ldc, int sj, int64_t n,
                double2* O, int64_t osc, int64_t osk, bool add, double alpha, const int* flag);
size_t bk_cholesky_state_bytes(int m);
void bk_cholesky(sbh_context* ctx, const double2* G, int m, double floor, int pass, void* state, double2* T);
void bk_to_rowmajor(sbh_context* ctx, const double2* in, int64_t ld, int cols, int64_t n, double2* out);
void bk_to_colmajor(sbh_context* ctx, const double2* in, int cols, int64_t n, const double2* d, double2* out,
                    int64_t ld);
void bk_residual_cm(sbh_context* ctx, const double2* B, const double2* AX, int s, int64_t n, const double2* d,
                    double2* R);
int bk_norm_chunks(int64_t n);
void bk_colnorms(sbh_context* ctx, const double2* X, int64_t ld, int cols, int64_t n, double* part, double* out);
int bk_frob_partials(sbh_context* ctx, const double2* X, int64_t count, double* part);
void bk_dgks_flag(sbh_context* ctx, const double* before, const double* after, int chunks, int* flag, double* frob);
void bk_true_metrics(sbh_context* ctx, const double2* B, const double2* AX, int s, int64_t n, double* part,
                     double* out);
size_t bk_qr_state_bytes();
size_t bk_qr_partial_elems(int64_t n);
void bk_block_qr(sbh_context* ctx, double2* W, double2* Q, int64_t n, int sj, int budget, void* state,
                 double2* part);
void zgemm_f64(sbh_context* ctx, const double2* A, int64_t lda, int64_t n, const double2* X, int64_t k, double2* Y);

namespace {

constexpr double TINY = 1e-30;

}  // namespace

struct BlockGmresParams {
    int64_t max_iterations = 100;
    int64_t restart = 30;
    double tol = 1e-6;
    bool true_residual_check = true;
    int64_t exact_interval = 0;
};

struct BlockGmresResult {
    int64_t iterations = 0, spmv = 0, exact_checks = 0, cycles = 0, max_basis = 0, deflated = 0;
    int64_t cholqr_blocks = 0, chain_blocks = 0;
    bool converged = false;
    std::vector<double> projected, true_res, backward;
};

class BlockGmresEngine {
   public:
    BlockGmresEngine(sbh_operator* op, const sbh_precond* M, int s, int64_t restart)
        : op_(op), ctx_(op->ctx), n_(op->n), s_(s), dinv_(M && M->kind == 1 ? M->d_dinv.ptr : nullptr),
          max_steps_((int)std::max<int64_t>(1, restart)), max_basis_((max_steps_ + 1) * s),
          ls_(ctx_, n_, s, max_basis_, max_steps_) {
        const size_t blk = (size_t)n_ * s;
        admit_device(ctx_,
                     (int64_t)(sizeof(double2) * ((size_t)(max_basis_ + s) * n_ + 6 * blk)) +
                         BlockLeastSquares::device_bytes(n_, s, max_steps_),
                     "the shared block Krylov basis", false);
        ls_.allocate();
        V_.allocate((size_t)(max_basis_ + s) * n_);
        W_.allocate(blk);
        Rcm_.allocate(blk);
        Xc_.allocate(blk);
        AX_.allocate(blk);
        Vrm_.allocate(blk);
        Yrm_.allocate(blk);
        gpart_.allocate((size_t)bk_gram_partial_elems(n_, max_basis_, s));
        gram_.allocate((size_t)max_basis_ * s + 16);
        hacc_.allocate((size_t)max_basis_ * s);
        chol_.allocate(bk_cholesky_state_bytes(s));
        chain_.allocate(bk_qr_state_bytes());
        qpart_.allocate(bk_qr_partial_elems(n_));
        nchunks_ = bk_norm_chunks((int64_t)n_ * s);
        npart_.allocate((size_t)std::max<int64_t>(3 * s, 4) * bk_norm_chunks(n_) + 2 * nchunks_ + 64);
        small_.allocate(4 * (size_t)s + 64);
        flag_.allocate(4);
        small_host_.allocate(4 * (size_t)s + 64);
        qg_.allocate((size_t)s * s + 16);
        // the QR chain's workgroup counter starts at zero and every launch leaves it there
        zero_on_stream(ctx_, chain_.ptr, chain_.bytes());
    }

    void run(const double2* B, double2* X, bool x_zero, const BlockGmresParams& prm, BlockGmresResult& out);

   private:
    sbh_operator* op_;
    sbh_context* ctx_;
    int64_t n_;
    int s_;
    const double2* dinv_;
    const int max_steps_, max_basis_;
    WorkArray<double2> V_, W_, Rcm_, Xc_, AX_, Vrm_, Yrm_, gram_, qpart_, hacc_;
    WorkArray<char> chol_, chain_;  // states of the two block QRs
    WorkArray<double> gpart_, npart_, small_;
    WorkArray<int> flag_;
    WorkArray<double, true> small_host_;
    WorkArray<double2> qg_;        // sj x sj Gram matrix of the block being factored
    BlockLeastSquares ls_;
    bool chol_queued_ = false;     // the block's Cholesky QR is on the stream
    int64_t cholqr_blocks_ = 0, chain_blocks_ = 0;
    int nchunks_ = 1;
    int64_t spmv_ = 0, exact_checks_ = 0;

    double2* vec(int i) { return V_.ptr + (size_t)i * n_; }

    // Y (n x k row-major) = A X (n x k row-major)
    void apply_rm(const double2* X, double2* Y, int k) {
        if (op_->dense()) {
            if (k == 1)
                zgemv_n(ctx_, op_->sys->d_A.ptr, op_->sys->lda, n_, n_, X, Y);
            else
                zgemm_f64(ctx_, op_->sys->d_A.ptr, op_->sys->lda, n_, X, k, Y);
        } else {
            // column by column through column-major scratch
            bk_to_colmajor(ctx_, X, k, n_, nullptr, Vrm_.ptr, n_);
            for (int c = 0; c < k; ++c) operator_apply_device(op_, Vrm_.ptr + (size_t)c * n_, Yrm_.ptr + (size_t)c * n_);
            bk_to_rowmajor(ctx_, Yrm_.ptr, n_, k, n_, Y);
        }
        spmv_ += k;
    }

    // W (column-major, sj vectors) = M^-1 A V[first .. first + sj)
    void apply_cm(int first, int sj) {
        if (op_->dense()) {
            bk_to_rowmajor(ctx_, vec(first), n_, sj, n_, Vrm_.ptr);
            if (sj == 1)
                zgemv_n(ctx_, op_->sys->d_A.ptr, op_->sys->lda, n_, n_, Vrm_.ptr, Yrm_.ptr);
            else
                zgemm_f64(ctx_, op_->sys->d_A.ptr, op_->sys->lda, n_, Vrm_.ptr, sj, Yrm_.ptr);
            bk_to_colmajor(ctx_, Yrm_.ptr, sj, n_, dinv_, W_.ptr, n_);
        } else {
            for (int c = 0; c < sj; ++c) {
                operator_apply_device(op_, vec(first + c), Yrm_.ptr);
                if (dinv_)
                    diag_scale(ctx_, dinv_, Yrm_.ptr, W_.ptr + (size_t)c * n_, n_);
                else
                    device_copy(ctx_, Yrm_.ptr, W_.ptr + (size_t)c * n_, n_);
            }
        }
        spmv_ += sj;
    }

    // One block Arnoldi step on the device: W = M^-1 A V_j, block CGS
    // against V[0:p] with the DGKS trigger, then the QR of W into V[p:]
    // (block_gmres.rs:918-1025).  Nothing is read back here.
    void queue_step(int p, int sj) {
        const int p_start = p - sj;
        apply_cm(p_start, sj);
        double* before = npart_.ptr;
        double* after = npart_.ptr + nchunks_;
        double* frob = small_.ptr;
        const int chunks = bk_frob_partials(ctx_, W_.ptr, (int64_t)sj * n_, before);
        bk_gram(ctx_, V_.ptr, n_, p, W_.ptr, n_, sj, n_, gpart_.ptr, gram_.ptr, hacc_.ptr, 1, nullptr);
        bk_combine(ctx_, V_.ptr, n_, p, gram_.ptr, sj, sj, n_, W_.ptr, n_, 1, true, -1.0, nullptr);
        bk_frob_partials(ctx_, W_.ptr, (int64_t)sj * n_, after);
        bk_dgks_flag(ctx_, before, after, chunks, flag_.ptr, frob);
        bk_gram(ctx_, V_.ptr, n_, p, W_.ptr, n_, sj, n_, gpart_.ptr, gram_.ptr, hacc_.ptr, 2, flag_.ptr);
        bk_combine(ctx_, V_.ptr, n_, p, gram_.ptr, sj, sj, n_, W_.ptr, n_, 1, true, -1.0, flag_.ptr);
        queue_qr(p, sj, max_basis_ - p);
    }

    // QR of the sj column-major vectors in W_ into the basis slots dst..:
    // Cholesky QR twice when every pivot is clearly positive (the block is far
    // from the rank-drop threshold) and the block fits the budget, which gives
    // the per-column CGS2 factors to rounding; otherwise the per-column CGS2
    // chain with rank-drop deflation (read_qr).  The first way runs on the
    // device without a decision of the host; it leaves W_ unchanged, so the
    // second can always follow.
    void queue_qr(int dst, int sj, int budget) {
        constexpr double kPivotFloor = 1e-4;  // four orders above sqrt(eps)
        chol_queued_ = sj <= budget;
        if (!chol_queued_) return;
        const int* ok = reinterpret_cast<const int*>(chol_.ptr);
        bk_gram(ctx_, W_.ptr, n_, sj, W_.ptr, n_, sj, n_, gpart_.ptr, qg_.ptr, nullptr, 0, nullptr);
        bk_cholesky(ctx_, qg_.ptr, sj, kPivotFloor, 0, chol_.ptr, gram_.ptr);
        bk_combine(ctx_, W_.ptr, n_, sj, gram_.ptr, sj, sj, n_, Yrm_.ptr, n_, 1, false, 1.0, ok);
        bk_gram(ctx_, Yrm_.ptr, n_, sj, Yrm_.ptr, n_, sj, n_, gpart_.ptr, qg_.ptr, nullptr, 0, ok);
        bk_cholesky(ctx_, qg_.ptr, sj, 0.5, 1, chol_.ptr, gram_.ptr);
        bk_combine(ctx_, Yrm_.ptr, n_, sj, gram_.ptr, sj, sj, n_, vec(dst), n_, 1, false, 1.0, ok);
    }

    // The outcome of the queued QR, with the CGS2 chain run where the Cholesky
    // QR did not hold.  step: the Hessenberg columns of that block are added to
    // the least-squares problem, whose residual norms come with the outcome.
    const BlockStep& finish_qr(int dst, int sj, int budget, bool step) {
        auto outcome = [&](const void* chain) {
            if (step)
                ls_.add(chol_.ptr, chain, hacc_.ptr, sj);
            else
                ls_.report(chol_.ptr, chain, sj);
            SBH_HIP(hipStreamSynchronize(ctx_->stream));
        };
        if (chol_queued_) {
            outcome(nullptr);
            cholqr_blocks_ += ls_.host().ok;
        }
        if (!chol_queued_ || !ls_.host().ok) {
            bk_block_qr(ctx_, W_.ptr, vec(dst), n_, sj, budget, chain_.ptr, qpart_.ptr);
            outcome(chain_.ptr);
            chain_blocks_ += 1;
        }
        if (step) ls_.accept(sj);
        return ls_.host();
    }

    std::vector<double> read_small(int count) {
        SBH_HIP(hipMemcpyAsync(small_host_.ptr, small_.ptr, sizeof(double) * count, hipMemcpyDeviceToHost,
                               ctx_->stream));
        SBH_HIP(hipStreamSynchronize(ctx_->stream));
        return std::vector<double>(small_host_.ptr, small_host_.ptr + count);
    }

    // per-column norms of a row-major n x s block: through the column-major scratch
    std::vector<double> colnorms_rm(const double2* X) {
        bk_to_colmajor(ctx_, X, s_, n_, nullptr, Rcm_.ptr, n_);
        bk_colnorms(ctx_, Rcm_.ptr, n_, s_, n_, npart_.ptr, small_.ptr);
        return read_small(s_);
    }

    // block_true_metrics (block_gmres.rs:567-612): ||b - A x||/||b|| and the
    // normwise backward error per column, with one block product.
    void true_metrics(const double2* B, const double2* Xd, const std::vector<double>& b_true,
                      std::vector<double>& tr, std::vector<double>& be) {
        apply_rm(Xd, AX_.ptr, s_);
        exact_checks_ += 1;
        bk_true_metrics(ctx_, B, AX_.ptr, s_, n_, npart_.ptr, small_.ptr);
        const std::vector<double> m = read_small(3 * s_);
        tr.assign(s_, 0.0);
        be.assign(s_, 0.0);
        for (int j = 0; j < s_; ++j) {
            const double ar = m[j], axn = m[s_ + j], bn = m[2 * s_ + j];
            tr[j] = b_true[j] <= TINY ? ar : ar / b_true[j];
            be[j] = ar / std::max(axn + bn, 2.2250738585072014e-308);
        }
    }

    // X (row-major) += V y with the least-squares solution y, apply_block_update
    void update(double2* Xd) {
        if (ls_.columns() == 0) return;
        ls_.solve(gram_.ptr);
        bk_combine(ctx_, V_.ptr, n_, ls_.columns(), gram_.ptr, s_, s_, n_, Xd, 1, s_, true, 1.0, nullptr);
    }
};

void BlockGmresEngine::run(const double2* B, double2* X, bool x_zero, const BlockGmresParams& prm,
                           BlockGmresResult& out) {
    const int s = s_;
    out = BlockGmresResult{};
    out.projected.assign(s, INFINITY);
    // ||M^-1 b_j|| for the convergence test and ||b_j|| for the true residuals
    std::vector<double> b_norms, b_true;
    bk_residual_cm(ctx_, B, nullptr, s, n_, dinv_, Rcm_.ptr);
    bk_colnorms(ctx_, Rcm_.ptr, n_, s, n_, npart_.ptr, small_.ptr);
    b_norms = read_small(s);
    b_true = colnorms_rm(B);
    std::vector<double>& projected = out.projected;
    std::vector<double> col_norms(s);
    int64_t total_iters = 0;
    bool x_known_zero = x_zero;

    for (int64_t cycle = 0; cycle < prm.max_iterations; ++cycle) {
        out.cycles += 1;
        // R0 = M^-1 (B - A X), column-major
        if (x_known_zero) {
            // A X = 0: the product is not formed (it is still counted)
            bk_residual_cm(ctx_, B, nullptr, s, n_, dinv_, Rcm_.ptr);
            spmv_ += s;
        } else {
            apply_rm(X, AX_.ptr, s);
            bk_residual_cm(ctx_, B, AX_.ptr, s, n_, dinv_, Rcm_.ptr);
        }
        bk_colnorms(ctx_, Rcm_.ptr, n_, s, n_, npart_.ptr, small_.ptr);
        col_norms = read_small(s);
        bool all_converged = true;
        for (int j = 0; j < s; ++j) {
            projected[j] = b_norms[j] >= TINY ? col_norms[j] / b_norms[j] : 0.0;
            if (b_norms[j] >= TINY && projected[j] > prm.tol) all_converged = false;
        }
        if (all_converged) break;
        // initial block QR with rank-drop deflation (CGS2 per column) of a copy of R0
        device_copy(ctx_, Rcm_.ptr, W_.ptr, n_ * s);
        queue_qr(0, s, 1 << 30);
        const int s1 = finish_qr(0, s, 1 << 30, false).next;
        out.deflated += s - s1;
        if (s1 == 0) break;
        // C0 = V1^H R0 (s1 x s)
        bk_gram(ctx_, V_.ptr, n_, s1, Rcm_.ptr, n_, s, n_, gpart_.ptr, gram_.ptr, nullptr, 0, nullptr);
        ls_.reset(gram_.ptr, s1);
        int p = s1;
        int sj = s1;
        bool converged_cycle = false;
        bool restart_cycle = false;
        for (int step = 0; step < max_steps_; ++step) {
            if (p >= max_basis_) break;
            queue_step(p, sj);
            const BlockStep& st = finish_qr(p, sj, max_basis_ - p, true);
            const int s_next = st.next;
            out.deflated += sj - s_next;
            total_iters += 1;
            for (int j = 0; j < s; ++j) projected[j] = b_norms[j] >= TINY ? st.tail[j] / b_norms[j] : 0.0;
            bool cycle_done = true;
            for (int j = 0; j < s; ++j) cycle_done = cycle_done && projected[j] <= prm.tol;
            const bool interval_due =
                prm.exact_interval > 0 && total_iters > 0 && total_iters % prm.exact_interval == 0;
            if (s_next > 0 && (interval_due || (cycle_done && prm.true_residual_check))) {
                device_copy(ctx_, X, Xc_.ptr, n_ * s);
                update(Xc_.ptr);
                std::vector<double> tr, be;
                true_metrics(B, Xc_.ptr, b_true, tr, be);
                bool exact_converged = true;
                for (int j = 0; j < s; ++j) exact_converged = exact_converged && tr[j] <= prm.tol;
                if (exact_converged) {
                    device_copy(ctx_, Xc_.ptr, X, n_ * s);
                    x_known_zero = false;
                    converged_cycle = true;
                    break;
                }
                if (cycle_done && prm.true_residual_check) {
                    device_copy(ctx_, Xc_.ptr, X, n_ * s);
                    x_known_zero = false;
                    restart_cycle = true;
                    break;
                }
            }
            if (cycle_done || s_next == 0) {
                update(X);
                x_known_zero = false;
                converged_cycle = cycle_done;
                break;
            }
            p += s_next;
            sj = s_next;
            out.max_basis = std::max<int64_t>(out.max_basis, p);
        }
        out.max_basis = std::max<int64_t>(out.max_basis, p);
        if (restart_cycle) continue;
        if (!converged_cycle && p > s1) {
            // budget exhausted: the square LS over the whole basis; its tail is
            // empty, as in the reference (rows == cols)
            for (int j = 0; j < s; ++j) projected[j] = 0.0;
            update(X);
            x_known_zero = false;
        }
        if (converged_cycle) break;
    }
    std::vector<double> tr, be;
    if (x_known_zero) {
        // A*0 = 0: the true residual is ||b|| / ||b||
        tr.assign(s, 0.0);
        be.assign(s, 0.0);
        for (int j = 0; j < s; ++j) {
            tr[j] = b_true[j] <= TINY ? b_true[j] : 1.0;
            be[j] = b_true[j] / std::max(b_true[j], 2.2250738585072014e-308);
        }
        spmv_ += s;
        exact_checks_ += 1;
    } else {
        true_metrics(B, X, b_true, tr, be);
    }
    bool conv = true;
    for (int j = 0; j < s; ++j) conv = conv && (prm.true_residual_check ? tr[j] <= prm.tol : projected[j] <= prm.tol);
    out.iterations = total_iters;
    out.true_res = tr;
    out.backward = be;
    out.converged = conv;
    out.spmv = spmv_;
    out.exact_checks = exact_checks_;
    out.cholqr_blocks = cholqr_blocks_;
    out.chain_blocks = chain_blocks_;
}

sbh_status run_block_gmres(sbh_operator* op, const sbh_precond* M, const double2* d_B, double2* d_X, int k,
                           bool x_zero, const sbh_block_gmres_config& cfg, sbh_block_gmres_info* info,
                           double* residuals, double* true_residuals, double* backward_errors) {
    BlockGmresParams prm;
    prm.max_iterations = cfg.max_iterations;
    prm.restart = cfg.restart;
    prm.tol = cfg.tolerance;
    prm.true_residual_check = cfg.true_residual_check != 0;
    prm.exact_interval = cfg.exact_residual_check_interval;
    BlockGmresEngine engine(op, M, k, cfg.restart);
    BlockGmresResult r;
    engine.run(d_B, d_X, x_zero, prm, r);
    bool finite = true;
    for (int j = 0; j < k; ++j)
        finite = finite && std::isfinite(r.projected[j]) && std::isfinite(r.true_res[j]) &&
                 std::isfinite(r.backward[j]);
    if (info) {
        *info = sbh_block_gmres_info{};
        info->iterations = r.iterations;
        info->converged = r.converged ? 1 : 0;
        info->status = !finite ? SBH_SOLVER_NUMERICAL_ERROR
                               : (r.converged ? SBH_SOLVER_CONVERGED : SBH_SOLVER_MAX_ITERATIONS);
        info->spmv_count = r.spmv;
        info->exact_residual_checks = r.exact_checks;
        info->restart_cycles = r.cycles;
        info->max_basis = r.max_basis;
        info->deflated = r.deflated;
        info->cholesky_qr_blocks = r.cholqr_blocks;
        info->chain_qr_blocks = r.chain_blocks;
    }
    for (int j = 0; j < k; ++j) {
        if (residuals) residuals[j] = r.projected[j];
        if (true_residuals) true_residuals[j] = r.true_res[j];
        if (backward_errors) backward_errors[j] = r.backward[j];
    }
    if (!finite) throw Error(SBH_ERR_NUMERICAL, "block GMRES generated NaN or infinity in residual metrics");
    return SBH_OK;
}

}  // namespace sbh
