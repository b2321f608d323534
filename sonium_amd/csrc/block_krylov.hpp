// Least-squares problem of the block GMRES on the device, shared by its kernels
// and its driver.

#pragma once

#include "internal.hpp"

namespace sbh {

// What the host reads of a block step (pinned, written by the device).
struct BlockStep {
    int ok;            // 0: the Cholesky QR did not hold and nothing was added
    int next;          // directions the block's QR accepted
    double tail[64];   // residual norms of the right-hand sides
};

// min ||g - H y|| over the block Hessenberg columns added so far.
class BlockLeastSquares {
   public:
    BlockLeastSquares(sbh_context* ctx, int s, int max_basis, int max_steps);

    // Queues the outcome of a block QR of sj columns (chain null: the Cholesky one's).
    void report(const void* chol, const void* chain, int sj);
    // Queues g = [C0; 0], C0 s1 x s row-major on the device.
    void reset(const double2* c0, int s1);
    // Queues the sj columns of the next step: hacc (rows 0 .. columns() + sj - 1,
    // row-major) over the QR's factor.  Nothing is added where the Cholesky QR
    // did not hold; accept() follows where it did.
    void add(const void* chol, const void* chain, const double2* hacc, int sj);
    void accept(int sj) {
        done_ += 1;
        cols_ += sj;
    }
    // Queues y (columns() x s, row-major) of the columns added.
    void solve(double2* y);
    int columns() const { return cols_; }
    const BlockStep& host() const { return *host_.ptr; }  // after a synchronization

   private:
    sbh_context* ctx_;
    int s_, done_ = 0, cols_ = 0;
    int64_t ldg_;
    WorkArray<int2> steps_;
    WorkArray<double2> refl_, qh_, R_, window_, g_, work_;
    WorkArray<BlockStep, true> host_;
};

}  // namespace sbh
