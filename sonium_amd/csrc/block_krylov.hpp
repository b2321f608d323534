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

// min ||g - H y|| over the block Hessenberg columns added so far, at most
// max_basis in max_steps steps.  A basis of an n-dimensional space has n
// directions as long as the numbers are good, so the arrays start with room for
// n + 2 s of them in n + 1 steps and grow when a step needs more: the rank-drop
// test measures a column against its norm after the projection, and once the
// basis fills the space (or the operator's range) the rounding errors left of a
// step pass it as new directions.
class BlockLeastSquares {
   public:
    BlockLeastSquares(sbh_context* ctx, int64_t n, int s, int max_basis, int max_steps);
    // Device bytes that allocate() takes in a solve of s columns on n rows.
    static int64_t device_bytes(int64_t n, int s, int64_t restart);
    void allocate();

    // Queues the outcome of a block QR of sj columns (chain null: the Cholesky one's).
    void report(const void* chol, const void* chain, int sj);
    // Queues g = [C0; 0], C0 s1 x s row-major on the device.
    void reset(const double2* c0, int s1);
    // Queues the sj columns of the next step: hacc (rows 0 .. columns() + sj - 1,
    // row-major) over the QR's factor.  Nothing is added where the Cholesky QR
    // did not hold; accept() follows where it did.
    void add(const void* chol, const void* chain, const double2* hacc, int sj);
    void accept(int sj);
    // Queues y (columns() x s, row-major) of the columns added.
    void solve(double2* y);
    int columns() const { return cols_; }
    const BlockStep& host() const { return *host_.ptr; }  // after a synchronization

   private:
    bool joins(int sj) const;  // a step of sj columns fits the last group's window
    static int64_t most_groups(int s, int64_t steps, int64_t cols);
    static int64_t room_bytes(int s, int64_t steps, int64_t cols);
    void make_room(int steps, int cols);

    sbh_context* ctx_;
    int64_t n_;
    int s_, done_ = 0, cols_ = 0;          // steps and columns added
    int ngroups_ = 0, open_ = 0;           // groups of steps, columns of the last
    int max_basis_, max_steps_;            // limits of a cycle
    int room_cols_ = 0, room_steps_ = 0;   // what the arrays hold
    int64_t ldg_ = 0;
    WorkArray<int4> groups_;
    WorkArray<double2> refl_, qh_, R_, window_, g_, work_;
    WorkArray<BlockStep, true> host_;
};

}  // namespace sbh
