// The launch rules behind C functions for tests/test_launch_rules.py.
#include "../../cannbench-operator-solutions_amd/csrc/launch_rules.hpp"

extern "C" {
int rule_grid_fits(int64_t blocks, int64_t threads) { return cb::grid_fits(blocks, threads); }
int64_t rule_dqsq_blocks(int64_t M, int64_t threads) { return cb::dqsq_blocks(M, threads); }
int rule_pick_deq(const int64_t* gl, int64_t E, int64_t M, int64_t K, int64_t N, int64_t batch, int ring_ok)
{
    return cb::pick_deq(gl, E, M, K, N, batch, ring_ok, 256);
}
int rule_pick_gmm(const int64_t* gl, int64_t E, int64_t M, int64_t K, int64_t N) { return cb::pick_gmm(gl, E, M, K, N, 256); }
int rule_gmsq_skips_empty(const int64_t* gl, int64_t E) { return cb::gmsq_skips_empty(gl, E); }
int64_t rule_gmsq_decode_grid(int64_t groups, int64_t ntl, int64_t cus) { return cb::gmsq_decode_grid(groups, ntl, cus); }
int rule_ring_skips_empty(const int64_t* gl, int64_t E) { return cb::ring_skips_empty(gl, E); }
}
