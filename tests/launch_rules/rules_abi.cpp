// The launch rules behind C functions for tests/test_launch_rules.py.
#include "../../cannbench-operator-solutions_amd/csrc/launch_rules.hpp"

extern "C" {
int rule_grid_fits(int64_t blocks, int64_t threads) { return cb::grid_fits(blocks, threads); }
int64_t rule_dqsq_blocks(int64_t M, int64_t threads) { return cb::dqsq_blocks(M, threads); }
}
