// Host build of haissinskijulia_amd/csrc/hm_rules.hpp for tests/test_rules.py.
#include "../haissinskijulia_amd/csrc/hm_rules.hpp"

extern "C" {
int64_t t_max_slabs(int64_t ntiles, int64_t ppt, int cus) { return hm::max_slabs(ntiles, ppt, cus); }
}
