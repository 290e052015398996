// Test access to a handle's kernel candidates (ldg.hip Cand, default_cand):
// the autotuner picks among them by time, tests pick them here.  Built with
// the library from the same headers; not part of the C ABI.
#include "handle.hpp"

extern "C" int ldg_test_candidates() { return ldg_host::kMaxCand; }

// The candidates of every order group from the next launch on.
extern "C" void ldg_test_set_candidates(ldg_handle *h, int grad, int rhs) {
  for (auto &g : h->groups) {
    g.cgrad = grad;
    g.crhs = rhs;
  }
}
