// Internal declarations shared by the npbcg translation units.
#ifndef NPBCG_INTERNAL_H
#define NPBCG_INTERNAL_H

#include <string>

namespace npbcg_detail {

// Records `msg` as this thread's last error and returns `code`.
int set_error(int code, const std::string &msg);
void clear_error();

// Worker threads of the generator used by npbcg_makea calls from the calling
// thread (0: the default, NPBCG_GEN_THREADS or up to 16).
void set_generator_threads(int threads);

}  // namespace npbcg_detail

struct npbcg_ctx;

// For tests of the resident engine's fallback: in the calls that follow, the
// launch that holds outer iteration `iteration` (0: conj_grad, a solve) waits
// for a word that nobody stores until its bounded wait runs out, a hundredth
// of the limit other launches have, and then ends as any launch does.  -1:
// none.  Also ends the device's rest after a launch that gave up.
// NPBCG_ERR_INVALID where the context does not run on that engine, or its order
// leaves no word of the exchange buffers unused.
extern "C" int npbcg_test_resident_give_up(npbcg_ctx *c, int iteration);

// For tests: while on, device buffers that a call of this context would add to
// run faster cannot be had, as on a full device.
extern "C" int npbcg_test_no_memory(npbcg_ctx *c, int on);

// For tests: the solve sequences that the context has captured as graphs.
extern "C" int npbcg_test_solve_graphs(npbcg_ctx *c);

#endif
