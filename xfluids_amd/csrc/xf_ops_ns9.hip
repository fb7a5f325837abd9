// Kernel instances for 9 species other than the sweeps (xf_sweeps.hip): states,
// viscous terms and chemistry, and the dispatch table.  One translation unit per
// species count so the build runs them in parallel.
#include "xf_context.h"

namespace xf {

Ops ops_ns9() { return Launch<9, true>::ops(); }

} // namespace xf
