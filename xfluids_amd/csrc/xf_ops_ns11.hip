// Kernel instances for 11 species other than the sweeps (xf_sweeps.hip): states,
// viscous terms and chemistry, and the dispatch table.  One translation unit per
// species count so the build runs them in parallel.
#include "xf_context.h"

namespace xf {

Ops ops_ns11() { return Launch<11, true>::ops(); }

} // namespace xf
