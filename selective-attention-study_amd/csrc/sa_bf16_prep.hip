// The backward preparation's bf16-storage instances (row statistics, the exempt keys' gradients), in a
// translation unit of their own: with sa_bf16.hip's options this compiler crashes on the head-dim-128
// instance, and its accumulators are not carried around a loop, so their placement does not matter.

#include "sa_kernels.h"

namespace sa_host {

void launch_rowprep_bf16(const BwdCall& c, const PrepLaunch& p) {
  if (c.head_dim == 32) launch_rowprep<OpBF16, 32>(c, p);
  else if (c.head_dim == 64) launch_rowprep<OpBF16, 64>(c, p);
  else launch_rowprep<OpBF16, 128>(c, p);
}

}  // namespace sa_host
