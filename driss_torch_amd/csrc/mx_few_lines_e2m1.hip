// The e2m1 instantiations of the kernel in mx_few_lines_kernels.hpp.
#include "mx_few_lines_kernels.hpp"

namespace dt {

int launch_few_lines_e2m1(const FewLinesArgs& p, bool ragged, int octets) { return few_lines::launch_rows<true>(p, ragged, octets); }

}  // namespace dt
