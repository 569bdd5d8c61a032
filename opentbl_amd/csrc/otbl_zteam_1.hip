// z kernels with several rows per wavefront: row lengths 12 to 160
#include "otbl_zteam_kernels.h"

namespace otbl {

bool zteam_part1(int n, ZTeamFns &f) { return team_find<12, 160>(n, f); }

} // namespace otbl
