// z kernels with several rows per wavefront: row lengths 162 to 336
#include "otbl_zteam_kernels.h"

namespace otbl {

bool zteam_part2(int n, ZTeamFns &f) { return team_find<162, 336>(n, f); }

} // namespace otbl
