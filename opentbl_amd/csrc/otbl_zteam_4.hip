// z kernels with several rows per wavefront: row lengths 602 to 1024
#include "otbl_zteam_kernels.h"

namespace otbl {

bool zteam_part4(int n, ZTeamFns &f) { return team_find<602, 1024>(n, f); }

} // namespace otbl
