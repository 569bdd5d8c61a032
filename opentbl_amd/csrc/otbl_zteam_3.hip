// z kernels with several rows per wavefront: row lengths 338 to 600
#include "otbl_zteam_kernels.h"

namespace otbl {

bool zteam_part3(int n, ZTeamFns &f) { return team_find<338, 600>(n, f); }

} // namespace otbl
