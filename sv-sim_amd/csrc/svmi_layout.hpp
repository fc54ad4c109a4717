// svmi_layout.hpp -- register layouts of planned sweeps (host only).
#pragma once

#include "svmi_plan.hpp"

namespace svmi {

// Fills prog.io, lphases and cols for every sweep of prog.
void build_layouts(Program& prog);

}  // namespace svmi
