// mla_screen_probe.hip -- the batched screens in their probe form: every
// screened value goes to memory, for tests that hold the screen's bound pair
// by pair (grm_mla_hip_probe_screen).  A code object of its own
// (mla_screen.hpp).
#include "mla_screen.hpp"

namespace grm {
namespace mla {

int launch_probe_screen(const ScreenLaunch& l) { return launch_screen<true>(l); }

}  // namespace mla
}  // namespace grm
