// The plain render's kernels for scenes of several lights, kRender<BIG, false,
// true>, in a translation unit of their own like the sampled render's
// (cgs_render_sampled.hip): only they and their launcher (launchRenderLights)
// are emitted here.
#define CGS_LIGHTS_TU 1
#include "cgs_trace.hip"
