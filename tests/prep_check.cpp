// The host half of scene creation by itself (validation, tables, tree), built
// for the CPU tests: prep() runs prepare_scene and reports its time and a few
// sizes.
#include <chrono>
#include <cstring>

#include "../povray_amd/csrc/scene_prep.h"

static pvx::HostScene g_scene;

extern "C" int prep(const pvx_scene_desc *d, const pvx_build_opts *o, double *ms, uint64_t *sizes, char *msg) {
    g_scene = pvx::HostScene();
    std::string err;
    const auto t = std::chrono::steady_clock::now();
    const int r = pvx::prepare_scene(*d, o, g_scene, err);
    *ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t).count();
    std::strncpy(msg, err.c_str(), 255);
    sizes[0] = g_scene.prims.size();
    sizes[1] = g_scene.nodes.size();
    sizes[2] = g_scene.depth;
    sizes[3] = g_scene.inf.size();
    return r;
}
