// The photon walk with its bounds as kernels that stage nothing have them:
// three arrays of their own, here 64 GiB apart, against the same walk with
// the three in one array.  A step that took one axis's bounds by their
// distance from another's read outside both.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../gegs_amd/csrc/event.hpp"

namespace gegs {
float lds_env[LDS_FLOATS];
}
using namespace gegs;

struct Push {
    void push(const Part &) {}
};

int main() {
    constexpr uint32_t N = 12;
    static gegs_media_tables mt;                     // zero: row 0 of medium 0 everywhere
    mt.gmfp[0] = {2.5f, 0.0f};
    mt.cohe[0] = {1.0f, 0.0f};
    gegs_region rec{0, 0, 1.0f, 0.0f, 0.0f};
    static uint16_t cls[N * N * N + VAC_AND_OTH];
    gegs_field field{};
    field.cos_angle = 1.0f;
    field.module_first = GEGS_M_PHANTOM;
    float *near[3];   // exactly N + 2 bounds each: a read beside them stops the run
    for (int a = 0; a < 3; ++a) {
        near[a] = (float *)malloc((N + 2) * sizeof(float));
        for (uint32_t i = 0; i < N + 2; ++i) near[a][i] = 0.5f * (float)i + 0.01f * (float)(a * i);
    }
    const size_t gap = (size_t)64 << 30;
    char *far = (char *)mmap(nullptr, 2 * gap + 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (far == MAP_FAILED) return 2;
    for (int a = 0; a < 3; ++a) memcpy(far + a * gap, near[a], (N + 2) * sizeof(float));
    Env env;
    env.mt = &mt;
    env.rcls = cls;
    env.rtab = &rec;
    env.pge = mt.ge;
    env.pgmfp = mt.gmfp;
    env.pcohe = mt.cohe;
    env.nx = env.ny = env.nz = N;
    env.nclass = 1;
    env.nmed = 1;
    env.fields = &field;
    env.njob = 1;
    env.mlc = nullptr;
    env.endnodes = nullptr;
    env.jaws = nullptr;
    env.mlc_next = env.jawx_next = GEGS_M_PHANTOM;
    env.seed = 9;
    const float dirs[6][3] = {{0.6f, 0.64f, 0.48f},   {-0.6f, 0.64f, -0.48f}, {0.0f, 0.6f, -0.8f},
                              {0.0f, 0.0f, 1.0f},     {-1.0f, 0.0f, 0.0f},    {0.36f, -0.48f, 0.8f}};
    for (int k = 0; k < 600; ++k) {
        Part out[2];
        uint32_t steps[2];
        for (int f = 0; f < 2; ++f) {
            env.xb = f ? (const float *)far : near[0];
            env.yb = f ? (const float *)(far + gap) : near[1];
            env.zb = f ? (const float *)(far + 2 * gap) : near[2];
            Part p{};
            p.e = 1.0f;
            p.x = p.y = p.z = 2.6f;
            p.u = dirs[k % 6][0];
            p.v = dirs[k % 6][1];
            p.w = dirs[k % 6][2];
            p.wt = 1.0f;
            p.module = GEGS_M_PHANTOM;
            p.leaf = OUTMLC;
            p.lin = 1000u + (uint64_t)k;
            p.spos = 4;
            p.region = VAC_AND_OTH + 5 + 5 * N + 5 * N * N;
            Stream s;
            s.begin(p, env.seed);
            Push sink;
            Tally t{};
            PhotonWalk w;
            photon_walk_begin(env, p, w);
            while (photon_walk_iter(env, s, p, w, sink, t) == PW_ON) {
            }
            photon_walk_leave(env, p, w);
            out[f] = p;
            steps[f] = t.steps;
        }
        if (steps[0] != steps[1] || out[0].region != out[1].region || out[0].x != out[1].x || out[0].y != out[1].y ||
            out[0].z != out[1].z) {
            printf("walk %d: %u and %u steps, regions %u and %u\n", k, steps[0], steps[1], out[0].region, out[1].region);
            return 1;
        }
    }
    printf("ok\n");
    return 0;
}
