// pm355_route.h's choice of experts as it stands, on the CPU: the 64 lanes of a wave are 64 contexts that run in turn from one meeting point of the wave to the next. Compared with the rule in plain
// words: the largest scores first, equal ones by index; groups beyond the kept ones have a score of -1 and no weight; a row without comparable scores names experts that exist, with a weight of 0.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <ucontext.h>
#include <algorithm>
#include <random>
#include <vector>

static struct { unsigned x; } threadIdx;
static ucontext_t host, lanes[64];
static char stacks[64][64 * 1024];
static int n_lanes_done;
static float slots[64];
static bool bits[64];
static void (*body)();

// a lane waits until all have come
static void meet() { const unsigned l = threadIdx.x; swapcontext(&lanes[l], &host); threadIdx.x = l; }
template <class T, class F> static T together(T (&slot)[64], T v, F && f) {
    slot[threadIdx.x] = v;
    meet();
    const T r = f();
    meet();
    return r;
}
static float wave_max(float v) { return together(slots, v, [] { float m = slots[0]; for (int i = 1; i < 64; ++i) m = fmaxf(m, slots[i]); return m; }); }
static float wave_sum(float v) { return together(slots, v, [] { float s = 0.0f; for (float x : slots) s += x; return s; }); }
static uint64_t ballot(bool v) {
    bits[threadIdx.x] = v;
    meet();
    uint64_t m = 0;
    for (int i = 0; i < 64; ++i) m |= (uint64_t) bits[i] << i;
    meet();
    return m;
}
#define __HIPCC__
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_fence(order, scope) ((void) 0)
#define __builtin_amdgcn_wave_barrier() meet()
#define __builtin_amdgcn_ballot_w64(v) ballot(v)
#include "pm355_route.h"

static struct { const float * z; int E, top, groups, keep; float s[1024], gs[1024], w[64]; int ids[64]; } a;
static void lane_main() { body(); ++n_lanes_done; }
static void wave() {
    body = [] { route_token([](int e) { return a.z[e]; }, a.E, a.top, a.groups, a.keep, a.s, a.gs, a.ids, a.w); };
    n_lanes_done = 0;
    for (int l = 0; l < 64; ++l) {
        getcontext(&lanes[l]);
        lanes[l].uc_stack.ss_sp = stacks[l]; lanes[l].uc_stack.ss_size = sizeof(stacks[l]); lanes[l].uc_link = &host;
        makecontext(&lanes[l], lane_main, 0);
    }
    while (n_lanes_done < 64) for (int l = 0; l < 64; ++l) { threadIdx.x = (unsigned) l; swapcontext(&host, &lanes[l]); }
}

int main() {
    std::mt19937 rng(1);
    std::normal_distribution<float> normal;
    const float inf = INFINITY, nan = NAN;
    struct Form { int E, top, groups, keep; };
    std::vector<Form> forms;
    for (int E : {1, 2, 5, 31, 32, 33, 63, 64, 65, 100})
        for (int top : {1, 4, 8, E})
            if (top <= E && top <= 64) forms.push_back({E, top, 1, 1});
    for (Form f : {Form{32, 4, 8, 3}, Form{33, 7, 11, 4}, Form{6, 4, 3, 1}, Form{64, 8, 4, 2}, Form{63, 9, 7, 1}, Form{96, 6, 8, 2}}) forms.push_back(f);
    int rows = 0, bad = 0;
    for (const Form & f : forms)
        for (int kind = 0; kind < 10; ++kind) {
            std::vector<float> z(f.E), p(f.E);
            for (float & v : z) v = kind == 1 ? (float) (int) (rng() % 3) : kind == 2 ? 0.5f : kind == 3 ? 300.0f * normal(rng) : normal(rng);
            const int at = (int) (rng() % (unsigned) f.E);
            if (kind == 4) z[at] = nan;
            if (kind == 5) z.assign(f.E, nan);
            if (kind == 6) z[at] = inf;
            if (kind == 7) z.assign(f.E, -inf);
            if (kind == 8) z[at] = -inf;
            if (kind == 9) z[at] = -nan;
            a.z = z.data(); a.E = f.E; a.top = f.top; a.groups = f.groups; a.keep = f.keep;
            for (int k = 0; k < 64; ++k) { a.ids[k] = -7; a.w[k] = -7.0f; }
            wave();
            float mx = -inf, sum = 0.0f, lane[64] = {};
            for (float v : z) mx = fmaxf(mx, v);
            for (int e = 0; e < f.E; ++e) { p[e] = expf(z[e] - mx); lane[e % 64] += p[e]; }
            for (float v : lane) sum += v;
            for (float & v : p) v /= sum;
            const int per = f.E / f.groups;
            std::vector<int> g(f.groups), want(f.E);
            auto best = [&](int i) { float m = p[i * per]; for (int j = 1; j < per; ++j) m = fmaxf(m, p[i * per + j]); return m; };
            for (int i = 0; i < f.groups; ++i) g[i] = i;
            if (sum == sum) {
                std::stable_sort(g.begin(), g.end(), [&](int x, int y) { return best(x) > best(y); });
                for (int i = f.keep; i < f.groups; ++i) for (int j = 0; j < per; ++j) p[g[i] * per + j] = -1.0f;
            }
            for (int i = 0; i < f.E; ++i) want[i] = i;
            if (sum == sum) std::stable_sort(want.begin(), want.end(), [&](int x, int y) { return p[x] > p[y]; });
            for (int k = 0; k < f.top; ++k) {
                const bool any = sum == sum;
                const int id = any ? want[k] : 0;
                const float w = any ? std::max(p[id], 0.0f) : 0.0f;
                if ((any ? a.ids[k] != id : a.ids[k] < 0 || a.ids[k] >= f.E) || a.w[k] != w) {
                    if (++bad <= 20) printf("E %d top %d groups %d keep %d kind %d slot %d: expert %d weight %g, wanted %d %g\n", f.E, f.top, f.groups, f.keep, kind, k, a.ids[k], a.w[k], id, w);
                }
            }
            for (int k = f.top; k < 64; ++k) if (a.ids[k] != -7) { ++bad; printf("E %d top %d: slot %d written\n", f.E, f.top, k); break; }
            ++rows;
        }
    printf("%d rows, %d wrong\n", rows, bad);
    return bad != 0;
}
