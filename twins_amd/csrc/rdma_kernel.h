// The RDMA slot kernel's launch, between the host side (rdma_core.cpp) and the kernel
// (rdma_kernel.hip; a CPU build of the same steps replaces it in the CPU check).
#pragma once
#include <hip/hip_runtime_api.h>
#include "rdma_model.h"

namespace rd
{
// a team's barrier and its world's slot decisions (device memory, zeroed before a launch)
struct TeamState
{
    unsigned arrive, gen;
    twc::CohWord<int> world;
    int err;
    twc::CohWord<unsigned> act;
    twc::CohWord<int> stop;
    twc::CohWord<unsigned long long> wake;
    unsigned long long prof[2]; // (profiling builds: the slot's longest host and switch items)
};
// one launch: teams of T workgroups take worlds queue[0 .. nq) in order (qnext: the next index);
// an entry is sim << QSHIFT | world: world `world` of the batch whose Sim is sims[sim] (a launch can
// run the worlds of several separately packed batches: the serving loop's requests)
constexpr int QSHIFT = 20;
constexpr int LAUNCH_WAVES = 4; // waves of a launch's 256-thread workgroups
struct LaunchCfg
{
    int T, nq, hpw; // hpw: hosts of a host item (side by side on a wave's lanes, at most 64)
    int by_group;   // 1: a world's switches run on a whole workgroup each where runs_by_group says so (0: never)
    const int *queue;
    unsigned *qnext;
    TeamState *teams;
    const Sim *const *sims;
    SwWorkWide *wide; // a device-memory switch workspace per wave of the launch (null: no switch of KS + 1 to KW ports)
};
// A world's work items, its hosts in items of hpw: a wave each, or by workgroup (a switch for a whole
// workgroup, a host item for each of its waves).
RD_HD int host_items(int hosts, int hpw) { return (hosts + hpw - 1) / hpw; }
RD_HD int wave_items(int hosts, int switches, int hpw) { return host_items(hosts, hpw) + switches; }
RD_HD int group_items(int hosts, int switches, int hpw) { return switches + (host_items(hosts, hpw) + LAUNCH_WAVES - 1) / LAUNCH_WAVES; }
// Does a team of T workgroups run the world by workgroup? Where all of it fits side by side: with a second
// round of workgroups a slot takes longer than with a wave each (kernel time by workgroup up to three
// rounds, and side by side only: FatTree k=16 (DCQCN) alone on 128 workgroups 62 and 38.5 ms, two k=16
// worlds 73 and 54, four k=8 worlds 39 and 30, 101 uneven ones on teams of 8 217 and 155; nothing of
// 17 batches was slower).
RD_HD bool runs_by_group(int hosts, int switches, int hpw, int T) { return group_items(hosts, switches, hpw) <= T; }

// The launch shape: one team size and hosts per host item. Every world that fits runs at once, each
// on its share of the GPU (worlds queued behind others leave it idle when few are left). A slot
// lasts as long as its longest item, and a wave runs unlike hosts one after another, so the fewest
// hosts per item (a power of two) of these: a switch a workgroup and four host items a workgroup,
// all side by side; else every item on a wave of its own; else every host item. Measured (kernel
// time): 24 FatTree k=8 worlds of 128 hosts (DCQCN, HPCC and DCTCP) 145 ms on teams of 16 at 64
// hosts per item (16 worlds at once), 88, 84 and 90 ms on teams of 10 at 2, 4 and 8 hosts; FatTree
// k=8 (HPCC) alone 104, 85 and 85 ms on 128 workgroups at 2 and 112 and 208 at 1; two 512-host
// leaf-spines 124, 107 and 121 ms on 128 workgroups each at 1, 2 and 4.
// A world alone takes at most half of the GPU (as one of the TCP model does), so that two callers'
// are resident together: a team of which a part waits for a place waits at its barrier meanwhile.
constexpr int ALONE = 128;
struct LaunchShape
{
    int T, hpw;
};
// of W worlds on a GPU that holds cap workgroups; grouped: switches may run by workgroup; team_blocks,
// hpw: as asked for (0: automatic)
inline LaunchShape launch_shape(const int *hosts, const int *switches, int W, int cap, bool grouped, int team_blocks, int hpw)
{
    const int share = W == 1 ? (cap < ALONE ? cap : ALONE) : cap / W > 1 ? cap / W : 1;
    int T = team_blocks <= 0 ? share : team_blocks < cap ? team_blocks : cap;
    for (int rule = grouped ? 0 : 1; hpw <= 0 && rule < 3; rule++)
        for (int h = 1; hpw <= 0 && h <= 64; h *= 2)
        {
            bool fits = true;
            for (int i = 0; i < W; i++)
                fits = fits && (rule == 0   ? group_items(hosts[i], switches[i], h) <= T
                                : rule == 1 ? wave_items(hosts[i], switches[i], h) <= LAUNCH_WAVES * T
                                            : host_items(hosts[i], h) <= LAUNCH_WAVES * T);
            if (fits)
                hpw = h;
        }
    hpw = hpw > 0 ? hpw : 64;
    int most = 1; // (no more workgroups than the largest world has items)
    for (int i = 0; i < W; i++)
    {
        const int n = grouped ? group_items(hosts[i], switches[i], hpw) : wave_items(hosts[i], switches[i], hpw);
        most = n > most ? n : most;
    }
    if (team_blocks <= 0 && T > most)
        T = most;
    return {T, hpw};
}

// the workgroups of 256 threads the GPU holds at once (-1: unknown)
int launch_capacity(int threads);
// one launch of nblocks workgroups (teams of cfg->T); cfg_dev is a device copy; 0 or a hipError_t
int launch_worlds(const LaunchCfg *cfg_dev, int nblocks, int threads, hipStream_t st);
} // namespace rd
