// The RDMA slot kernel for gfx950. A world runs on a team of T workgroups (256 threads, 4 waves
// each) for all of its slots; teams take worlds from a queue, longest first. In a slot the world's
// work items are dealt over the team's waves: a host item is up to hpw hosts side by side (a lane
// runs one host's events, src/rdma/rstep.cuh:1649-2112), a switch item is one switch on one wave or workgroup
// (its ports in LDS; a safe slot runs each egress port's events on a lane of its own, otherwise lane
// 0 runs them all; rdma_model.h switch_slot). Entities only read what earlier slots filed
// (src/rdma/rdma.h:12-16), so a slot needs one team barrier; the last workgroup to arrive decides the
// next slot (slot_end: finish, idle skip). A launch ends when the queue is empty or its time (about
// a second) is up; the host launches again for the worlds left.
#include <hip/hip_runtime.h>
#include "rdma_model.h"
#include "rdma_kernel.h"

namespace rd
{
constexpr long long LAUNCH_TICKS = 100000000;          // a launch's time: 1 s of the 100 MHz constant clock
constexpr unsigned long long WAIT_TICKS = 2000000000ull; // a barrier wait gives up after 20 s
constexpr int WAVES = LAUNCH_WAVES;                    // waves of a 256-thread workgroup

// (Four waves' workspaces of LDS: one workgroup per CU, one wave per SIMD, so all registers may be used.)
// A host item: `hpw` hosts side by side, lane i's events are host e0 + i's. The lanes share out the
// copying of the hosts' arrivals into their workspaces and of the frames sent out of them, 64 / hpw
// lanes a host: one round of loads and one of stores a slot, off the hosts' chains of events (24
// FatTree k=8 worlds as one batch 181 -> 156 ms of kernel; worlds alone, whose items have a host or
// two, within 3%: there the events' own instructions bound the item).
__device__ __forceinline__ bool host_item(SimRef s, int e0, int n, int hpw, int64_t slot, unsigned *flows_done, uint32_t *pend, int pend_n,
                                          int64_t *wake, char *mem, int lane)
{
    const int per = WAVE_LDS / hpw & ~15, group = 64 / hpw, mine = lane / group, words = (int)(sizeof(LFrame) / 8);
    HostSlot x = {false, 0, 0};
    if (lane < n)
        x = host_open(s, e0 + lane, slot, wake);
    const HostWork w = host_work(mem + (size_t)(lane < hpw ? lane : 0) * per, per);
    const int in_n = x.an < w.in_cap ? x.an : w.in_cap;
    {
        const HostWork g = host_work(mem + (size_t)(mine < hpw ? mine : 0) * per, per);
        const int k = __shfl(in_n, mine < hpw ? mine : 0) * (mine < hpw ? words : 0);
        const uint64_t at = __shfl(x.abase, mine < hpw ? mine : 0);
        for (int i = lane % group; i < k; i += group)
            in_word(g.in[i / words], i % words, in_load(s, at + i / words, i % words));
    }
    RD_WAVE_SYNC();
    bool act = false;
    int out_n = 0;
    if (x.runs)
        act = host_events(s, e0 + lane, slot, flows_done, pend, pend_n, wake, x.an, x.abase, w, in_n, &out_n);
    RD_WAVE_SYNC();
    {
        const HostWork g = host_work(mem + (size_t)(mine < hpw ? mine : 0) * per, per);
        const int k = __shfl(out_n, mine < hpw ? mine : 0) * (mine < hpw ? words : 0);
        for (int i = lane % group; i < k; i += group)
            out_store(g.out[i / words], i % words);
    }
    RD_WAVE_SYNC(); // (the workspace is reused by the next item)
    return act;
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) rdma_team_kernel(const LaunchCfg *__restrict__ lp)
{
    const LaunchCfg L = *lp;
    __shared__ __attribute__((aligned(16))) char work[WAVES][WAVE_LDS];
    __shared__ int64_t s_slot;
    __shared__ int s_w, s_stop, s_err;
    __shared__ unsigned s_act;
    __shared__ unsigned long long s_wake;
    // (the wave's number made a scalar: what a wave's item indexes is then loaded by scalar loads)
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int T = L.T;
    // a team's workgroups have consecutive ids, so they spread over the 8 XCDs (workgroups reach
    // the XCDs round-robin by id). Teams kept on one XCD each were measured slower: the reference's
    // 80 short RDMA jobs as one batch 13.0 s against 9.7 s, the 36 medium ones 21.9 s against 18.7 s.
    const int team = blockIdx.x / T, rank = blockIdx.x % T;
    TeamState *ts = L.teams + team;
    const long long t_launch = wall_clock64();
    unsigned gen = 0;

    // the team barrier; the last workgroup to arrive runs `last` first, whose stores are device-coherent
    // (a fenced barrier's release is ahead of it). Within a world (fenced
    // false) it has no cache fences: what the workgroups hand each other goes through coherent
    // accesses (rdma_model.h), so each wave only waits for its own stores to complete, and the
    // entities' own records stay in the caches from slot to slot (an agent-scope fence on the
    // multi-XCD GPU writes back and invalidates the L2). Claiming a world and leaving one are fenced.
    auto barrier = [&](auto last, bool fenced) -> bool {
        __builtin_amdgcn_s_waitcnt(0); // (this wave's stores have completed)
        __syncthreads();
        if (tid == 0)
        {
            if (fenced)
                __threadfence();
            if (T == 1)
                last();
            else
            {
                const unsigned g = gen;
                if (atomicAdd(&ts->arrive, 1u) == (unsigned)T - 1)
                {
                    last();
                    atomicExch(&ts->arrive, 0u);
                    __builtin_amdgcn_s_waitcnt(0); // (the ticket's stores before the release of the others)
                    atomicAdd(&ts->gen, 1u);
                }
                else
                {
                    const unsigned long long w0 = wall_clock64();
                    while (coh_load(&ts->gen) == g)
                    {
                        __builtin_amdgcn_s_sleep(1);
                        if (wall_clock64() - w0 > WAIT_TICKS)
                        {
                            atomicExch(&ts->err, 1);
                            break;
                        }
                    }
                }
                gen = g + 1;
            }
            if (fenced)
                __threadfence();
            s_err = T > 1 && __hip_atomic_load(&ts->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        return s_err;
    };

    for (;;)
    {
        // the team's next world (none once the launch's time is up: the host launches again)
        if (barrier([&] {
                ts->world.set(wall_clock64() - t_launch > LAUNCH_TICKS ? L.nq : (int)atomicAdd(L.qnext, 1u));
                ts->act.set(0);
                ts->wake.set(~0ull);
                ts->stop.set(0);
            }, true))
            return;
        if (tid == 0)
            s_w = ts->world.get();
        __syncthreads();
        if (s_w >= L.nq)
            return;
        const int qe = __builtin_amdgcn_readfirstlane(L.queue[s_w]), w = qe & ((1 << QSHIFT) - 1);
        const uint64_t sp = (uint64_t)L.sims[qe >> QSHIFT];
        // (the Sim record through a scalar pointer in the constant address space: its fields are
        // scalar loads; through a generic one every use of a field was a flat load, which waits for
        // the stores before it)
        SimRef s = *(const Sim RD_C *)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(sp >> 32)) << 32 |
                                       (uint32_t)__builtin_amdgcn_readfirstlane((int)sp));
        const World wd = s.wd[w];
        WorldRun &r = s.run[w];
        uint32_t *pend = s.pend + wd.pend_off;
        const int hpw = L.hpw, nhw = host_items(wd.nh, hpw);
        // Work items: a wave each, or, where the team has the workgroups (runs_by_group), a switch for a
        // whole workgroup (its ports over four waves: a wave's lanes run unlike events one after
        // another, so fewer ports a wave is a shorter slot: FatTree k=8 a2a, HPCC, the longest switch of
        // a slot 191 us on a wave, 134 us on four) and a host item for each of its waves.
        const bool by_group = L.by_group && runs_by_group(wd.nh, wd.ns, hpw, T);
        const int ngh = (nhw + WAVES - 1) / WAVES;
        const int first = by_group ? rank : rank * WAVES + wv, step = by_group ? T : T * WAVES;
        const int hosts = by_group ? ngh : nhw, items = hosts + wd.ns;
        const long long t_world = wall_clock64();
        for (;;)
        {
            if (tid == 0)
            {
                s_slot = __hip_atomic_load(&r.slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                s_stop = __hip_atomic_load(&r.finished, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ||
                         ts->stop.get();
                s_act = 0;
                s_wake = ~0ull;
            }
            __syncthreads();
            if (s_stop)
                break;
            const int64_t sl = s_slot;
            unsigned a = 0;
            unsigned long long wk = ~0ull;
#ifdef RD_PROF
            long long p0 = wall_clock64(), ph = 0, psw = 0;
#endif
            for (int it = first; it < items; it += step)
            {
#ifdef RD_PROF
                const long long q0 = wall_clock64();
#endif
                if (it < hosts)
                {
                    const int hi = by_group ? it * WAVES + wv : it;
                    const int e0 = hi * hpw, n = wd.nh - e0 < hpw ? wd.nh - e0 : hpw;
                    int64_t hw = INT64_MAX;
                    if (n > 0)
                        a |= host_item(s, wd.h0 + e0, n, hpw, sl, &r.flows_done, pend, wd.pend_n, &hw, work[wv], lane) ? 1u : 0u;
                    if (hw != INT64_MAX && (unsigned long long)hw < wk)
                        wk = (unsigned long long)hw;
                }
                else
                {
                    const int x = wd.s0 + (it - hosts);
                    const int deg = s.si[x].deg;
                    bool busy = false;
                    const bool run = s.sw_busy[x] || __any(switch_has_input(s, x, sl, lane, 64));
                    if (by_group)
                    {
                        // (every wave has looked before the first sync, and the switch is this workgroup's alone)
                        __syncthreads();
                        if (run)
                            busy = switch_slot_by(s, x, sl, pend, wd.pend_n, &work[0][0], WAVES * WAVE_LDS, lane * WAVES + wv, 64 * WAVES,
                                                  [] { __syncthreads(); });
                    }
                    else if (run)
                    {
                        if (deg <= KS)
                            busy = switch_slot(s, x, sl, pend, wd.pend_n, *reinterpret_cast<SwWork *>(work[wv]), lane, 64);
                        else if (deg <= KW && L.wide)
                            busy = switch_slot(s, x, sl, pend, wd.pend_n, L.wide[(size_t)blockIdx.x * WAVES + wv], lane, 64);
                        else
                        {
                            int b = 0;
                            if (lane == 0)
                                b = switch_step(s, x, sl, pend, wd.pend_n) ? 1 : 0;
                            busy = __shfl(b, 0) != 0;
                        }
                    }
                    if (lane == 0 && (!by_group || wv == 0))
                    {
                        s.sw_busy[x] = busy ? 1 : 0;
                        a |= busy ? 1u : 0u;
                    }
                }
#ifdef RD_PROF
                (it < hosts ? ph : psw) += wall_clock64() - q0;
#endif
            }
#ifdef RD_PROF
            // (profiling builds: the waves' host and switch item time, and the time to the slot's end)
            if (lane == 0)
            {
                atomicMax(&ts->prof[0], (unsigned long long)ph);
                atomicMax(&ts->prof[1], (unsigned long long)psw);
                if (ph)
                    atomicAdd(&s.ev[33], (unsigned long long)ph);
                if (psw)
                    atomicAdd(&s.ev[34], (unsigned long long)psw);
            }
            const long long pb = wall_clock64();
            (void)p0;
#endif
            if (a)
                atomicOr(&s_act, a);
            if (wk != ~0ull)
                atomicMin(&s_wake, wk);
            __syncthreads();
            // this workgroup's share joins the team's before it arrives at the barrier
            if (tid == 0)
            {
                if (s_act)
                    atomicOr(ts->act.at(), s_act);
                if (s_wake != ~0ull)
                    atomicMin(ts->wake.at(), s_wake);
            }
            if (barrier([&] {
#ifdef RD_PROF
                    atomicAdd(&s.ev[22], atomicExch(&ts->prof[0], 0ull));
                    atomicAdd(&s.ev[23], atomicExch(&ts->prof[1], 0ull));
#endif
                    slot_end(s, wd, r, pend, atomicOr(ts->act.at(), 0u), atomicMin(ts->wake.at(), ~0ull));
                    ts->act.set(0);
                    ts->wake.set(~0ull);
                    if (wall_clock64() - t_launch > LAUNCH_TICKS)
                        ts->stop.set(1);
                }, false))
                return;
#ifdef RD_PROF
            if (tid == 0 && rank == 0)
                atomicAdd(&s.ev[35], (unsigned long long)(wall_clock64() - pb));
#endif
        }
        if (tid == 0 && rank == 0)
            r.ticks += wall_clock64() - t_world;
    }
}

int launch_capacity(int threads)
{
    int dev = 0, per_cu = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, rdma_team_kernel, threads, 0) != hipSuccess)
        return -1;
    return per_cu * cus;
}

int launch_worlds(const LaunchCfg *cfg_dev, int nblocks, int threads, hipStream_t st)
{
    hipLaunchKernelGGL(rdma_team_kernel, dim3(nblocks), dim3(threads), 0, st, cfg_dev);
    return (int)hipGetLastError();
}
} // namespace rd
