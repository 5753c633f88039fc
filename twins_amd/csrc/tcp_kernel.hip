// The TCP slot kernels for gfx950.
//
// tcp_worlds_kernel: a persistent world-queue kernel run by teams of T workgroups. A team takes
// the next world from the batch's queue and runs its slots one after another until the world
// finishes or the launch's slot budget is spent. Within a slot the team's wavefronts share the
// world's entities: "work items" are groups of `hpw` hosts (one serial event loop per lane) and
// groups of 64/k switches (one lane per port), dealt round-robin over the team's waves, with no
// barrier between hosts and switches: both read only the two previous slots' link messages and
// write their own links' message for this slot (reference: src/kernel.cuh:5-113). The slot ends
// with the team barrier, whose last arrival is the ticket (finish test, exact idle-slot skip).
//
// The launch plan gives each team its size T, its workgroups and the queue of worlds it takes
// from, so one launch can run small worlds a workgroup each and large ones over many CUs.
// T = 1 needs only the workgroup barrier, so a world's state stays within one CU. T > 1
// synchronises through agent-scope words per team, one round trip a slot (TeamState, SlotGo); the grid is
// at most what the GPU holds at once, so all of a team's workgroups are resident, and every wait
// is bounded (a timeout ends the world with an error flag instead of hanging the queue). Each world's team
// accounts the device clock time it spent on it (WorldRun::ticks), the input of the autotuner.
#include <mutex>

#include "tcp_model.h"
#include "tcp_kernel.h"

namespace tw
{

// A wave's LDS, for the item it runs (one after another, so the items share it): a switch item's
// rows, in_win, base, cnt, sort and route slots; a host item's slots for its hosts' first frames out,
// an equal share each. Four waves take the CU's 160 KB but for the workgroup's own words.
constexpr int WAVE_LDS = 40704; // bytes
constexpr int LDS_PER_WAVE = WAVE_LDS / 4;
static_assert(Model<9>::SW_LDS_TOTAL * 4 <= WAVE_LDS, "a wave's LDS");
static_assert(4 * (size_t)WAVE_LDS + 512 <= 160 * 1024, "a 256-thread workgroup's LDS");
constexpr unsigned long long WAIT_TICKS = 2000000000ull;  // a team-barrier wait gives up after 20 s (100 MHz clock)
constexpr unsigned long long SERVER_MAX_WAIT = (unsigned long long)(SERVER_WAIT_S * 100e6); // (100 MHz clock)

__device__ __forceinline__ unsigned ld_acquire(const unsigned *p) { return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT); }

template <typename T>
__device__ __forceinline__ T *uniform_ptr(T *p)
{
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (T *)((uint64_t)hi << 32 | lo);
}

// The world loop of both persistent kernels: SRV = false takes worlds from a batch's queues
// (tcp_worlds_kernel), SRV = true takes requests from the serving loop's queues
// (tcp_server_kernel). One body, specialised at compile time, so the batch kernel carries nothing
// of the server's.
// ONE: every world's host items are of one host (Model::U).
template <int RUNS, bool SRV, bool ONE>
__device__ __forceinline__ void world_loop(const BatchT<RUNS> *__restrict__ Bp, const ServerCtl *__restrict__ Sp, int64_t slot_budget)
{
    typedef Model<RUNS, SRV> Md;
    typedef Model<RUNS, SRV, ONE> Mh; // the hosts'
    extern __shared__ __attribute__((aligned(128))) int lds[];
    __shared__ int s_w;
    __shared__ int64_t s_t;
    __shared__ int s_err;
    __shared__ unsigned s_act, s_flags;
    __shared__ unsigned long long s_wake;
    __shared__ const BatchT<RUNS> *s_b;
    __shared__ int s_id; // (serving: the request's id)
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = blockDim.x >> 6;
    const int32_t *team_of = SRV ? Sp->team_of : Bp->team_of;
    const TeamPlan *plans = SRV ? Sp->plan : Bp->plan;
    const int team = team_of[blockIdx.x] >> 8;
    const TeamPlan P = plans[team];
    const int T = P.T, rank = team_of[blockIdx.x] & 255;
    const int TW = T * nwaves, gw = rank * nwaves + wv; // the team's waves; this wave's place
    TeamState *ts = (SRV ? Sp->teams : Bp->teams) + team;
    int *wl = lds + wv * LDS_PER_WAVE;
    const int gwave = blockIdx.x * nwaves + wv; // this wave's global scratch
    int64_t *scr_ts = (SRV ? Sp->scr_ts : Bp->scr_ts) + (size_t)gwave * 64 * 2 * MAX_TX;
    uint32_t *scr_ref = (SRV ? Sp->scr_ref : Bp->scr_ref) + (size_t)gwave * 64 * 2 * MAX_TX;
    uint8_t *scr_up = (SRV ? Sp->scr_up : Bp->scr_up) + (size_t)gwave * 64 * 2 * MAX_TX;
    unsigned gen = 0; // the team barrier's generation this block has passed
    unsigned slot_count = 0; // slots run in this launch (thread 0)
    // a barrier wait's limit; the server's claim waits as long as a request may take to come
    unsigned long long wait_limit = WAIT_TICKS;

    // The barrier at a world's start and end; the last workgroup to arrive runs `last` first, whose
    // stores are device-coherent (the release is ahead of it). Agent-scope release and acquire, so that
    // the world's records, written with plain stores, are in memory when it ends and no stale copy is
    // read when it starts. The barrier between slots
    // (the end of the slot loop) has no cache fence: what workgroups hand each other from slot to
    // slot goes through device-coherent accesses only (coh_load / coh_store, tcp_state.h), so it is
    // enough that every wave's stores have completed (s_waitcnt) before its workgroup arrives; the
    // caches, and each entity's records in them, stay warm from slot to slot.
    auto team_barrier = [&](auto last) -> bool {
        __builtin_amdgcn_s_waitcnt(0); // (this wave's stores have completed)
        __syncthreads();
        if (tid == 0)
        {
            __threadfence();
            if (T == 1)
                last();
            else
            {
                unsigned g = gen;
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
                        if (wall_clock64() - w0 > (SRV ? wait_limit : WAIT_TICKS))
                        {
                            atomicExch(&ts->err, 1);
                            break;
                        }
                    }
                }
                gen = g + 1;
            }
            __threadfence();
            s_err = T > 1 && __hip_atomic_load(&ts->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        return s_err;
    };

    for (;;)
    {
        int w = 0;
        if constexpr (!SRV)
        {
            // the team's next world, from its queue
            if (team_barrier([&] { ts->world.set(atomicAdd(Bp->queue_next + P.queue, 1)); }))
                return;
            if (tid == 0)
                s_w = ts->world.get();
            __syncthreads();
            const int qi = s_w;
            if (qi >= Bp->wq_len[P.queue])
                return;
            w = Bp->world_order[Bp->wq_off[P.queue] + qi];
        }
        else
        {
            // claim the queue's next index, then wait until the host publishes its request: -1
            // when the server shuts down, or when idle and the claim could be given back
            const ServerCtl &S = *Sp;
            const int q = P.queue;
            wait_limit = SERVER_MAX_WAIT + WAIT_TICKS;
            const bool err = team_barrier([&] {
                unsigned i = atomicAdd(S.next + q, 1u);
                int got = -1;
                const unsigned long long w0 = wall_clock64();
                for (;;)
                {
                    if (__hip_atomic_load(S.shutdown, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM))
                        break;
                    if (i < __hip_atomic_load(S.tail + q, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM))
                    {
                        got = (int)i;
                        break;
                    }
                    const unsigned long long waited = wall_clock64() - w0;
                    if ((waited > S.idle_ticks && atomicCAS(S.next + q, i + 1, i) == i + 1) || waited > SERVER_MAX_WAIT)
                        break;
                    __builtin_amdgcn_s_sleep(8);
                }
                ts->world.set(got);
            });
            wait_limit = WAIT_TICKS;
            if (err)
                return;
            if (tid == 0)
            {
                s_w = ts->world.get();
                if (s_w >= 0)
                {
                    // (system-scope loads, as the tail's: the host writes a line's entries one after another
                    // while workgroups read the ones before, and only the workgroup that saw the tail has
                    // acquired at system scope)
                    ServerReq *r = S.req + (size_t)q * S.cap + s_w;
                    s_b = reinterpret_cast<const BatchT<RUNS> *>(
                        __hip_atomic_load(reinterpret_cast<uint64_t *>(&r->batch), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM));
                    s_id = __hip_atomic_load(&r->id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                }
            }
            __syncthreads();
            if (s_w < 0)
                return;
        }
        // (the request's batch pointer made wave-uniform, so its fields load into scalar registers
        // as a kernel argument's do)
        typename Md::Batch &B = *(typename Md::Batch *)(uint64_t)(SRV ? uniform_ptr(s_b) : Bp);
        typename Md::World &W = *(typename Md::World *)(uint64_t)(B.worlds + __builtin_amdgcn_readfirstlane(w));
        int hpw = P.hpw, spw = 64 / W.k;
        if (hpw <= 0)
            slot_items(W.H, W.S, W.k, T * nwaves, &hpw, &spw);
        if constexpr (ONE)
            hpw = 1; // (the launch's condition; a constant for the compiler)
        WorldRun *R = B.run + w;
        const int k = W.k;
        const int host_items = (W.H + hpw - 1) / hpw, items = host_items + (W.S + spw - 1) / spw;
        const unsigned long long c_begin = wall_clock64();
        if (tid == 0)
        {
            s_t = __hip_atomic_load(&R->slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_flags = (__hip_atomic_load(&R->finished, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ? SlotGo::FIN : 0) |
                      (__hip_atomic_load(&R->act_prev, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ? 0 : SlotGo::IDLE);
            s_act = __hip_atomic_load(&R->act_cur, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); // (a world's first slot)
            s_wake = ~0ull;
        }
        __syncthreads();
        for (int64_t it = 0;; it++)
        {
            const int64_t t = s_t;
            const unsigned flags = s_flags;
            if ((flags & SlotGo::FIN) || it >= slot_budget)
            {
                // every workgroup of the team leaves at the same slot, after a fenced barrier (the
                // world's records in memory before its results are read); the first writes where
                // the world stands, accounts the time (and, serving, tells the host)
                (void)team_barrier([] {});
                if (rank == 0 && tid == 0)
                {
                    R->slot = t;
                    R->slots_run += it;
                    R->act_cur = 0;
                    R->act_prev = flags & SlotGo::IDLE ? 0 : 1;
                    R->finished = flags & SlotGo::FIN ? 1 : 0;
                    R->ticks += wall_clock64() - c_begin;
                    R->team = T;
                    if constexpr (SRV)
                    {
                        __threadfence_system();
                        __hip_atomic_store(Sp->done + s_id, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
                    }
                }
                break;
            }
            unsigned act = 0;
            unsigned long long wk = ~0ull;
#ifdef TW_PROF
            __shared__ unsigned long long p_host, p_sw;
            const unsigned long long p0 = wall_clock64();
            unsigned long long p_h = 0, p_s = 0;
            if (tid == 0)
                p_host = p_sw = 0;
            __syncthreads();
#endif
            for (int item = gw; item < items; item += TW)
            {
                if (item < host_items)
                {
                    const int h0 = item * hpw, hl = h0 + lane;
#ifdef TW_PROF
                    const unsigned long long q0 = wall_clock64();
#endif
                    char *ws = reinterpret_cast<char *>(wl);
                    constexpr int FR = (int)sizeof(typename Md::Frame);
                    typename Md::HostIn in = {0, 0, 0, 0};
                    int64_t x = INT64_MAX;
                    const bool runs = lane < hpw && hl < W.H && Md::host_open(B, W, hl, t, in, &x);
                    // The frames out, from a host's workspace to its link's message, `group` lanes at it: one
                    // round of coherent stores, off the host's chain of events (a load after a frame's eight
                    // 8-byte stores waits 0.4 us for them, 0.09 us without).
                    auto send = [&](int host, const char *from, int frames, int first, int group) {
                        const uint64_t *f = reinterpret_cast<const uint64_t *>(from);
                        uint64_t TW_G *to = (uint64_t TW_G *)Md::msg_of(B, t, W.link0 + host);
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // (a wave's LDS accesses are in order)
                        for (int i = first; i < frames * (FR / 8); i += group)
                            coh_store(to + i, f[i]);
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    };
                    const int per = WAVE_LDS / hpw & ~15, group = 64 / hpw, mine = lane / group, src = mine < hpw ? mine : 0;
                    int out_n = 0;
                    if (runs)
                        act += Mh::host_run(B, W, R, hl, t, &x, typename Mh::HostIn{in.in, in.i2, in.n2, in.n1},
                                            (typename Mh::Frame *)(ws + lane * per), per / FR, &out_n);
                    const int n = __shfl(out_n, src);
                    send(h0 + src, ws + src * per, mine < hpw ? n : 0, lane % group, group);
                    if ((unsigned long long)x < wk)
                        wk = (unsigned long long)x;
#ifdef TW_PROF
                    p_h += wall_clock64() - q0;
#endif
                    continue;
                }
                const int g = item - host_items, sl = lane / k, base = (sl < spw ? sl : 0) * k;
                typename Md::SwLane x;
                x.swl = g * spw + sl;
                x.q = lane % k;
                x.active = sl < spw && x.swl < W.S;
                x.lid = W.link0 + W.H + x.swl * k + x.q;
                const size_t so = (size_t)base * 2 * MAX_TX;
                x.scr_ts = scr_ts + so;
                x.scr_ref = scr_ref + so;
                x.scr_up = scr_up + so;
                typename Md::SwLds L;
                L.rows = wl + base * (k + 1);
                L.in_win = wl + 64 * 33 + base * 3;
                L.base = wl + 64 * 33 + 64 * 3 + base;
                L.cnt = wl + 64 * 33 + 64 * 3 + 64 + base;
                L.wave = wl;
#ifdef TW_PROF
                const unsigned long long q0 = wall_clock64();
#endif
                act += Md::switch_step(B, W, R, x, t, L);
#ifdef TW_PROF
                p_s += wall_clock64() - q0;
#endif
            }
#ifdef TW_PROF
            atomicMax(&p_host, p_h);
            atomicMax(&p_sw, p_s);
#endif
            // The slot's end. A wake-up counts in a slot without any activity only, so a workgroup
            // with some brings one word, its arrival, and the others bring their wake-up before it.
            if (__ballot(act != 0))
            {
                if (lane == 0)
                    atomicOr(&s_act, 1u);
            }
            else if (wk != ~0ull)
                atomicMin(&s_wake, wk);
            __builtin_amdgcn_s_waitcnt(0); // (this wave's stores have completed)
            __syncthreads();
            if (tid == 0)
            {
#ifdef TW_PROF
                atomicMax(&ts->prof[0], p_host);
                atomicMax(&ts->prof[1], p_sw);
                atomicMax(&ts->prof[2], wall_clock64() - p0);
#endif
                const int par = slot_count++ & 1;
                const unsigned active = s_act != 0;
                unsigned arrived = 0; // before this workgroup
                if (T > 1)
                {
                    if (!active && s_wake != ~0ull)
                    {
                        atomicMax(&ts->wake[par], ~s_wake);
                        __builtin_amdgcn_s_waitcnt(0);
                    }
                    arrived = atomicAdd(&ts->slot_arrive[par], 1u | active << 16);
                }
                unsigned long long go;
                if ((arrived & 0xFFFFu) == (unsigned)T - 1)
                {
                    // the ticket (src/kernel.cuh:79-112): finish, or the next slot with the exact idle skip
                    const bool idle = (arrived >> 16) + active == 0;
                    const unsigned done = coh_load(&R->flows_done);
                    const int bad = T > 1 ? coh_load(&ts->err) : 0;
                    const bool fin = done >= (unsigned)W.M || t + 1 >= W.max_slots;
                    int64_t next = t + 1;
                    if (idle && (flags & SlotGo::IDLE))
                    {
                        const unsigned long long nw = T > 1 ? ~coh_load(&ts->wake[par]) : s_wake;
                        if (nw != ~0ull && (int64_t)nw > next)
                            next = (int64_t)nw < W.max_slots ? (int64_t)nw : W.max_slots;
                    }
                    go = SlotGo::pack(next, (fin ? SlotGo::FIN : 0) | (idle ? SlotGo::IDLE : 0) | (bad ? SlotGo::ERR : 0), slot_count);
                    if (T > 1)
                    {
                        coh_store(&ts->go, go);
                        // (these words are next used two slots on, after this wave's next wait for its stores)
                        coh_store(&ts->slot_arrive[par], 0u);
                        coh_store(&ts->wake[par], 0ull);
                    }
#ifdef TW_PROF
                    const unsigned long long now = wall_clock64();
                    const unsigned long long before = atomicExch(&ts->prof[3], now);
                    if (before)
                        atomicAdd(&R->ev[EV_PROF_PERIOD], now - before);
                    atomicAdd(&R->ev[EV_PROF_HOSTS], atomicExch(&ts->prof[0], 0ull));
                    atomicAdd(&R->ev[EV_PROF_SWITCHES], atomicExch(&ts->prof[1], 0ull));
                    atomicAdd(&R->ev[EV_PROF_WORK], atomicExch(&ts->prof[2], 0ull));
#endif
                }
                else
                {
                    const unsigned long long w0 = wall_clock64();
                    while (SlotGo::count(go = coh_load(&ts->go)) != (slot_count & 0xFFFFu))
                    {
                        __builtin_amdgcn_s_sleep(1);
                        if (wall_clock64() - w0 > WAIT_TICKS)
                        {
                            atomicExch(&ts->err, 1);
                            go = SlotGo::pack(t, SlotGo::ERR, slot_count);
                            break;
                        }
                    }
                }
                s_t = SlotGo::next(go);
                s_flags = SlotGo::flags(go);
                s_act = 0;
                s_wake = ~0ull;
            }
            __syncthreads();
            const bool err = s_flags & SlotGo::ERR;
            if (err)
            {
                if (tid == 0)
                {
                    coh_store(&R->error, 1);
                    coh_store(&R->finished, 1);
                    if constexpr (SRV)
                        if (rank == 0)
                        {
                            __threadfence_system();
                            __hip_atomic_store(Sp->done + s_id, 2, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
                        }
                }
                return;
            }
        }
    }
}

template <int RUNS, bool ONE>
__global__ void __launch_bounds__(256) tcp_worlds_kernel(const BatchT<RUNS> *__restrict__ Bp, int64_t slot_budget)
{
    world_loop<RUNS, false, ONE>(Bp, nullptr, slot_budget);
}

// The serving loop's persistent kernel. Requests are single-world batches already in device
// memory; the host appends them to per-queue rings in pinned host memory and publishes each
// queue's tail there. A team claims the next index of its queue, waits until the host has
// published it (or the server shuts down), runs the world to its end and flags it done in
// pinned memory. Every wait is bounded: an idle team gives its claim back and leaves after
// ServerCtl::idle_ticks, the host's shutdown flag ends every wait, and the host relaunches the
// kernel when it finds it gone.
template <int RUNS>
__global__ void __launch_bounds__(256) tcp_server_kernel(const ServerCtl *__restrict__ Sp)
{
    world_loop<RUNS, true, false>(nullptr, Sp, INT64_MAX);
}

// This file is compiled once per chain length (TW_RUNS = 9 or 25, two objects built in parallel:
// fully inlined, each takes minutes); tcp_kernel.h dispatches on the run count.
#ifndef TW_RUNS
#define TW_RUNS 9
#endif
#define TW_CAT(a, b) a##b
#define TW_NAME(a, b) TW_CAT(a, b)

hipError_t TW_NAME(tcp_launch_, TW_RUNS)(const void *batch_dev, const LaunchShape &s, hipStream_t stream)
{
    // an ordinary launch: the grid never exceeds the workgroups the GPU holds at once (the plan
    // checks it), so a team's workgroups are resident together, and a team barrier that still
    // waited too long ends the world with an error. No cooperative launch: it takes a device-wide
    // resource that one process can hold while another waits for it.
    const size_t lds = (size_t)(s.threads / 64) * LDS_PER_WAVE * sizeof(int);
    const BatchT<TW_RUNS> *b = reinterpret_cast<const BatchT<TW_RUNS> *>(batch_dev);
    if (s.one)
        hipLaunchKernelGGL((tcp_worlds_kernel<TW_RUNS, true>), dim3(s.blocks), dim3(s.threads), lds, stream, b, s.slot_budget);
    else
        hipLaunchKernelGGL((tcp_worlds_kernel<TW_RUNS, false>), dim3(s.blocks), dim3(s.threads), lds, stream, b, s.slot_budget);
    return hipGetLastError();
}

hipError_t TW_NAME(tcp_server_launch_, TW_RUNS)(const void *ctl_dev, int blocks, int threads, hipStream_t stream)
{
    const size_t lds = (size_t)(threads / 64) * LDS_PER_WAVE * sizeof(int);
    const ServerCtl *c = reinterpret_cast<const ServerCtl *>(ctl_dev);
    hipLaunchKernelGGL(tcp_server_kernel<TW_RUNS>, dim3(blocks), dim3(threads), lds, stream, c);
    return hipGetLastError();
}

hipError_t TW_NAME(tcp_max_blocks_, TW_RUNS)(int threads, int *per_cu)
{
    const size_t lds = (size_t)(threads / 64) * LDS_PER_WAVE * sizeof(int);
    // (the fewer of the two kernels')
    int one = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&one, tcp_worlds_kernel<TW_RUNS, true>, threads, lds);
    const hipError_t f = hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, tcp_worlds_kernel<TW_RUNS, false>, threads, lds);
    *per_cu = one < *per_cu ? one : *per_cu;
    return e != hipSuccess ? e : f;
}

#if TW_RUNS == 9
// clears the world-queue counters and the teams' barrier words before a launch (a kernel, not a
// memset, so that the pair can be captured in a graph)
__global__ void tcp_reset_kernel(uint32_t *__restrict__ a, int na, uint32_t *__restrict__ b, int nb)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < na + nb; i += gridDim.x * blockDim.x)
    {
        if (i < na)
            a[i] = 0;
        else
            b[i - na] = 0;
    }
}

hipError_t tcp_reset(uint32_t *queue_next, int nq, void *teams, size_t team_bytes, hipStream_t stream)
{
    const int nb = (int)(team_bytes / 4);
    int blocks = (nq + nb + 255) / 256;
    blocks = blocks < 1 ? 1 : blocks > 1024 ? 1024 : blocks;
    hipLaunchKernelGGL(tcp_reset_kernel, dim3(blocks), dim3(256), 0, stream, queue_next, nq, (uint32_t *)teams, nb);
    return hipGetLastError();
}

// The scratch memory of tw_batch_run_noalloc: a launch's batch record, team barrier words, queue
// counters and switch sort space, in a device array of the library's own (every GPU the library
// runs on holds one copy until the process ends), so that the entry point allocates nothing. Host
// code never passes the array's name to a kernel: the address to use is the one
// hipGetSymbolAddress gives, looked up once per device with that device current.
static __device__ __align__(256) unsigned char scratch[TW_SCRATCH_BYTES];

hipError_t tcp_static_scratch(void **ptr)
{
    static std::mutex mu;
    static void *per_dev[64] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return e;
    if (dev < 0 || dev >= 64)
        return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> g(mu);
    if (!per_dev[dev])
    {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess)
            return e;
        per_dev[dev] = p;
    }
    *ptr = per_dev[dev];
    return hipSuccess;
}
#endif

} // namespace tw
