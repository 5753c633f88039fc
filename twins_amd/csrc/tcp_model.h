// The TCP packet model on gfx950: one slot of a host (a lane runs its serial event loop) and one
// slot of a switch (a group of lanes of one wavefront, one lane per port), over the batch
// layout of tcp_state.h. The semantics follow TwiNS's model exactly (reference: src/step.cuh,
// src/kernel.cuh), so every flow's times equal sequential ns-3's; the comments cite the
// reference lines each part follows.
//
// Build with -ffp-contract=off: the only fused multiply-adds are the explicit fma() calls.
#pragma once
#include <cassert>
#include <cstddef>
#include <hip/hip_runtime.h>
#include "exact_math.h"
#include "tcp_state.h"

namespace tw
{

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// A condition that is seldom (usually) true where it stands: the code for the other case is laid out
// next, so the usual way through an event takes few branches.
#define TW_RARE(c) (ONE ? __builtin_expect((long)U(c), 0) : (long)U(c))
#define TW_USUAL(c) (ONE ? __builtin_expect((long)U(c), 1) : (long)U(c))

// ONE: the host code for a wave that runs one host at a time on one lane. Every branch is then the
// wave's, and U() says so: the compiler branches on a scalar instead of masking lanes in and out and
// merging the masks at every join (a third of the host code's instructions, and as many as its
// registers could not hold).
template <int RUNS, bool SRV = false, bool ONE = false>
struct Model
{
    static __device__ __forceinline__ bool U(bool c)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        if constexpr (ONE)
            return __builtin_amdgcn_ballot_w64(c) != 0;
#endif
        return c;
    }
    typedef typename ReadOnly<BatchT<RUNS>, SRV>::type Batch; // (const)
    typedef typename ReadOnly<WorldDesc, SRV>::type World;    // (const)
    typedef FrameT<RUNS> Frame;
    static constexpr int CW = RUNS + 1; // a chain's words: RUNS runs (code | count << 16), the root
    struct Chain
    {
        uint32_t r[CW];
    };

    // -------------------------------------------------------------- event-order chains
    // (src/step.cuh:58-159) the leads from an event back to its root, run-length encoded; codes
    // grow with the lead: ScheduleNow 1, Send's deferral 2, TransmitComplete len, arrival
    // 2048 + len, timers 4096 + lead/16 ns (saturating)
    static __device__ __forceinline__ uint32_t code_lead(int64_t lead_ps)
    {
        // (a lead is not negative; in 32 bits where it does not saturate)
        constexpr int64_t MOST = (int64_t)(0xFFFE - 4096) * 16000;
        return lead_ps < MOST ? 4096 + (uint32_t)lead_ps / 16000 : 0xFFFE;
    }
    static __device__ __forceinline__ void chain_load(Chain &c, const uint32_t *p)
    {
#pragma unroll
        for (int i = 0; i < CW; i++)
            c.r[i] = p[i];
    }
    static __device__ __forceinline__ void chain_store(uint32_t *p, const Chain &c)
    {
#pragma unroll
        for (int i = 0; i < CW; i++)
            p[i] = c.r[i];
    }
    // an application start scheduled at set-up: host then connection (world-local)
    static __device__ __forceinline__ void chain_root(Chain &c, int host_local, int conn_local)
    {
#pragma unroll
        for (int i = 0; i < RUNS; i++)
            c.r[i] = 0;
        c.r[RUNS] = (uint32_t)(0x8000 | (host_local + 1)) | (uint32_t)(conn_local & 0xFFFF) << 16;
    }
    // a message write scheduled in main(), by message (world-local)
    static __device__ __forceinline__ void chain_root_msg(Chain &c, int msg_local)
    {
#pragma unroll
        for (int i = 0; i < RUNS; i++)
            c.r[i] = 0;
        c.r[RUNS] = (uint32_t)((1 + (msg_local >> 16)) & 0xFFFF) | (uint32_t)(msg_local & 0xFFFF) << 16;
    }
    // dst = [code] + parent (dst may alias parent): a repeated code extends the first run
    static __device__ __forceinline__ void chain_child(Chain &dst, uint32_t code, const Chain &parent)
    {
        const Chain p = parent;
        if (U((p.r[0] & 0xFFFF) == code))
        {
            dst = p;
            if (U((p.r[0] >> 16) < 0xFFFF))
                dst.r[0] += 1u << 16;
            return;
        }
        dst.r[0] = code | 1u << 16;
#pragma unroll
        for (int i = 1; i < RUNS; i++)
            dst.r[i] = p.r[i - 1];
        dst.r[RUNS] = p.r[RUNS];
    }
    // < 0: a runs first, > 0: b, 0: undecided. Larger codes (earlier parents) first; a complete
    // chain (fewer than RUNS runs) ends at its root, before any other parent; else the roots.
    // (a(i), b(i): the chains' words; chain_cmp reads plain memory, frames of link messages are
    // read device-coherently, word by word as the comparison needs them)
    template <typename GA, typename GB>
    static __device__ int chain_cmp_by(GA a, GB b)
    {
        int ia = 0, ib = 0;
        uint32_t ra = a(0) >> 16, rb = b(0) >> 16;
        for (;;)
        {
            uint32_t ca = a(ia) & 0xFFFF, cb = b(ib) & 0xFFFF;
            if (U(ca == 0 && cb != 0 && (a(RUNS) & 0xFFFF) != 0))
                return -1;
            if (U(cb == 0 && ca != 0 && (b(RUNS) & 0xFFFF) != 0))
                return 1;
            if (U(ca == 0 || cb == 0))
                break;
            if (U(ca != cb))
                return ca > cb ? -1 : 1;
            uint32_t m = ra < rb ? ra : rb;
            ra -= m;
            rb -= m;
            if (U(ra == 0))
            {
                if (U(++ia == RUNS))
                    break;
                ra = a(ia) >> 16;
            }
            if (U(rb == 0))
            {
                if (U(++ib == RUNS))
                    break;
                rb = b(ib) >> 16;
            }
        }
        uint32_t xa = a(RUNS) << 16 | a(RUNS) >> 16, xb = b(RUNS) << 16 | b(RUNS) >> 16; // the root keys
        if (U(xa == 0 || xb == 0 || xa == xb))
            return 0;
        return xa < xb ? -1 : 1;
    }
    static __device__ int chain_cmp(const uint32_t *a, const uint32_t *b)
    {
        return chain_cmp_by([&](int i) { return a[i]; }, [&](int i) { return b[i]; });
    }
    // the message of link `link` in slot t's ring place
    static __device__ __forceinline__ auto msg_of(Batch &B, int64_t t, int link)
    {
        return B.msg + (uint64_t)(ring_of(t) * (uint32_t)B.nlinks + (uint32_t)link) * MAX_TX;
    }
    static __device__ __forceinline__ auto msg_cnt_of(Batch &B, int64_t t, int link) { return B.msg_cnt + (uint64_t)(ring_of(t) * (uint32_t)B.nlinks + (uint32_t)link); }
    // a link message's frame, read device-coherently: its head (all but the chain), its chain
    struct FrameHead
    {
        int64_t ts;
        uint32_t flow, sa;
        uint16_t len, dst;
        uint8_t flags, to_sender, up, pad;
    };
    static_assert(sizeof(FrameHead) == 24 && offsetof(Frame, chain) == 24, "a frame's head");
    static __device__ __forceinline__ FrameHead msg_head(const Frame *p) { return coh_get(reinterpret_cast<const FrameHead *>(p)); }
    static __device__ __forceinline__ void msg_chain(Chain &c, const Frame *p)
    {
#pragma unroll
        for (int i = 0; i < CW; i++)
            c.r[i] = coh_load(&p->chain[i]);
    }
    static __device__ __forceinline__ void count(WorldRun *R, int i, unsigned long long n = 1) { atomicAdd(&R->ev[i], n); }

    // -------------------------------------------------------------- egress queue
    // One sending queue per link (a host's NIC, a switch port): frames wait in a ring until the
    // link is free; a frame whose transmission starts in this slot goes to the link's message for
    // the slot with its arrival time at the far end. The queue's state lives in registers for the
    // entity's slot (load / store). Admission is RED with MinTh = MaxTh = K and QW = 1 on the
    // queue-disc length ns-3 would see (src/step.cuh:167-317 restates the same rules).
    struct Fifo
    {
        Batch *B;
        World *W;
        WorldRun *R;
        int lid, rt;
        Frame *ring;
        int cap, head, size, red_k, limit, sent, early;
        int64_t link_free, last_start, woke, idle_start, slot_end;
        Chain last; // the chain of the transmission in progress (kept in registers for the slot)
        Frame hd;   // the first queued frame (while size > 0); not yet in the ring if hd_new
        bool hd_new;
        Frame *out;
        // the slot's first frames out wait in the workspace (LDS), if the entity has one
        Frame *stage;
        int stage_cap;

        __device__ __forceinline__ void load(Batch &b, World &w, WorldRun *r, int link, int64_t t, int ring_t, Frame *st = nullptr, int st_cap = 0)
        {
            B = &b;
            W = &w;
            R = r;
            lid = link;
            rt = ring_t;
            ring = b.qring + b.q_base[link];
            cap = b.q_cap[link];
            head = b.q_head[link];
            size = b.q_size[link];
            red_k = b.q_red_k[link];
            limit = b.q_limit[link];
            link_free = b.q_link_free[link];
            last_start = b.q_last_start[link];
            chain_load(last, b.q_last_chain + (size_t)link * CW);
            woke = idle_start = -1;
            slot_end = (t + 1) * SLOT_PS;
            sent = early = 0;
            hd_new = false;
            if (U(size > 0))
                hd = ring[head];
            out = b.msg + ((size_t)ring_t * b.nlinks + link) * MAX_TX;
            stage = st;
            stage_cap = st_cap;
        }
        // the slot's message count word (msg_word) and the queue back to memory
        __device__ __forceinline__ void store(int64_t t, int ring_t)
        {
            coh_store(B->msg_cnt + (size_t)ring_t * B->nlinks + lid, msg_word(t, early, sent));
            if (TW_USUAL(size > 0 && hd_new))
                ring[head] = hd;
            B->q_head[lid] = head;
            B->q_size[lid] = size;
            B->q_link_free[lid] = link_free;
            B->q_last_start[lid] = last_start;
            chain_store(B->q_last_chain + (size_t)lid * CW, last);
            if (U(sent))
                count(R, EV_PKT_EVENTS, (unsigned long long)sent);
        }
        // frame i of the slot's message: into the workspace, or out device-coherently, 16 bytes a store
        // (the world's messages of a slot lie within the 2^31 bytes a buffer store reaches)
        __device__ __forceinline__ void put(int i, const Frame &o)
        {
            if (TW_USUAL(i < stage_cap))
            {
                stage[i] = o;
                return;
            }
#if defined(__HIP_DEVICE_COMPILE__)
            const uint64_t bytes = (uint64_t)W->L * MAX_TX * sizeof(Frame);
            if (U(bytes <= 0x7FFFFFF0ull))
            {
                const __amdgpu_buffer_rsrc_t r = twc::coh_buffer((const void *)(B->msg + ((size_t)rt * B->nlinks + W->link0) * MAX_TX), (uint32_t)bytes);
                const uint32_t at = ((uint32_t)(lid - W->link0) * MAX_TX + (uint32_t)i) * (uint32_t)sizeof(Frame);
                uint64_t w[sizeof(Frame) / 8];
                __builtin_memcpy(w, &o, sizeof o);
#pragma unroll
                for (int k = 0; k < (int)(sizeof(Frame) / 16); k++)
                    twc::coh_store16(r, at + 16 * k, w[2 * k], w[2 * k + 1]);
                return;
            }
#endif
            coh_put(out + i, o); // (read by the link's far end in a later slot)
        }
        // Starts, in order, the frames whose transmission begins by `until` within the slot. The
        // event that starts a frame is the previous frame's TransmitComplete when the frame had
        // to wait for the link (its chain: the last transmission's, one more run), else the
        // frame's own enqueue (a link that never sent counts as idle).
        // (Vector memory counts in order: a load waits for the stores issued before it. So the first
        // queued frame is in registers, a frame queued and sent while it was first passes through no
        // memory, and the next one's load is issued before the sent one's stores.)
        __device__ void advance(int64_t until)
        {
            while (U(size > 0))
            {
                if (TW_RARE(sent >= MAX_TX))
                {
                    count(R, EV_TXCAP);
                    return;
                }
                const int64_t start = hd.ts > link_free ? hd.ts : link_free;
                if (U(start >= slot_end || start > until))
                    return;
                Frame o = hd;
                head = head + 1 < cap ? head + 1 : 0;
                hd_new = false;
                if (U(--size > 0))
                    hd = ring[head];
                if (U(o.ts <= link_free && link_free > last_start))
                {
                    chain_child(last, (uint32_t)(link_free - last_start) / (uint32_t)PS_PER_BYTE, last);
                    chain_store(o.chain, last);
                }
                else
                {
                    chain_load(last, o.chain);
                    idle_start = start;
                }
                last_start = start;
                link_free = start + (int64_t)o.len * PS_PER_BYTE;
                o.ts = link_free + PROP_PS; // its arrival at the far end
                early += o.ts < slot_end + SLOT_PS;
                put(sent, o);
                sent++;
            }
        }
        // a queue-trace record (src/step.cuh:266-279), stored field by field (no record on the stack)
        __device__ __forceinline__ void trace(int64_t now, int qlen, uint32_t flow, uint32_t sa, uint16_t len, uint8_t flags, uint8_t to_sender)
        {
            const unsigned long long i = atomicAdd(B->qt.cnt, 1ull);
            if (U(i < B->qt.cap))
            {
                QRec *r = B->qt.rec + i;
                r->ts = now;
                r->link = lid;
                r->flow = flow;
                r->sa = sa;
                r->len = len;
                r->qlen = (uint16_t)qlen;
                r->flags = flags;
                r->to_sender = to_sender;
            }
        }
        // The queue-disc length ns-3's RED sees at `now`. The first queued frame sits in the
        // device's one-frame queue (outside the queue disc) once the device has pulled it: when a
        // transmission started before `now`, or when the device's Wake ran at this very instant
        // on an idle link; until then it still counts.
        __device__ __forceinline__ int qdisc_len(int64_t now) const
        {
            const bool pulled = last_start < now || (woke == now && idle_start == now);
            return size > 0 && link_free > now && pulled ? size - 1 : size;
        }
        // a frame offered at `now`, to which the queue has advanced: RED marks (ECN-capable) or drops it
        // at K, the queue limit drops it; false if dropped
        __device__ bool enqueue(const Frame &f, int64_t now)
        {
            const int len = qdisc_len(now);
            Frame g = f;
            g.ts = now;
            const bool over_k = len >= red_k && len > 1;
            if (TW_RARE(over_k && !(g.flags & F_ECT)))
            {
                count(R, EV_DROP);
                return false;
            }
            if (TW_RARE(over_k))
            {
                g.flags |= F_CE;
                count(R, EV_MARK);
            }
            if (TW_RARE(len >= limit))
            {
                count(R, EV_DROP);
                return false;
            }
            if (TW_RARE(B->qt.rec && now >= B->qt.from && now < B->qt.until))
                trace(now, len + 1, g.flow, g.sa, g.len, g.flags, g.to_sender);
            if (TW_RARE(size >= cap))
            {
                count(R, EV_RING_OVF);
                return false;
            }
            if (U(size == 0))
            {
                hd = g;
                hd_new = true;
            }
            else
                ring[head + size < cap ? head + size : head + size - cap] = g;
            size++;
            return true;
        }
    };

    // -------------------------------------------------------------- host context
    // a frame an event asks for: its sequence or acknowledgement number, length, flags and direction
    struct Out
    {
        uint32_t sa;
        uint16_t len;
        uint8_t flags, to_sender;
    };
    // what the events of a connection's sending (receiving) side use of its static record; way: its
    // frames' destination and equal-cost index
    struct ConnSnd
    {
        uint64_t it_off;
        uint32_t it_cap, way;
        int32_t m_first, m_cnt;
        bool fin_on;
    };
    struct ConnRcv
    {
        uint64_t oo_off;
        uint32_t oo_cap, way;
    };
    struct Host
    {
        Batch *B;
        World *W;
        WorldRun *R;
        Fifo nic;
        int h, hl; // global, world-local
        bool dctcp, cubic;
        Chain echain; // the chain of the event being processed
        Due *due;
        int nd, id;
        int64_t due_head; // due[id].at (INT64_MAX when none is left): the next timer of the slot
        int64_t slot_end;
        // The records of the connection sides that events work on, in registers: one sending side and one
        // receiving side (sf, rf: whose; -1: none), each with its connection's static record. A record is
        // read when its first event of the slot runs and written back when another connection's event
        // or the slot's end comes. (In LDS an event made some 160 accesses to them, 28 ns each when the
        // next waits for it.)
        SndState S;
        RcvState Q;
        ConnSnd cs;
        ConnRcv cr;
        int sf, rf;
        uint32_t max_it; // the longest sent ledger of the slot
        // What the running event sends, queued after its handler by the one place that builds frames
        // (host_run's loop): the frames asked for (at most 4: an ACK at a CE edge, one for the data,
        // the close's; or one segment sent again), then, if fill, segments while the window has room,
        // then one more asked for after that.
        Out ask[4], post;
        int n_ask, i_ask, fill_n;
        int f;        // the running event's connection
        uint32_t way; // where its frames go: the host (world-local) and, above it, the equal-cost index
        bool fill, has_post;
    };
    // A record between registers and device memory: words of 4 or 8 bytes as its fields lie (adjacent
    // ones become 16-byte accesses, issued together)
    typedef uint32_t __attribute__((may_alias)) word4;
    typedef uint64_t __attribute__((may_alias)) word8;
    template <typename W, int FROM, int TO, typename D, typename S>
    static __device__ __forceinline__ void words(D *dst, const S *src)
    {
#pragma unroll
        for (int i = FROM / (int)sizeof(W); i < TO / (int)sizeof(W); i++)
            reinterpret_cast<W *>(dst)[i] = reinterpret_cast<const W *>(src)[i];
    }
    static_assert(offsetof(SndState, srtt) == 120 && offsetof(SndState, cub_cnt) == 192 && offsetof(SndState, cub_k) == 224 &&
                      offsetof(RcvState, r_fin) == 32 && offsetof(RcvState, ecn_ce_seq) == 96,
                  "the records' words");
    // (a sender's Cubic state stays in memory: only Cubic's worlds look at it)
    template <typename D, typename S>
    static __device__ __forceinline__ void snd_move(D *dst, const S *src)
    {
        words<word4, 0, 120>(dst, src);
        words<word8, 120, 192>(dst, src);
    }
    template <typename D, typename S>
    static __device__ __forceinline__ void rcv_move(D *dst, const S *src)
    {
        words<word4, 0, 32>(dst, src);
        words<word8, 32, 104>(dst, src);
    }
    static __device__ __forceinline__ uint32_t way_to(const Host &x, int host, uint32_t hash)
    {
        return (uint32_t)(uint16_t)(host - x.W->host0) | (hash % (uint32_t)x.W->ecmp_n & 0xFF) << 16;
    }
    // The receiver's host reads a sender's end state (compact_rcv): the 4-byte word holding
    // SndState::st goes out device-coherently once the sender is done.
    static constexpr size_t ST_WORD = offsetof(SndState, st) & ~(size_t)3;
    static constexpr int ST_SHIFT = (int)(offsetof(SndState, st) & 3) * 8;
    static __device__ __forceinline__ void snd_flush(Host &x)
    {
        if (U(x.sf < 0))
            return;
        snd_move(&x.B->snd[x.sf], &x.S);
        if (U(x.S.st == S_DONE))
            coh_store(reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(&x.B->snd[x.sf]) + ST_WORD),
                      *reinterpret_cast<const word4 *>(reinterpret_cast<const char *>(&x.S) + ST_WORD));
    }
    static __device__ __forceinline__ void rcv_flush(Host &x)
    {
        if (U(x.rf >= 0))
            rcv_move(&x.B->rcv[x.rf], &x.Q);
    }
    static __device__ __forceinline__ SndState &snd_open(Host &x, int f)
    {
        if (TW_RARE(x.sf != f))
        {
            snd_flush(x);
            snd_move(&x.S, &x.B->snd[f]);
            const ConnStatic TW_G &c = x.B->cs[f];
            x.cs = ConnSnd{c.it_off, c.it_cap, way_to(x, c.dst, c.hash_data), c.m_first, c.m_cnt, c.fin_on != 0};
            x.sf = f;
        }
        x.f = f;
        x.way = x.cs.way;
        return x.S;
    }
    static __device__ __forceinline__ bool snd_done_seen(Batch &B, int f)
    {
        const uint32_t w = coh_load(reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(&B.snd[f]) + ST_WORD));
        return (uint8_t)(w >> ST_SHIFT) == S_DONE;
    }
    static __device__ __forceinline__ RcvState &rcv_open(Host &x, int f)
    {
        if (TW_RARE(x.rf != f))
        {
            rcv_flush(x);
            rcv_move(&x.Q, &x.B->rcv[f]);
            const ConnStatic TW_G &c = x.B->cs[f];
            x.cr = ConnRcv{c.oo_off, c.oo_cap, way_to(x, c.src, c.hash_ack)};
            x.rf = f;
        }
        x.f = f;
        x.way = x.cr.way;
        return x.Q;
    }

    // Active lists: a host's sending and receiving connections. A connection leaves its list at
    // the end of a slot in which it is finished (sender: closed; receiver: the sender closed and
    // no receiver timer pending), as in the reference (src/step.cuh:2470-2510; with a full list
    // the add is refused and counted, so the removal's timing decides results in that regime);
    // compact() drops those and returns the earliest timer of the rest.
    // (Both walk their list COMPACT_RUN entries at a time: the entries' records are all read
    // before any entry is written back, so the reads of a run are in flight together.)
    static constexpr int COMPACT_RUN = 4;
    static __device__ __forceinline__ int64_t compact_snd(Batch &B, int h)
    {
        int64_t next = INT64_MAX;
        int32_t *l = B.act_snd + (size_t)h * MAX_ACTIVE;
        int k = 0, n = B.n_snd[h];
        for (int i0 = 0; U(i0 < n); i0 += COMPACT_RUN)
        {
            int f[COMPACT_RUN];
            bool done[COMPACT_RUN];
            int64_t rto[COMPACT_RUN], syn[COMPACT_RUN];
#pragma unroll
            for (int j = 0; j < COMPACT_RUN; j++)
                if (U(i0 + j < n))
                {
                    f[j] = l[i0 + j];
                    const SndState &s = B.snd[f[j]];
                    done[j] = s.st == S_DONE;
                    rto[j] = s.rto_at;
                    syn[j] = s.syn_at;
                }
#pragma unroll
            for (int j = 0; j < COMPACT_RUN; j++)
                if (U(i0 + j < n && !done[j]))
                {
                    l[k++] = f[j];
                    if (U(rto[j] >= 0 && rto[j] < next))
                        next = rto[j];
                    if (U(syn[j] >= 0 && syn[j] < next))
                        next = syn[j];
                }
        }
        B.n_snd[h] = k;
        return next;
    }
    static __device__ __forceinline__ int64_t compact_rcv(Batch &B, int h)
    {
        int64_t next = INT64_MAX;
        int32_t *l = B.act_rcv + (size_t)h * MAX_ACTIVE;
        int k = 0, n = B.n_rcv[h];
        for (int i0 = 0; U(i0 < n); i0 += COMPACT_RUN)
        {
            int f[COMPACT_RUN];
            bool gone[COMPACT_RUN];
            int64_t tmin[COMPACT_RUN];
#pragma unroll
            for (int j = 0; j < COMPACT_RUN; j++)
                if (U(i0 + j < n))
                {
                    f[j] = l[i0 + j];
                    const RcvState &r = B.rcv[f[j]];
                    const int64_t v[4] = {r.delack_at, r.srv_syn_at, r.r_last_at, r.r_frx_at};
                    gone[j] = snd_done_seen(B, f[j]) && v[0] < 0 && v[2] < 0 && v[3] < 0;
                    tmin[j] = INT64_MAX;
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        if (U(v[q] >= 0 && v[q] < tmin[j]))
                            tmin[j] = v[q];
                }
#pragma unroll
            for (int j = 0; j < COMPACT_RUN; j++)
                if (U(i0 + j < n && !gone[j]))
                {
                    l[k++] = f[j];
                    next = tmin[j] < next ? tmin[j] : next;
                }
        }
        B.n_rcv[h] = k;
        return next;
    }

    static __device__ void due_insert(Host &x, int64_t at, int f, int kind)
    {
        if (U(at >= x.slot_end))
            return;
        if (TW_RARE(x.nd >= MAX_DUE))
        {
            count(x.R, EV_DUE_OVF);
            return;
        }
        int j = x.nd;
        while (U(j > x.id && x.due[j - 1].at > at))
        {
            x.due[j] = x.due[j - 1];
            j--;
        }
        x.due[j] = {at, f, kind};
        x.nd++;
        if (U(j == x.id))
            x.due_head = at;
    }
    static __device__ __forceinline__ void timer_chain(Host &x, uint32_t *base, int f, int64_t lead)
    {
        Chain c;
        chain_child(c, code_lead(lead), x.echain);
        chain_store(base + (size_t)f * CW, c);
    }
    static __device__ __forceinline__ Out out_of(uint8_t flags, uint32_t seq, uint32_t ack, uint16_t len, bool to_sender)
    {
        return Out{(flags & F_DATA) ? seq : ack, len, flags, (uint8_t)(to_sender ? 1 : 0)};
    }
    static __device__ __forceinline__ void emit(Host &x, int f, uint8_t flags, uint32_t seq, uint32_t ack, uint16_t len, bool to_sender, int64_t now)
    {
        const Out o = out_of(flags, seq, ack, len, to_sender);
        if (TW_RARE(x.fill))
        {
            x.post = o;
            x.has_post = true;
            return;
        }
        const int n = x.n_ask++;
#pragma unroll
        for (int i = 0; i < 4; i++) // (static places: registers)
            if (i == n)
                x.ask[i] = o;
    }
    // the frame of what the running event sends, with the event's chain
    static __device__ __forceinline__ Frame frame_of(const Host &x, const Out &o, int64_t now)
    {
        Frame fr;
        fr.ts = now;
        fr.flow = (uint32_t)x.f;
        fr.sa = o.sa;
        fr.len = o.len;
        fr.dst = (uint16_t)x.way; // (a side's frames all go one way)
        fr.flags = o.flags | (x.dctcp ? F_ECT : 0);
        fr.to_sender = o.to_sender;
        fr.up = (uint8_t)(x.way >> 16);
        fr.pad = 0;
        chain_store(fr.chain, x.echain);
        return fr;
    }
    // the next of it; false: all is out
    static __device__ __forceinline__ bool next_out(Host &x, int64_t now, Out *o)
    {
        if (U(x.i_ask < x.n_ask))
        {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i == x.i_ask)
                    *o = x.ask[i];
            x.i_ask++;
            return true;
        }
        if (U(x.fill && fill_next(x, x.f, now, o)))
            return true;
        x.fill = false;
        if (TW_USUAL(!x.has_post))
            return false;
        *o = x.post;
        x.has_post = false;
        return true;
    }

    // -------------------------------------------------------------- the sent ledger
    // ns-3's TcpTxBuffer sent list as this model uses it (no SACK blocks; Reno's emulated SACK on
    // duplicate ACKs): one entry per run of transmitted bytes - its first byte and its marks
    // (IT_SACKED, IT_LOST, IT_RETX) - in a ring per connection, oldest first; an entry ends where
    // the next begins (the last at s.high). The connection's record keeps what decisions need
    // without walking the ring: bytes per mark, the sacked entries, and the retransmission
    // candidates (lost, neither retransmitted nor sacked) with a lower bound of the first.
    struct Ledger
    {
        SndState &s;
        SentEntry TW_G *ring;
        uint32_t cap;
        __device__ __forceinline__ Ledger(Host &x) : s(x.S)
        {
            ring = x.B->it + x.cs.it_off;
            cap = x.cs.it_cap;
        }
        __device__ __forceinline__ uint32_t pos(uint32_t i) const { return s.it_head + i < cap ? s.it_head + i : s.it_head + i - cap; }
        __device__ __forceinline__ SentEntry at(uint32_t i) const { return ring[pos(i)]; }
        __device__ __forceinline__ uint32_t lo(uint32_t i) const { return ring[pos(i)].first; }
        __device__ __forceinline__ uint32_t hi(uint32_t i) const { return i + 1 < s.it_n ? ring[pos(i + 1)].first : s.high; }
        __device__ __forceinline__ uint8_t mk(uint32_t i) const { return (uint8_t)ring[pos(i)].mark; }
    };
    static __device__ __forceinline__ bool lg_candidate(uint8_t m) { return (m & (IT_LOST | IT_RETX | IT_SACKED)) == IT_LOST; }
    // adds (sign 1) or removes (sign -1) an entry of `len` bytes with marks m from the totals
    static __device__ __forceinline__ void lg_count(SndState &s, uint8_t m, uint32_t len, int sign)
    {
        const uint32_t d = sign > 0 ? len : 0u - len, one = sign > 0 ? 1u : 0u - 1u;
        if (U(m & IT_SACKED))
        {
            s.sack_b += d;
            s.sacked_n += one;
        }
        if (U(m & IT_LOST))
            s.lost_b += d;
        if (U(m & IT_RETX))
            s.rtx_b += d;
        if (TW_RARE(lg_candidate(m)))
            s.cand_n += one;
    }
    // entry i's marks become m
    static __device__ void lg_remark(Ledger &L, uint32_t i, uint8_t m)
    {
        const uint32_t k = L.pos(i);
        const uint8_t was = (uint8_t)L.ring[k].mark;
        if (U(was == m))
            return;
        const uint32_t len = L.hi(i) - L.ring[k].first;
        lg_count(L.s, was, len, -1);
        lg_count(L.s, m, len, 1);
        if (U(lg_candidate(m) && !lg_candidate(was) && i < L.s.cand))
            L.s.cand = i;
        L.ring[k].mark = m;
    }
    // a new entry at place i (the entries from i on move up one); its bytes were counted before
    // (a split) or are new (unmarked); false if the ring is full
    static __device__ bool lg_insert(Ledger &L, WorldRun *R, uint32_t i, uint32_t start, uint8_t m)
    {
        SndState &s = L.s;
        if (TW_RARE(s.it_n >= L.cap))
        {
            count(R, EV_RTT_OVF);
            return false;
        }
        for (uint32_t j = s.it_n; U(j > i); j--)
        {
            const uint32_t to = L.pos(j), from = L.pos(j - 1);
            L.ring[to] = L.ring[from];
        }
        L.ring[L.pos(i)] = SentEntry{start, m};
        s.it_n++;
        if (TW_RARE(s.cand > 0 && s.cand >= i))
            s.cand++;
        if (TW_RARE(lg_candidate(m)))
        {
            s.cand_n++;
            s.cand = i < s.cand ? i : s.cand;
        }
        return true;
    }
    // entry i leaves (the ones above move down); the caller has settled its counts
    static __device__ void lg_erase(Ledger &L, uint32_t i)
    {
        SndState &s = L.s;
        for (uint32_t j = i + 1; U(j < s.it_n); j++)
        {
            const uint32_t to = L.pos(j - 1), from = L.pos(j);
            L.ring[to] = L.ring[from];
        }
        s.it_n--;
        if (U(s.cand > i))
            s.cand--;
    }
    // the first entry starting at or after seq
    static __device__ uint32_t lg_find(const Ledger &L, uint32_t seq)
    {
        uint32_t a = 0, b = L.s.it_n;
        while (U(a < b))
        {
            const uint32_t m = (a + b) / 2;
            if (U(L.lo(m) < seq))
                a = m + 1;
            else
                b = m;
        }
        return a;
    }
    static __device__ __forceinline__ uint32_t lg_sent(const SndState &s) { return s.it_n ? s.high - s.una : 0u; }
    // bytes in flight (TcpTxBuffer::BytesInFlight without SACK blocks)
    static __device__ __forceinline__ uint32_t inflight(const SndState &s) { return lg_sent(s) - (s.sack_b + s.lost_b) + s.rtx_b; }
    // a duplicate ACK in recovery: the next unsacked entry after the ones already sacked (Reno's
    // emulation of a SACK block)
    static __device__ void lg_dup_sack(Ledger &L)
    {
        SndState &s = L.s;
        uint32_t i = s.sacked_n + 1;
        for (; U(i < s.it_n); i++)
            if (U(!(L.mk(i) & IT_SACKED)))
            {
                lg_remark(L, i, L.mk(i) | IT_SACKED);
                s.sack_seen = 1;
                s.hisack = L.lo(i);
                return;
            }
    }
    // the oldest entry lost (and no longer sacked or retransmitted)
    static __device__ void lg_head_lost(Ledger &L)
    {
        if (U(L.s.it_n))
            lg_remark(L, 0, (uint8_t)(IT_LOST | (L.mk(0) & ~(IT_SACKED | IT_RETX))));
    }
    // a retransmission timeout: every entry lost, nothing sacked or retransmitted
    static __device__ void lg_all_lost(Ledger &L)
    {
        SndState &s = L.s;
        for (uint32_t i = 0; U(i < s.it_n); i++)
            L.ring[L.pos(i)].mark = IT_LOST;
        s.lost_b = lg_sent(s);
        s.sack_b = s.rtx_b = 0;
        s.sacked_n = 0;
        s.cand_n = s.it_n;
        s.cand = 0;
        s.sack_seen = 0;
        s.hisack = 0;
    }
    // the bytes up to ack are acknowledged (DiscardUpTo): entries wholly below it leave, one cut by
    // it starts there; returns the bytes of the entries that left
    // (pre: the first LG_PRE entries, read together before they are needed: one after another each was
    // a wait of its own)
    static constexpr int LG_PRE = 4;
    static __device__ uint32_t lg_release(Ledger &L, uint32_t ack, const SentEntry *pre)
    {
        SndState &s = L.s;
        uint32_t freed = 0, gone = 0;
        SentEntry e = pre[0];
        while (U(s.it_n))
        {
            SentEntry nx = gone == 0 ? pre[1] : gone == 1 ? pre[2] : pre[3];
            if (TW_RARE(gone + 1 >= LG_PRE && s.it_n > 1))
                nx = L.at(1);
            const uint32_t a = e.first, b = s.it_n > 1 ? nx.first : s.high;
            if (U(b > ack))
            {
                if (TW_RARE(ack > a))
                {
                    // the entry's acknowledged front leaves its mark totals
                    const uint32_t cut = ack - a;
                    s.sack_b -= e.mark & IT_SACKED ? cut : 0u;
                    s.lost_b -= e.mark & IT_LOST ? cut : 0u;
                    s.rtx_b -= e.mark & IT_RETX ? cut : 0u;
                    L.ring[L.pos(0)].first = ack;
                }
                break;
            }
            if (TW_RARE(e.mark))
                lg_remark(L, 0, 0);
            s.it_head = L.pos(1);
            s.it_n--;
            gone++;
            freed += b - a;
            e = nx;
        }
        if (U(gone))
            s.cand = s.cand > gone ? s.cand - gone : 0;
        s.una = ack;
        if (TW_RARE(s.it_n && (e.mark & IT_SACKED)))
        {
            lg_remark(L, 0, (uint8_t)(L.mk(0) & ~IT_SACKED));
            lg_dup_sack(L);
            lg_head_lost(L);
        }
        if (U(s.hisack <= ack))
            s.sack_seen = 0, s.hisack = 0;
        return freed;
    }
    // where the next segment starts: the first retransmission candidate below the highest sack,
    // else new data; false: nothing to send
    static __device__ bool lg_next(Ledger &L, uint32_t *seq)
    {
        SndState &s = L.s;
        for (uint32_t i = s.cand; U(s.cand_n && i < s.it_n); i++)
        {
            if (U(!lg_candidate(L.mk(i))))
                continue;
            s.cand = i;
            if (U(s.sack_seen && L.lo(i) >= s.hisack))
                break;
            *seq = L.lo(i);
            return true;
        }
        if (U(s.high >= s.tail))
            return false;
        *seq = s.high;
        return true;
    }
    // is the oldest entry lost below the highest sack (a fast retransmit due)?
    static __device__ bool lg_head_is_lost(const Ledger &L)
    {
        const SndState &s = L.s;
        return s.sack_seen && s.una < s.hisack && s.it_n && (L.mk(0) & IT_LOST);
    }
    // does a retransmitted, unsacked entry end exactly at x?
    static __device__ bool lg_retx_ends_at(const Ledger &L, uint32_t x)
    {
        const SndState &s = L.s;
        if (U(!s.it_n || x <= s.una || x > s.high))
            return false;
        const uint32_t n = lg_find(L, x);
        if (U(!n || L.hi(n - 1) != x))
            return false;
        const uint8_t m = L.mk(n - 1);
        return (m & IT_RETX) && !(m & IT_SACKED);
    }
    // num bytes sent again from entry i (GetTransmittedSegment): it merges with the next entry
    // when that one is unsacked and equally lost (their retransmitted marks settled first), or is
    // split at num; the result is marked retransmitted. Returns the bytes.
    static __device__ uint32_t lg_resend(Ledger &L, WorldRun *R, uint32_t i, uint32_t num)
    {
        SndState &s = L.s;
        uint32_t len = L.hi(i) - L.lo(i);
        const bool has_next = i + 1 < s.it_n;
        const uint8_t a = L.mk(i), b = has_next ? L.mk(i + 1) : 0;
        const bool mergeable = has_next && !(b & IT_SACKED) && (a & IT_LOST) == (b & IT_LOST);
        const uint32_t most = mergeable ? len + (L.hi(i + 1) - L.lo(i + 1)) : len;
        const uint32_t sz = num < most ? num : most;
        if (U(sz > len))
        {
            // entry i + 1 joins entry i: only one of them may stay retransmitted-marked
            uint8_t nb = b;
            if (U((a ^ b) & IT_RETX))
            {
                if (U(a & IT_RETX))
                    lg_remark(L, i, (uint8_t)(a & ~IT_RETX));
                else
                    lg_remark(L, i + 1, nb = (uint8_t)(b & ~IT_RETX));
            }
            if (U(lg_candidate(nb)))
                s.cand_n--;
            lg_erase(L, i + 1);
            len = L.hi(i) - L.lo(i);
        }
        if (U(sz < len))
            lg_insert(L, R, i + 1, L.lo(i) + sz, L.mk(i));
        if (U(!(L.mk(i) & IT_RETX)))
            lg_remark(L, i, L.mk(i) | IT_RETX);
        return sz;
    }
    // the segment of up to num bytes at seq (CopyFromSequence): new data appends an entry, data
    // sent before is resent from its entry (*retx); a segment across s.high sends only the part
    // below it. 0: nothing (or the ledger cannot hold it)
    static __device__ uint32_t lg_take(Ledger &L, WorldRun *R, uint32_t num, uint32_t seq, bool *retx)
    {
        SndState &s = L.s;
        for (;;)
        {
            const uint32_t sz = s.tail <= seq ? 0u : num < s.tail - seq ? num : s.tail - seq;
            if (U(!sz))
                return 0;
            if (TW_USUAL(s.high <= seq))
            {
                if (U(!lg_insert(L, R, s.it_n, seq, 0)))
                    return 0;
                s.high = seq + sz;
                *retx = false;
                return sz;
            }
            if (TW_RARE(s.high >= seq + sz))
            {
                const uint32_t i = lg_find(L, seq);
                if (U(i >= s.it_n || L.lo(i) != seq))
                {
                    count(R, EV_RTT_OVF);
                    return 0;
                }
                *retx = true;
                return lg_resend(L, R, i, sz);
            }
            num = s.high - seq;
        }
    }

    // -------------------------------------------------------------- RTT
    // Each transmission is noted (first byte, length; the length's top bit once any of it is
    // resent, which removes it from sampling: Karn) in a ring beside the ledger; the oldest
    // unretransmitted record an ACK covers gives a sample (ns-3's RttMeanDeviation, in integer
    // picoseconds with its shifts), and the records it covers leave.
    static __device__ __forceinline__ uint32_t rtt_pos(const SndState &s, uint32_t cap, uint32_t j)
    {
        return s.h_head + j < cap ? s.h_head + j : s.h_head + j - cap;
    }
    static __device__ void rtt_note(Host &x, int f, uint32_t seq, uint32_t sz, bool retx, int64_t now)
    {
        SndState &s = x.S;
        const uint32_t cap = x.cs.it_cap;
        SentNote TW_G *ht = x.B->ht + x.cs.it_off;
        if (TW_RARE(retx))
        {
            // the record holding seq: resent up to seq + sz
            for (uint32_t j = 0; U(j < s.h_n); j++)
            {
                const uint32_t k = rtt_pos(s, cap, j);
                const SentNote e = ht[k];
                if (U(seq >= e.seq && seq - e.seq < (e.cnt & 0x7FFFFFFFu)))
                {
                    ht[k].cnt = 0x80000000u | (seq + sz - e.seq);
                    return;
                }
            }
            return;
        }
        if (TW_RARE(s.h_n >= cap))
        {
            count(x.R, EV_RTT_OVF);
            return;
        }
        ht[rtt_pos(s, cap, s.h_n++)] = SentNote{now, seq, sz};
    }
    // a measurement m: the smoothed RTT and its variation, then the timeout (at least MinRto)
    static __device__ void rtt_sample(SndState &s, int64_t m)
    {
        if (TW_RARE(s.srtt < 0))
        {
            s.srtt = m;
            s.rttvar = m / 2;
        }
        else
        {
            const int64_t err = m - s.srtt, mag = err < 0 ? -err : err;
            s.srtt = ((s.srtt << 3) + err) >> 3;
            s.rttvar = ((s.rttvar << 2) - s.rttvar + mag) >> 2;
        }
        const int64_t spread = 4 * s.rttvar > CLOCK_GRAN_PS ? 4 * s.rttvar : CLOCK_GRAN_PS;
        s.rto = s.srtt + spread > MIN_RTO_PS ? s.srtt + spread : MIN_RTO_PS;
    }
    // (pre: the first RTT_PRE notes, read together with the ledger's first entries)
    static constexpr int RTT_PRE = 3;
    static __device__ void rtt_on_ack(Host &x, uint32_t ack, int64_t now, const SentNote *pre)
    {
        SndState &s = x.S;
        if (TW_RARE(!s.h_n))
            return;
        const uint32_t cap = x.cs.it_cap;
        if (U(!(pre[0].cnt & 0x80000000u) && ack >= pre[0].seq + pre[0].cnt))
            rtt_sample(s, now - pre[0].t);
        for (int i = 0; U(s.h_n); i++, s.h_n--)
        {
            SentNote e = i == 0 ? pre[0] : i == 1 ? pre[1] : pre[2];
            if (TW_RARE(i >= RTT_PRE))
                e = x.B->ht[x.cs.it_off + rtt_pos(s, cap, 0)];
            if (U(e.seq + (e.cnt & 0x7FFFFFFFu) > ack))
                break;
            s.h_head = rtt_pos(s, cap, 1);
        }
    }

    // -------------------------------------------------------------- congestion control
    // Three controllers over the sender's record, each with ns-3's hooks: the slow-start threshold
    // after a loss or an echo (GetSsThresh), the per-ACK measurement (PktsAcked) and the window
    // growth (IncreaseWindow). Cubic follows ns-3's TcpCubic (with HyStart), DCTCP its alpha EWMA
    // per window of data, NewReno slow start and congestion avoidance.
    static __device__ __forceinline__ uint32_t to_u32(double d) { return (uint32_t)(uint64_t)(int64_t)d; }
    static __device__ void cubic_round_start(Host &x, int64_t now)
    {
        SndState &s = x.S;
        SndRec TW_G &c = x.B->snd[x.sf];
        c.cub_roundstart = now;
        c.cub_lastack = now;
        c.cub_endseq = s.st == S_EST ? s.high + 1 : 0;
        c.cub_currrtt = INT64_MIN;
        c.cub_samples = 0;
    }
    // ACKs per window increment in congestion avoidance (TcpCubic::Update): the cubic curve's
    // target at now + delay_min against the window, bounded by the TCP-friendly estimate
    static __device__ uint32_t cubic_acks_per_inc(Host &x, uint32_t segs, int64_t now)
    {
        SndState &s = x.S;
        SndRec TW_G &c = x.B->snd[x.sf];
        const double C = 0.4, BETA = 0.7;
        const uint32_t w = s.cwnd / MSS;
        c.cub_ackcnt += segs;
        if (U(c.cub_epoch == INT64_MIN))
        {
            // a new epoch: the curve's origin and the time K to reach it
            c.cub_epoch = now;
            c.cub_ackcnt = segs;
            c.cub_tcpcwnd = w;
            const bool below = c.cub_lastmax > w;
            c.cub_origin = below ? c.cub_lastmax : w;
            c.cub_k = below ? tw_pow((double)(c.cub_lastmax - w) / C, 1 / 3.) : 0.0;
        }
        const int64_t dt = (int64_t)((uint64_t)now + (uint64_t)c.cub_delaymin - (uint64_t)c.cub_epoch);
        const double t = tw_seconds(dt), k = c.cub_k;
        const uint32_t off = to_u32(C * tw_pow(t < k ? k - t : t - k, 3));
        const uint32_t target = t < k ? c.cub_origin - off : c.cub_origin + off;
        uint32_t n = target > w ? w / (target - w) : 100 * w;
        if (U(!c.cub_lastmax && n > 20))
            n = 20;
        // the TCP-friendly window: one segment per `per` ACKs
        const uint32_t per = (w * to_u32(8 * (1024 + BETA * 1024) / 3 / (1024 - BETA * 1024))) >> 3;
        for (; U(per > 0 && c.cub_ackcnt > per); c.cub_ackcnt -= per)
            c.cub_tcpcwnd++;
        if (U(c.cub_tcpcwnd > w))
        {
            const uint32_t cap = w / (c.cub_tcpcwnd - w);
            n = n > cap ? cap : n;
        }
        return n < 2 ? 2 : n;
    }
    // HyStart's delay check and the minimum delay (TcpCubic::PktsAcked)
    static __device__ void cubic_measure(Host &x, int64_t now)
    {
        SndState &s = x.S;
        SndRec TW_G &c = x.B->snd[x.sf];
        const int64_t ACK_DELTA = 2000000000, DELAY_MIN = 4000000000, DELAY_MAX = 1000000000000, CUBIC_DELTA = 10000000000;
        if (U(c.cub_epoch != INT64_MIN && now - c.cub_epoch < CUBIC_DELTA))
            return;
        const int64_t rtt = s.srtt;
        if (U(c.cub_delaymin == INT64_MIN || rtt < c.cub_delaymin))
            c.cub_delaymin = rtt;
        const bool slow_start_window = s.cwnd <= s.ssthresh && s.cwnd >= 16 * MSS;
        if (U(!slow_start_window || s.cub_found))
            return;
        if (U(now - c.cub_lastack <= ACK_DELTA))
        {
            // the ACK train
            c.cub_lastack = now;
            if (U(now - c.cub_roundstart > c.cub_delaymin))
                s.cub_found = 1;
        }
        if (U(c.cub_samples >= 8))
        {
            // the delay increase
            const int64_t dm = c.cub_delaymin, eta = dm < DELAY_MIN ? DELAY_MIN : dm > DELAY_MAX ? DELAY_MAX : dm;
            if (U(c.cub_currrtt > dm + eta))
                s.cub_found = 1;
        }
        else
        {
            if (U(c.cub_currrtt == INT64_MIN || rtt < c.cub_currrtt))
                c.cub_currrtt = rtt;
            c.cub_samples++;
        }
        if (U(s.cub_found))
            s.ssthresh = s.cwnd;
    }
    static __device__ void cubic_grow(Host &x, uint32_t segs, uint32_t ack, int64_t now)
    {
        SndState &s = x.S;
        SndRec TW_G &c = x.B->snd[x.sf];
        if (U(!s.cwnd_limited))
            return;
        if (U(s.cwnd < s.ssthresh))
        {
            if (U(ack + 1 > c.cub_endseq))
                cubic_round_start(x, now);
            s.cwnd += segs * MSS;
            segs = 0;
        }
        if (U(segs == 0 || s.cwnd < s.ssthresh))
            return;
        c.cub_cnt += segs;
        const uint32_t n = cubic_acks_per_inc(x, segs, now);
        if (U(c.cub_cnt >= n))
        {
            c.cub_cnt -= n;
            s.cwnd += MSS;
        }
    }
    // the threshold after a loss: beta times the window (fast convergence lowers the remembered
    // maximum when the window is below it); a new epoch starts
    static __device__ uint32_t cubic_ssthresh(Host &x)
    {
        SndState &s = x.S;
        SndRec TW_G &c = x.B->snd[x.sf];
        const double BETA = 0.7;
        const uint32_t w = s.cwnd / MSS;
        c.cub_lastmax = w < c.cub_lastmax ? to_u32((w * (1 + BETA)) / 2) : w;
        c.cub_epoch = INT64_MIN;
        const uint32_t th = to_u32(w * BETA);
        return (th < 2 ? 2 : th) * MSS;
    }
    static __device__ void cubic_timeout(Host &x, int64_t now)
    {
        SndState &s = x.S;
        SndRec TW_G &c = x.B->snd[x.sf];
        c.cub_origin = 0;
        c.cub_k = 0;
        c.cub_ackcnt = 0;
        c.cub_tcpcwnd = 0;
        c.cub_delaymin = INT64_MIN;
        s.cub_found = 0;
        cubic_round_start(x, now);
    }
    // DCTCP's alpha: the marked share of the bytes acknowledged over each window of data
    static __device__ void dctcp_measure(SndState &s, uint32_t segs, uint32_t ack)
    {
        const uint32_t bytes = segs * MSS;
        s.acked_total += bytes;
        if (U(s.ecn_s == E_ECE_RCVD))
            s.acked_ecn += bytes;
        if (U(!s.next_seq_flag))
        {
            s.next_seq_flag = 1;
            s.next_seq = s.nxt;
        }
        if (U(ack < s.next_seq))
            return;
        const double share = s.acked_total ? (double)s.acked_ecn / s.acked_total : 0.0;
        s.alpha = __builtin_fma(1.0 - DCTCP_G, s.alpha, DCTCP_G * share);
        s.next_seq = s.nxt;
        s.acked_total = s.acked_ecn = 0;
    }
    // DCTCP's growth: slow start up to the threshold, then a segment per window's worth of ACKs
    static __device__ void dctcp_grow(SndState &s, uint32_t segs)
    {
        if (U(s.cwnd < s.ssthresh))
        {
            if (U(segs))
            {
                const uint64_t w = (uint64_t)s.cwnd + (uint64_t)segs * MSS;
                s.cwnd = (uint32_t)(w < s.ssthresh ? w : s.ssthresh);
            }
            return;
        }
        const uint32_t per = s.cwnd / MSS ? s.cwnd / MSS : 1;
        uint32_t acc = s.cwnd_cnt;
        if (U(acc >= per))
        {
            acc = 0;
            s.cwnd += MSS;
        }
        acc += segs;
        if (U(acc >= per))
        {
            s.cwnd += acc / per * MSS;
            acc %= per;
        }
        s.cwnd_cnt = acc;
    }
    // NewReno: one segment per ACK in slow start, then about MSS^2 / cwnd bytes (at least 1)
    static __device__ void newreno_grow(SndState &s, uint32_t segs)
    {
        if (U(s.cwnd < s.ssthresh && segs))
        {
            s.cwnd += MSS;
            segs--;
        }
        if (U(s.cwnd >= s.ssthresh && segs))
        {
            const double add = (double)MSS * MSS / s.cwnd;
            s.cwnd += (uint32_t)(add < 1.0 ? 1.0 : add);
        }
    }
    static __device__ uint32_t cc_ssthresh(Host &x, SndState &s, uint32_t in_flight)
    {
        if (U(x.cubic))
            return cubic_ssthresh(x);
        if (U(x.dctcp))
            return (uint32_t)((1.0 - s.alpha / 2.0) * s.cwnd);
        return in_flight / 2 > 2 * MSS ? in_flight / 2 : 2 * MSS;
    }
    static __device__ void cc_acked(Host &x, SndState &s, uint32_t segs, uint32_t ack, int64_t now)
    {
        if (U(x.cubic))
            cubic_measure(x, now);
        else if (U(x.dctcp))
            dctcp_measure(s, segs, ack);
    }
    static __device__ void cc_grow(Host &x, SndState &s, uint32_t segs, uint32_t ack, int64_t now)
    {
        if (U(x.cubic))
            cubic_grow(x, segs, ack, now);
        else if (U(x.dctcp))
            dctcp_grow(s, segs);
        else
            newreno_grow(s, segs);
    }

    // -------------------------------------------------------------- the sending endpoint
    // A connection's sending side (TcpSocketBase with its TxBuffer, as the model restates it):
    // segments leave through the host's queue, the retransmission timer follows the oldest
    // unacknowledged byte, and ACKs drive ns-3's congestion states (open, disorder, CWR,
    // recovery, loss). Every function works on the record of the event's connection (Host::S).
    // one segment of up to max_size bytes at seq (SendDataPacket): CWR on the first new segment
    // after an echo, FIN on the last byte once the application closed; the timer is armed if
    // idle; *o: the frame; returns its bytes
    static __device__ uint32_t tx_segment(Host &x, int f, uint32_t seq, uint32_t max_size, int64_t now, Out *o)
    {
        Batch &B = *x.B;
        SndState &s = x.S;
        Ledger L(x);
        bool retx = false;
        const uint32_t len = lg_take(L, x.R, max_size, seq, &retx);
        if (TW_RARE(!len))
            return 0;
        uint8_t flags = F_DATA;
        if (U(!retx && s.ecn_s == E_ECE_RCVD && s.ecn_echo_seq > s.ecn_cwr_seq))
        {
            flags |= F_CWR;
            s.ecn_s = E_CWR_SENT;
            s.ecn_cwr_seq = seq;
        }
        if (TW_RARE((s.fin & FIN_CLOSE) && seq + len == s.tail))
        {
            flags |= F_FIN;
            s.fin |= FIN_SENT;
        }
        *o = out_of(flags, seq, 0, (uint16_t)(len + 42), false);
        if (TW_RARE(retx))
        {
            count(x.R, EV_RETX);
            count(x.R, EV_RETX_BY_STATE + s.cong);
        }
        if (TW_RARE(s.rto_at < 0))
        {
            s.rto_at = now + s.rto;
            timer_chain(x, B.rchain, f, s.rto);
        }
        s.cwnd_limited = s.cwnd < inflight(s) + MSS;
        rtt_note(x, f, seq, len, retx, now);
        s.high = seq + len > s.high ? seq + len : s.high;
        x.max_it = s.it_n > x.max_it ? s.it_n : x.max_it;
        return len;
    }
    // a segment asked for by the handler itself
    static __device__ void tx_now(Host &x, int f, uint32_t seq, int64_t now)
    {
        Out o;
        if (U(tx_segment(x, f, seq, MSS, now, &o)))
            emit(x, f, o.flags, o.sa, 0, o.len, false, now);
    }
    // sending while the window has room (SendPendingData), a segment at a time (fill_next) once the
    // handler is through: whole segments only, unless the rest of the data is smaller; nothing more
    // once a FIN is out in the open state
    static __device__ __forceinline__ void tx_fill(Host &x)
    {
        x.fill = true;
        x.fill_n = 0;
    }
    static __device__ bool fill_next(Host &x, int f, int64_t now, Out *o)
    {
        SndState &s = x.S;
        if (TW_RARE(s.st != S_EST || x.fill_n >= 4096))
            return false;
        x.fill_n++;
        Ledger L(x);
        const bool fin_out = (s.fin & (FIN_SENT | FIN_ACKED)) == FIN_SENT;
        if (TW_RARE(s.cong == C_OPEN && fin_out))
            return false;
        const uint32_t pipe = inflight(s), room = s.cwnd > pipe ? s.cwnd - pipe : 0;
        uint32_t seq;
        if (U(!room || !lg_next(L, &seq)))
            return false;
        if (TW_RARE(room < MSS && s.tail - seq > room))
            return false; // (no runt segment while more data waits)
        s.nxt = seq;
        const uint32_t len = tx_segment(x, f, seq, room < MSS ? room : MSS, now, o);
        if (TW_RARE(!len))
            return false;
        s.nxt = seq + len;
        return true;
    }
    // one segment again from the first candidate (else the oldest byte)
    static __device__ void tx_resend_one(Host &x, int f, int64_t now)
    {
        SndState &s = x.S;
        Ledger L(x);
        uint32_t seq;
        if (U(!lg_next(L, &seq)))
            seq = s.una;
        if (U(s.una >= s.tail))
            return;
        s.nxt = seq;
        tx_now(x, f, seq, now);
    }
    // the retransmission timer after new data is acknowledged (NewAck): restarted from the RTT
    // estimate when asked, stopped once all data (and no FIN) is acknowledged
    static __device__ void rto_after_ack(Host &x, int f, uint32_t ack, bool restart, int64_t now)
    {
        SndState &s = x.S;
        if (TW_USUAL(restart))
        {
            const int64_t base = s.srtt >= 0 ? s.srtt : INIT_RTT_PS, spread = 4 * s.rttvar > CLOCK_GRAN_PS ? 4 * s.rttvar : CLOCK_GRAN_PS;
            s.rto = base + spread > MIN_RTO_PS ? base + spread : MIN_RTO_PS;
            s.rto_at = now + s.rto;
            timer_chain(x, x.B->rchain, f, s.rto);
        }
        if (TW_RARE(ack >= s.tail && !(s.fin & FIN_SENT)))
            s.rto_at = -1;
        s.nxt = ack > s.nxt ? ack : s.nxt;
    }
    // fast retransmit: the oldest segment lost, the window halved (or as the controller says),
    // the segment sent again
    static __device__ void fast_retransmit(Host &x, int f, int64_t now)
    {
        SndState &s = x.S;
        Ledger L(x);
        lg_dup_sack(L);
        lg_head_lost(L);
        s.cong = C_RECOVERY;
        s.recover = s.high;
        s.recover_active = 1;
        s.ssthresh = cc_ssthresh(x, s, inflight(s) + MSS);
        s.cwnd = s.ssthresh;
        tx_now(x, f, s.una, now);
    }
    // messages wholly acknowledged complete (their completion time is the flow's); the connection
    // is done with its last message (and its FIN, if it sends one)
    static __device__ void msgs_complete(Host &x, int f, int64_t now)
    {
        Batch &B = *x.B;
        SndState &s = x.S;
        for (; U(s.m_dn < s.m_wr); s.m_dn++)
        {
            const int m = x.cs.m_first + s.m_dn;
            if (U(s.una < (s.m_dn + 1 == s.m_wr ? s.tail : B.mg_end[m]))) // (the last one written ends at the tail)
                break;
            B.mg_done[m] = now;
            atomicAdd(&x.R->flows_done, 1u);
        }
        if (TW_RARE(s.m_dn == x.cs.m_cnt && (!x.cs.fin_on || (s.fin & FIN_ACKED))))
        {
            s.st = S_DONE;
            s.rto_at = -1;
        }
    }
    // DCTCP's response to an echo (EnterCwr): a new echo beyond the last one cuts the window once
    static __device__ void ack_echo(Host &x, SndState &s, uint32_t ack, bool ece, bool advancing)
    {
        if (U(!(advancing && x.dctcp && ece)))
        {
            if (U(!ece && s.ecn_s == E_ECE_RCVD))
                s.ecn_s = E_IDLE;
            return;
        }
        if (TW_RARE((int64_t)ack <= s.ecn_echo_seq))
            return;
        s.ecn_echo_seq = ack;
        s.ecn_s = E_ECE_RCVD;
        if (U(s.cong == C_CWR))
            return;
        s.ssthresh = cc_ssthresh(x, s, inflight(s));
        s.cwnd = s.ssthresh;
        s.cong = C_CWR;
        s.recover = s.high;
    }
    // a duplicate ACK (below s.high): counted outside recovery and loss; in recovery it sacks
    // the next entry; the third (or a lost head below the highest sack) starts fast retransmit
    static __device__ void ack_duplicate(Host &x, int f, SndState &s, uint32_t una_before, int64_t now)
    {
        uint8_t state = s.cong;
        if (U(state == C_LOSS))
            return;
        if (U(state != C_RECOVERY))
            s.dupacks++;
        if (U(state == C_OPEN))
            s.cong = state = C_DISORDER;
        Ledger L(x);
        if (TW_RARE(state == C_RECOVERY))
            lg_dup_sack(L);
        else if (U(state == C_DISORDER))
        {
            const bool third = s.dupacks == (uint32_t)DUPTHRESH && (!s.recover_active || una_before >= s.recover);
            if (U(third || lg_head_is_lost(L)))
                fast_retransmit(x, f, now);
        }
    }
    // an ACK of new data below the recovery point: partial (recovery: the next hole is resent,
    // the timer restarted on the first partial ACK only) or during loss (slow start again)
    static __device__ void ack_partial(Host &x, int f, SndState &s, uint32_t ack, uint32_t segs, int64_t now)
    {
        if (U(s.cong == C_RECOVERY))
        {
            Ledger L(x);
            lg_head_lost(L);
            if (U(!lg_retx_ends_at(L, ack + MSS)))
                tx_resend_one(x, f, now);
            cc_acked(x, s, 1, ack, now);
            rto_after_ack(x, f, ack, s.first_partial, now);
            s.first_partial = 0;
            return;
        }
        cc_acked(x, s, segs, ack, now);
        cc_grow(x, s, segs, ack, now);
        rto_after_ack(x, f, ack, true, now);
    }
    // an ACK of new data otherwise: disorder and the ends of recovery and loss return to the
    // open state (the window settles at the threshold after recovery); open grows the window
    static __device__ void ack_advance(Host &x, int f, SndState &s, uint32_t ack, uint32_t una_before, uint32_t segs, uint32_t dups, int64_t now)
    {
        const uint8_t state = s.cong;
        if (U(state == C_CWR))
        {
            cc_acked(x, s, segs, ack, now);
            rto_after_ack(x, f, ack, true, now);
            return;
        }
        switch (state)
        {
        case C_OPEN:
            cc_acked(x, s, segs, ack, now);
            break;
        case C_DISORDER:
            if (U(segs >= dups))
                cc_acked(x, s, segs - dups, ack, now);
            break;
        case C_RECOVERY:
            segs = (ack - una_before) / MSS; // (the segments of the whole recovery)
            cc_acked(x, s, segs, ack, now);
            s.first_partial = 1;
            s.dupacks = 0;
            break;
        default: // C_LOSS
            segs = (ack - s.recover) / MSS;
            cc_acked(x, s, segs, ack, now);
            s.first_partial = 1;
            break;
        }
        s.cong = C_OPEN;
        if (U(ack >= s.recover))
            s.recover_active = 0;
        if (TW_RARE(state == C_RECOVERY))
        {
            rto_after_ack(x, f, ack, true, now);
            s.cwnd = s.ssthresh;
        }
        cc_grow(x, s, segs, ack, now);
        rto_after_ack(x, f, ack, true, now);
    }
    // an ACK at the sender (ReceivedAck + ProcessAck, no SACK option, classic recovery): old ones
    // are ignored; the RTT sample and the ledger come first, then the CWR end and the echo, then
    // by kind - a duplicate, an ACK of nothing new at s.high, one beyond it, or new data - and at
    // last the FIN's acknowledgment, the completed messages and more sending
    static __device__ void ack_in(Host &x, int f, uint32_t ack, bool ece, int64_t now)
    {
        SndState &s = x.S;
        if (TW_RARE(s.st != S_EST || ack < s.una))
            return;
        const uint32_t una_before = s.una;
        const bool advancing = ack > una_before;
        Ledger L(x);
        // (past the rings' ends their first entries again: read, not used)
        SentNote notes[RTT_PRE];
        SentEntry entries[LG_PRE];
#pragma unroll
        for (int i = 0; i < RTT_PRE; i++)
            notes[i] = x.B->ht[x.cs.it_off + rtt_pos(s, L.cap, (uint32_t)i < s.h_n ? i : 0)];
#pragma unroll
        for (int i = 0; i < LG_PRE; i++)
            entries[i] = L.at((uint32_t)i < s.it_n ? i : 0);
        rtt_on_ack(x, ack, now, notes);
        const uint32_t acked = advancing ? lg_release(L, ack, entries) : 0;
        if (TW_RARE(s.cong == C_CWR && ack > s.recover))
        {
            s.cong = C_OPEN;
            s.cwnd = s.ssthresh;
        }
        ack_echo(x, s, ack, ece, advancing);
        const uint32_t dups = s.dupacks;
        if (TW_RARE(!advancing))
        {
            if (U(ack < s.high))
            {
                ack_duplicate(x, f, s, una_before, now);
                cc_acked(x, s, 1, ack, now);
            }
            else if (U(ack > s.high))
                s.nxt = ack;
        }
        else
        {
            // whole segments acknowledged, the remainders carried over
            uint32_t segs = acked / MSS;
            s.ack_rem += acked % MSS;
            if (TW_RARE(s.ack_rem >= MSS))
            {
                s.ack_rem -= MSS;
                segs++;
            }
            s.dupacks = 0;
            if (TW_RARE(ack < s.recover && (s.cong == C_RECOVERY || s.cong == C_LOSS)))
                ack_partial(x, f, s, ack, segs, now);
            else
                ack_advance(x, f, s, ack, una_before, segs, dups, now);
        }
        if (TW_RARE((s.fin & FIN_SENT) && !s.it_n && ack == s.high + 1))
            s.fin |= FIN_ACKED;
        if (U(advancing))
        {
            msgs_complete(x, f, now);
            if (TW_RARE(s.st == S_DONE))
                return;
        }
        tx_fill(x);
    }
    // the retransmission timeout: every outstanding segment lost, the timeout doubled (to 60 s at
    // most), one segment's window, then sending again
    static __device__ void rto_fire(Host &x, int f, int64_t now)
    {
        SndState &s = x.S;
        s.rto_at = -1;
        if (U(s.st != S_EST))
            return;
        if (U(s.una >= s.tail))
        {
            if (U((s.fin & (FIN_SENT | FIN_ACKED)) == FIN_SENT))
                count(x.R, EV_RTT_OVF);
            return;
        }
        count(x.R, EV_RTO);
        const uint32_t was_in_flight = inflight(s);
        Ledger L(x);
        lg_all_lost(L);
        s.dupacks = 0;
        s.recover = s.high;
        s.recover_active = 1;
        s.rto = 2 * s.rto < 60000000000000ll ? 2 * s.rto : 60000000000000ll;
        s.h_n = 0;
        s.ssthresh = cc_ssthresh(x, s, was_in_flight);
        if (U(x.cubic))
            cubic_timeout(x, now);
        s.cong = C_LOSS;
        s.cwnd = MSS;
        tx_fill(x);
    }

    // -------------------------------------------------------------- the receiving endpoint
    // A connection's receiving side: the SYN-ACK and its retries, in-order delivery through the
    // reassembly ring, delayed ACKs (every second segment or after the delay), DCTCP's CE echo
    // state machine, and the passive close (FIN+ACK, LAST_ACK with its retries).
    // an ACK now (the delayed one, if pending, is folded in); ECE while echoing CE unless no_ece,
    // always with force_ece
    static __device__ void rcv_ack(Host &x, int f, uint32_t ack, bool force_ece, bool no_ece, int64_t now)
    {
        RcvState &r = x.Q;
        const bool echoing = r.ecn_r == E_CE_RCVD || r.ecn_r == E_SENDING_ECE;
        const bool ece = force_ece || (!no_ece && echoing);
        if (TW_RARE(!force_ece && ece))
            r.ecn_r = E_SENDING_ECE;
        r.delack_at = -1;
        r.delack_count = 0;
        emit(x, f, (uint8_t)(F_ACK | (ece ? F_ECE : 0)), 0, ack, CTRL_FRAME, true, now);
    }
    static __device__ void rcv_synack(Host &x, int f, int64_t now)
    {
        RcvState &r = x.Q;
        const int64_t backoff = CONN_TIMEOUT_PS << r.srv_syn_n++;
        if (U(r.r_synack_t < 0))
            r.r_synack_t = now;
        emit(x, f, F_SYN | F_ACK, 0, 0, SYN_FRAME, true, now);
        if (U(r.srv_syn_at >= 0))
            return;
        r.srv_syn_at = now + backoff;
        timer_chain(x, x.B->dchain, f, backoff);
    }
    static __device__ __forceinline__ void rcv_established(RcvState &r)
    {
        if (U(r.r_est))
            return;
        r.r_est = 1;
        r.srv_syn_at = -1;
    }
    // DCTCP's receiver: a change of the CE state flushes a pending delayed ACK for the bytes
    // before it, with the previous state's ECE (set when leaving CE, cleared when entering it)
    static __device__ void rcv_ce_edge(Host &x, int f, bool ce, int64_t now)
    {
        RcvState &r = x.Q;
        const bool flips = (bool)r.ce_state != ce;
        if (TW_RARE(flips && r.reserved && r.prior_flag))
            rcv_ack(x, f, r.prior_rcv_nxt, !ce, ce, now);
        r.ce_state = ce ? 1 : 0;
        if (U(ce))
            r.ecn_r = E_CE_RCVD;
        else if (U(r.ecn_r == E_CE_RCVD || r.ecn_r == E_SENDING_ECE))
            r.ecn_r = E_IDLE;
        r.prior_flag = 1;
        r.prior_rcv_nxt = r.rcv_nxt;
    }
    static __device__ void rcv_ecn_in(Host &x, int f, const Frame &p, int64_t now)
    {
        if (U(!x.dctcp))
            return;
        RcvState &r = x.Q;
        if (TW_RARE((p.flags & F_CE) && r.ecn_ce_seq < (int64_t)p.sa))
        {
            r.ecn_ce_seq = p.sa;
            r.ecn_r = E_CE_RCVD;
            rcv_ce_edge(x, f, true, now);
        }
        else if (U(p.flags & F_ECT))
            rcv_ce_edge(x, f, false, now);
    }
    // the CE state of the sending side's own ECN (ACKs carrying CE)
    static __device__ void snd_ecn_in(Host &x, SndState &s, const Frame &p)
    {
        if (U(!x.dctcp))
            return;
        if (TW_RARE((p.flags & F_CE) && !(s.s_ce & 1)))
        {
            s.s_ce = 3;
            s.ecn_s = E_CE_RCVD;
            return;
        }
        if (U(!(p.flags & F_ECT)))
            return;
        s.s_ce &= ~2;
        if (U(s.ecn_s == E_CE_RCVD || s.ecn_s == E_SENDING_ECE))
            s.ecn_s = E_IDLE;
    }
    // The reassembly ring (TcpRxBuffer::Add): out-of-order blocks, disjoint and sorted, in a ring
    // per connection. [seq, end) above rcv_nxt joins the blocks it touches; a block reaching
    // rcv_nxt is delivered. False if nothing was new (or the ring is full).
    static __device__ bool reasm_add(Host &x, int f, uint32_t seq, uint32_t end)
    {
        Batch &B = *x.B;
        RcvState &r = x.Q;
        const uint32_t from = seq > r.rcv_nxt ? seq : r.rcv_nxt;
        if (TW_RARE(from >= end))
            return false;
        uint32_t *lo = B.oo_s + x.cr.oo_off, *hi = B.oo_e + x.cr.oo_off;
        const uint32_t cap = x.cr.oo_cap, h0 = r.ooo_h;
        uint32_t n = r.ooo_n;
        if (TW_USUAL(n == 0 && from == r.rcv_nxt))
        {
            // in order, nothing held: delivered without a place in the ring
            r.rcv_nxt = end;
            r.ooo_h = 0;
            if (TW_RARE(r.r_fin >= 0 && r.rcv_nxt == (uint32_t)r.r_fin))
                r.rcv_nxt++; // (the FIN's sequence number)
            return true;
        }
        auto at = [&](uint32_t i) { return h0 + i < cap ? h0 + i : h0 + i - cap; };
        // the first block ending at or after `from`
        uint32_t i = n;
        if (U(n && hi[at(n - 1)] >= from))
        {
            uint32_t a = 0, b = n - 1;
            while (U(a < b))
            {
                const uint32_t m = (a + b) / 2;
                if (U(hi[at(m)] < from))
                    a = m + 1;
                else
                    b = m;
            }
            i = a;
        }
        if (U(i < n && lo[at(i)] <= from && hi[at(i)] >= end))
            return false; // (all of it is held already)
        // blocks i .. j - 1 touch [from, end): they merge into one
        uint32_t j = i, nlo = from, nhi = end;
        for (; U(j < n && lo[at(j)] <= nhi); j++)
        {
            nlo = lo[at(j)] < nlo ? lo[at(j)] : nlo;
            nhi = hi[at(j)] > nhi ? hi[at(j)] : nhi;
        }
        if (U(j == i))
        {
            // a new block at i
            if (U(n >= cap))
            {
                count(x.R, EV_OOO_OVF);
                return false;
            }
            for (uint32_t k = n; U(k > i); k--)
            {
                lo[at(k)] = lo[at(k - 1)];
                hi[at(k)] = hi[at(k - 1)];
            }
            n++;
        }
        else if (U(j - i > 1))
        {
            // the merged blocks after the first close up
            const uint32_t gone = j - i - 1;
            for (uint32_t k = j; U(k < n); k++)
            {
                lo[at(k - gone)] = lo[at(k)];
                hi[at(k - gone)] = hi[at(k)];
            }
            n -= gone;
        }
        lo[at(i)] = nlo;
        hi[at(i)] = nhi;
        uint32_t head = h0;
        if (U(from == r.rcv_nxt))
        {
            // the first block is in order now: delivered
            r.rcv_nxt = hi[at(0)];
            head = at(1);
            n--;
        }
        r.ooo_n = n;
        r.ooo_h = n ? head : 0;
        if (TW_RARE(r.r_fin >= 0 && r.rcv_nxt == (uint32_t)r.r_fin))
            r.rcv_nxt++; // (the FIN's sequence number)
        return true;
    }
    static __device__ __forceinline__ bool rcv_fin_in(const RcvState &r) { return r.r_fin >= 0 && (uint32_t)r.r_fin < r.rcv_nxt; }
    static __device__ __forceinline__ int64_t rcv_rto(const RcvState &r)
    {
        const int64_t base = r.r_srtt >= 0 ? r.r_srtt : INIT_RTT_PS, spread = 4 * r.r_rttvar > CLOCK_GRAN_PS ? 4 * r.r_rttvar : CLOCK_GRAN_PS;
        return base + spread;
    }
    // FIN+ACK of the passive close, with its retransmission timer (at least MinRto) if none runs
    static __device__ void rcv_fin_ack(Host &x, int f, int64_t now)
    {
        RcvState &r = x.Q;
        r.delack_at = -1;
        r.delack_count = 0;
        emit(x, f, F_ACK | F_FIN, 0, r.rcv_nxt, CTRL_FRAME, true, now);
        if (U(r.r_frx_at >= 0))
            return;
        const int64_t t = rcv_rto(r) > MIN_RTO_PS ? rcv_rto(r) : MIN_RTO_PS;
        r.r_frx_at = now + t;
        timer_chain(x, x.B->fchain, f, t);
    }
    // the peer closed: LAST_ACK, our FIN+ACK, and the LastAck timer with its retries
    static __device__ void rcv_peer_closed(Host &x, int f, int64_t now)
    {
        RcvState &r = x.Q;
        r.r_st = R_LAST_ACK;
        rcv_fin_ack(x, f, now);
        r.r_last_n = DATA_RETRIES;
        const int64_t t = rcv_rto(r);
        r.r_last_at = now + t;
        timer_chain(x, x.B->dchain, f, t);
    }
    static __device__ __forceinline__ void rcv_closed(RcvState &r)
    {
        r.r_st = R_CLOSED;
        r.delack_at = r.r_last_at = r.r_frx_at = -1;
    }
    // data delivered to the ring: an immediate ACK for anything out of order (a gap left, or one
    // filled), for nothing new, or for every second segment; else the delayed ACK
    static __device__ void rcv_data(Host &x, int f, uint32_t seq, uint32_t len, bool fin, int64_t now)
    {
        RcvState &r = x.Q;
        const uint32_t before = r.rcv_nxt;
        if (TW_RARE(!reasm_add(x, f, seq, seq + len)))
        {
            rcv_ack(x, f, r.rcv_nxt, false, false, now);
            return;
        }
        if (TW_RARE(!fin && before < r.rcv_nxt && rcv_fin_in(r)))
        {
            rcv_peer_closed(x, f, now);
            return;
        }
        const bool irregular = r.ooo_n > 0 || r.rcv_nxt > before + len;
        const uint32_t held = r.delack_count + 1u;
        if (U(irregular || held >= DELACK_COUNT))
        {
            r.reserved = 0;
            rcv_ack(x, f, r.rcv_nxt, false, false, now);
            return;
        }
        r.delack_count = (uint8_t)held;
        r.reserved = 1;
        if (U(r.delack_at >= 0))
            return;
        r.delack_at = now + DELACK_PS;
        timer_chain(x, x.B->dchain, f, DELACK_PS);
    }
    // a data (or FIN) segment at the receiver: old data in an established connection is answered
    // with an ACK (in LAST_ACK: anything but the next byte); the CE state; a CWR ends the echo;
    // the first segment establishes; in LAST_ACK only the close's ACK counts; a FIN is taken in
    // order, marks the end and closes passively once delivered
    static __device__ void rcv_segment(Host &x, int f, const Frame &p, int64_t now)
    {
        RcvState &r = x.Q;
        if (TW_RARE(!r.r_up || r.r_st == R_CLOSED))
            return;
        const bool fin = p.flags & F_FIN;
        const uint32_t seq = p.sa, len = (p.flags & F_DATA) ? p.len - 42u : 0u, end = seq + len;
        if (U(len && r.r_est))
        {
            const bool stale = r.r_st == R_LAST_ACK ? seq != r.rcv_nxt : end < r.rcv_nxt;
            if (TW_RARE(stale))
            {
                rcv_ack(x, f, r.rcv_nxt, false, true, now);
                return;
            }
        }
        rcv_ecn_in(x, f, p, now);
        if (TW_RARE((p.flags & F_CWR) && r.r_est && r.r_st == R_OPEN && r.ecn_r != E_CE_RCVD))
            r.ecn_r = E_IDLE;
        if (TW_RARE(!r.r_est))
        {
            if (U(fin && seq != r.rcv_nxt))
                return;
            rcv_established(r);
        }
        if (TW_RARE(r.r_st == R_LAST_ACK))
        {
            if (U(fin || seq == r.rcv_nxt))
                rcv_closed(r);
            return;
        }
        if (TW_USUAL(!fin))
        {
            rcv_data(x, f, seq, len, false, now);
            return;
        }
        if (U(seq < r.rcv_nxt))
            return;
        r.r_fin = end;
        if (U(r.rcv_nxt == end))
            r.rcv_nxt++;
        if (U(len))
            rcv_data(x, f, seq, len, true, now);
        if (U(rcv_fin_in(r)))
            rcv_peer_closed(x, f, now);
    }

    // -------------------------------------------------------------- application and dispatch
    static __device__ void add_active(Host &x, bool snd, int f)
    {
        int32_t *n = snd ? x.B->n_snd : x.B->n_rcv;
        const int k = n[x.h];
        if (U(k >= MAX_ACTIVE))
        {
            count(x.R, EV_ACTIVE_OVF);
            return;
        }
        (snd ? x.B->act_snd : x.B->act_rcv)[(size_t)x.h * MAX_ACTIVE + k] = f;
        n[x.h] = k + 1;
    }
    // the application writes its due messages (FlowSender::Write); Socket::Send defers
    // SendPendingData by 1 ps when the window has room (src/step.cuh:2120-2145); at: the write's chain
    static __device__ void app_write(Host &x, int f, int64_t now, const Chain &at)
    {
        Batch &B = *x.B;
        SndState &s = x.S;
        if (U(s.m_wr >= s.m_due))
            return;
        for (; U(s.m_wr < s.m_due); s.m_wr++)
        {
            const int m = x.cs.m_first + s.m_wr;
            B.mg_est[m] = now;
            s.tail = B.mg_end[m];
        }
        if (U(x.cs.fin_on && s.m_wr == x.cs.m_cnt))
            s.fin |= FIN_CLOSE;
        if (U(s.cwnd <= inflight(s) || s.syn_at >= 0))
            return;
        s.syn_at = now + 1;
        Chain ch;
        chain_child(ch, 2, at);
        chain_store(B.schain + (size_t)f * CW, ch);
        due_insert(x, now + 1, f, 2);
    }
    // a frame at its destination host (src/step.cuh:2147-2236): the sending side's part - the
    // SYN-ACK establishes (RTT sample, the handshake's ACK, the first write), a FIN+ACK (the
    // sender's close) is acknowledged once, any other ACK goes to ack_in
    static __device__ void on_frame_snd(Host &x, int f, const Frame &p, int64_t now)
    {
        SndState &s = x.S;
        if (TW_RARE(p.flags & F_SYN))
        {
            if (U(s.st != S_SYN_SENT))
                return;
            s.st = S_EST;
            s.syn_at = -1;
            rtt_sample(s, now - s.timing_time);
            emit(x, f, F_ACK, 0, 0, CTRL_FRAME, false, now);
            Chain w; // (the write is an event scheduled now; it sends nothing itself)
            chain_child(w, 1, x.echain);
            app_write(x, f, now, w);
            return;
        }
        if (TW_RARE(s.fin & FIN_TW))
            return;
        snd_ecn_in(x, s, p);
        ack_in(x, f, p.sa, p.flags & F_ECE, now);
        if (TW_USUAL(!(p.flags & F_FIN)))
            return;
        s.fin |= FIN_TW;
        emit(x, f, F_ACK, 0, 1, CTRL_FRAME, false, now);
    }
    // ... and the receiving side's: the handshake's RTT for the receiver, a SYN (the connection
    // comes up; a SYN-ACK unless established), data, or an ACK (establishes; ends LAST_ACK)
    static __device__ void on_frame_rcv(Host &x, int f, const Frame &p, int64_t now)
    {
        RcvState &r = x.Q;
        const bool syn = p.flags & F_SYN;
        if (TW_RARE(!syn && r.r_up && r.r_srtt < 0 && r.r_synack_t >= 0))
        {
            const int64_t m = now - r.r_synack_t;
            r.r_srtt = m;
            r.r_rttvar = m / 2;
        }
        if (TW_RARE(syn))
        {
            if (U(!r.r_up))
            {
                r.r_up = 1;
                r.delack_count = DELACK_COUNT;
                add_active(x, false, f);
            }
            if (U(r.r_est))
                return;
            x.nic.woke = now;
            chain_child(x.echain, 1, x.echain);
            rcv_synack(x, f, now);
            return;
        }
        if (TW_USUAL(p.flags & (F_DATA | F_FIN)))
        {
            rcv_segment(x, f, p, now);
            return;
        }
        if (TW_RARE(!r.r_up || r.r_st == R_CLOSED))
            return;
        rcv_ecn_in(x, f, p, now);
        rcv_established(r);
        if (TW_RARE(r.r_st == R_LAST_ACK))
            rcv_closed(r);
    }
    // one event per frame, on the side's record
    static __device__ void on_frame(Host &x, const Frame &p, int64_t now)
    {
        const int f = (int)p.flow;
        if (U(p.to_sender))
        {
            snd_open(x, f);
            on_frame_snd(x, f, p, now);
        }
        else
        {
            rcv_open(x, f);
            on_frame_rcv(x, f, p, now);
        }
    }
    static __device__ __forceinline__ const uint32_t *due_chain(const Host &x, const Due &d)
    {
        Batch &B = *x.B;
        const uint32_t *base = d.kind == 1 || d.kind == 3 || d.kind == 4 ? B.dchain
                               : d.kind == 5                            ? B.fchain
                               : (d.kind == 2 && (x.sf == d.flow ? x.S.st : B.snd[d.flow].st) == S_EST) ? B.schain
                                                                                                           : B.rchain;
        return base + (size_t)d.flow * CW;
    }
    // a timer and an arrival at one instant: the one scheduled first runs first (undecided: the timer)
    static __device__ __forceinline__ bool timer_before_arrival(Host &x, const Due &d, const Frame *p)
    {
        Chain arr, pc;
        msg_chain(pc, p);
        chain_child(arr, 2048u + msg_head(p).len, pc);
        int r = chain_cmp(due_chain(x, d), arr.r);
        if (U(r == 0))
            count(x.R, EV_UNDECIDED);
        return r <= 0;
    }

    // the slot of time `at`, from slot t's end E0 on without a 64-bit division
    static __device__ __forceinline__ int64_t slot_of(int64_t at, int64_t E0, int64_t t)
    {
        const uint64_t d = (uint64_t)(at - E0); // (huge before E0)
        return d < 0x100000000ull ? t + 1 + (uint32_t)d / (uint32_t)SLOT_PS : at / SLOT_PS;
    }

    // -------------------------------------------------------------- one slot of a host
    // its arrivals: the later part of slot t-2's message of its in-link, the earlier of t-1's
    struct HostIn
    {
        int in, i2, n2, n1;
    };
    // has the host events in this slot? If not, *wake: its next slot
    static __device__ __forceinline__ bool host_open(Batch &B, World &W, int hl, int64_t t, HostIn &in, int64_t *wake)
    {
        const int h = W.host0 + hl, lid = W.link0 + hl;
        in.in = B.in_link[lid];
        in.i2 = in.n2 = in.n1 = 0;
        const int64_t w = B.wake[h];
        const int queued = B.q_size[lid];
        if (t >= 2)
        {
            const long long v = coh_load(msg_cnt_of(B, t - 2, in.in));
            if (msg_slot(v) == t - 2)
                in.i2 = msg_early(v), in.n2 = msg_sent(v);
        }
        if (t >= 1)
        {
            const long long v = coh_load(msg_cnt_of(B, t - 1, in.in));
            in.n1 = msg_slot(v) == t - 1 ? msg_early(v) : 0;
        }
        if (in.i2 < in.n2 || in.n1 > 0 || t >= w || queued != 0)
            return true;
        *wake = w;
        return false;
    }
    // the slot of a host that has events (src/step.cuh:2263-2528): returns 1 if it sent or holds frames;
    // *wake: its next slot; st: the lane's workspace for the first st_cap frames out, which the caller
    // moves to the link's message (*staged of them)
    static __device__ int host_run(Batch &B, World &W, WorldRun *R, int hl, int64_t t, int64_t *wake, const HostIn &hi, Frame *st, int st_cap,
                                   int *staged)
    {
        const int64_t S0 = t * SLOT_PS, E0 = S0 + SLOT_PS;
        const int h = W.host0 + hl, lid = W.link0 + hl;
#ifdef TW_PROF
        const unsigned long long pr0 = wall_clock64();
        unsigned long long pr_ev = 0, pr_n = 0;
#endif
        const Frame *m2 = msg_of(B, t + NRING - 2, hi.in);
        const Frame *m1 = msg_of(B, t + NRING - 1, hi.in);
        const int n2 = hi.n2, n1 = hi.n1;
        int i2 = hi.i2, i1 = 0;
        const int rt = (int)ring_of(t);
        Host x;
        x.nic.load(B, W, R, lid, t, rt, st, st_cap);
        x.B = &B;
        x.W = &W;
        x.R = R;
        x.h = h;
        x.hl = hl;
        x.dctcp = B.host_cc[h] == CC_DCTCP;
        x.cubic = B.host_cc[h] == CC_CUBIC;
        x.due = B.due + (size_t)h * MAX_DUE;
        x.slot_end = E0;
        x.sf = x.rf = -1;
        x.S = SndState{};
        x.Q = RcvState{};
        x.cs = ConnSnd{};
        x.cr = ConnRcv{};
        x.max_it = 0;
        Due *due = x.due;
        // timers due in this slot, by time. A list is scanned only when one of its timers falls in
        // the slot: tmin_s / tmin_r are its earliest, exact since the end of the host's last slot
        // (timers change only while the host runs)
        int nd = 0;
        const int64_t bound_s = B.tmin_s[h], bound_r = B.tmin_r[h];
        const bool scan_s = bound_s < E0, scan_r = bound_r < E0;
        const int ns = scan_s ? B.n_snd[h] : 0, nr = scan_r ? B.n_rcv[h] : 0;
        const int32_t *as = B.act_snd + (size_t)h * MAX_ACTIVE, *ar = B.act_rcv + (size_t)h * MAX_ACTIVE;
        for (int i = 0; U(i < ns); i++)
        {
            int f = as[i];
            int64_t a = B.snd[f].rto_at, b = B.snd[f].syn_at;
            if (U(a >= 0 && a < E0 && nd < MAX_DUE))
                due[nd++] = {a, f, 0};
            if (U(b >= 0 && b < E0 && nd < MAX_DUE))
                due[nd++] = {b, f, 2};
        }
        for (int i = 0; U(i < nr); i++)
        {
            int f = ar[i];
            const RcvState &r = B.rcv[f];
            int64_t a = r.delack_at, b = r.srv_syn_at, l = r.r_last_at, xx = r.r_frx_at;
            if (U(a >= 0 && a < E0 && nd < MAX_DUE))
                due[nd++] = {a, f, 1};
            if (U(b >= 0 && b < E0 && nd < MAX_DUE))
                due[nd++] = {b, f, 3};
            if (U(l >= 0 && l < E0 && nd < MAX_DUE))
                due[nd++] = {l, f, 4};
            if (U(xx >= 0 && xx < E0 && nd < MAX_DUE))
                due[nd++] = {xx, f, 5};
        }
        if (U(nd >= MAX_DUE))
            count(R, EV_DUE_OVF);
        for (int i = 1; U(i < nd); i++)
        {
            Due v = due[i];
            int j = i - 1;
            while (U(j >= 0 && due[j].at > v.at))
            {
                due[j + 1] = due[j];
                j--;
            }
            due[j + 1] = v;
        }
        x.nd = nd;
        x.id = 0;
        x.due_head = nd ? due[0].at : INT64_MAX;
        int pn = B.pend_next[h];
        const int pe = B.pend_end[h];
        // The three candidates' times are kept between events, each read again only when its
        // own event is taken (the next reads are then in flight while that event runs): the
        // next arrival, the next timer (due_head, which due_insert keeps), the next application
        // start of the host's order.
        // (the next arrival's whole frame is read with its time, so taking it waits for no load)
        Frame fa;
        auto next_arrival = [&]() -> int64_t {
            if (U(i2 >= n2 && i1 >= n1))
                return INT64_MAX;
            fa = coh_get(i2 < n2 ? m2 + i2 : m1 + i1);
            return fa.ts;
        };
        auto next_start = [&](int &m) -> int64_t {
            m = pn < pe ? B.pend_msg[pn] : -1;
            if (U(m >= 0))
            {
                const int64_t at = B.mg_start[m];
                if (U(at < E0))
                    return at;
            }
            return INT64_MAX;
        };
        int pm;
        int64_t tr = next_arrival(), tp = next_start(pm);
#ifdef TW_PROF
        const unsigned long long pr1 = wall_clock64();
#endif
        x.fill = x.has_post = false;
        for (;;)
        {
            const int64_t td = x.due_head;
            int64_t now = tr < td ? tr : td;
            now = now < tp ? now : tp;
            const bool last = now == INT64_MAX;
            now = now < S0 ? S0 : now;
            x.nic.advance(last ? E0 - 1 : now);
            if (U(last))
                break;
            x.n_ask = x.i_ask = 0;
#ifdef TW_PROF
            const unsigned long long pq = wall_clock64();
            pr_n++;
#endif
            if (TW_RARE(now == tp && B.cs[B.mg_conn[pm]].m_first != pm))
            {
                // a later message of a connection (FlowSender::SendMessage)
                const int m = pm;
                pn++;
                tp = next_start(pm);
                int f = B.mg_conn[m];
                chain_root_msg(x.echain, m - W.msg0);
                SndState &s = snd_open(x, f);
                s.m_due++;
                if (U(s.st == S_EST))
                    app_write(x, f, now, x.echain);
            }
            else if (TW_RARE(now == tp))
            {
                // a connection's application starts: SYN
                const int m = pm;
                pn++;
                tp = next_start(pm);
                int f = B.mg_conn[m];
                SndState &s = snd_open(x, f);
                chain_root(x.echain, hl, f - W.conn0);
                s.m_due = 1;
                add_active(x, true, f);
                s.st = S_SYN_SENT;
                if (U(x.cubic))
                    cubic_round_start(x, now);
                s.rto = CONN_TIMEOUT_PS;
                s.syn_at = now + CONN_TIMEOUT_PS;
                timer_chain(x, B.rchain, f, CONN_TIMEOUT_PS);
                s.timing_time = now;
                emit(x, f, F_SYN, 0, 0, SYN_FRAME, false, now);
            }
            else if (TW_RARE(now == td && (now != tr || timer_before_arrival(x, due[x.id], i2 < n2 ? m2 + i2 : m1 + i1))))
            {
                Due d = due[x.id++];
                x.due_head = x.id < x.nd ? due[x.id].at : INT64_MAX;
                chain_load(x.echain, due_chain(x, d));
                const int f = d.flow;
                if (U(d.kind == 0))
                {
                    if (U((x.sf == f ? x.S.rto_at : B.snd[f].rto_at) == d.at))
                    {
                        snd_open(x, f);
                        rto_fire(x, f, now);
                    }
                }
                else if (U(d.kind == 2))
                {
                    SndState &s = snd_open(x, f);
                    if (U(s.syn_at == d.at && s.st == S_EST))
                    {
                        s.syn_at = -1; // the deferred SendPendingData
                        tx_fill(x);
                    }
                    else if (U(s.syn_at == d.at && s.st == S_SYN_SENT))
                    {
                        int tries = ++s.syn_tries; // SYN retransmission, backed off
                        s.rto = CONN_TIMEOUT_PS << tries;
                        s.syn_at = now + s.rto;
                        timer_chain(x, B.rchain, f, s.rto);
                        emit(x, f, F_SYN, 0, 0, SYN_FRAME, false, now);
                    }
                }
                else
                {
                    RcvState &r = rcv_open(x, f);
                    if (U(d.kind == 1 && r.delack_at == d.at))
                    {
                        r.delack_at = -1;
                        r.delack_count = 0;
                        r.reserved = 1;
                        rcv_ack(x, f, r.rcv_nxt, false, false, now);
                    }
                    else if (TW_RARE(d.kind == 4 && r.r_last_at == d.at && r.r_st == R_LAST_ACK))
                    {
                        if (U(r.r_last_n == 0))
                            rcv_closed(r);
                        else
                        {
                            r.r_last_n--;
                            rcv_fin_ack(x, f, now);
                            int64_t lr = rcv_rto(r);
                            r.r_last_at = now + lr;
                            timer_chain(x, B.dchain, f, lr);
                        }
                    }
                    else if (TW_RARE(d.kind == 5 && r.r_frx_at == d.at && r.r_st == R_LAST_ACK))
                    {
                        r.r_frx_at = -1;
                        rcv_fin_ack(x, f, now);
                    }
                    else if (TW_RARE(d.kind == 3 && r.srv_syn_at == d.at && !r.r_est))
                    {
                        r.srv_syn_at = -1;
                        rcv_synack(x, f, now);
                    }
                }
            }
            else
            {
                const Frame p = fa;
                if (U(i2 < n2))
                    i2++;
                else
                    i1++;
                tr = next_arrival();
                Chain pc;
                chain_load(pc, p.chain);
                chain_child(x.echain, 2048u + p.len, pc);
                on_frame(x, p, now);
            }
            // what the event sends, into the queue in order (made here once for all events: inlined at
            // every sender, the frame's making and the queue's advance were most of the code)
            bool first = true;
            Out o;
            while (U(next_out(x, now, &o)))
            {
                if (U(!first))
                    x.nic.advance(now); // (the event began with the queue advanced)
                first = false;
                x.nic.enqueue(frame_of(x, o, now), now);
            }
#ifdef TW_PROF
            pr_ev += wall_clock64() - pq;
#endif
        }
#ifdef TW_PROF
        const unsigned long long pr2 = wall_clock64();
#endif
        x.nic.store(t, rt);
        snd_flush(x);
        rcv_flush(x);
        if (U(x.max_it))
            atomicMax(&R->ev[EV_MAX_INFLIGHT], (unsigned long long)x.max_it);
        *staged = x.nic.sent < st_cap ? x.nic.sent : st_cap;
        B.pend_next[h] = pn;
        // drop finished connections from the active lists; their earliest timers; the next wake-up
        const int64_t nb_s = compact_snd(B, h), nb_r = compact_rcv(B, h);
        B.tmin_s[h] = nb_s;
        B.tmin_r[h] = nb_r;
        int64_t next = nb_s < nb_r ? nb_s : nb_r;
        if (U(pn < pe && B.mg_start[B.pend_msg[pn]] < next))
            next = B.mg_start[B.pend_msg[pn]];
        int64_t wk = x.nic.size > 0 ? t + 1 : (next == INT64_MAX ? INT64_MAX : slot_of(next, E0, t));
        B.wake[h] = wk;
        *wake = wk;
#ifdef TW_PROF
        const unsigned long long pr3 = wall_clock64();
        atomicAdd(&R->ev[EV_PROF_H_SETUP], pr1 - pr0);
        atomicAdd(&R->ev[EV_PROF_H_LOOP], pr2 - pr1);
        atomicAdd(&R->ev[EV_PROF_H_EVENTS], pr_ev);
        atomicAdd(&R->ev[EV_PROF_H_END], pr3 - pr2);
        atomicAdd(&R->ev[EV_PROF_H_COUNT], pr_n);
#endif
        return (x.nic.sent > 0 || x.nic.size > 0) ? 1 : 0;
    }

    // -------------------------------------------------------------- routing (src/step.cuh:2541-2630)
    static __device__ int epoch_of(Batch &B, World &W, int64_t ts)
    {
        int e = 0;
        while (e < W.n_fail && ts >= B.g_fail_t[W.o_fail + e])
            e++;
        return e;
    }
    static __device__ __forceinline__ size_t rt_index(World &W, int ep, int x, int e)
    {
        return (size_t)W.o_rt + ((size_t)ep * W.S + x) * W.S + e;
    }
    // the output port at switch sw (world-local) towards host dst; up: the equal-cost index
    static __device__ int route_up(Batch &B, World &W, int sw, int dst, int up, int ep)
    {
        if (W.kind == TOPO_GRAPH)
        {
            int e = B.g_host_sw[W.o_host + dst];
            if (e == sw)
                return B.g_host_port[W.o_host + dst];
            return B.g_rt_ports[W.o_rtp + B.g_rt_off[rt_index(W, ep, sw, e)] + up];
        }
        if (W.kind == TOPO_LEAFSPINE)
        {
            const int leaf = (int)div_small(dst, W.hpl_m);
            if (sw < W.leaves)
                return leaf == sw ? dst - leaf * W.hpl : W.hpl + up;
            return leaf;
        }
        const int hk = W.hk, E = W.k * hk;
        const int rack = (int)div_small(dst, W.hk_m), dst_pod = (int)div_small(dst, W.hk2_m);
        if (sw < E)
            return rack == sw ? dst - rack * hk : hk + up; // (edge switches in the racks' order)
        if (sw < 2 * E)
            return dst_pod == (int)div_small(sw - E, W.hk_m) ? rack - dst_pod * hk : hk + up;
        return dst_pod;
    }
    static __device__ int route(Batch &B, World &W, int sw, const FrameHead &p, int ep)
    {
        if (W.kind == TOPO_GRAPH)
        {
            int e = B.g_host_sw[W.o_host + p.dst];
            if (e == sw)
                return B.g_host_port[W.o_host + p.dst];
            const ConnStatic &c = B.cs[p.flow];
            uint32_t hh = p.to_sender ? c.hash_ack : c.hash_data;
            return route_up(B, W, sw, p.dst, (int)(hh % B.g_rt_n[rt_index(W, ep, sw, e)]), ep);
        }
        return route_up(B, W, sw, p.dst, p.up, ep);
    }
    static __device__ __forceinline__ bool port_down(Batch &B, World &W, int sw, int q, int ep)
    {
        return W.n_fail && B.g_port_dn[W.o_pdn + ((size_t)ep * W.S + sw) * W.k + q];
    }
    static __device__ int routes_to(Batch &B, World &W, int sw, int dst, int ep)
    {
        if (W.kind == TOPO_GRAPH)
        {
            int e = B.g_host_sw[W.o_host + dst];
            return e == sw ? 0 : B.g_rt_n[rt_index(W, ep, sw, e)];
        }
        if (W.kind == TOPO_LEAFSPINE)
            return sw < W.leaves ? ((int)div_small(dst, W.hpl_m) == sw ? 0 : W.ecmp_n) : 1;
        const int E = W.k * W.hk;
        if (sw < E)
            return (int)div_small(dst, W.hk_m) == sw ? 0 : W.ecmp_n; // (edge switches in the racks' order)
        if (sw < 2 * E)
            return div_small(dst, W.hk2_m) == div_small(sw - E, W.hk_m) ? 1 : W.ecmp_n;
        return 1;
    }
    // simultaneous arrivals: the longer frame first, then the upstream starts' chains, then
    // (undecided) the flow id (src/step.cuh:2691-2704)
    static __device__ bool frame_before(WorldRun *R, const Frame *a, const Frame *b)
    {
        const FrameHead ha = msg_head(a), hb = msg_head(b);
        if (ha.len != hb.len)
            return ha.len > hb.len;
        int c = chain_cmp_by([&](int i) { return coh_load(&a->chain[i]); }, [&](int i) { return coh_load(&b->chain[i]); });
        if (c == 0)
            count(R, EV_UNDECIDED);
        return c != 0 ? c < 0 : ha.flow < hb.flow;
    }

    // -------------------------------------------------------------- one slot of a switch
    // (src/step.cuh:2706-2886). The k lanes of one switch within one wavefront, lane q = port q;
    // phases separated by wave_sync(). LDS per switch: rows[k][k+1] counts, in_win[k][3], base[k],
    // cnt[k]; per-wave global scratch holds the arrivals sorted per egress.
    // a switch item's LDS: per lane rows (33 ints), in_win (3), base, cnt, then (after the
    // spray merge's 64) per lane SORT_LDS arrival times and refs for the egress sort, then per
    // lane its first EGRESS_LDS arrivals' times in the slot (20 bits) and egress ports (above: the
    // count phase reads and routes them, the scatter phase reads no frame), then per lane its port's
    // in-link
    static constexpr int SW_LDS_INTS = 64 * 33 + 64 * 3 + 64 + 64, SORT_LDS = 24, EGRESS_LDS = 40;
    static constexpr int SW_LDS_EGRESS = SW_LDS_INTS + 64 * SORT_LDS * 3;
    static constexpr int SW_LDS_INLINK = SW_LDS_EGRESS + 64 * EGRESS_LDS;
    static constexpr int SW_LDS_TOTAL = SW_LDS_INLINK + 64;
    static constexpr uint32_t NO_EGRESS = 0xFF;
    // an arrival in the sort lists: its frame's place among the messages of the world's links (MAX_TX
    // each), in those of slot t - 2 or, with REF_EARLY, t - 1
    static constexpr uint32_t REF_EARLY = 0x80000000u;
    static_assert(SLOT_PS < 1 << 20, "an arrival's time in its slot: 20 bits");
    static constexpr int COUNT_RUN = 4; // arrivals' heads read together
    struct SwLds
    {
        int *rows, *in_win, *base, *cnt;
        int *wave; // the wavefront's whole LDS region (33 ints per lane at the start)
    };
    struct In
    {
        const Frame *m2, *m1;
        int i2, n2, n1;
        __device__ int count() const { return (n2 - i2) + n1; }
        // the j-th arrival (a frame another entity wrote in an earlier slot: read it device-coherently)
        __device__ const Frame *at(int j) const { return j < n2 - i2 ? m2 + i2 + j : m1 + (j - (n2 - i2)); }
        __device__ FrameHead head(int j) const { return msg_head(at(j)); }
    };
    static __device__ In input_of(Batch &B, int link, int64_t t, const int *win)
    {
        In in;
        in.i2 = win[0];
        in.n2 = win[1];
        in.n1 = win[2];
        if (link < 0)
            link = 0; // (an unused port has an empty window)
        in.m2 = msg_of(B, t + NRING - 2, link);
        in.m1 = msg_of(B, t + NRING - 1, link);
        return in;
    }
    // One lane of a switch's slot: port q of world-local switch swl (inactive lanes idle).
    // The phases run in order for all lanes of a switch, with wave_sync() between them (a CPU
    // check may run each phase over the lanes one after another). Scratch: this switch's region
    // (k * 2 * MAX_TX entries) of the wave's arrival scratch.
    struct SwLane
    {
        int swl, q, lid;
        bool active;
        int64_t *scr_ts;
        uint32_t *scr_ref;
        uint8_t *scr_up;
    };
    // port q's input of the slot (its in-link from LDS, where the window phase put it)
    static __device__ In lane_input(Batch &B, World &W, const SwLane &x, int64_t t, const SwLds &L, int q)
    {
        return input_of(B, L.wave[SW_LDS_INLINK + sw_lane_of(L, x) - x.q + q], t, L.in_win + 3 * q);
    }
    // the switch lane's place in its wave (its switch's first lane, where L.cnt points, plus its port)
    static __device__ __forceinline__ int sw_lane_of(const SwLds &L, const SwLane &x)
    {
        return (int)(L.cnt - L.wave - (64 * 33 + 64 * 3 + 64)) + x.q;
    }
    static __device__ __forceinline__ uint32_t *lane_egress_lds(const SwLds &L, const SwLane &x)
    {
        return reinterpret_cast<uint32_t *>(L.wave + SW_LDS_EGRESS) + sw_lane_of(L, x) * EGRESS_LDS;
    }
    // (its equal-cost index in a sprayed world: the draw of arrival j)
    static __device__ __forceinline__ int lane_draw(World &W, const SwLane &x, int j)
    {
        return W.rng0 >= 0 ? x.scr_up[x.q * 2 * MAX_TX + j] : 0;
    }
    static __device__ int lane_egress(Batch &B, World &W, const SwLane &x, int draw, const FrameHead &p)
    {
        int ep = W.n_fail ? epoch_of(B, W, p.ts) : 0;
        if (port_down(B, W, x.swl, x.q, ep))
            return -1; // dropped on arrival at a down interface
        return W.rng0 >= 0 ? route_up(B, W, x.swl, p.dst, draw, ep) : route(B, W, x.swl, p, ep);
    }
    // 1: the ingress window of port q (tail of slot t-2's message from S0 on, head of t-1's
    // before E0) into LDS; the port's row of egress counts cleared
    static __device__ void sw_window(Batch &B, World &W, const SwLane &x, int64_t t, const SwLds &L)
    {
        if (!x.active)
            return;
        const int in_link = B.in_link[x.lid];
        L.wave[SW_LDS_INLINK + sw_lane_of(L, x)] = in_link;
        int w0 = 0, w1 = 0, w2 = 0;
        if (in_link >= 0)
        {
            if (t >= 2)
            {
                const long long v = coh_load(msg_cnt_of(B, t - 2, in_link));
                if (msg_slot(v) == t - 2)
                    w0 = msg_early(v), w1 = msg_sent(v);
            }
            if (t >= 1)
            {
                const long long v = coh_load(msg_cnt_of(B, t - 1, in_link));
                w2 = msg_slot(v) == t - 1 ? msg_early(v) : 0;
            }
        }
        L.in_win[3 * x.q] = w0;
        L.in_win[3 * x.q + 1] = w1;
        L.in_win[3 * x.q + 2] = w2;
        int *row = L.rows + x.q * (W.k + 1);
        for (int i = 0; i <= W.k; i++)
            row[i] = 0;
    }
    // 2: arrivals counted by egress (after the spray draws, if any)
    static __device__ void sw_count(Batch &B, World &W, WorldRun *R, const SwLane &x, int64_t t, const SwLds &L)
    {
        if (!x.active)
            return;
        In in = lane_input(B, W, x, t, L, x.q);
        int *row = L.rows + x.q * (W.k + 1);
        uint32_t *eg = lane_egress_lds(L, x);
        const int n = in.count();
        // (COUNT_RUN heads at a time: one after another each was a wait of its own)
        for (int j0 = 0; j0 < n; j0 += COUNT_RUN)
        {
            FrameHead h[COUNT_RUN];
            int draw[COUNT_RUN];
#pragma unroll
            for (int u = 0; u < COUNT_RUN; u++)
            {
                h[u] = in.head(j0 + u < n ? j0 + u : n - 1);
                draw[u] = lane_draw(W, x, j0 + u < n ? j0 + u : n - 1);
            }
#pragma unroll
            for (int u = 0; u < COUNT_RUN; u++)
            {
                const int j = j0 + u;
                if (j >= n)
                    break;
                const int e = lane_egress(B, W, x, draw[u], h[u]);
                if (j < EGRESS_LDS)
                    eg[j] = (uint32_t)(h[u].ts - t * SLOT_PS) | (e >= 0 ? (uint32_t)e : NO_EGRESS) << 20;
                if (e >= 0)
                    row[e]++;
                else
                    count(R, EV_DROP);
            }
        }
    }
    // 3: for egress q, each ingress's offset in its region and the region's size
    static __device__ void sw_prefix(World &W, const SwLane &x, const SwLds &L)
    {
        if (!x.active)
            return;
        int off = 0;
        for (int j = 0; j < W.k; j++)
        {
            int c = L.rows[j * (W.k + 1) + x.q];
            L.rows[j * (W.k + 1) + x.q] = off;
            off += c;
        }
        L.cnt[x.q] = off;
    }
    // 4: the start of egress q's region: the exclusive prefix sum of the switch's region sizes over
    // its ports. On the GPU the switch's k lanes are consecutive in the wavefront (port q on its
    // first lane + q) and every lane of the wave runs this phase, so a wave64 scan does it in six
    // shuffle steps; a CPU check, which runs the lanes one after another, sums in a loop.
    static __device__ void sw_base(const SwLane &x, const SwLds &L)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        const int v = x.active ? L.cnt[x.q] : 0;
        int incl = v;
        for (int d = 1; d < 64; d <<= 1)
        {
            const int u = __shfl_up(incl, d);
            if (x.active && x.q >= d)
                incl += u;
        }
        if (x.active)
            L.base[x.q] = incl - v;
#else
        if (!x.active)
            return;
        int b = 0;
        for (int j = 0; j < x.q; j++)
            b += L.cnt[j];
        L.base[x.q] = b;
#endif
    }
    // 5: every arrival of ingress q into its egress's region, in arrival order
    static __device__ void sw_scatter(Batch &B, World &W, const SwLane &x, int64_t t, const SwLds &L)
    {
        if (!x.active)
            return;
        In in = lane_input(B, W, x, t, L, x.q);
        int *row = L.rows + x.q * (W.k + 1);
        const uint32_t *eg = lane_egress_lds(L, x);
        const int n = in.count();
        const uint32_t first = (uint32_t)(L.wave[SW_LDS_INLINK + sw_lane_of(L, x)] - W.link0) * MAX_TX; // (of the in-link's message)
        auto scatter = [&](auto *ts, auto *ref) {
            for (int j = 0; j < n; j++)
            {
                int64_t at_ts;
                int e;
                if (j < EGRESS_LDS)
                {
                    const uint32_t v = eg[j];
                    at_ts = t * SLOT_PS + (v & 0xFFFFF);
                    e = v >> 20 == NO_EGRESS ? -1 : (int)(v >> 20);
                }
                else
                {
                    const FrameHead p = in.head(j);
                    at_ts = p.ts;
                    e = lane_egress(B, W, x, lane_draw(W, x, j), p);
                }
                if (e < 0)
                    continue;
                int at = L.base[e] + row[e]++;
                ts[at] = at_ts;
                const int late = in.n2 - in.i2; // (the arrivals of slot t - 2's message come first)
                ref[at] = first + (j < late ? (uint32_t)(in.i2 + j) : REF_EARLY | (uint32_t)(j - late));
            }
        };
        if (sw_lists_in_lds(W, L))
            scatter(sort_ts_lds(L, x), sort_ref_lds(L, x));
        else
            scatter(x.scr_ts, x.scr_ref);
    }
    // the switch's egress lists go to LDS (its lanes' SORT_LDS slots each, laid out by L.base)
    // when all of them fit there, else to the wave's device scratch
    static __device__ __forceinline__ bool sw_lists_in_lds(World &W, const SwLds &L)
    {
        return L.base[W.k - 1] + L.cnt[W.k - 1] <= W.k * SORT_LDS;
    }
    // the switch's sort slots in LDS (from its first lane's)
    static __device__ __forceinline__ int64_t *sort_ts_lds(const SwLds &L, const SwLane &x)
    {
        return reinterpret_cast<int64_t *>(L.wave + SW_LDS_INTS) + (sw_lane_of(L, x) - x.q) * SORT_LDS;
    }
    static __device__ __forceinline__ uint32_t *sort_ref_lds(const SwLds &L, const SwLane &x)
    {
        return reinterpret_cast<uint32_t *>(L.wave + SW_LDS_INTS + 2 * 64 * SORT_LDS) + (sw_lane_of(L, x) - x.q) * SORT_LDS;
    }
    // 6: egress q's arrivals sorted by (time, frame_before), enqueued with the arrival event's
    // chain (RED), and the slot's transmissions; returns 1 if the port sent or holds frames
    static __device__ int sw_egress(Batch &B, World &W, WorldRun *R, const SwLane &x, int64_t t, const SwLds &L)
    {
        if (!x.active)
            return 0;
        const int n = L.cnt[x.q], b0 = L.base[x.q];
        if (n == 0 && B.q_size[x.lid] == 0)
            return 0; // (nothing to send: the port's message of an older slot stands for an empty one)
        const Frame *const m2 = msg_of(B, t + NRING - 2, W.link0), *const m1 = msg_of(B, t + NRING - 1, W.link0);
        auto frame_at = [&](uint32_t r) -> const Frame * { return (r & REF_EARLY ? m1 : m2) + (r & ~REF_EARLY); };
        Fifo eg;
        const int rt = (int)ring_of(t);
        eg.load(B, W, R, x.lid, t, rt);
        // an insertion sort by (time, frame_before): chain comparison is no strict weak order
        // when chains are truncated, and this gives the reference's order in every case. (Inlined at
        // two calls, for a list in LDS and for one in device scratch, so that each copy's accesses have
        // one address space: LDS or global instructions, not flat ones that wait on both.)
        auto sort = [&](auto *ts, auto *ref) {
            for (int i = 1; i < n; i++)
            {
                const int64_t xv = ts[i];
                const uint32_t r = ref[i];
                int j = i - 1;
                while (j >= 0 && (ts[j] > xv || (ts[j] == xv && frame_before(R, frame_at(r), frame_at(ref[j])))))
                {
                    ts[j + 1] = ts[j];
                    ref[j + 1] = ref[j];
                    j--;
                }
                ts[j + 1] = xv;
                ref[j + 1] = r;
            }
        };
        // where the sorted refs are: in LDS when all of the switch's lists were scattered there, or for a
        // short list of a switch whose lists overflow LDS (copied to the lane's own slots: one round of
        // loads instead of a device-memory round trip per comparison and move), else in device scratch
        const bool all_lds = sw_lists_in_lds(W, L), in_lds = all_lds || n <= SORT_LDS;
        const int lane = sw_lane_of(L, x);
        int64_t *lts = all_lds ? sort_ts_lds(L, x) + b0 : reinterpret_cast<int64_t *>(L.wave + SW_LDS_INTS) + lane * SORT_LDS;
        uint32_t *lref = all_lds ? sort_ref_lds(L, x) + b0 : reinterpret_cast<uint32_t *>(L.wave + SW_LDS_INTS + 2 * 64 * SORT_LDS) + lane * SORT_LDS;
        if (in_lds)
        {
            if (!all_lds)
                for (int i = 0; i < n; i++)
                {
                    lts[i] = x.scr_ts[b0 + i];
                    lref[i] = x.scr_ref[b0 + i];
                }
            sort(lts, lref);
        }
        else
            sort(x.scr_ts + b0, x.scr_ref + b0);
        // in that order into the queue, then the slot's transmissions; the next arrival is read while one
        // is queued (before its transmissions' stores, which a later load would wait for)
        auto ref_at = [&](int i) -> uint32_t { return in_lds ? lref[i] : x.scr_ref[b0 + i]; };
        Frame nx;
        if (n > 0)
            nx = coh_get(frame_at(ref_at(0)));
        for (int i = 0;; i++)
        {
            Frame p = nx;
            if (i + 1 < n)
                nx = coh_get(frame_at(ref_at(i + 1)));
            eg.advance(i < n ? p.ts : (t + 1) * SLOT_PS - 1);
            if (i >= n)
                break;
            Chain up, c;
            chain_load(up, p.chain);
            chain_child(c, 2048u + p.len, up);
            chain_store(p.chain, c);
            eg.enqueue(p, p.ts);
        }
        eg.store(t, rt);
        return (eg.sent > 0 || eg.size > 0) ? 1 : 0;
    }
    // one slot of a switch on the GPU: the lanes of one wavefront, phases separated by wave_sync()
    static __device__ int switch_step(Batch &B, World &W, WorldRun *R, const SwLane &x, int64_t t, const SwLds &L)
    {
#ifdef TW_PROF
        // profiler builds: the phases' wall-clock ticks, summed over switch items (counters 20-23)
        unsigned long long p0 = wall_clock64();
#define TW_PHASE(i)                                                                                                         \
    {                                                                                                                       \
        unsigned long long p1 = wall_clock64();                                                                             \
        if ((threadIdx.x & 63) == 0)                                                                                        \
            atomicAdd(&R->ev[20 + (i)], p1 - p0);                                                                           \
        p0 = p1;                                                                                                            \
    }
#else
#define TW_PHASE(i)
#endif
        // (a switch with no arrivals and nothing queued has no events)
        const int queued = x.active ? B.q_size[x.lid] : 0;
        sw_window(B, W, x, t, L);
        const int *win = L.in_win + 3 * x.q;
        if (!__any(x.active && (queued || win[1] > win[0] || win[2])))
            return 0;
        if (W.rng0 >= 0)
        {
            wave_sync();
            Spray sp;
            spray_init(B, W, x, t, L, sp);
            wave_sync();
            while (!spray_pick(B, W, R, x, t, L, sp))
                ;
            wave_sync();
            spray_end(B, W, x, L, sp);
        }
        wave_sync();
        TW_PHASE(0);
        sw_count(B, W, R, x, t, L);
        wave_sync();
        sw_prefix(W, x, L);
        wave_sync();
        sw_base(x, L);
        wave_sync();
        TW_PHASE(1);
        sw_scatter(B, W, x, t, L);
        wave_sync();
        TW_PHASE(2);
        const int r = sw_egress(B, W, R, x, t, L);
        TW_PHASE(3);
#undef TW_PHASE
        return r;
    }
    // Per-packet ECMP (src/step.cuh:2706-2745): one GetInteger draw per forwarded packet from the
    // switch's stream, in the switch's arrival order over all ports: at each step the earliest head
    // of the ports' arrival lists, equal times decided in port order by frame_before. Packets
    // arriving at a down port draw nothing; a packet with no route draws nothing and gets 0.
    // The k lanes of the switch run the merge in lockstep, each holding its own port's list: a
    // step finds the earliest head over the lanes, every lane the same one, and every lane makes the
    // same draw (each carries the stream); the winner records it. Heads and route counts of the
    // first 32 arrivals of a port sit in LDS (computed by the port's lane beforehand); frames are
    // read only to break equal times. The phases (init, then pick until done, then end) run with
    // wave_sync() between them; a CPU check runs each phase over the lanes in turn, with a loop over them
    // for spray_pick's minimum, ballot and shuffles.
    static constexpr int SPRAY_CACHE = 32;
    static constexpr uint32_t SPRAY_NONE = 0xFFFFFFFFu;
    struct Spray
    {
        In in;
        int c, p;      // this port's arrivals, the next one's place
        uint32_t head; // its arrival time - slot start (SPRAY_NONE: none left)
        TwMrg g;       // the switch's stream (every lane the same)
        bool done;
    };
    // the packed entry of arrival j: time offset (20 bits), route count or 255 (a down port)
    static __device__ uint32_t spray_code(Batch &B, World &W, const SwLane &x, int64_t S0, const FrameHead &f)
    {
        const int ep = W.n_fail ? epoch_of(B, W, f.ts) : 0;
        const uint32_t nr = port_down(B, W, x.swl, x.q, ep) ? 255u : (uint32_t)routes_to(B, W, x.swl, f.dst, ep);
        return (uint32_t)(f.ts - S0) | nr << 20;
    }
    // this port's lane in the wavefront (its switch's first lane, base, plus the port)
    static __device__ int spray_lane(const SwLane &x, const SwLds &L) { return sw_lane_of(L, x); }
    static __device__ uint32_t spray_entry(Batch &B, World &W, const SwLane &x, const SwLds &L, const Spray &sp, int64_t S0, int j)
    {
        if (j < SPRAY_CACHE)
            return (uint32_t)L.wave[spray_lane(x, L) * 33 + j];
        return spray_code(B, W, x, S0, sp.in.head(j));
    }
    static __device__ void spray_init(Batch &B, World &W, const SwLane &x, int64_t t, const SwLds &L, Spray &sp)
    {
        sp.c = 0;
        sp.p = 0;
        sp.head = SPRAY_NONE;
        sp.done = !x.active;
        if (!x.active)
            return;
        const int64_t S0 = t * SLOT_PS;
        sp.in = lane_input(B, W, x, t, L, x.q);
        sp.c = sp.in.count();
        const int lane = spray_lane(x, L);
        const int n = sp.c < SPRAY_CACHE ? sp.c : SPRAY_CACHE;
        for (int j = 0; j < n; j++)
            L.wave[lane * 33 + j] = (int)spray_code(B, W, x, S0, sp.in.head(j));
        if (sp.c > 0)
            sp.head = (uint32_t)L.wave[lane * 33]; // (the lane's own write)
        const TwMrgState &gs = B.sw_rng[W.rng0 + x.swl];
#pragma unroll
        for (int i = 0; i < 6; i++)
            sp.g.s[i] = gs.s[i];
    }
    // a lane's head as the lanes' minimum takes it: its time, then its port
    static __device__ uint32_t spray_key(const SwLane &x, const Spray &sp)
    {
        return sp.head == SPRAY_NONE ? SPRAY_NONE : (sp.head & 0xFFFFFu) << 6 | (uint32_t)x.q;
    }
    // Equal times, of port `best` (the first) and the ports `same` after it: in port order, frame_before
    // decides (the reference's scan over the ports). L.base: each port's place in its list.
    static __device__ int spray_tie(Batch &B, World &W, WorldRun *R, const SwLane &x, int64_t t, const SwLds &L, int best, uint64_t same)
    {
        for (; same; same &= same - 1)
        {
            const int q = __builtin_ctzll(same);
            if (frame_before(R, lane_input(B, W, x, t, L, q).at(L.base[q]), lane_input(B, W, x, t, L, best).at(L.base[best])))
                best = q;
        }
        return best;
    }
    // port `best`'s head, with nr routes (255: a down port), has its draw; its lane goes on to the next
    static __device__ void spray_take(Batch &B, World &W, const SwLane &x, int64_t t, const SwLds &L, Spray &sp, int best, uint32_t nr)
    {
        uint8_t draw = 0;
        if (nr != 255u && nr)
            draw = (uint8_t)tw_mrg_integer(sp.g, nr);
        if (best == x.q)
        {
            if (nr != 255u)
                x.scr_up[x.q * 2 * MAX_TX + sp.p] = draw;
            sp.p++;
            sp.head = sp.p < sp.c ? spray_entry(B, W, x, L, sp, t * SLOT_PS, sp.p) : SPRAY_NONE;
        }
    }
#if defined(__HIPCC__)
    // one step of the merge; true when the switch has no arrivals left
    static __device__ bool spray_pick(Batch &B, World &W, WorldRun *R, const SwLane &x, int64_t t, const SwLds &L, Spray &sp)
    {
        if (!x.active || sp.done)
            return true;
        const int k = W.k;
        // the earliest head (the first port holding it): a minimum over the switch's lanes by shuffles
        // (a step reading every port's head from LDS in a loop, twice, was most of a sprayed slot)
        const int lane0 = sw_lane_of(L, x) - x.q;
        uint32_t m = spray_key(x, sp);
        for (int d = 1; d < k; d <<= 1)
        {
            const uint32_t u = __shfl_down(m, d);
            m = x.q + d < k && u < m ? u : m;
        }
        m = __shfl(m, lane0);
        if (m == SPRAY_NONE)
        {
            sp.done = true;
            return true;
        }
        int best = (int)(m & 63);
        uint64_t same = __ballot(sp.head != SPRAY_NONE && (sp.head & 0xFFFFFu) == m >> 6) >> lane0;
        same &= (k < 64 ? 1ull << k : 0ull) - 1;
        same &= same - 1; // (but the first)
        if (same)
        {
            L.base[x.q] = sp.p;
            wave_sync();
            best = spray_tie(B, W, R, x, t, L, best, same);
            wave_sync();
        }
        spray_take(B, W, x, t, L, sp, best, __shfl(sp.head, lane0 + best) >> 20);
        return false;
    }
#endif
    static __device__ void spray_end(Batch &B, World &W, const SwLane &x, const SwLds &L, Spray &sp)
    {
        if (!x.active)
            return;
        if (x.q == 0)
        {
            TwMrgState &gs = B.sw_rng[W.rng0 + x.swl];
#pragma unroll
            for (int i = 0; i < 6; i++)
                gs.s[i] = sp.g.s[i];
        }
        // the count matrix row this lane's cache overlapped starts from zero again
        int *row = L.rows + x.q * (W.k + 1);
        for (int i = 0; i <= W.k; i++)
            row[i] = 0;
    }
};

} // namespace tw
