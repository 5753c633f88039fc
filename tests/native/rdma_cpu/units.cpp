// TEST INFRASTRUCTURE: checks of single functions of the RDMA model and its launch rules on the CPU
// (twins_amd/csrc/rdma_model.h, rdma_kernel.h); "units CHECK" exits non-zero and says what differs.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>
#include "../../../twins_amd/csrc/rdma_model.h"
#include "../../../twins_amd/csrc/rdma_kernel.h"
#include "../../../include/twins.h"
#include "../../../include/twins_rdma.h"

static int bad = 0;
#define CHECK(c, ...)                                                                                                                     \
    do                                                                                                                                    \
    {                                                                                                                                     \
        if (!(c))                                                                                                                         \
        {                                                                                                                                 \
            bad++;                                                                                                                        \
            printf(__VA_ARGS__);                                                                                                          \
            printf(" (%s)\n", #c);                                                                                                        \
        }                                                                                                                                 \
    } while (0)

// A sender's frames over links whose delay is one slot to thousands: each is filed in the bucket of
// ts / D, and finding the slot's first one takes a step or two whatever the delay (the frame's own tx
// time is below a slot here).
static void out_buckets()
{
    const int64_t D = 1000;
    for (int64_t delay : {1000ll, 1001ll, 1999ll, 2000ll, 10000ll, 250500ll, 4000000ll})
    {
        rd::Sim s = {};
        rd::Link l = {};
        l.delay = delay;
        l.bps = 100000000000ull;
        l.nb = (uint32_t)(2 + (90 + delay - 1) / D);
        l.cap = 202;
        l.skip = (uint32_t)(delay / D);
        const int pend_n = (int)l.nb + 3;
        std::vector<rd::LFrame> msg((size_t)l.nb * l.cap);
        std::vector<int64_t> cnt(l.nb, 0);
        std::vector<uint32_t> pend(pend_n, 0);
        uint64_t ev[rd::NEV] = {};
        s.D = D;
        s.li = &l;
        s.msg = msg.data();
        s.msg_cnt = cnt.data();
        s.ev = (decltype(s.ev))ev;
        int64_t last = 0;
        for (int64_t slot : {(int64_t)1, (int64_t)2, (int64_t)3, (int64_t)l.nb * 5 - 1, (int64_t)1 << 33})
        {
            rd::OutBucket o;
            rd::ob_open(s, o, 0, last, slot, pend_n);
            const int64_t t0 = slot * D;
            for (int64_t at : {t0 + 1, t0 + 85, t0 + 400, t0 + 910})
            {
                const int64_t ts = at + 84 + delay, a = ts / D;
                CHECK(ts < o.end || (ts - o.end) / D < 2, "delay %lld slot %lld: %lld slots to step", (long long)delay, (long long)slot,
                      (long long)((ts - o.end) / D + 1));
                std::fill(pend.begin(), pend.end(), 0u);
                const bool opens = ts >= o.hi;
                rd::LFrame *f = rd::ob_push(s, pend.data(), pend_n, ts, o);
                CHECK(f && (f - msg.data()) / (long)l.cap == (long)(a % l.nb), "delay %lld slot %lld: bucket %ld, not %lld", (long long)delay,
                      (long long)slot, f ? (long)(f - msg.data()) / (long)l.cap : -1, (long long)(a % l.nb));
                CHECK(!opens || pend[a % pend_n] == 1, "delay %lld slot %lld: pending flag", (long long)delay, (long long)slot);
            }
            rd::ob_flush(s, o);
            last = o.last;
            const int64_t end = t0 + 910 + 84 + delay;
            CHECK(cnt[end / D % l.nb] >> 16 == end / D, "delay %lld slot %lld: count word", (long long)delay, (long long)slot);
        }
        CHECK(ev[rd::EV_TX_OVF] == 0, "overflow");
    }
}

// A world whose links all take 20 us beside one of 1 us links (the batch's slot is then 1 us, and the
// first world's delays are twenty slots): every flow as in the world alone, in slots of 20 us.
static void unlike_delays(const char *config, const char *topo, const char *flows)
{
    const char *ov[] = {"CC_MODE=3", "BUFFER_SIZE=1"};
    trd_world *w[2] = {};
    for (int i = 0; i < 2; i++)
        if (trd_world_create(config, ov, 2, topo, flows, 0, i ? 1000 : 20000, &w[i]))
        {
            CHECK(false, "%s", trd_last_error());
            return;
        }
    int32_t n = 0;
    trd_world_info(w[0], nullptr, nullptr, &n, nullptr, nullptr);
    std::vector<int64_t> fct[3];
    for (int run = 0; run < 2; run++) // both together, then the first alone
    {
        trd_batch *b = nullptr;
        trd_run_stats st;
        CHECK(trd_batch_create(w, run ? 1 : 2, nullptr, &b) == 0 && trd_batch_run(b, &st) == 0, "%s", trd_last_error());
        for (int i = 0; i < (run ? 1 : 2); i++)
        {
            std::vector<int64_t> &f = fct[run ? 2 : i];
            f.assign(n, -2);
            CHECK(trd_fct_get(b, i, nullptr, f.data()) == 0, "%s", trd_last_error());
        }
        trd_batch_destroy(b);
    }
    int64_t least = INT64_MAX;
    for (int64_t f : fct[2])
        least = f < least ? f : least;
    CHECK(n > 0 && least > 0 && fct[0] == fct[2], "the far world beside the near one");
    CHECK(fct[0] != fct[1], "the near world has the far one's times");
    for (auto *x : w)
        trd_world_destroy(x);
}

// The launch shapes of FatTree worlds on a GPU of 256 workgroups: what is resident, and what runs by workgroup.
static void fattrees(int k, int W, std::vector<int> &hosts, std::vector<int> &switches)
{
    hosts.assign(W, k * k * k / 4);
    switches.assign(W, 5 * k * k / 4);
}
static void lone_world()
{
    // two callers' worlds, each alone in its batch, are resident together
    for (int k : {4, 8, 16, 32})
        for (int cap : {1, 64, 256})
        {
            std::vector<int> h, s;
            fattrees(k, 1, h, s);
            const rd::LaunchShape x = rd::launch_shape(h.data(), s.data(), 1, cap, true, 0, 0);
            CHECK(x.T >= 1 && x.T <= cap && x.T <= 128, "k=%d alone on %d: %d workgroups", k, cap, x.T);
            CHECK(x.hpw >= 1 && x.hpw <= 64, "k=%d alone on %d: %d hosts an item", k, cap, x.hpw);
        }
}
static void one_rule()
{
    // what runs by workgroup has a workgroup for each of its items, and what does not was given hosts per
    // item for a wave each (where any number of them fits)
    for (int k : {4, 8, 16})
        for (int W : {1, 2, 3, 4, 12, 24, 40, 130, 256})
        {
            std::vector<int> h, s;
            fattrees(k, W, h, s);
            const rd::LaunchShape x = rd::launch_shape(h.data(), s.data(), W, 256, true, 0, 0);
            const bool by_group = rd::runs_by_group(h[0], s[0], x.hpw, x.T);
            const int group = rd::group_items(h[0], s[0], x.hpw), wave = rd::wave_items(h[0], s[0], x.hpw);
            CHECK(!by_group || group <= x.T, "%d of k=%d: %d workgroup items on %d", W, k, group, x.T);
            CHECK(by_group || wave <= 4 * x.T || s[0] + 1 > 4 * x.T, "%d of k=%d: %d wave items on %d workgroups", W, k, wave, x.T);
            CHECK(x.T * W <= 256, "%d of k=%d: teams of %d", W, k, x.T);
        }
}
// What a team's workgroups are told at a world's start takes no plain store (see the TCP check of it)
static void team_words()
{
    CHECK((!std::is_assignable<decltype(rd::TeamState::world) &, int>::value), "world");
    CHECK((!std::is_assignable<decltype(rd::TeamState::act) &, unsigned>::value), "act");
    CHECK((!std::is_assignable<decltype(rd::TeamState::stop) &, int>::value), "stop");
    CHECK((!std::is_assignable<decltype(rd::TeamState::wake) &, unsigned long long>::value), "wake");
}

int main(int argc, char **argv)
{
    const char *what = argc > 1 ? argv[1] : "";
    if (!strcmp(what, "out_buckets"))
        out_buckets();
    else if (!strcmp(what, "lone_world"))
        lone_world();
    else if (!strcmp(what, "team_words"))
        team_words();
    else if (!strcmp(what, "one_rule"))
        one_rule();
    else if (!strcmp(what, "unlike_delays") && argc > 4)
        unlike_delays(argv[2], argv[3], argv[4]);
    else
        return 2;
    printf("%s: %d differences\n", what, bad);
    return bad != 0;
}
