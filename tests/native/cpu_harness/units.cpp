// TEST INFRASTRUCTURE: checks of single functions of libtwins_core's TCP side on the CPU (the kernel's
// launch replaced by the harness, kernel_cpu.cpp); "units CHECK" exits non-zero and says what differs.
#include <cstdio>
#include <cstring>
#include <fstream>
#include <string>
#include <type_traits>
#include <vector>
#include "../../../include/twins.h"
#include "../../../twins_amd/csrc/tcp_state.h"

extern size_t shim_bytes;
namespace tw
{
extern bool cpu_time_out;
}
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

static tw_world *world(const char *dir, const char *flows, std::vector<std::string> more = {})
{
    const std::string path = std::string(dir) + "/units.csv";
    std::ofstream(path) << flows;
    more.insert(more.begin(), {"--k=4", "--flows=" + path});
    std::vector<const char *> a;
    for (auto &x : more)
        a.push_back(x.c_str());
    tw_world *w = nullptr;
    CHECK(tw_world_create_args((int)a.size(), a.data(), &w) == 0, "%s", tw_last_error());
    return w;
}
// the device memory of a batch of this world
static size_t packed(tw_world *w, int runs)
{
    tw_pack_cfg c = {};
    c.chain_runs = runs;
    c.blocks = c.team_blocks = 1; // (the same launch scratch for every world)
    tw_batch *b = nullptr;
    const size_t before = shim_bytes;
    CHECK(tw_batch_create(&w, 1, &c, &b) == 0, "%s", tw_last_error());
    tw_batch_destroy(b);
    return shim_bytes - before;
}

// The footprint that admission to the serving loop and tw_world_info give counts what a world's records
// take: between two worlds alike but for one quantity it grows by no less than the memory does (the
// rest of a batch, its launch's scratch, is the same for both).
static void footprint(const char *dir)
{
    const char *head = "src,dst,flow_size,start_ns\n";
    std::string many = head;
    for (int i = 0; i < 4000; i++)
        many += std::to_string(i % 16) + "," + std::to_string((i + 5) % 16) + ",1000," + std::to_string(i * 100) + "\n";
    struct
    {
        const char *what;
        std::string flows;
        std::vector<std::string> more;
    } const cases[] = {{"ledger places", std::string(head) + "0,5,900000000,0\n", {"--rtt_ring=600000"}},
                       {"flows", many, {}},
                       {"queue", std::string(head) + "0,5,1000,0\n", {"--queue=5000"}},
                       {"larger network", std::string(head) + "0,5,1000,0\n", {"--k=16"}},
                       {"spray streams", std::string(head) + "0,5,1000,0\n", {"--spray=1"}}};
    for (auto &c : cases)
    {
        tw_world *a = world(dir, (std::string(head) + "0,5,1000,0\n").c_str()), *b = world(dir, c.flows.c_str(), c.more);
        tw_world_info ia, ib;
        tw_world_info_get(a, &ia);
        tw_world_info_get(b, &ib);
        const long long info = (long long)(ib.device_bytes - ia.device_bytes), mem = (long long)(packed(b, 9) - packed(a, 9));
        printf("%s: footprint +%lld, memory +%lld\n", c.what, info, mem);
        CHECK(info >= mem && info <= mem + mem / 100 + 4096, "%s", c.what);
        tw_world_destroy(a);
        tw_world_destroy(b);
    }
}

// A barrier that times out in a world's first slot is reported as such, by both ways to run a batch.
static void timeout_error(const char *dir)
{
    tw_world *w[2] = {world(dir, "src,dst,flow_size,start_ns\n0,5,1000,0\n"), nullptr};
    w[1] = w[0];
    for (int n = 1; n <= 2; n++)
        for (int noalloc = 0; noalloc < 2; noalloc++)
        {
            tw_pack_cfg c = {};
            c.blocks = c.team_blocks = 1;
            tw_batch *b = nullptr;
            CHECK(tw_batch_create(w, n, &c, &b) == 0, "%s", tw_last_error());
            tw::cpu_time_out = true;
            tw_run_stats st;
            const int rc = noalloc ? tw_batch_run_noalloc(b, &st) : tw_batch_run(b, &st);
            tw::cpu_time_out = false;
            CHECK(rc == TW_EDEVICE && strstr(tw_last_error(), "a team barrier timed out"), "%d worlds, noalloc %d: error %d, %s", n, noalloc, rc,
                  tw_last_error());
            tw_batch_destroy(b);
        }
    tw_world_destroy(w[0]);
}

// The word that hands a team its next slot holds every slot whose time a 64-bit picosecond count can
// state, beside the flags and the count.
static void slot_word()
{
    using tw::SlotGo;
    const int64_t last = INT64_MAX / tw::SLOT_PS;
    for (int64_t t : {(int64_t)0, (int64_t)1, (int64_t)0x7FFFFFFF, (int64_t)0xFFFFFFFF, (int64_t)0x100000000, (int64_t)0x100000007, last})
        for (unsigned flags = 0; flags < 8; flags++)
            for (unsigned count : {0u, 1u, 0xFFFFu, 0x12345u})
            {
                const unsigned long long g = SlotGo::pack(t, flags, count);
                CHECK(SlotGo::next(g) == t && SlotGo::flags(g) == flags && SlotGo::count(g) == (count & 0xFFFFu), "slot %lld flags %u count %u: %lld %u %u",
                      (long long)t, flags, count, (long long)SlotGo::next(g), SlotGo::flags(g), SlotGo::count(g));
            }
}

// What a team's workgroups are told at a world's start takes no plain store: that would stay in the L2
// of the writer's XCD until a fence writes it back, and the others read it as soon as they are released.
static void team_words()
{
    CHECK((!std::is_assignable<decltype(tw::TeamState::world) &, int>::value), "TCP: world");
}

int main(int argc, char **argv)
{
    const char *what = argc > 1 ? argv[1] : "";
    if (!strcmp(what, "footprint") && argc > 2)
        footprint(argv[2]);
    else if (!strcmp(what, "team_words"))
        team_words();
    else if (!strcmp(what, "slot_word"))
        slot_word();
    else if (!strcmp(what, "timeout_error") && argc > 2)
        timeout_error(argv[2]);
    else
        return 2;
    printf("%s: %d differences\n", what, bad);
    return bad != 0;
}
