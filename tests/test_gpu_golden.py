"""The GPU path against sequential ns-3's stored outputs, through the drop-in `twins` command line
(the C ABI underneath): every flow's establishment and completion time must be identical, as the
reference's validation/check_exact.sh demands. Undecided ties are rerun with 25-run chains."""
import os

import pytest

import util

CASES = util.cases()


def run_gpu(args, flows, out, runs=9):
    return util.run(util.TWINS, args + [f"--flows={flows}", f"--chain_runs={runs}"], out)


@pytest.mark.gpu
@pytest.mark.parametrize("name,flows,ref,args", CASES, ids=[c[0] for c in CASES])
def test_gpu_matches_ns3(name, flows, ref, args, tmp_path):
    print(f"case {name}", flush=True)
    out = str(tmp_path / "g.csv")
    log = run_gpu(args, flows, out)
    same, n = util.same_times(os.path.join(util.GOLDEN, ref), out)
    if same != n and util.undecided(log):
        log = run_gpu(args, flows, out, runs=25)
        same, n = util.same_times(os.path.join(util.GOLDEN, ref), out)
    assert same == n, f"{name}: {same}/{n} flows identical to ns-3\n{log[-1500:]}"


@pytest.mark.gpu
def test_gpu_batch_equals_standalone(tmp_path):
    """Heterogeneous worlds in one batch (one persistent launch) give each world's own ns-3
    output: batching changes nothing (the reference's check_sweeps.sh property)."""
    import twins_amd
    pick = [c for c in CASES if c[0].split("-")[2] in ("base", "spray", "fin") and not c[0].startswith("k16")][:24]
    worlds = [twins_amd.World([a.replace("topo/", util.GOLDEN + "/topo/") for a in args] + [f"--flows={util.GOLDEN}/{fl}"])
              for _, fl, _, args in pick]
    print(f"batch of {len(worlds)} worlds", flush=True)
    b = twins_amd.Batch(worlds)
    st = b.run()
    assert st.worlds_done == len(worlds)
    tied = []
    for i, (name, fl, ref, args) in enumerate(pick):
        est, done = b.fct(i)
        exp = util.read_cols(os.path.join(util.GOLDEN, ref), (4, 5))
        got = [(str(e), str(d)) for e, d in zip(est, done)]
        if b.counters(i)[25]:
            tied.append(i)  # undecided ties with 9-run chains: run again below with 25
            continue
        assert got == exp, name
    b.close()
    if not tied:
        return
    # the worlds whose chains left ties undecided, again in one batch of 25-run chains (the
    # reference's twins128 rerun): each must now equal its ns-3 output
    print(f"rerun of {len(tied)} worlds with 25-run chains: {[pick[i][0] for i in tied]}", flush=True)
    b = twins_amd.Batch([worlds[i] for i in tied], chain_runs=25)
    assert b.run().worlds_done == len(tied)
    for j, i in enumerate(tied):
        name, fl, ref, args = pick[i]
        est, done = b.fct(j)
        exp = util.read_cols(os.path.join(util.GOLDEN, ref), (4, 5))
        assert b.counters(j)[25] == 0, name
        assert [(str(e), str(d)) for e, d in zip(est, done)] == exp, name
    b.close()


@pytest.mark.gpu
@pytest.mark.parametrize("runs", [9, 25])
@pytest.mark.parametrize("team,hosts", [(0, 0), (52, 1), (1, 1), (3, 5), (1, 64), (16, 33)])
def test_gpu_launch_shapes(team, hosts, runs):
    """One host to a wave (the kernel whose hosts' branches are wave-uniform, every frame of a slot
    staged) and 5 to 64 (a lane each, down to 9 staged frames a host, 4 with chains of 25, the others
    stored as they are sent), on teams of few and many waves: loss and its repair, sprayed reordering
    (the draws' merge by shuffles), FIN and a torus give ns-3's stored times. None of these runs leaves
    a tie undecided, with chains of 9 or 25."""
    import twins_amd
    pick = [c for c in CASES if c[0] in ("k8_incast16-cubic-fin", "k8_a2a30-newreno-spray", "torus6_a2a30-dctcp-base")]
    assert len(pick) == 3
    for name, fl, ref, args in pick:
        print(f"case {name}", flush=True)
        w = twins_amd.World([a.replace("topo/", util.GOLDEN + "/topo/") for a in args] + [f"--flows={util.GOLDEN}/{fl}"])
        b = twins_amd.Batch([w], chain_runs=runs, team_blocks=team, hosts_per_wave=hosts)
        assert b.run().worlds_done == 1
        est, done = b.fct(0)
        exp = util.read_cols(os.path.join(util.GOLDEN, ref), (4, 5))
        assert b.counters(0)[25] == 0, name
        assert [(str(e), str(d)) for e, d in zip(est, done)] == exp, name
        b.close()


@pytest.mark.gpu
@pytest.mark.parametrize("team,budget", [(1, 997), (16, 61), (52, 61), (0, 997)])
def test_gpu_resumed_launches(team, budget):
    """A run cut into launches of `budget` slots (idle skips, a world's end inside a launch) goes on
    where it stood: ns-3's times, and the slots and packet-events of one launch."""
    import twins_amd
    name, fl, ref, args = [c for c in CASES if c[0] == "k8_incast16-cubic-fin"][0]
    print(f"case {name}", flush=True)
    w = twins_amd.World(args + [f"--flows={util.GOLDEN}/{fl}"])
    whole = twins_amd.Batch([w])
    one = whole.run()
    whole.close()
    b = twins_amd.Batch([w], team_blocks=team, slot_budget=budget)
    st = b.run()
    assert (st.worlds_done, st.slots_max, st.packet_events) == (1, one.slots_max, one.packet_events)
    assert st.launches == -(-st.slots_max // budget)
    est, done = b.fct(0)
    assert [(str(e), str(d)) for e, d in zip(est, done)] == util.read_cols(os.path.join(util.GOLDEN, ref), (4, 5))
    b.close()


@pytest.mark.gpu
@pytest.mark.parametrize("team", [1, 3, 0])
def test_gpu_skip_past_32_bit_slots(team, tmp_path):
    """An idle world skips to a flow that starts after slot 2^32 and ends at its last slot (a link's
    messages are of slots below 2^31, so that flow's SYNs are lost there, on the CPU alike)."""
    import twins_amd
    flows = tmp_path / "late.csv"
    flows.write_text("src,dst,flow_size,start_ns\n0,5,100000,0\n1,9,100000,4300000000000\n")
    w = twins_amd.World(["--k=4", f"--flows={flows}", "--max_slots=4300100000"])
    b = twins_amd.Batch([w], team_blocks=team)
    print(f"team {team}", flush=True)
    st = b.run()
    est, done = b.fct(0)
    assert (st.worlds_done, st.launches, b.counters(0)[26]) == (1, 1, 652)
    assert (list(est), list(done)) == ([12044, -1], [71653, -1])
    b.close()
