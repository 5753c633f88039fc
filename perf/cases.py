"""The simulations this framework is used for, as timed cases: whole calls through its Python entry
points on inputs drawn from a seed.

A case is one job of a user's program. The program has its worlds in hand (topology and flow files
read, routes built: `twins_amd.World`, `twins_amd.rdma.World`); a pass packs them into a batch on the
GPU, runs it to the end and takes every flow's times and every counter, as the `twins` and
`twins-rdma` commands do for each run. A batch runs once, so packing belongs to the pass; the serving
case starts a server, submits its requests, polls until all are done and takes the results.

The results are whole numbers (picosecond-exact event times in ns, counters) and a simulation has one
right answer, so every output is compared exactly.
"""
import math
import os
import tempfile

import numpy as np

import twins_amd
from twins_amd import rdma, workloads

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HPCC_CFG = os.path.join(ROOT, "tests", "golden", "rdma", "inputs", "hpcc.cfg")
LINE_BYTES_PER_NS = 12.5  # 100 Gb/s


# ------------------------------------------------------------------ the cases
def _tcp(name, topo, flows, sizes, median, top, load, tcp, **more):
    case = dict(name=name, kind="tcp", topo=topo, flows=flows, sizes=sizes, median=median, top=top, load=load, tcp=tcp,
                ecn=30, queue=200, incast=0, conns=False, spray=False, fin=False, fail=False, runs=9, worlds=1)
    case.update(more)
    return case


def _rdma(name, topo, flows, sizes, median, top, load, cc, **more):
    case = dict(name=name, kind="rdma", topo=topo, flows=flows, sizes=sizes, median=median, top=top, load=load, cc=cc,
                buffer=32, kmin=400, payload=1000, incast=0, q3cap=0, worlds=1)
    case.update(more)
    return case


def listed():
    return [
        # the smallest job: a FatTree of 16 hosts and 64 short flows, where the slot barrier and the
        # launch are most of the time
        _tcp("tcp_k4", "fattree:4", 64, "lognormal", 20000, 10_000_000, 0.3, "dctcp"),
        # a FatTree of 128 hosts alone, one long flow per host (the permutation-like runs of a paper)
        _tcp("tcp_k8_long", "fattree:8", 128, "exponential", 800_000, 4_000_000, 0.5, "dctcp"),
        # the same network under loss: a 60-to-1 incast among short NewReno flows, no ECN to hold it
        _tcp("tcp_k8_incast", "fattree:8", 1500, "lognormal", 20000, 1_000_000, 0.3, "newreno", incast=60, queue=100),
        # all-to-all short flows on 1,024 hosts, one world over the whole GPU
        _tcp("tcp_k16_a2a", "fattree:16", 12000, "lognormal", 20000, 1_000_000, 0.5, "cubic"),
        # per-packet ECMP, FIN, persistent connections, a link failing and coming back: three TCPs side
        # by side
        _tcp("tcp_k16_spray", "fattree-file:16", 8000, "pareto", 1000, 3_000_000, 0.5, "all", conns=True, spray=True, fin=True,
             fail=True, worlds=3),
        # a torus of odd sizes with the long event chains a user asks for after an undecided tie
        _tcp("tcp_torus_runs25", "torus:7:9:3", 3000, "lognormal", 20000, 1_000_000, 0.4, "newreno", runs=25),
        # a sweep: worlds of every topology kind, ECN threshold, queue and TCP in one launch
        _tcp("tcp_sweep", "mixed", 1500, "pareto", 1000, 3_000_000, 0.4, "mixed", worlds=64),
        # the serving loop: a burst of requests of several sizes through one server
        _tcp("tcp_serve", "fattree-mixed", 1500, "pareto", 1000, 1_000_000, 0.4, "mixed", worlds=24, serve=True),
        # the smallest RDMA job: 15 senders to one receiver on 16 hosts, buffers small enough for PFC
        _rdma("rdma_k4_incast", "fattree:4", 16, "lognormal", 9000, 200_000, 0.3, "dcqcn", buffer=1, incast=15),
        # all-to-all on 128 hosts under HPCC (in-band telemetry in every frame)
        _rdma("rdma_k8_hpcc", "fattree:8", 3000, "lognormal", 20000, 1_000_000, 0.5, "hpcc"),
        # a 512-host leaf-spine with an incast in the middle, HPCC and DCQCN as two worlds of one batch
        _rdma("rdma_ls32_pair", "leafspine:32:16:16", 2400, "lognormal", 50000, 1_000_000, 0.4, "pair", incast=100, q3cap=16384,
              worlds=2),
        # a parameter sweep of 128-host worlds (congestion control x buffer x ECN threshold) as one batch
        _rdma("rdma_k8_sweep", "fattree:8", 600, "lognormal", 20000, 500_000, 0.4, "mixed", incast=20, buffer=2, worlds=24),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: network, flow count, sizes, load, protocol and options drawn."""
    kind = rng.choice(["tcp", "tcp", "tcp-batch", "rdma", "rdma", "rdma-batch"])
    if kind == "tcp":
        topo = rng.choice(["fattree", "leafspine", "torus", "jellyfish"])
        if topo == "fattree":
            k = rng.choice([4, 6, 8, 10, 12, 16])
            topo, hosts = "fattree:%d" % k, k ** 3 // 4
        elif topo == "leafspine":
            a, b, c = rng.randint(5, 32), rng.choice([3, 4, 7, 8]), rng.randint(3, 16)
            topo, hosts = "leafspine:%d:%d:%d" % (a, b, c), a * c
        elif topo == "torus":
            a, b, c = rng.randint(4, 13), rng.randint(4, 13), rng.randint(1, 6)
            topo, hosts = "torus:%d:%d:%d" % (a, b, c), a * b * c
        else:
            a, b, c = rng.randint(24, 120), rng.choice([4, 6, 7]), rng.randint(1, 6)
            a += a * b % 2
            topo, hosts = "jellyfish:%d:%d:%d" % (a, b, c), a * c
        queue = rng.choice([60, 100, 200, 400])
        return _tcp("", topo, _log(rng, 40, min(9000, 40 * hosts)), rng.choice(["lognormal", "pareto"]), rng.choice([1000, 9000, 20000]),
                    _log(rng, 200_000, 2_000_000), rng.choice([0.2, 0.3, 0.5]), rng.choice(["dctcp", "newreno", "cubic"]),
                    ecn=rng.choice([10, 30, 50]), queue=queue, incast=rng.choice([0, 0, min(hosts - 2, rng.randint(8, 50))]),
                    conns=rng.random() < 0.3, spray=rng.random() < 0.3, fin=rng.random() < 0.3, runs=rng.choice([9, 9, 9, 25])) | {"name": ""}
    if kind == "tcp-batch":
        return _tcp("", rng.choice(["mixed", "fattree-mixed"]), _log(rng, 150, 1500), rng.choice(["lognormal", "pareto"]), 1000,
                    _log(rng, 200_000, 2_000_000), rng.choice([0.2, 0.4]), "mixed", worlds=_log(rng, 2, 60), serve=rng.random() < 0.25)
    if kind == "rdma":
        if rng.random() < 0.5:
            k = rng.choice([4, 6, 8, 10])
            topo, hosts = "fattree:%d" % k, k ** 3 // 4
        else:
            a, b, c = rng.randint(4, 30), rng.choice([3, 4, 8, 16]), rng.randint(3, 17)
            topo, hosts = "leafspine:%d:%d:%d" % (a, b, c), a * c
        return _rdma("", topo, _log(rng, 30, min(2500, 20 * hosts)), rng.choice(["lognormal", "pareto"]), rng.choice([1000, 9000, 20000]),
                     _log(rng, 100_000, 1_000_000), rng.choice([0.2, 0.3, 0.5]), rng.choice(["dcqcn", "hpcc", "dctcp"]),
                     buffer=rng.choice([1, 2, 32]), kmin=rng.choice([20, 100, 400]), payload=rng.choice([1000, 1000, 1452]),
                     incast=rng.choice([0, min(hosts - 2, rng.randint(8, 60))]), q3cap=16384)
    return _rdma("", "fattree:%d" % rng.choice([4, 6, 8]), _log(rng, 60, 600), "lognormal", 20000, _log(rng, 100_000, 500_000), 0.4, "mixed",
                 buffer=2, incast=rng.randint(6, 12), worlds=_log(rng, 2, 24))


# ------------------------------------------------------------------ inputs
def _topology(spec, seed):
    """(arguments of a TCP world or None, topology file text or None, hosts) of a topology text."""
    name, *n = spec.split(":")
    n = [int(x) for x in n]
    if name == "fattree":
        return ["--k=%d" % n[0]], workloads.fattree_topology(n[0]), n[0] ** 3 // 4
    if name == "fattree-file":
        return None, workloads.fattree_topology(n[0]), n[0] ** 3 // 4
    if name == "leafspine":
        return (["--topo=leafspine", "--leaves=%d" % n[0], "--spines=%d" % n[1], "--hpl=%d" % n[2]],
                workloads.leafspine_topology(*n), n[0] * n[2])
    if name == "torus":
        return None, workloads.torus_topology(*n), n[0] * n[1] * n[2]
    return None, workloads.jellyfish_topology(n[0], n[1], n[2], seed), n[0] * n[2]


def _sizes(case, u):
    """Flow sizes of uniform draws u in (0, 1)."""
    m, top = case["median"], case["top"]
    if case["sizes"] == "pareto":
        s = m * (1 - u) ** (-1 / 1.2)
    elif case["sizes"] == "exponential":
        s = -m / math.log(2) * np.log(1 - u)
    else:  # lognormal with sigma 1.2, the normal quantile by its logistic neighbour
        s = m * np.exp(1.2 * np.log(u / (1 - u)) / 1.702)
    return np.clip(np.floor(s), 500, top).astype(np.int64)


def _flow_rows(case, hosts, seed, flows):
    """Flow rows (src, dst, bytes, start_ns[, conn]): Poisson starts at the case's load, then the incast."""
    rng = np.random.Generator(np.random.PCG64(seed))
    if case["sizes"] == "exponential":  # one long flow per host
        src = np.arange(flows) % hosts
    else:
        src = rng.integers(0, hosts, flows)
    dst = (src + rng.integers(1, hosts, flows)) % hosts
    size = _sizes(case, rng.uniform(1e-6, 1 - 1e-6, flows))
    mean = float(_sizes(case, (np.arange(4096) + 0.5) / 4096).mean())
    gap = mean / (case["load"] * hosts * LINE_BYTES_PER_NS)
    start = np.floor(np.cumsum(rng.exponential(gap, flows))).astype(np.int64)
    conn = np.full(flows, -1, dtype=np.int64)
    if case.get("conns"):  # a quarter of the flows are later messages of an earlier flow's connection
        last, cid = {}, 0
        for i in range(flows):
            s = int(src[i])
            if s in last and rng.random() < 0.5:
                j = last[s]
                if conn[j] < 0:
                    conn[j] = cid
                    cid += 1
                conn[i], dst[i] = conn[j], dst[j]
                start[i] = max(start[i], start[j] + 1)
            last[s] = i
    if case["incast"]:
        n = min(case["incast"], hosts - 1)
        to = int(rng.integers(0, hosts))
        who = (to + 1 + rng.permutation(hosts - 1)[:n]) % hosts
        at = int(start[flows // 2]) if flows else 1000
        src, dst = np.concatenate([src, who]), np.concatenate([dst, np.full(n, to)])
        size = np.concatenate([size, np.full(n, 64000 if case["kind"] == "rdma" else 50000)])
        start, conn = np.concatenate([start, np.full(n, at)]), np.concatenate([conn, np.full(n, -1)])
    order = np.lexsort((src, start))
    head = "src,dst,flow_size,start_ns,conn\n" if (conn >= 0).any() else "src,dst,flow_size,start_ns\n"
    cols = [src, dst, size, start] + ([conn] if (conn >= 0).any() else [])
    rows = np.stack(cols, 1)[order]
    return head + "".join(",".join(map(str, r)) + "\n" for r in rows.tolist())


def _write(folder, name, text):
    path = os.path.join(folder, name)
    with open(path, "w") as f:
        f.write(text)
    return path


MIX = ["fattree:4", "fattree:8", "leafspine:12:4:8", "torus:6:7:2", "jellyfish:32:6:4", "fattree:16", "leafspine:21:8:16", "torus:9:11:3"]
TCPS = ["newreno", "dctcp", "cubic"]


def _tcp_worlds(case, seed, folder):
    rng = np.random.Generator(np.random.PCG64(seed + 7))
    worlds = []
    for w in range(case["worlds"]):
        spec = case["topo"]
        flows = case["flows"]
        ecn, queue = case["ecn"], case["queue"]
        if spec in ("mixed", "fattree-mixed"):
            spec = MIX[w % len(MIX)] if spec == "mixed" else "fattree:%d" % (4, 8, 16, 8)[w % 4]
            flows = max(20, flows * (3 + w * 5 % 14) // 10)
            queue = (100, 200, 400)[w % 3]
            ecn = (10, 30, 65)[(w // 3) % 3]
        tcp = {"mixed": TCPS[int(rng.integers(3))], "all": TCPS[w % 3]}.get(case["tcp"], case["tcp"])
        args, text, hosts = _topology(spec, seed + w)
        if args is None or case["fail"]:
            args = ["--topo=graph", "--topofile=" + _write(folder, "t%d.txt" % w, text)]
        own = 0 if case["tcp"] == "all" else w  # the three TCPs run the same flows
        args = args + ["--flows=" + _write(folder, "f%d.csv" % w, _flow_rows(case, hosts, seed * 1000 + own, flows)), "--tcp=" + tcp,
                       "--ecnK=%d" % ecn, "--queue=%d" % queue]
        if case["spray"]:
            args += ["--spray=1", "--RngRun=%d" % (1 + seed % 5)]
        if case["fin"]:
            args += ["--fin=1"]
        if case["fail"]:  # a core - aggregation link of the k=16 FatTree, down and up again
            args += ["--fail=100000:s256:s128,300000:s256:s128:up"]
        worlds.append(twins_amd.World(args))
    return worlds


CC = {"dcqcn": 1, "hpcc": 3, "dctcp": 8}


def _rdma_worlds(case, seed, folder):
    _, text, hosts = _topology(case["topo"], seed)
    topo = _write(folder, "t.txt", text)
    worlds = []
    for w in range(case["worlds"]):
        cc, buf, kmin = case["cc"], case["buffer"], case["kmin"]
        if cc == "mixed":
            cc, buf, kmin = ("dcqcn", "hpcc", "dctcp")[w % 3], (2, 32)[w // 3 % 2], (20, 50, 100, 400)[w // 6 % 4]
        elif cc == "pair":
            cc = ("hpcc", "dcqcn")[w]
        own = 0 if case["cc"] == "pair" else w
        over = ["CC_MODE=%d" % CC[cc], "BUFFER_SIZE=%d" % buf, "PACKET_PAYLOAD_SIZE=%d" % case["payload"],
                "KMIN_MAP=1,100000000000,%d" % kmin, "KMAX_MAP=1,100000000000,%d" % (4 * kmin)]
        f = _write(folder, "f%d.csv" % own, _flow_rows(case, hosts, seed * 1000 + own, case["flows"]))
        worlds.append(rdma.World(HPCC_CFG, topo, f, over))
    return worlds


def prepare(case, seed):
    with tempfile.TemporaryDirectory() as folder:
        worlds = (_tcp_worlds if case["kind"] == "tcp" else _rdma_worlds)(case, seed, folder)
    return {"case": case, "worlds": worlds}


# ------------------------------------------------------------------ a pass
def run(state):
    case, worlds = state["case"], state["worlds"]
    times, counters = [], []
    if case.get("serve"):
        server = twins_amd.Server(arena_bytes=8 << 30, max_requests=256)
        ids = [server.submit(w) for w in worlds]
        while server.poll().done < len(ids):
            pass
        for i in ids:
            est, done, ev = server.result(i)
            times += [np.array(est), np.array(done)]
            counters.append(ev)
        server.close()
    elif case["kind"] == "tcp":
        batch = twins_amd.Batch(worlds, chain_runs=case["runs"])
        batch.run()
        for w in range(len(worlds)):
            est, done = batch.fct(w)
            times += [np.array(est), np.array(done)]
            counters.append(batch.counters(w))
        batch.close()
    else:
        batch = rdma.Batch(worlds, q3cap=case["q3cap"])
        batch.run()
        for w in range(len(worlds)):
            start, fct = batch.fct(w)
            times += [np.array(start), np.array(fct)]
        counters.append(batch.counters())
        batch.close()
    return {"times": np.concatenate(times), "counters": np.array(counters, dtype=np.uint64).astype(np.int64)}


# ------------------------------------------------------------------ what a pass cannot do without
def _links_on_path(spec):
    """Links a frame crosses from host to host, on average over random pairs."""
    name, *n = spec.split(":")
    n = [int(x) for x in n]
    if name.startswith("fattree") and n:
        k = n[0]
        hosts, edge, pod = k ** 3 / 4, k / 2, k * k / 4
        return (2 * (edge - 1) + 4 * (pod - edge) + 6 * (hosts - pod)) / (hosts - 1)
    if name == "leafspine":
        return 4 - 2 * (n[2] - 1) / (n[0] * n[2] - 1)
    if name == "torus":
        return 2 + (n[0] + n[1]) / 4
    if name == "jellyfish":
        return 2 + math.log(n[0]) / math.log(max(2, n[1] - 1))
    return 4.5


def work(case):
    """Every frame of every flow crosses its links one after another: on each it is written by the
    sending entity and read by the receiving one (64 bytes under TCP, 128 with 25-run chains; an RDMA
    link frame 176), and each crossing is one event. TCP: the data segments, an ACK for every second
    one and three frames of handshake; RDMA: an ACK for every data frame."""
    u = (np.arange(4096) + 0.5) / 4096
    payload = 1460 if case["kind"] == "tcp" else case["payload"]
    per_flow = float(np.ceil(_sizes(case, u) / payload).mean())
    data = per_flow * case["flows"] + case["incast"] * math.ceil((50000 if case["kind"] == "tcp" else 64000) / payload)
    flows = case["flows"] + case["incast"]
    frames = data * 1.5 + 3 * flows if case["kind"] == "tcp" else data * 2
    events = frames * case["worlds"] * _links_on_path(case["topo"])
    frame = (64 if case.get("runs", 9) == 9 else 128) if case["kind"] == "tcp" else 176
    return {"bytes": 2 * frame * events + 48 * flows * case["worlds"], "flops": events}


def tolerance(case):
    return "exact"
