"""What the speed of this framework is measured on: whole calls through its
public entry points, as programs that assemble reads make them.

A case is a dict of plain values.  Its "kind" names the way in:

  reads   reads already in device memory, one job that is used again and
          again (GraphJob.parse_count_device, run), FASTA bytes out
  files   host reads of uneven length fed in several portions (one per
          input file), as the driver's per-file loop does (parse_count)
  fastq   a FASTQ file's bytes from the host, split on the device, and
          every file that the driver writes out of it
  clean   reads, then the deadend / bubble cleaning loop
  batch   many independent jobs in one set of launches (GraphBatch)
  serve   requests with host reads through the request loop (Server)

The reads come from the package's seeded generator (bruno_amd.SynthConfig):
an i.i.d. genome with an optional repeat layer, sampled on both strands with
substitution and indel errors, which is what the counting, the filter and
the graph meet in earnest (most distinct k-mers are errors seen once, the
graph is long chains with few branches).

Outputs are bytes and integers.  The state holds a buffer for each, of a
size that any reads of the case fit in, and run() returns the buffer and how
much of it is filled.  "reads" and "batch" fetch the FASTA bytes into their
buffers through the C ABI, as a program does that keeps its output buffers;
the others call the Python getters.
"""
import ctypes
import math

import numpy as np

from bruno_amd import GraphBatch, GraphJob, SynthConfig, lib, thresholds_L
from bruno_amd._lib import check
from bruno_amd.device import DeviceBuffer
from bruno_amd.pipeline import estimate_distinct, job_first_read, synth_batch_device, synth_reads_device
from bruno_amd.planner import capacity
from bruno_amd.server import Server


def listed():
    return [
        # The smallest call: a file of the size of the short-read fixture
        # (243 reads of 36 bases).  Launches, read-backs and allocations.
        dict(name="fastq_fixture", kind="fastq", k=21, t=2, genome=1500, reads=243, read_len=36, sub=0.005),
        # The 1 Mbp workload (100 bp at 30x, k=31, -T -L 3): a small genome.
        dict(name="reads_1mbp", kind="reads", k=31, t=3, genome=1_000_000, reads=300_000, read_len=100, sub=0.005),
        # The benchmark's workload (150 bp at 50x, repeats, k=31) for a
        # bacterial genome, and at two fifths of the benchmark's size; "sized":
        # the table's size is asked for beforehand, as the benchmark does, and
        # not left to the job.
        dict(name="reads_4mbp", kind="reads", k=31, t=3, genome=4_600_000, reads=1_533_333, read_len=150, sub=0.01,
             families=50),
        dict(name="reads_40mbp", kind="reads", k=31, t=3, genome=40_000_000, reads=13_333_333, read_len=150,
             sub=0.01, families=50, sized=True),
        # Two-word k-mers: the k=63 workload (250 bp at 40x, indels) at half size.
        dict(name="reads_k63", kind="reads", k=63, t=3, genome=10_000_000, reads=1_600_000, read_len=250, sub=0.005,
             indel=0.0005, families=50, sized=True),
        # No thresholds (build_index): every k-mer is a node; low coverage,
        # the other list-ranking variant.
        dict(name="reads_unthresholded", kind="reads", k=21, t=0, genome=2_000_000, reads=200_001, read_len=101,
             sub=0.005, variant=0),
        # The block-construct driver's k+1-mer edge filter, an even k.
        dict(name="reads_edge_filter", kind="reads", k=26, t=3, genome=6_000_000, reads=1_600_003, read_len=125,
             sub=0.01, edge=True),
        # Several files of trimmed reads with Ns, from host memory, a
        # two-word k; the table is sized from the first file.
        dict(name="files_ragged", kind="files", k=47, t=2, genome=700_000, reads=170_000, read_len=151, sub=0.008,
             portions=5),
        # A FASTQ file with every output that the driver writes without -B.
        dict(name="fastq_outputs", kind="fastq", k=31, t=3, genome=900_000, reads=300_000, read_len=101, sub=0.008),
        # Cleaning: errors often enough to leave tips and bubbles behind.
        dict(name="clean_2mbp", kind="clean", k=31, t=2, genome=2_000_000, reads=800_000, read_len=100, sub=0.01),
        # 16 small jobs of uneven size and read length in one batch.
        dict(name="batch_16", kind="batch", k=31, t=3, jobs=16, lo=50_000, hi=2_000_000),
        # 16 requests through the request loop, k = 31 and 63.
        dict(name="serve_16", kind="serve", k=31, t=3, jobs=16, lo=20_000, hi=500_000),
    ]


def draw(rng):
    def spread(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    kind = rng.choice(["reads", "reads", "reads", "files", "fastq", "clean", "batch", "serve"])
    if kind == "batch":
        lo = int(spread(10_000, 200_000))
        return dict(kind=kind, k=rng.choice([21, 25, 31, 31, 41]), t=rng.choice([2, 3]), jobs=rng.randint(2, 16),
                    lo=lo, hi=int(lo * rng.uniform(2, 10)))
    if kind == "serve":
        lo = int(spread(5_000, 50_000))
        return dict(kind=kind, k=rng.choice([21, 27, 31, 31]), t=3, jobs=rng.randint(1, 16), lo=lo,
                    hi=int(lo * rng.uniform(2, 10)))
    read_len = rng.choice([76, 100, 101, 125, 150, 151, 250])
    k = rng.choice([k for k in (19, 21, 24, 25, 27, 31, 31, 31, 32, 47, 55, 63) if k + 10 <= read_len])
    cover = rng.uniform(15, 60)
    most = {"reads": 40e6, "files": 1e6, "fastq": 1e6, "clean": 3e6}[kind]
    if k > 31:
        most = min(most, 8e6)
    genome = int(spread(2e3 if kind == "fastq" else 5e4, most))
    c = dict(kind=kind, k=k, t=rng.choice([2, 3, 3]), genome=genome, reads=max(1, int(cover * genome / read_len)),
             read_len=read_len, sub=round(rng.uniform(0.002, 0.012), 4))
    if kind == "files":
        c["portions"] = rng.randint(1, 8)
    if kind == "reads":
        if rng.random() < 0.4:
            c["indel"] = 0.0005
        if genome >= 1_000_000 and rng.random() < 0.5:
            c["families"] = 50
        if rng.random() < 0.2:
            c["edge"] = True
        elif rng.random() < 0.2 and genome < 3e6 and k <= 31:
            c["t"] = 0
        c["variant"] = rng.choice([1, 1, 0])
        c["sized"] = rng.random() < 0.5
    # no more bases than the largest listed case has
    c["reads"] = min(c["reads"], int(2e9 / read_len))
    return c


def synth(case, seed):
    """The reads of a single-job case."""
    families = case.get("families", 0)
    repeats = dict(n_families=families, family_min_len=500, family_max_len=5000, repeat_fraction=0.02,
                   family_divergence=0.01) if families else {}
    return SynthConfig(seed=seed * 1009 + 17, genome_len=case["genome"], n_reads=case["reads"],
                       read_len=case["read_len"], sub_rate=case["sub"], indel_rate=case.get("indel", 0.0), **repeats)


def job_list(case, seed, ks):
    """Jobs of uneven size: genomes log-uniform in [lo, hi], read length 100,
    150 or 250, coverage 20-60x.  The sizes belong to the case and the reads
    to the seed.  Returns (generator settings, k of each)."""
    rng = np.random.default_rng([case["jobs"], case["lo"], case["hi"], case["k"]])
    jobs, kk = [], []
    for i in range(case["jobs"]):
        genome = int(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]))))
        read_len = int(rng.choice([100, 150, 250]))
        reads = int(rng.uniform(20, 60) * genome / read_len)
        jobs.append(SynthConfig(seed=seed * 100003 + i, genome_len=genome, n_reads=max(1, reads), read_len=read_len,
                                sub_rate=0.01))
        kk.append(ks[0] if rng.random() < 0.8 else ks[1])
    return jobs, kk


def on_device(cfg):
    bases, offsets = DeviceBuffer(max(1, cfg.n_bases)), DeviceBuffer((cfg.n_reads + 1) * 8)
    synth_reads_device(cfg, bases.ptr, offsets.ptr)
    return bases, offsets


def on_host(cfg):
    """The reads as a matrix of bases (reads x read length) in host memory."""
    bases, offsets = on_device(cfg)
    got = bases.to_numpy(np.uint8, cfg.n_bases).reshape(cfg.n_reads, cfg.read_len)
    bases.free()
    offsets.free()
    return got


def trimmed(cfg, seed, shortest):
    """Reads as a sequencer's trimmer leaves them: a third lose bases at the
    end, one in 200 holds an N.  Returns the matrix and each read's length."""
    rng = np.random.default_rng(seed)
    m = on_host(cfg)
    n, length = m.shape
    lens = np.full(n, length)
    cut = rng.random(n) < 1 / 3
    lens[cut] = rng.integers(min(shortest, length), length + 1, int(cut.sum()))
    at = np.flatnonzero(rng.random(n) < 0.005)
    m[at, rng.integers(0, length, at.size)] = ord("N")
    return m, lens


def fastq_bytes(m, lens, seed):
    """4-line records with a numbered name and qualities."""
    n, length = m.shape
    head = 12
    rec = np.empty((n, head + 2 * length + 4), np.uint8)
    rec[:, 0], rec[:, 1] = ord("@"), ord("r")
    number = np.arange(n)
    for d in range(9):
        rec[:, 10 - d] = ord("0") + number // 10 ** d % 10
    rec[:, 11] = ord("\n")
    s, q = head, head + length + 3
    rec[:, s:s + length] = m
    rec[:, s + length], rec[:, s + length + 1], rec[:, s + length + 2] = ord("\n"), ord("+"), ord("\n")
    rec[:, q:q + length] = np.random.default_rng(seed + 1).integers(33, 74, (n, length), np.uint8)
    rec[:, q + length] = ord("\n")
    keep = np.ones(rec.shape, bool)
    inside = np.arange(length)[None, :] < lens[:, None]
    keep[:, s:s + length] = inside
    keep[:, q:q + length] = inside
    return rec[keep]


def limits(case):
    return thresholds_L(case["t"]) if case["t"] else None


def room(case, genome):
    """(k-mers, FASTA bytes) that any reads of a case of this genome leave at
    most, generously: errors that pass the thresholds come on top of the
    genome's k-mers, all errors without thresholds."""
    if case["t"]:
        kmers = genome * (2 if case["t"] > 2 else 8)
    else:
        kmers = 2 * genome + int(2 * case["reads"] * case["read_len"] * case["sub"] * case["k"])
    return kmers + 1000, 4 * kmers + (1 << 16)


def prepare(case, seed):
    kind, k = case["kind"], case["k"]
    st = {"kind": kind, "t": case["t"], "variant": case.get("variant", 1)}
    if kind in ("batch", "serve"):
        jobs, ks = job_list(case, seed, (k, k if kind == "batch" else 63))
        st["out"] = []
        for c in jobs:
            size = room(case, c.genome_len)[1]
            st["out"].append([np.zeros(size, np.uint8), np.zeros(size, np.uint8)])
    else:
        kmers, size = room(case, case["genome"])
        st["out"] = [np.zeros(size, np.uint8), np.zeros(size, np.uint8)]
    if kind == "batch":
        bases = DeviceBuffer(sum(c.n_bases for c in jobs))
        offsets = DeviceBuffer((sum(c.n_reads for c in jobs) + 1) * 8)
        synth_batch_device(jobs, bases.ptr, offsets.ptr)
        st.update(bases=bases, offsets=offsets, first=job_first_read(jobs), n=sum(c.n_reads for c in jobs),
                  job=GraphBatch(k, limits(case), [capacity(c, k) for c in jobs]))
    elif kind == "serve":
        st["requests"] = []
        for c, kk in zip(jobs, ks):
            m = on_host(c)
            offsets = np.arange(c.n_reads + 1, dtype=np.uint64) * c.read_len
            st["requests"].append((kk, limits(case), m.reshape(-1), offsets, capacity(c, kk)))
        st["server"] = Server(hbm_budget=32 << 30, reserve_pool=False)
    elif kind == "fastq":
        m, lens = trimmed(synth(case, seed), seed, k)
        st.update(data=fastq_bytes(m, lens, seed), job=GraphJob(k, limits(case)))
        # records of 40 (chain and branch nodes) and 64 bytes (chain edges)
        st["records"] = [np.zeros(kmers * n, np.uint64) for n in (5, 5, 8)]
    elif kind == "files":
        m, lens = trimmed(synth(case, seed), seed, k)
        at = np.linspace(0, len(m), case["portions"] + 1).astype(int)
        st["files"] = []
        for a, b in zip(at[:-1], at[1:]):
            offsets = np.concatenate([[0], np.cumsum(lens[a:b])]).astype(np.uint64)
            st["files"].append((m[a:b][np.arange(m.shape[1])[None, :] < lens[a:b, None]], offsets))
        st["job"] = GraphJob(k, limits(case))
    else:  # reads, clean
        cfg = synth(case, seed)
        st["bases"], st["offsets"] = on_device(cfg)
        st["n"] = cfg.n_reads
        slots = estimate_distinct(k, st["bases"].ptr, st["offsets"].ptr, cfg.n_reads)[1] if case.get("sized") else 0
        st["job"] = GraphJob(k, limits(case), capacity=slots, edge_filter=case.get("edge", False))
        if kind == "reads":
            # a job that runs again and again and hands out FASTA only
            st["job"].set_recycle(True)
    return st


def fetch(getter, out, *handle):
    """A two-call getter of the C ABI into the caller's buffer."""
    n = ctypes.c_uint64(0)
    check(getter(*handle, None, ctypes.byref(n)), getter.__name__)
    if n.value > out.size:
        raise ValueError("%d bytes for a buffer of %d" % (n.value, out.size))
    check(getter(*handle, ctypes.c_void_p(out.ctypes.data), ctypes.byref(n)), getter.__name__)
    return [out, n.value]


def put(out, got):
    """What a Python getter returned (bytes or records), in the buffer."""
    got = np.frombuffer(got, out.dtype)
    out[:got.size] = got
    return [out, got.size]


def run(st):
    kind = st["kind"]
    if kind == "serve":
        srv = st["server"]
        tickets = [srv.submit_reads(*q) for q in st["requests"]]
        got = []
        for t, (unitigs, branches) in zip(tickets, st["out"]):
            srv.wait(t)
            got.append([put(unitigs, srv.unitigs(t)), put(branches, srv.branch_fasta(t))])
            srv.release(t)
        return got
    job = st["job"]
    job.reset()
    if kind == "batch":
        job.parse_count_device(st["bases"].ptr, st["offsets"].ptr, st["n"], st["first"])
        job.run(st["variant"])
        return [[fetch(lib().bruno_batch_get_unitigs, unitigs, job.h, i),
                 fetch(lib().bruno_batch_get_branch_fasta, branches, job.h, i)]
                for i, (unitigs, branches) in enumerate(st["out"])]
    if kind == "fastq":
        job.parse_count_fastq(st["data"])
    elif kind == "files":
        for bases, offsets in st["files"]:
            job.parse_count(bases, offsets)
    else:
        job.parse_count_device(st["bases"].ptr, st["offsets"].ptr, st["n"])
    job.run(st["variant"])
    unitigs, branches = st["out"]
    if kind == "reads":
        return [fetch(lib().bruno_get_unitigs, unitigs, job.h), fetch(lib().bruno_get_branch_fasta, branches, job.h)]
    got = []
    if kind == "clean":
        got.append(job.clean(st["variant"], st["t"]))
    got += [put(unitigs, job.unitigs()), put(branches, job.branch_fasta())]
    if kind == "fastq":
        for out, records in zip(st["records"], (job.chain_nodes(), job.branch_nodes(), job.chain_edges())):
            got.append(put(out, records))
    return got


def work(case):
    """Input bytes read once, output bytes written once (no floating-point
    work).  Kept k-mers: about the genome's, and without thresholds also the
    ones that each error creates."""
    k, kind = case["k"], case["kind"]
    if kind in ("batch", "serve"):
        jobs, _ = job_list(case, 1, (k, k))
        return {"bytes": sum(c.n_bases + 8 * c.n_reads + c.genome_len for c in jobs), "flops": 0}
    bases = case["reads"] * case["read_len"]
    kept = case["genome"]
    if not case["t"]:
        kept += bases * case["sub"] * min(k, case["read_len"] - k)
    moved = kept + (2 * bases + 16 * case["reads"] if kind == "fastq" else bases + 8 * case["reads"])
    if kind == "fastq":
        moved += 36 * kept
    return {"bytes": int(moved), "flops": 0}
