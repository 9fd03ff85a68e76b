"""What this framework is used for, as cases whose time can be measured.

Each case is a call (or the few calls) that a program mapping reads makes: the per-read API, one host-buffer
call, batches resident in HBM, the pair step on their NAMs, the seeding stage alone, index lookups alone, a
whole read file host to host, and building an index. The programs keep what a real one keeps: the index of
their reference (built once per process), the batches their reads sit in, and pinned output arrays.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the inputs (reads, keys or genome made from the seed) and handles
    run(state)          one pass; returns every output
    work(case)          bytes that one pass cannot do without
    exact(case, seed)   None: see there

Every output is a whole number or is returned as its bit pattern, so results compare bit for bit.
"""
import ctypes

import numpy as np

import gpu_index_test_amd as G
from gpu_index_test_amd import _native

# The references the programs hold an index of. "bacterial": two replicons, hardly any repeats, at the profiles
# of 150 bp and of 400+ bp reads. "mid": the 100 Mbp genome with 5% repeats of the default benchmark. "repeats":
# the repeat content of the human-scale benchmark (45% repeats, 2% tandem repeats) at 400 Mbp, which is far
# beyond every cache.
_GENOMES = {
    "bacterial": dict(total_length=5_000_000, n_contigs=2, gc=0.5, repeat_fraction=0.02, n_families=20,
                      family_len=(500, 5000), copies=(2, 10), seed=1),
    "mid": dict(total_length=100_000_000, n_contigs=8, gc=0.41, repeat_fraction=0.05, n_families=500,
                family_len=(1000, 10000), copies=(2, 50), divergence=(0.01, 0.05), seed=1),
    "repeats": dict(total_length=400_000_000, n_contigs=24, gc=0.41, repeat_fraction=0.45, n_families=645,
                    family_len=(300, 6000), copies=(2, 50), divergence=(0.02, 0.20), tandem_fraction=0.02,
                    tandem_unit=(2, 50), seed=1),
}
# reference -> (genome, read length of the index profile)
_REFERENCES = {"bacterial": ("bacterial", 150), "bacterial-long": ("bacterial", 400), "mid": ("mid", 150),
               "repeats": ("repeats", 150)}
# read length mixtures: the fixed 150 bp of most sequencing runs, the uneven mixture of the batched benchmark,
# older short runs, and merged or long reads beyond the longest profile
_MIXES = {
    "150": ((150,), (1.0,)),
    "uneven": ((50, 100, 150, 250, 300), (0.1, 0.2, 0.4, 0.2, 0.1)),
    "short": ((50, 75, 101), (0.2, 0.4, 0.4)),
    "long": ((400, 500, 1000, 2500), (0.4, 0.4, 0.15, 0.05)),
}
# NAMs per read of each reference's reads, and the room that a program leaves for them
_NAMS = {"bacterial": 7.8, "bacterial-long": 24, "mid": 7.9, "repeats": 10.4}
_NAM_ROOM = {"bacterial": 12, "bacterial-long": 40, "mid": 14, "repeats": 24}
_MODES = {"plain": G.MODE_PLAIN, "fused": G.MODE_FUSED}

_genomes, _indexes = {}, {}


def listed():
    return [
        # an aligner's worker thread: one read through the reference's per-read calls
        {"name": "read", "kind": "read", "reference": "mid", "length": 150},
        # a small interactive or served request: a few hundred reads in one host-buffer call
        {"name": "call_293", "kind": "call", "reference": "mid", "mix": "150", "reads": 293, "mode": "plain"},
        # a microbial sample: small index, nearly all reads unique; reads resident, results copied back
        {"name": "batch_bacterial", "kind": "batch", "reference": "bacterial", "mix": "150", "reads": 65536,
         "mode": "plain", "lanes": 1},
        # the default benchmark: 65,536-read batches, several in flight
        {"name": "batch_150", "kind": "batch", "reference": "mid", "mix": "150", "reads": 65536, "mode": "plain",
         "lanes": 3},
        # the batched benchmark: uneven paired reads through the fused form
        {"name": "batch_uneven_fused", "kind": "batch", "reference": "mid", "mix": "uneven", "reads": 131072,
         "mode": "fused", "lanes": 1},
        # a repeat-rich genome: rescue and heavy merges
        {"name": "batch_repeats", "kind": "batch", "reference": "repeats", "mix": "150", "reads": 100003,
         "mode": "plain", "lanes": 1},
        # merged and long reads on a long-read profile
        {"name": "batch_long", "kind": "batch", "reference": "bacterial-long", "mix": "long", "reads": 8191,
         "mode": "plain", "lanes": 1},
        # the step after mapping: pair types, MAPQ and joint NAM pairs of a paired batch
        {"name": "pairs_32k", "kind": "pairs", "reference": "mid", "mix": "uneven", "pairs": 32768},
        # the seeding stage alone (randstrobes_query of a batch), for callers with a search of their own
        {"name": "seeds_20k", "kind": "seeds", "reference": "mid", "mix": "150", "reads": 20011},
        # the index search alone (find of a list of hashes)
        {"name": "find_1m", "kind": "find", "reference": "repeats", "keys": 1_000_003},
        # a read file from host memory to NAMs in host memory
        {"name": "stream_500k", "kind": "stream", "reference": "mid", "mix": "150", "reads": 500_000,
         "batch_reads": 65536, "lanes": 4, "mode": "plain"},
        # building the index of a new reference, its table handed to the host
        {"name": "build_20m", "kind": "build", "bases": 20_000_000, "contigs": 7, "profile": 150},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["read", "call", "call", "batch", "batch", "batch", "batch", "pairs", "seeds", "find",
                       "stream", "build"])
    if kind == "read":
        return {"kind": kind, "reference": rng.choice(["bacterial", "mid"]), "length": rng.randint(50, 300)}
    if kind == "call":
        return {"kind": kind, "reference": rng.choice(["bacterial", "mid", "repeats"]),
                "mix": rng.choice(["150", "uneven", "short"]), "reads": _log_int(rng, 1, 4096),
                "mode": rng.choice(["plain", "plain", "fused"])}
    if kind == "batch":
        reference = rng.choice(list(_REFERENCES))
        if reference == "bacterial-long":
            return {"kind": kind, "reference": reference, "mix": "long", "reads": _log_int(rng, 1000, 16000),
                    "mode": "plain", "lanes": 1}
        lanes = rng.choice([1, 1, 2, 3])
        return {"kind": kind, "reference": reference, "mix": rng.choice(["150", "150", "uneven", "short"]),
                "reads": _log_int(rng, 8000, 131072 // lanes), "mode": rng.choice(["plain", "plain", "fused"]),
                "lanes": lanes}
    if kind == "pairs":
        return {"kind": kind, "reference": rng.choice(["bacterial", "mid"]), "mix": rng.choice(["150", "uneven"]),
                "pairs": _log_int(rng, 1000, 65536)}
    if kind == "seeds":
        return {"kind": kind, "reference": rng.choice(["bacterial", "mid"]),
                "mix": rng.choice(["150", "uneven", "short"]), "reads": _log_int(rng, 500, 65536)}
    if kind == "find":
        return {"kind": kind, "reference": rng.choice(["bacterial", "mid", "repeats"]),
                "keys": _log_int(rng, 1000, 4_000_000)}
    if kind == "stream":
        return {"kind": kind, "reference": rng.choice(["bacterial", "mid"]), "mix": rng.choice(["150", "uneven"]),
                "reads": _log_int(rng, 150_000, 500_000), "batch_reads": rng.choice([32768, 65536]),
                "lanes": rng.randint(2, 4), "mode": rng.choice(["plain", "fused"])}
    return {"kind": kind, "bases": _log_int(rng, 500_000, 20_000_000), "contigs": rng.randint(1, 40),
            "profile": rng.choice([100, 150, 250, 400])}


# ---------------- what the programs keep ----------------

def _genome(name):
    if name not in _genomes:
        spec = dict(_GENOMES[name])
        _genomes[name] = G.synth_genome(spec.pop("total_length"), **spec)
    return _genomes[name]


def _index(reference):
    if reference not in _indexes:
        name, profile = _REFERENCES[reference]
        genome, contigs = _genome(name)
        index = G.StrobemerIndex(None, G.IndexParameters.from_read_length(profile))
        index.populate_arrays(genome, contigs)
        _indexes[reference] = index
    return _indexes[reference]


def _reads(reference, mix, n, seed, paired=False):
    genome, contigs = _genome(_REFERENCES[reference][0])
    lengths, weights = _MIXES[mix]
    seqs, offsets, lens, _ = G.synth_reads(genome, contigs, n // 2 if paired else n, lengths=lengths,
                                           weights=weights, paired=paired, sub_rate=0.005, indel_rate=0.0005,
                                           insert=(400.0, 50.0), seed=seed + 1)
    if paired:  # mate 1 block, then mate 2 block
        order = np.concatenate([np.arange(0, n, 2), np.arange(1, n, 2)])
        offsets, lens = offsets[order], lens[order]
    return seqs, offsets, lens


def _zeros(n, dtype, pinned=True):
    """An array that a program keeps for results (pinned unless it is a plain host array)."""
    a = G.pinned_empty(n, dtype) if pinned else np.empty(n, dtype)
    a.view(np.uint8)[...] = 0
    return a


class _Nams:
    """The arrays a program keeps for the NAMs of n reads: results land at their front, the rest stays zero."""

    def __init__(self, reference, n, pinned=True):
        self.pinned = pinned
        self.offsets, self.nams = _zeros(n + 1, np.uint64, pinned), None
        self.fraction, self.flags = _zeros(n, np.float32, pinned), _zeros(n, np.uint8, pinned)
        self.out = _native.NamOut(nam_offsets=self.offsets.ctypes.data,
                                  nonrepetitive_fraction=self.fraction.ctypes.data,
                                  flags=self.flags.ctypes.data)
        self.grow(_NAM_ROOM[reference] * n + 8192)

    def grow(self, nams):
        self.nams = _zeros(nams, G.NAM, self.pinned)
        self.out.nams, self.out.nam_capacity = self.nams.ctypes.data, nams

    def call(self, ctx, fn):
        """fn(NamOut), again with more room where the arrays were too small; then the results."""
        code = fn(ctypes.byref(self.out))
        if code == 5 and self.out.n_nams > len(self.nams):  # GIS_ERR_CAPACITY: the count is set
            self.grow(self.out.n_nams + self.out.n_nams // 8)
            code = fn(ctypes.byref(self.out))
        ctx.check(code)
        return [_bits(self.offsets), _words(self.nams), _bits(self.fraction), self.flags]


class _Batch:
    """A resident batch and the pinned arrays its results are copied to."""

    def __init__(self, reference, reads, mode, own_stream=False):
        seqs, offsets, lens = reads
        self.m = G.Mapper(_index(reference), len(lens), int(lens.sum()), own_stream=own_stream)
        self.m.upload(seqs, offsets, lens)
        self.mode, self.nams = mode, _Nams(reference, len(lens))

    def download(self):
        ctx = self.m.ctx
        return self.nams.call(ctx, lambda out: ctx.L.gis_batch_download(self.m.h, out))


class _Pairs:
    """A resident paired batch, mapped, and the pinned arrays of the pair step's results."""

    def __init__(self, reference, reads):
        self.b = _Batch(reference, reads, G.MODE_PLAIN)
        self.b.m.run()
        n = self.n = self.b.m.n // 2
        self.offsets, self.types, self.ids = _zeros(2 * n + 1, np.uint64), _zeros(n, np.uint8), _zeros(n, np.uint32)
        self.dropoff, self.mapq = _zeros(2 * n, np.float32), _zeros(2 * n, np.uint8)
        self.joint_offsets = _zeros(n + 1, np.uint64)
        self.params = _native.PairParams()
        self.b.m.ctx.L.gis_pair_params_default(ctypes.byref(self.params))
        self.params.flags = _native.PAIRS_JOINT
        self.out = _native.PairOut(nam_offsets=self.offsets.ctypes.data, types=self.types.ctypes.data,
                                   type_ids=self.ids.ctypes.data, top_dropoff=self.dropoff.ctypes.data,
                                   mapq=self.mapq.ctypes.data, joint_offsets=self.joint_offsets.ctypes.data)
        self.grow(2 * _NAM_ROOM[reference] * n + 8192, 12 * n + 8192)

    def grow(self, nams, joint):
        self.nams, self.joint = _zeros(nams, G.NAM), _zeros(joint, G.NAM_PAIR)
        self.out.nams, self.out.nam_capacity = self.nams.ctypes.data, nams
        self.out.joint, self.out.joint_capacity = self.joint.ctypes.data, joint

    def run(self):
        m, out = self.b.m, self.out
        m.ctx.check(m.ctx.L.gis_batch_pairs(m.h, ctypes.byref(self.params)))
        code = m.ctx.L.gis_batch_pairs_download(m.h, ctypes.byref(out))
        if code == 5:  # GIS_ERR_CAPACITY: the counts are set
            self.grow(max(out.n_nams, len(self.nams)), max(out.n_joint, len(self.joint)))
            code = m.ctx.L.gis_batch_pairs_download(m.h, ctypes.byref(out))
        m.ctx.check(code)
        return [_bits(self.offsets), _words(self.nams), self.types, _bits(self.ids), list(out.type_counts),
                _bits(self.dropoff), self.mapq, _bits(self.joint_offsets), _words(self.joint)]


def _words(records):
    """A record array as rows of 32-bit words."""
    return records.view(np.int32).reshape(len(records), records.dtype.itemsize // 4)


def _bits(a):
    return a.view({4: np.int32, 8: np.int64}[a.dtype.itemsize])


def _queries(q):
    """Query randstrobes by field (is_reverse and its padding as one word pair)."""
    w = q.view(np.int32).reshape(len(q), 6)
    return [q["hash"].view(np.int64), w[:, 2:5]]


def _kept(kept, got):
    """`got` at the front of the array that the program keeps, the rest zero."""
    kept[:len(got)] = got
    return kept


# ---------------- the cases ----------------

def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "build":
        s["genome"] = G.synth_genome(case["bases"], n_contigs=case["contigs"], gc=0.45, repeat_fraction=0.05,
                                     n_families=30, family_len=(500, 5000), copies=(2, 20), seed=seed + 1)
        s["index"] = G.StrobemerIndex(None, G.IndexParameters.from_read_length(case["profile"]))
        # the table that the host keeps: about a randstrobe per k - s + 1 bases
        s["table"], s["starts"] = _zeros(case["bases"] // 3, _native.REF_RANDSTROBE), None
        return s
    index = s["index"] = _index(case["reference"])
    if kind == "read":
        genome, contigs = _genome(_REFERENCES[case["reference"]][0])
        seqs, _, lens, _ = G.synth_reads(genome, contigs, 1, lengths=(case["length"],), sub_rate=0.005,
                                         indel_rate=0.0005, seed=seed + 1)
        s["read"], s["rescue_cutoff"] = seqs[:int(lens[0])].tobytes(), 2 * index.filter_cutoff
        s["queries"], s["nams"] = _zeros(128, G.QUERY_RANDSTROBE, False), _zeros(4096, G.NAM, False)
    elif kind == "call":
        s["reads"] = _reads(case["reference"], case["mix"], case["reads"], seed)
        s["nams"] = _Nams(case["reference"], case["reads"], pinned=False)
        s["options"] = _options(index, case["mode"])
    elif kind == "seeds":
        s["reads"] = _reads(case["reference"], case["mix"], case["reads"], seed)
        s["queries"] = _zeros(int(case["reads"] * (1.25 * _seeds_of(_mean_length(case["mix"])) + 8)) + 4096,
                              G.QUERY_RANDSTROBE, False)
        s["offsets"] = _zeros(case["reads"] + 1, np.uint64, False)
    elif kind == "batch":
        # lanes: batches with a stream of their own each, all in flight at once
        s["batches"] = [_Batch(case["reference"],
                               _reads(case["reference"], case["mix"], case["reads"], 16 * seed + lane),
                               _MODES[case["mode"]], own_stream=case["lanes"] > 1)
                        for lane in range(case["lanes"])]
    elif kind == "pairs":
        s["pairs"] = _Pairs(case["reference"],
                            _reads(case["reference"], case["mix"], 2 * case["pairs"], seed, paired=True))
    elif kind == "find":
        # hashes of randstrobes of the reference's own reads, and a tenth that no index holds
        n = case["keys"]
        rng = np.random.default_rng(seed)
        known = _hashes(case["reference"])
        keys = known[rng.integers(0, len(known), n)]
        keys[rng.random(n) < 0.1] ^= np.uint64(0x5555)
        s["keys"] = keys
    elif kind == "stream":
        s["reads"] = [G.pinned_copy(a) for a in _reads(case["reference"], case["mix"], case["reads"], seed)]
        s["nams"], s["options"] = _Nams(case["reference"], case["reads"]), _options(index, case["mode"])
    return s


def _options(index, mode):
    options = _native.MapOptions()
    index.ctx.L.gis_map_options_default(ctypes.byref(options))
    options.mode = _MODES[mode]
    return options


def _addresses(reads):
    return [a.ctypes.data for a in reads]


def _hashes(reference):
    """Query hashes of some reads of a reference (one sample per process)."""
    key = ("hashes", reference)
    if key not in _indexes:
        reads = _reads(reference, "150", 30_000, 7)
        _indexes[key] = np.ascontiguousarray(G.randstrobes_batch(_index(reference), *reads)[1]["hash"])
    return _indexes[key]


def run(s):
    case, kind, index = s["case"], s["case"]["kind"], s["index"]
    if kind == "read":
        # the caller's loop over its reads (randstrobes_query, find_nams, find_nams_rescue when needed)
        q = G.randstrobes_query(s["read"], index)
        fraction, nams = G.find_nams(q, index)
        if fraction < 0.7 or len(nams) == 0:
            nams = G.find_nams_rescue(q, index, s["rescue_cutoff"])
        return [*_queries(_kept(s["queries"], q)), fraction, _words(_kept(s["nams"], nams))]
    ctx = index.ctx
    if kind == "call":
        return s["nams"].call(ctx, lambda out: ctx.L.gis_find_nams_batch(
            ctx.h, *_addresses(s["reads"]), case["reads"], ctypes.byref(s["options"]), out))
    if kind == "batch":
        batches = s["batches"]
        if len(batches) == 1:
            batches[0].m.run(mode=batches[0].mode)
            return batches[0].download()
        for b in batches:
            b.m.launch(mode=b.mode)
        out = []
        for b in batches:
            b.m.wait()
            out.append(b.download())
        return out
    if kind == "pairs":
        return s["pairs"].run()
    if kind == "seeds":
        count = ctypes.c_uint64()
        ctx.check(ctx.L.gis_randstrobes_batch(ctx.h, *_addresses(s["reads"]), case["reads"],
                                              s["offsets"].ctypes.data, s["queries"].ctypes.data,
                                              len(s["queries"]), ctypes.byref(count)))
        return [_bits(s["offsets"]), int(count.value), *_queries(s["queries"])]
    if kind == "find":
        return index.find_many(s["keys"]).view(np.int64)
    if kind == "stream":
        return s["nams"].call(ctx, lambda out: ctx.L.gis_find_nams_stream(
            ctx.h, *_addresses(s["reads"]), case["reads"], case["batch_reads"], case["lanes"],
            ctypes.byref(s["options"]), out, None))
    # build: the index, then its table copied to the host
    genome, contigs = s["genome"]
    index.populate_arrays(genome, contigs)
    info = index.info()
    if info.n_randstrobes > len(s["table"]):
        s["table"] = _zeros(info.n_randstrobes, _native.REF_RANDSTROBE)
    if s["starts"] is None:
        s["starts"] = _zeros((1 << info.bits) + 1, np.uint64)
    ctx.check(ctx.L.gis_index_download(ctx.h, s["table"].ctypes.data, s["starts"].ctypes.data))
    return [_words(s["table"]), _bits(s["starts"]), int(info.bits), int(info.filter_cutoff),
            int(info.distinct_strobemers), int(info.tot_occur_once)]


def _mean_length(mix):
    lengths, weights = _MIXES[mix]
    return sum(a * b for a, b in zip(lengths, weights)) / sum(weights)


def _seeds_of(length):
    """Query randstrobes of a read: both strands, about one syncmer per 5 bases, w_min of them without one."""
    return max(0.0, 2 * ((length - 19) / 5 - 5))


def work(case):
    """Bytes: reads, keys or genome in, results out, and per looked-up randstrobe the 57 table bytes that its
    search reads (bucket bounds, records up to the key, filter probe). The path is integer work; its
    operations are left out."""
    kind = case["kind"]
    if kind == "find":
        return {"bytes": case["keys"] * (8 + 57 + 8), "flops": 0}
    if kind == "build":
        records = case["bases"] / 5
        return {"bytes": case["bases"] + records * (16 + 8), "flops": 0}
    if kind == "pairs":
        per_pair = 2 * (_NAMS[case["reference"]] * 44 * 2 + 8 + 4 + 1) + 1 + 4 + 8 + 12 * 4
        return {"bytes": case["pairs"] * per_pair, "flops": 0}
    length = case["length"] if kind == "read" else _mean_length(case["mix"])
    seeds = _seeds_of(length)
    n = 1 if kind == "read" else case["reads"]
    if kind == "batch":
        n *= case["lanes"]
    if kind == "seeds":
        return {"bytes": n * (length + 12 + seeds * 24 + 8), "flops": 0}
    return {"bytes": n * (length + 12 + seeds * 57 + _NAMS[case["reference"]] * 44 + 8 + 4 + 1), "flops": 0}


def exact(case, seed):
    """Outputs are whole numbers, or ratios and scores of whole numbers returned as bit patterns: they are equal
    or they are wrong, and there is no value in more digits to compare them with."""
    return None
