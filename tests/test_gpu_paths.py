"""Edges of single kernels and dispatch branches, against the oracle, bit for bit."""
import ctypes
import time

import numpy as np
import pytest

import gpu_index_test_amd as G
from oracle import oracle_lib as O
from tests.helpers import tiny_index_arrays
from tests.test_gpu_pairs import _compare, _flatten, _proper_rich_pair
from tests.test_pairs_oracle import rand_list

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [8, 13])
def test_bucket_lines_of_every_size(ctx, bits):
    """Buckets of 0 to 9 records, equal, adjacent and apart, up to the bucket's
    ends; every hash, its neighbours and the ends are looked up."""
    rng = np.random.default_rng(bits)
    low = 64 - bits - 9
    ents, keys = [], [0, 1, 2 ** 64 - 1]
    for top in range(2, 250):
        base = top << (64 - bits)
        n = top % 10
        fps = rng.choice([0, 1, 255, 256, 510, 511], size=n) if top % 3 else np.full(n, rng.integers(0, 512))
        hashes = [base | (int(f) << low) | int(rng.choice([0, 1, 2, 3, (1 << low) - 1])) for f in fps]
        ents += [(h, 1000 + 10 * i + top, (top % 5) << 8 | int(rng.integers(0, 60))) for i, h in enumerate(hashes)]
        keys += hashes + [h + 1 for h in hashes] + [h - 1 for h in hashes]
        keys += [base, base + 1, base | (511 << low), base | ((1 << (64 - bits)) - 1)]
    arr, starts = tiny_index_arrays(ents, bits)
    op = O.params_from_read_length(150)
    oidx = O.Index.wrap(arr, starts, bits, 30, op)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.upload(arr, starts, bits, 30)
    keys = np.array(keys, dtype=np.uint64)
    assert np.array_equal(idx.find_many(keys), np.array([oidx.find(int(k)) for k in keys], dtype=np.uint64))
    for part in np.array_split(keys, 40):
        q = np.zeros(len(part), dtype=O.QUERY_RANDSTROBE)
        q["hash"], q["start"] = part, np.arange(len(part)) * 2
        q["end"] = q["start"] + 20 + np.arange(len(part)) % 45
        fr, nams = G.find_nams(q, idx)
        efr, enams, _ = O.find_nams(oidx, q, canonical=True)
        assert np.float32(fr).tobytes() == np.float32(efr).tobytes()
        assert nams.tobytes() == enams.tobytes()
    idx.ctx.close()



@pytest.mark.parametrize("profile", [150, 300, 400])
def test_seeding_pass_edges(ctx, profile):
    """Read lengths around the seeding's pass sizes (4, 64, 256 bases, the
    320-base and 4096-base LDS limits, more and fewer than 448 syncmers), at every alignment of a read's first byte, with every
    kind of byte (either case, U, IUPAC codes, bytes outside ASCII) and
    windows with equal s-mers, through randstrobes_query."""
    rng = np.random.default_rng(profile)
    acgt = np.frombuffer(b"ACGT", dtype=np.uint8)
    reads = []
    for L in list(range(0, 26)) + [62, 63, 64, 65, 127, 128, 129, 150, 151, 252, 253, 254, 255, 256, 257, 258, 259,
                                   260, 318, 319, 320, 321, 322, 511, 512, 513, 767, 1025, 2600, 4000, 4096, 4097]:
        r = acgt[rng.integers(0, 4, L)]
        reads.append(r)
        for byte in (b"N", b"U", b"u", b"t", b"a", b"M", b"!", b"\x00", b"\xc1", b"\xff", b"3", b"\x14"):
            if L:
                x = r.copy()
                x[rng.integers(0, L, 1 + L // 200)] = byte[0]
                reads.append(x)
        if L > 40:  # a tandem of period 1 .. 7: tied windows
            x = r.copy()
            u = r[: 1 + L % 7]
            x[5:40] = np.resize(u, 35)
            reads.append(x)
    p = G.IndexParameters.from_read_length(profile)
    op = O.params_from_read_length(profile)
    ents = [(h, 10 * i, 5) for i, h in enumerate(rng.integers(1, 2 ** 63, 50).tolist())]
    arr, starts = tiny_index_arrays(ents)
    idx = G.StrobemerIndex(None, p)
    idx.upload(arr, starts, 8, 30)
    s, o, l = G.pack_reads([r.tobytes() for r in reads])
    off, q = G.randstrobes_batch(idx, s, o, l)
    soff, sy = G.syncmers_batch(idx, s, o, l)
    for i, r in enumerate(reads):
        e = O.randstrobes_query(r.tobytes(), op)
        assert q[int(off[i]): int(off[i + 1])].tobytes() == e.tobytes(), (i, len(r))
        e = O.syncmers(r.tobytes(), op)
        assert sy[int(soff[i]): int(soff[i + 1])].tobytes() == e.tobytes(), (i, len(r))
    idx.ctx.close()


@pytest.mark.parametrize("mode", [G.MODE_PLAIN, G.MODE_FUSED])
def test_filter_cutoff_inside_a_bucket_line(ctx, mode):
    """A filter cutoff below seven filters runs that fit a bucket's line; a
    rescued read takes them all the same (count <= hard cutoff)."""
    g, lens = G.synth_genome(200_000, n_contigs=2, gc=0.45, repeat_fraction=0.5, n_families=12,
                             family_len=(400, 1500), copies=(2, 12), divergence=(0.0, 0.005), seed=3)
    op = O.params_from_read_length(150)
    built = O.Index.build_arrays(g, lens, op, n_threads=4)
    oidx = O.Index.wrap(built.randstrobes, built.starts, built.bits, 2, op)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.upload(built.randstrobes, built.starts, built.bits, 2)
    s, o, l, _ = G.synth_reads(g, lens, 600, lengths=(100, 150, 250), weights=(1, 1, 1), sub_rate=0.005, seed=4)
    res = G.find_nams_batch(idx, s, o, l, mode=mode)
    eo, en, ef, efl = O.map_batch(oidx, s, o, l, 2 * 2, 1000, 4)
    assert (efl & 1).sum() > 50
    assert np.array_equal(res.nam_offsets, eo) and res.nams.tobytes() == en.tobytes()
    assert res.nonrepetitive_fraction.tobytes() == ef.tobytes() and np.array_equal(res.flags & 1, efl & 1)
    idx.ctx.close()


@pytest.mark.parametrize("n", [1, 15, 17, 1023, 1024, 1025, 65537, 1_048_576, 1_048_577])
def test_output_offsets_over_tiles(ctx, n):
    """NAM offsets and the dense output around the scan's tile (1024 reads)
    and the count of tiles each wave sums itself: one mapped read among reads
    too short to map, again and again, equals that read's NAMs repeated."""
    g, lens = G.synth_genome(100_000, n_contigs=1, gc=0.45, seed=21)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.populate_arrays(g, lens)
    s = g[5000:5150].copy()
    l = np.full(n, 25, dtype=np.uint32)
    l[::29] = 150
    o = np.zeros(n, dtype=np.uint64)
    one = G.find_nams_batch(idx, s, o[:1], np.array([150], dtype=np.uint32))
    assert len(one.nams) > 0
    res = G.find_nams_batch(idx, s, o, l)
    k = len(range(0, n, 29))
    assert np.array_equal(np.diff(res.nam_offsets), np.where(l == 150, len(one.nams), 0))
    assert res.nam_offsets[0] == 0 and res.nams.tobytes() == one.nams.tobytes() * k
    idx.ctx.close()


@pytest.mark.parametrize("mode", [G.MODE_PLAIN, G.MODE_FUSED])
def test_host_calls_of_any_size(ctx, mode):
    """Host-buffer calls around the size up to which inputs and results go
    through pinned memory, empty and single ones, and reads with more NAMs
    than that way has room for; each size three times (the third replays a
    captured graph), interleaved with the others."""
    g, lens = G.synth_genome(300_000, n_contigs=2, gc=0.45, repeat_fraction=0.5, n_families=3,
                             family_len=(2000, 3000), copies=(40, 50), divergence=(0.0, 0.01), seed=31)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.populate_arrays(g, lens)
    oidx = O.Index.build_arrays(g, lens, O.params_from_read_length(150), n_threads=4)
    cases = []
    for n in (0, 1, 2, 63, 700, 4095, 4096, 4097, 9000):
        s, o, l, _ = G.synth_reads(g, lens, n, lengths=(60, 150, 201), weights=(1, 2, 1), sub_rate=0.004, seed=n + 1)
        cases.append((s, o, l) + (O.map_batch(oidx, s, o, l, 2 * oidx.filter_cutoff, 1000, 4) if n else
                                  (np.zeros(1, np.uint64), np.zeros(0, G.NAM), np.zeros(0, np.float32), np.zeros(0, np.uint8))))
    assert any(len(en) > 16 * len(l) + 1024 for _, _, l, _, en, _, _ in cases if 0 < len(l) <= 4096)
    for _ in range(3):
        for s, o, l, eo, en, ef, efl in cases:
            res = G.find_nams_batch(idx, s, o, l, mode=mode)
            assert np.array_equal(res.nam_offsets, eo) and res.nams.tobytes() == en.tobytes()
            assert res.nonrepetitive_fraction.tobytes() == ef.tobytes() and np.array_equal(res.flags & 1, efl & 1)
    # the seeding entry points over the same sizes
    if mode == G.MODE_PLAIN:
        op = O.params_from_read_length(150)
        for s, o, l, *_ in cases:
            off, q = G.randstrobes_batch(idx, s, o, l)
            soff, sy = G.syncmers_batch(idx, s, o, l)
            assert off[0] == 0 and off[-1] == len(q) and soff[0] == 0 and soff[-1] == len(sy)
            for r in range(0, len(l), 97):
                read = s[int(o[r]): int(o[r]) + int(l[r])].tobytes()
                assert q[int(off[r]): int(off[r + 1])].tobytes() == O.randstrobes_query(read, op).tobytes()
                assert sy[int(soff[r]): int(soff[r + 1])].tobytes() == O.syncmers(read, op).tobytes()
    idx.ctx.close()


@pytest.mark.parametrize("hits", [1, 15, 16, 17, 33, 63, 64, 65, 66, 127, 128, 129, 255, 256, 257, 400, 512, 513, 700])
@pytest.mark.parametrize("refs", [1, 3, 20, 300])
def test_merge_path_edges(ctx, hits, refs):
    """Merges around the limits of their ways (16 and 64 NAMs a strand, 64,
    128, 256 and 512 hits): a strand of hits that each open a NAM, one of hits
    on a few diagonals, and runs of equal query starts, on one and on several
    references and split between the strands in several ways, against the
    oracle."""
    rng = np.random.default_rng(100 * hits + refs)
    ents, reads, used = [], [], set()

    def query(starts, style, rev):
        q = np.zeros(len(starts), dtype=O.QUERY_RANDSTROBE)
        q["start"], q["end"], q["is_reverse"] = starts, starts + rng.integers(20, 60, len(starts)), rev
        for i in range(len(q)):
            h = int(rng.integers(1 << 50, 1 << 63))
            assert h not in used
            used.add(h)
            q["hash"][i] = h
            s = int(starts[i])
            if style == "apart":       # a NAM a hit
                pos = [2_000_000 - 300 * i]
            elif style == "diagonals":  # mostly extended or contained, four diagonals
                pos = [50_000 + s + int(rng.choice([0, 0, 0, 7, 200, 5000]))]
            else:                      # a tandem: several hits of one query start
                pos = sorted(set((70_000 + s + 11 * rng.integers(0, 40, 6)).tolist()))
            for p in pos:
                ents.append((h, p, int(rng.integers(0, refs)) << 8 | int(rng.integers(0, 40))))
        return q

    for style in ("apart", "diagonals", "tandem"):
        per = 5 if style == "tandem" else 1
        for cut in (0, 1, hits // 2, hits):
            n = max(1, hits // per)
            f = min(n, cut // per)
            starts = np.arange(n, dtype=np.int64) * 5
            reads.append(np.concatenate([query(starts[:f], style, 0), query(starts[f:], style, 1)]))
    arr, starts = tiny_index_arrays(ents, 12)
    op = O.params_from_read_length(150)
    oidx = O.Index.wrap(arr, starts, 12, 30, op)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.upload(arr, starts, 12, 30)
    res = G._qrs_call(idx, reads, 0, 0, 1000)
    resc = G._qrs_call(idx, reads, 1, 60, 1000)
    for r, q in enumerate(reads):
        _, exp, _ = O.find_nams(oidx, q, canonical=True)
        assert res.read_nams(r).tobytes() == exp.tobytes(), r
        assert resc.read_nams(r).tobytes() == O.find_nams_rescue(oidx, q, 60, 1000, canonical=True).tobytes(), r
    idx.ctx.close()


@pytest.mark.parametrize("profile", [50, 150, 400])
@pytest.mark.parametrize("lens", [[60_000], [30_000, 20_000, 12_345, 4096], [25_000, 8, 24, 31, 300, 25_000, 1], [45_000, 5000]])
def test_index_build_edges(ctx, profile, lens):
    """One and several contigs, equal sequence at equal positions of several
    contigs, contigs too short for a randstrobe, runs of tied s-mers, N runs,
    lengths off every tile and hashes of thousands of records."""
    rng = np.random.default_rng(len(lens) + profile)
    lens = np.array(lens, dtype=np.uint64)
    g = rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), size=int(lens.sum()))
    at = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    for c in range(len(lens)):
        if lens[c] > 20_000:
            s = g[at[c]:at[c + 1]]
            s[:4000] = g[:4000]
            s[5000:5400] = ord("A")
            s[6000:6600] = np.frombuffer(b"AC" * 300, dtype=np.uint8)
            s[7000:7150] = ord("N")
            s[8000:8100] = np.frombuffer(b"acgtN" * 20, dtype=np.uint8)
            s[-25:] = ord("T")
    if lens[0] == 45_000:
        g[:45_000] = np.resize(g[:11], 45_000)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(profile))
    idx.populate_arrays(g, lens)
    oidx = O.Index.build_arrays(g, lens, O.params_from_read_length(profile), n_threads=4)
    assert idx.randstrobes.tobytes() == oidx.randstrobes.tobytes()
    assert np.array_equal(idx.randstrobe_start_indices, oidx.starts)
    assert idx.filter_cutoff == oidx.filter_cutoff
    idx.ctx.close()


@pytest.mark.parametrize("max_tries", [1, 20, 31, 32, 64])
def test_pair_list_edges(ctx, max_tries):
    """List lengths around the lanes of a row, of a wave and of a pass over a
    pair's cells; many and few proper cells, equal scores, equal entries."""
    rng = np.random.default_rng(max_tries)
    sizes = [0, 1, 2, 3, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 100]
    m1, m2 = [], []
    for a in sizes:
        for b in sizes:
            if (a + b) % 2:
                x, y = _proper_rich_pair(rng, max(a, b, 1))
                x["score"], y["score"] = x["score"] // 30, y["score"] // 30
                x, y = x[:a], y[:b]
            else:
                x, y = rand_list(rng, a, 2), rand_list(rng, b, 2)
            m1.append(x[rng.permutation(len(x))])
            m2.append(y[rng.permutation(len(y))])
    offs, flat = _flatten(m1 + m2)
    n = len(m1)
    _compare(G.pairs_from_nams(ctx, offs, flat, n, max_tries=max_tries),
             O.pairs_batch(offs, flat, n, max_tries=max_tries), offs)


@pytest.mark.parametrize("n", [1, 65_535, 65_536, 131_071, 131_072, 131_073, 400_000, 1_300_000])
def test_lookups_of_any_size(ctx, n):
    """Key counts around the chunks that pageable arrays go through, from and to
    pageable and pinned arrays."""
    rng = np.random.default_rng(n)
    ents = [(h, 10 * i, 5) for i, h in enumerate(rng.integers(1, 2 ** 63, 500).tolist())]
    arr, starts = tiny_index_arrays(ents)
    oidx = O.Index.wrap(arr, starts, 8, 30, O.params_from_read_length(150))
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.upload(arr, starts, 8, 30)
    pool = np.concatenate([arr["hash"], rng.integers(0, 2 ** 64, 500, dtype=np.uint64)])
    exp = np.array([oidx.find(int(k)) for k in pool], dtype=np.uint64)
    at = rng.integers(0, len(pool), n)
    keys = pool[at]
    assert np.array_equal(idx.find_many(keys), exp[at])
    pk, po = G.pinned_copy(keys), G.pinned_empty(n, np.uint64)
    for k, o in ((pk, np.empty(n, np.uint64)), (keys, po), (pk, po)):
        o[:] = 7
        idx.ctx.check(idx.ctx.L.gis_lookup_batch(idx.ctx.h, k.ctypes.data, n, o.ctypes.data))
        assert np.array_equal(o, exp[at])
    idx.ctx.close()


@pytest.mark.parametrize("mode", [G.MODE_PLAIN, G.MODE_FUSED])
def test_launch_bursts(ctx, mode):
    """Large and small batches on streams of their own, launched together and
    again out of step, waited for in any order, against a run alone."""
    g, lens = G.synth_genome(300_000, n_contigs=2, gc=0.45, repeat_fraction=0.05, n_families=5,
                             family_len=(300, 1500), copies=(2, 10), seed=5)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.populate_arrays(g, lens)
    mappers, exp = [], []
    for n in (20_000, 16_384, 700, 16_383):
        s, o, l, _ = G.synth_reads(g, lens, n, lengths=(100, 150), weights=(0.5, 0.5), sub_rate=0.01, seed=n)
        m = G.Mapper(idx, n, int(l.sum()), own_stream=True)
        m.upload(s, o, l)
        m.run(mode=mode)
        mappers.append(m)
        exp.append(m.download().nams.tobytes())
    for order in ([0, 1, 2, 3], [3, 2, 1, 0], [2, 0, 3, 1]):
        for m in mappers:
            m.launch(mode=mode)
        for i in order:
            mappers[i].wait()
            assert mappers[i].download().nams.tobytes() == exp[i]
            mappers[i].launch(mode=mode)
        for i in order:
            mappers[i].wait()
            assert mappers[i].download().nams.tobytes() == exp[i]
    for m in mappers:
        m.close()
    idx.ctx.close()


@pytest.mark.parametrize("at", [0, 16, 4096, 8, 1])
def test_results_inside_pinned_arrays(ctx, at):
    """Offsets, fractions and flags downloaded to places inside pinned arrays,
    aligned and not, with nothing written beside them."""
    g, lens = G.synth_genome(200_000, seed=3)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.populate_arrays(g, lens)
    n = 5001
    s, o, l, _ = G.synth_reads(g, lens, n, seed=4)
    m = G.Mapper(idx, n, int(l.sum()))
    m.upload(s, o, l)
    m.run()
    exp = m.download()
    sizes = {"nam_offsets": 8 * (n + 1), "nonrepetitive_fraction": 4 * n, "flags": n,
             "nams": len(exp.nams) * G.NAM.itemsize}
    buf = {k: G.pinned_empty(at + b + 64, np.uint8) for k, b in sizes.items()}
    for b in buf.values():
        b[:] = 0xA5
    out = G._native.NamOut(nam_capacity=len(exp.nams), **{k: b.ctypes.data + at for k, b in buf.items()})
    idx.ctx.check(idx.ctx.L.gis_batch_download(m.h, ctypes.byref(out)))
    want = {"nam_offsets": exp.nam_offsets, "nonrepetitive_fraction": exp.nonrepetitive_fraction, "flags": exp.flags,
            "nams": exp.nams}
    for k, b in buf.items():
        assert b[at: at + sizes[k]].tobytes() == np.ascontiguousarray(want[k]).tobytes(), k
        assert (b[:at] == 0xA5).all() and (b[at + sizes[k]:] == 0xA5).all(), k
    m.close()
    idx.ctx.close()


def _long_mates(rng, c1, c2, hits1, hits2, ref=0):
    """Two lists on one contig, opposite strands, diagonals inside the insert limit
    or far apart, in any order."""
    out = []
    for n, hits, rc, off in ((c1, hits1, 0, 0), (c2, hits2, 1, 300)):
        x = np.zeros(n, dtype=O.NAM)
        i = np.arange(n)
        x["nam_id"], x["query_start"], x["query_end"] = i, i % 50, 100 + i % 50
        x["ref_start"] = 1000 + rng.integers(0, 3, n) * 100_000 + 40 * i + off
        x["ref_end"], x["n_hits"], x["score"] = x["ref_start"] + 100, hits, 10.0 * np.asarray(hits)
        x["ref_id"], x["is_rc"] = ref, rc
        out.append(x[rng.permutation(n)])
    return out


@pytest.mark.parametrize("max_tries", [1, 20, 31])
@pytest.mark.parametrize("c1,c2", [(1, 200), (200, 1), (63, 64), (64, 65), (65, 63), (70, 70), (130, 129), (300, 90), (90, 700)])
def test_joint_rows_left_at_any_cell(ctx, c1, c2, max_tries):
    """The joint scan leaves a row at the first cell whose hits fall below half the
    best: at its first cell, inside a pass of 64 cells, at its ends, or never."""
    rng = np.random.default_rng(1000 * c1 + c2)
    m1, m2 = [], []
    for kind in range(12):
        h1, h2 = rng.integers(1, 6, c1), rng.integers(1, 6, c2)
        if kind % 4 == 1:  # a few rows above the others
            h1[rng.integers(0, c1, 1 + c1 // 30)] = 200
            h2[rng.integers(0, c2, 1 + c2 // 2)] = 150
        elif kind % 4 == 2:  # a best that ends most rows at once, or at a column
            h1[0], h2[: 1 + int(rng.integers(0, c2))] = 300, 100
        elif kind % 4 == 3:
            h1, h2 = rng.integers(1, 400, c1), rng.integers(1, 400, c2)
        a, b = _long_mates(rng, c1, c2, h1, h2)
        m1.append(a)
        m2.append(b)
    offs, flat = _flatten(m1 + m2)
    _compare(G.pairs_from_nams(ctx, offs, flat, 12, max_tries=max_tries),
             O.pairs_batch(offs, flat, 12, max_tries=max_tries), offs)


def test_joint_time_of_rows_left(ctx):
    """A pair of 1000 x 1000 NAMs whose rows end at their first cell: 0.1 ms beside
    the other steps, where visiting every cell of the rows left took 10 ms."""
    rng = np.random.default_rng(3)
    h1, h2 = np.ones(1000, int), np.ones(1000, int)
    h1[0], h2[:] = 300, 100
    offs, flat = _flatten(_long_mates(rng, 1000, 1000, h1, h2))
    best = {}
    for joint in (True, False) * 4:
        t = time.perf_counter()
        G.pairs_from_nams(ctx, offs, flat, 1, joint=joint)
        best[joint] = min(best.get(joint, 1.0), time.perf_counter() - t)
    assert best[True] - best[False] < 3e-3, best


def test_order_time_of_long_lists(ctx):
    """128 lists of 1000 NAMs are ordered beside each other, as long as one pair's two
    lists (four of them one after the other on a wave: 2.3 times that), 33 to 64 and
    more NAMs beside short ones in their order."""
    rng = np.random.default_rng(4)
    ones = np.ones(1000, int)
    best = {}
    pairs = [_long_mates(rng, 1000, 1000, ones, ones) for _ in range(64)]
    for n in (1, 64) * 4:
        offs, flat = _flatten([a for a, _ in pairs[:n]] + [b for _, b in pairs[:n]])
        t = time.perf_counter()
        G.pairs_from_nams(ctx, offs, flat, n, joint=False)
        best[n] = min(best.get(n, 1.0), time.perf_counter() - t)
    assert best[64] < 1.6 * best[1], best
    for n in (1, 7, 8, 9, 40, 300):
        c = [int(x) for x in rng.choice([0, 1, 16, 31, 32, 33, 63, 64, 65, 128, 129], 2 * n)]
        lists = [_long_mates(rng, max(x, 1), 1, rng.integers(1, 9, max(x, 1)), [1])[0][:x] for x in c]
        offs, flat = _flatten(lists)
        _compare(G.pairs_from_nams(ctx, offs, flat, n, joint=False), O.pairs_batch(offs, flat, n, joint=False), offs)


@pytest.mark.parametrize("n,max_tries", [(1, 256), (3000, 1), (3000, 40), (3000, 256), (72_500, 256), (75_000, 256)])
def test_joint_entries_placed_by_any_bound(ctx, n, max_tries):
    """The pairs' places come from the smaller of two bounds linear in their lists'
    lengths, and from their exact bounds where that is more than 2^25 entries (the
    last case; the one before it just is not)."""
    rng = np.random.default_rng(5)
    sizes = [0, 1, 2, 5, 17, 33, 70]
    some = [_long_mates(rng, max(a, 1), max(b, 1), rng.integers(1, 9, max(a, 1)), rng.integers(1, 9, max(b, 1)))
            for a in sizes for b in sizes]
    some = [(x[:a], y[:b]) for (x, y), a, b in zip(some, np.repeat(sizes, 7), np.tile(sizes, 7))]
    if n == 3000:  # mostly short lists
        some += [some[8]] * 100
    reps = -(-n // len(some))
    lists = ([x for x, _ in some] * reps)[:n] + ([y for _, y in some] * reps)[:n]
    offs, flat = _flatten(lists)
    linear = len(flat) + min(int(len(flat) * np.sqrt(2 * max_tries + 1) / 2), n * (2 * max_tries + 1))
    assert (linear > 2 ** 25) == (n == 75_000) and (n < 72_500 or abs(linear / 2 ** 25 - 1) < 0.03)
    _compare(G.pairs_from_nams(ctx, offs, flat, n, max_tries=max_tries), O.pairs_batch(offs, flat, n, max_tries=max_tries),
             offs)


@pytest.mark.parametrize("n", [2, 16, 17, 32, 33, 64, 65, 128, 129, 300])
def test_equal_nams_are_refused_in_lists_of_any_length(ctx, n):
    rng = np.random.default_rng(n)
    a, b = _long_mates(rng, n, 3, rng.integers(1, 9, n), rng.integers(1, 9, 3))
    for i, j in {(0, 1), (0, n - 1), (n // 2, n // 2 - 1)}:
        x = a.copy()
        x[i] = x[j]
        if i == j:
            continue
        for lists in ([x, b], [b, x]):
            offs, flat = _flatten(lists)
            with pytest.raises(G.GisError):
                G.pairs_from_nams(ctx, offs, flat, 1, joint=False)
        offs, flat = _flatten([a, b])
        _compare(G.pairs_from_nams(ctx, offs, flat, 1, joint=False), O.pairs_batch(offs, flat, 1, joint=False), offs)


def test_pair_results_are_of_the_last_run(ctx):
    """A pair step's results can be read until other reads are run, or the same ones with
    other cutoffs; reads run again as they were have the same NAMs."""
    g, lens = G.synth_genome(200_000, n_contigs=2, gc=0.45, repeat_fraction=0.5, n_families=12,
                             family_len=(400, 1500), copies=(2, 40), divergence=(0.0, 0.005), seed=3)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.populate_arrays(g, lens)
    s, o, l, _ = G.synth_reads(g, lens, 3000, lengths=(100, 150), weights=(1, 1), sub_rate=0.01, seed=4)
    m = G.Mapper(idx, 20, 20 * 150)
    m.upload(s, o[:20], l[:20])
    m.run()
    want = m.pairs()
    m.run()
    m.run(mode=G.MODE_FUSED)
    again = m.pairs_download()
    assert again.nams.tobytes() == want.nams.tobytes() and np.array_equal(again.nam_offsets, want.nam_offsets)
    m.run(rescue_level=100, hard_cutoff=5)
    with pytest.raises(G.GisError):
        m.pairs_download()
    m.run()
    assert m.pairs_download().nams.tobytes() == want.nams.tobytes()
    m2 = G.Mapper(idx, 20, 20 * 150, share=m)
    m.upload(s, o, l)  # (the batch's arrays grow with the run)
    m.run()
    with pytest.raises(G.GisError):
        m.pairs_download()
    assert len(m.pairs().types) == 1500
    # another batch of the workspace between
    m2.upload(s, o[:20], l[:20])
    m2.run()
    with pytest.raises(G.GisError):
        m.pairs_download()
    assert m2.pairs().nams.tobytes() == want.nams.tobytes()
    m.run()
    with pytest.raises(G.GisError):
        m2.pairs_download()
    m2.run()
    assert m2.pairs_download().nams.tobytes() == want.nams.tobytes()
    for x in (m2, m):
        x.close()
    idx.ctx.close()
