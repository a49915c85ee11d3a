"""Scoring of the MFMA kernels' work units: the sets at the edges of a 3-way
unit (tiles 3, 4 and 5: X pairs, 32 Y, 32 Z) and of a 2-way one, classes of one
and several chunks, and the top-k bound that the kernels tighten from their own
candidates.  Winners, rankings and FP64 scores are the oracle's, bit for bit."""
import math

import pytest

import episdet
import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(3, 1, 1), (4, 31, 1100), (33, 1024, 1025), (64, 700, 3000), (65, 2049, 2048), (98, 40, 25)]


@pytest.mark.parametrize("n,Nc,Nt", SIZES)
@pytest.mark.parametrize("score", [episdet.K2, episdet.MI])
def test_unit_edges(n, Nc, Nt, score):
    syn = episdet.generate(n, Nc, Nt, seed=300 + n, planted_sets=1 if n >= 64 else 0)
    ref_p, ref_s = O.ranked(syn.cases, syn.controls, Nc, Nt, 3, score)
    with episdet.Dataset.from_synthetic(syn) as ds:
        for tile in (3, 4, 5):
            print(f"edges n={n} Nc={Nc} Nt={Nt} score={score} tile={tile}", flush=True)
            r = ds.run(3, score, path=episdet.PATH_FUSED_MFMA, tile=tile)
            assert r["packed"] == int(ref_p[0]) and r["best_score"] == float(ref_s[0])
            for k in (2, 65, 1024):
                p, s, _ = ds.topk(3, k, score=score, path=episdet.PATH_FUSED_MFMA, tile=tile)
                m = min(k, math.comb(n, 3))
                assert p == [int(x) for x in ref_p[:m]] and s == [float(x) for x in ref_s[:m]]


@pytest.mark.parametrize("n,Nc,Nt", [(2, 1, 1), (63, 40, 25), (64, 1024, 1025), (65, 3000, 31), (130, 700, 2049),
                                     (1030, 600, 500)])
@pytest.mark.parametrize("score", [episdet.K2, episdet.MI])
def test_pair_unit_edges(n, Nc, Nt, score):
    """The 2-way kernel's 64 x 64 units (MFMA tile 1), in triangular order and
    (from 16 tiles up) in XCD blocks."""
    syn = episdet.generate(n, Nc, Nt, seed=400 + n, planted_sets=1 if n >= 64 else 0, planted_order=2)
    ref_p, ref_s = O.ranked(syn.cases, syn.controls, Nc, Nt, 2, score)
    with episdet.Dataset.from_synthetic(syn) as ds:
        print(f"pair edges n={n} Nc={Nc} Nt={Nt} score={score}", flush=True)
        r = ds.run(2, score, path=episdet.PATH_FUSED_MFMA, tile=1)
        assert r["packed"] == int(ref_p[0]) and r["best_score"] == float(ref_s[0])
        for k in (2, 65, 1024):
            p, s, _ = ds.topk(2, k, score=score, path=episdet.PATH_FUSED_MFMA, tile=1)
            m = min(k, math.comb(n, 2))
            assert p == [int(x) for x in ref_p[:m]] and s == [float(x) for x in ref_s[:m]]


@pytest.mark.parametrize("score", [episdet.K2, episdet.MI])
def test_batch_seeds_every_three_way_job(score):
    """The 3-way jobs of a batch are seeded in grids sized for the largest one:
    one triplet (not seeded), the smallest seeded job, larger ones with 2-way jobs
    between, and more SNPs than the pair ranking has workgroups (1024)."""
    sizes = [(3, 3, 40), (2, 90, 700), (3, 4, 1030), (3, 65, 900), (2, 5, 64), (3, 130, 300)]
    syns = [episdet.generate(n, N // 3, N - N // 3, seed=500 + j, planted_sets=int(n >= 64), planted_order=o)
            for j, (o, n, N) in enumerate(sizes)]
    ref = [O.search(s.cases, s.controls, s.num_cases, s.num_controls, o, score) for (o, _, _), s in zip(sizes, syns)]
    # too many triplets for the oracle: the search without a starting bound is the reference
    sizes.append((3, 1030, 200))
    syns.append(episdet.generate(1030, 90, 110, seed=550))
    dss = [episdet.Dataset.from_synthetic(s) for s in syns]
    r = dss[-1].run_noalloc(3, score)
    ref.append({"packed": r["packed"], "score": r["best_score"]})
    for rep in range(3):
        print(f"batch score={score} rep={rep}", flush=True)
        res, _ = episdet.run_batch(dss, [o for o, _, _ in sizes], [score] * len(sizes), rebuild=rep == 1)
        assert [x["seeded"] for x in res] == [int(o == 3 and n > 3) for o, n, _ in sizes]
        for x, o in zip(res, ref):
            assert x["packed"] == o["packed"] and x["best_score"] == o["score"]
    for d in dss:
        d.close()


@pytest.mark.parametrize("n,Nc,Nt", [(2, 1, 1), (16, 40, 25), (17, 1024, 1025), (432, 700, 300), (433, 300, 700)])
@pytest.mark.parametrize("score", [episdet.K2, episdet.MI])
def test_small_valu_pair_units(n, Nc, Nt, score):
    """VALU pair tile 1 takes 16 x 16 units up to 432 SNPs (256 CUs) and 32 x 32
    units beyond and for top-k; candidate_cap 64 forces windows of units."""
    syn = episdet.generate(n, Nc, Nt, seed=600 + n, planted_sets=int(n >= 64), planted_order=2)
    ref_p, ref_s = O.ranked(syn.cases, syn.controls, Nc, Nt, 2, score)
    V = episdet.PATH_FUSED_VALU
    with episdet.Dataset.from_synthetic(syn) as ds:
        print(f"valu pair units n={n} Nc={Nc} Nt={Nt} score={score}", flush=True)
        for r in (ds.run(2, score, path=V, tile=1), ds.run(2, score, path=V, tile=1, candidate_cap=64),
                  ds.run_noalloc(2, score, path=V, tile=1)):
            assert r["packed"] == int(ref_p[0]) and r["best_score"] == float(ref_s[0]) and r["tile"] == 1
        m = min(1024, math.comb(n, 2))
        p, s, _ = ds.topk(2, 1024, score=score, path=V, tile=1)
        assert p == [int(x) for x in ref_p[:m]] and s == [float(x) for x in ref_s[:m]]


def test_upload_through_the_pinned_pool():
    """Planes of 4 MB and more a class go to the device in chunks of whole SNPs
    (239 of them here); the rows on both sides of a chunk's edge, the caller's
    own padding and the last rows arrive whole."""
    n, Nc, Nt, words = 300, 70001, 69000, 2190
    syn = episdet.generate(n, Nc, Nt, seed=77, cases_words=words, controls_words=words, planted_sets=1,
                           planted_order=2)
    sets = [(0, 238), (238, 239), (239, 240), (1, 299), (237, 298)]
    with episdet.Dataset.from_synthetic(syn) as ds:
        t = ds.tables(2, sets)
        for i, s in enumerate(sets):
            assert (t[i, 0] == O.table_bits(syn.cases, Nc, s)).all() and (t[i, 1] == O.table_bits(syn.controls, Nt, s)).all()
        for score in (episdet.K2, episdet.MI):
            r, o = ds.run(2, score), O.search(syn.cases, syn.controls, Nc, Nt, 2, score)
            assert r["packed"] == o["packed"] and r["best_score"] == o["score"]
