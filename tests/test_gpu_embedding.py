"""The owner's token-embedding gradient on the GPU, against torch's own aten.embedding_dense_backward on the same
device (the routine the reference calls, yoco/models/decoder/layer_graphs.py:92, ce_reduce.py:230) and against the
oracle.  aten takes its sort-based path for more than 3072 indices and another kernel for fewer; this build follows
the order of each (bit-exact)."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def zipf_ids(rng, R, V, a=1.2):
    ids = rng.zipf(a, R) - 1
    return np.where(ids < V, ids, rng.integers(0, V, R)).astype(np.int64)


def bits(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.mark.parametrize('padding_idx', [-1, 1])
@pytest.mark.parametrize('D', [3072, 200])
def test_matches_aten_sort_path(pkg, dev, padding_idx, D):
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(D + padding_idx)
    R, V = 8 * 2048, 100288
    ids = torch.from_numpy(zipf_ids(rng, R, V)).to(dev)
    assert int((ids == 0).sum()) > 100                       # long runs: many partials of 10
    g = (torch.randn(R, D, device=dev) * 1e-2).to(torch.bfloat16)
    ref = torch.ops.aten.embedding_dense_backward(g, ids, V, padding_idx, False)
    got = embedding.embedding_dense_backward(g, ids, V, padding_idx)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got), bits(ref))
    # the reference's two 1/world placements
    ref2 = torch.ops.aten.embedding_dense_backward(g, ids, V, padding_idx, False).mul_(1.0 / 8)
    got2 = embedding.owner_embedding_grad(g, ids, V, padding_idx, 8)
    ref3 = torch.ops.aten.embedding_dense_backward(g.clone().mul_(1.0 / 8), ids, V, padding_idx, False)
    got3 = embedding.ce_owner_embedding_grad(g, ids, V, padding_idx, 8)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got2), bits(ref2)) and np.array_equal(bits(got3), bits(ref3))


@pytest.mark.parametrize('R', [65536, 1_500_000])
def test_matches_aten_at_larger_row_counts(pkg, dev, R):
    """More rows than the recipe's 16,384: the sort runs rocPRIM's other algorithms (merge sort up to 1M items,
    onesweep above); still bit-exact against aten."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(R)
    V, D = 100288, 64
    ids = torch.from_numpy(zipf_ids(rng, R, V)).to(dev)
    g = (torch.randn(R, D, device=dev) * 1e-2).to(torch.bfloat16)
    ref = torch.ops.aten.embedding_dense_backward(g, ids, V, -1, False)
    got = embedding.embedding_dense_backward(g, ids, V, -1)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got), bits(ref))


@pytest.mark.parametrize('D', [3072, 40, 13])
def test_heavy_ids_at_the_run_boundaries(pkg, dev, D):
    """Ids with 20 occurrences (the rows kernel's most), 21 (the heavy passes' fewest), 30, 31, 320 (the most one
    wave chains: 32 runs), 321 and 9,878; 400 ids
    with exactly 21 each, which fill every run slot the workspace holds (R / 7); one id taking every row.  Against
    aten's sort path (more than 3072 rows in every case), on the vector path with several and with one partial
    column group, and on the element path."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(D)
    V = 5000
    mix = np.concatenate([np.full(c, t) for t, c in ((7, 20), (8, 21), (9, 30), (10, 31), (11, 9878), (12, 1),
                                                     (13, 320), (14, 321))] + [rng.integers(15, V, 3000)])
    cases = [rng.permutation(mix), rng.permutation(np.repeat(np.arange(100, 500), 21)), np.full(16384, 4)]
    for ids in cases:
        ids = torch.from_numpy(ids.astype(np.int64)).to(dev)
        R = ids.numel()
        g = (torch.randn(R, D, device=dev) * 1e-2).to(torch.bfloat16)
        for pad in (-1, 8):
            ref = torch.ops.aten.embedding_dense_backward(g, ids, V, pad, False)
            got = embedding.embedding_dense_backward(g, ids, V, pad)
            torch.cuda.synchronize()
            assert np.array_equal(bits(got), bits(ref)), (R, pad)


@pytest.mark.parametrize('D', [3072, 40, 13])
def test_matches_aten_at_3072_rows_or_fewer(pkg, dev, D):
    """At most 3072 rows: aten's kernel for few indices, whose order (chunks of 16 indices, each chunk's sum rounded to
    bf16 and added to the bf16 row) this build follows there.  Bit-exact against torch's aten for 1 row, for chunk
    boundaries (15, 16, 17 rows), and up to 3072 rows with heavy repeats, padding and both 1/world placements."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(100 + D)
    for R, V in ((1, 5), (15, 3), (16, 3), (17, 3), (1000, 7), (2048, 300), (3072, 40), (3072, 100288)):
        ids = torch.from_numpy(rng.integers(0, V, R).astype(np.int64)).to(dev)
        g = (torch.randn(R, D, device=dev) * 1e-2).to(torch.bfloat16)
        for pad in (-1, 2):
            ref = torch.ops.aten.embedding_dense_backward(g, ids, V, pad, False)
            got = embedding.embedding_dense_backward(g, ids, V, pad)
            torch.cuda.synchronize()
            assert np.array_equal(bits(got), bits(ref)), (R, V, pad)
        ref2 = torch.ops.aten.embedding_dense_backward(g, ids, V, -1, False).mul_(1.0 / 8)
        ref3 = torch.ops.aten.embedding_dense_backward(g.clone().mul_(1.0 / 8), ids, V, -1, False)
        got2 = embedding.owner_embedding_grad(g, ids, V, -1, 8)
        got3 = embedding.ce_owner_embedding_grad(g, ids, V, -1, 8)
        torch.cuda.synchronize()
        assert np.array_equal(bits(got2), bits(ref2)) and np.array_equal(bits(got3), bits(ref3)), R


@pytest.mark.parametrize('V', [1023, 1024, 1025, 2049])
@pytest.mark.parametrize('few', [True, False])
@pytest.mark.parametrize('D', [3080, 520, 5])
def test_occurrence_counts(pkg, dev, D, few, V):
    """Ids with as many occurrences as the parts of the work split at -- 4 and 5 (the row's own wave / by runs), 10 and 11
    (one run / several), 32 and 33, 320 and 321 (chained by a wave / a workgroup), 1200 -- ids at both ends of tables
    around a multiple of the rows one round of XCDs takes, an output off the 16-byte boundary, a heavy padding row.
    Bit-exact against aten."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(D + V)
    counts = [1, 2, 3, 4, 5, 9, 10, 11, 12, 16, 17, 20, 21, 30, 31, 32, 33, 64, 65, 320, 321, 1200]
    where = rng.choice(np.arange(1, V - 1), len(counts), replace=False)
    ids = np.concatenate([np.repeat(where, counts), [0, V - 1, V - 1], rng.integers(0, V, 0 if few else 2000)])
    ids = torch.from_numpy(rng.permutation(ids).astype(np.int64)).to(dev)
    assert (ids.numel() <= 3072) == few
    g = (torch.randn(ids.numel(), D, device=dev) * 1e-2).to(torch.bfloat16)
    for pad in (-1, int(where[-1]), 0):
        ref = torch.ops.aten.embedding_dense_backward(g, ids, V, pad, False)
        out = torch.full((V * D + 1,), 7.0, dtype=torch.bfloat16, device=dev)[pad % 2:][:V * D].view(V, D)
        embedding.embedding_dense_backward(g, ids, V, pad, out=out)
        torch.cuda.synchronize()
        assert np.array_equal(bits(out), bits(ref)), pad


# the bounds of a dense table: 2 indices per row, 16,384 indices
@pytest.mark.parametrize('R,V', [(16383, 700), (16384, 700), (16384, 8192), (16384, 8193), (40000, 1500), (60000, 30000)])
@pytest.mark.parametrize('D', [5, 520, 3083])
def test_dense_tables(pkg, dev, R, V, D):
    """Tables of many indices per row, where the wave of a row sums up to 20 occurrences: ids with as many as the parts of
    the work split at, ids at both ends, an output off the 16-byte boundary, a heavy and a light padding row, all three
    placements of the scale.  Bit-exact against aten."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(R + V + D)
    counts = [1, 2, 4, 5, 9, 10, 11, 19, 20, 21, 30, 31, 320, 321]
    where = rng.choice(np.arange(1, V - 1), len(counts), replace=False)
    rest = np.setdiff1d(np.arange(V), where)
    ids = np.concatenate([np.repeat(where, counts), rng.choice(rest, R - sum(counts))])
    ids = torch.from_numpy(rng.permutation(ids).astype(np.int64)).to(dev)
    g = (torch.randn(R, D, device=dev) * 1e-2).to(torch.bfloat16)
    aten = torch.ops.aten.embedding_dense_backward
    for pad in (-1, int(where[-1]), int(where[8])):
        ref = aten(g, ids, V, pad, False)
        out = torch.full((V * D + 1,), 7.0, dtype=torch.bfloat16, device=dev)[pad % 2:][:V * D].view(V, D)
        embedding.embedding_dense_backward(g, ids, V, pad, out=out)
        torch.cuda.synchronize()
        assert np.array_equal(bits(out), bits(ref)), pad
    got, got_ce = (f(g, ids, V, 1, 8) for f in (embedding.owner_embedding_grad, embedding.ce_owner_embedding_grad))
    ref, ref_ce = aten(g, ids, V, 1, False) * 0.125, aten(g * 0.125, ids, V, 1, False)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got), bits(ref)) and np.array_equal(bits(got_ce), bits(ref_ce))


@pytest.mark.parametrize('V', [2 ** 25, 2 ** 25 + 1, 2 ** 26 + 2000])
def test_more_rows_than_one_round_of_waves(pkg, dev, V):
    """Tables of 2^25 rows (the most one launch has waves for) and more, past the former limit of one grid as well:
    bit-exact against aten."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(V)
    ids = np.concatenate([rng.integers(0, V, 500), [0, V - 1, 2 ** 25 - 1, V - 1], np.full(40, V - 2)])
    ids = torch.from_numpy(ids.astype(np.int64)).to(dev)
    g = (torch.randn(ids.numel(), 2, device=dev) * 1e-2).to(torch.bfloat16)
    ref = torch.ops.aten.embedding_dense_backward(g, ids, V, -1, False)
    out = torch.full((V, 2), 7.0, dtype=torch.bfloat16, device=dev)
    embedding.embedding_dense_backward(g, ids, V, -1, out=out)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize('R', [1, 63, 1024, 1025, 16384, 16385, 20000, 49152, 49153])
@pytest.mark.parametrize('V', [1, 2, 513, 65537, 524288, 524289])
def test_order_of_occurrences(pkg, dev, R, V):
    """Row counts and vocabularies at the edges of the one-launch ordering (a wave's 64 positions, one register tile of
    16 x 1024 ids, its largest R and V and one beyond, where the library sort takes over): bit-exact against aten, with
    skewed ids, the first and last id and (mapped to padding for aten) ids outside the vocabulary."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(R * 7 + V)
    ids = zipf_ids(rng, R, V, 1.3)
    ids[rng.integers(0, R, R // 3)] = rng.integers(0, V, R // 3)
    ids[0] = V - 1
    bad = rng.integers(0, R, R // 50)
    D = 8 if V > 100000 else 24
    g = (torch.randn(R, D, device=dev) * 1e-2).to(torch.bfloat16)
    ours = ids.copy()
    ours[bad] = rng.choice([-1, V, V + 3, 2 ** 31 - 1, 2 ** 40], bad.size)
    theirs = ids.copy()
    theirs[bad] = V
    ref = torch.ops.aten.embedding_dense_backward(g, torch.from_numpy(theirs).to(dev), V + 1, V, False)[:V]
    got = embedding.embedding_dense_backward(g, torch.from_numpy(ours).to(dev), V, -1)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got), bits(ref))


@pytest.mark.parametrize('R', [262144, 262145])
@pytest.mark.parametrize('V', [1, 255, 256, 257, 70001])
def test_places_of_the_library_sort(pkg, dev, R, V):
    """Either side of the largest row count whose places are found in one launch, vocabularies at the edge of a workgroup:
    skewed ids, the last id among them, and ids outside the vocabulary.  Bit-exact against aten."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(R + V)
    ids = zipf_ids(rng, R, V, 1.3)
    ids[rng.integers(0, R, R // 3)] = rng.integers(0, V, R // 3)
    ids[0] = V - 1
    g = (torch.randn(R, 24, device=dev) * 1e-2).to(torch.bfloat16)
    ours, theirs = ids.copy(), ids.copy()
    bad = rng.integers(1, R, R // 50)
    ours[bad] = rng.choice([-1, V, V + 3, 2 ** 31 - 1, 2 ** 40], bad.size)
    theirs[bad] = V
    ref = torch.ops.aten.embedding_dense_backward(g, torch.from_numpy(theirs).to(dev), V + 1, V, False)[:V]
    got = embedding.embedding_dense_backward(g, torch.from_numpy(ours).to(dev), V, -1)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got), bits(ref))


@pytest.mark.parametrize('step', [2, 256, 512, 514, 1024, 4096])
@pytest.mark.parametrize('V', [1000, 65536, 100288, 524288])
def test_ids_a_step_apart(pkg, dev, V, step):
    """Multiples of a step, which the one-launch ordering spreads over its buckets by turning each round of them: bit-exact
    against aten, an id next to each among them."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(V + step)
    ids = rng.integers(0, V, 6000) // step * step
    ids[::97] = np.minimum(ids[::97] + 1, V - 1)
    ids = torch.from_numpy(ids.astype(np.int64)).to(dev)
    g = (torch.randn(6000, 16, device=dev) * 1e-2).to(torch.bfloat16)
    ref = torch.ops.aten.embedding_dense_backward(g, ids, V, -1, False)
    got = embedding.embedding_dense_backward(g, ids, V, -1)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got), bits(ref))


@pytest.mark.parametrize('R', [700, 4000])
@pytest.mark.parametrize('D', [1, 7, 8, 9, 511, 512, 513, 1027, 1536, 2563, 3079, 4104, 6151])
def test_row_widths(pkg, dev, R, D):
    """Widths at the edges of a lane's column groups (8 columns, 64 lanes, up to 6 groups a step, several steps) and
    rows at odd addresses, in both summation orders: bit-exact against aten, rows of -0.0 included."""
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(D)
    V = 900
    ids = torch.from_numpy(np.concatenate([rng.integers(0, V, R - 300), rng.integers(0, 9, 300)])).to(dev)
    g = (torch.randn(R, D, device=dev) * 1e-2).to(torch.bfloat16)
    g[::5] = -0.0
    ref = torch.ops.aten.embedding_dense_backward(g, ids, V, 3, False)
    got = embedding.embedding_dense_backward(g, ids, V, 3)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got), bits(ref))


@pytest.mark.parametrize('few', [True, False])
def test_every_bf16_value(pkg, dev, few):
    """All 65,536 bf16 patterns (every NaN, infinities, denormals, both zeros) as an id's first occurrence, alone and
    before 3, 4, 10 and 40 others (the row's own wave, one run, several, a long chain), in the three placements of the
    scale: the bits of aten and aten's multiplication, whose NaN is 0x7fc0."""
    from faster_yoco_amd import embedding
    counts, D = [1, 4, 5, 11, 41], 16384
    pattern = torch.arange(-2 ** 15, 2 ** 15, device=dev).to(torch.int16).view(torch.bfloat16).view(4, D)
    for n in counts:
        g = (torch.randn(4 * n + (0 if few else 3100), D, device=dev) * 1e-2).to(torch.bfloat16)
        g[:4] = pattern
        ids = torch.full((g.shape[0],), 9, device=dev)
        ids[:4 * n] = torch.arange(4 * n, device=dev) % 4
        aten = torch.ops.aten.embedding_dense_backward
        ref, ref_ce = aten(g, ids, 10, 9, False), aten(g * 0.125, ids, 10, 9, False)
        got = embedding.embedding_dense_backward(g, ids, 10, 9)
        got_owner = embedding.owner_embedding_grad(g, ids, 10, 9, 8)
        got_ce = embedding.ce_owner_embedding_grad(g, ids, 10, 9, 8)
        torch.cuda.synchronize()
        for a, b in ((got, ref), (got_owner, ref * 0.125), (got_ce, ref_ce)):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16)), n


def test_matches_oracle_and_edge_cases(pkg, dev):
    from faster_yoco_amd import embedding
    rng = np.random.default_rng(3)
    R, V, D = 4000, 300, 13                                   # D % 8 != 0: the element path
    ids = zipf_ids(rng, R, V, 1.5)
    ids[:4] = [-5, V, V + 7, 2 ** 40]                         # outside [0, V): contribute nothing
    g16 = oracle.bf16_rne((rng.standard_normal((R, D)) * 1e-2).astype(np.float32))
    for pad, scale, first in ((-1, None, False), (3, 0.125, False), (0, 0.125, True)):
        exp = oracle.embedding_backward(ids, g16, V, padding_idx=pad, scale=scale, scale_first=first)
        gt = torch.from_numpy(g16.view(np.int16)).to(dev).view(torch.bfloat16)
        got = embedding.embedding_dense_backward(gt, torch.from_numpy(ids).to(dev), V, pad, scale=scale,
                                                 scale_first=first)
        torch.cuda.synchronize()
        assert np.array_equal(bits(got), exp)
    # no rows at all: a zero table; a preexisting out buffer is fully overwritten
    out = torch.full((V, 16), 7.0, dtype=torch.bfloat16, device=dev)
    embedding.embedding_dense_backward(torch.zeros(0, 16, dtype=torch.bfloat16, device=dev),
                                       torch.zeros(0, dtype=torch.int64, device=dev), V, -1, out=out)
    torch.cuda.synchronize()
    assert not out.float().abs().sum().item()
    with pytest.raises(RuntimeError, match='scale_grad_by_freq'):
        embedding.embedding_dense_backward(gt, torch.from_numpy(ids).to(dev), V, -1, True)


def test_aten_few_indices_order_known_answer(pkg, dev):
    """Guard of the bit-exact claim for at most 3072 rows, whose order follows torch's own ROCm aten kernel (chunks
    of 16 indices, each chunk's fp32 sum rounded to bf16 before it is added to the row).  On one id, rows 1.0, 2^-9,
    fourteen zeros, 2^-8: chunks of 16 give 0x3F80; one chunk of 32, or the sort path, 0x3F81.  If a torch build
    walks the indices otherwise, this fails here, loudly, instead of the bf16 copies drifting in their last bit."""
    from faster_yoco_amd import embedding
    vals = [1.0, 2.0 ** -9] + [0.0] * 14 + [2.0 ** -8]
    g = torch.tensor(vals, dtype=torch.float32).reshape(-1, 1).to(torch.bfloat16).to(dev)
    ids = torch.zeros(len(vals), dtype=torch.int64, device=dev)
    aten = torch.ops.aten.embedding_dense_backward(g, ids, 1, -1, False)
    ours = embedding.embedding_dense_backward(g, ids, 1, -1)
    torch.cuda.synchronize()
    assert int(aten.view(torch.int16).item()) & 0xFFFF == 0x3F80, 'torch\'s few-indices order changed'
    assert int(ours.view(torch.int16).item()) & 0xFFFF == 0x3F80
