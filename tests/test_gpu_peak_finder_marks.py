"""The peak finder in one and in two steps, and by the rule between them, bit for bit against the
kernel that also forms the float64 variances, which visits every candidate in order in one time
segment: where values leave the range in which the two-step kernel's first step is exact, and
over bin lengths, boxcar lengths, multiplets and chunks that the time segments do not divide."""

import numpy as np
import pytest

from gpu_cases import BASE, pt
from gpu_harness import random_weights

pytestmark = pytest.mark.gpu


def make_all(rank, bands, widths, dtype, B, T, time_ds=0):
    """The same search with the two-step kernel (where there is one), with one step, by the rule
    between the two, and with the one that forms variances."""
    import pirate_amd as pa
    trees = [dict(pt(0, w, min(64, 2**(rank - 1)), min(64, (T >> p) & -(T >> p))), time_downsampling=time_ds)
             for p, w in enumerate(widths)]
    cfg = dict(BASE, dtype=dtype, zone_nfreq=[2**rank], zone_freq_edges=[400, 800], toplevel_tree_rank=rank,
               time_samples_per_chunk=T, beams_per_gpu=B, beams_per_batch=B, num_active_batches=1,
               frequency_subband_counts=bands, primary_trees=trees)
    plan = pa.DedispersionPlan(pa.DedispersionConfig.from_dict(cfg))
    dds = [pa.GpuDedisperser(plan, enable_variances=v) for v in (False, False, False, True)]
    rng = np.random.default_rng(rank)
    for dd, two_step in zip(dds, (1, 0, -1, -1)):
        dd.allocate()
        dd.set_tuning('pf_two_step', two_step)
    for it in range(plan.ntrees):
        w = random_weights(rng, dds[0], it)
        for dd in dds:
            dd.fill_all_weights(it, w)
    return plan, dds


def outputs(plan, dds, c, x):
    """Bit patterns of (out_max, out_argmax) and values of every tree, for each of the dedispersers."""
    import torch
    x = torch.from_numpy(x).cuda()
    bits = torch.int32 if plan.dtype == 'float32' else torch.int16
    res = []
    for dd in dds:
        with dd.get_input(c) as arr:
            arr.copy_(x)
        with dd.get_output(c) as out:
            res.append([(m.view(bits).cpu().numpy(), a.cpu().numpy(), m.float().cpu().numpy())
                        for m, a in zip(out.out_max, out.out_argmax)])
    return res


def assert_equal(plan, res, c):
    for it in range(plan.ntrees):
        for i, what in enumerate(('out_max', 'out_argmax')):
            b = res[-1][it][i]
            for a, name in zip((r[it][i] for r in res[:-1]), ('two steps', 'one step', 'rule')):
                assert np.array_equal(a, b), f'{name}: chunk {c} tree {it} {what}: {int(np.sum(a != b))} of {a.size} differ'


# bins of 16, 8 and 16 samples; 16, 34 and 91 multiplets
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('rank,bands', [(13, [0, 0, 0, 0, 1]), (11, [4, 5, 3, 1]), (14, [5, 9, 7, 3, 1])])
def test_sums_that_overflow(rank, bands, dtype):
    """Pairs of neighbouring samples of -1.72e38 at zero DM on a small positive background, each pair
    on both sides of a bin's start: their sum is -inf, while all sums on the boxcar levels' grids (and of the
    other multiplets, which smear a pair over more samples) are finite. Such a sum is then the first candidate of its level, and times a zero weight NaN: the level
    is out for this bin and stream, whatever its later candidates are. Weights are zero but for the second and
    third profile of one level."""
    B, T = 2, 512
    print(f'[peak finder marks] overflow rank {rank} {bands} {dtype}', flush=True)
    plan, dds = make_all(rank, bands, [16], dtype, B, T)
    bin_len = T // plan.trees[0].nt_out
    rng = np.random.default_rng(1)
    w = np.zeros(dds[0].wt_shape(0), dtype=np.float32)          # (slots, B, ndm_wt, nt_wt, P, N)
    lev = rng.integers(1, 4, size=w.shape[:4] + w.shape[5:])
    for l in (1, 2, 3):
        for p in (3 * l + 2, 3 * l + 3):
            w[:, :, :, :, p, :] = (lev == l) * rng.uniform(0.5, 1, size=lev.shape)
    for dd in dds:
        dd.fill_all_weights(0, w)
    for c in range(3):
        v = 1e30 * (1 + 0.3 * rng.standard_normal((B, plan.nfreq, T)))
        for b in range(B):
            for k in rng.choice(np.arange(1, T // bin_len), T // bin_len // 3, replace=False):
                v[b, :, k * bin_len - 1:k * bin_len + 1] = -1.72e38
        x = (v * 2.0 ** (-rank / 2)).astype(np.float32)
        res = outputs(plan, dds, c, x)
        assert_equal(plan, res, c)


# (rank, subband counts, boxcars, chunk, beams): 1 to 63 tiles per chunk, launches on both sides of the rule
SEGMENTS = [
    (4, [1], [32], 1984, 3), (8, [1], [16, 4], 1408, 1), (8, [2, 2, 1], [32], 4032, 2), (10, [1], [2], 320, 4),
    (10, [3, 3, 1], [16, 8], 1408, 1), (12, [1], [32, 1], 2944, 1), (14, [1], [16], 64, 1), (14, [1], [8], 1984, 1),
]


@pytest.mark.parametrize('dtype', ['float32', 'float16'])
@pytest.mark.parametrize('rank,bands,widths,T,B', SEGMENTS)
def test_segments(rank, bands, widths, T, B, dtype):
    print(f'[peak finder marks] segments rank {rank} {bands} {widths} T {T} B {B} {dtype}', flush=True)
    plan, dds = make_all(rank, bands, widths, dtype, B, T)
    rng = np.random.default_rng(2)
    for c in range(3):
        res = outputs(plan, dds, c, rng.standard_normal((B, plan.nfreq, T)).astype(np.float32))
        assert_equal(plan, res, c)


# (rank, subband counts, boxcars, output bin or 0): 2 to 91 multiplets, bins of 1 to 32 samples
SHAPES = {
    'm4_bins1': (8, [1], [32], 1), 'm2_bins2': (4, [1], [16], 2), 'm10_bins4': (8, [2, 2, 1], [16, 4], 0),
    'm8_bins8': (10, [1], [32, 2], 0), 'm34_bins8': (11, [4, 5, 3, 1], [8, 32], 0), 'm16_bins16': (13, [0, 0, 0, 0, 1], [16, 8], 0),
    'm91_bins16': (14, [5, 9, 7, 3, 1], [16], 0), 'm8_bins32': (10, [1], [16], 32),
}


@pytest.mark.parametrize('dtype', ['float32', 'float16', 'bfloat16'])
@pytest.mark.parametrize('name', list(SHAPES))
def test_sparse_marks(name, dtype):
    """Three infinities or NaN per beam and chunk, so that marked and clean bins and streams lie side by
    side, on inputs of few values (1 or 2 in one of 50 dedispersed samples), all weights 1: the
    largest value occurs in several multiplets and profiles."""
    rank, bands, widths, time_ds = SHAPES[name]
    B, T = 2, 512
    print(f'[peak finder marks] sparse {name} {dtype}', flush=True)
    plan, dds = make_all(rank, bands, widths, dtype, B, T, time_ds)
    for it in range(plan.ntrees):
        for dd in dds:
            dd.fill_all_weights(it, np.ones(dd.wt_shape(it), dtype=np.float32))
    rng = np.random.default_rng(4)
    finite, bad, tied = (np.zeros(plan.ntrees, dtype=int) for _ in range(3))
    for c in range(4):
        x = np.zeros((B, plan.nfreq, T), dtype=np.float32)
        n = max(1, int(0.02 * x.size / plan.nfreq))
        x.reshape(-1)[rng.choice(x.size, n, replace=False)] = rng.integers(1, 3, size=n)
        if c > 0:
            for b in range(B):
                # one at each end of the band: at one of them no DM delays it past the last chunk
                for f, v in zip((0, plan.nfreq - 1, rng.integers(plan.nfreq)), rng.choice([np.inf, -np.inf, np.nan], 3)):
                    x[b, f, rng.integers(T)] = v
        res = outputs(plan, dds, c, x)
        assert_equal(plan, res, c)
        for it in range(plan.ntrees):
            v = res[0][it][2]
            finite[it] += np.sum(np.isfinite(v))
            bad[it] += np.sum(~np.isfinite(v))
            # the same nonzero maximum in neighbouring DM rows: multiplets of both share its samples
            tied[it] += np.sum((v[:, 1:] == v[:, :-1]) & (v[:, 1:] > 0))
    assert np.all(finite > 0) and np.all(bad > 0) and np.all(tied > 0), (finite, bad, tied)
