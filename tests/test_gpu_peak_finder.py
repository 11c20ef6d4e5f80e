"""The two-step peak finder against the one that visits every candidate in order (the kernel that
also forms the float64 variances), bit for bit, on inputs where the two could part: ties (long
stretches of zeros), infinities, NaN, values that overflow, and zero weights; over the numbers of
multiplets (whole DM rows in a wave or not), bin lengths, boxcar lengths and storage types."""

import numpy as np
import pytest

from gpu_cases import BASE, pt
from gpu_harness import random_weights

pytestmark = pytest.mark.gpu

# (rank, subband counts, boxcars per primary tree): M = 2..91 multiplets, bins of 2..16 samples
SHAPES = {
    'r4_m2': (4, [1], [32, 4]),                  # bins of 2 samples
    'r7_m4': (7, [1], [1, 16]),                  # a tree without boxcars
    'r10_m8': (10, [1], [32, 2]),
    'r13_m16': (13, [0, 0, 0, 0, 1], [16, 8]),
    'r8_m10': (8, [2, 2, 1], [16, 8, 4]),        # DM rows straddle waves
    'r11_m34': (11, [4, 5, 3, 1], [8, 32]),
    'r14_m91': (14, [5, 9, 7, 3, 1], [16]),      # two DM rows per workgroup
}


def chunk(kind, rng, shape):
    x = rng.standard_normal(shape).astype(np.float32)
    if kind == 'ties':
        x *= rng.random(shape) < 0.002
    elif kind == 'nonfinite':
        for v in (np.inf, -np.inf, np.nan, 3e38, -3e38):
            x[rng.random(shape) < 2e-5] = v
    return x


@pytest.mark.parametrize('dtype', ['float32', 'float16'])
@pytest.mark.parametrize('kind', ['ties', 'nonfinite'])
@pytest.mark.parametrize('name', list(SHAPES))
def test_two_steps_equal_one(name, kind, dtype):
    import torch
    import pirate_amd as pa
    rank, bands, widths = SHAPES[name]
    B, T = 2, 512
    cfg = dict(BASE, dtype=dtype, zone_nfreq=[2**rank - 3], zone_freq_edges=[400, 800], toplevel_tree_rank=rank,
               time_samples_per_chunk=T, beams_per_gpu=B, beams_per_batch=B, num_active_batches=1,
               frequency_subband_counts=bands, primary_trees=[pt(0, w, min(64, 2**(rank - 1)), 64) for w in widths])
    plan = pa.DedispersionPlan(pa.DedispersionConfig.from_dict(cfg))
    print(f'[peak finder] {name} {kind} {dtype} M={[t.nmultiplets_M for t in plan.trees]}', flush=True)
    dds = [pa.GpuDedisperser(plan, enable_variances=v) for v in (False, True)]
    rng = np.random.default_rng(3)
    for dd in dds:
        dd.allocate()
    for it in range(plan.ntrees):
        w = random_weights(rng, dds[0], it)
        for dd in dds:
            dd.fill_all_weights(it, w)
    for c in range(3):
        x = torch.from_numpy(chunk(kind, rng, (B, plan.nfreq, T))).cuda()
        got = []
        for dd in dds:
            with dd.get_input(c) as arr:
                arr.copy_(x)
            with dd.get_output(c) as out:
                bits = torch.int32 if dtype == 'float32' else torch.int16
                got.append([(m.view(bits).cpu().numpy(), a.cpu().numpy()) for m, a in zip(out.out_max, out.out_argmax)])
        for it in range(plan.ntrees):
            for i, what in enumerate(('out_max', 'out_argmax')):
                a, b = got[0][it][i], got[1][it][i]
                assert np.array_equal(a, b), f'chunk {c} tree {it} {what}: {int(np.sum(a != b))} of {a.size} differ'
