"""Device memory per beam, and lag rings of more than 2^31 elements per beam."""

import numpy as np
import pytest

from gpu_cases import BASE, chord16k_with_beams, pt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype,batch,limit', [('float32', 0, 1.500), ('float16', 0, 0.767), ('float32', 2, 1.195), ('float16', 2, 0.614)])
def test_bytes_per_beam(dtype, batch, limit):
    """16384 channels, four primary trees: what each beam beyond the first 16 takes (GiB), all beams in
    one batch and in batches of 2, whose trees run in several time segments."""
    import pirate_amd as pa

    def nbytes(n):
        cfg = dict(chord16k_with_beams(n, batch), dtype=dtype, num_active_batches=2 if batch else 1)
        dd = pa.GpuDedisperser(pa.DedispersionPlan(pa.DedispersionConfig.from_dict(cfg)))
        dd.allocate()
        return dd.gpu_bytes()

    per_beam = (nbytes(32) - nbytes(16)) / 16 / 2**30
    print(f'[memory] {dtype} {batch}: {per_beam:.5f} GiB per beam', flush=True)
    assert per_beam <= limit


def test_ring_beyond_2_31_elements():
    """One beam of rank 16 whose lag ring has 2.16e9 elements, against the same search with most of
    the ring in host memory, bit for bit, until the largest lag (65025 samples) is covered."""
    import torch
    import pirate_amd as pa
    T = 16640
    cfg = dict(BASE, dtype='float16', zone_nfreq=[2048], zone_freq_edges=[400, 800], toplevel_tree_rank=16,
               time_samples_per_chunk=T, beams_per_gpu=1, beams_per_batch=1, num_active_batches=1,
               frequency_subband_counts=[1], primary_trees=[pt(0, 8, 64, 64)])
    dds = []
    for c in (cfg, dict(cfg, max_gpu_clag=0)):
        dd = pa.GpuDedisperser(pa.DedispersionPlan(pa.DedispersionConfig.from_dict(c)))
        dd.allocate()
        dd.fill_all_weights(0, np.ones(dd.wt_shape(0), dtype=np.float32))
        dds.append(dd)
    assert dds[1].host_bytes() > 0 and dds[0].host_bytes() == 0
    gen = torch.Generator('cuda').manual_seed(1)
    for c in range(5):
        x = torch.randn(1, 2048, T, device='cuda', generator=gen).half()
        got = []
        for dd in dds:
            print(f'[memory] ring chunk {c}', flush=True)
            with dd.get_input(c) as arr:
                arr.copy_(x)
            with dd.get_output(c) as out:
                got.append([a.clone() for a in (out.out_max[0], out.out_argmax[0])])
        for a, b in zip(*got):
            assert torch.equal(a, b), f'chunk {c}'
