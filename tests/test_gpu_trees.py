"""Tree kernels at the edges of their tiles and time segments, bit for bit against the oracle:
every stage rank 1..8, chunks of one half tile, of tile counts that the segments do not divide,
and of segments that end in a half tile; subband searches with every level and with none."""

import pytest

from gpu_cases import BASE, pt
from gpu_harness import run_and_compare

pytestmark = pytest.mark.gpu

# name: (rank, chunk, beams, subband counts, dtype, chunks run)
SHAPES = {
    'r3_16_tiles': (3, 1024, 1, [1], 'float32', 3),
    'r4_half_tile_only': (4, 32, 1, [1], 'float32', 6),
    'r5_11_tiles': (5, 704, 2, [2, 1], 'float16', 3),
    'r7_tile_and_half': (7, 96, 3, [2, 2, 1], 'float32', 6),
    'r8_45_tiles': (8, 2848, 1, [2, 2, 1], 'float32', 2),
    'r9_levels': (9, 1088, 1, [8, 7, 3, 1], 'bfloat16', 3),
    'r11_31_tiles': (11, 1984, 1, [0, 3, 1], 'float32', 3),
    'r12_all_levels': (12, 832, 2, [8, 15, 7, 3, 1], 'float32', 2),
    'r13_19_tiles': (13, 1216, 1, [16, 15, 7, 3, 1], 'float16', 2),
    'r14_half_tile': (14, 608, 1, [5, 9, 7, 3, 1], 'float32', 2),
    'r15_13_tiles': (15, 832, 1, [0, 0, 3, 2, 1], 'float16', 3),
    'r16_half_tile': (16, 608, 1, [1], 'float32', 2),
}


@pytest.mark.parametrize('name', list(SHAPES))
def test_tiles_and_segments(name):
    rank, T, beams, bands, dtype, nchunks = SHAPES[name]
    print(f'[trees] {name}', flush=True)
    cfg = dict(BASE, dtype=dtype, zone_nfreq=[2**min(rank, 11) + 5], zone_freq_edges=[400, 800], toplevel_tree_rank=rank,
               time_samples_per_chunk=T, beams_per_gpu=beams, beams_per_batch=beams, num_active_batches=1,
               frequency_subband_counts=bands, primary_trees=[pt(0, 4, min(64, 2**(rank - 1)), T & -T if T & -T <= 64 else 64)])
    bad, _, _ = run_and_compare(cfg, nchunks, seed=rank, log=lambda m: print(m, flush=True))
    assert not bad, f'first mismatch: {bad[0]}'
