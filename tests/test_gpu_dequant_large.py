"""Dequantization of more samples than one launch has threads for (2^34 float32 samples, 64 GiB out)."""

import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def test_more_than_2_32_threads():
    import torch
    import pirate_amd as pa
    B, F, T = 4, 16384 + 1, 2**18
    nmin = T // 256
    if torch.cuda.mem_get_info()[0] < 90 * 2**30:
        pytest.skip('needs 90 GiB of GPU memory')
    gen = torch.Generator('cuda').manual_seed(1)
    data = torch.randint(-2**62, 2**62, (B, F, T // 16), dtype=torch.int64, device='cuda', generator=gen).view(torch.uint8)
    so = torch.rand(B, F, nmin, 2, device='cuda', generator=gen).half()
    out = torch.full((B, F, T), 7.0, device='cuda')
    print('[dequantization] 2^34 samples', flush=True)
    pa.GpuDequantizationKernel('float32', B, F, T).launch(out, so, data)
    flat, fd, fs = out.view(-1), data.view(-1), so.view(-1, 2)
    n = flat.numel()
    assert n > 2**34
    for at in (0, 2**31, 2**32, 2**33, 2**33 + 2**32, 2**34 - 512, n - 1024):
        got = flat[at:at + 1024].cpu().numpy()
        want = orc.dequantize(fd[at // 2:at // 2 + 512].cpu().numpy().reshape(1, 1, 512),
                              fs[at // 256:at // 256 + 4].cpu().numpy().reshape(1, 1, 4, 2), 1, 1, 1024)
        np.testing.assert_array_equal(got, np.asarray(want).reshape(-1), err_msg=f'samples from {at}')
