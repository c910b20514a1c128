"""2^20-point FFTs in natural order on both tile sizes of their 10-bit row pass:
2^13-point tiles up to 2^24 points in all, 2^14-point tiles from 2^25. Against
numpy's complex128 FFT, row by row (reference FFT plans, src/c_api.cpp:4981-5064)."""
import numpy as np
import pytest

import cubutterfly_amd as cb

pytestmark = pytest.mark.gpu

N = 1 << 20


@pytest.mark.parametrize("batch,reversed_out,lines", [(31, False, 8), (32, False, 16), (33, False, 16), (32, True, 8)])
@pytest.mark.parametrize("inverse", [False, True])
def test_row_tiles(torch_gpu, lib, stream, batch, reversed_out, lines, inverse):
    orders = [cb.LogicalOrder.BIT_REVERSED if reversed_out else cb.LogicalOrder.NATURAL]
    t = cb.describe(cb.Operator.FFT, cb.DataType.COMPLEX_FP32, [N], batch, compute=cb.ComputeType.FP32,
                    inverse=inverse, output_orders=orders)
    g = torch_gpu.Generator(device="cuda")
    g.manual_seed(batch)
    x = torch_gpu.view_as_complex(torch_gpu.randn(batch, N, 2, generator=g, device="cuda"))
    y = torch_gpu.empty_like(x)
    with cb.Plan(lib, t, stream=stream) as plan:
        assert plan.mapping()["row_tile_lines"] == lines
        size = plan.workspace_size()
        ws = torch_gpu.empty(size, dtype=torch_gpu.uint8, device="cuda")
        plan.set_workspace(ws, size)
        plan.execute(x, y)
        torch_gpu.cuda.synchronize()
    perm = np.zeros(N, np.int64)
    for b in range(20):
        perm |= ((np.arange(N) >> b) & 1) << (19 - b)
    for row in (0, batch // 2, batch - 1):
        ref = (np.fft.ifft if inverse else np.fft.fft)(x[row].cpu().numpy().astype(np.complex128))
        if reversed_out:
            ref = ref[perm]
        err = np.linalg.norm(y[row].cpu().numpy() - ref) / np.linalg.norm(ref)
        assert err <= 1e-6, err  # 5.7e-7 at 2^24 points
