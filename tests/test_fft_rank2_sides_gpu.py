"""Rank-2 FFT column plans between a gather and a scatter (strided images on
both sides): two packed copies of workspace, as the transposing rows take, so
plans up to half the no-allocation array run from it. Against numpy's
complex128 fftn (reference rank-two lowering, src/c_api.cpp:5231-5327)."""
import numpy as np
import pytest

import cubutterfly_amd as cb
from gpu_util import to_device, to_host

pytestmark = pytest.mark.gpu

LIMIT = 32 << 20  # CUBUTTERFLY_NOALLOC_SCRATCH_BYTES


@pytest.mark.parametrize("extents,batch", [((512, 1024), 4), ((1024, 256), 8), ((2048, 2048), 1), ((4096, 512), 1)])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("in_place", [False, True])
def test_strided_sides(torch_gpu, lib, stream, extents, batch, inverse, in_place):
    n0, n1 = extents
    pitch = n1 + 8
    span = (batch * n0 - 1) * pitch + n1
    rng = np.random.default_rng(n0 + batch)
    flat = (rng.standard_normal(span) + 1j * rng.standard_normal(span)).astype(np.complex64)
    strides = {"input_strides": [pitch, 1], "input_batch_stride": n0 * pitch,
               "output_strides": [pitch, 1], "output_batch_stride": n0 * pitch}
    t = cb.describe(cb.Operator.FFT, cb.DataType.COMPLEX_FP32, list(extents), batch, compute=cb.ComputeType.FP32,
                    inverse=inverse, placement=int(in_place), **strides)
    index = (np.arange(batch * n0)[:, None] * pitch + np.arange(n1)).reshape(batch, n0, n1)
    ref = (np.fft.ifftn if inverse else np.fft.fftn)(flat[index].astype(np.complex128), axes=(1, 2))
    fill = flat if in_place else np.full(span, 7 + 7j, np.complex64)
    gaps = np.ones(span, bool)
    gaps[index] = False
    with cb.Plan(lib, t, stream=stream) as plan:
        assert plan.algorithm_name().startswith("rank2-columns[") and "+direct" not in plan.algorithm_name()
        size = plan.workspace_size()
        assert size == 2 * 8 * batch * n0 * n1
        ws = torch_gpu.empty(size, dtype=torch_gpu.uint8, device="cuda")
        plan.set_workspace(ws, size)
        for entry in ("Execute", "ExecuteNoAlloc"):
            if entry == "ExecuteNoAlloc" and size > LIMIT:
                continue
            x = to_device(torch_gpu, flat)
            y = x if in_place else to_device(torch_gpu, fill)
            lib(entry, plan.context, plan.handle, x.data_ptr(), y.data_ptr())
            torch_gpu.cuda.synchronize()
            got = to_host(torch_gpu, y, np.complex64)
            err = np.linalg.norm(got[index] - ref) / np.linalg.norm(ref)
            assert err <= 1e-6, err  # 5.7e-7 at 2^24 points
            np.testing.assert_array_equal(got[gaps], fill[gaps])
