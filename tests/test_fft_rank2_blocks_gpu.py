"""Rank-2 FFTs of small blocks in one pass (whole blocks in a workgroup) and the
single column pass of 2^9 to 2^11 points, against numpy's complex128 fftn
(reference rank-two lowering, src/c_api.cpp:5231-5327)."""
import numpy as np
import pytest

import cubutterfly_amd as cb
from gpu_util import run_plan

pytestmark = pytest.mark.gpu

BLOCKS = "rank2-blocks[fft-c64-rank2-blocks-r16]+direct-input+direct-output"
COLUMNS = "rank2-columns[fft-c64-rank2-columns-r16]+direct-input+direct-output"


def fft_t(extents, batch, **kw):
    return cb.describe(cb.Operator.FFT, cb.DataType.COMPLEX_FP32, list(extents), batch, compute=cb.ComputeType.FP32, **kw)


def check(torch, lib, stream, extents, batch, name, inverse=False, normalize=True, in_place=False, **plan_args):
    rng = np.random.default_rng(extents[0] * 3 + extents[1] + batch)
    x = (rng.standard_normal((batch, *extents)) + 1j * rng.standard_normal((batch, *extents))).astype(np.complex64)
    t = fft_t(extents, batch, inverse=inverse, normalize_inverse=normalize, placement=int(in_place))
    with cb.Plan(lib, t, **plan_args) as plan:
        assert plan.algorithm_name() == name
    got = run_plan(torch, lib, t, x, stream, in_place=in_place, **plan_args).astype(np.complex128)
    ref = (np.fft.ifftn if inverse else np.fft.fftn)(x.astype(np.complex128), axes=(1, 2))
    if inverse and not normalize:
        ref = ref * (extents[0] * extents[1])
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= 1e-6, err  # 5.7e-7 at 2^24 points


# Digits of 1 to 4 bits on either axis, both tile limits (a window above a short
# axis 0, 2^14-point blocks), a partial last tile.
@pytest.mark.parametrize("l0,l1", [(1, 1), (1, 2), (3, 1), (2, 5), (4, 4), (5, 5), (5, 8), (8, 5), (6, 6), (7, 5), (1, 8),
                                   (9, 3), (4, 8), (4, 9), (13, 1), (6, 7), (9, 4), (7, 7), (4, 10), (5, 9), (12, 2)])
@pytest.mark.parametrize("inverse", [False, True])
def test_blocks(torch_gpu, lib, stream, l0, l1, inverse):
    batch = ((8 << max(12, l0 + l1)) >> (l0 + l1)) + 3
    check(torch_gpu, lib, stream, (1 << l0, 1 << l1), batch, BLOCKS, inverse=inverse)


def test_blocks_in_place_unnormalised(torch_gpu, lib, stream):
    for extents in ((32, 64), (64, 256)):
        check(torch_gpu, lib, stream, extents, 41, BLOCKS, inverse=True, normalize=False, in_place=True)


def test_few_blocks_and_long_rows_keep_other_lowerings(lib, torch_gpu):
    # Fewer tiles than XCDs; an axis-1 window of 4 bits above it leaves the tile.
    for extents, batch in (((64, 64), 7), ((2, 1 << 12), 16), ((1 << 7, 1 << 8), 64)):
        with cb.Plan(lib, fft_t(extents, batch)) as plan:
            assert not plan.algorithm_name().startswith("rank2-blocks[")
        with pytest.raises(cb.AbiError) as e:
            cb.Plan(lib, fft_t(extents, batch), algorithm=BLOCKS)
        assert e.value.status == cb.Status.NOT_SUPPORTED


def test_transposes_by_name(torch_gpu, lib, stream):
    name = "rank2-transpose[fft-c64-resident-r16,fft-c64-resident-r16]+direct-input+direct-output"
    check(torch_gpu, lib, stream, (64, 32), 20, name, algorithm=name)


def test_measure_times_the_blocks_and_the_cache_replays(torch_gpu, lib, stream, tmp_path):
    for extents, other in (((32, 64), "rank2-transpose["), ((64, 256), "rank2-columns[")):
        cache = tmp_path / f"{extents[1]}.tsv"
        t = fft_t(extents, 64)
        with cb.Plan(lib, t, policy=cb.AlgorithmPolicy.MEASURE, stream=stream, cache_path=cache) as plan:
            chosen, reason = plan.algorithm_name(), plan.selection_reason()
        assert "rank2-blocks[" in reason and other in reason, reason
        with cb.Plan(lib, t, stream=stream, cache_path=cache) as plan:
            assert plan.algorithm_name() == chosen
            assert plan.selection_source() == cb.SelectionSource.USER_CACHE


@pytest.mark.parametrize("l0,l1", [(9, 5), (9, 8), (9, 11), (10, 4 + 1), (10, 10), (11, 5), (11, 9), (11, 11), (7, 7),
                                   (9, 6)])
@pytest.mark.parametrize("inverse", [False, True])
def test_single_column_pass(torch_gpu, lib, stream, l0, l1, inverse):
    extents = (1 << l0, 1 << l1)
    check(torch_gpu, lib, stream, extents, 1 if l0 + l1 > 18 else 3, COLUMNS, inverse=inverse, algorithm=COLUMNS)
    with cb.Plan(lib, fft_t(extents, 1), algorithm=COLUMNS) as plan:
        assert plan.mapping()["schedule"][0]["child"]["column_passes"] == 1


@pytest.mark.parametrize("extents,batch,columns", [((512, 1024), 3, False), ((512, 1024), 4, True), ((512, 256), 16, True),
                                                   ((256, 512), 64, False), ((256, 256), 64, False)])
def test_default_rule(torch_gpu, lib, extents, batch, columns):
    with cb.Plan(lib, fft_t(extents, batch)) as plan:
        assert plan.algorithm_name().startswith("rank2-columns[" if columns else "rank2-transposing[")


# Two-pass 1-D lengths whose passes take halved tiles: 9-bit columns and 9- and
# 10-bit rows always, 10-bit columns while their tiles are fewer than the CUs.
@pytest.mark.parametrize("log_n,batch", [(17, 3), (18, 1), (18, 5), (19, 3), (20, 1), (20, 5), (21, 1), (21, 3)])
@pytest.mark.parametrize("inverse", [False, True])
def test_two_pass_tiles(torch_gpu, lib, stream, log_n, batch, inverse):
    rng = np.random.default_rng(log_n + batch)
    n = 1 << log_n
    x = (rng.standard_normal((batch, n)) + 1j * rng.standard_normal((batch, n))).astype(np.complex64)
    for orders in ([cb.LogicalOrder.NATURAL], [cb.LogicalOrder.BIT_REVERSED]):
        t = cb.describe(cb.Operator.FFT, cb.DataType.COMPLEX_FP32, [n], batch, compute=cb.ComputeType.FP32,
                        inverse=inverse, output_orders=orders)
        got = run_plan(torch_gpu, lib, t, x, stream).astype(np.complex128)
        ref = (np.fft.ifft if inverse else np.fft.fft)(x.astype(np.complex128), axis=1)
        if orders[0] == cb.LogicalOrder.BIT_REVERSED:
            perm = np.zeros(n, np.int64)
            for b in range(log_n):
                perm |= ((np.arange(n) >> b) & 1) << (log_n - 1 - b)
            ref = ref[:, perm]
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err <= 1e-6, err
