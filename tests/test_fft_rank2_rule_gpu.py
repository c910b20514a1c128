"""The default lowering of rank-2 FFTs around the edges of its rule, the names
and the measurements that the shapes beside them keep (reference rank-two
lowering, src/c_api.cpp:5231-5327). Parity against numpy's complex128 fftn."""
import numpy as np
import pytest

import cubutterfly_amd as cb
from gpu_util import run_plan

pytestmark = pytest.mark.gpu

ROWS, COLUMNS, TRANSPOSES = "rank2-transposing[", "rank2-columns[", "rank2-transpose["


def fft_t(extents, batch, **kw):
    return cb.describe(cb.Operator.FFT, cb.DataType.COMPLEX_FP32, list(extents), batch, compute=cb.ComputeType.FP32, **kw)


def check(torch, lib, stream, extents, batch, prefix, inverse=False, **plan_args):
    rng = np.random.default_rng(extents[0] + extents[1])
    x = (rng.standard_normal((batch, *extents)) + 1j * rng.standard_normal((batch, *extents))).astype(np.complex64)
    t = fft_t(extents, batch, inverse=inverse)
    with cb.Plan(lib, t, **plan_args) as plan:
        assert plan.algorithm_name().startswith(prefix)
    got = run_plan(torch, lib, t, x, stream, **plan_args).astype(np.complex128)
    ref = (np.fft.ifftn if inverse else np.fft.fftn)(x.astype(np.complex128), axes=(1, 2))
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= 1e-6, err  # 5.7e-7 at 2^24 points


# Rows of 2^6 and 2^7 points: one column pass up to axis 0 = 2^11, transposing
# rows at 2^12, two column passes beyond (where the rows end).
@pytest.mark.parametrize("l0,l1,prefix", [(11, 6, COLUMNS), (11, 7, COLUMNS), (12, 6, ROWS), (12, 7, ROWS),
                                          (13, 6, COLUMNS), (13, 7, COLUMNS), (16, 6, COLUMNS), (12, 8, COLUMNS)])
@pytest.mark.parametrize("inverse", [False, True])
def test_short_rows(torch_gpu, lib, stream, l0, l1, prefix, inverse):
    check(torch_gpu, lib, stream, (1 << l0, 1 << l1), 2 if l0 < 13 else 1, prefix, inverse=inverse)


# One column pass of 9 to 11 bits over short rows: up to 2^24 points in all.
@pytest.mark.parametrize("extents,batch,prefix", [
    ((2048, 32), 256, COLUMNS), ((2048, 32), 512, ROWS), ((512, 256), 255, COLUMNS), ((512, 256), 256, ROWS),
    ((2048, 512), 32, ROWS), ((1024, 512), 63, COLUMNS), ((1024, 512), 64, ROWS), ((512, 1024), 64, ROWS),
    ((1024, 1024), 32, COLUMNS), ((256, 2048), 64, COLUMNS), ((512, 2048), 32, COLUMNS)])
def test_large_batches(torch_gpu, lib, extents, batch, prefix):
    with cb.Plan(lib, fft_t(extents, batch)) as plan:
        assert plan.algorithm_name().startswith(prefix)


def transposes(l0, l1):
    leaf = {6: "resident-r16", 7: "resident-r16", 13: "resident-r32", 15: "two-pass-r16"}
    return f"{TRANSPOSES}fft-c64-{leaf[l1]},fft-c64-{leaf[l0]}]+direct-input+direct-output"


@pytest.mark.parametrize("l0,l1", [(13, 6), (15, 7)])
def test_transposes_keep_their_name(torch_gpu, lib, stream, l0, l1):
    check(torch_gpu, lib, stream, (1 << l0, 1 << l1), 1, TRANSPOSES, algorithm=transposes(l0, l1))


def test_transposes_are_no_lowering_beside_the_others(lib, torch_gpu):
    name = f"{TRANSPOSES}fft-c64-resident-r16,fft-c64-resident-r16]+direct-input+direct-output"
    for extents in ((4096, 64), (2048, 64), (2048, 256)):
        with pytest.raises(cb.AbiError) as e:
            cb.Plan(lib, fft_t(extents, 1), algorithm=name)
        assert e.value.status == cb.Status.NOT_SUPPORTED


def test_measure_times_columns_and_transposes(torch_gpu, lib, stream, tmp_path):
    t = fft_t((1 << 13, 64), 2)
    cache = tmp_path / "sel.tsv"
    with cb.Plan(lib, t, policy=cb.AlgorithmPolicy.MEASURE, stream=stream, cache_path=cache) as plan:
        chosen, reason = plan.algorithm_name(), plan.selection_reason()
        assert plan.selection_source() == cb.SelectionSource.RUNTIME_MEASURED
    assert COLUMNS in reason and TRANSPOSES in reason, reason
    # Either record replays as what it names.
    records = cache.read_text().splitlines()
    key = next(line.split("\t")[0] for line in records if line.split("\t")[0].endswith("|rank2-fft|8192x64"))
    with cb.Plan(lib, t, stream=stream, cache_path=cache) as plan:
        assert plan.algorithm_name() == chosen and plan.selection_source() == cb.SelectionSource.USER_CACHE
    name = transposes(13, 6)
    other = tmp_path / "other.tsv"
    other.write_text(f"{key}\t{name}\n")
    with cb.Plan(lib, t, stream=stream, cache_path=other) as plan:
        assert plan.algorithm_name() == name and plan.selection_source() == cb.SelectionSource.USER_CACHE
