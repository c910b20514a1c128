"""The rank-1 zero-extended embedding of FFTs up to 2^14 points in one pass: the
transform reads (forward) or writes (inverse) rows of the logical length itself
(reference docs/c_api.md:74-79; src/c_api.cpp:5231-5245, 5312-5325). Against
numpy's padded transform, whole output buffers with sentinels."""
import numpy as np
import pytest

import cubutterfly_amd as cb
from gpu_util import to_device, to_host

pytestmark = pytest.mark.gpu

EMB = cb.LengthMode.ZERO_EXTENDED_EMBEDDING


def pow2(n):
    return 1 << (n - 1).bit_length()


def run(torch, lib, stream, n, batch, inverse, pad=0, normalize=True, fused=True, offset=0, **fields):
    """`pad`: elements between the ragged rows; `offset`: elements both buffers
    start past a 256-byte boundary."""
    full, pitch = pow2(n), n + pad
    side = "output" if inverse else "input"
    if pad and batch > 1:
        fields.update({f"{side}_strides": [1], f"{side}_batch_stride": pitch})
    t = cb.describe(cb.Operator.FFT, cb.DataType.COMPLEX_FP32, [n], batch, compute=cb.ComputeType.FP32,
                    inverse=inverse, normalize_inverse=normalize, length_mode=EMB, **fields)
    rng = np.random.default_rng(n * 8 + batch)
    span = (batch - 1) * pitch + n
    n_in, n_out = (batch * full, span) if inverse else (span, batch * full)
    sentinel = np.complex64(7 - 3j)
    x = (rng.standard_normal(n_in) + 1j * rng.standard_normal(n_in)).astype(np.complex64)
    xd = to_device(torch, np.concatenate([np.full(offset, np.nan, np.complex64), x, np.full(3, np.nan, np.complex64)]))
    yd = to_device(torch, np.full(offset + n_out + 5, sentinel))
    with cb.Plan(lib, t, stream=stream) as plan:
        assert plan.mapping()["ragged_rows"] is fused
        size = plan.workspace_size()
        assert size >= 8 * full * batch  # as with the copies
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        plan.set_workspace(ws, size)
        plan.execute(xd[offset:], yd[offset:])
        torch.cuda.synchronize()
    got = to_host(torch, yd, np.complex64)
    assert np.all(got[:offset] == sentinel) and np.all(got[offset + n_out:] == sentinel)
    got = got[offset:offset + n_out]
    if inverse:
        want = np.fft.ifft(x.reshape(batch, full).astype(np.complex128), axis=1)[:, :n] * (1 if normalize else full)
        rows = np.stack([got[b * pitch:b * pitch + n] for b in range(batch)])
        gaps = [got[b * pitch + n:(b + 1) * pitch] for b in range(batch - 1)]
        assert all(np.all(g == sentinel) for g in gaps)
    else:
        rows_in = np.stack([x[b * pitch:b * pitch + n] for b in range(batch)])
        want = np.fft.fft(rows_in.astype(np.complex128), n=full, axis=1)
        rows = got.reshape(batch, full)
    err = np.linalg.norm(rows - want) / np.linalg.norm(want)
    assert err <= 1e-6, err  # 5.7e-7 at 2^24 points


# Lengths just past a power of two, just below one, and odd ones; batches that
# leave the last tile partial.
@pytest.mark.parametrize("n", [3, 5, 7, 9, 33, 100, 127, 257, 1000, 2047, 2049, 4095, 4097, 6000, 8191, 8193, 16383])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("batch", [1, 37])
def test_lengths(torch_gpu, lib, stream, n, inverse, batch):
    run(torch_gpu, lib, stream, n, batch, inverse, offset=1)


@pytest.mark.parametrize("n", [5, 300, 4099, 12001])
@pytest.mark.parametrize("inverse,normalize", [(False, True), (True, True), (True, False)])
@pytest.mark.parametrize("pad", [1, 64])
def test_pitched_rows(torch_gpu, lib, stream, n, inverse, normalize, pad):
    run(torch_gpu, lib, stream, n, 19, inverse, pad=pad, normalize=normalize)


@pytest.mark.parametrize("n", [3, 300])
@pytest.mark.parametrize("inverse", [False, True])
def test_single_row_with_a_short_batch_stride(torch_gpu, lib, stream, n, inverse):
    """One transform: the batch stride says nothing, so rows a tile lacks must
    not be written next to the first."""
    side = "output" if inverse else "input"
    run(torch_gpu, lib, stream, n, 1, inverse, **{f"{side}_strides": [1], f"{side}_batch_stride": 1})


def test_many_tiles(torch_gpu, lib, stream):
    # More rows than workgroups stay resident: the persistent walk.
    for n in (6000, 12000, 130):
        for inverse in (False, True):
            run(torch_gpu, lib, stream, n, 1100, inverse)


def test_other_layouts_keep_the_copies(torch_gpu, lib, stream):
    run(torch_gpu, lib, stream, 20000, 2, False, fused=False)  # two passes
