"""One-pass NTTs of 2^13 and 2^14 points (whole polynomials in one workgroup),
and the u64 arithmetic classes by modulus (fully reduced, lazy, lazy with
headroom), against the oracle, bit-exact (reference_ntt,
src/reference.cpp:584-630)."""
import numpy as np
import pytest

import cubutterfly_amd as cb
import oracle
from cubutterfly_amd import rns, workloads
from gpu_util import run_plan, to_device, to_host

pytestmark = pytest.mark.gpu

THREADS = oracle.default_threads()


def prime_below(limit, log_order):
    """The largest prime below `limit` that is 1 modulo 2^log_order."""
    q = ((limit - 2) >> log_order << log_order) + 1
    while not oracle.is_prime(q):
        q -= 1 << log_order
    return q


def prime_above(limit, log_order):
    q = (limit >> log_order << log_order) + 1
    while q < limit or not oracle.is_prime(q):
        q += 1 << log_order
    return q


# Fully reduced, lazy, and both ends of the headroom range.
U64 = {"strict": prime_below(1 << 63, 21), "lazy": prime_below(1 << 62, 21), "lazy-60": prime_above(1 << 60, 21),
       "headroom-top": prime_below(1 << 60, 21), "headroom-bottom": prime_above(1 << 33, 21),
       "lazy-small": prime_below(1 << 33, 21)}
U32 = {"strict": 2013265921, "lazy": workloads.C2_MODULUS}


def bitrev_perm(log_n):
    idx = np.arange(1 << log_n)
    rev = np.zeros_like(idx)
    for b in range(log_n):
        rev |= ((idx >> b) & 1) << (log_n - 1 - b)
    return rev


def check(torch, lib, stream, bits, log_n, batch, q, ring, inverse, rin, rout, algorithm=None):
    n = 1 << log_n
    words = np.uint32 if bits == 32 else np.uint64
    layout = {False: cb.NttLayout.NATURAL, True: cb.NttLayout.BIT_REVERSED}
    t = cb.describe(cb.Operator.NTT, cb.DataType.UINT32 if bits == 32 else cb.DataType.UINT64, [n], batch,
                    compute=cb.ComputeType.UINT32 if bits == 32 else cb.ComputeType.UINT64, modulus=q, word_bits=bits,
                    ntt_ring=ring, inverse=inverse, ntt_input_layout=layout[rin], ntt_output_layout=layout[rout])
    rng = np.random.default_rng(log_n * 64 + bits + inverse)
    x = rng.integers(0, np.iinfo(words).max, (batch, n), dtype=np.uint64, endpoint=True).astype(words)
    x.reshape(-1)[:4] = [0, np.iinfo(words).max, q - 1, q]
    perm = bitrev_perm(log_n)
    ref = oracle.ntt_negacyclic if ring == cb.NttRing.NEGACYCLIC else oracle.ntt_cyclic
    logical = x.astype(np.uint64) % np.uint64(q)
    expected = ref(logical[:, perm] if rin else logical, q, inverse=inverse, threads=THREADS)
    if rout:
        expected = expected[:, perm]
    plan_args = {"algorithm": algorithm} if algorithm else {}
    got = run_plan(torch, lib, t, x, stream, **plan_args)
    np.testing.assert_array_equal(got, expected.astype(words))


@pytest.mark.parametrize("bits,kind", [(32, k) for k in U32] + [(64, k) for k in ("strict", "lazy", "headroom-top")])
@pytest.mark.parametrize("log_n", [13, 14])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("rin,rout", [(False, False), (True, False), (False, True), (True, True)])
def test_resident_rows(torch_gpu, lib, stream, bits, kind, log_n, inverse, rin, rout):
    ring = cb.NttRing.NEGACYCLIC if rin == rout else cb.NttRing.CYCLIC
    name = f"ntt-u{bits}-{'negacyclic' if ring == cb.NttRing.NEGACYCLIC else 'cyclic'}-resident-r16"
    q = (U32 if bits == 32 else U64)[kind]
    check(torch_gpu, lib, stream, bits, log_n, 97, q, ring, inverse, rin, rout, name)


@pytest.mark.parametrize("kind", list(U64))
@pytest.mark.parametrize("log_n", [1, 3, 4, 7, 11, 12, 13, 16, 19])
@pytest.mark.parametrize("inverse", [False, True])
def test_u64_moduli(torch_gpu, lib, stream, kind, log_n, inverse):
    check(torch_gpu, lib, stream, 64, log_n, 3, U64[kind], cb.NttRing.NEGACYCLIC, inverse, False, False)


def test_mapping_names_the_arithmetic(torch_gpu, lib):
    for log_n, batch in ((10, 3), (13, 200), (16, 2)):
        for kind, q in U64.items():
            t = cb.describe(cb.Operator.NTT, cb.DataType.UINT64, [1 << log_n], batch, compute=cb.ComputeType.UINT64,
                            modulus=q, word_bits=64)
            with cb.Plan(lib, t) as plan:
                m = plan.mapping()
                assert m["headroom"] == kind.startswith("headroom") and m["lazy_reduction"] == (kind != "strict")


# (256 CUs) More than two 2^12-point rows per CU, inverse from natural to bit-reversed
# order, keep the lazy form; fewer, shorter ones and other orders take headroom.
@pytest.mark.parametrize("log_n,batch,inverse,rin,rout", [(12, 512, True, False, True), (12, 513, True, False, True),
                                                          (11, 1025, True, False, True), (12, 513, True, False, False),
                                                          (12, 513, False, False, True), (1, 5, True, False, True)])
def test_staged_inverse_rows_are_lazy(torch_gpu, lib, stream, log_n, batch, inverse, rin, rout):
    q = U64["headroom-top"]
    t = cb.describe(cb.Operator.NTT, cb.DataType.UINT64, [1 << log_n], batch, compute=cb.ComputeType.UINT64, modulus=q,
                    word_bits=64, inverse=inverse, ntt_input_layout=LAYOUT[rin], ntt_output_layout=LAYOUT[rout])
    with cb.Plan(lib, t) as plan:
        m = plan.mapping()
    assert m["lazy_reduction"] and m["headroom"] == (not (inverse and rout and log_n == 12 and batch > 512))
    check(torch_gpu, lib, stream, 64, log_n, batch, q, cb.NttRing.NEGACYCLIC, inverse, rin, rout)


# Tile counts that no multiple of 8 divides: every tile is some block's.
@pytest.mark.parametrize("bits,log_n,batch", [(64, 13, 1), (64, 13, 7), (64, 16, 3), (32, 14, 157), (32, 10, 29), (64, 12, 9),
                                              (32, 15, 1)])
def test_odd_tile_counts(torch_gpu, lib, stream, bits, log_n, batch):
    q = U32["lazy"] if bits == 32 else U64["headroom-top"]
    for inverse in (False, True):
        check(torch_gpu, lib, stream, bits, log_n, batch, q, cb.NttRing.NEGACYCLIC, inverse, False, False)


# Nontemporal intermediates: u64 2 .. 12 MiB, u32 with 32-column tiles 8 .. 12 MiB,
# forward only.
@pytest.mark.parametrize("bits,log_n,batch,inverse,streams", [
    (64, 16, 3, False, False), (64, 16, 4, False, True), (64, 16, 24, False, True), (64, 16, 25, False, False),
    (64, 16, 8, True, False), (64, 13, 31, False, False), (64, 13, 32, False, True), (32, 16, 31, False, False),
    (32, 16, 32, False, True), (32, 16, 48, False, True), (32, 16, 49, False, False), (32, 15, 64, False, False)])
def test_intermediate_stores(torch_gpu, lib, stream, bits, log_n, batch, inverse, streams):
    q = U32["lazy"] if bits == 32 else U64["headroom-top"]
    t = cb.describe(cb.Operator.NTT, cb.DataType.UINT32 if bits == 32 else cb.DataType.UINT64, [1 << log_n], batch,
                    compute=cb.ComputeType.UINT32 if bits == 32 else cb.ComputeType.UINT64, modulus=q, word_bits=bits,
                    ntt_ring=cb.NttRing.NEGACYCLIC, inverse=inverse)
    with cb.Plan(lib, t) as plan:
        assert plan.mapping()["shape"]["streams_intermediate"] == streams
    check(torch_gpu, lib, stream, bits, log_n, batch, q, cb.NttRing.NEGACYCLIC, inverse, False, False)


# (256 CUs) The edges of the rule, in natural order: a round half full (u64 2^14:
# four fifths of one, and no more rounds), two rounds three quarters full; u64 2^13
# any number of rounds beyond.
@pytest.mark.parametrize("bits,log_n,batch,resident", [(32, 13, 4, False), (32, 13, 8, True), (32, 14, 128, False),
                                                       (32, 14, 129, True), (64, 13, 128, False), (64, 13, 129, True),
                                                       (64, 14, 204, False), (64, 14, 205, True), (64, 14, 256, True),
                                                       (64, 14, 257, False), (64, 14, 410, False), (64, 14, 512, False),
                                                       (64, 13, 257, False), (64, 13, 383, False), (64, 13, 384, True),
                                                       (64, 13, 513, True), (32, 14, 300, False), (32, 14, 383, False),
                                                       (32, 14, 384, True), (32, 14, 513, False)])
def test_default_rule(torch_gpu, lib, bits, log_n, batch, resident):
    expect_resident(lib, bits, log_n, batch, resident)


# More than two rounds of u64 2^13 without headroom: seven eighths full.
@pytest.mark.parametrize("batch,resident", [(384, True), (513, False), (671, False), (672, True)])
def test_default_rule_without_headroom(torch_gpu, lib, batch, resident):
    for kind in ("lazy", "strict"):
        expect_resident(lib, 64, 13, batch, resident, kind)


# u32 2^14 by direction and order: forward to natural order from bit-reversed input,
# or with full reduction, in the first round only; rows that need no permutation in
# every round; the others two thirds of two rounds, seven eighths of more.
@pytest.mark.parametrize("batch,inverse,rin,rout,strict,resident", [
    (160, False, True, False, False, False), (192, False, True, False, False, True),
    (512, False, True, False, False, False), (160, False, False, False, True, False),
    (192, False, False, False, True, True), (512, False, False, False, True, False),
    (257, False, False, True, True, True), (700, False, False, True, False, True),
    (257, True, True, False, False, True), (128, True, True, False, False, False),
    (341, True, False, False, False, False), (342, True, False, False, False, True),
    (671, True, False, True, False, False), (672, True, False, True, False, True)])
def test_default_rule_by_order(torch_gpu, lib, batch, inverse, rin, rout, strict, resident):
    expect_resident(lib, 32, 14, batch, resident, "strict" if strict else "lazy", inverse=inverse, ntt_input_layout=LAYOUT[rin],
                    ntt_output_layout=LAYOUT[rout])


LAYOUT = {False: cb.NttLayout.NATURAL, True: cb.NttLayout.BIT_REVERSED}


def expect_resident(lib, bits, log_n, batch, resident, kind=None, **fields):
    q = U32[kind or "lazy"] if bits == 32 else U64[kind or "headroom-top"]
    t = cb.describe(cb.Operator.NTT, cb.DataType.UINT32 if bits == 32 else cb.DataType.UINT64, [1 << log_n], batch,
                    compute=cb.ComputeType.UINT32 if bits == 32 else cb.ComputeType.UINT64, modulus=q, word_bits=bits,
                    **fields)
    with cb.Plan(lib, t) as plan:
        assert ("resident" in plan.algorithm_name()) == resident
        assert (plan.workspace_size() == 0) == resident


@pytest.mark.parametrize("log_n", [13, 14])
@pytest.mark.parametrize("in_place,moving", [(False, True), (True, False), (True, True)])
def test_rns_offers_resident_rows(torch_gpu, lib, log_n, in_place, moving):
    """RNS Prepare times the one-pass mapping except where an in-place
    polynomial moves; irregular offsets and mixed domains stay bit-exact."""
    n, limbs, per = 1 << log_n, 3, 32
    moduli = [U64["headroom-top"], U64["headroom-bottom"], 576460756061519873]
    roots = [oracle.find_primitive_root(log_n + 1, q) for q in moduli]
    count = limbs * per
    order = np.random.default_rng(log_n).permutation(count)
    polys = [{"domain": int(order[i]) % limbs, "input_offset": i * (n + 16) + (5 if i > 7 else 0),
              "output_offset": (int(order[i]) if moving else i) * (n + 16) + (5 if i > 7 or moving else 0)}
             for i in range(count)]
    words = count * (n + 16) + 32
    rng = np.random.default_rng(7)
    data = np.full(words, 3, np.uint64)
    for p in polys:
        data[p["input_offset"]:p["input_offset"] + n] = rng.integers(0, moduli[p["domain"]], n, dtype=np.uint64)
    want = data.copy() if in_place else np.full(words, 3, np.uint64)
    for p in polys:
        row = data[p["input_offset"]:p["input_offset"] + n]
        want[p["output_offset"]:p["output_offset"] + n] = oracle.rns(row[None], [moduli[p["domain"]]], [roots[p["domain"]]],
                                                                     output_bit_reversed=True)[0]
    x = to_device(torch_gpu, data)
    y = x if in_place else to_device(torch_gpu, np.full(words, 3, np.uint64))
    cfg = rns.request(log_n, list(zip(moduli, roots)), polynomials=polys)
    s = torch_gpu.cuda.current_stream().cuda_stream
    with rns.RnsPlan(lib, cfg) as plan:
        plan.prepare(s, in_place=in_place, repetitions=1)
        names = [c["mapping"] for c in plan.info()["candidates"]]
        assert ("lazy-resident" in names) == (not (in_place and moving))
        plan.execute(x, y, s)
        torch_gpu.cuda.synchronize()
    np.testing.assert_array_equal(to_host(torch_gpu, y, np.uint64), want)
