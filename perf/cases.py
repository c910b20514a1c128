"""The transforms that a program using this library runs, as timing cases.

Each case names one call pattern by its sizes and options: batched FWHTs (FP32
and FP16 with the final-storage epilogue), negacyclic NTTs over one prime and
over an RNS basis, and complex FFTs of one and two axes, of power-of-two and of
ragged lengths (the zero-extended embedding). Plans, twiddles and workspaces
are made once in `prepare`, as a program keeps them; `run` is one pass through
the public entry points on the current stream.

`listed()` holds the representative sizes, `draw()` any size of the same
ranges, odd batches and ragged lengths among them.
"""
import math

import torch

import cubutterfly_amd as cb
from cubutterfly_amd import ntt_roots, rns, workloads

# NTT primes of the single-modulus plans: 30-bit (2^30 - 2^18 + 1) and the
# largest 60-bit prime that is 1 modulo 2^21, so every length drawn has roots.
Q32 = workloads.C2_MODULUS
Q64 = workloads.ntt_primes(1, 60, 21)[0]

_library = None


def library():
    global _library
    if _library is None:
        _library = cb.Native()
    return _library


def listed():
    return [
        # A few short vectors to the Walsh domain and back: two short launches.
        {"name": "fwht32-few-rows", "kind": "fwht", "dtype": "fp32", "n": 1024, "rows": 61, "layout": "packed",
         "direction": "both"},
        # The library's headline FP32 batch: whole rows resident in a workgroup.
        {"name": "fwht32-rows", "kind": "fwht", "dtype": "fp32", "n": 4096, "rows": 4096, "layout": "packed",
         "direction": "forward"},
        # Signals longer than a workgroup holds, back from the Walsh domain (scaled by 1/n).
        {"name": "fwht32-long-inverse", "kind": "fwht", "dtype": "fp32", "n": 1 << 18, "rows": 40, "layout": "packed",
         "direction": "inverse"},
        # Activations of a hidden size, rotated before quantisation; the rows lie in a wider matrix.
        {"name": "fwht16-hidden", "kind": "fwht", "dtype": "fp16", "n": 4096, "rows": 8191, "layout": "pitched",
         "direction": "forward"},
        # A batch of polynomials modulo one 30-bit prime, to the NTT domain and back.
        {"name": "ntt32-batch", "kind": "ntt", "bits": 32, "log_n": 16, "rows": 64, "order": "natural"},
        # One ciphertext (two polynomials) of a small homomorphic-encryption parameter set.
        {"name": "rns-small", "kind": "rns", "log_n": 13, "limbs": 4, "per_limb": 2},
        # A batch of ciphertexts at the middle ring size, six limbs each.
        {"name": "rns-ciphertexts", "kind": "rns", "log_n": 14, "limbs": 6, "per_limb": 35},
        # A wide basis at the largest common ring size, one polynomial a limb.
        {"name": "rns-limbs", "kind": "rns", "log_n": 16, "limbs": 32, "per_limb": 1},
        # Many rows of a spectrogram-like length that one workgroup holds.
        {"name": "fft-rows", "kind": "fft", "log_n": 14, "rows": 1000, "inverse": False, "order": "natural"},
        # One transform of a long record.
        {"name": "fft-long", "kind": "fft", "log_n": 24, "rows": 1, "inverse": False, "order": "natural"},
        # A stack of images, back from their spectra.
        {"name": "fft2-images", "kind": "fft2", "log_h": 9, "log_w": 10, "rows": 13, "inverse": True},
        # Records of a length that is no power of two, zero-extended to the next.
        {"name": "fft-ragged", "kind": "ragged", "op": "fft", "n": 6000, "rows": 777, "inverse": False},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _rows(rng, n, least, most):
    """Rows of n elements so that rows * n lies between `least` and `most` elements (at least one row)."""
    return max(1, _spread(rng, least, most) // n)


def draw(rng):
    kind = rng.choice(["fwht", "fwht", "ntt", "rns", "rns", "fft", "fft", "fft2", "ragged"])
    if kind == "fwht":
        if rng.random() < 0.5:
            n = 1 << rng.randint(7, 16)
            return {"kind": kind, "dtype": "fp16", "n": n, "rows": _rows(rng, n, 1 << 14, 1 << 25),
                    "layout": rng.choice(["packed", "packed", "pitched"]) if n <= 8192 else "packed",
                    "direction": "forward"}
        n = 1 << rng.randint(5, 22)
        return {"kind": kind, "dtype": "fp32", "n": n, "rows": _rows(rng, n, 1 << 14, 1 << 24),
                "layout": rng.choice(["packed", "packed", "pitched", "bit_reversed"]) if n <= 8192 else "packed",
                "direction": rng.choice(["forward", "inverse", "both"])}
    if kind == "ntt":
        bits = rng.choice([32, 64])
        log_n = rng.randint(10, 17 if bits == 32 else 19)
        return {"kind": kind, "bits": bits, "log_n": log_n,
                "rows": _rows(rng, 1 << log_n, 1 << 14, 1 << (23 if bits == 32 else 22)),
                "order": rng.choice(["natural", "bit_reversed"])}
    if kind == "rns":
        log_n = rng.randint(12, 16)
        limbs = rng.randint(1, 16 if log_n < 16 else 32)
        most = max(1, (1 << 22) // (limbs << log_n))
        return {"kind": kind, "log_n": log_n, "limbs": limbs, "per_limb": _spread(rng, 1, most)}
    if kind == "fft":
        log_n = rng.randint(5, 23)
        return {"kind": kind, "log_n": log_n, "rows": _rows(rng, 1 << log_n, 1 << 14, 1 << 23),
                "inverse": rng.random() < 0.4, "order": rng.choice(["natural", "natural", "bit_reversed"])}
    if kind == "fft2":
        log_h, log_w = rng.randint(5, 11), rng.randint(5, 11)
        return {"kind": kind, "log_h": log_h, "log_w": log_w,
                "rows": _rows(rng, 1 << (log_h + log_w), 1 << 15, 1 << 23), "inverse": rng.random() < 0.4}
    n = _spread(rng, 50, 16000)
    return {"kind": kind, "op": rng.choice(["fft", "fft", "fwht"]), "n": n, "rows": _rows(rng, n, 1 << 14, 1 << 22),
            "inverse": rng.random() < 0.4}


# ---- inputs ------------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _complex(shape, seed):
    return torch.view_as_complex(torch.randn(*shape, 2, generator=_generator(seed), device="cuda"))


def _padded(n):
    return 1 << (n - 1).bit_length()


def _pitch(case):
    """Elements from one input row to the next: a row and 64 elements more where the rows lie in a wider matrix."""
    return case["n"] + (64 if case["layout"] == "pitched" else 0)


def _fwht_input(case, seed):
    shape = (case["rows"], _pitch(case))
    x = torch.randn(shape, generator=_generator(seed), device="cuda")
    if case["dtype"] == "fp16":
        # Activations: a few channels are 50 times as large as the others.
        x *= torch.where(torch.arange(shape[1], device="cuda") % 509 == 17, 50.0, 1.0)
        x = x.half()
    return x


def _residues(shape, moduli, seed, dtype):
    g = _generator(seed)
    rows = [torch.randint(0, q, shape, generator=g, device="cuda", dtype=torch.int64) for q in moduli]
    return torch.stack(rows).to(dtype).contiguous()


# ---- plans -------------------------------------------------------------------


def _plan(stream, *args, **fields):
    plan = cb.Plan(library(), cb.describe(*args, **fields), stream=stream)
    size = plan.workspace_size()
    if size:
        plan.set_workspace(torch.empty(size, dtype=torch.uint8, device="cuda"), size)
    return plan


_ORDERS = {"natural": cb.LogicalOrder.NATURAL, "bit_reversed": cb.LogicalOrder.BIT_REVERSED}


def prepare(case, seed):
    stream = torch.cuda.current_stream().cuda_stream
    kind = case["kind"]
    if kind == "fwht":
        x = _fwht_input(case, seed)
        fields = {}
        if case["dtype"] == "fp16":
            fields.update(output_scale=case["n"] ** -0.5, output_rounding=cb.OutputRounding.FINAL_STORAGE)
        if case["layout"] == "pitched":
            fields.update(input_strides=[1], input_batch_stride=_pitch(case))
        elif case["layout"] == "bit_reversed":
            fields.update(input_orders=[_ORDERS["bit_reversed"]])
        storage = cb.DataType.FP16 if case["dtype"] == "fp16" else cb.DataType.FP32
        plans = []
        if case["direction"] != "inverse":
            plans.append(_plan(stream, cb.Operator.FWHT, storage, [case["n"]], case["rows"],
                               compute=cb.ComputeType.FP32, **fields))
        if case["direction"] != "forward":
            back = {} if plans else fields  # the forward result is packed, in natural order
            plans.append(_plan(stream, cb.Operator.FWHT, storage, [case["n"]], case["rows"],
                               compute=cb.ComputeType.FP32, inverse=True, **back))
        outs = [torch.empty((case["rows"], case["n"]), dtype=x.dtype, device="cuda") for _ in plans]
        return {"kind": kind, "plans": plans, "x": x, "outs": outs}
    if kind == "ntt":
        wide = case["bits"] == 64
        q = Q64 if wide else Q32
        layout = cb.NttLayout.BIT_REVERSED if case["order"] == "bit_reversed" else cb.NttLayout.NATURAL
        plans = []
        for inverse in (False, True):
            sides = {"ntt_input_layout" if inverse else "ntt_output_layout": layout}
            plans.append(_plan(stream, cb.Operator.NTT, cb.DataType.UINT64 if wide else cb.DataType.UINT32,
                               [1 << case["log_n"]], case["rows"],
                               compute=cb.ComputeType.UINT64 if wide else cb.ComputeType.UINT32, modulus=q,
                               word_bits=case["bits"], ntt_ring=cb.NttRing.NEGACYCLIC, inverse=inverse, **sides))
        x = _residues((case["rows"], 1 << case["log_n"]), [q], seed, torch.int64 if wide else torch.int32)[0]
        return {"kind": kind, "plans": plans, "x": x, "outs": [torch.empty_like(x), torch.empty_like(x)]}
    if kind == "rns":
        n = 1 << case["log_n"]
        moduli = workloads.ntt_primes(case["limbs"], 60, case["log_n"] + 1)
        domains = [(q, ntt_roots.primitive_root(case["log_n"] + 1, q)) for q in moduli]
        polynomials = [{"domain": i // case["per_limb"], "input_offset": i * n, "output_offset": i * n}
                       for i in range(case["limbs"] * case["per_limb"])]
        plans = []
        for inverse in (False, True):
            plan = rns.RnsPlan(library(), rns.request(case["log_n"], domains, inverse=inverse,
                                                      polynomials=polynomials))
            plans.append(plan.prepare(stream))
        x = _residues((case["per_limb"], n), moduli, seed, torch.int64)
        return {"kind": kind, "plans": plans, "x": x, "outs": [torch.empty_like(x), torch.empty_like(x)],
                "stream": stream}
    if kind == "fft":
        n = 1 << case["log_n"]
        fields = {"output_orders": [_ORDERS["bit_reversed"]]} if case["order"] == "bit_reversed" else {}
        plan = _plan(stream, cb.Operator.FFT, cb.DataType.COMPLEX_FP32, [n], case["rows"],
                     compute=cb.ComputeType.FP32, inverse=case["inverse"], **fields)
        x = _complex((case["rows"], n), seed)
        return {"kind": kind, "plans": [plan], "x": x, "outs": [torch.empty_like(x)]}
    if kind == "fft2":
        shape = (1 << case["log_h"], 1 << case["log_w"])
        plan = _plan(stream, cb.Operator.FFT, cb.DataType.COMPLEX_FP32, shape, case["rows"],
                     compute=cb.ComputeType.FP32, inverse=case["inverse"])
        x = _complex((case["rows"],) + shape, seed)
        return {"kind": kind, "plans": [plan], "x": x, "outs": [torch.empty_like(x)]}
    full = _padded(case["n"])
    n_in, n_out = (full, case["n"]) if case["inverse"] else (case["n"], full)
    fft = case["op"] == "fft"
    plan = _plan(stream, cb.Operator.FFT if fft else cb.Operator.FWHT,
                 cb.DataType.COMPLEX_FP32 if fft else cb.DataType.FP32, [case["n"]], case["rows"],
                 compute=cb.ComputeType.FP32, inverse=case["inverse"],
                 length_mode=cb.LengthMode.ZERO_EXTENDED_EMBEDDING)
    x = _ragged_input(case, n_in, seed)
    y = torch.empty((case["rows"], n_out), dtype=x.dtype, device="cuda")
    return {"kind": kind, "plans": [plan], "x": x, "outs": [y]}


def _ragged_input(case, n_in, seed):
    if case["op"] == "fft":
        return _complex((case["rows"], n_in), seed)
    return torch.randn((case["rows"], n_in), generator=_generator(seed), device="cuda")


def run(state):
    x, outs = state["x"], state["outs"]
    if state["kind"] == "rns":
        state["plans"][0].execute(x, outs[0], state["stream"])
        state["plans"][1].execute(outs[0], outs[1], state["stream"])
        return outs
    for plan, y in zip(state["plans"], outs):
        plan.execute(x, y)
        x = y
    return outs


# ---- what a pass cannot do without -------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "fwht":
        size = 2 if case["dtype"] == "fp16" else 4
        total = case["rows"] * case["n"] * (2 if case["direction"] == "both" else 1)
        return {"bytes": 2 * size * total, "flops": total * (case["n"].bit_length() - 1)}
    if kind in ("ntt", "rns"):
        # To the NTT domain and back: each direction reads and writes every
        # word once; a butterfly is one modular product, one sum, one difference.
        total = (case["rows"] if kind == "ntt" else case["limbs"] * case["per_limb"]) << case["log_n"]
        size = 4 if kind == "ntt" and case["bits"] == 32 else 8
        return {"bytes": 2 * 2 * size * total, "flops": 2 * 3 * (total // 2) * case["log_n"]}
    if kind == "fft":
        total = case["rows"] << case["log_n"]
        return {"bytes": 16 * total, "flops": 5 * total * case["log_n"]}
    if kind == "fft2":
        log = case["log_h"] + case["log_w"]
        total = case["rows"] << log
        return {"bytes": 16 * total, "flops": 5 * total * log}
    full = _padded(case["n"])
    log = full.bit_length() - 1
    size, per = (8, 5) if case["op"] == "fft" else (4, 1)
    return {"bytes": size * case["rows"] * (case["n"] + full), "flops": per * case["rows"] * full * log}


def tolerance(case):
    if case["kind"] in ("ntt", "rns"):
        return "exact"  # canonical residues
    if case["kind"] == "fwht" and case["dtype"] == "fp16":
        return {"rel": 4e-4, "max": 2e-3}  # sums in another order: a few results round to the neighbouring FP16
    if case["kind"] == "fwht" or (case["kind"] == "ragged" and case["op"] == "fwht"):
        return {"rel": 4e-7}  # 1.2e-7 from 64 bits at 2^18 points
    return {"rel": 2e-6}  # 5.7e-7 from 64 bits at 2^24 points


# ---- the same in 64 bits -----------------------------------------------------


def _hadamard(x):
    n = x.shape[-1]
    h = 1
    while h < n:
        v = x.reshape(-1, n // (2 * h), 2, h)
        x = torch.stack((v[:, :, 0] + v[:, :, 1], v[:, :, 0] - v[:, :, 1]), dim=2)
        h *= 2
    return x.reshape(-1, n)


def _reversal(n):
    bits = n.bit_length() - 1
    j = torch.arange(n, device="cuda")
    r = torch.zeros_like(j)
    for b in range(bits):
        r |= ((j >> b) & 1) << (bits - 1 - b)
    return r


def exact(case, seed):
    kind = case["kind"]
    if kind == "fwht":
        n = case["n"]
        x = _fwht_input(case, seed)[:, :n].double()
        if case["layout"] == "bit_reversed":
            x = x[:, _reversal(n)]
        if case["direction"] == "both":
            return [_hadamard(x), x]
        y = _hadamard(x)
        return [y * n ** -0.5 if case["dtype"] == "fp16" else y / n if case["direction"] == "inverse" else y]
    if kind in ("ntt", "rns"):
        return None  # residues are whole numbers: compared bit by bit
    if kind == "fft":
        n = 1 << case["log_n"]
        x = _complex((case["rows"], n), seed).to(torch.complex128)
        y = torch.fft.ifft(x) if case["inverse"] else torch.fft.fft(x)
        return [y[:, _reversal(n)] if case["order"] == "bit_reversed" else y]
    if kind == "fft2":
        x = _complex((case["rows"], 1 << case["log_h"], 1 << case["log_w"]), seed).to(torch.complex128)
        return [torch.fft.ifft2(x) if case["inverse"] else torch.fft.fft2(x)]
    full, n = _padded(case["n"]), case["n"]
    x = _ragged_input(case, full if case["inverse"] else n, seed)
    if case["op"] == "fft":
        x = x.to(torch.complex128)
        return [torch.fft.ifft(x)[:, :n].contiguous() if case["inverse"] else torch.fft.fft(x, n=full)]
    x = x.double()
    if case["inverse"]:
        return [(_hadamard(x) / full)[:, :n].contiguous()]
    return [_hadamard(torch.nn.functional.pad(x, (0, full - n)))]
