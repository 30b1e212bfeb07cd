"""The work this codec is used for, as measurable cases.

A case is a dict of plain values:

  op      "compress", "decompress" or "batch"
  type    "f32", "f64", "i32", "i64"
  size    extents, x (fastest) first: "512x512x512"
  mode    "rate", "precision", "accuracy" or "reversible", with its `value`
  view    "contiguous", or "permuted": the last axis fastest in memory, x
          slowest with a negative stride (a transposed, flipped view)
  index   (decompress, variable length) True: the stream was compressed by
          this process, so its block index is at hand; False: it was read from
          somewhere else, behind a 16-byte header of the file it came in
  arrays  (batch) how many arrays one batch holds

Fields and streams are resident in device memory, as a simulation or an
analysis on the GPU holds them.
"""
import math

import numpy as np
import torch

import zfp_amd as Z

DEVICE = "cuda:0"
ZTYPE = {"i32": Z.zfp_type_int32, "i64": Z.zfp_type_int64, "f32": Z.zfp_type_float, "f64": Z.zfp_type_double}
DTYPE = {"i32": torch.int32, "i64": torch.int64, "f32": torch.float32, "f64": torch.float64}
BITS = {"i32": 32, "i64": 64, "f32": 32, "f64": 64}
# zfp_stream_set_reversible: ZFP_MIN_BITS, ZFP_MAX_BITS, ZFP_MAX_PREC, ZFP_MIN_EXP - 1
REVERSIBLE = (1, 16658, 64, -1075)
HEADER_WORDS = 2


def _case(op, ztype, size, mode, value, view="contiguous", index=True, **name):
    return dict(name, op=op, type=ztype, size=size, mode=mode, value=value, view=view, index=index)


def listed():
    return [
        # a large simulation field written at the middle rate: the usual checkpoint
        _case("compress", "f64", "512x512x512", "rate", 16, name="f64_3d_rate16_compress"),
        # and read back
        _case("decompress", "f64", "512x512x512", "rate", 16, name="f64_3d_rate16_decompress"),
        # read back at high quality into a transposed, flipped view
        _case("decompress", "f64", "512x512x512", "rate", 32, "permuted", name="f64_3d_rate32_permuted_decompress"),
        # an ordinary in-memory array of a single-precision code
        _case("compress", "f32", "128x128x128", "rate", 8, name="f32_3d_rate8_compress"),
        # the smallest calls, odd extents: a brick of a larger array
        _case("decompress", "f32", "65x33x17", "rate", 8, name="f32_3d_brick_decompress"),
        # an image-like field stored within an error bound
        _case("compress", "f32", "8191x8193", "accuracy", 1e-3, name="f32_2d_accuracy_compress"),
        # the same kind of field at high precision, read where it was written
        _case("decompress", "f32", "8191x8193", "precision", 28, name="f32_2d_precision_decompress"),
        # and from a file another program wrote
        _case("decompress", "f32", "8191x8193", "precision", 16, index=False, name="f32_2d_file_decompress"),
        # space-time data (three space axes and time)
        _case("compress", "f64", "96x96x96x24", "precision", 28, name="f64_4d_precision_compress"),
        _case("decompress", "f64", "96x96x96x24", "accuracy", 1e-3, name="f64_4d_accuracy_decompress"),
        # lossless storage of a ragged field
        _case("compress", "f64", "257x129x191", "reversible", 0, name="f64_3d_reversible_compress"),
        # a mesh of many small patches, written and read back as one batch each way
        dict(name="mixed_patches_batch", op="batch", arrays=1024),
    ]


def _extents(case):
    return [int(v) for v in case["size"].split("x")]


def _size(rng, dims, low, high):
    """Extents with a product spread over [low, high] by its logarithm, the axes up to a factor of two apart."""
    values = math.exp(rng.uniform(math.log(low), math.log(high)))
    lean = [rng.uniform(-0.35, 0.35) for _ in range(dims)]
    mean = sum(lean) / dims
    edge = values ** (1.0 / dims)
    return "x".join(str(max(1, int(edge * math.exp(a - mean)))) for a in lean)


def draw(rng):
    kind = rng.choice(["rate", "rate", "rate", "variable", "variable", "4d", "reversible", "file", "batch"])
    if kind == "batch":
        return dict(op="batch", arrays=rng.randint(64, 1024))
    op = rng.choice(["compress", "decompress"])
    if kind == "rate":
        ztype = rng.choice(["f64", "f32", "f64", "f32", "i32", "i64"])
        dims = rng.choice([1, 2, 3, 3, 3])
        view = rng.choice(["contiguous", "contiguous", "permuted"]) if dims > 1 else "contiguous"
        return _case(op, ztype, _size(rng, dims, 1 << 12, 1 << 27), "rate",
                     rng.choice([4, 8, 16, rng.randint(3, 32)]), view)
    if kind == "variable":
        ztype, dims = rng.choice([("f32", 2), ("f32", 3), ("f64", 2), ("f64", 3)])
        mode, value = _quality(rng)
        return _case(op, ztype, _size(rng, dims, 1 << 14, 1 << 26), mode, value)
    if kind == "4d":
        mode, value = _quality(rng)
        return _case(op, rng.choice(["f64", "f64", "f32"]), _size(rng, 4, 1 << 14, 96 * 96 * 96 * 24), mode, value)
    if kind == "reversible":
        ztype, dims = rng.choice([("f32", 2), ("f32", 3), ("f64", 3), ("i32", 3)])
        return _case(op, ztype, _size(rng, dims, 1 << 14, 1 << 24), "reversible", 0)
    mode, value = _quality(rng)
    return _case("decompress", "f32", _size(rng, rng.choice([2, 3]), 1 << 16, 1 << 26), mode, value, index=False)


def _quality(rng):
    if rng.random() < 0.5:
        return "precision", rng.randint(10, 28)
    return "accuracy", float("%.1e" % 10.0 ** rng.uniform(-7, -2))


def _params(mode, value, ztype, dims):
    return REVERSIBLE if mode == "reversible" else Z.stream_params(mode, value, ZTYPE[ztype], dims)


def _typed(f, ztype):
    """A field of values within about +-1 as the given type; integers use 28 or 60 bits."""
    if ztype == "i32":
        return torch.round(f * 2.0 ** 28).to(torch.int32)
    if ztype == "i64":
        return torch.round(f * 2.0 ** 60).to(torch.int64)
    return f.to(DTYPE[ztype])


def _field(n, ztype, seed, box):
    """A smooth field (four plane waves) with a little measurement noise; with `box`, a corner of about a
    tenth of it is turbulent (uniform noise), as variable-length modes are made for."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    r = np.random.default_rng(seed)
    dims, shape = len(n), list(reversed(n))
    f = torch.randn(shape, device=DEVICE, dtype=torch.float64, generator=g).mul_(1e-3)
    for _ in range(4):
        # sin(a + b) by its parts: one product of the last axis's waves with the others'
        phase = torch.full(shape[:-1] or [1], float(r.uniform(0, 2 * math.pi)), device=DEVICE, dtype=torch.float64)
        waves = [2 * math.pi * int(r.integers(1, 7)) / v for v in n]
        for d in range(1, dims):
            view = [1] * (dims - 1)
            view[dims - 1 - d] = n[d]
            phase = phase + (torch.arange(n[d], device=DEVICE, dtype=torch.float64) * waves[d]).view(view)
        x = torch.arange(n[0], device=DEVICE, dtype=torch.float64) * waves[0]
        amp = float(r.uniform(0.1, 0.22))
        phase = phase.reshape(shape[:-1] + [1])
        f.addcmul_(torch.sin(phase) * amp, torch.cos(x))
        f.addcmul_(torch.cos(phase) * amp, torch.sin(x))
    if box:
        edge = 0.1 ** (1.0 / dims)
        corner = f[tuple(slice(0, int(v * edge)) for v in shape)]
        corner.copy_(torch.rand(corner.shape, device=DEVICE, dtype=torch.float64, generator=g).mul_(2).sub_(1))
    return _typed(f, ztype)


def _memory(f, view):
    """The field as its view keeps it in memory (flat), the strides and the offset of element 0 of that view."""
    if view == "contiguous":
        return f.contiguous(), None, 0
    dims = f.dim()
    n = list(reversed(f.shape))
    # x slowest and reversed, the last axis fastest
    m = torch.flip(f.permute(*reversed(range(dims))), dims=[0]).contiguous()
    strides = [0] * dims
    step = 1
    for d in range(dims - 1, -1, -1):
        strides[d] = step
        step *= n[d]
    strides[0] = -strides[0]
    return m, strides, (n[0] - 1) * -strides[0]


def _source(case, seed):
    return _memory(_field(_extents(case), case["type"], seed, case["mode"] in ("precision", "accuracy")), case["view"])


def prepare(case, seed):
    if case["op"] == "batch":
        return _prepare_batch(case, seed)
    n = _extents(case)
    data, strides, first = _source(case, seed)
    params = _params(case["mode"], case["value"], case["type"], len(n))
    words = torch.zeros(Z.max_stream_words(ZTYPE[case["type"]], n, params), dtype=torch.int64, device=DEVICE)
    state = dict(op=case["op"], ztype=ZTYPE[case["type"]], n=n, strides=strides, params=params, words=words, offset=0,
                 data=data, at=data.data_ptr() + first * data.element_size())
    if case["op"] == "decompress":
        bits = Z.encode(state["ztype"], n, strides, state["at"], params, words.data_ptr())
        if not case["index"]:
            # the stream as a file holds it: a header, then exactly its words
            used = (bits + 63) // 64
            state["words"] = torch.zeros(HEADER_WORDS + used, dtype=torch.int64, device=DEVICE)
            state["words"][HEADER_WORDS:] = words[:used]
            state["offset"] = 64 * HEADER_WORDS
        state["data"] = torch.zeros_like(data)
        state["at"] = state["data"].data_ptr() + first * data.element_size()
    torch.cuda.synchronize()
    return state


def run(state):
    if state["op"] == "batch":
        bits_out = state["compress"].run()
        bits_in = state["decompress"].run()
        return [np.array(bits_out, dtype=np.int64), np.array(bits_in, dtype=np.int64), state["words"]] + state["arrays"]
    words = state["words"]
    if state["op"] == "compress":
        bits = Z.encode(state["ztype"], state["n"], state["strides"], state["at"], state["params"], words.data_ptr())
        return [bits, words]
    bits = Z.decode(state["ztype"], state["n"], state["strides"], state["at"], state["params"], words.data_ptr(),
                    offset=state["offset"], nwords=words.numel())
    return [bits, state["data"]]


def exact(case, seed):
    """Streams are whole numbers.  A decoded floating-point array stands for the array that was compressed:
    its values, in the same memory order."""
    if case["op"] == "compress":
        return None
    if case["op"] == "batch":
        values = _patches(case, seed)
        return [None, None, None] + [_pool(values, t).double() if t[0] == "f" else None for t in DTYPE]
    if case["type"][0] == "i":
        return None
    return [None, _source(case, seed)[0].double()]


# ---------------------------------------------------------------------------
# many arrays per call: patches of one to three axes, every type, two rates
# and two variable-length modes
# ---------------------------------------------------------------------------
PATCH_MODES = (("rate", 8), ("rate", 16), ("precision", 20), ("accuracy", 1e-4))


def _patch_specs(case):
    """(type, extents, mode) of every patch: the same mesh for every seed of its values."""
    r = np.random.default_rng(case["arrays"])
    specs = []
    for _ in range(case["arrays"]):
        dims = int(r.integers(1, 4))
        n = [int(round(math.exp(r.uniform(math.log(5), math.log(300))))) for _ in range(dims)]
        specs.append((list(DTYPE)[int(r.integers(0, 4))], n, PATCH_MODES[int(r.integers(0, 4))]))
    return specs


def _patches(case, seed):
    return [(t, n, mode, _field(n, t, seed * 4099 + k, False)) for k, (t, n, mode) in enumerate(_patch_specs(case))]


def _pool(patches, ztype):
    """The patches of one type as one flat buffer, each patch on a 64-byte boundary."""
    each = 64 * 8 // BITS[ztype]
    flat = [torch.nn.functional.pad(f.reshape(-1), (0, -f.numel() % each)) for t, _, _, f in patches if t == ztype]
    return torch.cat(flat) if flat else torch.zeros(0, dtype=DTYPE[ztype], device=DEVICE)


def _prepare_batch(case, seed):
    patches = _patches(case, seed)
    sources = {t: _pool(patches, t) for t in DTYPE}
    results = {t: torch.zeros_like(v) for t, v in sources.items()}
    plans = [_params(*mode, t, len(n)) for t, n, mode, _ in patches]
    caps = [Z.max_stream_words(ZTYPE[t], n, p) for (t, n, _, _), p in zip(patches, plans)]
    blocks = [math.prod((v + 3) // 4 for v in n) for _, n, _, _ in patches]
    words = torch.zeros(sum(caps), dtype=torch.int64, device=DEVICE)
    index = torch.zeros(sum(b + 1 for b in blocks), dtype=torch.int64, device=DEVICE)
    at = dict.fromkeys(DTYPE, 0)
    jobs = ([], [])
    w = i = 0
    for (t, n, _, f), p, cap, b in zip(patches, plans, caps, blocks):
        step = f.element_size()
        own = index.data_ptr() + 8 * i if p[0] != p[1] else None
        for job, pool in zip(jobs, (sources[t], results[t])):
            job.append(Z.make_job(ZTYPE[t], n, None, pool.data_ptr() + at[t] * step, p, words.data_ptr() + 8 * w, 0, cap,
                                  own))
        each = 64 // step
        at[t] += -(-f.numel() // each) * each
        w += cap
        i += b + 1
    torch.cuda.synchronize()
    return dict(op="batch", compress=Z.Batch(jobs[0], Z.ZFP_HIP_BATCH_COMPRESS),
                decompress=Z.Batch(jobs[1], Z.ZFP_HIP_BATCH_DECOMPRESS), words=words, index=index, sources=sources,
                arrays=list(results.values()))


# ---------------------------------------------------------------------------
# the bytes a pass cannot do without: the field once and its stream once
# ---------------------------------------------------------------------------
def _stream_bits(ztype, mode, value):
    """Bits per value of the fields above, to first order: a rate is exact; variable-length modes code the
    planes above the noise cheaply and about one bit per plane and value below it."""
    width = BITS[ztype]
    if mode == "rate":
        return float(value)
    if mode == "reversible":
        return 0.7 * width
    planes = value if mode == "precision" else 6 - math.log2(value)
    return min(float(width), max(0.5, 0.52 * (min(planes, width) - 8)))


def work(case):
    if case["op"] == "batch":
        values = stream = field = 0.0
        for t, n, mode in _patch_specs(case):
            v = math.prod(n)
            values += 2 * v
            field += 2 * v * BITS[t] / 8
            stream += 2 * v * _stream_bits(t, *mode) / 8
        return {"bytes": field + stream, "flops": values}
    n = _extents(case)
    v = math.prod(n)
    stream = v * _stream_bits(case["type"], case["mode"], case["value"])
    # one multiplication per value: the scale of its block
    return {"bytes": (v * BITS[case["type"]] + stream) / 8, "flops": float(v)}
