"""Workloads of the codec, each one pass through the package's public entry points.

A case is a dict of plain values.  ``path`` names what a program does:

* ``compress``   one device field through ``DeviceCompressor`` (stream, record
                 index and result words stay on the device; nothing waits)
* ``decode``     a stream that still has its record index, through
                 ``DeviceDecompressor`` (a program that compressed the field
                 itself and kept the index beside the stream)
* ``restore``    a stream alone, as read back from a file or received from
                 another program: no record index
* ``roundtrip``  compress, learn the stream's size, decode: a program that
                 checks or replays what it stored.  Used for the block sizes
                 that are not powers of two
* ``nonblocked`` the same for fastMode 1, one record over the whole array
* ``batch``      many fields of mixed size and type through ``BatchCodec``,
                 both directions
* ``fixed_rate`` one field to a target number of bits per value, with the
                 learned proposer
* ``host``       the drop-in C API on host arrays, both directions

The other keys are ``shape`` (extents, slowest first), ``dtype``, ``field``
(the kind of data, see szx_amd.fields), ``bs`` (block size), ``mode`` ("abs" or
"rel"), ``rel`` (the bound over the value range), ``fast_mode``, and for
``batch`` the number of fields and the largest one's bytes.

Decoded values are returned as their bit patterns: the format fixes every bit
of a decode, as it fixes every byte of a stream.
"""
import math

import numpy as np
import torch

import szx_amd as Z
from szx_amd.fields import grf_field_torch, sinusoid_field_torch

MIB = 1 << 20


def listed():
    return [
        # the smallest call: one small patch of a simulation, where launches and host calls count
        dict(name="compress_f32_16x40x40_rel", path="compress", shape="16x40x40", dtype="float32", field="waves",
             bs=128, mode="rel", rel=1e-3, fast_mode=2),
        # an ordinary 3D snapshot with an absolute bound known beforehand (no range pass)
        dict(name="compress_f32_100x500x500_abs", path="compress", shape="100x500x500", dtype="float32",
             field="waves", bs=128, mode="abs", rel=1e-3, fast_mode=2),
        # a large snapshot, the bound relative to its range: the headline workload
        dict(name="compress_f32_512x512x512_rel", path="compress", shape="512x512x512", dtype="float32",
             field="waves", bs=128, mode="rel", rel=1e-3, fast_mode=2),
        # a large double field of wide dynamic range with denormal-scale entries
        dict(name="compress_f64_8192x8192_rel", path="compress", shape="8192x8192", dtype="float64", field="grf",
             bs=64, mode="rel", rel=1e-6, fast_mode=2),
        # the same two fields back, with the index the compressor left
        dict(name="decode_f32_512x512x512", path="decode", shape="512x512x512", dtype="float32", field="waves",
             bs=128, mode="rel", rel=1e-3, fast_mode=2),
        dict(name="decode_f64_8192x8192", path="decode", shape="8192x8192", dtype="float64", field="grf", bs=64,
             mode="rel", rel=1e-6, fast_mode=2),
        # a stream read from a file: its records have to be located first
        dict(name="restore_f32_100x500x500", path="restore", shape="100x500x500", dtype="float32", field="waves",
             bs=128, mode="rel", rel=1e-3, fast_mode=2),
        # a block size chosen to match the data's row length (100)
        dict(name="roundtrip_f32_256x256x256_bs100", path="roundtrip", shape="256x256x256", dtype="float32",
             field="waves", bs=100, mode="rel", rel=1e-3, fast_mode=2),
        # the non-blocked mode, for smooth data without constant regions
        dict(name="nonblocked_f32_256x256x256", path="nonblocked", shape="256x256x256", dtype="float32",
             field="waves", bs=0, mode="rel", rel=1e-3, fast_mode=1),
        # one output step of a multi-field application: sizes log-uniform from 64 KiB, 60 % fp32, own bounds
        dict(name="batch_30_fields_64MiB", path="batch", fields=30, max_bytes=64 * MIB, bs=128),
        # a storage quota: 4 bits per value, whatever bound that takes
        dict(name="fixed_rate_f32_256x256x256_4bpv", path="fixed_rate", shape="256x256x256", dtype="float32",
             field="spectral", bs=128, bpv=4.0),
        # an existing C caller's host arrays, both directions, transfers included
        dict(name="host_f32_100x500x500_abs", path="host", shape="100x500x500", dtype="float32", field="waves",
             bs=128, mode="abs", rel=1e-3, fast_mode=2),
    ]


def _shape(rng, values):
    """Random 3D extents, odd ones among them, with about `values` cells and no more."""
    a = max(1, int(values ** rng.uniform(0.2, 0.4)))
    b = max(1, int((values / a) ** rng.uniform(0.4, 0.6)))
    c = max(1, int(values / (a * b)))
    return "%dx%dx%d" % (a, b, c)


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    path = rng.choice(["compress", "compress", "decode", "decode", "restore", "roundtrip", "nonblocked", "batch",
                       "fixed_rate", "host"])
    if path == "batch":
        return dict(path=path, fields=rng.randint(4, 30), max_bytes=int(_log(rng, MIB, 64 * MIB)), bs=128)
    dtype = rng.choice(["float32", "float32", "float64"])
    w = 4 if dtype == "float32" else 8
    if path == "fixed_rate":
        return dict(path=path, shape=_shape(rng, _log(rng, MIB, 16 * MIB)), dtype="float32", field="spectral", bs=128,
                    bpv=rng.choice([1.0, 2.0, 4.0, 8.0]))
    top = {"compress": 512, "decode": 512, "restore": 512, "roundtrip": 64, "nonblocked": 64, "host": 64}[path] * MIB
    rel = _log(rng, 1e-5, 1e-2) if w == 4 else _log(rng, 1e-8, 1e-4)
    c = dict(path=path, shape=_shape(rng, _log(rng, 100 * 1024, top) / w), dtype=dtype, field="waves",
             bs=rng.choice([32, 64, 128, 128, 128, 256]), mode=rng.choice(["abs", "rel"]), rel=float("%.3g" % rel),
             fast_mode=2)
    if path in ("compress", "restore"):
        c["fast_mode"] = rng.choice([2, 2, 2, 4])   # 4: the random-access container
    elif path == "roundtrip":
        c["bs"] = rng.choice([20, 50, 100, 125, 200, 250])
    elif path == "nonblocked":
        c["bs"], c["fast_mode"] = 0, 1
    elif path == "host":
        c["bs"] = 128   # the drop-in call's own block size
    return c


def _extents(case):
    return tuple(int(s) for s in case["shape"].split("x"))


def _values(case):
    return math.prod(_extents(case))


def _bytes(dtype):
    return 4 if dtype == "float32" else 8


def _field(case, seed):
    """The case's field on the GPU, flat."""
    shape, dtype = _extents(case), case["dtype"]
    if case["field"] == "grf":
        x = grf_field_torch(shape, seed, dtype=dtype)
    elif case["field"] == "spectral":   # slope and noise level differ from field to field
        r = np.random.default_rng([seed, 1])
        x = sinusoid_field_torch(shape, seed, n_waves=32, kmax=16, slope=r.uniform(1.5, 4.0),
                                 noise=10 ** r.uniform(-6, -2), n_boxes=1, box_frac=0.25, box_value="zero",
                                 dtype=dtype)
    elif _values(case) >= 64 * MIB:
        x = sinusoid_field_torch(shape, seed, dtype=dtype)
    else:
        x = sinusoid_field_torch(shape, seed, n_waves=32, kmax=16, slope=2.0, noise=1e-3, n_boxes=1, box_frac=0.25,
                                 box_value="zero", dtype=dtype)
    return x.reshape(-1).contiguous()


def _bound(case, x):
    """(errBoundMode, keyword arguments) of the case's bound; an absolute one is known before the call."""
    if case["mode"] == "rel":
        return Z.REL, dict(relBoundRatio=case["rel"])
    return Z.ABS, dict(absErrBound=float(np.float32(float(x.max() - x.min()) * case["rel"])))


def _compressor(case, x):
    comp = Z.DeviceCompressor(x.numel(), case["dtype"], case["bs"], fastMode=case["fast_mode"])
    comp.out.zero_()   # bytes outside the stream are not written
    return comp


def _batch_fields(case, seed):
    """Fields with log-uniform sizes, 60 % fp32, each with its own REL bound."""
    r = np.random.default_rng(seed)
    sizes = np.random.default_rng([case["fields"], case["max_bytes"]])   # one seed's work is another's
    out = []
    for i in range(case["fields"]):
        dtype = "float32" if sizes.random() < 0.6 else "float64"
        nbytes = 65536 * (case["max_bytes"] / 65536) ** sizes.random()
        values = nbytes / _bytes(dtype)
        a = max(1, int(values ** sizes.uniform(0.2, 0.4)))
        b = max(1, int((values / a) ** sizes.uniform(0.4, 0.6)))
        shape = (a, b, max(1, int(values / (a * b))))
        x = sinusoid_field_torch(shape, int(r.integers(1 << 30)), n_waves=32, kmax=16, slope=2.0, noise=1e-3,
                                 n_boxes=1, box_frac=0.25, box_value="zero", dtype=dtype)
        out.append((x.reshape(-1).contiguous(), Z.REL, float(10 ** sizes.uniform(-5, -2))))
    return out


def prepare(case, seed):
    path = case["path"]
    if path == "batch":
        codec = Z.BatchCodec(_batch_fields(case, seed), case["bs"])
        for o in codec.outs:
            o.zero_()
        return dict(path=path, codec=codec)
    x = _field(case, seed)
    n = x.numel()
    if path == "fixed_rate":
        comp = Z.FixedRateCompressor(n, case["dtype"], case["bs"], model=Z.RateModel())
        return dict(path=path, x=x, comp=comp, bpv=case["bpv"], slot=torch.zeros_like(comp.out))
    mode, bound = _bound(case, x)
    s = dict(path=path, mode=mode, bound=bound)
    if path == "host":
        s.update(x=x.cpu().numpy().reshape(_extents(case)), fast_mode=case["fast_mode"],
                 slot=np.zeros(Z.lib().szx_amd_compress_bound(n, Z._dtype_code(case["dtype"]), case["bs"]), np.uint8))
        return s
    if path == "nonblocked":
        codec = Z.DeviceNonBlocked(n, case["dtype"])
        codec.out.zero_()
        s.update(x=x, codec=codec)
        return s
    comp = _compressor(case, x)
    s.update(x=x, comp=comp)
    if path == "roundtrip":
        s["dec"] = Z.DeviceDecompressor(n, case["dtype"], case["bs"], comp.capacity)
    if path in ("decode", "restore"):
        comp(x, mode, **bound)
        stream, _, size, _ = comp.stream_view()
        s = dict(path=path, stream=stream.clone(), index=comp.index if path == "decode" else None,
                 dec=Z.DeviceDecompressor(n, case["dtype"], case["bs"], size, fastMode=case["fast_mode"]))
    return s


def _bits(t):
    return t.view(torch.int32 if t.dtype == torch.float32 else torch.int64)


def run(s):
    path = s["path"]
    if path == "compress":
        s["comp"](s["x"], s["mode"], **s["bound"])
        return [s["comp"].out, s["comp"].index, s["comp"].result]
    if path in ("decode", "restore"):
        s["dec"](s["stream"], index=s["index"])
        return [_bits(s["dec"].out), s["dec"].status]
    if path == "roundtrip":
        s["comp"](s["x"], s["mode"], **s["bound"])
        stream, _, size, _ = s["comp"].stream_view()
        s["dec"](stream, size, index=s["comp"].index)
        return [s["comp"].out, s["comp"].index, _bits(s["dec"].out), s["dec"].status]
    if path == "nonblocked":
        s["codec"].compress(s["x"], s["mode"], **s["bound"])
        stream, size, _ = s["codec"].stream_view()
        s["codec"].decompress(stream, size)
        return [s["codec"].out, _bits(s["codec"].dec), s["codec"].status]
    if path == "batch":
        s["codec"].compress()
        s["codec"].decompress()
        return s["codec"].outs + [_bits(d) for d in s["codec"].decs] + [s["codec"].status()]
    if path == "fixed_rate":
        s["comp"](s["x"], s["bpv"])
        stream = s["comp"].stream_view()
        s["slot"][:stream.numel()] = stream   # the field's place among a file's records
        return [s["slot"], s["comp"].result]
    stream = Z.SZx_fast_compress_args(s["fast_mode"], s["x"], s["mode"], **s["bound"])
    back = Z.SZx_fast_decompress(s["fast_mode"], s["x"].dtype, stream, s["x"].shape)
    s["slot"][:len(stream)] = np.frombuffer(stream, np.uint8)   # the program's own output block
    return [s["slot"], len(stream), back.view(np.int32 if back.dtype == np.float32 else np.int64)]


def _stream_bytes(values, rel):
    """A stream's size, near enough: about 0.95 log2(1 / rel) bits per value on these fields."""
    return values * 0.95 * math.log2(1 / rel) / 8


def work(case):
    """Each input read once, each output written once."""
    path = case["path"]
    if path == "batch":
        sizes = [(x, r) for x, r in _batch_work(case)]
        return {"bytes": 2 * sum(b + c for b, c in sizes), "flops": 0}
    n, w = _values(case), _bytes(case["dtype"])
    if path == "fixed_rate":
        return {"bytes": n * w + n * case["bpv"] / 8, "flops": 0}
    one_way = n * w + _stream_bytes(n, case["rel"])
    return {"bytes": one_way * (2 if path in ("roundtrip", "nonblocked", "host") else 1), "flops": 0}


def _batch_work(case):
    """(field bytes, stream bytes) of every field, with the sizes and bounds that _batch_fields draws."""
    sizes = np.random.default_rng([case["fields"], case["max_bytes"]])
    for _ in range(case["fields"]):
        w = 4 if sizes.random() < 0.6 else 8
        values = int(65536 * (case["max_bytes"] / 65536) ** sizes.random() / w)
        sizes.uniform(0.2, 0.4), sizes.uniform(0.4, 0.6)
        yield values * w, _stream_bytes(values, 10 ** sizes.uniform(-5, -2))
