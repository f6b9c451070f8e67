"""The transforms whose speed this repository keeps track of, each through a public entry point.

A case is a dict of plain values.  Its "kind" names the entry point:

  plan    one execute of a ``Plan`` over a batch that is resident on the device;
  chain   ``Plan.chain``: m transforms, each scaled by 1/sqrt(V), the state ping-ponged;
  multi   one ``MultiPlan`` launch over several geometries;
  host    the host-pointer ABI (``fft3d_create`` / ``fft3d_execute``): the batch starts and
          ends in the caller's own host memory;
  serve   a burst of requests through a continuously batching ``Server``, submitted and waited
          for one by one.

listed() holds fixed cases, draw(rng) gives further ones of the same ranges, prepare / run
make and run one, work(case) counts the bytes and flops that one run cannot do without, and
exact(case, seed) is the result in 64 bits from torch.fft alone.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """opt-fft_amd/ (not a Python identifier) loaded as the module ``optfft_amd``."""
    if "optfft_amd" not in sys.modules:
        path = os.path.join(ROOT, "opt-fft_amd")
        spec = importlib.util.spec_from_file_location(
            "optfft_amd", os.path.join(path, "__init__.py"), submodule_search_locations=[path])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["optfft_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["optfft_amd"]


# Every geometry the library serves; the first five also run in mixed launches and on the
# matrix cores.
FUSED = ["6x6x6", "8x8x8", "12x12x12", "17x17x17", "8x8x16"]
GEOMS = FUSED + ["24x24x24", "36x36x36", "24x24x48"]
CUBES = [6, 8, 12, 17, 24, 36]
MOST_BYTES = 400 << 20       # input bytes of a drawn batch, below the mixed launch's 441 MB
FEW_BYTES = 4 << 20
MOST_BATCH = 65536


def _shape(text):
    return tuple(int(n) for n in text.split("x"))


def _elem(prec):
    return 16 if prec == "c128" else 8


def listed():
    return [
        # One volume at a time: the latency of a solver that transforms a field per step.
        dict(name="l17_c128_b1_bwd", kind="plan", shape="17x17x17", batch=1, prec="c128",
             direction=1, normalize=True, matrix="", dist="uniform"),
        # A handful of the largest cube: the common request of the serving mix at low load.
        dict(name="l36_c128_b5", kind="plan", shape="36x36x36", batch=5, prec="c128",
             direction=-1, normalize=False, matrix="", dist="normal"),
        # The benchmark's batches in double precision.
        dict(name="l8_c128_b4096", kind="plan", shape="8x8x8", batch=4096, prec="c128",
             direction=-1, normalize=False, matrix="", dist="uniform"),
        dict(name="l17_c128_b1024", kind="plan", shape="17x17x17", batch=1024, prec="c128",
             direction=-1, normalize=False, matrix="", dist="uniform"),
        dict(name="l36_c128_b128", kind="plan", shape="36x36x36", batch=128, prec="c128",
             direction=-1, normalize=False, matrix="", dist="normal"),
        dict(name="24x24x48_c128_b64", kind="plan", shape="24x24x48", batch=64, prec="c128",
             direction=-1, normalize=False, matrix="", dist="normal"),
        # Ragged batches, backward: the return leg of a convolution.
        dict(name="l24_c128_b365_bwd", kind="plan", shape="24x24x24", batch=365, prec="c128",
             direction=1, normalize=True, matrix="", dist="uniform"),
        dict(name="l36_c64_b255_bwd", kind="plan", shape="36x36x36", batch=255, prec="c64",
             direction=1, normalize=True, matrix="", dist="uniform"),
        # Uneven batches of four geometries in one launch: single precision, and the
        # split-bf16 matrix-core form.
        dict(name="mix_c64", kind="multi", prec="c64", direction=-1, normalize=False, matrix="",
             items="6x6x6*65536,8x8x8*32768,12x12x12*8192,17x17x17*2048"),
        dict(name="mix_c64_bf16x3", kind="multi", prec="c64", direction=-1, normalize=False,
             matrix="bf16", items="6x6x6*65536,8x8x8*32768,12x12x12*8192,17x17x17*2048"),
        # A C program that keeps its field in host memory.
        dict(name="host_l17_b1024", kind="host", L=17, batch=1024),
        # Requests of the serving mix that arrive while others run.
        dict(name="serve_burst_48", kind="serve", requests=48, mix_seed=0),
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _most(shape, prec, limit=MOST_BYTES):
    n = _shape(shape)
    return max(1, min(MOST_BATCH, limit // (n[0] * n[1] * n[2] * _elem(prec))))


def draw(rng):
    kind = rng.choice(["plan"] * 7 + ["chain", "multi", "multi", "host", "serve"])
    if kind == "host":
        L = rng.choice(CUBES)
        return dict(kind="host", L=L, batch=_log_uniform(rng, 1, _most(f"{L}x{L}x{L}", "c128", 76 << 20)))
    if kind == "serve":
        while True:              # a burst no larger than the listed one
            case = dict(kind="serve", requests=rng.randint(4, 40), mix_seed=rng.randrange(1 << 16))
            if work(case)["bytes"] <= 1200 << 20:
                return case
    prec = "c128" if rng.random() < 0.6 else "c64"
    if kind == "multi":
        matrix = rng.choice(["", "", "bf16", "fp16"]) if prec == "c64" else ""
        some = rng.sample(FUSED, rng.randint(2, 5))
        items = ",".join("%s*%d" % (s, _log_uniform(rng, 1, _most(s, prec, 96 << 20)))
                         for s in some)
        return dict(kind="multi", prec=prec, direction=rng.choice([-1, 1]),
                    normalize=rng.random() < 0.5, matrix=matrix, items=items)
    shape = rng.choice(GEOMS)
    matrix = ""
    if kind == "plan" and prec == "c64" and shape in FUSED and rng.random() < 0.3:
        matrix = rng.choice(["bf16", "fp16"])
    # A single execute of less than FEW_BYTES takes under 5 us, most of it the launch: such
    # batches are drawn as chains, and the matrix-core ones from there upwards.
    steps = rng.randint(2, 4)
    batch = _log_uniform(rng, _most(shape, prec, FEW_BYTES) if matrix else 1,
                         _most(shape, prec, MOST_BYTES // (steps if kind == "chain" else 1)))
    if batch < _most(shape, prec, FEW_BYTES) and shape in FUSED:
        kind = "chain"
    case = dict(kind=kind, shape=shape, prec=prec, direction=rng.choice([-1, 1]), batch=batch,
                dist=rng.choice(["uniform", "normal"]))
    if kind == "chain":
        case["steps"] = steps
    else:
        case.update(normalize=rng.random() < 0.5, matrix=matrix)
    return case


# Inputs, on the device, from the seed alone: real and imaginary parts iid uniform(-1, 1), or
# standard complex normal (variance 1/2 each).
def _field(seed, k, batch, shape, prec, dist):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 4096 + k)
    real = torch.float64 if prec == "c128" else torch.float32
    size = (batch,) + _shape(shape) + (2,)
    if dist == "normal":
        x = torch.randn(size, generator=g, device="cuda", dtype=real).mul_(math.sqrt(0.5))
    else:
        x = torch.rand(size, generator=g, device="cuda", dtype=real).mul_(2).sub_(1)
    return torch.view_as_complex(x)


def _host_field(case, seed):
    L = case["L"]
    x = np.random.default_rng(seed).uniform(-1, 1, (case["batch"], L, L, L, 2))
    return x.view(np.complex128)[..., 0]


def _items(case):
    for part in case["items"].split(","):
        shape, batch = part.split("*")
        yield shape, int(batch)


def _requests(case):
    """[(shape text, batch, direction, precision text)] of the serving mix."""
    f = _package().fft3d
    for shape, batch, direction, prec in _package().serving.draw_mix(case["requests"],
                                                                    case["mix_seed"]):
        yield "x".join(map(str, shape)), batch, direction, "c128" if prec == f.C128 else "c64"


def _inputs(case, seed):
    if case["kind"] == "host":
        return [_host_field(case, seed)]
    if case["kind"] == "multi":
        return [_field(seed, k, b, s, case["prec"], "uniform")
                for k, (s, b) in enumerate(_items(case))]
    if case["kind"] == "serve":
        return [_field(seed, k, b, s, p, "uniform")
                for k, (s, b, _, p) in enumerate(_requests(case))]
    return [_field(seed, 0, case["batch"], case["shape"], case["prec"], case["dist"])]


def prepare(case, seed):
    f = _package().fft3d
    kind = case["kind"]
    ins = _inputs(case, seed)
    if kind == "host":
        lib = f.load()
        return dict(kind=kind, x=ins[0], y=np.empty_like(ins[0]),
                    plan=_HostPlan(lib, case["L"], case["batch"]))
    outs = [torch.empty_like(x) for x in ins]
    state = dict(kind=kind, ins=ins, outs=outs, stream=torch.cuda.current_stream().cuda_stream)
    if kind == "serve":
        state["server"] = f.Server(budget_bytes=4 << 30, streams=16, batched=True, max_items=16,
                                   window_us=30.0)
        state["requests"] = [(_shape(s), b, d, f.C128 if p == "c128" else f.C64)
                             for s, b, d, p in _requests(case)]
        torch.cuda.synchronize()       # the server's streams do not follow torch's
        return state
    prec = f.C128 if case["prec"] == "c128" else f.C64
    flags = f.NORMALIZE if case.get("normalize") else 0
    flags |= {"": 0, "bf16": f.MFMA_BF16, "fp16": f.MFMA_FP16}[case.get("matrix", "")]
    if kind == "multi":
        state["plan"] = f.MultiPlan([(_shape(s), b, case["direction"]) for s, b in _items(case)],
                                    prec, flags)
        return state
    shape = _shape(case["shape"])
    state["plan"] = f.Plan(shape, case["batch"], case["direction"], prec, flags)
    if kind == "chain":
        state["pong"] = torch.empty_like(ins[0])
        state["steps"] = case["steps"]
        state["scale"] = 1.0 / math.sqrt(shape[0] * shape[1] * shape[2])
    return state


class _HostPlan:
    """fft3d_create / fft3d_execute / fft3d_destroy, as a C program calls them."""

    def __init__(self, lib, L, batch):
        self.lib, self.handle = lib, lib.fft3d_create(L, batch)
        if not self.handle:
            raise RuntimeError("fft3d_create failed")

    def execute(self, x, y):
        self.lib.fft3d_execute(self.handle, x.ctypes.data, y.ctypes.data)

    def __del__(self):
        if getattr(self, "handle", None):
            self.lib.fft3d_destroy(self.handle)
            self.handle = None


def run(state):
    kind = state["kind"]
    if kind == "host":
        state["plan"].execute(state["x"], state["y"])
        return state["y"]
    ins, outs = state["ins"], state["outs"]
    if kind == "plan":
        state["plan"].execute(ins[0].data_ptr(), outs[0].data_ptr(), stream=state["stream"])
        return outs[0]
    if kind == "chain":
        state["plan"].chain(ins[0].data_ptr(), outs[0].data_ptr(), state["pong"].data_ptr(),
                            state["steps"], state["scale"], stream=state["stream"])
        return outs[0]
    if kind == "multi":
        state["plan"].execute([x.data_ptr() for x in ins], [y.data_ptr() for y in outs],
                              stream=state["stream"])
        return outs
    server = state["server"]
    ids = [server.submit(s, b, d, p, x.data_ptr(), y.data_ptr())
           for (s, b, d, p), x, y in zip(state["requests"], ins, outs)]
    for i in ids:
        server.wait(i)
    return outs


def _parts(case):
    """(shape, batch, precision, transforms) of everything one run transforms."""
    kind = case["kind"]
    if kind == "host":
        L = case["L"]
        return [((L, L, L), case["batch"], "c128", 1)]
    if kind == "multi":
        return [(_shape(s), b, case["prec"], 1) for s, b in _items(case)]
    if kind == "serve":
        return [(_shape(s), b, p, 1) for s, b, _, p in _requests(case)]
    return [(_shape(case["shape"]), case["batch"], case["prec"], case.get("steps", 1))]


def work(case):
    """Each transform reads its batch once and writes it once; 5 V log2 V flops a volume."""
    total, flops = 0, 0.0
    for (a, b, c), batch, prec, times in _parts(case):
        V = a * b * c
        total += 2 * V * batch * _elem(prec) * times
        flops += 5.0 * V * math.log2(V) * batch * times
    return {"bytes": total, "flops": flops}


def _dft(x, direction, normalize):
    dims = (-3, -2, -1)
    if direction < 0:
        y = torch.fft.fftn(x, dim=dims)
        return y / (x.shape[-3] * x.shape[-2] * x.shape[-1]) if normalize else y
    return torch.fft.ifftn(x, dim=dims, norm="backward" if normalize else "forward")


def exact(case, seed):
    xs = [torch.as_tensor(x).cpu().to(torch.complex128) for x in _inputs(case, seed)]
    kind = case["kind"]
    if kind == "host":
        return _dft(xs[0], -1, False).numpy()
    if kind == "plan":
        return _dft(xs[0], case["direction"], case["normalize"])
    if kind == "chain":
        x = xs[0]
        for _ in range(case["steps"]):
            x = _dft(x, case["direction"], False)
            x /= math.sqrt(x.shape[-3] * x.shape[-2] * x.shape[-1])
        return x
    if kind == "multi":
        return [_dft(x, case["direction"], case["normalize"]) for x in xs]
    return [_dft(x, d, False) for x, (_, _, d, _) in zip(xs, _requests(case))]
