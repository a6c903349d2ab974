"""Performance cases of the tensor-bundle path, each one pass of a program that uses it.

A bundle is packed (N tensors -> one payload and a header) and unpacked (payload -> N tensors).
`fresh` paths see their tensors for the first time in every pass, as an RPC does: describe, plan,
pack, decode the header, bind, unpack, release.  `kept` paths hold their plans, as a training or
serving loop that moves the same tensors again and again does.
"""
import functools
import math
import random

import numpy as np
import torch

import __graft_entry__

axon = __graft_entry__.load_package()
from execution_ucx_amd import workloads  # noqa: E402  (the package is importable once it is loaded)
from execution_ucx_amd import _capi  # noqa: E402

MIB = 1 << 20


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the tensor arguments of one call: four tensors of 64 KiB, new in every call
        {"name": "call_arguments", "path": "fresh", "tensors": 4, "lo": 65536, "hi": 65536, "align": 256, "sizes": 1},
        # 64 host arrays of 16,384 fp32 to a device payload and back into host arrays
        {"name": "host_arguments", "path": "host", "tensors": 64, "lo": 65536, "hi": 65536, "align": 256, "sizes": 1},
        # parameters and states of a model's small layers, sent once: 4096 tensors of 256 B to
        # 64 KiB in the tight layout
        {"name": "mixed_once", "path": "fresh", "tensors": 4096, "lo": 256, "hi": 65536, "align": 1, "sizes": 0},
        # the same mix as the steady state of a worker: one bundle packed and another one, received
        # before, unpacked, handed over together
        {"name": "mixed_steady", "path": "submit", "tensors": 4096, "lo": 256, "hi": 65536, "align": 256, "sizes": 0},
        # one transformer layer's bf16 weights handed to another worker
        {"name": "layer_weights", "path": "layer", "hidden": 4096, "ffn": 11008, "align": 256},
        # cache blocks of a request moved between two KV caches: strided views of every layer
        {"name": "cache_blocks", "path": "cache", "layers": 32, "blocks": 4096, "picks": 512, "tokens": 16, "heads": 8, "dim": 128,
         "align": 256},
        # a payload too large for one message, streamed in chunks of pitched views
        {"name": "streamed_chunks", "path": "stream", "chunks": 8, "views": 64, "rows": 1024, "cols": 2048, "align": 256},
        # transposed matrices whose rows do not start on lines
        {"name": "transposed_odd", "path": "transposed", "matrices": 4, "rows": 4097, "cols": 4099, "item": 2, "align": 256},
        # a batch of interleaved images sent channel by channel
        {"name": "image_planes", "path": "images", "images": 256, "height": 224, "width": 224, "channels": 3, "item": 1, "align": 256},
        # the leading columns of a wide table: rows of 250 bytes at a 1 KiB pitch
        {"name": "row_slices", "path": "rows", "rows": 1 << 20, "cols": 125, "pitch": 512, "item": 2, "align": 256},
        # very many short tensors (norm scales, biases, optimizer scalars), sent once
        {"name": "short_once", "path": "fresh", "tensors": 65536, "lo": 8, "hi": 512, "align": 256, "sizes": 3},
        # and moved again and again in the tight layout
        {"name": "short_steady", "path": "kept", "tensors": 65536, "lo": 8, "hi": 512, "align": 1, "sizes": 3},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["call", "host", "mixed_once", "mixed_steady", "layer", "cache", "stream", "transposed", "images", "rows",
                       "short_once", "short_steady"])
    align = rng.choice([1, 64, 256])
    sizes = rng.randrange(1 << 20)
    if kind == "call":
        lo = _log(rng, 64, 65536)
        return {"path": "fresh", "tensors": _log(rng, 1, 64), "lo": lo, "hi": _log(rng, lo, 65536), "align": align, "sizes": sizes}
    if kind == "host":
        lo = _log(rng, 1024, 65536)
        return {"path": "host", "tensors": _log(rng, 1, 64), "lo": lo, "hi": _log(rng, lo, 65536), "align": align, "sizes": sizes}
    if kind in ("mixed_once", "mixed_steady"):
        return {"path": "fresh" if kind == "mixed_once" else "submit", "tensors": _log(rng, 128, 4096), "lo": 256, "hi": 65536,
                "align": align, "sizes": sizes}
    if kind == "layer":
        hidden = 128 * rng.randint(8, 32)
        return {"path": "layer", "hidden": hidden, "ffn": min(11008, hidden * rng.choice([2, 3, 4]) - rng.choice([0, 32, 8])),
                "align": align}
    if kind == "cache":
        blocks = _log(rng, 128, 4096)
        return {"path": "cache", "layers": _log(rng, 4, 32), "blocks": blocks, "picks": _log(rng, 8, blocks // 8),
                "tokens": rng.choice([8, 16]), "heads": rng.choice([1, 2, 4, 8]), "dim": rng.choice([64, 128]), "align": align}
    if kind == "stream":
        return {"path": "stream", "chunks": rng.randint(2, 8), "views": rng.randint(8, 64), "rows": _log(rng, 128, 1024),
                "cols": _log(rng, 512, 2048), "align": align}
    if kind == "transposed":
        item = rng.choice([1, 2, 2, 4, 8])
        edge = 4096 if item < 8 else 2900
        return {"path": "transposed", "matrices": rng.randint(1, 4 if item <= 2 else 2), "rows": _log(rng, 257, edge), "cols": _log(rng, 257, edge),
                "item": item, "align": align}
    if kind == "images":
        return {"path": "images", "images": _log(rng, 8, 256), "height": rng.randint(64, 224), "width": rng.randint(64, 224),
                "channels": rng.choice([3, 3, 4]), "item": rng.choice([1, 1, 2, 4]), "align": align}
    if kind == "rows":
        item = rng.choice([1, 2, 4])
        cols = _log(rng, 64, 1024) // item
        return {"path": "rows", "rows": _log(rng, 1 << 14, 1 << 18), "cols": cols, "pitch": int(cols * rng.uniform(1.2, 4.0)) + 1,
                "item": item, "align": align}
    if kind == "short_once":
        return {"path": "fresh", "tensors": _log(rng, 1024, 65536), "lo": 8, "hi": 512, "align": align, "sizes": sizes}
    return {"path": "kept", "tensors": _log(rng, 4096, 65536), "lo": 8, "hi": 512, "align": align, "sizes": sizes}


# ---------------------------------------------------------------- inputs

_BITS = {1: torch.uint8, 2: torch.bfloat16, 4: torch.float32, 8: torch.float64}


@functools.lru_cache(maxsize=4)
def _mixed(tensors, lo, hi, sizes):
    if lo == hi:    # equal sizes: fp32 tensors
        segs = [workloads.Segment((2, 32, 1), "float32", lo, i * ((lo + 255) // 256 * 256)) for i in range(tensors)]
        return workloads.MixedBundle(segs, tensors * ((lo + 255) // 256 * 256), tensors * lo)
    return workloads.mixed_bundle(n=tensors, lo=lo, hi=hi, seed=sizes)


def _spec(case):
    return _mixed(case["tensors"], case["lo"], case["hi"], case["sizes"])


def _carve(arena, spec):
    at = {name: getattr(torch, name) for name in {s.dtype_name for s in spec.segments}}
    return [arena[s.arena_offset:s.arena_offset + s.nbytes].view(at[s.dtype_name]) for s in spec.segments]


def _random_bytes(nbytes, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randint(0, 256, (nbytes,), dtype=torch.uint8, device="cuda", generator=g)


def _normal(shape, scale, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, scale, generator=g)


def _layer_shapes(case):
    h, f = case["hidden"], case["ffn"]
    return [(h, h)] * 4 + [(f, h), (f, h), (h, f), (h,), (h,)]


def _view_state(case, seed):
    """(storage of the sources, views of it, storage of the destinations, views of that)"""
    path, item = case["path"], case.get("item", 2)
    if path == "transposed":
        per = case["rows"] * case["cols"]
        src = _random_bytes(case["matrices"] * per * item, seed)
        dst = torch.zeros_like(src)

        def views(store):
            return [m.t() for m in store.view(_BITS[item]).view(case["matrices"], case["rows"], case["cols"])]
    elif path == "images":
        shape = (case["images"], case["height"], case["width"], case["channels"])
        src = _random_bytes(math.prod(shape) * item, seed)
        dst = torch.zeros_like(src)

        def views(store):
            return [store.view(_BITS[item]).view(shape).permute(0, 3, 1, 2)]
    else:
        src = _random_bytes(case["rows"] * case["pitch"] * item, seed)
        dst = torch.zeros_like(src)

        def views(store):
            return [store.view(_BITS[item]).view(case["rows"], case["pitch"])[:, :case["cols"]]]
    return src, views(src), dst, views(dst)


def prepare(case, seed):
    path = case["path"]
    state = {"path": path, "align": case["align"]}
    if path in ("fresh", "kept", "submit"):
        spec = _spec(case)
        src = _random_bytes(spec.arena_bytes, seed)
        dst = torch.zeros_like(src)
        state.update(keep=src, src=_carve(src, spec), out=dst, dst=_carve(dst, spec))
    elif path == "host":
        spec = _spec(case)
        rng = np.random.default_rng(seed)
        src = rng.uniform(-1.0, 1.0, size=spec.arena_bytes // 4).astype(np.float32).view(np.uint8)
        dst = np.zeros_like(src)

        def carve(arena):
            return [arena[s.arena_offset:s.arena_offset + s.nbytes // 4 * 4].view(np.float32) for s in spec.segments]
        state.update(keep=src, src=carve(src), out=dst, dst=carve(dst))
    elif path == "layer":
        src = [_normal(s, 0.02, seed * 64 + i) for i, s in enumerate(_layer_shapes(case))]
        dst = [torch.zeros_like(t) for t in src]
        state.update(src=src, out=dst, dst=dst)
    elif path == "cache":
        shape = (case["layers"], 2, case["blocks"], case["tokens"], case["heads"], case["dim"])
        src, dst = _normal(shape, 1.0, seed), torch.zeros(shape, dtype=torch.bfloat16, device="cuda")
        rng = random.Random(seed)
        take, put = (rng.sample(range(case["blocks"]), case["picks"]) for _ in range(2))
        state.update(keep=src, src=[src[:, :, b] for b in take], out=dst, dst=[dst[:, :, b] for b in put])
    elif path == "stream":
        pitch = case["cols"] * 3 // 2
        shape = (case["chunks"], case["views"], case["rows"], pitch)
        src, dst = _normal(shape, 1.0, seed), torch.zeros(shape, dtype=torch.bfloat16, device="cuda")
        state.update(keep=src, out=dst,
                     src=[[v[:, :case["cols"]] for v in chunk] for chunk in src],
                     dst=[[v[:, :case["cols"]] for v in chunk] for chunk in dst],
                     transfer=axon.StreamedTransfer(_payload_bound(case), align=case["align"]))
    else:
        src, sv, dst, dv = _view_state(case, seed)
        state.update(keep=src, src=sv, out=dst, dst=dv)
    if path in ("kept", "submit", "transposed", "images", "rows"):
        # plans and payload buffers that the program keeps from one pass to the next
        send = axon.BundlePlan.create(state["src"], align=case["align"])
        recv = axon.BundlePlan.from_header(send.header).bind(state["dst"])
        n = send.payload_bytes
        payload = torch.zeros(n, dtype=torch.uint8, device="cuda")
        state.update(send=send, recv=recv, payload=payload, bytes=n)
        if path == "submit":
            # a second bundle has arrived before: it is what this pass unpacks
            spec = _spec(case)
            other = _random_bytes(spec.arena_bytes, seed + (1 << 30))
            arrived = torch.zeros(n, dtype=torch.uint8, device="cuda")
            with axon.BundlePlan.create(_carve(other, spec), align=case["align"]) as plan:
                plan.pack(arrived.data_ptr(), n)
            jobs = (_capi.Job * 2)()
            jobs[0].plan, jobs[0].payload, jobs[0].payload_bytes, jobs[0].unpack = send._h, payload.data_ptr(), n, 0
            jobs[1].plan, jobs[1].payload, jobs[1].payload_bytes, jobs[1].unpack = recv._h, arrived.data_ptr(), n, 1
            state.update(arrived=arrived, jobs=jobs, lib=_capi.load())
        else:
            send.prepare()
            recv.prepare()
    return state


# ---------------------------------------------------------------- one pass

def run(state):
    path = state["path"]
    if path in ("fresh", "host", "layer", "cache"):
        bundle = axon.pack_bundle(state["src"], align=state["align"])
        plan = axon.unpack_bundle(bundle.header, bundle.payload, payload_bytes=bundle.payload_bytes, out=state["dst"])
        plan.close()
        bundle.close()
        return {"header": np.frombuffer(bundle.header, np.uint8), "tensors": state["out"]}
    if path == "stream":
        transfer = state["transfer"]
        for src, dst in zip(state["src"], state["dst"]):
            transfer.submit(src, dst)
        transfer.finish()
        return state["out"]
    if path == "submit":
        _capi.check(state["lib"].axr_submit(state["jobs"], 2, None))
        return {"payload": state["payload"], "tensors": state["out"]}
    at, n = state["payload"].data_ptr(), state["bytes"]
    state["send"].pack(at, n)
    state["recv"].unpack(at, n)
    return {"payload": state["payload"], "tensors": state["out"]}


# ---------------------------------------------------------------- what a pass needs

def _data_bytes(case):
    path = case["path"]
    if path == "host":
        return sum(s.nbytes // 4 * 4 for s in _spec(case).segments)
    if path in ("fresh", "kept", "submit"):
        return _spec(case).data_bytes
    if path == "layer":
        return 2 * sum(math.prod(s) for s in _layer_shapes(case))
    if path == "cache":
        return 2 * case["picks"] * case["layers"] * 2 * case["tokens"] * case["heads"] * case["dim"]
    if path == "stream":
        return 2 * case["chunks"] * case["views"] * case["rows"] * case["cols"]
    if path == "transposed":
        return case["matrices"] * case["rows"] * case["cols"] * case["item"]
    if path == "images":
        return case["images"] * case["height"] * case["width"] * case["channels"] * case["item"]
    return case["rows"] * case["cols"] * case["item"]


def _payload_bound(case):
    per = 2 * case["rows"] * case["cols"]
    return case["views"] * ((per + case["align"] - 1) // case["align"] * case["align"])


def work(case):
    # packing reads the tensors and writes the payload, unpacking reads the payload and writes the tensors
    return {"bytes": 4 * _data_bytes(case), "flops": 0}


def tolerance(case):
    return "exact"    # bytes are moved, never computed
