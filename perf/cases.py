"""Performance cases: in-place transposes as programs call them.

Three kinds of call, all on tensors that already live on the GPU:

* single: one tensor, ``transpose_tensor`` on the current stream or
  synchronously;
* batch: many small tensors, one replay of a built ``Batch``;
* server: a burst of requests through ``Server.submit`` and ``drain``.

An in-place pass permutes whatever the buffer holds, so it can be run again
on the same state.  Outputs are the permuted bytes themselves (whole
numbers), hence no 64-bit values are given for them.
"""
import math

import torch

import eithot_amd as E
from eithot_amd.workloads import batch_specs, serve_specs

DTYPE = {1: torch.uint8, 2: torch.int16, 4: torch.int32, 8: torch.int64}
ALIGN = 256  # bytes between tensors packed in one buffer


def single(name, dims, perm, elem, sync=False, n_sub=1):
    case = {"kind": "single", "dims": ",".join(map(str, dims)), "perm": ",".join(map(str, perm)),
            "elem": elem, "sync": sync, "n_sub": n_sub}
    return dict(case, name=name) if name else case


def ints(text):
    return [int(x) for x in text.split(",")]


def listed():
    return [
        # a few tens of KB, odd dims, waited for: latency and launches
        single("small_3d", [61, 7, 45], [3, 1, 2], 4, sync=True),
        # a few MB of 8-byte elements, odd dims: the low end of the served sizes
        single("medium_4d_8byte", [129, 33, 65, 2], [4, 2, 3, 1], 8, sync=True),
        # 4-D, 64 MB, pairs swapped inside (the benchmark's smallest workload)
        single("pairs_64mb", [2, 4096, 1024, 2], [1, 3, 2, 4], 4),
        # 0.2 GB, 4 bytes: the published experiment's 2-, 5- and 6-d tensors
        single("matrix_7248", [7248, 7248], [2, 1], 4),
        single("exp2_5d", [352, 4, 28, 48, 28], [4, 3, 2, 5, 1], 4),
        single("exp2_6d", [32, 15, 15, 32, 15, 15], [4, 3, 6, 2, 1, 5], 4),
        # image batch, channels last to channels first, bytes, odd height
        single("images_uint8", [3, 640, 481, 256], [2, 3, 1, 4], 1),
        # 16-bit attention keys, (head dim, position, heads, batch) with an
        # odd number of positions, to positions fastest
        single("keys_16bit", [128, 2049, 16, 8], [2, 1, 3, 4], 2),
        # 6-D, 4.5 GB: the benchmark's high-order workload
        single("six_d_4.5gb", [32, 48, 64, 40, 36, 8], [6, 4, 2, 5, 1, 3], 4),
        # 10.7 GB, the 4-D shape of the largest workload scaled down, inverse
        single("pairs_10.7gb", [2, 16384, 40960, 2], [1, 3, 2, 4], 4),
        # many small tensors of uneven orders, shapes and element sizes
        {"name": "batch_512", "kind": "batch", "count": 512, "seed": 3},
        # a burst of requests of 1 to 256 MB
        {"name": "server_32", "kind": "server", "count": 32, "seed": 4, "hi_mb": 256},
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def split_dims(rng, vol, order):
    """Dims of about `vol` elements in random log proportions, each >= 2."""
    w = [rng.expovariate(1.0) for _ in range(order)]
    return [max(2, int(round(vol ** (x / sum(w))))) for x in w]


def draw(rng):
    pick = rng.random()
    if pick < 0.12:
        return {"kind": "batch", "count": log_int(rng, 16, 256), "seed": rng.randrange(1 << 16)}
    if pick < 0.24:
        return {"kind": "server", "count": log_int(rng, 4, 48), "seed": rng.randrange(1 << 16),
                "hi_mb": log_int(rng, 4, 256)}
    nbytes = math.exp(rng.uniform(math.log(16 << 10), math.log(1 << 30)))
    shape = rng.random()
    if shape < 0.25:
        # as in the published experiment: two lengths that recur over the dims
        elem, order = rng.choice([4, 4, 8]), rng.randint(2, 6)
        a = (nbytes / elem) ** (1.0 / order) * rng.uniform(0.6, 1.4)
        b = (nbytes / elem / a ** (order // 2)) ** (1.0 / (order - order // 2))
        dims = [max(2, round(a))] * (order // 2) + [max(2, round(b))] * (order - order // 2)
        rng.shuffle(dims)
    elif shape < 0.4:
        # images or activations: a few channels or heads, a plane, a batch
        elem, order = rng.choice([1, 2]), 4
        c, b = rng.choice([3, 4, 16, 32, 64, 128]), rng.randint(1, 32)
        side = max(2.0, math.sqrt(nbytes / elem / c / b))
        dims = [c, max(2, round(side * rng.uniform(0.7, 1.4))), max(2, round(side)), b]
    else:
        elem, order = rng.choice([1, 2, 4, 8]), rng.randint(2, 6)
        dims = split_dims(rng, max(2.0 ** order, nbytes / elem), order)
    perm = list(range(1, order + 1))
    while perm == sorted(perm):
        rng.shuffle(perm)
    n_sub = rng.choice([2, 3, 4]) if rng.random() < 0.1 else 1
    return single(None, dims, perm, elem, sync=rng.random() < 0.3, n_sub=n_sub)


def specs_of(case):
    if case["kind"] == "batch":
        return batch_specs(seed=case["seed"], count=case["count"])
    return serve_specs(seed=case["seed"], count=case["count"], hi=case["hi_mb"] << 20)


def tensor_bytes(spec):
    dims, _, elem = spec
    return math.prod(dims) * elem


def random_bytes(n, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = torch.empty(n, dtype=dtype, device="cuda")
    if dtype == torch.int64:
        return t.random_(generator=g)
    info = torch.iinfo(dtype)
    return t.random_(info.min, info.max + 1, generator=g)


def prepare(case, seed):
    if case["kind"] == "single":
        dims, perm = ints(case["dims"]), ints(case["perm"])
        t = random_bytes(math.prod(dims), DTYPE[case["elem"]], seed)
        return {"kind": "single", "t": t, "dims": dims, "perm": perm, "sync": case["sync"],
                "n_sub": case["n_sub"]}
    specs = specs_of(case)
    offsets, end = [], 0
    for s in specs:
        offsets.append(end)
        end += -(-tensor_bytes(s) // ALIGN) * ALIGN
    buf = random_bytes(end, torch.uint8, seed)
    state = {"kind": case["kind"], "t": buf}
    calls = [(buf.data_ptr() + o, *s) for s, o in zip(specs, offsets)]
    torch.cuda.current_stream().synchronize()  # batches and servers have streams of their own
    if case["kind"] == "batch":
        state["batch"] = E.Batch()
        for c in calls:
            state["batch"].add(*c)
        state["batch"].build()
    else:
        pool = max(1 << 20, int(0.05 * end))
        state["server"] = E.Server(pool, max_inflight=16, nstreams=4)
        state["calls"] = calls
    return state


def run(state):
    if state["kind"] == "single":
        stream = None if state["sync"] else torch.cuda.current_stream().cuda_stream
        E.transpose_tensor(state["t"], state["dims"], state["perm"], n_sub=state["n_sub"],
                           stream=stream)
    elif state["kind"] == "batch":
        state["batch"].run()
    else:
        for c in state["calls"]:
            state["server"].submit(*c)
        state["server"].drain()
    return state["t"]


def work(case):
    """Each byte read once and written once."""
    if case["kind"] == "single":
        return {"bytes": 2 * math.prod(ints(case["dims"])) * case["elem"], "flops": 0}
    return {"bytes": 2 * sum(tensor_bytes(s) for s in specs_of(case)), "flops": 0}
