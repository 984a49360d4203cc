"""The work whose speed this framework is judged by, one case per way of using it.

Scattered tokens in pinned host memory are assembled in HBM (and written back),
through every public entry point that serves a running KV-cache or MoE program:
host-submitted lists (Direct), kernels over a page table or an entry list,
GPU-written descriptors (Queue), GPU-planned lists, MoE routing, and the two
wave-specialised sessions with their consumers.  Sizes are those of the tests
and of bench.py; draw() spreads over the ranges around them, odd sizes and
alignments among them.

A case's "kind" names the entry point.  Long-lived handles (the poller and its
staging, the descriptor ring, a session) are made once, as a program keeps them.
"""
import math
import weakref

import numpy as np
import torch

import gfd_amd

DEV = "cuda"
MIB = 1 << 20
QUEUE_TIMEOUT_US = 10_000_000
STAGING_BYTES = 64 * MIB  # the poller's staging: the largest list that is submitted


def listed():
    return [
        # A decode step fetching a handful of KV blocks: latency is everything.
        dict(name="direct-16x4k", kind="direct", n=16, size=4096, ragged=False, align=16, paged=False),
        # A prefix-cache hit of 32 MiB (bench.py's headline workload).
        dict(name="direct-8192x4k", kind="direct", n=8192, size=4096, ragged=False, align=16, paged=False),
        # Variable-length records (compressed KV, embeddings) packed one behind the other.
        dict(name="direct-ragged-700", kind="direct", n=700, size=9000, ragged=True, align=1, paged=False),
        # The same bytes into the free pages of a paged KV cache.
        dict(name="direct-paged-1024x4k", kind="direct", n=1024, size=4096, ragged=False, align=16, paged=True),
        # Kernel-only gather through a page table in HBM, small tokens.
        dict(name="gather-2048x512", kind="gather", n=2048, size=512),
        # Eviction to host slots; a token size that is no multiple of 16 bytes.
        dict(name="offload-4096x3000", kind="offload", n=4096, size=3000),
        # An entry list in HBM with few, large and unequal entries (blocks of several layers).
        dict(name="sg-48-ragged", kind="sg", n=48, size=300000, align=16),
        # GPU kernels request tokens from the polling thread and wait for them.
        dict(name="queue-2048x2k", kind="queue", n=2048, size=2048),
        # MoE routing: top-2 experts and the per-expert row lists.
        dict(name="route-4096x64", kind="route", tokens=4096, experts=64),
        # A list planned on the GPU from a routing table, then moved by the host path.
        dict(name="planned-4096of8x4k", kind="planned", tokens=4096, experts=8, size=4096),
        # MoE rows fetched for their experts and RMS-normalised on arrival.
        dict(name="moe-1024x7168", kind="moe", tokens=1024, experts=64, dim=7168),
        # Prefill: linear tiles streamed in while compute waves reduce the landed chunks.
        dict(name="warpspec-8192x16k", kind="warpspec", n=8192, size=16384, tile=128, chunk=32, double=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["direct", "direct", "gather", "offload", "sg", "queue", "route", "planned", "moe", "warpspec"])
    if kind == "direct":
        ragged = rng.random() < 0.5
        align = rng.choice([1, 4, 16])
        size = max(align, _log(rng, 64, 65536) // align * align)
        return dict(kind=kind, n=_log(rng, 2, min(8192, 32 * MIB // size)), size=size, ragged=ragged, align=align,
                    paged=rng.random() < 0.4)
    if kind in ("gather", "offload"):
        size = _log(rng, 64, 65536)
        size = size if rng.random() < 0.4 else max(16, size // 16 * 16)
        return dict(kind=kind, n=_log(rng, 4, min(8192, 32 * MIB // size)), size=size)
    if kind == "sg":
        align = rng.choice([1, 4, 16])
        size = max(align, _log(rng, 256, 1 * MIB) // align * align)
        return dict(kind=kind, n=_log(rng, 1, min(4096, 64 * MIB // size)), size=size, align=align)
    if kind == "queue":
        size = _log(rng, 256, 16384)
        size = size if rng.random() < 0.3 else size // 16 * 16
        return dict(kind=kind, n=_log(rng, 16, min(8192, 32 * MIB // size)), size=size)
    if kind == "route":
        return dict(kind=kind, tokens=_log(rng, 16, 65536), experts=rng.choice([4, 5, 8, 16, 32, 64]))
    if kind == "planned":
        experts = rng.choice([4, 7, 8, 16, 64])
        tokens = _log(rng, 256, 65536)
        size = max(256, min(_log(rng, 256, 8192), 64 * MIB // tokens) // 16 * 16)
        return dict(kind=kind, tokens=tokens, experts=experts, size=size)
    if kind == "moe":
        dim = 512 * rng.randint(1, 14)
        return dict(kind=kind, tokens=_log(rng, 16, min(4096, 48 * MIB // (4 * dim))),
                    experts=rng.choice([5, 8, 16, 64]), dim=dim)
    tile, chunk, double = rng.choice([(128, 32, True), (128, 32, False), (64, 8, False), (64, 16, True)])
    size = 4 * _log(rng, 256, 4096)
    size = size if rng.random() < 0.3 else size // 16 * 16
    return dict(kind="warpspec", n=_log(rng, tile, min(8192, 64 * MIB // size)), size=size, tile=tile, chunk=chunk,
                double=double)


# ------------------------------------------------------------------ handles

class _Shared:
    """One handle for all the states that use it at a time; closed with the last of them."""

    def __init__(self, make):
        self._make, self._ref = make, None

    def get(self):
        h = self._ref() if self._ref else None
        if h is None:
            h = self._make()
            self._ref = weakref.ref(h)
        return h


class _Direct:
    def __init__(self):
        gfd_amd.lib().gfd_set_device(0)
        self.poller = gfd_amd.CpuPollingThread(None, None, None, STAGING_BYTES, numa_node=-1)
        if not self.poller.init_direct_ce():
            raise RuntimeError("init_direct_ce failed")


class _Queue:
    """The ring, its polling thread, and the slot that the next request starts at."""

    def __init__(self):
        gfd_amd.lib().gfd_set_device(0)
        self.ring = gfd_amd.DescriptorQueue()
        self.base = 0
        self.poller = gfd_amd.CpuPollingThread(self.ring, None, None, STAGING_BYTES, numa_node=-1)
        if not self.poller.init_copy_engine():
            raise RuntimeError("init_copy_engine failed")
        self.poller.start()

    def __del__(self):
        try:
            torch.cuda.synchronize()  # the last wait kernel reads the ring
            self.poller.stop()
            self.poller.close()
            self.ring.free()
        except Exception:
            pass


_direct, _queue = _Shared(_Direct), _Shared(_Queue)


# ------------------------------------------------------------------- inputs

def _rng(case, seed):
    return np.random.Generator(np.random.SFC64([int(seed), sum(map(ord, case["kind"]))]))


def _random_host(rng, nbytes):
    """Pinned host memory holding random bytes."""
    host = gfd_amd.HostBuffer((nbytes + 7) // 8 * 8)
    host.array.view(np.uint64)[:] = rng.integers(0, 1 << 64, host.nbytes // 8, dtype=np.uint64)
    return host


class _Slots:
    """A HostBuffer's bytes as an array that keeps the buffer alive: np.asarray(_Slots(host))."""

    def __init__(self, host):
        self.host, self.__array_interface__ = host, host.array.__array_interface__


def _device_u64(values):
    return torch.from_numpy(np.ascontiguousarray(values, dtype=np.uint64).view(np.int64)).to(DEV)


def _slots(rng, n, stride):
    """Offsets of n tokens at `stride` bytes, in random order."""
    return rng.permutation(n).astype(np.uint64) * np.uint64(stride)


def _ragged(rng, n, top, align):
    """n sizes of up to `top` bytes, and where the entries lie in host memory:
    gaps between them, in random order, at multiples of `align`."""
    sizes = rng.integers(1, top // align + 1, n).astype(np.uint64) * np.uint64(align)
    room = sizes * np.uint64(2) + rng.integers(0, 40, n).astype(np.uint64) * np.uint64(align)
    starts = np.concatenate([[0], np.cumsum(room[:-1])]).astype(np.uint64) + np.uint64(3 * align if align < 16 else 0)
    order = rng.permutation(n)
    return sizes[order], starts[order], int(starts[-1] + room[-1]) + 64


def _entries(dst, src, size):
    arr = (gfd_amd.SGEntry * len(src))()
    a = np.frombuffer(arr, dtype=np.uint64).reshape(-1, 3)
    a[:, 0], a[:, 1], a[:, 2] = dst, src, size
    return arr


def _list_of(case, rng):
    """(host, dst, dst addresses, src addresses, sizes) of an entry list."""
    n, top, align = case["n"], case["size"], case["align"]
    if case.get("ragged", True):
        sizes, src, nbytes = _ragged(rng, n, top, align)
    else:
        sizes = np.full(n, top, np.uint64)
        src, nbytes = _slots(rng, n, 2 * top), 2 * top * n
    host = _random_host(rng, nbytes)
    if case.get("paged"):
        at, room = rng.permutation(2 * n)[:n].astype(np.uint64) * np.uint64(top), 2 * n * top
    else:
        at, room = np.concatenate([[0], np.cumsum(sizes[:-1])]).astype(np.uint64), n * top
    dst = torch.zeros(room, dtype=torch.uint8, device=DEV)
    return host, dst, np.uint64(dst.data_ptr()) + at, np.uint64(host.ptr) + src, sizes


def _prepare_direct(case, rng):
    host, dst, to, src, sizes = _list_of(case, rng)
    return dict(keep=_direct.get(), host=host, dst=dst, entries=_entries(to, src, sizes))


def _prepare_sg(case, rng):
    host, dst, to, src, sizes = _list_of(case, rng)
    return dict(host=host, dst=dst, table=_device_u64(np.stack([to, src, sizes], 1)))


def _prepare_gather(case, rng):
    n, size = case["n"], case["size"]
    host = _random_host(rng, 2 * size * n)
    return dict(host=host, table=_device_u64(np.uint64(host.ptr) + _slots(rng, n, 2 * size)),
                dst=torch.zeros(n * size, dtype=torch.uint8, device=DEV))


def _prepare_offload(case, rng):
    n, size = case["n"], case["size"]
    host = gfd_amd.HostBuffer(2 * size * n)
    host.array[:] = 0
    src = torch.from_numpy(rng.integers(0, 256, n * size, dtype=np.uint8)).to(DEV)
    return dict(host=host, slots=np.asarray(_Slots(host)), src=src,
                table=_device_u64(np.uint64(host.ptr) + _slots(rng, n, 2 * size)))


def _prepare_queue(case, rng):
    n, size = case["n"], case["size"]
    host = _random_host(rng, 2 * size * n)
    tokens = np.zeros((n, 2), np.uint64)  # gfd::TokenInfo {cpu_addr, token_id, expert_id}
    tokens[:, 0] = np.uint64(host.ptr) + _slots(rng, n, 2 * size)
    tokens[:, 1] = np.arange(n)
    return dict(keep=_queue.get(), host=host, tokens=_device_u64(tokens),
                dst=torch.zeros(n * size, dtype=torch.uint8, device=DEV),
                status=gfd_amd.HostBuffer(64, gfd_amd.HOST_COHERENT))


def _logits(case, rng):
    return rng.standard_normal((case["tokens"], case["experts"]), dtype=np.float32)


def _prepare_route(case, rng):
    t, e = case["tokens"], case["experts"]
    return dict(logits=torch.from_numpy(_logits(case, rng)).to(DEV),
                top2=torch.zeros((t, 2), dtype=torch.int32, device=DEV),
                offsets=torch.zeros(e + 1, dtype=torch.int32, device=DEV),
                rows=torch.zeros(2 * t, dtype=torch.int32, device=DEV))


def _prepare_planned(case, rng):
    t, size = case["tokens"], case["size"]
    routing = rng.integers(0, case["experts"], t).astype(np.int32)
    expert = int(routing[0])
    host = _random_host(rng, 2 * size * t)
    return dict(keep=_direct.get(), host=host, routing=torch.from_numpy(routing).to(DEV), expert=expert,
                entries=gfd_amd.HostBuffer(24 * t), count=gfd_amd.HostBuffer(64),
                dst=torch.zeros(t * size, dtype=torch.uint8, device=DEV))


def _moe_inputs(case, rng):
    t, dim = case["tokens"], case["dim"]
    logits = _logits(case, rng)
    weight = torch.from_numpy(1 + 0.1 * rng.standard_normal(dim, dtype=np.float32)).to(torch.bfloat16)
    values = torch.from_numpy(rng.standard_normal((t, dim), dtype=np.float32)).to(torch.bfloat16)
    return logits, weight, values


def _prepare_moe(case, rng):
    t, e, dim = case["tokens"], case["experts"], case["dim"]
    logits, weight, values = _moe_inputs(case, rng)
    host = gfd_amd.HostBuffer(t * dim * 2)
    host.array.view(np.uint16).reshape(t, dim)[:] = values.view(torch.int16).numpy().view(np.uint16)
    s = dict(host=host, logits=torch.from_numpy(logits).to(DEV), weight=weight.to(DEV),
             top2=torch.zeros((t, 2), dtype=torch.int32, device=DEV),
             offsets=torch.zeros(e + 1, dtype=torch.int32, device=DEV),
             rows=torch.zeros(2 * t, dtype=torch.int32, device=DEV),
             dst=torch.zeros((2 * t, dim), dtype=torch.bfloat16, device=DEV),
             out=torch.zeros((2 * t, dim), dtype=torch.bfloat16, device=DEV),
             session=gfd_amd.SGWarpSpecSession(num_compute_warps=3, num_blocks=40, idle_limit_ms=10000))
    gfd_amd.moe_route(s["logits"].data_ptr(), t, e, s["top2"].data_ptr(), s["offsets"].data_ptr(),
                      s["rows"].data_ptr())
    return s


def _warpspec_values(case, rng):
    return rng.standard_normal((case["n"], case["size"] // 4), dtype=np.float32)


def _prepare_warpspec(case, rng):
    n, size = case["n"], case["size"]
    host = gfd_amd.HostBuffer(n * size)
    host.array.view(np.float32).reshape(n, size // 4)[:] = _warpspec_values(case, rng)
    return dict(host=host, dst=torch.zeros((n, size // 4), dtype=torch.float32, device=DEV),
                out=torch.zeros(n, dtype=torch.float32, device=DEV))


def prepare(case, seed):
    gfd_amd.lib().gfd_set_device(0)
    state = globals()["_prepare_" + case["kind"]](case, _rng(case, seed))
    state["case"] = case
    torch.cuda.synchronize()  # other engines write the zeroed destinations next
    return state


# --------------------------------------------------------------------- runs

def _stream():
    return torch.cuda.current_stream().cuda_stream or None


def _check(rc):
    if rc:
        raise RuntimeError(gfd_amd.lib().gfd_last_error().decode(errors="replace"))


def _submit(s, entries, count):
    if s["keep"].poller.submit_direct(entries, count) < 0:
        raise RuntimeError("submit_direct failed")


def _run_direct(s, case):
    _submit(s, s["entries"], case["n"])
    return s["dst"]


def _run_gather(s, case):
    gfd_amd.zero_copy_gather_tokens(s["table"].data_ptr(), s["dst"].data_ptr(), case["size"], case["n"], _stream())
    return s["dst"]


def _run_offload(s, case):
    gfd_amd.zero_copy_scatter_tokens(s["table"].data_ptr(), s["src"].data_ptr(), case["size"], case["n"], _stream())
    return s["slots"]


def _run_sg(s, case):
    gfd_amd.zero_copy_gather(s["table"].data_ptr(), case["n"], _stream())
    return s["dst"]


def _run_queue(s, case):
    q, lib, st = s["keep"], gfd_amd.lib(), _stream()
    _check(lib.gfd_queue_submit_tokens(q.ring.ptr, s["tokens"].data_ptr(), s["dst"].data_ptr(), case["n"],
                                       case["size"], q.base, st))
    q.base += case["n"]
    _check(lib.gfd_queue_wait(q.ring.ptr, q.base, QUEUE_TIMEOUT_US, s["status"].ptr, st))
    torch.cuda.current_stream().synchronize()  # the ring has room for the next request
    return s["dst"]


def _run_route(s, case):
    gfd_amd.moe_route(s["logits"].data_ptr(), case["tokens"], case["experts"], s["top2"].data_ptr(),
                      s["offsets"].data_ptr(), s["rows"].data_ptr(), _stream())
    return {"top2": s["top2"], "offsets": s["offsets"], "rows": s["rows"]}


def _run_planned(s, case):
    gfd_amd.plan_expert_entries(s["routing"].data_ptr(), case["tokens"], s["expert"], s["host"].ptr,
                                2 * case["size"], s["dst"].data_ptr(), case["size"], s["entries"].ptr,
                                s["count"].ptr, _stream())
    torch.cuda.current_stream().synchronize()  # the list is the host's next
    count = int(s["count"].array.view(np.int32)[0])
    _submit(s, s["entries"].ptr, count)
    return {"count": count, "dst": s["dst"]}


def _run_moe(s, case):
    session, rows = s["session"], 2 * case["tokens"]
    session.reset()
    session.launch_moe(s["host"].ptr, 2 * case["dim"], case["tokens"], s["offsets"].data_ptr(),
                       s["rows"].data_ptr(), case["experts"], rows, 2 * case["dim"], s["dst"].data_ptr(),
                       s["out"].data_ptr(), s["weight"].data_ptr(), stream=_stream())
    torch.cuda.current_stream().synchronize()  # the kernel ends itself; synchronize() then reports
    session.synchronize(0)
    return {"dst": s["dst"].view(torch.int16), "out": s["out"]}


def _run_warpspec(s, case):
    gfd_amd.warp_spec_run_rms_sin(s["host"].ptr, s["dst"].data_ptr(), case["n"], case["size"], s["out"].data_ptr(),
                                  case["tile"], case["chunk"], case["double"])
    return {"dst": s["dst"].view(torch.int32), "out": s["out"]}


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state, state["case"])


# ------------------------------------------------------- work and tolerances

def work(case):
    kind = case["kind"]
    if kind in ("direct", "sg"):
        mean = (case["size"] + case["align"]) / 2 if case.get("ragged", True) else case["size"]
        return {"bytes": case["n"] * (2 * mean + 24), "flops": 0}
    if kind in ("gather", "offload"):
        return {"bytes": case["n"] * (2 * case["size"] + 8), "flops": 0}
    if kind == "queue":
        return {"bytes": case["n"] * (2 * case["size"] + 16), "flops": 0}
    if kind == "route":
        return {"bytes": case["tokens"] * (4 * case["experts"] + 16) + 4 * case["experts"], "flops": 0}
    if kind == "planned":
        return {"bytes": 4 * case["tokens"] + case["tokens"] / case["experts"] * (2 * case["size"] + 24), "flops": 0}
    if kind == "moe":
        row = 2 * case["dim"]
        return {"bytes": 2 * case["tokens"] * 3 * row + row, "flops": 2 * case["tokens"] * 5 * case["dim"]}
    moved = case["n"] // case["tile"] * case["tile"]
    return {"bytes": moved * (2 * case["size"] + 4), "flops": moved * case["size"] // 4 * 6}


def tolerance(case):
    """Copies, routing and lists are exact.  The RMSNorm rounds to bf16 (1.7e-3
    against 64 bits), the sin sums add 32-bit products (7e-8)."""
    return {"moe": {"rel": 7e-3, "max": 1.6e-2}, "warpspec": {"rel": 4e-7, "max": 4e-6}}.get(case["kind"], "exact")


def exact(case, seed):
    rng = _rng(case, seed)
    if case["kind"] == "moe":
        logits, weight, values = _moe_inputs(case, rng)
        top2 = torch.from_numpy(logits).topk(2, dim=1).indices
        rows = torch.argsort(top2.reshape(-1) * case["tokens"] + torch.arange(2 * case["tokens"]) // 2) // 2
        x = values.to(DEV).double()
        x = x / torch.sqrt(x.square().mean(1, keepdim=True) + 1e-6) * weight.to(DEV).double()
        return {"dst": None, "out": x[rows.to(DEV)]}
    if case["kind"] == "warpspec":
        moved = case["n"] // case["tile"] * case["tile"]
        x = torch.from_numpy(_warpspec_values(case, rng)).to(DEV).double()
        x = x / torch.sqrt(x.square().mean(1, keepdim=True) + 1e-6)
        out = (torch.sin(x) * x).sum(1)
        out[moved:] = 0
        return {"dst": None, "out": out}
    return None
