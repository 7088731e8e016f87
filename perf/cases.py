"""Timed cases of the receive path: what callers have it do, each through the entry point that they call.

Four ways in, and a case names its own in ``path``:

  plugin   A receive comm of the plugin (include/tcpx_plugin.h): irecv, control messages, fragments, test until done,
           iflush, irecvConsumed, with ``window`` requests posted at a time.  What NCCL's proxy thread drives; one call of
           tcpxSynthRunRequests receives the whole message.
  engine   A plugin of somebody else's that has only the GPU side from here (include/tcpx_unpack_hip.h, part 4): every
           request that is complete goes to the persistent engine, then the completion words are polled.
  batch    A consumer of the UNPACK device type, or any caller that launches per batch (part 3): one launch for a list of
           descriptors, on the caller's stream.
  noalloc  A tight serving loop that may not allocate (part 5): one slot on the caller's stream.

The wire decides the rest.  ``fragments`` is how the NIC cut the message: "page" -- whole 4 KiB pages, each at a page of
its own; "wire" -- nine in ten a whole page, the others 64 to 4095 bytes, anywhere in a page; "ragged" -- 1 to 4096 bytes
anywhere in a page and one descriptor in ten empty.  ``run`` fragments in turn arrive on one of ``flows`` flows (one
control message for each such run).  ``misalign`` is where the receive buffer starts, in bytes from a 256-byte boundary.
``descs`` is where a launch finds its descriptors: "mapped" -- in host memory that the GPU reads over PCIe, as a comm's
unpack queue is; "device" -- in the GPU's memory.
"""
import ctypes
import math
import time
import weakref

import numpy as np
import torch

import __graft_entry__

pkg = __graft_entry__.load_package()

PAGE = pkg.PAGE_SIZE
SLOT_BYTES = 4 << 20  # the most one slot of an unpack queue takes
REGION_BYTES = 1 << 30  # bounce memory of one state; the plugin's arena holds four
SMALL_POOL_BYTES = 256 << 20  # bounce memory that a message of up to a quarter of it is scattered over
MEAN_FRAGMENT = {"page": 4096.0, "wire": 0.9 * 4096 + 0.1 * 2079.5, "ragged": 2048.5}
EMPTIES = 1.0 / 9.0  # empty descriptors per fragment of a ragged message: one descriptor in ten

DESC = np.dtype([("src_off", "<u4"), ("len", "<u4"), ("dst_off", "<u8")])
FRAG = np.dtype([("frag_offset", "<u4"), ("frag_size", "<u4"), ("frag_token", "<u4"), ("flow", "<u4")])
REQUEST = np.dtype([("first_desc", "<u8"), ("dst_off", "<u8"), ("n_descs", "<u4"), ("bytes", "<u4"), ("window", "<u4"), ("reserved", "<u4")])
SUBMISSION = np.dtype(
    [("bounce_base", "<u8"), ("dst_base", "<u8"), ("descs", "<u8"), ("flag", "<u8"), ("value", "<u8"), ("n_descs", "<u4"), ("bytes", "<u4")]
)


def _case(path, total, request, fragments, name=None, run=1, flows=4, window=16, misalign=0, descs="mapped"):
    case = {"path": path, "bytes": total, "request_bytes": request, "fragments": fragments, "misalign": misalign}
    if path == "plugin":
        case.update(run=run, flows=flows, window=window)
    if path in ("batch", "noalloc"):
        case.update(descs=descs)
    if name:
        case["name"] = name
    return case


def listed():
    K, M = 1 << 10, 1 << 20
    return [
        # A lone small message through the plugin: a small all-reduce's step, where the way to the GPU and back is all there is.
        _case("plugin", 64 * K, 64 * K, "page", "plugin-64K-alone", flows=1, window=1),
        # An 8 MiB chunk whose fragments of four flows arrive interleaved, one control message each.
        _case("plugin", 8 * M, 4 * M, "wire", "plugin-8M-interleaved"),
        # A storm of small messages, a full window of them posted.
        _case("plugin", 128 * M, 64 * K, "page", "plugin-2048x64K", flows=1),
        # A bulk transfer in chunks of 128 KiB, which is how the sender cuts a message.
        _case("plugin", 256 * M, 4 * M, "page", "plugin-256M-bulk", run=32),
        # Fragments of any length with empty ones among them, two flows, an odd receive buffer.
        _case("plugin", 32 * M, 3 * M, "ragged", "plugin-32M-ragged", flows=2, misalign=3),
        # The engine with one small request at a time: latency.
        _case("engine", 64 * K, 64 * K, "page", "engine-64K-alone"),
        # One comm's unpack queue, sixteen slots of 4 MiB, handed over together.
        _case("engine", 64 * M, 4 * M, "wire", "engine-16x4M"),
        # Many comms' slots of ragged fragments queued at once.
        _case("engine", 256 * M, 3 * M, "ragged", "engine-256M-ragged", misalign=3),
        # A consumer kernel's launch for one small slot of the unpack queue.
        _case("batch", 64 * K, 64 * K, "page", "batch-64K-slot"),
        # And for a full slot.
        _case("batch", 4 * M, 4 * M, "wire", "batch-4M-slot"),
        # A backlog of slots copied by one launch, its descriptors gathered in the GPU's memory.
        _case("batch", 512 * M, 512 * M, "wire", "batch-512M", descs="device"),
        # A full slot in a loop that may not allocate.
        _case("noalloc", 4 * M, 4 * M, "wire", "noalloc-4M-slot"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    K, M = 1 << 10, 1 << 20
    path = rng.choice(["plugin", "plugin", "plugin", "engine", "engine", "batch", "batch", "noalloc"])
    fragments = rng.choice(["page", "wire", "ragged"])
    misalign = rng.choice([0, rng.randrange(256)])
    most_request = 3 * M if fragments == "ragged" else SLOT_BYTES  # (as many ragged fragments as a slot has descriptors for)
    if path == "plugin":
        # (Ragged fragments, small runs and few requests posted at a time cost the host the most: less of those.)
        run, window = _log_uniform(rng, 1, 64), rng.choice([1, 4, 16])
        total = _log_uniform(rng, 4 * K, (256 if run >= 16 and fragments == "page" else 96) * M)
        request = min(total, max(_log_uniform(rng, 4 * K, most_request), -(-total // (128 * window))))
        return _case(path, total, request, fragments, run=run, flows=rng.randint(1, 4), window=window, misalign=misalign)
    if path == "engine":
        total = _log_uniform(rng, 4 * K, 256 * M)
        request = min(total, max(_log_uniform(rng, 4 * K, most_request), -(-total // 2048)))
        return _case(path, total, request, fragments, misalign=misalign)
    if path == "batch":
        descs = rng.choice(["mapped", "device"])
        total = _log_uniform(rng, 4 * K, most_request if descs == "mapped" else (256 if fragments == "ragged" else 512) * M)
        return _case(path, total, total, fragments, misalign=misalign, descs=descs)
    total = _log_uniform(rng, 4 * K, most_request)
    return _case(path, total, total, fragments, misalign=misalign, descs=rng.choice(["mapped", "device"]))


def _message(case, rng, first_page, n_pages):
    """A message of case["bytes"] as the NIC left it in the pages from first_page on: descriptors of the whole list (dst_off
    from each request's own buffer), the page each lies in and the requests."""
    total, request, kind = case["bytes"], case["request_bytes"], case["fragments"]
    n = int(total / MEAN_FRAGMENT[kind] * 1.05) + 64
    if kind == "page":
        lens = np.full(-(-total // PAGE), PAGE, dtype=np.int64)
    elif kind == "wire":
        lens = np.where(rng.random(n) < 0.9, PAGE, rng.integers(64, PAGE, n))
    else:
        lens = rng.integers(1, PAGE + 1, n)
    ends = np.cumsum(lens)
    ends = ends[ends < total]
    # A request's last fragment ends it.
    ends = np.unique(np.concatenate([ends, np.arange(request, total, request), [total]]))
    lens = np.diff(ends, prepend=0)
    if kind == "ragged":
        lens = np.insert(lens, np.flatnonzero(rng.random(len(lens)) < EMPTIES) + 1, 0)
    n = len(lens)
    if kind == "page" and n <= n_pages:
        page, at = rng.permutation(n_pages)[:n], np.zeros(n, dtype=np.int64)
    else:
        page = rng.integers(0, n_pages, n)
        at = np.zeros(n, dtype=np.int64) if kind == "page" else rng.integers(0, PAGE + 1 - np.maximum(lens, 1))
    page = page + first_page
    start = np.cumsum(lens) - lens
    of = np.minimum(start // request, (total - 1) // request)  # the request that each descriptor belongs to
    descs = np.zeros(n, dtype=DESC)
    descs["src_off"], descs["len"], descs["dst_off"] = page * PAGE + at, lens, start - of * request
    first = np.searchsorted(of, np.arange(-(-total // request)))
    requests = np.zeros(len(first), dtype=REQUEST)
    requests["first_desc"], requests["n_descs"] = first, np.diff(first, append=n)
    requests["dst_off"] = np.arange(len(first)) * request
    requests["bytes"] = np.minimum(request, total - requests["dst_off"].astype(np.int64))
    assert case["path"] == "batch" or int(requests["n_descs"].max()) <= pkg.SLOT_PAGES
    return descs, page, requests


class _Arena:
    """A view of device memory that torch did not allocate."""

    def __init__(self, ptr, nbytes):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (nbytes,), "typestr": "|u1", "version": 2}


class _Process:
    """What a process keeps for its life: an engine, and the plugin with its bounce arena and a receive comm."""

    engine = plugin = None

    @classmethod
    def get_engine(cls):
        if cls.engine is None:
            hip, engine = pkg.hip_layer(), ctypes.c_void_p()
            pkg.check(hip.tcpxuEngineCreate(0, None, ctypes.byref(engine)), "tcpxuEngineCreate")
            pkg.check(hip.tcpxuEngineStart(engine), "tcpxuEngineStart")
            cls.engine = engine
        return cls.engine

    @classmethod
    def get_plugin(cls):
        if cls.plugin is None:
            from nccl_plugin_gpudirecttcpx_amd import synth_driver

            lib, base = pkg.plugin_lib(), ctypes.c_void_p()
            synth_driver.ok(lib.tcpxInit(None), "tcpxInit")
            synth_driver.ok(lib.tcpxSynthArenaCreate(0, 4 * REGION_BYTES, ctypes.byref(base)), "tcpxSynthArenaCreate")
            cls.arena = torch.as_tensor(_Arena(base.value, 4 * REGION_BYTES), device="cuda:0")
            cls.regions = [3, 2, 1, 0]  # free quarters of the arena
            cls.plugin = synth_driver.RecvComm(0)
        return cls.plugin


class State:
    pass


def _mapped(state, nbytes):
    hip, host, dev = pkg.hip_layer(), ctypes.c_void_p(), ctypes.c_void_p()
    pkg.check(hip.tcpxuMappedAlloc(0, nbytes, ctypes.byref(host), ctypes.byref(dev)), "tcpxuMappedAlloc")
    weakref.finalize(state, hip.tcpxuMappedFree, 0, host.value)
    return np.frombuffer((ctypes.c_uint8 * nbytes).from_address(host.value), dtype=np.uint8), dev.value


def prepare(case, seed):
    s = State()
    s.case, path = case, case["path"]
    rng = np.random.default_rng(seed)
    pool_bytes = SMALL_POOL_BYTES if case["bytes"] <= SMALL_POOL_BYTES // 4 else REGION_BYTES
    if path == "plugin":
        comm = _Process.get_plugin()
        region = _Process.regions.pop()
        weakref.finalize(s, _Process.regions.append, region)
        first_page = region * (REGION_BYTES // PAGE)
        pool = _Process.arena[region * REGION_BYTES :][:pool_bytes]
    else:
        first_page, pool = 0, torch.empty(pool_bytes, dtype=torch.uint8, device="cuda:0")
    pool.view(torch.int64).random_(generator=torch.Generator(device="cuda:0").manual_seed(seed))
    descs, page, requests = _message(case, rng, first_page, pool_bytes // PAGE)
    buffer = torch.zeros(case["bytes"] + 512, dtype=torch.uint8, device="cuda:0")
    s.pool, s.out = pool, buffer[case["misalign"] :][: case["bytes"]]
    if path == "plugin":
        s.frags = np.zeros(len(descs), dtype=FRAG)
        s.frags["frag_offset"], s.frags["frag_size"], s.frags["frag_token"] = descs["src_off"], descs["len"], page
        in_request = np.arange(len(descs)) - np.repeat(requests["first_desc"].astype(np.int64), requests["n_descs"])
        s.frags["flow"] = in_request // case["run"] % case["flows"]
        s.requests, s.seconds, s.call = requests, ctypes.c_double(), comm.lib.tcpxSynthRunRequests
        s.args = (comm.comm, s.frags.ctypes.data, requests.ctypes.data, len(requests), s.out.data_ptr(), case["bytes"], case["window"], 60000, ctypes.byref(s.seconds), None)
    elif path == "engine":
        s.engine = _Process.get_engine()
        n, first_flag = len(requests), descs.nbytes
        memory, dev = _mapped(s, first_flag + 64 * n)
        memory[:first_flag] = descs.view(np.uint8)
        s.flags = memory[first_flag:].view(np.uint64)[::8]  # a completion word to a line
        s.value = 0
        s.subs = np.zeros(n, dtype=SUBMISSION)
        s.subs["bounce_base"], s.subs["dst_base"] = pool.data_ptr(), s.out.data_ptr() + requests["dst_off"]
        s.subs["descs"], s.subs["flag"] = dev + 16 * requests["first_desc"], dev + first_flag + 64 * np.arange(n, dtype=np.uint64)
        s.subs["n_descs"], s.subs["bytes"] = requests["n_descs"], requests["bytes"]
        s.subs_ptr = ctypes.cast(s.subs.ctypes.data, ctypes.POINTER(pkg.Submission))
        s.accepted = ctypes.c_uint32()
        s.call = pkg.hip_layer().tcpxuEngineSubmitMany
    else:
        if case["descs"] == "mapped":
            memory, dev = _mapped(s, descs.nbytes + 64)
            memory[: descs.nbytes] = descs.view(np.uint8)
        else:
            s.descs = torch.from_numpy(descs.view(np.uint8)).to("cuda:0")
            dev = s.descs.data_ptr()
        stream = torch.cuda.current_stream().cuda_stream
        if path == "batch":
            s.call = pkg.hip_layer().tcpxuUnpackBatch
            s.args = (0, pool.data_ptr(), s.out.data_ptr(), dev, len(descs), stream)
        else:
            _, flag = _mapped(s, 64)
            s.call = pkg.hip_layer().tcpxuUnpackSlotNoAlloc
            s.args = (0, pool.data_ptr(), s.out.data_ptr(), dev, len(descs), flag, 1 + seed, stream)
    torch.cuda.synchronize()
    return s


def run(s):
    if s.case["path"] != "engine":
        rc = s.call(*s.args)
        if rc != pkg.SUCCESS:
            raise pkg.HipError(s.case["path"], rc, pkg.hip_layer().tcpxuLastError().decode(errors="replace"))
        return s.out
    s.value += 1
    s.subs["value"] = s.value
    pkg.check(s.call(s.engine, s.subs_ptr, len(s.subs), ctypes.byref(s.accepted)), "tcpxuEngineSubmitMany")
    deadline = time.perf_counter() + 60
    while not (s.flags == s.value).all():
        if time.perf_counter() > deadline:
            raise TimeoutError("the engine left completion words unwritten")
    return s.out


def work(case):
    """The payload read once and written once, and the descriptors read once."""
    n = case["bytes"] / MEAN_FRAGMENT[case["fragments"]] * (1 + (EMPTIES if case["fragments"] == "ragged" else 0))
    return {"bytes": 2 * case["bytes"] + 16 * math.ceil(n), "flops": 0}


def tolerance(case):
    return "exact"
