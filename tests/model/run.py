"""Runs crukx_sync's Python layer on the CPU model of the library (tests/model/, libcrukx_model.so):
the library's own kernels and host code, built for the CPU under AddressSanitizer and UBSan, with
every kernel run by the wave64 emulator of simt.cpp.  Test infrastructure only.

The process must start with the sanitizer runtime preloaded (`env()` gives the environment); it then
binds crukx_sync to the model library and routes the few device-only pieces of the Python layer to
the CPU: tensors live in host memory, the "device" is the CPU, every stream is the null stream.  The
rest of the Python layer (argument checks, caches, the receiver's exponent counts and their
lifecycle) runs unchanged.

    python tests/model/run.py <scenario> [args]   (scenarios below)
"""

from __future__ import annotations

import contextlib
import ctypes
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
LIB = os.path.join(HERE, "_build", "libcrukx_model.so")
CLANG = "/opt/rocm/llvm/bin/clang++"


def build() -> str:
    """Builds the model library (make in tests/model); returns its path."""
    subprocess.run(["make", "-s", "-C", HERE], check=True)
    return LIB


def asan_runtime() -> str:
    out = subprocess.run([CLANG, "-print-file-name=libclang_rt.asan-x86_64.so"], capture_output=True, text=True)
    path = out.stdout.strip()
    if not os.path.isabs(path):  # this clang keeps it under its resource directory
        res = subprocess.run([CLANG, "-print-resource-dir"], capture_output=True, text=True).stdout.strip()
        path = os.path.join(res, "lib", "linux", "libclang_rt.asan-x86_64.so")
    return path


def env(lib: str | None = None) -> dict:
    """The environment of a model process: the sanitizer runtime first, leaks not reported (the
    interpreter keeps its own until exit), a sanitizer report ends the process with status 86."""
    e = dict(os.environ)
    e["LD_PRELOAD"] = asan_runtime()
    # every allocation filled with 0xFF: device memory that no kernel wrote reads as all ones (the
    # kernels' "none" value, and the value closest to wrapping in index arithmetic)
    e["ASAN_OPTIONS"] = ("detect_leaks=0:detect_stack_use_after_return=0:exitcode=86:abort_on_error=0:"
                         "malloc_fill_byte=255:max_malloc_fill_size=4294967295")
    e["UBSAN_OPTIONS"] = "print_stacktrace=1:halt_on_error=1:exitcode=86"
    e["CRX_LIBRARY"] = lib or LIB
    e["OMP_NUM_THREADS"] = "1"
    return e


def install():
    """Binds crukx_sync to the model library (CRX_LIBRARY) and routes its device plumbing to the CPU."""
    for p in (os.path.join(ROOT, "crukx-sync_amd"), os.path.join(ROOT, "oracle"), os.path.join(ROOT, "tests")):
        if p not in sys.path:
            sys.path.insert(0, p)
    assert os.environ.get("CRX_LIBRARY"), "start the process with run.env()"
    import torch

    import crukx_sync  # noqa: F401
    from crukx_sync import _native, codec, wire

    assert os.path.samefile(_native.LIB_PATH, os.environ["CRX_LIBRARY"])
    codec._hip_device = lambda dev: dev          # the model's device is the CPU
    _native.stream_of = lambda dev: 0            # the null stream
    torch.cuda.device = lambda d: contextlib.nullcontext()

    def parse_tensor(t, L, err):
        """wire._parse_tensor's device branch for a host tensor: the header and block table are parsed
        from a copy of the leading bytes, and apply reads the block table and payload from `t` itself."""
        if t.dtype != torch.uint8 or t.dim() != 1 or not t.is_contiguous():
            raise TypeError("an update tensor must be a contiguous 1-D uint8 tensor")
        total = t.numel()
        if total == 0:
            return wire.parse(b"")
        have = min(total, 1 << 16)
        while True:
            host = torch.empty(have + 1, dtype=torch.uint8)
            host[:have].copy_(t[:have])
            host[have:].copy_(t[total - 1:])
            h, need = ctypes.c_void_p(), ctypes.c_uint64()
            rc = L.crx_parse_prefix(ctypes.c_void_p(host.data_ptr()), have, total, int(host[have]), ctypes.byref(h),
                                    ctypes.byref(need), err, 512)
            if rc == _native.INVALID and need.value > have:
                have = min(total, max(need.value + 64, 2 * have))
                continue
            _native.raise_for(rc, err)
            return wire.ParsedUpdate(h.value, host, dev_bytes=t)

    wire._parse_tensor = parse_tensor


# ------------------------------------------------------------------ scenarios

def scenario_parity() -> None:
    """Encode (bytes and the device-resident form) and apply of the small scenarios against the oracle."""
    import torch

    import crukx_sync
    import oracle
    import scenarios
    sc = scenarios.single_scenarios()
    names = sorted(sc)
    for name in names:
        old, new = sc[name]
        upd = crukx_sync.encode_update(old, new)
        ref = oracle.encode_update(old, new)
        assert upd == ref, f"{name}: model bytes differ from the oracle ({len(upd)} vs {len(ref)})"
        dev = crukx_sync.encode_update_device(old, new)
        assert bytes(dev.numpy()) == ref, name
        for u in (upd, dev):
            w = {k: v.clone() for k, v in old.items()}
            crukx_sync.apply_update(w, u)
            for k in new:
                assert torch.equal(w[k].view(torch.int16), new[k].view(torch.int16)), (name, k)
        print(f"parity {name}: {len(upd)} bytes", flush=True)


def scenario_small4_flips(first: int = 0, count: int = -1, every: int = 1, widened: int = 0) -> None:
    """The four-tensor exhaustive corruption sequences of tests/test_full_sizes.py (tests/corruption.py),
    on the model: the same weights, steps, caches, device-resident update and flips in the same order.
    Flips [first, first + count) of the list are applied (every `every`-th; SMALL4_LIST: an explicit
    list of flip indices), starting from the warm state.  widened=1: the widened sequence, with
    slabs of at most 16,384 elements (8,192, or 16,384 with CRX_LARGE_PATHS set)."""
    import corruption
    from crukx_sync import codec

    if widened:
        codec._SLAB = 1 << 14
    only = [int(v) for v in os.environ["SMALL4_LIST"].split(",")] if os.environ.get("SMALL4_LIST") else None
    rejected, applied = corruption.run("cpu", bool(widened), lambda m: print(m, flush=True), first, count, every,
                                       check_every=1, verbose=bool(os.environ.get("SMALL4_VERBOSE")), only=only)
    print(f"small4 done: {rejected} rejected, {applied} applied", flush=True)


def scenario_rejected_early() -> None:
    """Updates the decoder rejects, applied to multi-slab tensors (4096-element slabs) while device
    memory starts as all ones: each raises CorruptUpdate and leaves the receiver as it was.  Two
    neighbouring block-table entries are moved by one bit in opposite directions (the header and the
    payload length still parse), so both blocks fail to decode and the update is rejected before its
    changes are located; the receivers' caches are warm, as in a training run.  The undo pass once
    took such an update's never-written record offsets (all ones) as a range to restore and walked
    past the record buffer."""
    import struct

    import torch

    import crukx_sync
    import scenarios
    from crukx_sync import CorruptUpdate, _native, codec, wire

    codec._SLAB = 4096
    old, new = {}, {}
    for i, n in enumerate([300_000, 50_001, 4_097]):
        a, b = scenarios.rl_pair(n, lr=4e-6, seed=80 + i)
        old[f"t{i}"], new[f"t{i}"] = a, b
    send, rc = {}, {}
    recv = {k: v.clone() for k, v in old.items()}
    crukx_sync.apply_update(recv, crukx_sync.encode_update(old, new, send), rc)  # caches warm
    old, new = new, old  # the updates below take the receiver back
    upd = bytearray(crukx_sync.encode_update(old, new, send))
    u = wire.parse(bytes(upd))
    L = _native.lib()
    n_blocks, pay = L.crx_update_n_blocks(u.handle), L.crx_update_payload_offset(u.handle)
    pay_len = L.crx_update_payload_len(u.handle)
    n = 1
    while pay_len >= 128 ** n:
        n += 1
    bt = pay - n - 4 * n_blocks
    bits = list(struct.unpack_from(f"<{n_blocks}I", upd, bt))
    rejected = 0
    for b in range(0, n_blocks - 1, max(1, n_blocks // 12)):
        bad = bytearray(upd)
        struct.pack_into("<II", bad, bt + 4 * b, bits[b] + 1, bits[b + 1] - 1)
        for form in (bytes(bad), torch.frombuffer(bytearray(bad), dtype=torch.uint8)):
            try:
                crukx_sync.apply_update(recv, form, rc)
            except CorruptUpdate:
                rejected += 1
            else:
                raise AssertionError(f"blocks {b}, {b + 1} moved by one bit: applied")
            for k in old:
                assert torch.equal(recv[k].view(torch.int16), old[k].view(torch.int16)), (b, k)
    crukx_sync.apply_update(recv, bytes(upd), rc)
    for k in new:
        assert torch.equal(recv[k].view(torch.int16), new[k].view(torch.int16)), k
    print(f"rejected early: {rejected} updates rejected, the receiver unchanged each time", flush=True)


def scenario_group_message() -> None:
    """The group-size check covers tensors of more than codec._SLAB elements (codec.py:598-604): a
    20,000-element tensor whose group outnumbers the receiver's elements of its exponent is refused by
    the verification with the default _SLAB, and with "group has more changes than elements" once
    _SLAB is 4096; the receiver is unchanged either way."""
    import torch

    import crukx_sync
    from crukx_sync import CorruptUpdate, codec

    n = 20_000
    base = torch.full((n,), 0x3F80, dtype=torch.int16)
    sender = base.clone()
    sender[100:105] = 0x3C00
    target = sender.clone()
    target[100:105] += 1
    upd = crukx_sync.encode_update({"w": sender}, {"w": target})
    short = base.clone()
    short[100:103] = 0x3C00
    msgs = []
    for slab in (1 << 24, 4096):
        codec._SLAB = slab
        w = {"w": short.clone()}
        try:
            crukx_sync.apply_update(w, upd)
        except CorruptUpdate as e:
            msgs.append(str(e))
        assert torch.equal(w["w"], short)
    assert len(msgs) == 2 and msgs[0] != msgs[1] and msgs[1] == "group has more changes than elements", msgs
    print(f"group message: {msgs}", flush=True)


def scenario_device_offsets() -> None:
    """A device-resident update applied from views at every byte offset within an 8-byte word (the
    decoder then reads the payload in place, from the aligned words around it) and from the end of an
    allocation of exactly its size (then from a padded copy, or in place when its last word ends
    there): every access stays inside the update's allocation, and every apply is exact."""
    import torch

    import crukx_sync
    import scenarios

    a, b = scenarios.rl_pair(70_000, seed=21)
    upd = crukx_sync.encode_update_device({"w": a}, {"w": b})
    n = upd.numel()
    views = []
    for shift in range(9):
        buf = torch.zeros(n + shift + 40, dtype=torch.uint8)
        views.append(buf[shift:shift + n])
    for cut in (0, 3, 5):
        buf = torch.empty(n + cut, dtype=torch.uint8)  # the update at the very end of its allocation
        views.append(buf[cut:])
    for view in views:
        view.copy_(upd)
        w = {"w": a.clone()}
        crukx_sync.apply_update(w, view)
        assert torch.equal(w["w"].view(torch.int16), b.view(torch.int16))
    print(f"device offsets: {len(views)} applies exact", flush=True)


def scenario_parts() -> None:
    """The part-wise encode and apply (CRX_PART_ELEMENTS=60000: parts of one to three tensors) on the
    multi-tensor scenarios: the bytes equal the oracle's single-pass bytes (also with the sender's
    checksum cache), two chained applies with both caches are exact (the receiver's exponent counts kept
    part by part), and a corruption in the last part is rejected with every tensor unchanged (the
    verdict is taken on the whole update before any part is written)."""
    import torch

    import crukx_sync
    import oracle
    import scenarios
    from crukx_sync import CorruptUpdate

    def equal(x, y):
        return all(torch.equal(x[k].view(torch.int16), y[k].view(torch.int16)) for k in y)

    os.environ["CRX_PART_ELEMENTS"] = "60000"
    sc = scenarios.single_scenarios()
    for name in ("many_tensors", "three_tensors"):
        old, new = sc[name]
        ref = oracle.encode_update(old, new)
        assert crukx_sync.encode_update(old, new) == ref, name
        assert bytes(crukx_sync.encode_update_device(old, new).numpy()) == ref, name
        send, rc = {}, {}
        w = {k: v.clone() for k, v in old.items()}
        crukx_sync.apply_update(w, crukx_sync.encode_update(old, new, send), rc)
        assert equal(w, new), name
        chk = dict(send)
        back = crukx_sync.encode_update(new, old, send)
        assert back == oracle.encode_update(new, old, dict(chk)), name
        # bytes near the payload's end (blocks of the last part), until one that parses is rejected by
        # the device passes
        found = None
        for k in range(2, 40):
            bad = bytearray(back)
            bad[-k] ^= 0x10
            try:
                crukx_sync.apply_update(w, bytes(bad), rc)
            except CorruptUpdate as e:
                if "verify" in str(e) or "outside" in str(e):
                    found = (k, str(e))
            else:
                raise AssertionError(f"{name}: a corrupted update applied")
            assert equal(w, new), (name, k)
            if found:
                break
        assert found, name
        print(f"parts {name}: byte -{found[0]} flipped, rejected by the device passes ({found[1]})", flush=True)
        crukx_sync.apply_update(w, back, rc)
        assert equal(w, old), name
        assert send == {k: v[0] for k, v in rc.items()}, name
        print(f"parts {name}: {len(ref)} bytes as the oracle's; chained applies exact", flush=True)


def scenario_pinned_exhausted() -> None:
    """A call that runs out of pinned memory writes nothing: an update of many small tensors that does not
    verify, applied by a thread whose pinned memory cannot grow past its first block, at the number of
    tensors from which the call no longer fits there (found by bisection: up to it the verdict is
    reported, from it on the failed allocation is)."""
    import threading

    import torch

    import crukx_sync
    import oracle
    from crukx_sync import CorruptUpdate, _native

    left = ctypes.c_int.in_dll(_native.lib(), "simt_host_mallocs_left")

    def attempt(n: int) -> str:
        """The error of an update of n tensors against a receiver whose last tensor is another; the
        receiver is unchanged."""
        old = {f"{i}": torch.full((8,), 0x3F80, dtype=torch.int16) for i in range(n)}
        new = {k: v.clone() for k, v in old.items()}
        for v in new.values():
            v[3] += 1
        upd = oracle.encode_update(old, new)
        recv = {k: v.clone() for k, v in old.items()}
        recv[f"{n - 1}"][5] ^= 1
        want = {k: v.clone() for k, v in recv.items()}
        got = []

        def work():  # a thread of its own: its pinned memory starts empty
            left.value = 1
            try:
                crukx_sync.apply_update(recv, upd)
            except Exception as e:
                got.append(e)
            left.value = -1

        t = threading.Thread(target=work)
        t.start()
        t.join()
        assert all(torch.equal(recv[k], want[k]) for k in recv), f"{n} tensors, {got}: written"
        if isinstance(got[0], CorruptUpdate):
            return "verdict"
        assert "hipHostMalloc" in str(got[0]), got
        return "memory"

    fits, fails = 3000, 4096
    assert attempt(fits) == "verdict" and attempt(fails) == "memory"
    while fails - fits > 1:
        n = (fits + fails) // 2
        if attempt(n) == "verdict":
            fits = n
        else:
            fails = n
        print(f"pinned memory: {n} tensors {'fit' if fits == n else 'do not fit'}", flush=True)
    print(f"pinned memory: out of it from {fails} tensors on, nothing written", flush=True)


def launches() -> list:
    """The kernel launches since the last call: (workgroups, work-items each, collectives) of each."""
    from crukx_sync import _native
    f = _native.lib().simt_launches
    f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_void_p, ctypes.c_uint64]
    buf = (ctypes.c_uint64 * 30000)()
    return [tuple(buf[3 * i:3 * i + 3]) for i in range(f(buf, 10000))]


def scenario_long_codes() -> None:
    """Blocks of unary runs past a 64-bit window (a dense run and changes `spread` apart in one exponent
    group, whose Rice parameter suits neither): exact, rejected when a payload byte is flipped, and the
    wave decoder's work grows with the payload's bits and not with the number of such codes."""
    import torch

    import crukx_sync
    import oracle
    import scenarios
    from crukx_sync import _native, codec

    per_bit, lanes = {}, "CRX_LARGE_PATHS" in os.environ  # (a lane per block then: its work is not checked)
    for spread, far in ((8, 2048), (40, 2048), (64, 2048), (200, 1024), (2000, 256), (4000, 128)):
        dense = int(0.6 * far * spread)
        n = far * spread + dense
        a = torch.full((n,), 0x3F80, dtype=torch.int16)
        b = a.clone()
        b[:dense] += 1
        b[dense::spread] += 3
        upd = oracle.encode_update({"w": a}, {"w": b})
        u = crukx_sync.parse(upd)
        blocks = _native.lib().crx_update_n_blocks(u.handle)
        pay = _native.lib().crx_update_payload_len(u.handle)
        chk = {"w": (codec.checksum(a), a._version)}
        launches()
        w = {"w": a}
        crukx_sync.apply_update(w, upd, chk)
        assert torch.equal(a, b)
        decode = [c for g, t, c in launches() if g == blocks and t == 64]
        if lanes:
            decode = [0]
        per_bit[spread] = max(decode) / (8 * pay + 512 * blocks)
        print(f"long codes {spread}: {blocks} blocks, {8 * pay // blocks} bits each: {max(decode)} collectives, "
              f"{per_bit[spread]:.3f} per bit", flush=True)
        if spread in (64, 4000):
            w["w"].copy_(torch.full((n,), 0x3F80, dtype=torch.int16))
            want = w["w"].clone()
            for at in range(len(upd) - pay, len(upd), pay // 6):
                bad = bytearray(upd)
                bad[at] ^= 0x41
                try:
                    crukx_sync.apply_update(w, bytes(bad))
                except crukx_sync.CorruptUpdate:
                    pass
                else:
                    raise AssertionError(f"byte {at} flipped: applied")
                assert torch.equal(w["w"], want)
    a, b = scenarios.far_pair()
    crukx_sync.apply_update({"w": a}, oracle.encode_update({"w": a}, {"w": b}))
    assert torch.equal(a, b)
    # a block is decoded in segments of whole 512-bit rounds (hence 512 bits more per block)
    assert lanes or max(per_bit.values()) < 3 * per_bit[8], per_bit
    print("long codes: exact" if lanes else "long codes: work in proportion to the bits", flush=True)


def scenario_kept_counts() -> None:
    """The counts that a receiver keeps stay within their limit however many of its tensors are applied in
    calls of their own, are used where they are kept, and give their room back with their tensors; every
    apply is exact, of each tensor alone and of all together."""
    import torch

    import crukx_sync
    import oracle
    import scenarios
    from crukx_sync import codec

    codec._FINE_COUNTS = 24 << 10
    states = [{}, {}]
    for i in range(12):
        states[0][f"t{i}"], states[1][f"t{i}"] = scenarios.rl_pair(3000, lr=4e-5, seed=70 + i)  # 6 slabs: 6 KiB

    def kept():
        return sum(4 * e[2].numel() for e in codec._hist.values())

    def exact(names, s):
        for k in names:
            assert torch.equal(recv[k].view(torch.int16), states[s][k].view(torch.int16)), k

    recv, chk = {k: v.clone() for k, v in states[0].items()}, {}
    for s in (1, 0, 1):
        for k in recv:
            a, b = {k: states[1 - s][k]}, {k: states[s][k]}
            crukx_sync.apply_update(recv, oracle.encode_update(a, b), chk)
            assert kept() == codec._fine <= codec._FINE_COUNTS, (k, kept())
        exact(recv, s)
    assert sorted(codec._hist) == sorted(id(recv[f"t{i}"]) for i in range(4))
    bufs = {k: e[2] for k, e in codec._hist.items()}
    for s in (0, 1):
        crukx_sync.apply_update(recv, oracle.encode_update(states[1 - s], states[s]), chk)
        exact(recv, s)
        assert kept() == codec._fine <= codec._FINE_COUNTS
    assert all(codec._hist[k][2] is b for k, b in bufs.items())
    del bufs
    for k in ("t0", "t2"):
        del recv[k], states[0][k], states[1][k]
    assert kept() == codec._fine == 12 << 10
    bad = bytearray(oracle.encode_update(states[1], states[0]))
    bad[-9] ^= 0x20
    try:
        crukx_sync.apply_update(recv, bytes(bad), chk)
    except crukx_sync.CorruptUpdate:
        assert kept() == codec._fine == 0
    else:
        raise AssertionError("a corrupted update applied")
    for s in (0, 1):
        crukx_sync.apply_update(recv, oracle.encode_update(states[1 - s], states[s]), chk)
        exact(recv, s)
        assert kept() == codec._fine == 24 << 10
    # slabs as large as _SLAB allows are not under the limit
    codec._SLAB = 512
    for s in (0, 1):
        crukx_sync.apply_update(recv, oracle.encode_update(states[1 - s], states[s]), chk)
        exact(recv, s)
        assert kept() == 60 << 10 and codec._fine == 0
    del recv
    assert kept() == codec._fine == 0
    print("kept counts: within the limit", flush=True)


def scenario_fork() -> None:
    """The decoder has a stream of its own where the receiver's weights are streamed beside it, from 2^25 of
    them on: not with counts kept, nor in smaller calls."""
    import torch

    import crukx_sync
    import oracle
    from crukx_sync import _native

    waits = ctypes.c_int.in_dll(_native.lib(), "simt_stream_waits")
    for n, forks in ((1 << 25, True), ((1 << 25) - 1, False)):
        a = torch.full((n,), 0x3F80, dtype=torch.int16)
        b = a.clone()
        b[::100_003] += 1
        w, chk = {"w": a.clone()}, {}
        for upd, to, expect in ((oracle.encode_update({"w": a}, {"w": b}), b, forks),
                                (oracle.encode_update({"w": b}, {"w": a}), a, False)):
            waits.value = 0
            crukx_sync.apply_update(w, upd, chk)
            assert torch.equal(w["w"], to)
            assert (waits.value > 0) == expect, (n, waits.value)
    print("fork: by the weights streamed", flush=True)


SCENARIOS = {"parity": scenario_parity, "small4_flips": scenario_small4_flips, "rejected_early": scenario_rejected_early,
             "group_message": scenario_group_message, "parts": scenario_parts, "long_codes": scenario_long_codes, "kept_counts": scenario_kept_counts, "fork": scenario_fork,
             "pinned_exhausted": scenario_pinned_exhausted,
             "device_offsets": scenario_device_offsets}

if __name__ == "__main__":
    install()
    SCENARIOS[sys.argv[1]](*[int(a) for a in sys.argv[2:]])
