"""Calls of different sizes take different slab sizes (crx_apply_count_slab) and kernels: results are the
oracle's at the sizes where the choice changes."""

import ctypes

import pytest
import torch

import crukx_sync
import oracle
import scenarios
from crukx_sync import _native, codec


def _cuda(d):
    return {k: v.to("cuda") for k, v in d.items()}


def test_count_slab_follows_the_size():
    """Slabs grow with the call, are multiples of a 128-element row, stay within _SLAB, and are halved
    for updates whose largest slabs would average more than 1600 changes."""
    def f(elements, slab, changes=0):
        return _native.lib().crx_apply_count_slab(elements, changes, slab)

    sizes = [f(1 << k, 1 << 24) for k in range(33)]
    assert sizes == sorted(sizes) and sizes[0] == 512 and sizes[-1] == 65536
    assert all(s % 128 == 0 for s in sizes)
    assert f(512 * 4096, 1 << 24) == 512 and f(512 * 4096 + 1, 1 << 24) == 1024
    assert f(1 << 32, 1 << 24, 65536 * 1600) == 65536 and f(1 << 32, 1 << 24, 65536 * 1600 + 1) == 32768
    assert [f(1 << 32, s) for s in (1, 128, 1000, 4096, 1 << 14)] == [128, 128, 896, 4096, 1 << 14]


@pytest.mark.parametrize("n,kept,want", [
    (1_700_000, 512, 65536), (12_800_000, 4096, 65536), (26_600_000, 8192, 65536), (100_000_000, 32768, 32768)])
def test_count_slab_of_a_whole_model_applied_in_pieces_before(n, kept, want):
    """A model of 7.6 billion weights after applies of its tensors (n weights) one by one: its slabs are the
    whole's again (or half of them, whose counts are used), and a piece's thereafter too."""
    L, pieces = _native.lib(), 7_600_000_000 // n
    changes = 76_000_000
    assert L.crx_apply_count_slab(n, n // 100, 1 << 24) == kept
    assert codec._count_slab(lambda: changes, [kept] * pieces, [n] * pieces, 1 << 24) == want
    assert codec._count_slab(lambda: changes, [kept, 65536] * (pieces // 2), [n] * (pieces // 2 * 2), 1 << 24) == (want if 2 * kept >= want else 65536)
    assert codec._count_slab(lambda: changes, [], [n] * pieces, 1 << 24) == 65536
    assert codec._count_slab(lambda: n // 100, [want], [n], 1 << 24) == want
    assert codec._count_slab(lambda: n // 100, [kept], [n], 1 << 24) == kept
    # the same tensors at a few more changes or elements than the rule's lines: their counts are used
    assert codec._count_slab(lambda: changes * 3, [65536] * pieces, [n] * pieces, 1 << 24) == 65536
    assert codec._count_slab(lambda: changes, [32768] * pieces, [n] * pieces, 1 << 24) == 32768


def test_count_slab_of_counts_of_one_size():
    """Counts of one size (that some call takes) are used when it is at least half of what suits the call,
    at every call size."""
    f = _native.lib().crx_apply_count_slab
    calls = [e for k in range(8, 34) for e in ((1 << k) - 1, 1 << k, (1 << k) + 1)]
    for slab in (0, 128, 600, 1000, 4096, 40_000, 1 << 24):
        for size in {f(e, 0, slab) for e in calls}:
            for elements in calls:
                for changes in (0, elements // 30):
                    suits = f(elements, changes, slab)
                    got = codec._count_slab(lambda: changes, [size], [elements], slab)
                    assert got == (size if 2 * size >= suits else suits), (elements, slab, changes, size)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 511, 512, 513, 512 * 128, 512 * 128 + 1, 512 * 2048, 512 * 2048 + 1, 512 * 4096,
                               512 * 4096 + 1])
def test_bytes_and_apply_at_slab_edges(n):
    a, b = scenarios.rl_pair(n, lr=4e-6, seed=n)
    b[-1] = (b[-1:].view(torch.int16) + 1).view(torch.bfloat16)[0]  # at least one change, in the last slab
    old, new = {"w": a}, {"w": b}
    upd = crukx_sync.encode_update(_cuda(old), _cuda(new))
    assert upd == oracle.encode_update(old, new)
    recv = _cuda(old)
    crukx_sync.apply_update(recv, upd)
    assert torch.equal(recv["w"].cpu().view(torch.int16), b.view(torch.int16))


@pytest.mark.gpu
def test_counts_kept_while_updates_hold_more_and_fewer_tensors():
    """Updates of all of a receiver's tensors and of its smallest alone, in turn: each is exact, and the
    counts of the many stay in use for the few (one slab size), while a receiver that knows only the few
    takes the many's slab size for all."""
    shapes = {"big": 3_000_001, "small": 20_003}
    states = [{}, {}]
    for i, (k, n) in enumerate(shapes.items()):
        states[0][k], states[1][k] = scenarios.rl_pair(n, lr=4e-6, seed=900 + i)
    for first in ("small", "all"):
        cur = dict(states[0])
        recv, chk = _cuda(cur), {}
        sizes = []
        for which in (first, "all", "small", "all"):
            nxt = {k: (states[1][k] if cur[k] is states[0][k] else states[0][k]) if which in ("all", k) else cur[k]
                   for k in shapes}
            crukx_sync.apply_update(recv, crukx_sync.encode_update(_cuda(cur), _cuda(nxt)), chk)
            for k in shapes:
                assert torch.equal(recv[k].cpu().view(torch.int16), nxt[k].view(torch.int16)), (first, which, k)
            sizes.append(codec._hist[id(recv["small"])][6])
            cur = nxt
        assert sizes == ([512, 1024, 1024, 1024] if first == "small" else [1024] * 4)
        assert {k: v[0] for k, v in chk.items()} == {k: codec.checksum(recv[k]) for k in shapes}


def _many_groups(tensors, n=600):
    """Every element of `tensors` random int16 tensors changed: 256 groups each, most of one block."""
    g = torch.Generator().manual_seed(tensors)
    old = {f"t{i}": torch.randint(-32768, 32768, (n,), generator=g, dtype=torch.int16) for i in range(tensors)}
    return old, {k: v ^ torch.randint(1, 32768, (n,), generator=g, dtype=torch.int16) for k, v in old.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["host", "device"])
@pytest.mark.parametrize("tensors", [1, 50, 60])
def test_decoder_by_number_of_blocks(tensors, form):
    """Updates on both sides of the number of blocks up to which a wavefront decodes a block: exact, and
    rejected with the weights unchanged when a payload byte is flipped."""
    old, new = _many_groups(tensors)
    upd = crukx_sync.encode_update(_cuda(old), _cuda(new))
    assert upd == oracle.encode_update(old, new)
    pay = len(upd) - _native.lib().crx_update_payload_len(crukx_sync.parse(upd).handle)
    recv = _cuda(old)
    for at in range(pay, len(upd), max(1, (len(upd) - pay) // 40)):
        bad = bytearray(upd)
        bad[at] ^= 0x41
        with pytest.raises(crukx_sync.CorruptUpdate):
            crukx_sync.apply_update(recv, bytes(bad) if form == "host" else
                                    torch.frombuffer(bad, dtype=torch.uint8).cuda())
    assert all(torch.equal(recv[k].cpu(), old[k]) for k in old)
    crukx_sync.apply_update(recv, upd if form == "host" else torch.frombuffer(bytearray(upd), dtype=torch.uint8).cuda())
    assert all(torch.equal(recv[k].cpu(), new[k]) for k in new)


@pytest.mark.gpu
@pytest.mark.parametrize("n,lanes", [(1_900_000, False), (2_900_000, True)])
def test_decoder_by_bits_of_the_payload(n, lanes):
    """Updates of few enough blocks for a wavefront each, in payloads on both sides of 12288 * 3072 bits."""
    old, new = _many_groups(1, n)
    upd = crukx_sync.encode_update(_cuda(old), _cuda(new))
    u, L = crukx_sync.parse(upd), _native.lib()
    assert L.crx_update_n_blocks(u.handle) <= 12288 and (8 * L.crx_update_payload_len(u.handle) > 12288 * 3072) == lanes
    recv = _cuda(old)
    crukx_sync.apply_update(recv, upd)
    assert torch.equal(recv["t0"].cpu(), new["t0"])


@pytest.mark.gpu
@pytest.mark.parametrize("spread", [3, 700, 9_001, 120_000])
def test_blocks_of_long_codes(spread):
    """Blocks of one to many decoder segments, with unary runs past a 64-bit window: changes in dense runs
    and `spread` elements apart in one exponent group, whose Rice parameter suits neither."""
    n = 256 * spread + 2048
    a = torch.full((n,), 0x3F80, dtype=torch.int16)
    b = a.clone()
    b[:2048] += 1
    b[2048::spread] += 3
    old, new = {"w": a}, {"w": b}
    upd = crukx_sync.encode_update(_cuda(old), _cuda(new))
    assert upd == oracle.encode_update(old, new)
    recv = _cuda(old)
    crukx_sync.apply_update(recv, upd)
    assert torch.equal(recv["w"].cpu(), b)


@pytest.mark.gpu
def test_blocks_of_long_remainders():
    a, b = scenarios.far_pair()
    upd = crukx_sync.encode_update({"w": a.cuda()}, {"w": b.cuda()})
    assert upd == oracle.encode_update({"w": a}, {"w": b})
    assert crukx_sync.parse(upd).tensors[0].groups[0].rice_r == 16
    recv = {"w": a.cuda()}
    crukx_sync.apply_update(recv, upd)
    assert torch.equal(recv["w"].cpu(), b)


@pytest.mark.gpu
@pytest.mark.parametrize("gap,extra", [(14, 0), (15, 0), (16, 0), (66, 0), (67, 0), (67, 15), (90, 0)])
def test_workgroups_of_long_bit_strings(gap, extra):
    """Workgroups of 4096 changes that take gap + 1 bits each (a million changes in one run hold the Rice
    parameter at 0): as many bits as are staged at most (16 per change), more, as many as LDS surely holds
    (67; its 8704 words hold 68 where the string begins with a word, as after a run of 15 changes more),
    and as many as it does not."""
    dense, far = (1 << 20) + extra, 3 * 4096 + 17
    a = torch.full((dense + gap * far,), 0x3F80, dtype=torch.int16)
    b = a.clone()
    b[:dense] += 1
    b[dense::gap] += 1
    old, new = {"w": a}, {"w": b}
    upd = crukx_sync.encode_update(_cuda(old), _cuda(new))
    assert upd == oracle.encode_update(old, new)
    bits = 8 * _native.lib().crx_update_payload_len(crukx_sync.parse(upd).handle)
    # the first of the far changes follows the run at once
    assert 0 <= bits - (2 * dense + 2 + (far - 1) * (gap + 1)) < 8
    # change 2^20 + 4096, with which a workgroup begins, as the 4096 after it
    assert ((2 * dense + 2 + (4096 - extra - 1) * (gap + 1)) % 32 == 0) == (extra == 15)
    recv = _cuda(old)
    crukx_sync.apply_update(recv, upd)
    assert torch.equal(recv["w"].cpu(), b)


def _packed(tensors, lead):
    """The tensors one behind another in one GPU buffer, from element `lead` of it on."""
    flat = torch.zeros(lead + sum(t.numel() for t in tensors.values()), dtype=torch.int16, device="cuda")
    out, at = {}, lead
    for k, t in tensors.items():
        out[k] = flat[at:at + t.numel()].view(t.dtype).view(t.shape)
        out[k].copy_(t)
        at += t.numel()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("leads", [(0, 0), (1, 1), (0, 1), (1, 0)])
@pytest.mark.parametrize("cached", [False, True])
def test_packed_tensors_at_odd_elements(leads, cached):
    """Old and new state dicts packed into flat buffers, beginning in the same or in different halves of
    a 32-bit word, with and without the sender's cache: the oracle's bytes, and the inputs unchanged."""
    old, new = {}, {}
    for i, n in enumerate([1, 2, 511, 513, 70_001, 1025]):
        old[f"t{i}"], new[f"t{i}"] = scenarios.rl_pair(n, lr=4e-6, seed=300 + i)
        new[f"t{i}"][-1] = (new[f"t{i}"][-1:].view(torch.int16) ^ 1).view(torch.bfloat16)[0]
        new[f"t{i}"][0] = (old[f"t{i}"][:1].view(torch.int16) ^ 3).view(torch.bfloat16)[0]
    chk = {k: oracle.checksum(t) for k, t in old.items()} if cached else None
    a, b = _packed(old, leads[0]), _packed(new, leads[1])
    assert crukx_sync.encode_update(a, b, chk) == oracle.encode_update(old, new)
    for k in old:
        assert torch.equal(a[k].cpu().view(torch.int16), old[k].view(torch.int16))
        assert torch.equal(b[k].cpu().view(torch.int16), new[k].view(torch.int16))
        assert chk is None or chk[k] == oracle.checksum(new[k])


@pytest.mark.gpu
def test_a_small_calls_workspace_after_a_large_call_of_as_many_slabs():
    """134 million weights in slabs of 32768 and 2 million in slabs of 512 are as many slabs: the small
    encode and apply take no more memory after the large ones than after their like."""
    def peaks(n):
        a = torch.zeros(n, dtype=torch.int16, device="cuda")
        b = a.clone()
        b[::100] += 1
        out = []
        for f in (lambda: crukx_sync.encode_update_device({"w": a}, {"w": b}), lambda: crukx_sync.apply_update({"w": a}, upd)):
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            before = torch.cuda.memory_allocated()
            upd = f()
            out.append(torch.cuda.max_memory_allocated() - before)
        assert torch.equal(a, b)
        return out

    small, large = 2_090_000, 134_000_000
    peaks(small)
    alone = peaks(small)
    peaks(large)
    after = peaks(small)
    # without a hint of its own size a call takes its workspace in chunks of 8 MiB, the last not full
    assert all(x <= y + (8 << 20) for x, y in zip(after, alone)), (alone, after)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [513, 20_003, 700_001])
@pytest.mark.parametrize("slab", [0, 4096])
def test_apply_entries_of_the_c_interface(n, slab):
    """crx_apply, crx_apply_cached with counts of the largest slabs that `slab` allows (written, then kept
    over two updates) and crx_apply_counts with smaller ones: exact, and nothing written when a checksum
    is not the receiver's."""
    a, b = scenarios.rl_pair(n, lr=4e-5, seed=n)
    L, dev = _native.lib(), torch.device("cuda")
    there, back = (crukx_sync.parse(oracle.encode_update({"w": x}, {"w": y})) for x, y in ((a, b), (b, a)))
    ups, target = (there, back), a.cuda()
    err, changed = _native.errbuf(), ctypes.c_uint64()

    def call(entry, u, *args, cached=None):
        ws = _native.Workspace(target.device)
        rc = entry(u.handle, None, (ctypes.c_void_p * 1)(target.data_ptr()), (ctypes.c_uint64 * 1)(n),
                   (ctypes.c_int32 * 1)(cached is not None), (ctypes.c_uint64 * 1)(cached or 0), *args, slab,
                   _native.stream_of(target.device), ws.fn, None, ctypes.byref(changed), err, 512)
        ws.check()
        torch.cuda.synchronize()
        ws.release()
        return rc

    def holds(x):
        return torch.equal(target.cpu().view(torch.int16), x.view(torch.int16))

    def counts(size):
        buf = torch.full((L.crx_apply_hist_words(n, size),), -1, dtype=torch.int32, device=dev)
        return buf, (ctypes.c_void_p * 1)(buf.data_ptr())

    assert call(L.crx_apply, ups[0]) == _native.OK and holds(b) and changed.value > 0
    assert call(L.crx_apply, ups[0]) == _native.CORRUPT and holds(b)
    assert call(L.crx_apply, ups[1]) == _native.OK and holds(a)
    for entry, size in ((L.crx_apply_cached, ()), (L.crx_apply_counts, (256,))):
        buf, p = counts(size[0] if size else slab)  # (held: p is its address)
        none = (ctypes.c_void_p * 1)()
        assert call(entry, ups[0], none, p, *size) == _native.OK and holds(b)
        assert call(entry, ups[1], p, p, *size, cached=oracle.checksum(b)) == _native.OK and holds(a)
        assert call(entry, ups[0], p, p, *size, cached=oracle.checksum(a) ^ 1) == _native.CORRUPT and holds(a)
