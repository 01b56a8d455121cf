"""What the host layer keeps between calls -- descriptor tables, blocks -- against what it was made from, on a stand-in
for the device (no GPU needed)."""
import ctypes

import numpy as np
import pytest


def _quant_weights(n=2):
    from ancora_cutile_amd import DevBuf
    return {f"w{i}": dict(p16=DevBuf.zeros((128, 256), np.uint16), K=128, N=256) for i in range(n)}


def test_fp8_cache_follows_its_weights_addresses(fake_device):
    """The table is written once, again when a weight's address changes, in the same buffer object or another, and
    not for another object at the same address; a freed weight is refused and nothing launched."""
    from ancora_cutile_amd import DevBuf, Mxfp8WeightCache, _lib
    w = _quant_weights()
    cache = Mxfp8WeightCache(w)

    def refreshed():
        n = len(fake_device.calls("anc_quant_mxfp8_w_multi"))
        cache.mark_dirty()
        assert cache.refresh(0)
        calls = fake_device.calls("anc_quant_mxfp8_w_multi")[n:]
        assert len(calls) == 1
        raw = bytes(fake_device.at(calls[0][0], ctypes.sizeof(_lib.QuantDesc) * calls[0][1]))
        return calls[0][0], [_lib.QuantDesc.from_buffer_copy(raw, i * ctypes.sizeof(_lib.QuantDesc)).w for i in range(calls[0][1])]

    table, ptrs = refreshed()
    assert ptrs == [w["w0"]["p16"].ptr, w["w1"]["p16"].ptr]
    cache.w["w1"]["p16"] = DevBuf(shape=(128, 256), dtype=np.uint16, ptr=ptrs[1])
    assert refreshed() == (table, ptrs)
    other = DevBuf.zeros((128, 256), np.uint16)
    cache.w["w1"]["p16"].ptr = other.ptr                       # the same object elsewhere
    assert refreshed()[1] == [ptrs[0], other.ptr]
    w["w0"]["p16"].free()
    n = len(fake_device.calls("anc_quant_mxfp8_w_multi"))
    cache.mark_dirty()
    with pytest.raises(_lib.AncoraError):
        cache.refresh(0)
    assert cache.dirty and len(fake_device.calls("anc_quant_mxfp8_w_multi")) == n
    cache.free()


def _muon_weights(dev, shapes):
    from ancora_cutile_amd import DevBuf
    return [dict(buf=DevBuf.zeros((K, N), np.float32), p32=DevBuf.zeros((K, N), np.float32),
                 p16=DevBuf.zeros((K, N), np.uint16), G=DevBuf.zeros((K, N), np.float32), K=K, N=N) for K, N in shapes]


@pytest.mark.parametrize("fused_update", [True, False])
def test_muon_tables_follow_the_weights_addresses(fake_device, fused_update):
    """One table for many steps, also with fresh views of the same memory; another one when a gradient's address or
    type changes, in the same object or another; a freed buffer is refused and nothing launched. With the
    group's table and with a table per batch."""
    from ancora_cutile_amd import DevBuf, _lib
    from ancora_cutile_amd.muon import MuonEngine
    ws = _muon_weights(fake_device, [(128, 256), (256, 128), (128, 128)])
    eng = MuonEngine(ws, chunk=None)
    eng.fused_update = fused_update
    G = ws[1]["G"]

    def step():
        """(table, weights) of each momentum launch"""
        n = len(fake_device.calls("anc_muon_momentum_multi_pair"))
        eng.step(0)
        return [a[:2] for a in fake_device.calls("anc_muon_momentum_multi_pair")[n:]]

    def entry(launches):
        """(gradient's address, its type) of weight 1"""
        for ptr, n in launches:
            raw = bytes(fake_device.at(ptr, ctypes.sizeof(_lib.MuonDesc) * n))
            for i in range(n):
                d = _lib.MuonDesc.from_buffer_copy(raw, i * ctypes.sizeof(_lib.MuonDesc))
                if d.buf == ws[1]["buf"].ptr:
                    return d.g, d.g_dtype

    first = step()
    assert len(first) == (1 if fused_update else 2) and entry(first) == (G.ptr, _lib.F32)
    ws[1]["G"] = G.view((256, 128))
    assert step() == first
    ws[1]["G"] = G.view((256, 128), np.uint16)
    assert entry(step()) == (G.ptr, _lib.BF16)
    other = DevBuf.zeros((256, 128), np.uint16)
    ws[1]["G"].ptr = other.ptr
    assert entry(step()) == (other.ptr, _lib.BF16)
    ws[1]["G"] = G
    before = step()
    assert entry(before) == (G.ptr, _lib.F32)
    for key in ("buf", "G", "p32"):
        keep, n = ws[2][key], len(fake_device.calls("anc_muon_ns_update_multi"))
        ws[2][key] = keep.view(keep.shape)
        ws[2][key].free()
        with pytest.raises(_lib.AncoraError):
            eng.step(0)
        assert len(fake_device.calls("anc_muon_ns_update_multi")) == n
        ws[2][key] = keep
    assert step() == before
    eng.free()


def test_id_groups_are_in_place_before_a_captured_launch(fake_device):
    """A launch on a stream under capture finds the arrays uploaded outside the graph, whether they were on their way
    on another stream or not at all, and allocates nothing; outside a capture they go in the stream's order."""
    from ancora_cutile_amd import DevBuf, _lib
    from ancora_cutile_amd.embed import IdGroups, embed_dw_scatter
    dy, out = DevBuf.zeros((6, 64), np.uint16), DevBuf.zeros((8, 64), np.float32)
    for first, uploads in ((None, ["anc_upload_now"]), (3, ["anc_upload_async", "anc_stream_sync"]), (7, ["anc_upload_async"])):
        fake_device.capturing = set()
        grp = IdGroups([5, 2, 5, 5, 0, 2])
        if first is not None:
            embed_dw_scatter(grp, dy, first, out=out)
        fake_device.capturing = {7}
        mallocs = len(fake_device.calls("anc_malloc"))
        embed_dw_scatter(grp, dy, 7, out=out)
        assert len(fake_device.calls("anc_malloc")) == mallocs
        names = [n for n, _ in fake_device.log]
        last = len(names) - 1 - names[::-1].index("anc_malloc") if first is None else 0
        assert [n for n in names[last:] if n in ("anc_upload_now", "anc_upload_async", "anc_stream_sync")] == uploads
        cnt = fake_device.calls("anc_embed_dw_scatter")[-1][0]
        assert list(np.frombuffer(fake_device.at(cnt, 24), np.int32)) == [1, 2, 3, 0, 0, 0]
        grp.free()
        with pytest.raises(_lib.AncoraError):
            embed_dw_scatter(grp, dy, 7, out=out)
        fake_device.log.clear()
    with pytest.raises(ValueError):
        IdGroups(np.zeros(0, np.int32))


def test_group_blocks_are_reused_after_a_synchronisation_and_stay_on_their_device(fake_device, monkeypatch):
    """Blocks of 3 * KEEP batches on two devices in turn: one that was given back is handed out again only after a
    synchronisation of its device, on its device alone, within a factor of its size; a bounded number is kept and all
    are given back."""
    from ancora_cutile_amd import embed
    pool = embed._Blocks()
    monkeypatch.setattr(embed, "_blocks", pool)
    rng = np.random.default_rng(0)
    dirty, live = set(), []                    # given back and not synchronised since; in use

    def sync():
        fake_device.log.append(("anc_device_sync", ()))
        dirty.difference_update([p for p in dirty if fake_device.home[p] == fake_device.current])
    monkeypatch.setattr(embed.api, "anc_device_sync", sync)
    for i in range(6 * pool.KEEP):
        fake_device.current = i & 1
        grp = embed.IdGroups(rng.integers(0, 50, int(rng.integers(1, 20000))))
        base = grp.base_on(4)
        assert fake_device.home[base] == fake_device.current and base not in dirty and base not in live
        live.append(base)
        grp.free()
        live.remove(base)
        dirty.add(base)
    assert len(fake_device.calls("anc_device_sync")) <= 6
    assert len(fake_device.blocks) <= 2 * 2 * pool.KEEP
    pool.trim()
    assert not fake_device.blocks


def test_weight_gradient_sizes_of_any_number_type(fake_device):
    """Sizes, segments and addresses as numpy numbers or whole floats reach the native call as integers."""
    from ancora_cutile_amd import DevBuf, _lib
    from ancora_cutile_amd.grads import DwWorkspace, gemm_dW
    b = DevBuf.zeros((256, 256), np.float32)
    problem = dict(x=b, dy=b, dW=b, T=256.0, K=np.int64(128), N=np.float32(256), workspace=DwWorkspace(),
                   gn_partials=np.uint64(b.ptr), accumulate=np.True_)
    gemm_dW([problem], segments=np.int32(2))
    arr, n = fake_device.calls("anc_gemm_dw_multi")[-1][:2]
    d = arr[0]
    assert n == 1 and (d.T, d.K, d.N, d.segments, d.gn_partials, d.accumulate) == (256, 128, 256, 2, b.ptr, 1)
    assert d.workspace_bytes == 2 * 128 * 256 * 4 and d.x_row_major == 1 and (d.xT, d.dy, d.dW, d.g16) == (b.ptr, b.ptr, b.ptr, 0)
