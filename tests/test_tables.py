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
