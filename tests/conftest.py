import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def gpu():
    """Initialise the library on device 0; a missing library or GPU is an error, not a skip."""
    from ancora_cutile_amd import _lib, muon_ns
    _lib.init(0)
    # modes that force one tile size instead of the rule by launch size (ANC_NS_FORCE_T*)
    muon_ns.MODES.update({f"{m}_t{t}": muon_ns.MODES[m] | flag for m in ("bf16", "bf16_late3", "bf16_x3")
                          for t, flag in ((64, 0x200), (128, 0x400), (256, 0x800))})
    return _lib


class FakeDevice:
    """Host memory behind the library's memory entry points, so that what the host layer uploads and launches can be
    looked at without a GPU. Freed addresses are not handed out again."""

    def __init__(self):
        self.blocks = {}             # address -> bytearray
        self.next = 1 << 20
        self.log = []                # (entry point, arguments) of every call
        self.capturing = set()       # streams
        self.current = 0
        self.home = {}               # address -> device

    def at(self, ptr, n):
        base = max(b for b in self.blocks if b <= ptr)
        assert ptr + n <= base + len(self.blocks[base]), "access outside an allocation"
        return memoryview(self.blocks[base])[ptr - base: ptr - base + n]

    def calls(self, name):
        return [a for n, a in self.log if n == name]

    def anc_malloc(self, out, n):
        self.blocks[self.next] = bytearray(n)
        out._obj.value = self.next
        self.home[self.next] = self.current
        self.next += (n + 511) // 256 * 256

    def anc_free(self, ptr):
        del self.blocks[ptr]

    def anc_fill_u32(self, ptr, value, n, stream):
        self.at(ptr, 4 * n)[:] = int(value).to_bytes(4, "little") * n

    def anc_current_device(self, out):
        out._obj.value = self.current

    def anc_stream_is_capturing(self, stream, out):
        out._obj.value = stream in self.capturing

    def _upload(self, ptr, src, n, *stream):
        import ctypes
        src = src.value if isinstance(src, ctypes.c_void_p) else src
        self.at(ptr, n)[:] = ctypes.string_at(src, n)


@pytest.fixture
def fake_device(monkeypatch):
    from ancora_cutile_amd import _lib
    _lib.load()
    dev = FakeDevice()
    monkeypatch.setattr(_lib, "init", lambda device=0: None)
    for name, (restype, _) in _lib._PROTOS.items():
        if restype is not None or name in ("anc_id_groups", "anc_unique_ids"):      # host arithmetic
            continue
        real = getattr(dev, name, None)
        if name in ("anc_memcpy_h2d", "anc_upload_async", "anc_upload_now"):
            real = dev._upload
        def call(*args, name=name, real=real):
            dev.log.append((name, args))
            if real is not None:
                real(*args)
        monkeypatch.setattr(_lib.api, name, call)
    return dev
