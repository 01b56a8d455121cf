"""The recorded HBM traffic is tied to the kernels it was counted on: every source they are compiled from changes the hash."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join("ancora-cutile_amd", "csrc")


def _compiled_from(src):
    """What the preprocessor reads of this repository for `src`, system headers aside."""
    out = subprocess.run(["g++", "-x", "c++", "-std=c++17", "-MM", "-MG", src], cwd=os.path.join(ROOT, CSRC),
                         capture_output=True, text=True, check=True).stdout
    names = out.replace("\\\n", " ").split(":", 1)[1].split()
    paths = {os.path.normpath(os.path.join(ROOT, CSRC, n)) for n in names}
    return {os.path.relpath(p, ROOT) for p in paths if os.path.exists(p) and p.startswith(ROOT)}


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a preprocessor")
def test_every_source_of_the_counted_kernels_is_hashed(tmp_path, monkeypatch):
    import bench
    files = set().union(*(_compiled_from(f) for f in ("ns.hip", "ns_gemm_big.hip", "ns_gemm_tile.hip")))
    assert {os.path.basename(f) for f in files} >= {"ns_common.h", "lds_dma.h", "ns.hip"}
    for f in files:
        os.makedirs(tmp_path / os.path.dirname(f), exist_ok=True)
        shutil.copy(os.path.join(ROOT, f), tmp_path / f)
    here = bench.kernel_source_sha16()
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.kernel_source_sha16() == here
    seen = {here}
    for f in sorted(files):
        with open(tmp_path / f, "a") as fh:
            fh.write("// changed\n")
        assert bench.kernel_source_sha16() not in seen, f
        seen.add(bench.kernel_source_sha16())
