"""Pins of oracle/embed_ref.py and of the host-side group builder (CPU only)."""
import numpy as np
import pytest

from oracle.bf16_ref import bf16_rne_bits, bits_to_f32
from oracle.embed_ref import id_groups, embed_dw_rows, embed_dw_scatter


def test_group_arrays_have_their_defining_properties():
    rng = np.random.default_rng(0)
    for M, V in ((512, 2048), (512, 64), (1, 5), (300, 1)):
        ids = rng.integers(0, V, M).astype(np.int32)
        srt, start, cnt, gid = id_groups(ids)
        assert sorted(srt.tolist()) == list(range(M))                  # a permutation
        assert np.all(np.diff(ids[srt]) >= 0)                          # ids non-decreasing
        assert cnt.sum() == M and np.all(cnt > 0) and np.all(np.diff(gid) > 0)
        assert np.array_equal(gid, np.unique(ids))
        for g in range(gid.size):
            seg = srt[start[g]:start[g] + cnt[g]]
            assert np.all(ids[seg] == gid[g]) and np.all(np.diff(seg) > 0)   # original order kept
        assert np.array_equal(cnt, np.bincount(ids, minlength=V)[gid])


def test_host_builder_matches_the_oracle_and_pads():
    from ancora_cutile_amd.embed import build_id_groups
    rng = np.random.default_rng(1)
    ids = rng.integers(0, 97, 400).astype(np.int32)
    srt, start, cnt, gid = build_id_groups(ids)
    o_srt, o_start, o_cnt, o_gid = id_groups(ids)
    U = o_gid.size
    for a in (srt, start, cnt, gid):
        assert a.shape == (400, 1) and a.dtype == np.int32
    assert np.array_equal(srt[:, 0], o_srt)
    assert np.array_equal(start[:U, 0], o_start) and np.array_equal(cnt[:U, 0], o_cnt)
    assert np.array_equal(gid[:U, 0], o_gid) and not cnt[U:].any() and not start[U:].any()


@pytest.mark.parametrize("ids", [np.zeros(1), np.array([5, 5, 5]), np.array([-3, 7, -3, 0, 7]), np.array([2**31 - 1, -2**31, 0, 2**31 - 1]),
                                 np.arange(300)[::-1], np.array([63, 64, 65, 127, 128, 64, 0])], ids=str)
def test_host_builder_at_the_edges(ids):
    """One id, one group, negative ids, the whole 32-bit range (sorted instead of ranked by bitmap), word borders."""
    from ancora_cutile_amd.embed import build_id_groups, _lib, api
    ids = ids.astype(np.int32)
    srt, start, cnt, gid = (a[:, 0] for a in build_id_groups(ids))
    o_srt, o_start, o_cnt, o_gid = id_groups(ids)
    U = o_gid.size
    assert np.array_equal(srt, o_srt) and np.array_equal(start[:U], o_start)
    assert np.array_equal(cnt[:U], o_cnt) and np.array_equal(gid[:U], o_gid) and not cnt[U:].any()
    out, n = np.empty(ids.size, np.int32), _lib.i64(0)
    api.anc_unique_ids(ids.ctypes.data, ids.size, out.ctypes.data, n)
    assert np.array_equal(out[:n.value], np.unique(ids))


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.float16, np.int64, np.uint16, np.uint32, np.int8, bool])
def test_host_builder_takes_ids_of_any_type(dtype):
    """Token ids as a data loader may hold them, floating point among them, group as their int32 values."""
    from ancora_cutile_amd.embed import build_id_groups
    ids = np.random.default_rng(3).integers(0, 97, 400).astype(dtype)
    for got, want in zip(build_id_groups(ids.reshape(20, 20)), build_id_groups(ids.astype(np.int32))):
        assert np.array_equal(got, want)
    if dtype is np.uint32:
        ids[::9] = 0xFFFFFFFF                                        # padding
        srt, start, cnt, gid = (a[:, 0] for a in build_id_groups(ids))
        o_srt, o_start, o_cnt, o_gid = id_groups(ids.view(np.int32))
        U = o_gid.size
        assert np.array_equal(gid[:U], o_gid) and -1 in o_gid and np.array_equal(srt, o_srt) and np.array_equal(cnt[:U], o_cnt)
    assert [a.shape for a in build_id_groups([])] == [(0, 1)] * 4


def test_scatter_sum_exact_case_and_reference_gate():
    rng = np.random.default_rng(2)
    M, V, H = 512, 64, 128
    ids = rng.integers(0, V, M).astype(np.int32)
    ints = rng.integers(-8, 9, (M, H)).astype(np.float32)            # exact in bf16, sums exact in fp32
    gid, rows = embed_dw_rows(ids, bf16_rne_bits(ints).reshape(M, H))
    want = np.zeros((V, H), np.int64)
    np.add.at(want, ids, ints.astype(np.int64))
    assert np.array_equal(rows.astype(np.int64), want[gid])
    dyb = bf16_rne_bits(rng.standard_normal((M, H)).astype(np.float32)).reshape(M, H)
    base = (0.1 * rng.standard_normal((V, H))).astype(np.float32)
    got = embed_dw_scatter(ids, dyb, base)
    ref = base.astype(np.float64)
    np.add.at(ref, ids, bits_to_f32(dyb).reshape(M, H).astype(np.float64))
    assert np.abs(got - ref).max() / np.abs(ref).max() < 5e-5      # tests/kernels/test_embed_dw_scatter.py:91
    untouched = np.setdiff1d(np.arange(V), gid)
    assert np.array_equal(got[untouched], base[untouched])
