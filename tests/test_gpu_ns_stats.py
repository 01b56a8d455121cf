"""GPU parity: how the gates' statistics of a matrix are made and decided on, by the launches that can make them."""
import numpy as np
import pytest

from util import bits_equal
from test_gpu_ns import run_ns

pytestmark = pytest.mark.gpu


def _input(M, N, kind, seed):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((M, N)).astype(np.float32)
    if kind == "rows":
        X[rng.choice(M, max(1, M // 100), replace=False)] *= 100
    elif kind == "cols":
        X[:, rng.choice(N, max(1, N // 100), replace=False)] *= 100
    return X


@pytest.mark.parametrize("E,M,N", [(1, 1024, 1024), (1, 1024, 4096), (3, 1024, 1152), (7, 1152, 2304)])
def test_the_last_block_decides_on_the_column_statistic(gpu, E, M, N):
    """Batches that no launch takes in another order: matrices in the band (no statistic asked for), above it with columns that
    explain the proxy and without, and plain ones. The flags are the model's, each call again (the count of arrivals starts over),
    and the matrices have the bits they have alone."""
    from ancora_cutile_amd.muon_ns import PE_SCHEDULE
    from test_gpu_ns import _hard_count
    rng = np.random.default_rng(E + N)
    kinds = ("lowrank", "cols", "plain", "band", "lowrank", "cols", "band")

    def make(kind):
        X = rng.standard_normal((M, N)).astype(np.float32)
        if kind == "lowrank":
            X = (_input(M, 8, "plain", 7) @ _input(8, N, "plain", 8) + 0.01 * X).astype(np.float32)
        elif kind == "band":
            X[:, rng.choice(N, N // 10, replace=False)] *= 10
        elif kind == "cols":
            X[:, rng.choice(N, N // 100, replace=False)] *= 100
        return X
    X = np.stack([make(k) for k in kinds[:E]])
    wide = sum(k in ("lowrank", "band") for k in kinds[:E])
    want = run_ns(X, schedule=None)
    for _ in range(3):
        assert _hard_count(E, M, N, "bf16_late3")[0] == wide
        assert bits_equal(run_ns(X, schedule=None), want)
    for e in range(E):
        assert bits_equal(run_ns(X[e: e + 1], schedule=None)[0], want[e]), e
        assert _hard_count(1, M, N, "bf16_late3")[0] == int(kinds[e] in ("lowrank", "band")), e
    run_ns(X[:1], schedule=PE_SCHEDULE)                    # one matrix under the proxy's gates has no order either
    assert _hard_count(1, M, N)[0] == 1


@pytest.mark.parametrize("M,N", [(1024, 1024), (1024, 3072), (1152, 2432), (1408, 1408), (1536, 1536)])
@pytest.mark.parametrize("sched", ["keller", "pe"])
def test_statistics_beside_the_second_product(gpu, M, N, sched):
    """One matrix whose B has up to 256 tiles of 64 has its statistics made in that launch (1408: 253; 1536 has them made by kernels of
    their own, like two matrices and tiles of 128): flags and bits of the same matrix among two, for each answer of the statistics, call after call."""
    from ancora_cutile_amd import DevBuf, newton_schulz_resident_e
    from ancora_cutile_amd.muon_ns import NsWorkspace, PE_SCHEDULE, ns_hard_info
    from oracle.bf16_ref import bf16_rne_bits
    schedule, counted = (PE_SCHEDULE, "bf16") if sched == "pe" else (None, "bf16_late3")
    ws = NsWorkspace()

    def run(X, mode="bf16"):
        g = DevBuf(bf16_rne_bits(X).reshape(-1, N))
        newton_schulz_resident_e(g, None, None, None, None, None, X.shape[0], M, N, 0, schedule=schedule, mode=mode, workspace=ws)
        out, flags = g.to_numpy().reshape(X.shape), ns_hard_info(ws.buf.ptr, X.shape[0], M, N, 5, counted)
        g.free()
        return out, flags
    band = _input(M, N, "plain", 5)
    band[:, :: 10] *= 10
    low = (_input(M, 8, "plain", 7) @ _input(8, N, "plain", 8) + 0.01 * _input(M, N, "plain", 9)).astype(np.float32)
    for X in (_input(M, N, "plain", 1), _input(M, N, "cols", 2), band, low, _input(M, N, "rows", 3), np.zeros((M, N), np.float32)):
        pair, (n2, extra2) = run(np.stack([X, X]))
        one, (n1, extra1) = run(X[None])
        assert bits_equal(one[0], pair[0]) and bits_equal(pair[0], pair[1])
        assert 2 * n1 == n2 and abs(2 * extra1 - extra2) <= 1e-9 * extra2
    assert run(band[None])[1][0] == 1 and run(low[None])[1][0] == 1 and run(_input(M, N, "plain", 1)[None])[1][0] == 0
    t128 = run(low[None], "bf16_t128" if sched == "pe" else "bf16_late3_t128")[0]
    assert bits_equal(t128, run(low[None])[0])
    ws.free()


@pytest.mark.parametrize("M,N,beside", [(1024, 1024, True), (1408, 8192, True), (1024, 12288, True), (1024, 12416, False),
                                        (1152, 16384, False), (1536, 1536, False)])
def test_long_rows_have_the_statistics_in_launches_of_their_own(gpu, M, N, beside):
    """Beside B the column statistic is read for every matrix: only up to 12288 columns. Either way the flags and bits are those of
    the same matrix among two, which always have launches of their own."""
    from ancora_cutile_amd import DevBuf, _lib, newton_schulz_resident_e
    from ancora_cutile_amd.muon_ns import NsWorkspace, ns_hard_info
    from oracle.bf16_ref import bf16_rne_bits
    ws = NsWorkspace()

    def run(X):
        g = DevBuf(bf16_rne_bits(X).reshape(-1, N))
        _lib.profile_enable(True)
        _lib.profile_read()
        newton_schulz_resident_e(g, None, None, None, None, None, X.shape[0], M, N, 0, schedule=None, workspace=ws)
        launches = _lib.profile_read()["ns_fro"][1]
        _lib.profile_enable(False)
        out, flags = g.to_numpy().reshape(X.shape), ns_hard_info(ws.buf.ptr, X.shape[0], M, N, 5, "bf16_late3")
        g.free()
        return out, flags, launches
    for kind in ("plain", "cols"):
        X = _input(M, N, kind, M + N)
        pair, (n2, _), two = run(np.stack([X, X]))
        one, (n1, _), alone = run(X[None])
        assert bits_equal(one[0], pair[0]) and 2 * n1 == n2
        assert alone == two - (1 if beside else 0)       # (the proxy's and the column statistic's launches share a counter's scope)
    ws.free()


@pytest.mark.parametrize("sched,groups", [
    ("keller", [(3, 1024, 1152, ("lowrank", "cols", "plain")), (2, 1024, 2304, ("cols", "lowrank")), (1, 1408, 1408, ("band",)),
                (2, 256, 512, ("plain", "plain")), (4, 1152, 1280, ("plain", "band", "cols", "plain"))]),
    ("pe", [(1, 1024, 1024, ("cols",)), (1, 1024, 1152, ("lowrank",)), (1, 1152, 2432, ("plain",)), (1, 1280, 1280, ("band",))]),
])
def test_each_batch_of_a_call_decides_by_its_own_statistic(gpu, sched, groups):
    """Several batches in one call, none of them in another order: every batch has the flags and bits that it has in a call of
    its own, in each order of the batches and call after call on the same workspaces."""
    from ancora_cutile_amd import DevBuf, _lib
    from ancora_cutile_amd._lib import api
    from ancora_cutile_amd.muon_ns import MODES, PE_SCHEDULE, coef_array, ns_hard_info, ns_workspace_bytes
    from oracle.bf16_ref import bf16_rne_bits, bits_to_f32
    schedule, mode = (PE_SCHEDULE, "bf16") if sched == "pe" else (None, "bf16_late3")
    coef, rng = coef_array(schedule, 5), np.random.default_rng(3)
    bufs, probs = [], []
    for E, M, N, kinds in groups:
        X = np.stack([_input(M, N, k if k == "cols" else "plain", i + N) for i, k in enumerate(kinds)])
        for e, k in enumerate(kinds):
            if k == "lowrank":
                X[e] = _input(M, 8, "plain", 7) @ _input(8, N, "plain", 8) + 0.01 * X[e]
            elif k == "band":
                X[e][:, rng.choice(N, N // 10, replace=False)] *= 10
        hi = bf16_rne_bits(X).reshape(E, M, N)
        lo = bf16_rne_bits(X - bits_to_f32(hi).reshape(E, M, N)).reshape(E, M, N)
        nb = ns_workspace_bytes(E, M, N, mode)
        b = [DevBuf(hi.reshape(-1, N)), DevBuf(lo.reshape(-1, N)), DevBuf((X.astype(np.float64) ** 2).sum(axis=(1, 2))),
             DevBuf.empty((E * M, N), np.float32), DevBuf.empty((nb // 4 + 64,), np.float32)]
        ws = (b[4].ptr + 255) // 256 * 256
        bufs.append(b)
        probs.append((_lib.NsProblem(b[0].ptr, b[1].ptr, b[2].ptr, b[3].ptr, ws, 1, E, M, N, nb), ws))

    def call(which, wipe=True):
        for q in which if wipe else ():                 # (nothing is left of an earlier call)
            for d in bufs[q][3:]:
                api.anc_fill_u32(d.ptr, 0x7F7F7F7F, d.size, 0)
        api.anc_ns_batched_pair_multi((_lib.NsProblem * len(which))(*[probs[q][0] for q in which]), len(which), 5, coef, 1e-7, MODES[mode], 0)
        return [(bufs[q][3].to_numpy(), ns_hard_info(probs[q][1], *groups[q][:3], 5, mode)) for q in which]
    alone = [call([q])[0] for q in range(len(groups))]
    for (E, M, N, kinds), (_, (n, _)) in zip(groups, alone):
        taken = ("lowrank", "band") if sched == "keller" else ("lowrank", "band", "cols")     # (Polar Express: by the proxy's gates too)
        assert n == sum(k in taken for k in kinds), (M, N)
    for which in (list(range(len(groups))), list(range(len(groups)))[::-1], [0, 1], [1, 0], [len(groups) - 1, 0, 1]):
        for wipe in (True, False):
            for q, (out, info) in zip(which, call(which, wipe)):
                assert bits_equal(out, alone[q][0]) and info == alone[q][1], (which, q)
    for b in bufs:
        for d in b:
            d.free()
