"""Batched solves of many molecules (stda_hip_batch_*) and the serving loop.

Mixed-precision bar (batched kernel and single-molecule mixed path): every
root within 1 meV and every oscillator strength (fL, fV) within 1e-4 of the
FP64 reference -- the FP64 oracle for the small molecules, the plain FP64 GPU
path (itself held to the oracle by test_gpu_parity.py) for all of them.  The
same molecule solved alone and inside a batch must give the same result
bit for bit: each molecule's kernels touch only its own data and reduce in a
fixed order.
"""
import sys

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

EV = 27.211385050
E_MIX = 1e-3 / EV          # 1 meV in Hartree
F_MIX = 1e-4


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def molecules():
    from stda_amd import synth
    # 10 molecules of 10-40 atoms plus two of ~80 atoms (nci > 4096: single path)
    cis = synth.mixed_batch(10, lo=10, hi=40, base_seed=500, workers=4)
    from stda_amd.prep import prepare
    for na, seed in ((80, 77), (84, 78)):
        mol, ints = synth.cluster(na, seed=seed, basis="minimal")
        cis.append(prepare(mol, 7.0, 0.25, ints))
    return cis


@pytest.fixture(scope="module")
def plain(molecules):
    """Plain FP64 GPU results per molecule: (omega, props) or the error status."""
    from stda_amd.core import StdaHip, StdaHipError
    out = []
    with StdaHip(0) as h:
        for ci in molecules:
            try:
                h.setup(ci, 7.0, 0.25)
                s = h.solve_tda(20, velcorr=True, tol=1e-8, vectors=False)
                out.append((s.omega.copy(), s.props.copy(), h.nci))
            except StdaHipError as e:
                out.append(e.status)
    return out


def test_batch_matches_fp64(molecules, plain):
    from stda_amd.core import StdaHipBatch
    say(f"batch of {len(molecules)} molecules, 4 workers")
    with StdaHipBatch(0, workers=4) as b:
        b.configure(nmax_batched=4096)     # the two ~80-atom molecules take the single path
        b.configure_wide(False)
        res = b.solve_tda(molecules, 7.0, 0.25, nroots=20, tol=1e-8, velcorr=True)
        t, cnt = b.timings()
        assert b.wide_count() == 0
    say(f"  paths {cnt}, timings {t}")
    assert cnt["batched"] >= 8 and cnt["single"] == 2
    for i, ((om, pr, st), ref) in enumerate(zip(res, plain)):
        if isinstance(ref, int):
            assert st == ref, (i, st, ref)
            continue
        assert st == 0, (i, st)
        rom, rpr, nci = ref
        assert len(om) == len(rom) == min(20, nci)
        say(f"  mol {i}: nci={nci} max|dE|={np.abs(om - rom).max() * EV:.2e} eV "
            f"max|dfL|={np.abs(pr[:, 0] - rpr[:, 0]).max():.2e}")
        np.testing.assert_allclose(om, rom, atol=E_MIX, rtol=0)
        np.testing.assert_allclose(pr[:, :2], rpr[:, :2], atol=F_MIX, rtol=0)


def test_batch_worker_solves(molecules):
    """A worker's own solves are laid out for the shared device: FP32 products at every size,
    subspace problems on the host, one FP64 step at the end (and the velocity correction's
    product), while a context alone solves the same molecules in FP64 with the kernel."""
    from stda_amd.core import StdaHip, StdaHipBatch
    stats = lambda x: {k: x.kernel_stats(k)["launches"] for k in
                       ("ao_matvec", "ao_matvec_f32", "dav_rr_eig", "mixed_fp64_refine")}
    with StdaHipBatch(0, workers=2) as b:
        b.configure(nmax_batched=4096)
        b.configure_wide(False)
        res = b.solve_tda(molecules[-2:], 7.0, 0.25, nroots=20)
        assert b.timings()[1]["single"] == 2
        k = stats(b)
    assert all(st == 0 for _, _, st in res)
    assert k["ao_matvec"] == 4 and k["mixed_fp64_refine"] == 2
    assert k["ao_matvec_f32"] == k["dav_rr_eig"] - 2 > 2
    with StdaHip(0) as h:
        h.setup(molecules[-1], 7.0, 0.25)
        h.set_precision("mixed")
        h.solve_tda(20)
        k = stats(h)
    assert k["ao_matvec"] > 2 and k["ao_matvec_f32"] == k["dav_rr_eig"] == k["mixed_fp64_refine"] == 0


def test_batch_bf16_single_path(molecules, plain):
    """Split-bfloat16 operator products on the single-molecule path of the
    workers (stda_hip_batch_set_precision 2): same bar against plain FP64."""
    from stda_amd.core import StdaHipBatch
    with StdaHipBatch(0, workers=3) as b:
        b.configure(nmax_batched=0)
        b.configure_wide(False)
        b.set_precision("bf16")
        res = b.solve_tda(molecules, 7.0, 0.25, nroots=20, tol=1e-8, velcorr=True)
        t, cnt = b.timings()
    say(f"  bf16 single path: paths {cnt}")
    assert cnt["single"] >= 10
    for i, ((om, pr, st), ref) in enumerate(zip(res, plain)):
        if isinstance(ref, int):
            assert st == ref, (i, st, ref)
            continue
        assert st == 0, (i, st)
        rom, rpr, nci = ref
        assert len(om) == len(rom) == min(20, nci)
        np.testing.assert_allclose(om, rom, atol=E_MIX, rtol=0)
        np.testing.assert_allclose(pr[:, :2], rpr[:, :2], atol=F_MIX, rtol=0)


def test_wide_matches_fp64(molecules, plain):
    """Matrix-free lock step: every molecule above 128 CSFs in the grouped
    kernels (FP32 operator products, FP64 Davidson numerics and refinement)."""
    from stda_amd.core import StdaHipBatch
    say(f"wide lock step: {len(molecules)} molecules, nmax_batched 128")
    with StdaHipBatch(0, workers=3) as b:
        b.configure(nmax_batched=128)
        res = b.solve_tda(molecules, 7.0, 0.25, nroots=20, tol=1e-8, velcorr=True)
        t, cnt = b.timings()
        nw = b.wide_count()
    say(f"  paths {cnt}, wide {nw}, timings {t}")
    assert nw >= 6 and cnt["single"] == 0
    for i, ((om, pr, st), ref) in enumerate(zip(res, plain)):
        if isinstance(ref, int):
            assert st == ref, (i, st, ref)
            continue
        assert st == 0, (i, st)
        rom, rpr, nci = ref
        assert len(om) == len(rom) == min(20, nci)
        say(f"  mol {i}: nci={nci} max|dE|={np.abs(om - rom).max() * EV:.2e} eV "
            f"max|dfL|={np.abs(pr[:, 0] - rpr[:, 0]).max():.2e} "
            f"max|dfV|={np.abs(pr[:, 1] - rpr[:, 1]).max():.2e}")
        np.testing.assert_allclose(om, rom, atol=E_MIX, rtol=0)
        np.testing.assert_allclose(pr[:, :2], rpr[:, :2], atol=F_MIX, rtol=0)


def test_wide_alone_equals_in_batch(molecules):
    from stda_amd.core import StdaHipBatch
    with StdaHipBatch(0, workers=3) as b:
        b.configure(nmax_batched=128)
        mix = b.solve_tda(molecules, 7.0, 0.25, nroots=20)
        for i in (1, len(molecules) - 1):
            alone = b.solve_tda([molecules[i]], 7.0, 0.25, nroots=20)[0]
            assert b.wide_count() == (1 if alone[2] == 0 else 0)
            np.testing.assert_array_equal(alone[0], mix[i][0])
            np.testing.assert_array_equal(alone[1], mix[i][1])
            assert alone[2] == mix[i][2]


def test_batch_matches_oracle(molecules):
    from stda_amd.core import StdaHipBatch
    small = [ci for ci in molecules if ci.ncent <= 25]
    assert small
    with StdaHipBatch(0, workers=2) as b:
        res = b.solve_tda(small, 7.0, 0.25, nroots=20, tol=1e-8, velcorr=True)
    for ci, (om, pr, st) in zip(small, res):
        try:
            ref = O.run(ci, 7.0, 0.25, nroots=20)
        except RuntimeError:      # no CSF
            assert st == 2
            continue
        assert st == 0
        np.testing.assert_allclose(om, ref.omega, atol=E_MIX, rtol=0)
        np.testing.assert_allclose(pr[:, :2], ref.props[:, :2], atol=F_MIX, rtol=0)


def test_alone_equals_in_batch(molecules):
    from stda_amd.core import StdaHipBatch
    with StdaHipBatch(0, workers=3) as b:
        mix = b.solve_tda(molecules, 7.0, 0.25, nroots=20)
        for i in (0, 3, len(molecules) - 1):
            alone = b.solve_tda([molecules[i]], 7.0, 0.25, nroots=20)[0]
            np.testing.assert_array_equal(alone[0], mix[i][0])
            np.testing.assert_array_equal(alone[1], mix[i][1])
            assert alone[2] == mix[i][2]


def test_server_alone_equals_in_mix(molecules, plain):
    """Continuous batching: spectrum jobs and polarizability jobs admitted as
    they arrive; every result equals the same job run alone."""
    from stda_amd.serve import Server, Job
    jobs = []
    for i, ci in enumerate(molecules):
        kind = "polar" if i % 3 == 2 else "spectrum"
        jobs.append(Job(jid=i, kind=kind, ci=ci, omegas=(0.0, 0.05)))
    with Server(workers=4, hbm_budget=64e9, batch_workers=4) as srv:
        st = srv.run(jobs, realtime=False)
        say(f"  served {st.n} jobs in {st.wall:.3f}s; p50 {st.p50_ms:.1f} ms")
        for j in jobs:
            alone = Job(jid=j.jid, kind=j.kind, ci=j.ci, omegas=j.omegas)
            srv.run([alone], realtime=False)
            assert j.error == alone.error
            if j.error:
                continue
            if j.kind == "spectrum":
                np.testing.assert_array_equal(j.result[0], alone.result[0])
                np.testing.assert_array_equal(j.result[1], alone.result[1])
                ref = plain[j.jid]
                np.testing.assert_allclose(j.result[0], ref[0], atol=E_MIX, rtol=0)
            else:
                for (w1, a1), (w2, a2) in zip(j.result, alone.result):
                    assert w1 == w2
                    np.testing.assert_array_equal(a1, a2)


def test_continuous_mode_equals_closed(molecules):
    """Continuous mode (stda_hip_batch_submit/result): molecules submitted in two waves,
    the second while the first are in the running lock-step set, give bit for bit the
    results of the closed batch call; the closed call works again after stop."""
    import time
    from stda_amd.core import StdaHipBatch
    with StdaHipBatch(0, workers=3) as b:
        closed = b.solve_tda(molecules, 7.0, 0.25, nroots=20)
        first = [b.submit(ci, 7.0, 0.25, 20) for ci in molecules[:6]]
        time.sleep(0.002)
        second = [b.submit(ci, 7.0, 0.25, 20) for ci in molecules[6:]]
        got = [b.result(t) for t in first + second]
        b.stop()
        again = b.solve_tda(molecules[:2], 7.0, 0.25, nroots=20)
    for i, ((om, pr, st), (om0, pr0, st0)) in enumerate(zip(got, closed)):
        assert st == st0, (i, st, st0)
        np.testing.assert_array_equal(om, om0)
        np.testing.assert_array_equal(pr, pr0)
    for (om, pr, st), (om0, pr0, st0) in zip(again, closed[:2]):
        assert st == st0
        np.testing.assert_array_equal(om, om0)
