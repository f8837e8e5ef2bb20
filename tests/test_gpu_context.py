"""What a context keeps between calls: scratch memory, idle search tables and
captured graphs never change a result, whichever call came before."""
import threading

import numpy as np
import pytest

import cdocker_amd as cdk
from cdocker_amd import workloads

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu]", *a, flush=True)


@pytest.fixture(scope="module")
def ctx():
    c = cdk.Context(0)
    yield c
    c.close()


def make(ctx, n=48, natom_protein=500):
    vals, radii, mid, ln = cdk.synth_protein(15, natom_protein, 0.5 * n, n, 0.5)
    return cdk.Protein(ctx, vals, radii, 0.5, mid, ln)


def bits(*arrays):
    return [np.ascontiguousarray(a).view(np.uint8).tobytes() for a in arrays if a is not None]


def test_scratch_is_counted_and_given_back(ctx):
    """The bytes kept for the next calls can be read, are given back when the
    limit is lowered, stay given back while it is 0, and do not change results."""
    say("scratch")
    prot = make(ctx)
    x, q, e, r = cdk.synth_ligand(3, 12)
    lig = cdk.Ligand(prot, q, e, r)
    quats = cdk.QuaternionUniformSampling(cdk.Rng(5), 40)
    rot, mv, ex = workloads.chain_topology(12)
    poses = x[None].astype(np.float64) + np.linspace(9, 12, 30)[:, None, None]

    def calls():
        return bits(*cdk.search(ctx, prot, lig, x[None], quats), *cdk.rescore_poses(prot, lig, poses, want_grad=True),
                    *cdk.refine_poses(prot, lig, poses, steps=4),
                    *cdk.generate_conformers(ctx, x, rot, mv, ex, 60, 3, 0.6), prot.grids())

    assert ctx.get_option("scratch_keep_bytes") == 128 << 20
    first = calls()
    kept = ctx.get_option("scratch_bytes")
    assert 0 < kept <= 3 * (128 << 20)
    try:
        ctx.set_option("scratch_keep_bytes", 0)
        assert ctx.get_option("scratch_bytes") == 0
        assert calls() == first
        assert ctx.get_option("scratch_bytes") == 0
        with pytest.raises(cdk.CdkError):
            ctx.set_option("scratch_keep_bytes", -1)
    finally:
        ctx.set_option("scratch_keep_bytes", 128 << 20)
    assert calls() == first and ctx.get_option("scratch_bytes") > 0
    lig.close()
    prot.close()


def test_conformers_that_all_pass_need_no_more_memory(ctx):
    """A call that keeps every one of many trials runs them in sets of bounded
    memory: the scratch it leaves is below the coordinates it returns, trial
    numbers are complete, and conformers across sets are those of a call for
    fewer (trials depend on their number alone)."""
    natom, ntrial = 24, 150000
    x, q, e, r = cdk.synth_ligand(77, natom)
    rot, mv, ex = workloads.chain_topology(natom)
    ctx.set_option("scratch_keep_bytes", 0)
    try:
        ctx.set_option("scratch_keep_bytes", 1 << 40)
        say("conformers, all kept")
        conf, trial = cdk.generate_conformers(ctx, x, rot, mv, ex, ntrial, 9, 1e-6)
        used = ctx.get_option("scratch_bytes")
    finally:
        ctx.set_option("scratch_keep_bytes", 128 << 20)
    assert np.array_equal(trial, np.arange(ntrial))
    assert used < ntrial * natom * 24 + (24 << 20)
    few, t = cdk.generate_conformers(ctx, x, rot, mv, ex, 70000, 9, 1e-6, max_keep=69990)
    assert np.array_equal(t, np.arange(69990)) and np.array_equal(few, conf[:69990])


@pytest.mark.parametrize("natom,npose", [(40, 4346), (40, 9000), (1, 120000), (300, 601), (512, 342)])
def test_poses_in_pieces(ctx, natom, npose):
    """Rescoring and refinement of more poses than one piece of the pinned
    memory holds (two and more pieces, whole and odd remainders): bit for bit
    the results of the same poses in calls of their own."""
    say("pieces natom=%d npose=%d" % (natom, npose))
    prot = make(ctx)
    rs = np.random.default_rng(natom)
    _, q, e, r = cdk.synth_ligand(19, natom)
    lig = cdk.Ligand(prot, q, e, r)
    x = rs.normal(0, 2.0, (natom, 3))
    poses = x[None] + rs.uniform(7, 16, (npose, 1, 3))
    cuts = np.unique([0, 50, npose // 4, npose // 2, 3 * npose // 4, npose - 1, npose])
    parts = list(zip(cuts, cuts[1:]))
    for grad in (True, False):
        E, g, ins = cdk.rescore_poses(prot, lig, poses, want_grad=grad)
        assert np.isfinite(E).all() and len(np.unique(E)) > 100
        for a, b in parts:
            for lo, hi in ((a, min(a + 300, b)), (max(a, b - 300), b)):
                Es, gs, inss = cdk.rescore_poses(prot, lig, poses[lo:hi], want_grad=grad)
                assert bits(Es, gs, inss) == bits(E[lo:hi], g[lo:hi] if grad else None, ins[lo:hi]), (lo, hi)
    X, E = cdk.refine_poses(prot, lig, poses, steps=2)
    for a, b in parts:
        for lo, hi in ((a, min(a + 200, b)), (max(a, b - 200), b)):
            Xs, Es = cdk.refine_poses(prot, lig, poses[lo:hi], steps=2)
            assert bits(Xs, Es) == bits(X[lo:hi], E[lo:hi]), (lo, hi)
    lig.close()
    prot.close()


@pytest.mark.parametrize("nch", [2, 15, 16])
def test_protein_memory_by_size(ctx, nch):
    """32^3 proteins on both sides of the size from which one allocation holds
    every array (16 channels): grids read back bit for bit, spectra are the
    grids' transforms, and the fused engine (which reads another copy of the
    spectra) agrees with the reference dataflow."""
    say("protein channels", nch)
    rs = np.random.default_rng(nch)
    n = 32
    v = rs.normal(0, 1, (nch, n, n, n)).astype(np.float32)
    radii = np.linspace(1.0, 2.2, nch - 1).astype(np.float32)
    prot = cdk.Protein(ctx, v, radii, 0.5)
    H = nch * n * n * (n // 2 + 1) * 8
    assert v.nbytes + 2 * H <= prot.device_bytes() <= v.nbytes + 2 * H + 5 * 256
    assert bits(prot.grids()) == bits(v)
    for c in (0, nch - 1):
        ref = np.fft.rfftn(v[c].astype(np.float64))
        assert np.abs(prot.spectrum(c) - ref).max() <= 1e-5 * np.abs(ref).max()
    x, q, e, r = cdk.synth_ligand(23, 7)
    lig = cdk.Ligand(prot, q, e, r)
    quats = cdk.QuaternionUniformSampling(cdk.Rng(7), 9)
    E, idx, _ = cdk.search(ctx, prot, lig, x[None], quats)
    R, ridx, _ = cdk.search(ctx, prot, lig, x[None], quats, engine=cdk.ENGINE_REFERENCE)
    assert np.isfinite(R).all() and np.abs(E - R).max() <= 1e-4 * np.abs(R).max()
    lig.close()
    prot.close()


@pytest.mark.parametrize("n,pipeline,chunk", [(64, 2, 0), (64, 2, 7), (64, 1, 16), (64, 0, 16), (48, 0, 9), (96, 2, 11)])
@pytest.mark.parametrize("overlap", [0, 1])
def test_batch_graph_capture_and_replays(ctx, n, pipeline, chunk, overlap):
    """One Batch run again and again: launched eagerly, captured, then replayed,
    with eager searches on the same context between the runs, and captured anew
    after the schedule changes, the working memory moves or a job is added.
    Every run has the bits of a Batch that never uses a graph."""
    say("graph n=%d pipeline=%d chunk=%d overlap=%d" % (n, pipeline, chunk, overlap))
    prot = make(ctx, n)
    jobs = []
    for i in range(4):
        x, q, e, r = cdk.synth_ligand(40 + i, 9 + 5 * i)
        jobs.append((cdk.Ligand(prot, q, e, r), x[None], cdk.QuaternionUniformSampling(cdk.Rng(50 + i), 11)))

    def eager(k):
        ctx.set_option("use_graph", 0)
        b = cdk.Batch(ctx, prot)
        for j in jobs[:k]:
            b.add(*j)
        out = []
        for _ in range(2):
            b.run()
            out.append([bits(*b.results(i)) for i in range(k)])
        b.close()
        ctx.set_option("use_graph", 1)
        assert out[0] == out[1]
        return out[0]

    try:
        ctx.set_option("overlap_z", overlap)
        ctx.set_option("pipeline", pipeline)
        ctx.set_option("fused_chunk", chunk)
        want = {k: eager(k) for k in (3, 4)}
        b = cdk.Batch(ctx, prot)
        for j in jobs[:3]:
            b.add(*j)
        for run in range(9):
            if run == 4:
                ctx.set_option("mid_group", 3)  # captured anew
            if run == 6:
                ctx.set_option("mid_group", 0)
                ctx.set_option("fused_chunk", 40)
                cdk.search(ctx, prot, *jobs[3])  # the working memory grows
                ctx.set_option("fused_chunk", chunk)
            b.run()
            assert [bits(*b.results(i)) for i in range(3)] == want[3], run
            cdk.search(ctx, prot, *jobs[run % 4])
        b.add(*jobs[3])
        for run in range(4):
            b.run()
            assert [bits(*b.results(i)) for i in range(4)] == want[4], run
        b.close()
    finally:
        for k, v in (("overlap_z", 1), ("pipeline", -1), ("fused_chunk", 0), ("mid_group", 0), ("use_graph", 1)):
            ctx.set_option(k, v)
        for j in jobs:
            j[0].close()
        prot.close()


def test_searches_of_several_threads(ctx):
    """Threads that search, rescore and make conformers on one context at once
    get what each gets alone: no two calls share kept tables or scratch."""
    say("threads")
    prots = {n: make(ctx, n) for n in (48, 64)}
    rot, mv, ex = workloads.chain_topology(14)

    def call(k):
        prot = prots[(48, 64)[k % 2]]
        x, q, e, r = cdk.synth_ligand(60 + k, 6 + 2 * k)
        lig = cdk.Ligand(prot, q, e, r)
        quats = cdk.QuaternionUniformSampling(cdk.Rng(70 + k), 5 + 9 * k)
        out = bits(*cdk.search(ctx, prot, lig, x[None], quats))
        poses = x[None].astype(np.float64) + np.linspace(9, 12, 20 + k)[:, None, None]
        out += bits(*cdk.rescore_poses(prot, lig, poses, want_grad=True))
        xc = cdk.synth_ligand(80 + k, 14)[0]
        out += bits(*cdk.generate_conformers(ctx, xc, rot, mv, ex, 200, k, 0.6))
        lig.close()
        return out

    for k in (0, 1):
        call(k)  # the forms are chosen
    want = [call(k) for k in range(8)]
    got, errors = [[] for _ in range(8)], []

    def work(k):
        try:
            for _ in range(6):
                got[k].append(call(k))
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for k in range(8):
        assert len(got[k]) == 6 and all(g == want[k] for g in got[k]), k
    for p in prots.values():
        p.close()


def test_calls_after_calls_that_failed(ctx):
    """A call that is refused, before or after its tables are built, leaves
    nothing behind: the next calls have the results of a fresh context."""
    say("failed calls")
    prot = make(ctx)
    x, q, e, r = cdk.synth_ligand(5, 11)
    lig = cdk.Ligand(prot, q, e, r)
    quats = cdk.QuaternionUniformSampling(cdk.Rng(9), 33)
    rot, mv, ex = workloads.chain_topology(11)
    poses = x[None].astype(np.float64) + np.linspace(9, 12, 12)[:, None, None]

    def calls():
        return bits(*cdk.search(ctx, prot, lig, x[None], quats), *cdk.refine_poses(prot, lig, poses, steps=3),
                    *cdk.generate_conformers(ctx, x, rot, mv, ex, 50, 3, 0.6))

    want = calls()
    bad_quats = quats.copy()
    bad_quats[-1, 2] = np.nan
    bad_x = np.repeat(x[None], 2, 0)
    bad_x[1, -1, 0] = np.inf
    bad_rot = rot.copy()
    bad_rot[-1, 3] = 99
    for refused in (lambda: cdk.search(ctx, prot, lig, x[None], bad_quats),
                    lambda: cdk.search(ctx, prot, lig, bad_x, quats),
                    lambda: cdk.generate_conformers(ctx, x, bad_rot, mv, ex, 50, 3, 0.6),
                    lambda: cdk.Protein(ctx, np.zeros((1, 48, 48, 48)), [1.0], 0.5),
                    lambda: cdk.Protein(ctx, np.zeros((3, 40, 40, 40)), [1.0, 1.5], 0.5)):
        with pytest.raises(cdk.CdkError):
            refused()
        assert calls() == want
    lig.close()
    prot.close()


@pytest.mark.parametrize("engine", [cdk.ENGINE_FUSED, cdk.ENGINE_REFERENCE])
def test_searches_too_large_to_keep(ctx, engine):
    """A search whose tables are not kept for the next call copies them and its
    results in pieces (one, four slots and more, remainders): bit for bit the
    results of a kept one, with and without the optional arrays' poses found."""
    prot = make(ctx, 32, 200)
    x, q, e, r = cdk.synth_ligand(29, 5)
    x = np.stack([x, 20.0 * x]).astype(np.float32)  # the second conformer does not fit the grid
    lig = cdk.Ligand(prot, q, e, r)
    sizes = (1, 14527, 14528, 14529, 60000) if engine == cdk.ENGINE_FUSED else (70, 15000)
    try:
        for n in sizes:
            say("search not kept, engine %d, 2 x %d poses" % (engine, n))
            quats = np.resize(cdk.QuaternionUniformSampling(cdk.Rng(n), min(n, 4000)), (n, 4))
            ctx.set_option("scratch_keep_bytes", 128 << 20)
            want = cdk.search(ctx, prot, lig, x, quats, engine=engine)
            ctx.set_option("scratch_keep_bytes", 0)
            got = cdk.search(ctx, prot, lig, x, quats, engine=engine)
            assert ctx.get_option("scratch_bytes") == 0
            assert bits(*got) == bits(*want)
            assert np.isfinite(want[0][0]).all() and not np.isfinite(want[0][1]).all()
    finally:
        ctx.set_option("scratch_keep_bytes", 128 << 20)
        lig.close()
        prot.close()
