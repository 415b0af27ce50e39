"""Parity of the GPU CCSD path with the FP64 oracle, through the C ABI.

Bar (FP64 path): correlation energy within 1e-9 Eh of the oracle, amplitudes
within 1e-8 relative; single residuum evaluations within 1e-12 relative.
"""

import json
import pathlib

import numpy as np
import pytest

from cc4s_amd import api
from cc4s_amd import synthetic as syn
from oracle import ccsd_oracle as O
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

GOLDEN = pathlib.Path(__file__).parent / "golden"
E_TOL = 1e-9       # Eh
T_TOL = 1e-8       # relative
R_TOL = 1e-12      # relative, one residuum


def _setup(No, Nv, NG, field, seed, **kw):
    inp = syn.generate(No, Nv, NG, field, seed)
    cc = api.CoupledCluster(No, Nv, NG, field=field, **kw)
    cc.set_inputs(inp.gamma, inp.eps)
    P = O.CcsdProblem(inp.gamma, inp.eps, No, field, ppl=kw.get("ppl", True),
                      integrals_slice_size=kw.get("integralsSliceSize") or None)
    return cc, P, inp


def _amps(No, Nv, field, seed, scale=0.05):
    T1, T2 = syn.random_amplitudes(No, Nv, field, seed, t1_scale=scale,
                                   t2_scale=scale)
    if field == "real":
        return T1.real.copy(), T2.real.copy()
    return T1, T2


@pytest.mark.parametrize("field", ["complex", "real"])
@pytest.mark.parametrize("shape", [(3, 7, 5), (4, 12, 30), (8, 40, 200)],
                         ids=["o3v7G5", "o4v12G30", "o8v40G200"])
def test_residuum_parity(field, shape):
    No, Nv, NG = shape
    print(f"residuum parity {field} {shape}", flush=True)
    cc, P, _ = _setup(No, Nv, NG, field, seed=21, integralsSliceSize=3)
    T = _amps(No, Nv, field, 13)
    R1, R2 = cc.residuum(T)
    Q1, Q2 = P.residuum(T)
    assert rel_err(R1, Q1) < R_TOL
    assert rel_err(R2, Q2) < R_TOL
    # first residuum: R1 = 0, R2 = V_abij
    R1, R2 = cc.residuum(None)
    Q1, Q2 = P.residuum(None)
    assert np.all(R1 == 0) and rel_err(R2, Q2) < 1e-14
    cc.close()


def test_residuum_parity_non_hermitian_vertex():
    """A vertex without Gamma_qp = conj Gamma_pq: V_hhpp is then formed and
    stored instead of being read as the conjugate transpose of V_pphh."""
    No, Nv, NG = 4, 12, 30
    inp = syn.generate(No, Nv, NG, "complex", 21)
    rng = np.random.default_rng(4)
    g = inp.gamma + 0.003 * (rng.standard_normal(inp.gamma.shape)
                             + 1j * rng.standard_normal(inp.gamma.shape))
    cc = api.CoupledCluster(No, Nv, NG, field="complex", integralsSliceSize=5)
    cc.set_inputs(g, inp.eps)
    P = O.CcsdProblem(g, inp.eps, No, "complex", integrals_slice_size=5)
    T = _amps(No, Nv, "complex", 13)
    R1, R2 = cc.residuum(T)
    Q1, Q2 = P.residuum(T)
    assert rel_err(R1, Q1) < R_TOL
    assert rel_err(R2, Q2) < R_TOL
    cc.close()


@pytest.mark.parametrize("placement,chunk,pinned", [
    ("host", None, True), ("host", 4096, True), ("host_all", None, True),
    ("host_all", 4096, True), ("host_all", 4096, False)])
@pytest.mark.parametrize("field", ["complex", "real"])
def test_diis_slots_on_host(field, placement, chunk, pinned, monkeypatch):
    """DIIS slots in host memory (the amplitude slots, or every slot,
    streamed through HBM in chunks; 4096-byte chunks split the sets many
    times, across the T1/T2 boundary; pinned, or pageable as when the
    system's pinned memory is exhausted) give the oracle's run."""
    monkeypatch.setenv("CC4S_DIIS_PLACEMENT", placement)
    if chunk:
        monkeypatch.setenv("CC4S_DIIS_CHUNK_BYTES", str(chunk))
    if not pinned:
        monkeypatch.setenv("CC4S_DIIS_PINNED", "0")
    print(f"placement {placement} chunk {chunk} pinned {pinned} field {field}", flush=True)
    kw = dict(maxIterations=30, energyConvergence=1e-10,
              amplitudesConvergence=1e-8, maxResidua=5)
    gpu, T_gpu, ref = _run_both(4, 14, 25, field, 17, **kw)
    _check_run(gpu, T_gpu, ref)


@pytest.mark.parametrize("field", ["complex", "real"])
def test_energy_parity(field):
    No, Nv, NG = 5, 16, 40
    cc, P, _ = _setup(No, Nv, NG, field, seed=4)
    T = _amps(No, Nv, field, 8)
    E, D, X = cc.energy(T)
    Eo, Do, Xo = O.energy(P, T)
    assert abs(E - Eo) < 1e-14 and abs(D - Do) < 1e-14 and abs(X - Xo) < 1e-14
    cc.close()


def _run_both(No, Nv, NG, field, seed, **kw):
    cc, P, inp = _setup(No, Nv, NG, field, seed, **kw)
    gpu = cc.run()
    T_gpu = cc.amplitudes()
    cc.close()
    ref = O.coupled_cluster(
        P, max_iterations=kw.get("maxIterations", 16),
        energy_convergence=kw.get("energyConvergence", 1e-7),
        amplitudes_convergence=kw.get("amplitudesConvergence", 1e-6),
        level_shift=kw.get("levelShift", 0.0),
        max_residua=kw.get("maxResidua", 4))
    return gpu, T_gpu, ref


def _check_run(gpu, T_gpu, ref):
    assert gpu["convergenceReached"] == ref["convergenceReached"]
    assert gpu["iterations"] == ref["iterations"]
    for key in ("correlation", "direct", "exchange", "secondOrder"):
        assert abs(gpu["energy"][key] - ref["energy"][key]) < E_TOL, key
    for g, r in zip(gpu["trace"], ref["trace"]):
        assert abs(g["energy"] - r[0]) < E_TOL
    assert rel_err(T_gpu[0], ref["amplitudes"][0]) < T_TOL
    assert rel_err(T_gpu[1], ref["amplitudes"][1]) < T_TOL


def test_run_parity_real_no8_nv40_ng200():
    """The real No=8, Nv=40, NG=200 workload to convergence, DIIS 8."""
    cfg = syn.WORKLOADS["real_no8_nv40_ng200"]
    print("run parity, real No=8 Nv=40 NG=200", flush=True)
    kw = dict(maxIterations=cfg.max_iterations,
              energyConvergence=cfg.energy_convergence,
              amplitudesConvergence=cfg.amplitudes_convergence,
              maxResidua=cfg.max_residua)
    gpu, T_gpu, ref = _run_both(cfg.No, cfg.Nv, cfg.NG, cfg.field, cfg.seed, **kw)
    _check_run(gpu, T_gpu, ref)
    gold = json.loads((GOLDEN / "real_no8_nv40_ng200.json").read_text())
    assert gpu["iterations"] == gold["iterations"]
    assert abs(gpu["energy"]["correlation"] - gold["energy"]["correlation"]) < E_TOL
    for g, r in zip(gpu["trace"], gold["trace"]):
        assert abs(g["energy"] - r[0]) < E_TOL


def test_run_parity_small_complex():
    gold = json.loads((GOLDEN / "small_complex.json").read_text())
    c = gold["config"]
    print("run parity small complex", flush=True)
    kw = dict(maxIterations=c["max_iterations"],
              energyConvergence=c["energy_convergence"],
              amplitudesConvergence=c["amplitudes_convergence"],
              maxResidua=c["max_residua"])
    gpu, T_gpu, ref = _run_both(c["No"], c["Nv"], c["NG"], c["field"], c["seed"], **kw)
    _check_run(gpu, T_gpu, ref)
    assert abs(gpu["energy"]["correlation"] - gold["energy"]["correlation"]) < E_TOL


@pytest.mark.parametrize("field", ["complex", "real"])
@pytest.mark.parametrize("opts", [
    dict(levelShift=0.2), dict(ppl=False), dict(maxResidua=1),
    dict(integralsSliceSize=5), dict(maxIterations=2)],
    ids=["levelShift", "noPpl", "jacobi", "slice5", "notConverged"])
def test_run_options(field, opts):
    print(f"run options {field} {opts}", flush=True)
    kw = dict(maxIterations=30, energyConvergence=1e-10,
              amplitudesConvergence=1e-8)
    kw.update(opts)
    gpu, T_gpu, ref = _run_both(4, 14, 25, field, 17, **kw)
    _check_run(gpu, T_gpu, ref)


def test_initial_amplitudes_and_zero_iterations():
    """maxIterations 0 evaluates the energy of given amplitudes
    (CoupledCluster.cxx:177-178)."""
    No, Nv, NG = 4, 12, 20
    cc, P, _ = _setup(No, Nv, NG, "complex", 3, maxIterations=0)
    T = _amps(No, Nv, "complex", 2)
    cc.set_amplitudes(*T)
    out = cc.run()
    E, D, X = O.energy(P, T)
    assert out["iterations"] == 0 and not out["convergenceReached"]
    assert abs(out["energy"]["correlation"] - E.real) < 1e-14
    cc.close()


def test_zero_iterations_without_amplitudes_fails():
    cc, _, _ = _setup(3, 6, 5, "complex", 3, maxIterations=0)
    with pytest.raises(api.CcsdError, match="initialAmplitudes"):
        cc.run()
    cc.close()


def test_config1_properties():
    """The complex No=32, Nv=256, NG=1500 workload: properties that do
    not need the oracle at this size.  The residuum of symmetric amplitudes
    is pair-symmetric (R_abij = R_baji), independent of the ladder slice
    size, and its first iteration reproduces the MP2 energy."""
    cfg = syn.WORKLOADS["complex_no32_nv256_ng1500"]
    print("config1 properties: generating inputs", flush=True)
    inp = syn.generate_config(cfg)
    T = _amps(cfg.No, cfg.Nv, "complex", 5, scale=0.01)
    res = {}
    for s in (32, 64):
        print(f"config1 residuum, integralsSliceSize {s}", flush=True)
        with api.CoupledCluster(cfg.No, cfg.Nv, cfg.NG, field="complex",
                                integralsSliceSize=s) as cc:
            cc.set_inputs(inp.gamma, inp.eps)
            res[s] = cc.residuum(T)
            if s == 32:
                R1, R2 = cc.residuum(None)
                V = R2
                it = cc.iterate()
    R1, R2 = res[32]
    assert rel_err(R2, R2.transpose(1, 0, 3, 2)) < 1e-13
    assert rel_err(res[64][1], R2) < 1e-12
    assert rel_err(res[64][0], R1) < 1e-12
    eh, ep = inp.eps[:cfg.No], inp.eps[cfg.No:]
    dph = ep[:, None] - eh[None, :]
    Dpphh = dph[:, None, :, None] + dph[None, :, None, :]
    Tm = np.conj(V) / Dpphh
    mp2 = (-2.0 * np.sum(V * Tm) + np.sum(V.transpose(0, 1, 3, 2) * Tm)).real
    assert abs(it["energy"] - mp2) < 1e-13 * abs(mp2)


@pytest.mark.parametrize("field", ["complex", "real"])
@pytest.mark.parametrize("opts", [dict(), dict(linearized=True),
                                  dict(adjacentPairsExchange=True)],
                         ids=["quadratic", "linearized", "adjacentPairsExchange"])
def test_drccd_parity(field, opts):
    """Drccd (Drccd.cxx:31-109): one residuum against the oracle's explicit-V
    statements, then a run to convergence."""
    No, Nv, NG = 4, 12, 30
    print(f"drccd {field} {opts}", flush=True)
    inp = syn.generate(No, Nv, NG, field, 5)
    kw = dict(maxIterations=40, energyConvergence=1e-10, amplitudesConvergence=1e-8)
    P = O.CcsdProblem(inp.gamma, inp.eps, No, field, method="Drccd",
                      linearized=opts.get("linearized", False),
                      adjacent_pairs_exchange=opts.get("adjacentPairsExchange", False))
    with api.CoupledCluster(No, Nv, NG, field=field, method="Drccd", **opts, **kw) as cc:
        cc.set_inputs(inp.gamma, inp.eps)
        T = _amps(No, Nv, field, 13)
        T = (np.zeros_like(T[0]), T[1])
        R1, R2 = cc.residuum(T)
        Q1, Q2 = P.residuum(T)
        assert np.all(R1 == 0)
        assert rel_err(R2, Q2) < R_TOL
        gpu = cc.run()
        T_gpu = cc.amplitudes()
    ref = O.coupled_cluster(P, max_iterations=40, energy_convergence=1e-10,
                            amplitudes_convergence=1e-8)
    _check_run(gpu, T_gpu, ref)


def test_ueg_energies_of_the_reference_test_suite():
    """Uniform electron gas rs=1, No=7, Nv=26 (inputs restated from
    UegVertexGenerator.cxx): the GPU Drccd and Ccsd energies equal those the
    reference recorded in test/tests/ueg/rs1.0-7occ-26virt/correct.out.yaml,
    within 1e-9 Eh (the reference's own check uses 1e-7)."""
    from oracle import ueg
    gamma, eps, _ = ueg.generate(7, 26, 1.0)
    ref = ueg.UEG_RS1_NO7_NV26
    s = ref["settings"]
    kw = dict(maxIterations=s["maxIterations"], energyConvergence=s["energyConvergence"],
              amplitudesConvergence=s["amplitudesConvergence"], maxResidua=s["maxResidua"])
    for method, extra in (("Drccd", {}), ("Ccsd", dict(integralsSliceSize=s["integralsSliceSize"]))):
        with api.CoupledCluster(7, 26, gamma.shape[0], method=method, **kw, **extra) as cc:
            cc.set_inputs(gamma, eps)
            out = cc.run()
        print(method, out["energy"], out["iterations"], flush=True)
        assert out["convergenceReached"]
        for key in ("correlation", "direct", "exchange", "secondOrder"):
            assert abs(out["energy"][key] - ref[method][key]) < 1e-9, (method, key)


@pytest.mark.parametrize("field", ["complex", "real"])
@pytest.mark.parametrize("shape", [(3, 7, 5), (4, 12, 30), (5, 33, 20)],
                         ids=["o3v7G5", "o4v12G30", "o5v33G20"])
def test_triples_parity(field, shape):
    """(T) of given amplitudes (PerturbativeTriplesReference.cxx:55-180)
    against the oracle's restatement, 1e-12 relative.  The complex field
    pairs each particle term (K = Nv) with a hole term (K = No) in one
    two-segment contraction; Nv = 7 and 33 pad the first segment to whole
    K-stages of 16."""
    No, Nv, NG = shape
    print(f"triples {field} {shape}", flush=True)
    inp = syn.generate(No, Nv, NG, field, 23)
    T = _amps(No, Nv, field, 29, scale=0.1)
    with api.CoupledCluster(No, Nv, NG, field=field) as cc:
        cc.set_inputs(inp.gamma, inp.eps)
        cc.set_amplitudes(*T)
        e = cc.triples()
    ref = O.perturbative_triples(inp.gamma, inp.eps, No, field, T)
    assert abs(e - ref) <= 1e-12 * abs(ref)


# (shape, bytes of connected amplitudes per chunk): Nv on both sides of the 8 x 8
# blocks of (x2, x3), of the 64- and 96-column tiles and of two of them; all hole
# triples in one launch, one triple in three parts, one triple part by part
TRIPLES_CASES = [((2, 3, 5), None), ((3, 8, 9), None), ((17, 18, 9), None), ((2, 64, 10), None),
                 ((2, 65, 10), None), ((2, 96, 10), None), ((2, 97, 10), None),
                 ((3, 33, 20), "three"), ((3, 33, 20), "one"), ((3, 66, 10), "one")]


@pytest.mark.parametrize("field", ["complex", "real"])
@pytest.mark.parametrize("shape,chunk", TRIPLES_CASES)
def test_triples_tile_edges_and_chunks(field, shape, chunk, monkeypatch):
    """As test_triples_parity: sums of 2 (Nv + No) products per amplitude, same
    1e-12 relative."""
    No, Nv, NG = shape
    print(f"triples {field} {shape} {chunk}", flush=True)
    if chunk:
        part = Nv ** 3 * (16 if field == "complex" else 8)
        monkeypatch.setenv("CC4S_TRIPLES_W_BYTES", str({"three": 3, "one": 1}[chunk] * part))
    inp = syn.generate(No, Nv, NG, field, 31)
    T = _amps(No, Nv, field, 37, scale=0.1)
    with api.CoupledCluster(No, Nv, NG, field=field) as cc:
        cc.set_inputs(inp.gamma, inp.eps)
        cc.set_amplitudes(*T)
        e = cc.triples()
        assert e == cc.triples()
    ref = O.perturbative_triples(inp.gamma, inp.eps, No, field, T)
    assert abs(e - ref) <= 1e-12 * abs(ref)


def test_ueg_triples_of_the_reference_test_suite():
    """(T) of the GPU CCSD amplitudes of the uniform electron gas rs=1, No=7,
    Nv=26 equals the reference's recorded PerturbativeTriplesReference
    energy (correct.out.yaml:166-170) within 1e-10 Eh."""
    from oracle import ueg
    gamma, eps, _ = ueg.generate(7, 26, 1.0)
    ref = ueg.UEG_RS1_NO7_NV26
    s = ref["settings"]
    with api.CoupledCluster(7, 26, gamma.shape[0], maxIterations=s["maxIterations"],
                            energyConvergence=s["energyConvergence"],
                            amplitudesConvergence=s["amplitudesConvergence"],
                            maxResidua=s["maxResidua"],
                            integralsSliceSize=s["integralsSliceSize"]) as cc:
        cc.set_inputs(gamma, eps)
        assert cc.run()["convergenceReached"]
        e = cc.triples()
    assert abs(e - ref["Triples"]["correlation"]) < 1e-10


def test_ueg_under_an_orbital_phase_gauge():
    """The electron-gas vertex with its orbitals' phases changed
    (Gamma^G_pq -> conj(u_p) Gamma^G_pq u_q): V becomes complex, the
    physics stays.  The GPU's converged CCSD energies equal the recorded
    ones (1e-9 Eh), and its (T) of those amplitudes equals the oracle's
    restatement of the reference's expression (1e-12 relative), which for
    complex V moves away from the recorded (T) energy: the reference's
    Re sum conj(W Z)/D is not invariant under the gauge."""
    from oracle import ueg
    from tests import properties as PR
    gamma, eps, _ = ueg.generate(7, 26, 1.0)
    ref = ueg.UEG_RS1_NO7_NV26
    s = ref["settings"]
    g = np.asfortranarray(gamma.copy())
    PR.gauge_vertex(g, PR.phases(g.shape[1], 11))
    with api.CoupledCluster(7, 26, g.shape[0], maxIterations=s["maxIterations"],
                            energyConvergence=s["energyConvergence"],
                            amplitudesConvergence=s["amplitudesConvergence"],
                            maxResidua=s["maxResidua"],
                            integralsSliceSize=s["integralsSliceSize"]) as cc:
        cc.set_inputs(g, eps)
        out = cc.run()
        e_t = cc.triples()
        T = cc.amplitudes()
    assert out["convergenceReached"]
    for key in ("correlation", "direct", "exchange", "secondOrder"):
        assert abs(out["energy"][key] - ref["Ccsd"][key]) < 1e-9, key
    e_oracle = O.perturbative_triples(g, eps, 7, "complex", T)
    print(f"gauged UEG (T): GPU {e_t:.15f} oracle {e_oracle:.15f} "
          f"recorded (real V) {ref['Triples']['correlation']:.15f}", flush=True)
    assert abs(e_t - e_oracle) <= 1e-12 * abs(e_oracle)
    assert abs(e_t - ref["Triples"]["correlation"]) > 1e-3
