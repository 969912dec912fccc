"""Density fitting with orbital f shells (cc-pVTZ), and the factor formed over
several chunks of tile rows (src/df.rs:60-127; the 3-index tensor exists one
chunk at a time, and a shell pair whose functions lie in two chunks is
evaluated for both), against the oracle: DF J/K to 1e-9 per element (the
reference's own DF element bound, tests/df_hf_test.rs; the metric's smallest
kept eigenvalues amplify last-digit differences to ~1e-10, between chunk sizes
as between programs), DF-RHF energies within 1e-8 Eh with the iteration count
within 1, also with split-BF16 exchange before the final FP64 builds.
HFG_DF_CHUNK=1 (bytes) makes every 32-function tile row a chunk of its own;
without it these molecules have one chunk."""
import numpy as np
import pytest

import oracle as O
import molecules as M
from conftest import load_package

pytestmark = pytest.mark.gpu

JKFIT = "def2-universal-jkfit"


@pytest.fixture(scope="module")
def hf():
    mod = load_package()
    if mod.device_count() < 1:
        pytest.fail("no GPU visible to the HIP engine")
    return mod


@pytest.fixture(params=["one chunk", "a chunk a tile row"])
def chunks(request, monkeypatch):
    if request.param == "one chunk":
        monkeypatch.delenv("HFG_DF_CHUNK", raising=False)
    else:
        monkeypatch.setenv("HFG_DF_CHUNK", "1")
    return request.param


def bases(hf, mol, name):
    return (hf.Basis.from_g94(M.basis_text(name), mol.symbols, mol.xyz),
            hf.Basis.from_g94(M.basis_text(JKFIT), mol.symbols, mol.xyz))


def oracle_bases(mol, name):
    return (O.Basis.build(M.basis_text(name), mol.symbols, mol.xyz),
            O.Basis.build(M.basis_text(JKFIT), mol.symbols, mol.xyz))


# water dimer / cc-pVTZ: n 130, f shells, five tile rows; (H2O)4 / cc-pVDZ: n 100, four
@pytest.fixture(scope="module", params=["dimer cc-pvtz", "tetramer cc-pvdz"])
def system(request):
    mol, basis = {"dimer cc-pvtz": (M.water_cluster((2, 1, 1), seed=2), "cc-pvtz"),
                  "tetramer cc-pvdz": (M.water_cluster((2, 2, 1), seed=2), "cc-pvdz")}[request.param]
    ob, oa = oracle_bases(mol, basis)
    first = ob.shells()  # first function of every shell, and n
    # shells whose functions lie in two tile rows
    assert any(a // 32 != (b - 1) // 32 for a, b in zip(first[:-1], first[1:])), "no shell straddles"
    return mol, basis, O.df_build(ob, oa)


def test_df_jk_matches_oracle_over_chunks(hf, system, chunks):
    mol, basis, bt = system
    df = hf.DfTensor(*bases(hf, mol, basis))
    assert df.rank == bt.shape[0]
    c = np.random.default_rng(6).standard_normal((df.n, 10)) * 0.2
    j, k = df.coulomb_exchange_rhf(c)
    jr, kr = O.df_jk(bt, df.n, c)
    print("%s, %s: n=%d rank=%d  J %.2e K %.2e" % (basis, chunks, df.n, df.rank, np.abs(j - jr).max(),
                                                  np.abs(k - kr).max()))
    assert np.abs(j - jr).max() < 1e-9 and np.abs(k - kr).max() < 1e-9
    scale = np.abs(k).max()
    for prec, bound in (("fp32", 1e-5), ("bf16x3", 1e-3)):
        jp, kp, _ = df.jk_precision(c, prec)
        assert np.abs(jp - j).max() < 1e-12 * max(1, np.abs(j).max())
        assert np.abs(kp - k).max() < bound * scale
    df.close()


def test_df_rhf_cc_pvtz_water_matches_oracle(hf, chunks):
    mol = M.water_config1()
    r = hf.df_rhf(*bases(hf, mol, "cc-pvtz"), mol.zxyz)
    o, _, _, _, _ = O.df_rhf(*oracle_bases(mol, "cc-pvtz"), mol.zxyz)
    print("DF-RHF water cc-pVTZ, %s: E %.12f vs %.12f, iters %d vs %d" % (
        chunks, r["total_energy"], o.total_energy, r["iterations"], o.iterations))
    assert r["converged"] and o.converged
    assert abs(r["total_energy"] - o.total_energy) < 1e-8
    assert abs(r["iterations"] - o.iterations) <= 1


def test_df_rhf_split_bf16_reaches_the_fp64_energy_with_f_shells(hf):
    """Split-BF16 exchange in the early iterations, FP64 builds at the end:
    the water-dimer cc-pVTZ energy equals the oracle's FP64 DF-RHF energy to
    1e-8 Eh (no reference counterpart; the reference is FP64 throughout)."""
    mol = M.water_cluster((2, 1, 1), seed=2)
    r = hf.df_rhf(*bases(hf, mol, "cc-pvtz"), mol.zxyz, k_precision="bf16x3")
    o, _, _, _, _ = O.df_rhf(*oracle_bases(mol, "cc-pvtz"), mol.zxyz)
    print("DF-RHF dimer cc-pVTZ bf16x3: E %.12f vs %.12f, iters %d vs %d" % (
        r["total_energy"], o.total_energy, r["iterations"], o.iterations))
    assert r["converged"] and o.converged
    assert abs(r["total_energy"] - o.total_energy) < 1e-8
    assert r["iterations"] <= o.iterations + 4
