"""The matrix-core exchange products over the tiled factor (coulomb_exchange_rhf,
src/df.rs:133-174) at the sizes where their tiles end: molecules whose n lies
below, at and above multiples of the 32-wide factor tiles and the 64-row
output tiles, with one, two and three column tiles (of at most 160) to the
first row of them, and column counts around the 16-column blocks and the 160
columns of one workgroup.

Two references.  The oracle's B gives J and K to 1e-9 per element (the
reference's own DF bound).  And K is a sum over the columns of C, so K of all
columns equals the sum of K over a split of them, which runs other kernel
variants: FP64 sums of rank * o <= 1e5 products differ by at most
sqrt(1e5) * 1.1e-16 ~ 4e-14 of the summed magnitudes, stated 1e-12; FP32 and
split BF16 are compared with FP64 within FP32's and the split's own rounding
(2^-24 and 2^-16 per product and operand: 1e-5 and 1e-4 of the largest element)."""
import numpy as np
import pytest

import molecules as M
import oracle as O
from conftest import load_package

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hf():
    mod = load_package()
    if mod.device_count() < 1:
        pytest.fail("no GPU visible to the HIP engine")
    return mod


# n: 7, 25, 33 (33 = 32 + 1), 114 and 133 (around 128)
MOLECULES = {"water_sto3g": (M.water_config1, "sto-3g"), "water_ccpvdz": (M.water_config1, "cc-pvdz"),
             "methane_def2svp": (lambda: M.alkane(1), "def2-svp"),
             "water6_631gs": (lambda: M.water_cluster_m(6, 1), "6-31g*"),
             "water7_631gs": (lambda: M.water_cluster_m(7, 1), "6-31g*")}
AUX = "def2-svp-rifit"


# n: 175 and 325, two and three column tiles
LARGE = {"water7_ccpvdz": (lambda: M.water_cluster_m(7, 1), "cc-pvdz"),
         "water13_ccpvdz": (lambda: M.water_cluster_m(13, 1), "cc-pvdz")}


def factors(hf, make, basis):
    mol = make()
    b = hf.Basis.from_g94(M.basis_text(basis), mol.symbols, mol.xyz)
    a = hf.Basis.from_g94(M.basis_text(AUX), mol.symbols, mol.xyz)
    return hf.DfTensor(b, a), O.df_build(O.Basis.build(M.basis_text(basis), mol.symbols, mol.xyz),
                                         O.Basis.build(M.basis_text(AUX), mol.symbols, mol.xyz))


@pytest.fixture(scope="module", params=sorted(MOLECULES))
def system(hf, request):
    df, bt = factors(hf, *MOLECULES[request.param])
    yield df, bt
    df.close()


@pytest.fixture(scope="module", params=sorted(LARGE))
def large_system(hf, request):
    df, bt = factors(hf, *LARGE[request.param])
    assert (df.n + 15) // 16 > 10
    yield df, bt
    df.close()


@pytest.mark.parametrize("o", [1, 5, 16, 17, 48, 100, 160, 161, 330])
def test_exchange_over_tiles(system, o):
    check_exchange(*system, o)


@pytest.mark.parametrize("o", [17, 160, 161])
def test_exchange_over_several_column_tiles(large_system, o):
    check_exchange(*large_system, o)


def check_exchange(df, bt, o):
    c = np.random.default_rng(100 + o).standard_normal((df.n, o)) / np.sqrt(df.n)
    j, k, _ = df.jk_precision(c, "fp64")
    jr, kr = O.df_jk(bt, df.n, c)
    scale = max(1.0, np.abs(kr).max())
    assert np.abs(j - jr).max() < 1e-9 * max(1.0, np.abs(jr).max())
    assert np.abs(k - kr).max() < 1e-9 * scale
    assert np.array_equal(k, k.T)
    if o > 1:
        cut = (o + 2) // 3
        parts = [df.jk_precision(x, "fp64")[:2] for x in (c[:, :cut], c[:, cut:])]
        assert np.abs(k - parts[0][1] - parts[1][1]).max() < 1e-12 * scale
        assert np.abs(j - parts[0][0] - parts[1][0]).max() < 1e-12 * max(1.0, np.abs(j).max())
    for precision, bound in (("fp32", 1e-5), ("bf16x3", 1e-4)):
        jp, kp, _ = df.jk_precision(c, precision)
        assert np.abs(jp - j).max() < 1e-12 * max(1.0, np.abs(j).max())
        assert np.abs(kp - k).max() < bound * scale
        assert np.array_equal(kp, kp.T)
