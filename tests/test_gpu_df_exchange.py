"""The matrix-core exchange products over the tiled factor (coulomb_exchange_rhf,
src/df.rs:133-174) at the sizes where their tiles end: molecules whose n lies
below, at and above multiples of the 32-wide factor tiles and the 128-row
output tiles, and column counts around the 16-column blocks and the 160
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


@pytest.fixture(scope="module", params=sorted(MOLECULES))
def system(hf, request):
    make, basis = MOLECULES[request.param]
    mol = make()
    b = hf.Basis.from_g94(M.basis_text(basis), mol.symbols, mol.xyz)
    a = hf.Basis.from_g94(M.basis_text(AUX), mol.symbols, mol.xyz)
    df = hf.DfTensor(b, a)
    bt = O.df_build(O.Basis.build(M.basis_text(basis), mol.symbols, mol.xyz),
                    O.Basis.build(M.basis_text(AUX), mol.symbols, mol.xyz))
    yield df, bt
    df.close()


@pytest.mark.parametrize("o", [1, 5, 16, 17, 48, 100, 160, 161, 330])
def test_exchange_over_tiles(system, o):
    df, bt = system
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
