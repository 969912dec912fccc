"""Gradients of a basis with d shells from several live contexts: their
(fd|dd) blocks ask for the largest private segments of the library, which the
runtime keeps per hardware queue, and each context has streams of its own.
Every context's gradient equals the first one's of the same molecule (the
sums differ by the order of atomic additions only: 1e-12 of the largest
component), and forces sum to zero as translational invariance has it
(tests/test_gpu_gradient.py holds the values against PySCF)."""
import numpy as np
import pytest

import molecules as M
from conftest import load_package

pytestmark = pytest.mark.gpu


def test_gradients_of_many_live_contexts():
    hf = load_package()
    if hf.device_count() < 1:
        pytest.fail("no GPU visible to the HIP engine")
    mol = M.alkane(1)
    b = hf.Basis.from_g94(M.basis_text("def2-svp"), mol.symbols, mol.xyz)
    c = np.linalg.qr(np.random.default_rng(4).standard_normal((b.n, 5)))[0]
    p = 2.0 * c @ c.T
    w = 2.0 * (c * -np.arange(1.0, 6.0)) @ c.T
    contexts = [hf.Context(b) for _ in range(6)]
    g = [ctx.rhf_gradient(mol.zxyz, p, w) for ctx in contexts]
    scale = np.abs(g[0]).max()
    for x in g:
        assert np.abs(x - g[0]).max() < 1e-12 * scale
        assert np.abs(x.sum(0)).max() < 1e-10 * scale
    for ctx in contexts:
        ctx.close()
