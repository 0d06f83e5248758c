"""The training GEMMs and loss kernels at the edges of their tiles: hidden sizes that are no multiple of 4, 16 or 32 (no
16-byte loads, partial K steps and tiles), a single sample, samples past one round of 32 x 32 tiles.  Bounds: those of
the bf16-emulating oracle for the ordinary sizes (2e-3 of the gradient, 5e-3 of each tensor: flips of a bf16 rounding)."""
import numpy as np
import pytest

import mlp_oracle as MO

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,Np,kind,rank,hidden,B", [(64, 16, 1, 8, 17, 1), (36, 9, 1, 4, 100, 33), (64, 16, 0, 8, 31, 64),
                                                      (64, 16, 1, 4, 256, 300), (36, 9, 0, 8, 40, 7)])
def test_loss_gradient_at_odd_sizes(nb, Np, kind, rank, hidden, B):
    from dpgsolver_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(hidden + B)
    m = _lib.MLP(nb, Np, hidden=hidden, rank=rank, seed=7, kind=kind)
    w = (m.get_params() + 0.05 * rng.standard_normal(m.nparam)).astype(np.float32)
    m.set_params(w)
    X = rng.standard_normal((B, m.nf)).astype(np.float32)
    A = -(rng.standard_normal((B, nb, nb)) * 0.3 + 2.0 * np.eye(nb))
    sigma = rng.uniform(0.3, 0.7, B).astype(np.float32)
    Xd, Ad, sd = (torch.from_numpy(a).to(dev) for a in (X, A, sigma))
    loss, g = m.loss_grad(Xd.data_ptr(), sd.data_ptr(), Ad.data_ptr(), B)
    Lref, gref = MO.loss_and_grad(w, X, sigma, A, nb, rank, hidden, emulate_bf16=True, kind=kind, Np=Np)
    assert abs(loss - Lref) <= 1e-4 * Lref
    assert np.linalg.norm(g - gref) < 2e-3 * np.linalg.norm(gref)
    offs, _, n = MO.layout(m.nf, hidden, m.nout)
    for a, b in zip(offs, offs[1:] + [n]):
        assert np.linalg.norm(g[a:b] - gref[a:b]) <= 5e-3 * np.linalg.norm(gref[a:b]) + 1e-12
    m.close()


def test_inference_takes_no_training_planes():
    """dgx_mlp_predict over many samples holds three activations, their gradients and the losses, not the split planes of
    the backward pass (4 B hidden floats more); training after it still finds them."""
    from dpgsolver_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    B, hidden = 100000, 512
    m = _lib.MLP(36, 9, hidden=hidden, rank=4, seed=7, kind=1)
    X = torch.zeros((B, m.nf), dtype=torch.float32, device="cuda:0")
    out = torch.empty((B, m.nout), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    m.predict(X.data_ptr(), B, out.data_ptr())
    torch.cuda.synchronize()
    took = free0 - torch.cuda.mem_get_info()[0]
    need = 4 * B * (4 * hidden + 2 * m.nout) + 8 * B
    assert took <= need + 64 * 2 ** 20, (took, need)      # (the planes alone: 819 MB)
    A = torch.eye(36, dtype=torch.float64, device="cuda:0").repeat(40, 1, 1)
    assert np.isfinite(m.train(X.data_ptr(), None, A.data_ptr(), 40, epochs=1, batch=16, lr=1e-4))
    m.close()
