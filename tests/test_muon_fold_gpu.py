"""Newton-Schulz iterations folded into one (short sides of 2048 and more, long enough): against 64-bit arithmetic.

Every bound is the error of the single iterations on the same input: each product in bf16 with fp32 accumulation, in the
order of torch/optim/_muon.py:50-68, by torch's own products."""
import pytest
import torch

from matrix_fsdp_amd.optim import functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
A, B, C = F.NS_COEFFICIENTS


def single_iterations(x, steps, dtype):
    x = x.to(dtype)
    for _ in range(steps):
        gram = x @ x.T
        x = torch.addmm(x, torch.addmm(gram, gram, gram, beta=B, alpha=C), x, beta=A)
    return x.double()


def spectrum(kind, m, n, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    normal = lambda *shape: torch.randn(shape, generator=gen, device=DEV)
    if kind == "normal":
        g = normal(m, n)
    elif kind == "spike":
        g = normal(m, n) + 0.3
    elif kind == "low rank":
        g = normal(m, m // 16) @ normal(m // 16, n) * (m // 16) ** -0.5 + 0.05 * normal(m, n)
    elif kind == "graded rows":
        g = normal(m, n) * torch.logspace(0, -2, m, device=DEV)[:, None]
    else:
        g = normal(m, n) * torch.logspace(0, -3, n, device=DEV)
    return g.bfloat16()


def errors(update, have, steps):
    """Relative errors of ``have`` and of the single iterations."""
    tall = update.shape[0] > update.shape[1]
    x = (update.T if tall else update) / update.float().norm().bfloat16().clamp(min=1e-7)
    want = single_iterations(x, steps, torch.float64)
    have = (have.T if tall else have).double()
    return float((have - want).norm() / want.norm()), float((single_iterations(x, steps, torch.bfloat16) - want).norm() / want.norm())


@pytest.fixture
def tuned():
    from matrix_fsdp_amd import _lib

    yield _lib.lib().mfsdp_set_muon_tuning
    _lib.lib().mfsdp_set_muon_tuning(3, 3, 0, 1, 16)


@pytest.mark.parametrize("kind", ["normal", "spike", "low rank", "graded rows", "graded columns"])
@pytest.mark.parametrize("shape,steps", [((2048, 4096), 5), ((5001, 2111), 5), ((2100, 8190), 6), ((4096, 5000), 8)])
def test_folded_iterations_are_no_less_precise(kind, shape, steps):
    update = spectrum(kind, *sorted(shape), 5)
    update = update.T.contiguous() if shape[0] > shape[1] else update
    mine, theirs = errors(update, F.newton_schulz(update, ns_steps=steps), steps)
    assert mine <= theirs, (mine, theirs)


@pytest.mark.parametrize("variant", [1, 2, 4])
@pytest.mark.parametrize("split", [1, 2])
def test_folded_iterations_on_every_tile(variant, split, tuned):
    """Each tile variant, whole and cut K walks, a ragged matrix in a workspace full of NaN."""
    tuned(variant, variant, 0, split, 16)
    update = spectrum("normal", 2090, 4330, 6)
    workspace = F.MuonWorkspace(torch.device(DEV))
    workspace.get(*update.shape).fill_(0xFF)
    mine, theirs = errors(update, F.newton_schulz(update, workspace=workspace), 5)
    assert mine <= theirs, (mine, theirs)


def test_folded_and_single_iterations_in_one_group():
    """Folded matrices between square and small ones, more of them than one launch has room for the two products of a stage:
    every parameter gets the update that its matrix gets from ``newton_schulz``, to the bound above."""
    shapes = [(2048, 2500)] * 9 + [(2111, 2111), (300, 520)] + [(2560, 2065)] * 9
    kw = dict(lr=0.5, weight_decay=0.0, momentum=0.0, nesterov=False)
    updates = [spectrum("normal", r, c, 20 + i) for i, (r, c) in enumerate(shapes)]
    params = [torch.zeros(s, device=DEV) for s in shapes]
    F.muon_step_many([(p, u.float(), torch.zeros_like(p), kw) for p, u in zip(params, updates)])
    for p, u in zip(params, updates):
        mine, theirs = errors(u, p / -F.adjust_lr(0.5, None, p.shape), 5)
        # the single iterations of the square and the small one differ from torch's in the order of their sums only
        assert mine <= theirs * (1.0 if min(u.shape) >= 2048 and u.shape[0] != u.shape[1] else 1.05), (u.shape, mine, theirs)


def test_what_stays_single():
    """Other coefficients and fewer iterations run one by one, as on bf16 parameters: their error is torch's, not less."""
    update = spectrum("normal", 2048, 6144, 7)
    mine, theirs = errors(update, F.newton_schulz(update, ns_steps=4), 4)
    assert abs(mine / theirs - 1) < 0.02, (mine, theirs)
    x = update / update.float().norm().bfloat16()
    for _ in range(5):
        gram = x @ x.T
        x = torch.addmm(x, torch.addmm(gram, gram, gram, beta=-4.0, alpha=2.0), x, beta=3.0)
    have = F.newton_schulz(update, ns_coefficients=(3.0, -4.0, 2.0))
    # the same roundings, sums in another order: 0.003 to 0.004 at this size with any coefficients; folded, 0.0085
    assert float((have.float() - x.float()).norm() / x.float().norm()) < 6e-3
    param, grad = torch.zeros(2048, 6144, device=DEV, dtype=torch.bfloat16), update.clone()
    F.muon_step(param, grad, torch.zeros_like(grad), lr=1.0, weight_decay=0.0, momentum=0.0, nesterov=False)
    mine, theirs = errors(update, param / -F.adjust_lr(1.0, None, param.shape), 5)
    assert abs(mine / theirs - 1) < 0.02, (mine, theirs)
