"""Newton-Schulz iterations of the sizes that training has, against 64-bit arithmetic.

Every bound comes from the error of torch's iterations on the same input: each product in bf16 with fp32 accumulation, in the
order of torch/optim/_muon.py:50-68, by torch's own products.  The kernels round where those round and sum in another order, so
the errors differ by chance only: with the rows and columns of the update in another order torch's own move by up to 1.5 % (all
elements together) and 21 % (the row that is furthest off)."""
import pytest
import torch

from matrix_fsdp_amd.optim import functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
A, B, C = F.NS_COEFFICIENTS
ALL, ROW = 1.03, 1.5  # largest error, in torch's


def torch_iterations(x, steps, dtype, coefficients=(A, B, C)):
    a, b, c = coefficients
    x = x.to(dtype)
    for _ in range(steps):
        gram = x @ x.T
        x = torch.addmm(x, torch.addmm(gram, gram, gram, beta=b, alpha=c), x, beta=a)
    return x.double()


def spectrum(kind, m, n, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    normal = lambda *shape: torch.randn(shape, generator=gen, device=DEV)
    if kind == "normal":
        g = normal(m, n)
    elif kind == "spike":
        g = normal(m, n) + 0.3
    elif kind == "offset":
        g = normal(m, n) + 3.0
    elif kind.startswith("direction"):  # one direction, so many times as long as a row or a column of the rest
        g = float(kind.split()[1]) * normal(m, 1) @ normal(1, n) + normal(m, n)
    elif kind == "low rank":
        g = normal(m, m // 16) @ normal(m // 16, n) * (m // 16) ** -0.5 + 0.05 * normal(m, n)
    elif kind == "cross entropy":  # of 512 tokens, with regard to the weight of the classifier
        tokens, classes = normal(512, n), torch.randint(0, m, (512,), generator=gen, device=DEV)
        g = (torch.softmax(2.0 * normal(512, m), 1) - torch.nn.functional.one_hot(classes, m)).T @ tokens
    elif kind == "graded rows":
        g = normal(m, n) * torch.logspace(0, -2, m, device=DEV)[:, None]
    else:
        g = normal(m, n) * torch.logspace(0, -3, n, device=DEV)
    return g.bfloat16()


KINDS = ["normal", "spike", "offset", "direction 3", "direction 10", "direction 30", "low rank", "cross entropy", "graded rows", "graded columns"]


def errors(update, have, steps):
    """Of ``have`` and of torch's iterations, relative: of all elements together, and of the row that is furthest off."""
    tall = update.shape[0] > update.shape[1]
    x = (update.T if tall else update) / update.float().norm().bfloat16().clamp(min=1e-7)
    want = torch_iterations(x, steps, torch.float64)
    result = []
    for got in ((have.T if tall else have).double(), torch_iterations(x, steps, torch.bfloat16)):
        rows = (got - want).norm(dim=1) / want.norm(dim=1)
        result.append((float((got - want).norm() / want.norm()), float(rows.max())))
    return result


def check(update, have, steps, what=None):
    mine, theirs = errors(update, have, steps)
    print(what, tuple(update.shape), "mine", mine, "torch", theirs, flush=True)
    assert mine[0] <= ALL * theirs[0] and mine[1] <= ROW * theirs[1], (what, tuple(update.shape), mine, theirs)


@pytest.fixture
def tuned():
    from matrix_fsdp_amd import _lib

    yield _lib.lib().mfsdp_set_muon_tuning
    _lib.lib().mfsdp_set_muon_tuning(3, 3, 0, 1, 16)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape,steps", [((2048, 6144), 5), ((5001, 2111), 5), ((2100, 8190), 6), ((4096, 8192), 8), ((8200, 4100), 5), ((768, 2304), 5)])
def test_precision_is_that_of_torch(kind, shape, steps):
    update = spectrum(kind, *sorted(shape), 5)
    update = update.T.contiguous() if shape[0] > shape[1] else update
    check(update, F.newton_schulz(update, ns_steps=steps), steps, kind)


@pytest.mark.parametrize("kind", KINDS)
def test_a_step_is_as_precise_as_its_iterations(kind):
    """The same bits from ``newton_schulz`` and from ``muon_step``, whatever the dtype of the parameter."""
    update = spectrum(kind, 2048, 6144, 6)
    want = F.newton_schulz(update)
    scale = -F.adjust_lr(1.0, None, update.shape)
    for dtype in (torch.float32, torch.bfloat16):
        param = torch.zeros(update.shape, device=DEV, dtype=dtype)
        F.muon_step(param, update.to(dtype), torch.zeros_like(param), lr=1.0, weight_decay=0.0, momentum=0.0, nesterov=False)
        assert torch.equal(param, (want.float() * scale).to(dtype)), dtype


@pytest.mark.parametrize("variant", [1, 2, 4])
@pytest.mark.parametrize("split", [1, 2])
def test_precision_on_every_tile(variant, split, tuned):
    """Each tile variant, whole and cut K walks, a ragged matrix in a workspace full of NaN."""
    tuned(variant, variant, 0, split, 16)
    update = spectrum("direction 10", 2090, 4330, 6)
    workspace = F.MuonWorkspace(torch.device(DEV))
    workspace.get(*update.shape).fill_(0xFF)
    check(update, F.newton_schulz(update, workspace=workspace), 5)


@pytest.mark.parametrize("kind", ["normal", "direction 10", "cross entropy"])
def test_precision_does_not_depend_on_the_other_matrices(kind):
    """Long matrices between square and small ones, in more than one group."""
    shapes = [(2048, 3072)] * 9 + [(2111, 2111), (300, 520)] + [(2560, 2065)] * 9
    kw = dict(lr=0.5, weight_decay=0.0, momentum=0.0, nesterov=False)
    updates = [spectrum(kind, r, c, 20 + i) for i, (r, c) in enumerate(shapes)]
    params = [torch.zeros(s, device=DEV) for s in shapes]
    F.muon_step_many([(p, u.float(), torch.zeros_like(p), kw) for p, u in zip(params, updates)])
    for p, u in zip(params, updates):
        check(u, p / -F.adjust_lr(0.5, None, p.shape), 5, kind)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [(2048, 6144), (2111, 5001), (300, 520)])
def test_distance_from_torch_and_from_a_call_alone(kind, shape):
    """Five iterations: 0.0007 to 0.0065 of the update from torch's, 0.0005 to 0.006 between a call with other matrices and one
    without, on every spectrum.  The bound is the path's tolerance."""
    update = spectrum(kind, *shape, 5)
    others = [spectrum("normal", *shape, 9 + i) for i in range(3)] + [spectrum("normal", 700, 1800, 3)]
    kw = dict(lr=1.0, weight_decay=0.0, momentum=0.0, nesterov=False)
    params = [torch.zeros(u.shape, device=DEV) for u in [update] + others]
    F.muon_step_many([(p, u.float(), torch.zeros_like(p), kw) for p, u in zip(params, [update] + others)])
    alone = F.newton_schulz(update).double()
    theirs = torch_iterations(update / update.float().norm().bfloat16().clamp(min=1e-7), 5, torch.bfloat16)
    together = params[0].double() / -F.adjust_lr(1.0, None, shape)
    for have, want in ((alone, theirs), (together, theirs), (together, alone)):
        assert float((have - want).norm() / want.norm()) < 1e-2


def test_other_coefficients():
    update = spectrum("normal", 2048, 6144, 7)
    check(update, F.newton_schulz(update, ns_steps=4), 4)
    x = update / update.float().norm().bfloat16()
    want = torch_iterations(x, 5, torch.bfloat16, (3.0, -4.0, 2.0))
    have = F.newton_schulz(update, ns_coefficients=(3.0, -4.0, 2.0)).double()
    # the same roundings, sums in another order: 0.003 to 0.004 at this size with any coefficients
    assert float((have - want).norm() / want.norm()) < 6e-3
