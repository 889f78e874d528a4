"""Groups whose update products fill more than a round of 256 tiles keep X alone, not its transpose: the same bits."""
import pytest
import torch

from matrix_fsdp_amd import _lib
from matrix_fsdp_amd.optim import functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SHAPES = [(1090, 1500), (1500, 1090), (1037, 1283), (1283, 1037), (1025, 1409), (1111, 1111)] * 4  # 30 tiles of 256 or so each
# one slab of K, rows shorter than a tile, remainders of tiles and of slabs
SMALL = [(1, 7), (65, 63), (300, 257), (64, 1153), (1153, 128), (1100, 2040)]
KW = dict(lr=1.0, weight_decay=0.0, momentum=0.0, nesterov=False)


@pytest.fixture
def tuned():
    yield _lib.lib().mfsdp_set_muon_tuning
    _lib.lib().mfsdp_set_muon_tuning(3, 3, 0, 1, 16)


def transposes(shapes):
    """Bytes of all the matrices in the workspace, and of those the two X^T of each."""
    lib, total, xt = _lib.lib(), 0, 0
    shared = lib.mfsdp_muon_workspace_bytes(1, 1) - 6 * 256 * 256 * 2
    for r, c in shapes:
        bytes_ = lib.mfsdp_muon_workspace_bytes(r, c) - shared
        side = -(-min(r, c) // 256) * 256
        total += bytes_
        xt += (bytes_ - 2 * side * side * 2) // 2  # what A and B leave is X and X^T, two of each
    return total, xt


def step_together(shapes, dtype):
    """Ragged, wide, tall and square matrices of one group in a workspace of NaN: gradients, parameters, how many bytes of the
    matrices nothing was stored to."""
    gen = torch.Generator(device=DEV).manual_seed(1)
    grads = [torch.randn(s, generator=gen, device=DEV).bfloat16().to(dtype) for s in shapes]
    params = [torch.zeros(s, device=DEV, dtype=dtype) for s in shapes]
    total, _ = transposes(shapes)
    workspace = F.MuonWorkspace(torch.device(DEV))
    storage = workspace.get_bytes(_lib.lib().mfsdp_muon_workspace_bytes(1, 1) + total)
    storage.fill_(0xFF)
    F.muon_step_many([(p, g, torch.zeros_like(p), KW) for p, g in zip(params, grads)], workspace=workspace)
    return grads, params, 2 * int((storage[:total].view(torch.int16) == -1).sum())  # this NaN comes of no finite input


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("variant,split", [(1, 2), (1, 1), (3, 1)])
def test_groups_without_stored_transposes(variant, split, dtype, tuned):
    """Alone each matrix fills less than a round and keeps its transpose.  On 256 tiles with whole K walks both ways sum in the
    same order: the same bits.  With walks cut, or the library's own choice of tiles, the sums are in another order: 0.003 to
    0.005 apart after five iterations in bf16, up to 0.01 of the few elements of the small ones."""
    tuned(variant, variant, 0, split, 16)
    shapes = SHAPES + SMALL
    grads, together, untouched = step_together(shapes, dtype)
    assert untouched >= transposes(shapes)[1], "X^T was stored"
    for p, g in zip(together, grads):
        alone = torch.zeros_like(p)
        F.muon_step(alone, g, torch.zeros_like(p), **KW)
        if (variant, split) == (1, 2):
            assert torch.equal(p, alone), p.shape
        else:
            assert float((p - alone).float().norm() / alone.float().norm()) < 1e-2, p.shape


def test_smaller_tiles_store_transposes(tuned):
    """What the test above takes for stored transposes is there when they are."""
    tuned(2, 2, 0, 1, 16)
    shapes = SHAPES + SMALL
    assert step_together(shapes, torch.float32)[2] < transposes(shapes)[1]


@pytest.mark.parametrize("steps", [1, 2, 5])
@pytest.mark.parametrize("shape", [(2200, 9100), (9100, 2200)])
def test_newton_schulz_without_stored_transposes(shape, steps, tuned):
    """One matrix of 324 tiles, wide and tall: the last product leaves the orientation of the update.  On 256 tiles with whole K
    walks the same bits as from a matrix short enough to keep its transpose, for the rows and columns that reach it: with zeros
    behind them the norm and the Gram matrix of the short one are the same."""
    tuned(1, 1, 0, 2, 16)
    gen = torch.Generator(device=DEV).manual_seed(3)
    short = torch.randn(2200, 8000, generator=gen, device=DEV).bfloat16()  # 288 tiles
    long = torch.zeros(2200, 9100, device=DEV, dtype=torch.bfloat16)
    long[:, :8000] = short
    tall = shape[0] > shape[1]
    want = F.newton_schulz(short.T.contiguous() if tall else short, ns_steps=steps)
    have = F.newton_schulz(long.T.contiguous() if tall else long, ns_steps=steps)
    want, have = (want.T, have.T) if tall else (want, have)
    assert torch.equal(have[:, :8000], want) and not have[:, 8000:].any()


@pytest.mark.parametrize("shapes,stored", [
    ([(2500, 2500)] * 3, True), ([(2048, 5000)] * 2, False),  # 300 tiles and 320
    ([(5632, 5700)], False), ([(5700, 5633)], True), ([(8192, 8192)], True),
    ([(3072, 3072)] * 4, False), ([(3200, 3600)] * 4, True), ([(3328, 3328)] * 5, True),
    ([(1700, 1700)] * 20, False), ([(1800, 1800)] * 20, True),
    ([(2560, 5120)] * 6, False), ([(2304, 2880)] * 12, True), ([(2816, 5632)] * 5, True),
    ([(1536, 4096)] * 16, False), ([(1536, 4096)] * 17, True),  # 192 MiB of X
])
def test_where_the_transpose_is_stored(shapes, stored):
    """Both sides of every line of the choice."""
    assert (step_together(shapes, torch.bfloat16)[2] < transposes(shapes)[1]) == stored


@pytest.mark.parametrize("shape", [(1, 1 << 22), ((1 << 22) - 3, 24)])
def test_longest_matrices_keep_their_transpose(shape, tuned):
    """On 256 tiles: X padded to whole tiles is 2 GiB, more than a product takes by columns.  The roundings are torch's and the
    sums in another order, see above."""
    tuned(1, 1, 0, 1, 16)
    gen = torch.Generator(device=DEV).manual_seed(2)
    grad = torch.randn(shape, generator=gen, device=DEV).bfloat16()
    param = torch.zeros_like(grad)
    F.muon_step(param, grad, torch.zeros_like(grad), **KW)
    a, b, c = F.NS_COEFFICIENTS
    x = grad.T if shape[0] > shape[1] else grad
    x = (x / x.float().norm().bfloat16()).contiguous()
    for _ in range(5):
        gram = x @ x.T
        x = torch.addmm(x, torch.addmm(gram, gram, gram, beta=b, alpha=c), x, beta=a)
    want = (x.T if shape[0] > shape[1] else x).float()
    have = param.float() / -F.adjust_lr(1.0, None, shape)
    assert float((have - want).norm() / want.norm()) < 1e-2
