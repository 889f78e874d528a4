"""Parity of the HIP Muon / AdamW kernels (through the C ABI) with the CPU oracle.

Tolerances: the Muon update must be within rel-Frobenius 1e-2 of the reference arithmetic on the
same seeded inputs (bf16 products, fp32 accumulation; only the summation order differs); AdamW is
fp32 element-wise and must agree to 1e-6 relative."""
import numpy as np
import pytest
import torch

from matrix_fsdp_amd.optim import functional as F
from oracle import optim_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
MUON_TOL = 1e-2


def rel_fro(have: torch.Tensor, want: torch.Tensor) -> float:
    have, want = have.detach().double().cpu(), want.detach().double().cpu()
    return float(torch.linalg.norm(have - want) / torch.linalg.norm(want))


def max_err_over_scale(have: torch.Tensor, want: torch.Tensor) -> float:
    """Largest element error relative to the tensor's largest magnitude (fp32 element-wise kernels
    differ from the CPU only by fused multiply-adds: a few 1e-7 of the operand scale)."""
    want = want.detach().double().cpu()
    return float((have.detach().double().cpu() - want).abs().max() / want.abs().max().clamp(min=1e-300))


def make(shape, seed, std=1e-3):
    gen = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=gen) * std


@pytest.mark.parametrize("shape", [(256, 256), (256, 512), (512, 256), (64, 96), (100, 36), (300, 520), (1, 7), (1024, 1024)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_newton_schulz_parity(shape, dtype):
    u = make(shape, 11).to(dtype)
    for steps in (0, 1, 5):
        want = O.newton_schulz(u, steps=steps)
        have = F.newton_schulz(u.to(DEV), ns_steps=steps)
        assert have.dtype == torch.bfloat16 and have.shape == want.shape
        assert rel_fro(have, want) < MUON_TOL, (shape, dtype, steps)


def test_newton_schulz_diagonal_closed_form():
    sigma = torch.tensor([0.9, 0.5, 0.25, 0.1, 0.01, 0.0])
    x = torch.diag(sigma)
    have = F.newton_schulz(x.to(DEV)).float().cpu()
    want = O.newton_schulz(x).float()
    assert torch.count_nonzero(have - torch.diag(torch.diag(have))) == 0
    assert torch.allclose(torch.diag(have), torch.diag(want), atol=0.02)


def test_newton_schulz_singular_values_land_near_one():
    u = make((384, 640), 12)
    sv = torch.linalg.svdvals(F.newton_schulz(u.to(DEV)).float().cpu())
    assert sv.max() < 1.3 and sv.min() > 0.3


@pytest.mark.parametrize("coefficients", [(1.5, -0.5, 0.0), (2.0, -1.5, 0.5), (0.0, 1.0, 1.0)])
def test_newton_schulz_other_polynomials(coefficients):
    """torch.optim.Muon takes any three coefficients; with c = 0 (the cubic iteration) addmm leaves b * A, with a = 0
    the update product has no X term."""
    for shape in ((256, 256), (300, 520), (512, 256)):
        u = make(shape, 17)
        want = O.newton_schulz(u, coefficients=coefficients, steps=3)
        have = F.newton_schulz(u.to(DEV), ns_coefficients=coefficients, ns_steps=3)
        assert rel_fro(have, want) < MUON_TOL, (shape, coefficients)
    p, g, buf = make((256, 384), 18, 0.02), make((256, 384), 19).bfloat16().float(), make((256, 384), 20)
    p_dev, buf_dev = p.to(DEV), buf.to(DEV)
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    F.muon_step(p_dev, g.to(DEV), buf_dev, ns_coefficients=coefficients, ns_steps=3, **kw)
    p_ref, buf_ref = p.clone(), buf.clone()
    O.muon_step(p_ref, g, buf_ref, coefficients=coefficients, steps=3, **kw)
    assert rel_fro(p_dev.cpu() - p, p_ref - p) < MUON_TOL


@pytest.mark.parametrize("shape", [(192, 320), (320, 192), (100, 36), (37, 101)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("steps", [0, 1])
def test_muon_step_with_no_or_one_newton_schulz_step(shape, dtype, steps):
    """Without a Newton-Schulz step there is no product whose epilogue could carry the parameter update (the separate
    update kernel runs on the normalised update); with one step the only update product is also the last one.  Wide,
    tall and unaligned shapes (tall parameters are updated from the transposed tile)."""
    p = make(shape, 31, 0.02).to(dtype)
    g, buf = make(shape, 32).to(dtype), make(shape, 33).to(dtype)
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    p_dev, buf_dev = p.to(DEV), buf.to(DEV)
    F.muon_step(p_dev, g.to(DEV), buf_dev, ns_steps=steps, **kw)
    p_ref, buf_ref = p.clone(), buf.clone()
    O.muon_step(p_ref, g, buf_ref, steps=steps, **kw)
    tol = MUON_TOL if dtype == torch.float32 else 0.05  # a bf16 parameter moves in steps of its own last bit
    assert rel_fro(p_dev.cpu().float() - p.float(), p_ref.float() - p.float()) < tol
    if dtype == torch.float32:
        assert torch.allclose(buf_dev.cpu(), buf_ref, rtol=1e-6, atol=1e-9)
    else:
        assert (buf_dev.cpu().view(torch.int16).int() - buf_ref.view(torch.int16).int()).abs().max() <= 1


def test_non_finite_coefficients_are_refused_before_anything_runs():
    p, g, buf = make((64, 64), 21, 0.02).to(DEV), make((64, 64), 22).to(DEV), make((64, 64), 23).to(DEV)
    before = (p.clone(), buf.clone())
    for bad in ((float("nan"), -4.775, 2.0315), (3.4445, float("inf"), 2.0315), (3.4445, -4.775, 1e-45)):
        with pytest.raises(RuntimeError, match="coefficients must be finite"):
            F.muon_step(p, g, buf, lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True, ns_coefficients=bad)
        with pytest.raises(RuntimeError, match="coefficients must be finite"):
            F.newton_schulz(g, ns_coefficients=bad)
    torch.cuda.synchronize()
    assert torch.equal(p, before[0]) and torch.equal(buf, before[1])  # the momentum buffer was not touched


def test_zero_update_stays_zero():
    have = F.newton_schulz(torch.zeros(64, 128, device=DEV))
    assert torch.count_nonzero(have) == 0


@pytest.mark.parametrize("shape", [(256, 512), (512, 256), (192, 192)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nesterov,adjust", [(True, None), (True, "match_rms_adamw"), (False, "original")])
def test_muon_step_parity(shape, dtype, nesterov, adjust):
    p0 = make(shape, 1, 0.02).to(dtype)
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=nesterov, adjust_lr_fn=adjust)
    p_cpu, buf_cpu = p0.clone(), make(shape, 2).to(dtype)
    p_dev, buf_dev = p_cpu.to(DEV), buf_cpu.to(DEV)
    ws = F.MuonWorkspace(DEV)
    for step in range(2):
        g = make(shape, 20 + step).to(dtype)
        before = p_cpu.clone()
        O.muon_step(p_cpu, g.clone(), buf_cpu, **kw)
        before_dev = p_dev.clone()
        F.muon_step(p_dev, g.to(DEV), buf_dev, workspace=ws, **kw)
        # the parameter delta, which the orthogonalised update dominates
        # bf16 parameters move by whole bf16 steps (2^-8 relative), so their delta and value carry that grain
        delta_err = rel_fro(p_dev.float().cpu() - before_dev.float().cpu(), p_cpu.float() - before.float())
        buf_ok = bool(torch.allclose(buf_dev.cpu(), buf_cpu, rtol=1e-6, atol=1e-9)) if dtype == torch.float32 else rel_fro(buf_dev.float(), buf_cpu.float()) < 4e-3
        value_err = rel_fro(p_dev.float(), p_cpu.float())
        assert delta_err < (MUON_TOL if dtype == torch.float32 else 0.05), delta_err
        assert buf_ok
        assert value_err < MUON_TOL, value_err
        p_cpu, buf_cpu = p_dev.cpu().clone(), buf_dev.cpu().clone()  # re-sync so that steps are compared one at a time


def test_muon_step_matches_torch_optim_muon_on_device_inputs():
    """Same check against the optimizer class the reference instantiates (CPU execution)."""
    shape = (512, 768)
    p0, g, buf0 = make(shape, 1, 0.02), make(shape, 3).bfloat16().float(), make(shape, 4)
    p_ref = torch.nn.Parameter(p0.clone())
    opt = torch.optim.Muon([p_ref], lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    opt.state[p_ref]["momentum_buffer"] = buf0.clone()
    p_ref.grad = g.clone()
    opt.step()
    p, buf = p0.to(DEV), buf0.to(DEV)
    F.muon_step(p, g.to(DEV), buf, lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    assert rel_fro(p.cpu() - p0, p_ref.detach() - p0) < MUON_TOL
    assert torch.allclose(buf.cpu(), opt.state[p_ref]["momentum_buffer"], rtol=1e-6, atol=1e-9)


def test_muon_step_many_matches_one_matrix_at_a_time():
    """Independent matrices of two sets of hyper-parameters, which share launches with their like: the same bits as one
    call per matrix (together they are few enough for the 64 x 64 tiles that each takes alone), work enqueued afterwards
    sees the updates, and an optimizer over several parameter groups goes the same way."""
    shapes = [(512, 768), (768, 512), (256, 256), (320, 200), (1024, 512)]
    hypers = [dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True), dict(lr=0.01, weight_decay=0.0, momentum=0.9, nesterov=False, adjust_lr_fn="match_rms_adamw")]
    params = [make(sh, 100 + i, 0.02) for i, sh in enumerate(shapes)]
    grads = [make(sh, 200 + i).bfloat16().float() for i, sh in enumerate(shapes)]
    bufs = [make(sh, 300 + i) for i, sh in enumerate(shapes)]
    one_p, one_b = [p.to(DEV) for p in params], [b.to(DEV) for b in bufs]
    ws = F.MuonWorkspace(DEV)
    for i in range(len(shapes)):
        F.muon_step(one_p[i], grads[i].to(DEV), one_b[i], workspace=ws, **hypers[i % 2])
    many_p, many_b = [p.to(DEV) for p in params], [b.to(DEV) for b in bufs]
    dev_grads = [g.to(DEV) for g in grads]
    F.muon_step_many([(many_p[i], dev_grads[i], many_b[i], hypers[i % 2]) for i in range(len(shapes))])
    total = sum(p.sum() for p in many_p)  # enqueued on the calling stream right behind the batch
    for i in range(len(shapes)):
        assert torch.equal(many_p[i], one_p[i]) and torch.equal(many_b[i], one_b[i])
        p_ref, b_ref = params[i].clone(), bufs[i].clone()
        O.muon_step(p_ref, grads[i], b_ref, **hypers[i % 2])
        assert rel_fro(many_p[i].cpu() - params[i], p_ref - params[i]) < MUON_TOL
    assert float(total) == float(sum(p.sum() for p in one_p))
    F.muon_step_many([])
    F.muon_step_many([(many_p[0], dev_grads[0], many_b[0], hypers[0])])
    F.muon_step(one_p[0], dev_grads[0], one_b[0], workspace=ws, **hypers[0])
    assert torch.equal(many_p[0], one_p[0])


@pytest.mark.parametrize("shapes", [[(3072, 3072), (3072, 3328), (3072, 3072)], [(512, 512), (512, 300)] * 8])
def test_muon_step_many_side_by_side_switch(monkeypatch, shapes):
    """With ``side_by_side=False`` (argument or environment) every matrix gets the bits of a call of its own, whatever else
    the call holds; sharing launches stays within the parity bar of the same result.  Matrices that change tiles and K
    cuts together (m = 3072: the triangle of 256 x 256 tiles occupies 78 of the CUs), and sixteen small ones that are more
    than one round of the 64 x 64 tiles each takes alone."""
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    params = [make(sh, 400 + i, 0.02).to(DEV) for i, sh in enumerate(shapes)]
    grads = [make(sh, 500 + i).bfloat16().float().to(DEV) for i, sh in enumerate(shapes)]
    ws = F.MuonWorkspace(DEV)
    alone_p, alone_b = [p.clone() for p in params], [torch.zeros_like(p) for p in params]
    for i in range(len(shapes)):
        F.muon_step(alone_p[i], grads[i], alone_b[i], workspace=ws, **kw)

    def batch(**how):
        ps, bs = [p.clone() for p in params], [torch.zeros_like(p) for p in params]
        F.muon_step_many([(ps[i], grads[i], bs[i], kw) for i in range(len(shapes))], **how)
        torch.cuda.synchronize()
        return ps, bs

    ps, bs = batch(side_by_side=False)
    assert all(torch.equal(a, b) for a, b in zip(ps, alone_p)) and all(torch.equal(a, b) for a, b in zip(bs, alone_b))
    monkeypatch.setenv("MATRIX_FSDP_MUON_SIDE_BY_SIDE", "0")
    ps, bs = batch()
    assert all(torch.equal(a, b) for a, b in zip(ps, alone_p))
    monkeypatch.delenv("MATRIX_FSDP_MUON_SIDE_BY_SIDE")
    for how in (dict(), dict(side_by_side=True)):
        ps, bs = batch(**how)
        for i in range(len(shapes)):
            assert rel_fro((ps[i] - params[i]).cpu(), (alone_p[i] - params[i]).cpu()) < MUON_TOL
            assert torch.equal(bs[i], alone_b[i])  # the momentum depends on no product


@pytest.mark.parametrize("side_by_side", [None, True, False])
def test_muon_step_many_on_the_streams_of_a_pool(side_by_side):
    """A caller's own side streams, used twice with new gradients: the update of one call per matrix within the parity bar,
    the momentum exactly, and work enqueued afterwards on the calling stream sees them.  A machine-filling matrix rides
    along; its launches stay on the calling stream unless every matrix is sent to the streams."""
    shapes = [(512, 768), (768, 512), (100, 36), (5120, 5120), (1024, 512)]
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    params = [make(sh, 960 + i, 0.02).to(DEV) for i, sh in enumerate(shapes)]
    bufs = [make(sh, 970 + i).to(DEV) for i, sh in enumerate(shapes)]
    one_p, one_b = [p.clone() for p in params], [b.clone() for b in bufs]
    many_p, many_b = [p.clone() for p in params], [b.clone() for b in bufs]
    pool, ws = F.MuonStreamPool(DEV), F.MuonWorkspace(DEV)
    for step in range(2):
        grads = [make(sh, 980 + 10 * step + i).to(DEV) for i, sh in enumerate(shapes)]
        for p, g, b in zip(one_p, grads, one_b):
            F.muon_step(p, g, b, workspace=ws, **kw)
        F.muon_step_many([(p, g, b, kw) for p, g, b in zip(many_p, grads, many_b)], workspace=ws, pool=pool, side_by_side=side_by_side)
        seen = [p.clone() for p in many_p]  # enqueued right behind the call
        torch.cuda.synchronize()
        for i in range(len(shapes)):
            assert torch.equal(many_b[i], one_b[i]) and torch.equal(many_p[i], seen[i])
            assert rel_fro(many_p[i] - params[i], one_p[i] - params[i]) < MUON_TOL, shapes[i]


def test_muon_step_many_takes_the_keywords_of_muon_step():
    """``shared_machine`` among a job's keywords: that matrix gets the bits of ``muon_step`` with the flag."""
    shapes = [(3072, 3072), (200, 100)]
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    params, grads = [make(sh, 990 + i, 0.02).to(DEV) for i, sh in enumerate(shapes)], [make(sh, 995 + i).to(DEV) for i, sh in enumerate(shapes)]
    many_p, one_p = [p.clone() for p in params], [p.clone() for p in params]
    keywords = [dict(kw, shared_machine=True), kw]
    F.muon_step_many([(p, g, torch.zeros_like(p), k) for p, g, k in zip(many_p, grads, keywords)])
    for p, g, k, have in zip(one_p, grads, keywords, many_p):
        F.muon_step(p, g, torch.zeros_like(p), **k)
        assert torch.equal(p, have)


def test_muon_argument_errors():
    p = torch.zeros(8, 8, device=DEV)
    with pytest.raises(ValueError, match="2D"):
        F.muon_step(p.view(-1), p.view(-1), p.view(-1), lr=0.1, weight_decay=0.0, momentum=0.9, nesterov=True)
    with pytest.raises(RuntimeError, match="dtype"):
        F.muon_step(p, p.bfloat16(), p, lr=0.1, weight_decay=0.0, momentum=0.9, nesterov=True)
    with pytest.raises(ValueError, match="less than 100"):
        F.newton_schulz(p, ns_steps=100)
    with pytest.raises(ValueError, match="2D"):
        F.newton_schulz(p.view(-1))
    with pytest.raises(RuntimeError, match="Learning rate"):
        F.muon_step(p, p.clone(), p.clone(), lr=-1.0, weight_decay=0.0, momentum=0.9, nesterov=True)


@pytest.mark.parametrize("n", [1, 3, 1000, 4099, 1 << 20])
@pytest.mark.parametrize("grad_dtype", [torch.float32, torch.bfloat16])
def test_adamw_parity(n, grad_dtype):
    p_cpu, m_cpu, v_cpu = make((n,), 5, 0.02), torch.zeros(n), torch.zeros(n)
    p, m, v = p_cpu.to(DEV), m_cpu.to(DEV), v_cpu.to(DEV)
    kw = dict(lr=3e-4, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)
    for t in (1, 2, 3):
        g = make((n,), 30 + t).to(grad_dtype)
        O.adamw_step(p_cpu, g.float(), m_cpu, v_cpu, t, **kw)
        F.adamw_step(p, g.to(DEV), m, v, t, **kw)
        assert max_err_over_scale(p, p_cpu) < 1e-6
        assert max_err_over_scale(m, m_cpu) < 1e-6
        assert max_err_over_scale(v, v_cpu) < 1e-6


@pytest.mark.parametrize("amsgrad,maximize", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("n", [1000, 4099])
def test_adamw_amsgrad_and_maximize_parity(n, amsgrad, maximize):
    p_cpu, m_cpu, v_cpu = make((n,), 5, 0.02), torch.zeros(n), torch.zeros(n)
    x_cpu = torch.zeros(n) if amsgrad else None
    p, m, v = p_cpu.to(DEV), m_cpu.to(DEV), v_cpu.to(DEV)
    x = torch.zeros(n, device=DEV) if amsgrad else None
    kw = dict(lr=3e-3, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1, maximize=maximize)
    for t, scale in enumerate((1.0, 0.05, 0.2, 0.01), start=1):  # shrinking grads: the running maximum matters
        g = make((n,), 30 + t) * scale
        O.adamw_step(p_cpu, g, m_cpu, v_cpu, t, max_exp_avg_sq=x_cpu, **kw)
        F.adamw_step(p, g.to(DEV), m, v, t, max_exp_avg_sq=x, **kw)
        assert max_err_over_scale(p, p_cpu) < 1e-6
        assert max_err_over_scale(m, m_cpu) < 1e-6
        assert max_err_over_scale(v, v_cpu) < 1e-6
        if amsgrad:
            assert max_err_over_scale(x, x_cpu) < 1e-6
    if amsgrad:
        assert not torch.equal(x, v)


def test_optimizer_scalars_are_formed_in_double():
    """``1 - beta2`` for beta2 = 0.999 is 1.3e-5 off when it is formed from an fp32 beta2, and ``1 - momentum``
    for 0.95 is 2.4e-7 off: the entry points take doubles and round once, as the tensor operations of torch do, so
    the moments agree with the oracle to an fp32 rounding or two element by element."""
    n = 5000
    p_cpu, m_cpu, v_cpu = make((n,), 5, 0.02), torch.zeros(n), torch.zeros(n)
    p, m, v = p_cpu.to(DEV), m_cpu.to(DEV), v_cpu.to(DEV)
    kw = dict(lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01)
    for t in (1, 2, 3):
        g = make((n,), 50 + t)
        O.adamw_step(p_cpu, g, m_cpu, v_cpu, t, **kw)
        F.adamw_step(p, g.to(DEV), m, v, t, **kw)
        # the same operations in the same order as torch's single-tensor path, each rounded once; torch's CPU
        # kernels fuse some multiply-adds depending on the host's vector ISA, so the last bit may differ
        assert float(((v.cpu() - v_cpu).abs() / v_cpu.abs().clamp_min(1e-30)).max()) < 4e-7
        assert float((m.cpu() - m_cpu).abs().max()) <= 1.2e-7 * float(m_cpu.abs().max())
        assert float((p.cpu() - p_cpu).abs().max()) <= 1.2e-7 * float(p_cpu.abs().max())
    # Muon's momentum buffer (fp32 lerp with weight 1 - 0.95)
    shape = (64, 128)
    grad, buf = make(shape, 60), make(shape, 61)
    param = make(shape, 62, 0.02)
    buf_cpu = buf.clone()
    O.muon_step(param.clone(), grad, buf_cpu, lr=0.02, weight_decay=0.0, momentum=0.95, nesterov=True)
    buf_dev = buf.to(DEV)
    F.muon_step(param.to(DEV), grad.to(DEV), buf_dev, lr=0.02, weight_decay=0.0, momentum=0.95, nesterov=True)
    assert float((buf_dev.cpu() - buf_cpu).abs().max()) <= 1.2e-7 * float(buf_cpu.abs().max())


def test_adamw_unaligned_views_and_errors():
    n = 1001
    base = [torch.zeros(n + 1, device=DEV) for _ in range(3)]
    p, m, v = (b[1:] for b in base)
    p.copy_(make((n,), 6, 0.02))
    g = make((n,), 7).to(DEV)
    p_cpu, m_cpu, v_cpu = p.cpu().clone(), torch.zeros(n), torch.zeros(n)
    O.adamw_step(p_cpu, g.cpu(), m_cpu, v_cpu, 1, lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01)
    F.adamw_step(p, g, m, v, 1, lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01)
    assert max_err_over_scale(p, p_cpu) < 1e-6
    assert all(float(b[0]) == 0.0 for b in base)
    with pytest.raises(RuntimeError, match="step"):
        F.adamw_step(p, g, m, v, 0, lr=1e-3)
    with pytest.raises(RuntimeError, match="float32"):
        F.adamw_step(p.bfloat16(), g, m, v, 1, lr=1e-3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("short", [1, 63, 64, 65, 127, 129, 255, 257])
def test_muon_group_at_tile_edges(short, dtype):
    """Matrices around the edges of 64, 128 and 256 tiles, wide and tall, in one launch per stage: the momentum and the
    bits of a call of their own (all of them together are within one round of 64 x 64 tiles, which each takes alone too,
    and no K walk is cut), and the oracle's update."""
    shapes = [(short, short), (short, 200), (200, short), (short, 700), (700, short), (320, 256)]
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    params = [make(sh, 800 + i, 0.02).to(dtype) for i, sh in enumerate(shapes)]
    grads = [make(sh, 820 + i).to(dtype) for i, sh in enumerate(shapes)]
    bufs = [make(sh, 840 + i).to(dtype) for i, sh in enumerate(shapes)]
    many_p, many_b = [p.to(DEV) for p in params], [b.to(DEV) for b in bufs]
    F.muon_step_many([(p, g.to(DEV), b, kw) for p, g, b in zip(many_p, grads, many_b)])
    for i in range(len(shapes)):
        p, b = params[i].to(DEV), bufs[i].to(DEV)
        F.muon_step(p, grads[i].to(DEV), b, **kw)
        assert torch.equal(many_p[i], p) and torch.equal(many_b[i], b), shapes[i]
        p_ref, b_ref = params[i].clone(), bufs[i].clone()
        O.muon_step(p_ref, grads[i], b_ref, **kw)
        # a bf16 parameter moves in steps of its own last bit (see test_muon_step_matches_oracle)
        assert rel_fro((many_p[i].cpu() - params[i]).float(), (p_ref - params[i]).float()) < (MUON_TOL if dtype == torch.float32 else 5e-2), shapes[i]


def test_muon_group_larger_than_a_launch_and_than_the_workspace():
    """More matrices than one launch carries, a workspace that holds only the largest of them (so that every launch has
    one or two) and parameters at odd offsets of a flat shard: bits of the one-by-one calls."""
    import ctypes

    from matrix_fsdp_amd import _lib

    shapes = [(96, 160), (33, 70), (160, 96)] * 13
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.9, nesterov=False)
    flats = [[torch.randn(r * c + 3, generator=torch.Generator().manual_seed(900 + 3 * i + k)) for k in range(3)] for i, (r, c) in enumerate(shapes)]

    def views():
        return [[f.to(DEV)[1 : 1 + r * c].view(r, c) for f in three] for three, (r, c) in zip(flats, shapes)]

    one = views()
    for p, g, b in one:
        F.muon_step(p, g, b, **kw)
    many = views()
    F.muon_step_many([(p, g, b, kw) for p, g, b in many])
    tight = views()
    ws = torch.empty(F.muon_workspace_bytes(96, 160), dtype=torch.uint8, device=DEV)
    jobs = (_lib.MuonJob * len(tight))(*((p.data_ptr(), g.data_ptr(), b.data_ptr(), *p.shape, 0.02, 0.1, F.adjust_lr(0.02, None, p.shape)) for p, g, b in tight))
    args = (_lib.DT_F32, 0.9, 0, *F.NS_COEFFICIENTS, 5, F.NS_EPS)
    _lib.check(_lib.lib().mfsdp_muon_step_many(len(tight), jobs, *args, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    for a, b, c in zip(one, many, tight):
        assert torch.equal(a[0], b[0]) and torch.equal(a[2], b[2]) and torch.equal(a[0], c[0])
    before = tight[0][0].clone()
    jobs[5].rows = 0  # one bad job: nothing is enqueued
    assert _lib.lib().mfsdp_muon_step_many(len(tight), jobs, *args, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream) == 1
    jobs[5].rows = shapes[5][0]
    assert _lib.lib().mfsdp_muon_step_many(len(tight), jobs, *args, ws.data_ptr(), ws.numel() - 256, torch.cuda.current_stream().cuda_stream) == 1
    torch.cuda.synchronize()
    assert torch.equal(tight[0][0], before)
    assert _lib.lib().mfsdp_muon_many_workspace_bytes(1, (ctypes.c_int64 * 1)(96), (ctypes.c_int64 * 1)(160)) == ws.numel()


def test_muon_group_with_a_side_too_long_is_refused_whole():
    """A matrix whose long side no product takes, behind an ordinary one: the call raises and neither has changed."""
    shapes = [(64, 96), (1, (1 << 22) + 1)]
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.9, nesterov=True)
    mats = [[make(sh, 950 + 3 * i + k).to(DEV) for k in range(3)] for i, sh in enumerate(shapes)]
    before = [[t.clone() for t in three] for three in mats]
    with pytest.raises(RuntimeError, match="2\\^22"):
        F.muon_step_many([(p, g, b, kw) for p, g, b in mats])
    torch.cuda.synchronize()
    assert all(torch.equal(t, u) for three, old in zip(mats, before) for t, u in zip(three, old))
    torch.cuda.empty_cache()  # the workspace of the long matrix


def test_muon_step_many_machine_filling_matrices_go_alone():
    """Two matrices that fill the machine between small ones: they get the bits of a call of their own and the small ones
    those of a call without them, whether or not the workspace has room for more."""
    shapes = [(64, 96), (4865, 5120), (300, 520), (5120, 4900), (96, 64)]
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    params = [make(sh, 940 + i, 0.02).to(DEV) for i, sh in enumerate(shapes)]
    grads = [make(sh, 945 + i).to(DEV) for i, sh in enumerate(shapes)]

    def update(which, workspace=None):
        ps, bs = [params[i].clone() for i in which], [torch.zeros_like(params[i]) for i in which]
        F.muon_step_many([(p, grads[i], b, kw) for i, p, b in zip(which, ps, bs)], workspace=workspace)
        return dict(zip(which, ps))

    want = {**update([0, 2, 4]), **update([1]), **update([3])}
    roomy = F.MuonWorkspace(DEV)
    roomy.get_bytes(3 * F.muon_workspace_bytes(5120, 5120))
    for workspace in (None, roomy):
        have = update(list(range(5)), workspace)
        assert all(torch.equal(have[i], want[i]) for i in range(5))


def test_muon_group_with_ragged_partial_sums():
    """Matrices whose numbers of partial sums leave every remainder by four, beside ones so large that the norms are summed
    by a launch of their own: the oracle's update and momentum."""
    shapes = [(1, 7), (33, 70), (40, 60), (20, 200), (777, 1411), (600, 900), (1, 700)]
    partials = [max(1, -(-(r * c // 4) // 128)) for r, c in shapes]
    assert {n % 4 for n in partials} == {0, 1, 2, 3} and max(partials) > 1024
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    params = [make(sh, 600 + i, 0.02) for i, sh in enumerate(shapes)]
    grads = [make(sh, 610 + i, 1e-3 * 4.0**i) for i, sh in enumerate(shapes)]  # norms far apart
    bufs = [make(sh, 620 + i, 1e-3 * 4.0**i) for i, sh in enumerate(shapes)]
    for order in (range(len(shapes)), reversed(range(len(shapes)))):
        order = list(order)
        dev_p, dev_b = [params[i].to(DEV) for i in order], [bufs[i].to(DEV) for i in order]
        F.muon_step_many([(p, grads[i].to(DEV), b, kw) for i, p, b in zip(order, dev_p, dev_b)])
        for i, p, b in zip(order, dev_p, dev_b):
            p_ref, b_ref = params[i].clone(), bufs[i].clone()
            O.muon_step(p_ref, grads[i], b_ref, **kw)
            assert rel_fro(p.cpu() - params[i], p_ref - params[i]) < MUON_TOL, shapes[i]
            assert torch.allclose(b.cpu(), b_ref, rtol=1e-6, atol=1e-6 * float(b_ref.abs().max()))


@pytest.mark.parametrize("variant", [1, 2, 3, 4])
def test_muon_group_reads_nothing_stale_and_nothing_of_its_neighbours(variant):
    """Sides around the 64 that operands are zero-padded to, some K walks cut: a workspace full of NaN gives the bits of a
    cleared one, and a matrix whose gradient is NaN or infinite leaves those of the others alone."""
    from matrix_fsdp_amd import _lib

    shapes = [(63, 65), (130, 2100), (64, 1153), (300, 257), (1, 7), (1200, 190)]
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    params, grads = [make(sh, 700 + i, 0.02).to(DEV) for i, sh in enumerate(shapes)], [make(sh, 710 + i).to(DEV) for i, sh in enumerate(shapes)]

    def update(fill, bad=None):
        ps, bs, gs = [p.clone() for p in params], [torch.zeros_like(p) for p in params], [g.clone() for g in grads]
        if bad is not None:
            gs[1][5, 7] = bad
            gs[3][0, 0] = bad
        workspace = F.MuonWorkspace(DEV)
        workspace.get_bytes(256 << 20).fill_(fill)
        F.muon_step_many([(p, g, b, kw) for p, g, b in zip(ps, gs, bs)], workspace=workspace)
        return ps

    _lib.lib().mfsdp_set_muon_tuning(variant, variant, 0, 0, 0)
    try:
        want, stale = update(0), update(0xFF)
        spoiled = [update(0, float("nan")), update(0xFF, float("inf"))]
    finally:
        _lib.lib().mfsdp_set_muon_tuning(3, 3, 0, 0, 0)
    for i in range(len(shapes)):
        assert torch.isfinite(want[i]).all() and torch.equal(stale[i], want[i]), shapes[i]
        for ps in spoiled:
            assert torch.isnan(ps[i]).all() if i in (1, 3) else torch.equal(ps[i], want[i]), shapes[i]


def test_muon_group_with_cut_k_walks():
    """Sides beyond 1024, where the tiles of the last round are cut along K: several K in one launch, against the oracle."""
    shapes = [(192, 1088), (130, 2100), (4160, 200), (70, 8200)]
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    params = [make(sh, 860 + i, 0.02) for i, sh in enumerate(shapes)]
    grads = [make(sh, 870 + i) for i, sh in enumerate(shapes)]
    dev_p, dev_b = [p.to(DEV) for p in params], [torch.zeros(sh, device=DEV) for sh in shapes]
    F.muon_step_many([(p, g.to(DEV), b, kw) for p, g, b in zip(dev_p, grads, dev_b)])
    for i, sh in enumerate(shapes):
        p_ref, b_ref = params[i].clone(), torch.zeros(sh)
        O.muon_step(p_ref, grads[i], b_ref, **kw)
        assert rel_fro(dev_p[i].cpu() - params[i], p_ref - params[i]) < MUON_TOL, sh


@pytest.mark.parametrize("number", [np.array, np.float64, torch.tensor, lambda x: torch.tensor(x, device=DEV)], ids=["0-d array", "numpy scalar", "tensor", "device tensor"])
def test_hyper_parameters_of_any_number_type(number):
    """Learning rates and the like as numpy or torch numbers, which a scheduler may leave in a group: the bits of floats."""
    p0, g0 = make((40, 60), 1, 0.02).to(DEV), make((40, 60), 2).to(DEV)
    adam = dict(lr=1e-3, eps=1e-8, weight_decay=0.1)
    muon = dict(lr=0.02, weight_decay=0.1, momentum=0.95, eps=1e-7)
    results = []
    for convert in (float, lambda x: number(float(x))):
        p, q, r = p0.clone(), p0.clone(), p0.clone()
        F.adamw_step(p, g0, torch.zeros_like(p), torch.zeros_like(p), 1, betas=(convert(0.5), convert(0.75)), **{k: convert(v) for k, v in adam.items()})
        F.muon_step_many([(t, g0, torch.zeros_like(t), dict(nesterov=True, ns_coefficients=tuple(convert(c) for c in (3.0, -4.0, 2.0)), **{k: convert(v) for k, v in muon.items()}))
                          for t in (q, r)])
        results.append((p, q, r))
    tight = number is np.array or number is np.float64
    for have, want in zip(results[1], results[0]):
        # a torch number is rounded to fp32 on its way
        assert torch.equal(have, want) if tight else rel_fro(have - p0, want - p0) < 1e-4


@pytest.mark.parametrize("amsgrad", [False, True])
@pytest.mark.parametrize("count", [1, 4, 5, 56, 57, 130])
def test_adamw_batch_has_the_bits_of_single_spans(count, amsgrad):
    """Spans of 0 to a few thousand elements at any element offset, with step counts and gradient types of their own, in
    launches of up to 56: the bits of one call per span, and nothing outside the spans is touched."""
    edges = [0, 1, 3, 4, 5, 255, 256, 257, 511, 512, 513, 1023, 1025, 4099]
    sizes = [edges[(7 * i + count) % len(edges)] for i in range(count)]
    starts = [sum(sizes[:i]) + i + 1 for i in range(count)]  # a gap of one element before every span
    total = sum(sizes) + count + 8
    flats = [make((total,), 70 + k, 0.02).to(DEV) for k in range(5)]
    flats[3].abs_()
    flats[4].abs_()
    expect = [f.clone() for f in flats]

    def run(tensors, batch):
        p, g, m, v, x = tensors
        for i, (a, n) in enumerate(zip(starts, sizes)):
            cut = slice(a, a + n)
            grad = g[cut].bfloat16() if i % 5 == 3 else g[cut]
            F.adamw_step(p[cut], grad, m[cut], v[cut], 1 + i % 3, lr=1e-3, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1,
                         max_exp_avg_sq=x[cut] if amsgrad else None, batch=batch)

    run(expect, None)
    batch = F.AdamWBatch()
    run(flats, batch)
    batch.launch()
    for have, want in zip(flats, expect):
        assert torch.equal(have, want)
    batch.launch()  # nothing is left in it
    assert torch.equal(flats[0], expect[0])
    # overlapping parameters keep their order
    p, q = flats[0].clone(), flats[0].clone()
    g, m, v = flats[1], torch.zeros(total, device=DEV), torch.zeros(total, device=DEV)
    for target, b in ((p, None), (q, F.AdamWBatch())):
        first, second = (torch.zeros(4, device=DEV) for _ in range(2))
        F.adamw_step(target[0:4], g[0:4], first, second, 1, lr=0.1, batch=b)
        F.adamw_step(target[2:6], g[2:6], m[2:6].clone(), v[2:6].clone(), 1, lr=0.1, batch=b)
        if b is not None:
            b.launch()
    assert torch.equal(p, q)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shapes", [[(1, 1)], [(64, 64), (65, 63)], [(1024, 1024)], [(960, 1100)], [(1000, 40), (40, 1000), (33, 2047)], [(512, 1536)] * 2,
                                    [(200, 3000)], [(128, 130)] * 9, [(100, 300)] * 33])
def test_muon_small_tiles_against_the_oracle(shapes, dtype):
    """Launches of at most one round of 64 x 64 tiles: every K length of a wave's share (no step, one to four, several
    batches), up to 8 and more problems per launch, matrices whose norm is summed on the way and larger ones, wide and
    tall.  The same launches forced to 128 x 128 tiles give the same update to bf16 rounding."""
    from matrix_fsdp_amd import _lib

    params = [make(s, 300 + i, 0.02).to(dtype) for i, s in enumerate(shapes)]
    grads = [make(s, 400 + i).to(dtype) for i, s in enumerate(shapes)]
    bufs = [make(s, 500 + i).to(dtype) for i, s in enumerate(shapes)]
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    results = []
    try:
        for variant in (4, 2, 3):
            _lib.lib().mfsdp_set_muon_tuning(variant, variant, 0, 0, 0)
            p, b = [t.to(DEV) for t in params], [t.to(DEV) for t in bufs]
            F.muon_step_many([(pi, g.to(DEV), bi, kw) for pi, g, bi in zip(p, grads, b)])
            results.append((p, b))
    finally:
        _lib.lib().mfsdp_set_muon_tuning(3, 3, 0, 0, 0)
    for i in range(len(shapes)):
        want_p, want_b = params[i].clone(), bufs[i].clone()
        O.muon_step(want_p, grads[i], want_b, **kw)
        step = (want_p.double() - params[i].double()).norm()
        # bf16 rounding of the five iterations' products in another order: the bar the other variants are held to; a bf16
        # parameter adds its own rounding, 2^-9 of its value on either side
        bar = 1e-2 * step + (0.0 if dtype == torch.float32 else 2.0**-8 * params[i].double().norm())
        for have_p, have_b in results:
            assert (have_p[i].double().cpu() - want_p.double()).norm() <= bar, shapes[i]
            # one lerp in fp32, in bf16 rounded once: a last bit where the host fuses a multiply-add
            assert rel_fro(have_b[i], want_b) < (1e-6 if dtype == torch.float32 else 4e-3), shapes[i]


@pytest.mark.parametrize("variant", [1, 2, 3])
def test_muon_many_matrices_of_several_k_over_several_rounds(variant):
    """Thirteen matrices in one launch per stage (the argument table of 32), of three K lengths in every product, with more
    tiles than the machine holds at a time (update product: 423 of 256 x 256, 1479 of 128 x 128), wide and tall, by 256 and
    128 tiles and as the library chooses: ``torch.optim.Muon`` on this GPU, every matrix and its momentum."""
    from matrix_fsdp_amd import _lib

    shapes = [(1024, 1024), (1100, 2100), (4100, 640)] * 2 + [(1024, 1024), (2100, 1100)] * 2 + [(1024, 1024), (2100, 1100), (1024, 1024)]
    kw = dict(lr=0.02, weight_decay=0.1, momentum=0.95, nesterov=True)
    params, grads, bufs = ([make(sh, base + i, std).to(DEV) for i, sh in enumerate(shapes)] for base, std in ((1000, 0.02), (1020, 1e-3), (1040, 1e-3)))
    have_p, have_b = [p.clone() for p in params], [b.clone() for b in bufs]
    _lib.lib().mfsdp_set_muon_tuning(variant, variant, 0, 0, 0)
    try:
        F.muon_step_many([(p, g, b, kw) for p, g, b in zip(have_p, grads, have_b)])
    finally:
        _lib.lib().mfsdp_set_muon_tuning(3, 3, 0, 0, 0)
    torch_params = [torch.nn.Parameter(p.clone()) for p in params]
    optimizer = torch.optim.Muon(torch_params, **kw)
    for p, g, b in zip(torch_params, grads, bufs):
        optimizer.state[p]["momentum_buffer"] = b.clone()
        p.grad = g
    optimizer.step()
    for i, p in enumerate(torch_params):
        assert rel_fro(have_p[i] - params[i], p.detach() - params[i]) < MUON_TOL, (i, shapes[i])
        assert torch.allclose(have_b[i], optimizer.state[p]["momentum_buffer"], rtol=1e-6, atol=1e-9)
