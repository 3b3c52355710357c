"""The ``AdamW`` class and the side entry points on the GPU: several steps
against the reference's own op sequence, unbiasedness of the Philox rounding,
grad-norm clip, centralization, copy_stochastic_.  Run with ``-m gpu``.
"""
import copy
import time

import numpy as np
import pytest
import torch

import oracle
from oracle import torch_ops
import ramtorch_amd
from ramtorch_amd import _native as N
from ramtorch_amd import functional as F

pytestmark = pytest.mark.gpu
HP0 = dict(lr=1e-4, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01)


def dev16(a, dt=torch.bfloat16):
    return torch.from_numpy(a.view(np.int16).copy()).view(dt).cuda()


def nmis(a, b):
    """Number of elements whose bits differ (keeps assertion messages short)."""
    a, b = a.detach().cpu().contiguous(), b.detach().cpu().contiguous()
    assert a.shape == b.shape and a.dtype == b.dtype, (a.shape, b.shape, a.dtype, b.dtype)
    it = {2: torch.int16, 4: torch.int32}[a.element_size()]
    return int((a.view(it) != b.view(it)).sum())


def bits16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16).ravel()


def _make_params(shapes, seed, device="cuda"):
    ps, grads = [], []
    for i, shp in enumerate(shapes):
        n = int(np.prod(shp)) if len(shp) else 1
        p, g, _, _ = oracle.synth_inputs(n, seed + i)
        ps.append(torch.nn.Parameter(dev16(p).view(shp).to(device)))
        grads.append(dev16(g).view(shp))
    return ps, grads


def test_three_steps_match_the_reference_op_sequence():
    """GPU params, GPU states, explicit noise: bit-exact against the ATen op
    sequence of the reference (adamw.py:160-222) run on the same GPU."""
    shapes = [(64, 48), (1000,), (3, 5, 7), ()]
    ps, grads = _make_params(shapes, 100)
    ref_p = [p.detach().clone() for p in ps]
    opt = ramtorch_amd.AdamW([{"params": ps[:2]}, {"params": ps[2:], "lr": 5e-4, "weight_decay": 0.0}], lr=1e-3,
                             storage_device="cuda")
    ref_m = [torch.zeros_like(p) for p in ref_p]
    ref_v = [torch.zeros_like(p) for p in ref_p]
    for step in (1, 2, 3):
        noise = {}
        for i, p in enumerate(ps):
            p.grad = (grads[i].float() * (1.0 + 0.1 * step)).bfloat16()
            noise[p] = tuple(torch.randint(-32768, 32768, p.shape, dtype=torch.int16, device="cuda",
                                           generator=torch.Generator("cuda").manual_seed(step * 10 + i * 3 + k))
                             for k in range(3))
        opt.step(noise=noise)
        torch.cuda.synchronize()
        for i, p in enumerate(ps):
            grp = opt.param_groups[0 if i < 2 else 1]
            torch_ops.reference_step_ops(ref_p[i], p.grad, ref_m[i], ref_v[i], lr=grp["lr"], betas=grp["betas"],
                                         eps=grp["eps"], weight_decay=grp["weight_decay"], step=step, noise=noise[p])
            assert nmis(p.detach(), ref_p[i]) == 0, f"step {step} param {i}"
            assert nmis(opt.state[p]["ema"], ref_m[i]) == 0, f"step {step} ema {i}"
            assert nmis(opt.state[p]["ema_squared"], ref_v[i]) == 0, f"step {step} ema_squared {i}"
            assert opt.state[p]["step"] == step


def _nmis_any(a, b):
    a, b = a.detach().cpu().contiguous(), b.detach().cpu().contiguous()
    assert a.shape == b.shape and a.dtype == b.dtype, (a.shape, b.shape, a.dtype, b.dtype)
    it = {2: torch.int16, 4: torch.int32, 8: torch.int64}[a.element_size()]
    return int((a.view(it) != b.view(it)).sum())


@pytest.mark.parametrize("p_dt,s_dt", [(torch.float16, torch.float16), (torch.float32, torch.float16),
                                        (torch.float64, torch.float64), (torch.bfloat16, torch.float16),
                                        (torch.float16, torch.bfloat16)])
@pytest.mark.parametrize("where", ["cuda", "cpu"])
def test_other_param_and_state_dtypes_match_the_reference_op_sequence(p_dt, s_dt, where):
    """The reference accepts any float dtype: everything is upcast to fp32 (adamw.py:160-170) and what
    is not bf16 is written back with a plain copy_ (adamw.py:208,214,221-222).  Two steps, GPU
    states and host-resident (pinned) states, against the same ATen calls on the GPU."""
    shapes = [(40, 33), (8192 + 11,), (5,)]
    ps, grads, ref_p = [], [], []
    for i, shp in enumerate(shapes):
        n = int(np.prod(shp))
        p, g, _, _ = oracle.synth_inputs(n, 700 + i)
        p32 = torch.from_numpy(oracle.bf16_to_f32(p).copy()).view(shp) * 1.001
        t = p32.to(p_dt)
        if where == "cpu":
            t = t.pin_memory()
        else:
            t = t.cuda()
        ps.append(torch.nn.Parameter(t, requires_grad=False))
        ref_p.append(t.detach().clone().cuda())
        grads.append(dev16(g).view(shp))
    opt = ramtorch_amd.AdamW(ps, lr=1e-3, dtype=s_dt, storage_device=where, stream_chunk_bytes=16384)
    ref_m = [torch.zeros_like(p, dtype=s_dt) for p in ref_p]
    ref_v = [torch.zeros_like(p, dtype=s_dt) for p in ref_p]
    for step in (1, 2):
        noise, gmap = {}, {}
        for i, p in enumerate(ps):
            # the gradient has the parameter's dtype and lives where the parameter lives, as autograd
            # leaves it (fp64 and CPU gradients included: adamw.py:167 takes any float dtype, any device)
            gmap[p] = (grads[i].float() * (1.0 + 0.25 * step)).to(p_dt)
            p.grad = gmap[p].to(p.device)
            noise[p] = tuple(torch.randint(-32768, 32768, p.shape, dtype=torch.int16, device="cuda",
                                           generator=torch.Generator("cuda").manual_seed(step * 10 + i * 3 + k))
                             for k in range(3))
        opt.step(noise=noise)
        torch.cuda.synchronize()
        for i, p in enumerate(ps):
            st = opt.state[p]
            assert st["ema"].dtype == s_dt and st["ema_squared"].dtype == s_dt and p.dtype == p_dt
            assert st["ema"].device.type == where
            torch_ops.reference_step_ops(ref_p[i], gmap[p], ref_m[i], ref_v[i], lr=1e-3, betas=(0.9, 0.999),
                                         eps=1e-8, weight_decay=1e-2, step=step, noise=noise[p])
            assert _nmis_any(p.detach(), ref_p[i]) == 0, f"step {step} param {i}"
            assert _nmis_any(st["ema"], ref_m[i]) == 0, f"step {step} ema {i}"
            assert _nmis_any(st["ema_squared"], ref_v[i]) == 0, f"step {step} ema_squared {i}"


@pytest.mark.parametrize("where", ["cuda", "cpu"])
def test_reference_noise_mode_is_bit_identical_to_the_reference_step(where):
    """noise_source="reference": the rounding noise is drawn exactly as adamw.py:10-21 does
    (generators seeded step+42 / +69 / +420), so whole steps equal the reference's op
    sequence drawing its own noise -- nothing is passed in from outside."""
    shapes = [(64, 48), (1000,), (3, 5, 7), (8192 * 2 + 3,)]
    ps, grads = _make_params(shapes, 1300, device="cuda")
    if where == "cpu":
        ps = [torch.nn.Parameter(p.detach().cpu().pin_memory()) for p in ps]
    ref_p = [p.detach().clone().cuda() for p in ps]
    opt = ramtorch_amd.AdamW(ps, lr=2e-3, storage_device=where, noise_source="reference", stream_chunk_bytes=32768)
    ref_m = [torch.zeros_like(p) for p in ref_p]
    ref_v = [torch.zeros_like(p) for p in ref_p]
    for step in (1, 2, 3):
        gmap = {p: (grads[i].float() * (1.0 + 0.3 * step)).bfloat16() for i, p in enumerate(ps)}
        opt.step(grads=gmap)
        torch.cuda.synchronize()
        for i, p in enumerate(ps):
            torch_ops.reference_step_ops(ref_p[i], gmap[p], ref_m[i], ref_v[i], lr=2e-3, betas=(0.9, 0.999), eps=1e-8,
                                         weight_decay=1e-2, step=step, noise=None)
            assert nmis(p.detach(), ref_p[i]) == 0, f"step {step} param {i}"
            assert nmis(opt.state[p]["ema"], ref_m[i]) == 0, f"step {step} ema {i}"
            assert nmis(opt.state[p]["ema_squared"], ref_v[i]) == 0, f"step {step} ema_squared {i}"


def test_skipped_and_sparse_gradients():
    ps, grads = _make_params([(32, 8), (40,)], 200)
    opt = ramtorch_amd.AdamW(ps, storage_device="cuda")
    ps[0].grad = grads[0]
    before = ps[1].detach().clone()
    opt.step()
    torch.cuda.synchronize()
    assert opt.state[ps[0]]["step"] == 1 and opt.state[ps[1]]["step"] == 0  # adamw.py:114: no grad, no step
    assert nmis(ps[1].detach(), before) == 0
    emb = torch.nn.Parameter(torch.zeros(10, 4, device="cuda"))
    emb.grad = torch.sparse_coo_tensor(torch.tensor([[1], [2]]), torch.tensor([1.0]), (10, 4)).cuda()
    with pytest.raises(RuntimeError, match="sparse"):
        ramtorch_amd.AdamW([emb], storage_device="cuda").step()


def test_lr_schedule_is_reread_every_step():
    ps, grads = _make_params([(128,)], 300)
    opt = ramtorch_amd.AdamW(ps, lr=1e-3, storage_device="cuda", seed=4)
    sched = torch.optim.lr_scheduler.LambdaLR(opt, lambda e: 0.5 ** e)
    p_ref, m_ref, v_ref = (bits16(ps[0]), np.zeros(128, np.uint16), np.zeros(128, np.uint16))
    g = bits16(grads[0])
    for step in (1, 2, 3):
        ps[0].grad = grads[0]
        opt.step()
        lr = opt.param_groups[0]["lr"]
        sc = oracle.scalars_from_hparams(lr, (0.9, 0.999), 1e-8, 1e-2, step)
        oracle.step_tensor(p_ref, g, m_ref, v_ref, sc, seed=4, step=step, tensor_id=0)
        sched.step()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(bits16(ps[0]), p_ref, err_msg=f"step {step} lr {lr}")
    assert opt.param_groups[0]["lr"] == pytest.approx(1e-3 * 0.125)


def test_state_dict_resume_continues_bit_exactly():
    ps, grads = _make_params([(300,), (16, 16)], 400)
    a = ramtorch_amd.AdamW(ps, storage_device="cuda", seed=11)
    for _ in range(2):
        for p, g in zip(ps, grads):
            p.grad = g
        a.step()
    sd = copy.deepcopy(a.state_dict())   # state_dict() hands out the live tensors; a checkpoint would not
    ps2 = [torch.nn.Parameter(p.detach().clone()) for p in ps]
    b = ramtorch_amd.AdamW(ps2, storage_device="cuda", seed=11)
    b.load_state_dict(sd)
    for opt, params in ((a, ps), (b, ps2)):
        for p, g in zip(params, grads):
            p.grad = g
        opt.step()
    torch.cuda.synchronize()
    for p, q in zip(ps, ps2):
        assert nmis(p.detach(), q.detach()) == 0
        assert nmis(a.state[p]["ema_squared"], b.state[q]["ema_squared"]) == 0 and b.state[q]["step"] == 3


def test_non_contiguous_param_round_trips():
    base = torch.nn.Parameter(dev16(oracle.synth_inputs(64 * 32, 500)[0]).view(64, 32).t())  # transposed view
    assert not base.is_contiguous()
    g = dev16(oracle.synth_inputs(64 * 32, 500)[1]).view(64, 32).t()
    ref = torch.nn.Parameter(base.detach().contiguous())
    o1 = ramtorch_amd.AdamW([base], storage_device="cuda", seed=2)
    o2 = ramtorch_amd.AdamW([ref], storage_device="cuda", seed=2)
    base.grad, ref.grad = g, g.contiguous()
    o1.step(), o2.step()
    torch.cuda.synchronize()
    assert nmis(base.detach().contiguous(), ref.detach()) == 0


def test_philox_rounding_is_unbiased_over_1e8_elements():
    """Mean signed rounding error of each of p, m, v below 1e-3 bf16 ulp over 1e8 elements."""
    n = 100_000_000
    h = N.Handle(0)
    gen = torch.Generator("cuda").manual_seed(1234)
    P = (torch.randn(n, device="cuda", generator=gen) * 0.02).bfloat16()
    G = (torch.randn(n, device="cuda", generator=gen) * 1e-3).bfloat16()
    M = (torch.randn(n, device="cuda", generator=gen) * 1e-4).bfloat16()
    V = ((torch.randn(n, device="cuda", generator=gen) * 1e-3) ** 2).bfloat16()
    dbg = tuple(torch.empty(n, device="cuda") for _ in range(3))
    e = F.Entry(p=P, g=G, m=M, v=V, step=100, scalars_idx=0, tensor_id=0, dbg=dbg)
    F.step_resident(h, [e], [F.make_scalars(step=100, **HP0)], seed=1234, explicit_noise=False)
    torch.cuda.synchronize()
    for name, out, pre in zip("pmv", (P, M, V), dbg):
        # one bf16 ulp at the magnitude of the fp32 value: 2^(exponent - 7)
        ulp = torch.ldexp(torch.ones_like(pre), torch.frexp(pre)[1] - 8)
        err = ((out.double() - pre.double()) / ulp.double())
        err = err[pre != 0]
        assert float(err.abs().max()) < 1.0 + 1e-9, name          # never further than one ulp
        mean = float(err.mean())
        assert abs(mean) < 1e-3, f"{name}: mean rounding error {mean:.3e} ulp"
        assert 0.05 < float(err.std()) < 0.5, name                 # it does randomise
    # the three arrays do not share noise: errors of p and m are uncorrelated
    ep = (P.float() - dbg[0])[:10_000_000]
    em = (M.float() - dbg[1])[:10_000_000]
    c = torch.corrcoef(torch.stack([ep / ep.std(), em / em.std()]))[0, 1]
    assert abs(float(c)) < 5e-3
    h.close()


def test_philox_noise_matches_oracle_stream_and_differs_between_steps_and_tensors():
    n = 10_000
    p, g, m, v = oracle.synth_inputs(n, 600)
    h = N.Handle(0)
    outs = {}
    for step, tid, seed in ((5, 0, 1), (6, 0, 1), (5, 1, 1), (5, 0, 2)):
        e = F.Entry(p=dev16(p), g=dev16(g), m=dev16(m), v=dev16(v), step=step, scalars_idx=0, tensor_id=tid)
        F.step_resident(h, [e], [F.make_scalars(step=5, **HP0)], seed=seed, explicit_noise=False)
        torch.cuda.synchronize()
        outs[(step, tid, seed)] = bits16(e.p)
        po, mo, vo = p.copy(), m.copy(), v.copy()
        oracle.step_tensor(po, g, mo, vo, oracle.scalars_from_hparams(step=5, **HP0), seed=seed, step=step,
                           tensor_id=tid)
        np.testing.assert_array_equal(outs[(step, tid, seed)], po)
    keys = list(outs)
    for i in range(len(keys)):
        for j in range(i + 1, len(keys)):
            assert (outs[keys[i]] != outs[keys[j]]).mean() > 0.05
    h.close()


def test_grad_norm_clip_and_skip():
    h = N.Handle(0)
    rng = np.random.default_rng(0)
    grads_np = [(rng.normal(0, 1e-3, n).astype(np.float32) * 1024) for n in (1, 1000, 8192 * 3 + 7, 250_000)]
    grads = [torch.from_numpy(g).cuda() for g in grads_np] + [torch.zeros(0, device="cuda")]
    grads.append(dev16(oracle.f32_to_bf16_rne(grads_np[1])))
    out = F.grad_norm(h, grads, inv_loss_scale=1 / 1024, max_norm=0.01)
    torch.cuda.synchronize()
    want = sum(oracle.grad_sumsq(g, oracle.DT_F32, 1 / 1024) for g in grads_np)
    want += oracle.grad_sumsq(oracle.f32_to_bf16_rne(grads_np[1]), oracle.DT_BF16, 1 / 1024)
    total = float(out[0])
    assert total == pytest.approx(want ** 0.5, rel=1e-6)
    assert np.float32(out[1].item()) == oracle.clip_coef(np.float32(total), 0.01)
    assert out.view(torch.int32)[2].item() == 0
    again = F.grad_norm(h, grads, inv_loss_scale=1 / 1024, max_norm=0.01)
    assert nmis(out[:2], again[:2]) == 0  # deterministic reduction order
    grads[2][5] = float("inf")
    bad = F.grad_norm(h, grads, inv_loss_scale=1 / 1024, max_norm=0.01)
    assert bad.view(torch.int32)[2].item() == 1 and float(bad[1]) == 1.0
    h.close()


def test_optimizer_with_loss_scale_and_max_grad_norm():
    """Config-4 layout: bf16 p, fp32 grads pre-scaled by 1024, global clip to 1.0."""
    shapes = [(256, 64), (512,)]
    ps, _ = _make_params(shapes, 700)
    opt = ramtorch_amd.AdamW(ps, storage_device="cuda", seed=8, loss_scale=1024.0, max_grad_norm=1.0, **HP0)
    gnp = [np.random.default_rng(i).normal(0, 0.05, int(np.prod(s))).astype(np.float32) * 1024 for i, s in
           enumerate(shapes)]
    gmap = {p: torch.from_numpy(g).cuda().view(p.shape) for p, g in zip(ps, gnp)}  # fp32 grads of bf16 params
    before = [bits16(p) for p in ps]
    opt.step(grads=gmap)
    torch.cuda.synchronize()
    total = float(opt.last_grad_norm[0])
    coef = np.float32(opt.last_grad_norm[1].item())
    assert total == pytest.approx(sum(oracle.grad_sumsq(g, oracle.DT_F32, 1 / 1024) for g in gnp) ** 0.5, rel=1e-6)
    assert coef < 1.0
    sc = oracle.scalars_from_hparams(step=1, inv_loss_scale=1 / 1024, apply_clip=True, **HP0)
    for i, (p, g) in enumerate(zip(ps, gnp)):
        n = g.size
        po, mo, vo = before[i].copy(), np.zeros(n, np.uint16), np.zeros(n, np.uint16)
        oracle.step_tensor(po, g, mo, vo, sc, g_dtype=oracle.DT_F32, clip_coef=coef, seed=8, step=1, tensor_id=i)
        np.testing.assert_array_equal(bits16(p), po)
        np.testing.assert_array_equal(bits16(opt.state[p]["ema_squared"]), vo)
    # a non-finite gradient skips the whole update
    snap = [p.detach().clone() for p in ps]
    gmap[ps[0]][0, 0] = float("nan")
    opt.step(grads=gmap)
    torch.cuda.synchronize()
    assert all(nmis(a, b.detach()) == 0 for a, b in zip(snap, ps))
    assert opt.last_grad_norm.view(torch.int32)[2].item() == 1


@pytest.mark.parametrize("shape", [(37, 24), (4, 3, 10), (129,), (), (64, 300), (3000, 8), (5, 4099), (16, 1024, 3),
                                   (20_000,), (4, 8192), (2500, 7), (2, 40_000), (70_001,), (3, 32_768), (3, 32_769)])
def test_centralization(shape):
    n = int(np.prod(shape)) if len(shape) else 1
    p, g, _, _ = oracle.synth_inputs(n, 800)
    P = torch.nn.Parameter(dev16(p).view(shape))
    P.grad = dev16(g).view(shape)
    opt = ramtorch_amd.AdamW([P], storage_device="cuda", seed=3, centralization=0.5, **HP0)
    opt.step()
    torch.cuda.synchronize()
    rows = shape[0] if len(shape) >= 2 else 1
    row_len = n // rows
    h = N.Handle(0)
    means = F.row_means(h, P.grad.contiguous(), rows, row_len).cpu().numpy()
    np.testing.assert_allclose(means, oracle.row_means(g, rows, row_len), rtol=2e-6, atol=1e-9)
    # same means in, bit-exact out: g' = g - fl(mean * c), then the usual update
    g32 = oracle.bf16_to_f32(g) - (np.repeat(means, row_len) * np.float32(0.5)).astype(np.float32)
    po, mo, vo = p.copy(), np.zeros(n, np.uint16), np.zeros(n, np.uint16)
    oracle.step_tensor(po, g32.astype(np.float32), mo, vo, oracle.scalars_from_hparams(step=1, **HP0),
                       g_dtype=oracle.DT_F32, seed=3, step=1, tensor_id=0)
    np.testing.assert_array_equal(bits16(P), po)
    # and against torch's own formulation (adamw.py:179-184), within the mean's tolerance
    gt = P.grad.float()
    gt = gt - gt.mean(dim=tuple(range(1, gt.dim())), keepdim=True) * 0.5
    np.testing.assert_allclose(g32.reshape(shape), gt.cpu().numpy(), rtol=1e-5, atol=1e-9)
    h.close()


@pytest.mark.parametrize("shape", [(64, 300), (3, 70_001), (9000, 12)])
def test_centralization_in_pieces_equals_whole(shape):
    """Host-resident states: the tensor is updated in staged pieces that start in the middle of rows
    (and of the tensor); whole units of a piece take the fast kernel's centralizing variant, the
    rest the generic kernel.  Same bits as the resident step."""
    n = int(np.prod(shape))
    p, g, _, _ = oracle.synth_inputs(n, 810)
    out = []
    for storage, extra in (("cuda", {}), ("cpu", dict(stream_chunk_bytes=2 * 10_000))):
        P = torch.nn.Parameter(dev16(p).view(shape))
        P.grad = dev16(g).view(shape)
        opt = ramtorch_amd.AdamW([P], storage_device=storage, seed=3, centralization=0.25, **extra, **HP0)
        for _ in range(2):
            opt.step()
        torch.cuda.synchronize()
        out.append((bits16(P), bits16(opt.state[P]["ema"]), bits16(opt.state[P]["ema_squared"])))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_row_means_of_many_gradients_in_one_launch():
    """rt_row_means_multi = rt_row_means tensor by tensor, bit for bit (same summation), for row
    lengths around the vector width and on both sides of the length from which a row takes a whole
    workgroup, unaligned views and every gradient dtype."""
    rng = np.random.default_rng(11)
    h = N.Handle(0)
    jobs, singles = [], []
    for k in range(40):
        row_len = int(rng.choice([1, 3, 8, 12, 100, 511, 4096, 5000, 32_768, 33_001, 70_001]))   # one wavefront per row up to 32 768 elements, a workgroup beyond
        rows = int(rng.integers(1, 40))
        dt = [torch.bfloat16, torch.float32, torch.float16][k % 3]
        off = int(rng.integers(0, 3))                     # a view that does not start on 16 bytes
        g = (torch.randn(rows * row_len + off, device="cuda") * 1e-3).to(dt)[off:]
        e = F.Entry(p=g, g=g, m=g, v=g, step=1, scalars_idx=0, tensor_id=k)
        jobs.append((e, rows, row_len))
        singles.append(F.row_means(h, g, rows, row_len, 0.5))
    F.row_means_multi(h, jobs, 0.5)
    torch.cuda.synchronize()
    for k, ((e, rows, row_len), one) in enumerate(zip(jobs, singles)):
        assert e.row_len == row_len and e.row_mean.numel() == rows
        assert nmis(e.row_mean, one) == 0, (k, rows, row_len)
        want = (e.g.double().view(rows, row_len) * 0.5).mean(dim=1).cpu().numpy()
        np.testing.assert_allclose(e.row_mean.cpu().numpy(), want, rtol=3e-6, atol=1e-9)
    h.close()


def test_clip_with_centralization():
    """max_grad_norm and centralization together (neither the combination nor the clip is in the
    reference): the clip coefficient scales the gradient and its row means alike, as clip_grad_norm_
    followed by step() would; then fl(mean * coef) * c is subtracted.  Both kernels that centralize."""
    shapes = [(64, 300), (37, 24), (5, 4099)]
    ps, gs = [], []
    for i, shp in enumerate(shapes):
        p, g, _, _ = oracle.synth_inputs(int(np.prod(shp)), 830 + i)
        ps.append(torch.nn.Parameter(dev16(p).view(shp)))
        gs.append(g)
        ps[-1].grad = (dev16(g).float() * 40.0).bfloat16().view(shp)   # large enough for the clip to bite
    before = [bits16(p) for p in ps]
    opt = ramtorch_amd.AdamW(ps, storage_device="cuda", seed=5, centralization=0.5, max_grad_norm=1.0, **HP0)
    opt.step()
    torch.cuda.synchronize()
    total, coef, skip = opt.last_grad_norm.cpu().numpy()[:3]
    coef = np.float32(coef)
    assert 0.0 < coef < 1.0
    h = N.Handle(0)
    for i, (p, shp) in enumerate(zip(ps, shapes)):
        n = p.numel()
        rows, row_len = shp[0], n // shp[0]
        means = F.row_means(h, p.grad.contiguous(), rows, row_len).cpu().numpy()
        gb = bits16(p.grad)
        g32 = (oracle.bf16_to_f32(gb) * coef).astype(np.float32)
        g32 = (g32 - ((np.repeat(means, row_len) * coef).astype(np.float32) * np.float32(0.5)).astype(np.float32)).astype(np.float32)
        po, mo, vo = before[i].copy(), np.zeros(n, np.uint16), np.zeros(n, np.uint16)
        oracle.step_tensor(po, g32, mo, vo, oracle.scalars_from_hparams(step=1, **HP0), g_dtype=oracle.DT_F32, seed=5,
                           step=1, tensor_id=i)
        np.testing.assert_array_equal(bits16(p), po, err_msg=f"param {i}")
        np.testing.assert_array_equal(bits16(opt.state[p]["ema_squared"]), vo, err_msg=f"param {i} v")
    h.close()


def test_copy_stochastic_with_a_cpu_source():
    """adamw.py:6-30 rounds wherever ``source`` lives; here a CPU source goes through the GPU.  Same bits as
    the integer closed form, into a CPU target and into a GPU target, with Philox and with explicit noise."""
    n = 70_001
    src = torch.randn(n) * 0.02
    noise = torch.randint(-32768, 32768, (n,), dtype=torch.int16)
    for tgt in (torch.empty(n, dtype=torch.bfloat16), torch.empty(n, dtype=torch.bfloat16, device="cuda")):
        ramtorch_amd.copy_stochastic_(tgt, src, seed=5)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(bits16(tgt), oracle.sr_copy(src.numpy(), seed=5))
        ramtorch_amd.copy_stochastic_(tgt, src, noise=noise)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(bits16(tgt), oracle.sr_copy(src.numpy(), noise=noise.numpy()))
    # 2-d, a non-contiguous CPU target
    src2 = (torch.randn(60, 50) * 0.02)
    tgt2 = torch.empty(50, 60, dtype=torch.bfloat16).t()
    ramtorch_amd.copy_stochastic_(tgt2, src2, seed=6)
    np.testing.assert_array_equal(bits16(tgt2.contiguous()), oracle.sr_copy(src2.numpy().ravel(), seed=6))


@pytest.mark.parametrize("storage", ["cuda", "cpu"])
def test_a_step_cancelled_by_a_non_finite_norm_does_not_count(storage):
    """max_grad_norm with an infinite gradient: the kernels leave everything as it is, and the step counts
    the call had advanced are taken back, so that the next step is the one after the last that happened --
    same bias corrections, same Philox counter word (the reference increments right before its arithmetic,
    adamw.py:177; torch's GradScaler does not call step() at all on such gradients)."""
    shapes = [(256, 64), (3 * 8192 + 11,)]
    ps, grads = _make_params(shapes, 720, device=storage if storage == "cuda" else "cpu")
    if storage == "cpu":
        ps = [torch.nn.Parameter(p.detach().pin_memory()) for p in ps]
    opt = ramtorch_amd.AdamW(ps, storage_device=storage, seed=21, max_grad_norm=1e9, **HP0)
    gmap = {p: g.clone() for p, g in zip(ps, grads)}
    sc = lambda step: oracle.scalars_from_hparams(step=step, apply_clip=True, **HP0)
    model = [(bits16(p), np.zeros(p.numel(), np.uint16), np.zeros(p.numel(), np.uint16)) for p in ps]

    def good_step(step):
        opt.step(grads=gmap)
        torch.cuda.synchronize()
        for i, (p, (po, mo, vo)) in enumerate(zip(ps, model)):
            oracle.step_tensor(po, bits16(gmap[p]), mo, vo, sc(step), clip_coef=np.float32(1.0), seed=21, step=step, tensor_id=i)
            np.testing.assert_array_equal(bits16(p), po, err_msg=f"step {step} param {i}")
            np.testing.assert_array_equal(bits16(opt.state[p]["ema"]), mo, err_msg=f"step {step} ema {i}")
            np.testing.assert_array_equal(bits16(opt.state[p]["ema_squared"]), vo, err_msg=f"step {step} ema_squared {i}")

    good_step(1)
    assert not opt.step_was_skipped()
    keep = gmap[ps[1]][5].clone()
    gmap[ps[1]][5] = float("inf")
    opt.step(grads=gmap)                       # cancelled on the GPU
    torch.cuda.synchronize()
    for p, (po, mo, vo) in zip(ps, model):
        np.testing.assert_array_equal(bits16(p), po)
        np.testing.assert_array_equal(bits16(opt.state[p]["ema"]), mo)
    assert opt.step_was_skipped()
    assert [opt.state[p]["step"] for p in ps] == [1, 1]
    assert [v["step"] for v in opt.state_dict()["state"].values()] == [1, 1]
    gmap[ps[1]][5] = keep
    good_step(2)                               # the step after step 1, bit for bit
    assert not opt.step_was_skipped() and [opt.state[p]["step"] for p in ps] == [2, 2]
    # cancelled again, and this time the next step() itself finds out
    gmap[ps[0]][0, 0] = float("nan")
    opt.step(grads=gmap)
    gmap[ps[0]][0, 0] = 0.0
    good_step(3)


def test_step_param_that_raises_leaves_the_step_count_alone():
    ps, grads = _make_params([(64, 32)], 730)
    opt = ramtorch_amd.AdamW(ps, storage_device="cuda", seed=2, **HP0)
    opt.step_param(ps[0], grads[0])
    opt.step()
    assert opt.state[ps[0]]["step"] == 1
    before = bits16(ps[0])
    with pytest.raises(ValueError):
        opt.step_param(ps[0], grads[0].view(-1)[:100])           # a gradient of the wrong size
    torch.cuda.synchronize()
    assert opt.state[ps[0]]["step"] == 1 and id(ps[0]) not in opt._stepped_early
    np.testing.assert_array_equal(bits16(ps[0]), before)
    opt.step_param(ps[0], grads[0])                             # and the parameter can still be stepped
    opt.step()
    assert opt.state[ps[0]]["step"] == 2


def test_copy_stochastic():
    n = 100_003
    src = torch.randn(n, device="cuda") * 0.02
    noise = torch.randint(-32768, 32768, (n,), dtype=torch.int16, device="cuda")
    tgt = torch.empty(n, dtype=torch.bfloat16, device="cuda")
    ramtorch_amd.copy_stochastic_(tgt, src, noise=noise)
    torch.cuda.synchronize()
    want = oracle.sr_copy(src.cpu().numpy(), noise=noise.cpu().numpy())
    np.testing.assert_array_equal(bits16(tgt), want)
    ref = torch.empty_like(tgt)
    torch_ops.sr_write_(ref, src, torch_ops.noise_to_i32(noise))   # the reference's integer ops on the GPU
    assert nmis(ref, tgt) == 0
    ramtorch_amd.copy_stochastic_(tgt, src, seed=42)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bits16(tgt), oracle.sr_copy(src.cpu().numpy(), seed=42))
    cpu_tgt = torch.empty(n, dtype=torch.bfloat16)
    ramtorch_amd.copy_stochastic_(cpu_tgt, src, seed=42)
    assert nmis(cpu_tgt, tgt.cpu()) == 0
    # whole 2048-element blocks, short tails, sizes below one block, unaligned views
    big_t = torch.empty(3 * 2048 + 16, dtype=torch.bfloat16, device="cuda")
    for off, m in ((0, 2048), (0, 3 * 2048), (0, 2047), (0, 7), (1, 2048 + 5), (3, 4096), (8, 3 * 2048)):
        s_view, n_view, t_view = src[off:off + m], noise[off:off + m], big_t[off:off + m]
        for kw in (dict(seed=9), dict(noise=n_view)):
            big_t.zero_()
            ramtorch_amd.copy_stochastic_(t_view, s_view, **kw)
            torch.cuda.synchronize()
            want = (oracle.sr_copy(s_view.cpu().numpy(), seed=9) if "seed" in kw
                    else oracle.sr_copy(s_view.cpu().numpy(), noise=n_view.cpu().numpy()))
            np.testing.assert_array_equal(bits16(t_view), want, err_msg=f"offset {off} n {m} {list(kw)}")
            assert int(big_t[:off].view(torch.int16).abs().sum()) == 0 and int(big_t[off + m:].view(torch.int16).abs().sum()) == 0
    # the reference's own draw (adamw.py:10-21): a fresh generator seeded with `seed`
    src2 = src.view(-1)[:100_000].view(250, 400)
    tgt2 = torch.empty(250, 400, dtype=torch.bfloat16, device="cuda")
    ramtorch_amd.copy_stochastic_(tgt2, src2, seed=77, reference_noise=True)
    ref2 = torch.empty_like(tgt2)
    torch_ops.sr_write_(ref2, src2, torch_ops.draw_noise(src2.shape, 77, src2.device))
    assert nmis(ref2, tgt2) == 0


def test_gathered_step_equals_the_python_loop():
    """With many tensors AdamW.step collects descriptors in C++.  Same parameters through that
    path and through the Python loop (gatherer switched off): identical bits and step counts,
    also with skipped gradients, a non-contiguous parameter, two groups."""
    from ramtorch_amd import _gather as G
    if G.module() is None:
        pytest.skip("gather helper not built")
    rng = np.random.default_rng(11)
    lens = [int(x) for x in np.exp(rng.uniform(0, np.log(20000), 600)).astype(np.int64).clip(1, 20000)]

    def make():
        ps = []
        for i, n in enumerate(lens):
            p, g, _, _ = oracle.synth_inputs(n, 5000 + i)
            t = dev16(p)
            if i == 17:
                t = torch.stack([t, t], 1)[:, 0]  # not contiguous
            q = torch.nn.Parameter(t, requires_grad=False)
            ps.append(q)
        return ps

    def set_grads(ps, step):
        for i, (p, n) in enumerate(zip(ps, lens)):
            if (i + step) % 11 == 0:
                p.grad = None
                continue
            _, g, _, _ = oracle.synth_inputs(n, 5000 + i + 100 * step)
            p.grad = dev16(g).view(p.shape)

    a, b = make(), make()
    kw = dict(storage_device="cuda", seed=77)
    oa = ramtorch_amd.AdamW([{"params": a[:400]}, {"params": a[400:], "lr": 3e-4, "weight_decay": 0.0}], **kw)
    ob = ramtorch_amd.AdamW([{"params": b[:400]}, {"params": b[400:], "lr": 3e-4, "weight_decay": 0.0}], **kw)
    ob.gather_min_tensors = 10 ** 9  # Python loop only
    assert oa.gather_min_tensors <= len(a)
    for step in (1, 2, 3):
        set_grads(a, step)
        set_grads(b, step)
        oa.step()
        ob.step()
        torch.cuda.synchronize()
        for i, (p, q) in enumerate(zip(a, b)):
            assert oa.state[p]["step"] == ob.state[q]["step"], (step, i)
            assert nmis(p.detach(), q.detach()) == 0, (step, i)
            assert nmis(oa.state[p]["ema"], ob.state[q]["ema"]) == 0, (step, i)
            assert nmis(oa.state[p]["ema_squared"], ob.state[q]["ema_squared"]) == 0, (step, i)
    assert max(oa.state[p]["step"] for p in a) == 3 and min(oa.state[p]["step"] for p in a) >= 2


@pytest.mark.parametrize("option", ["clip", "central", "central_apart", "given_f32", "clip_central_given"])
def test_gathered_step_equals_the_python_loop_with_every_option(option):
    """The C++ gatherer under a clip, with centralization (row means inside the update and before it) and with
    gradients that are given, against the Python loop: the same bits and step counts, also with a parameter
    that only the loop can take, parameters without gradients, two step counts in a group, and a step that a
    non-finite norm cancels."""
    from ramtorch_amd import _gather as G
    if G.module() is None:
        pytest.skip("gather helper not built")
    shapes = [(33, 24), (9000,), (4, 512), (16, 3, 3, 3), (5,), (2, 4104), (40, 700), (3, 7), (1,), (64, 64)]
    kw = dict(storage_device="cuda", seed=31, loss_scale=4.0 if "given" in option else 1.0,
              max_grad_norm=0.02 if "clip" in option else None, centralization=0.5 if "central" in option else 0.0)

    def make():
        ps, _ = _make_params(shapes, 9000)
        ps[6] = torch.nn.Parameter(torch.stack([ps[6].detach()] * 2, 2)[..., 0], requires_grad=False)  # not contiguous
        opt = ramtorch_amd.AdamW([{"params": ps[:4]}, {"params": ps[4:], "lr": 3e-4, "centralization": 0.0}], **kw, **{k: v for k, v in HP0.items() if k != "lr"})
        opt.fuse_row_means = option != "central_apart"
        return ps, opt

    (a, oa), (b, ob) = make(), make()
    ob.gather_min_tensors = 10 ** 9
    for step in range(1, 6):
        given = []
        for ps in (a, b):
            own = {}
            for i, p in enumerate(ps):
                g = dev16(oracle.synth_inputs(p.numel(), 9100 + 17 * step + i)[1]).view(p.shape)
                if step == 4 and "clip" in option and i == 2:
                    g = g * float("inf")
                g = None if (i + step) % 7 == 0 else g
                if "given" in option and i != 3:
                    own[p] = None if g is None else g.float()
                    g = torch.ones_like(p)            # must not be used
                p.grad = g
            given.append(own if "given" in option else None)
        oa.step(grads=given[0])
        ob.step(grads=given[1])
        assert oa.step_was_skipped() == ob.step_was_skipped() == (step == 4 and "clip" in option)
        for i, (p, q) in enumerate(zip(a, b)):
            assert oa.state[p]["step"] == ob.state[q]["step"], (step, i)
            for x, y in ((p.detach(), q.detach()), (oa.state[p]["ema"], ob.state[q]["ema"]),
                         (oa.state[p]["ema_squared"], ob.state[q]["ema_squared"])):
                assert nmis(x, y) == 0, (step, i)
    assert len({oa.state[p]["step"] for p in a}) > 1


def test_pooled_state_placement_changes_nothing_but_addresses():
    """state_placement="auto": ema and ema_squared are views into two pools (placed in different
    HBM regions when the probe finds such a placement).  Results, state_dict and resume are the
    same as with plain per-tensor states."""
    shapes = [(9000, 8192), (70_000_003,), (4096,)]          # 143.7 M elements: 287 MB per pool
    def make():
        ps = []
        for i, shp in enumerate(shapes):
            g = torch.Generator("cuda").manual_seed(40 + i)
            ps.append(torch.nn.Parameter((torch.randn(shp, device="cuda", generator=g) * 0.02).bfloat16(),
                                         requires_grad=False))
        return ps
    a, b = make(), make()
    oa = ramtorch_amd.AdamW(a, storage_device="cuda", seed=5, ema_squared_dtype=torch.float32,
                            state_pool_min_bytes=64 << 20, **HP0)
    ob = ramtorch_amd.AdamW(b, storage_device="cuda", seed=5, ema_squared_dtype=torch.float32, state_placement="plain",
                            **HP0)
    rep = oa.state_placement_report
    assert rep is not None and rep["tries"] >= 1 and ob.state_placement_report is None
    pm, pv = oa._state_pools["ema"], oa._state_pools["ema_squared"]
    for p in a:
        st = oa.state[p]
        assert st["ema"].dtype == torch.bfloat16 and st["ema_squared"].dtype == torch.float32
        assert st["ema"].shape == p.shape and st["ema"].is_contiguous() and st["ema"].data_ptr() % 256 == 0
        assert pm.data_ptr() <= st["ema"].data_ptr() < pm.data_ptr() + pm.numel()
        assert pv.data_ptr() <= st["ema_squared"].data_ptr() < pv.data_ptr() + pv.numel()
        assert float(st["ema"].float().abs().max()) == 0.0 and float(st["ema_squared"].abs().max()) == 0.0
    for step in (1, 2):
        for i, (p, q) in enumerate(zip(a, b)):
            g = torch.Generator("cuda").manual_seed(100 * step + i)
            p.grad = (torch.randn(p.shape, device="cuda", generator=g) * 1e-3).bfloat16()
            q.grad = p.grad.clone()
        oa.step()
        ob.step()
    torch.cuda.synchronize()
    for p, q in zip(a, b):
        assert nmis(p.detach(), q.detach()) == 0
        assert nmis(oa.state[p]["ema"], ob.state[q]["ema"]) == 0
        assert _nmis_any(oa.state[p]["ema_squared"], ob.state[q]["ema_squared"]) == 0
    # resume into a fresh optimizer: the loaded values land in its own pools
    c = [torch.nn.Parameter(p.detach().clone(), requires_grad=False) for p in a]
    oc = ramtorch_amd.AdamW(c, storage_device="cuda", seed=0, ema_squared_dtype=torch.float32,
                            state_pool_min_bytes=64 << 20, **HP0)
    oc.load_state_dict(copy.deepcopy(oa.state_dict()))
    cm = oc._state_pools["ema"]
    for p, r in zip(a, c):
        assert oc.state[r]["step"] == 2 and oc.seed == 5
        assert cm.data_ptr() <= oc.state[r]["ema"].data_ptr() < cm.data_ptr() + cm.numel()
        assert nmis(oc.state[r]["ema"], oa.state[p]["ema"]) == 0
        assert _nmis_any(oc.state[r]["ema_squared"], oa.state[p]["ema_squared"]) == 0
        r.grad = p.grad.clone()
    oa.step()
    oc.step()
    torch.cuda.synchronize()
    for p, r in zip(a, c):
        assert nmis(p.detach(), r.detach()) == 0


def test_random_parameter_sets_match_the_oracle():
    """Seeded random optimizer-level cases: 1 to 300 tensors, GPU / pinned / pageable parameters,
    GPU or host states, one or two groups, skipped gradients, C++ gatherer on or off, three steps."""
    rng = np.random.default_rng(77)

    def t16(a, where, pin):
        t = torch.from_numpy(a.view(np.int16).copy()).view(torch.bfloat16)
        if where == "cuda":
            return t.cuda()
        return t.pin_memory() if pin else t

    hp = dict(lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01)
    hp2 = dict(lr=3e-4, betas=(0.8, 0.99), eps=1e-8, weight_decay=0.0)
    for case in range(40):
        k = int(rng.choice([1, 3, 17, 40, 300]))
        p_where, s_where = str(rng.choice(["cuda", "cpu"])), str(rng.choice(["cuda", "cpu"]))
        pin = bool(rng.random() < 0.7)
        seed = int(rng.integers(0, 1 << 40))
        lens = [max(1, int(x)) for x in np.exp(rng.uniform(0, np.log(30000), k))]
        if rng.random() < 0.3:
            lens[0] = 8192 * int(rng.integers(1, 5))
        ps, ref = [], []
        for i, n in enumerate(lens):
            p, _, _, _ = oracle.synth_inputs(n, seed % 1000 + i)
            shape = (n,) if n % 4 or rng.random() < 0.5 else (n // 4, 4)
            ps.append(torch.nn.Parameter(t16(p, p_where, pin).view(shape), requires_grad=False))
            ref.append([p.copy(), np.zeros(n, np.uint16), np.zeros(n, np.uint16), 0])
        cut = k if k < 3 or rng.random() < 0.5 else int(rng.integers(1, k))
        groups = [{"params": ps[:cut]}] + ([{"params": ps[cut:], **hp2}] if cut < k else [])
        opt = ramtorch_amd.AdamW(groups, storage_device=s_where, seed=seed,
                                 stream_chunk_bytes=int(rng.choice([4096, 65536, 1 << 20])), **hp)
        opt.gather_min_tensors = int(rng.choice([1, 10 ** 9]))
        for step in (1, 2, 3):
            grads = []
            for i, p in enumerate(ps):
                if rng.random() < 0.15:
                    p.grad = None
                    grads.append(None)
                    continue
                _, g, _, _ = oracle.synth_inputs(lens[i], seed % 1000 + 7 * i + step)
                p.grad = t16(g, p_where, False).view(p.shape)
                grads.append(g)
            opt.step()
            torch.cuda.synchronize()
            for i, p in enumerate(ps):
                r = ref[i]
                if grads[i] is not None:
                    r[3] += 1
                    sc = oracle.scalars_from_hparams(step=r[3], **(hp if i < cut else hp2))
                    oracle.step_tensor(r[0], grads[i], r[1], r[2], sc, seed=seed, step=r[3], tensor_id=i)
                st = opt.state[p]
                what = f"case {case} ({k} tensors, params {p_where}, states {s_where}) tensor {i} step {step}"
                assert st["step"] == r[3], what
                assert int((bits16(p) != r[0]).sum()) == 0, what
                assert int((bits16(st["ema"]) != r[1]).sum()) == 0, what
                assert int((bits16(st["ema_squared"]) != r[2]).sum()) == 0, what


def test_deepcopied_optimizer_steps_like_the_original():
    ps, grads = _make_params([(300,), (16, 16)], 1500)
    opt = ramtorch_amd.AdamW(ps, storage_device="cuda", seed=9, **HP0)
    for p, g in zip(ps, grads):
        p.grad = g
    opt.step()
    twin = copy.deepcopy(opt)          # copies parameters, states and the configuration
    qs = twin.param_groups[0]["params"]
    assert twin.seed == 9 and all(q is not p for p, q in zip(ps, qs))
    for q, g in zip(qs, grads):
        q.grad = g.clone()
    opt.step()
    twin.step()
    torch.cuda.synchronize()
    for p, q in zip(ps, qs):
        assert nmis(p.detach(), q.detach()) == 0
        assert nmis(opt.state[p]["ema"], twin.state[q]["ema"]) == 0
        assert opt.state[p]["step"] == twin.state[q]["step"] == 2


@pytest.mark.parametrize("n_params", [4, 300])  # 300: the C++ gatherer has advanced step counts before the error
@pytest.mark.parametrize("kind", ["sparse", "bad dtype"])
def test_a_step_that_raises_leaves_step_counts_and_tensors_untouched(n_params, kind):
    """The reference raises before it touches the offending tensor (adamw.py:118-119); here whatever
    the step had already counted for the tensors before it is put back."""
    shapes = [(16, 8)] * (n_params - 1) + [(10, 4)]
    ps, grads = _make_params(shapes, 5000)
    kw = {}
    if kind == "bad dtype":
        ps[-1] = torch.nn.Parameter(torch.zeros(10, 4, device="cuda", dtype=torch.float8_e4m3fn), requires_grad=False)
    groups = [{"params": ps[:-1]}, {"params": ps[-1:]}]
    opt = ramtorch_amd.AdamW(groups, storage_device="cuda", dtype=torch.bfloat16, **kw)
    for p, g in zip(ps[:-1], grads):
        p.grad = g
    opt.step()  # one good step first (the last parameter has no gradient yet), so that the counts are not all zero
    torch.cuda.synchronize()
    snap = [(p.detach().clone(), opt.state[p]["ema"].clone(), opt.state[p]["ema_squared"].clone()) for p in ps[:-1]]
    steps = [opt.state[p]["step"] for p in ps]
    if kind == "sparse":
        ps[-1].grad = torch.sparse_coo_tensor(torch.tensor([[1], [2]]), torch.tensor([1.0]), (10, 4)).cuda().bfloat16()
        err = RuntimeError
    else:
        ps[-1].grad = torch.zeros(10, 4, device="cuda", dtype=torch.float8_e4m3fn)
        err = NotImplementedError
    with pytest.raises(err):
        opt.step()
    torch.cuda.synchronize()
    assert [opt.state[p]["step"] for p in ps] == steps
    for p, (p0, m0, v0) in zip(ps[:-1], snap):
        assert nmis(p.detach(), p0) == 0 and nmis(opt.state[p]["ema"], m0) == 0
        assert nmis(opt.state[p]["ema_squared"], v0) == 0
    # and the optimizer still steps once the offending gradient is gone
    ps[-1].grad = None
    opt.step()
    assert [opt.state[p]["step"] for p in ps[:-1]] == [s + 1 for s in steps[:-1]]


def test_short_sqrt_sequence_equals_sqrtf_on_its_whole_domain():
    """The update kernels' sqrt for wavefronts whose second moments all lie in [2^-96, inf) against the
    compiler's correctly rounded sqrtf, on every one of the 1 879 048 192 floats of that range."""
    h = N.Handle(0)
    try:
        assert h.selftest_sqrt() == 0
    finally:
        h.close()


def test_zeros_denormals_and_tiny_second_moments_take_the_full_sqrt():
    """Wavefronts with a zero, a denormal or a tiny second moment leave the short sqrt path; both paths
    must give the oracle's bits, also side by side in one launch (fp32 states carry the small values)."""
    n = 64 * 8 * 6 + 24
    rng = np.random.default_rng(3)
    p = rng.normal(0, 0.02, n).astype(np.float32)
    g = np.zeros(n, np.float32)
    m = rng.normal(0, 1e-4, n).astype(np.float32)
    v = (rng.normal(0, 1e-3, n).astype(np.float32)) ** 2
    v[512:1024] = 0.0                                   # a whole wavefront of zeros
    v[1024 + 7] = np.float32(1e-40)                     # one denormal in an otherwise ordinary wavefront
    v[1536:2048] = np.float32(2.0 ** -100)              # tiny but normal
    v[2048 + 5] = np.float32(np.inf)
    g[2560:] = rng.normal(0, 1e-3, n - 2560).astype(np.float32)
    P, G, M, V = (torch.from_numpy(a.copy()).cuda() for a in (p, g, m, v))
    h = N.Handle(0)
    try:
        e = F.Entry(p=P, g=G, m=M, v=V, step=7, scalars_idx=0, tensor_id=0)
        F.step_resident(h, [e], [F.make_scalars(step=7, **HP0)], seed=5, explicit_noise=False)
        torch.cuda.synchronize()
    finally:
        h.close()
    po, mo, vo = p.copy(), m.copy(), v.copy()
    oracle.step_tensor(po, g, mo, vo, oracle.scalars_from_hparams(step=7, **HP0), p_dtype=oracle.DT_F32,
                       g_dtype=oracle.DT_F32, m_dtype=oracle.DT_F32, v_dtype=oracle.DT_F32, seed=5, step=7, tensor_id=0)
    for name, t, a in (("p", P, po), ("m", M, mo), ("v", V, vo)):
        got, want = t.cpu().numpy().view(np.uint32), a.view(np.uint32)
        both_nan = np.isnan(t.cpu().numpy()) & np.isnan(a)
        assert ((got == want) | both_nan).all(), name


def test_state_placement_with_most_of_hbm_occupied_falls_back_quietly():
    """The constructor's placement search occupies memory only through the library and only a bounded
    share of what is free: with most of HBM taken it ends at once, leaves torch's caching allocator
    alone, and the optimizer steps exactly like one with plainly allocated states."""
    GIB = 1 << 30
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    hog = [torch.empty(8 * GIB, dtype=torch.uint8, device="cuda") for _ in range(int((free - 16 * GIB) // (8 * GIB)))]
    try:
        n = 1 << 29   # 1 GiB of bf16 per array: the smallest set the search is used for
        gen = torch.Generator("cuda").manual_seed(5)
        base = (torch.randn(n, device="cuda", generator=gen) * 0.02).bfloat16()
        grad = (torch.randn(n, device="cuda", generator=gen) * 1e-3).bfloat16()
        p1 = torch.nn.Parameter(base.clone(), requires_grad=False)
        p2 = torch.nn.Parameter(base.clone(), requires_grad=False)
        del base
        torch.cuda.synchronize()
        reserved0 = torch.cuda.memory_reserved()
        t0 = time.monotonic()
        opt1 = ramtorch_amd.AdamW([p1], storage_device="cuda", seed=3, state_placement="auto", **HP0)
        took = time.monotonic() - t0
        rep = opt1.state_placement_report
        assert rep is not None and rep["tries"] >= 1 and isinstance(rep["placed"], bool), rep
        assert took < 10.0, took
        # torch holds the two pools and nothing else that it did not hold before
        assert torch.cuda.memory_reserved() - reserved0 <= 2 * GIB + (64 << 20)
        st = opt1.state[p1]
        assert float(st["ema"].float().abs().max()) == 0.0 and float(st["ema_squared"].float().abs().max()) == 0.0
        opt2 = ramtorch_amd.AdamW([p2], storage_device="cuda", seed=3, state_placement="plain", **HP0)
        for _ in range(2):
            p1.grad = grad
            p2.grad = grad
            opt1.step()
            opt2.step()
        torch.cuda.synchronize()
        assert torch.equal(p1.view(torch.int16), p2.view(torch.int16))
        for k in ("ema", "ema_squared"):
            assert torch.equal(opt1.state[p1][k].view(torch.int16), opt2.state[p2][k].view(torch.int16))
    finally:
        del hog
        torch.cuda.empty_cache()


def test_state_placement_of_two_large_optimizers_in_a_row():
    """A process that has allocated and released tens of GiB before (a second model, a second run in one
    process): the search must still end quickly, and say what it settled for.  Whatever place the states
    got, the steps are those of an optimizer with plainly allocated states."""
    n = 1 << 30    # 2 GiB of bf16 per array
    for round_ in range(2):
        gen = torch.Generator("cuda").manual_seed(50 + round_)
        base = (torch.randn(n, device="cuda", generator=gen) * 0.02).bfloat16()
        grad = (torch.randn(n, device="cuda", generator=gen) * 1e-3).bfloat16()
        ballast = [torch.empty(8 << 30, dtype=torch.uint8, device="cuda") for _ in range(4 + 2 * round_)]
        p1 = torch.nn.Parameter(base.clone(), requires_grad=False)
        p2 = torch.nn.Parameter(base, requires_grad=False)
        t0 = time.monotonic()
        opt1 = ramtorch_amd.AdamW([p1], storage_device="cuda", seed=3, state_placement="auto", **HP0)
        took = time.monotonic() - t0
        rep = opt1.state_placement_report
        assert rep is not None and rep["tries"] >= 1, rep
        assert rep["placed"] or rep["reason"], rep
        # about a second where measured; memory that the driver is still clearing makes every allocation slower
        assert rep["seconds"] < 5.0 and took < 6.0, (rep, took)
        opt2 = ramtorch_amd.AdamW([p2], storage_device="cuda", seed=3, state_placement="plain", **HP0)
        p1.grad = p2.grad = grad
        opt1.step(); opt2.step()
        torch.cuda.synchronize()
        assert torch.equal(p1.view(torch.int16), p2.view(torch.int16))
        assert torch.equal(opt1.state[p1]["ema_squared"].view(torch.int16), opt2.state[p2]["ema_squared"].view(torch.int16))
        del opt1, opt2, p1, p2, base, grad, ballast
        torch.cuda.empty_cache()       # tens of GiB go back to the driver: the next round starts in a used process


def test_state_placement_with_scattered_free_memory_is_as_clean_as_in_a_fresh_process():
    """Free device memory in scattered order -- every other block of many released -- is where one
    allocation of several GiB straddles HBM regions.  The pools are mapped from 1 GiB chunks that were
    probed one by one against the parameter's own memory: both are complete, they show the gain of lying
    in different regions, the probing has left every bit of the parameter as it was, and the steps are
    those of an optimizer with plainly allocated states."""
    GIB = 1 << 30
    blocks = [torch.empty(3 * GIB // 2, dtype=torch.uint8, device="cuda") for _ in range(120)]
    keep = blocks[::2]
    del blocks
    torch.cuda.empty_cache()
    try:
        n = 1 << 30    # 2 GiB of bf16 per array
        gen = torch.Generator("cuda").manual_seed(77)
        base = (torch.randn(n, device="cuda", generator=gen) * 0.02).bfloat16()
        grad = (torch.randn(n, device="cuda", generator=gen) * 1e-3).bfloat16()
        p1 = torch.nn.Parameter(base.clone(), requires_grad=False)
        p2 = torch.nn.Parameter(base, requires_grad=False)
        opt1 = ramtorch_amd.AdamW([p1], storage_device="cuda", seed=3, state_placement="auto", **HP0)
        torch.cuda.synchronize()
        rep = opt1.state_placement_report
        assert torch.equal(p1.view(torch.int16), p2.view(torch.int16)), "the placement probes changed the parameter"
        assert rep.get("by_chunks") and rep["placed"] and rep["share_apart"] == 1.0, rep
        assert rep["cross_GBps"] >= 1.03 * rep["same_GBps"], rep      # 6 - 7 % where measured
        assert rep["seconds"] < 3.0, rep                              # 0.2 s where measured
        st = opt1.state[p1]
        assert not bool(st["ema"].view(torch.int16).any()) and not bool(st["ema_squared"].view(torch.int16).any())
        opt2 = ramtorch_amd.AdamW([p2], storage_device="cuda", seed=3, state_placement="plain", **HP0)
        for _ in range(2):
            p1.grad = p2.grad = grad
            opt1.step(); opt2.step()
        torch.cuda.synchronize()
        assert torch.equal(p1.view(torch.int16), p2.view(torch.int16))
        for k in ("ema", "ema_squared"):
            assert torch.equal(opt1.state[p1][k].view(torch.int16), opt2.state[p2][k].view(torch.int16))
        # the pools go back to the driver with their last views
        free_before = torch.cuda.mem_get_info()[0]
        del opt1, st
        import gc
        gc.collect()
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] - free_before >= 4 * GIB - (64 << 20)
    finally:
        del keep
        torch.cuda.empty_cache()


def test_state_placement_without_probing_parameter_memory(monkeypatch):
    """placement.PROBE_WITH_PARAMETERS = False: chunks are sorted relative to the first chunk taken; the pools
    still come from individually probed chunks, lie apart from each other, hold zeros, and step like plain states."""
    from ramtorch_amd import placement
    monkeypatch.setattr(placement, "PROBE_WITH_PARAMETERS", False)
    n = 1 << 30
    gen = torch.Generator("cuda").manual_seed(78)
    base = (torch.randn(n, device="cuda", generator=gen) * 0.02).bfloat16()
    grad = (torch.randn(n, device="cuda", generator=gen) * 1e-3).bfloat16()
    p1 = torch.nn.Parameter(base.clone(), requires_grad=False)
    p2 = torch.nn.Parameter(base, requires_grad=False)
    opt1 = ramtorch_amd.AdamW([p1], storage_device="cuda", seed=3, state_placement="auto", **HP0)
    rep = opt1.state_placement_report
    assert rep.get("by_chunks") and (rep["placed"] or rep["reason"]), rep
    if rep["placed"]:
        assert rep["cross_GBps"] >= 1.03 * rep["same_GBps"], rep
    opt2 = ramtorch_amd.AdamW([p2], storage_device="cuda", seed=3, state_placement="plain", **HP0)
    p1.grad = p2.grad = grad
    opt1.step(); opt2.step()
    torch.cuda.synchronize()
    assert torch.equal(p1.view(torch.int16), p2.view(torch.int16))
    assert torch.equal(opt1.state[p1]["ema_squared"].view(torch.int16), opt2.state[p2]["ema_squared"].view(torch.int16))


@pytest.mark.parametrize("pdt,sdt", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                     (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("clip", [None, 0.05])
def test_centralization_inside_the_update_gives_the_bits_of_the_separate_row_mean_pass(pdt, sdt, clip, monkeypatch):
    """adamw.py:179-184.  Matrices whose rows fit a wavefront (a multiple of 8, 512 .. 32768 elements) have their
    rows summed inside the update kernel; everything else gets its means from the row-mean pass first.  Both
    ways sum a row in the same order, so an optimizer that never sums inside the update steps to the same bits
    (that path is checked against the oracle and the reference's op sequence elsewhere), with a loss
    scale and with a clip coefficient on gradient and mean."""
    shapes = [(64, 512), (7, 4096), (3, 14336), (5, 520), (3, 32768), (2, 3, 256), (40, 504), (9, 1000), (4, 516),
              (4096,), (3, 32776), (1, 512), (300, 8)]
    eligible = {0, 1, 2, 3, 4, 5, 7, 9, 11}   # rows a multiple of 8 and 512 .. 32768 long ((2,3,256): rows of 768)
    from ramtorch_amd import functional as F
    passes = []
    real = F.row_means_multi
    monkeypatch.setattr(F, "row_means_multi", lambda h, jobs, *a, **k: (passes.append(len(jobs)), real(h, jobs, *a, **k))[1])

    def make(**attrs):
        ps, grads = _make_params(shapes, 9100)
        ps = [torch.nn.Parameter(p.detach().to(pdt)) for p in ps]
        opt = ramtorch_amd.AdamW(ps, lr=2e-3, centralization=0.7, storage_device="cuda", dtype=sdt, seed=5,
                                 loss_scale=8.0, max_grad_norm=clip)
        for k, v in attrs.items():
            setattr(opt, k, v)
        return ps, grads, opt

    ps_a, grads, a = make()
    ps_b, _, b = make(fuse_row_means=False)
    for step in range(3):
        for x, y, g in zip(ps_a, ps_b, grads):
            x.grad = (g.float() * (8.0 + step)).to(pdt).cuda()
            y.grad = x.grad.clone()
        passes.clear()
        a.step()
        assert passes == [len(shapes) - len(eligible)], passes     # the rest is summed inside the update
        passes.clear()
        b.step()
        assert passes == [len(shapes)]
        torch.cuda.synchronize()
        for i, (x, y) in enumerate(zip(ps_a, ps_b)):
            assert nmis(x.detach(), y.detach()) == 0, (step, shapes[i])
            assert nmis(a.state[x]["ema"], b.state[y]["ema"]) == 0, (step, shapes[i])
            assert nmis(a.state[x]["ema_squared"], b.state[y]["ema_squared"]) == 0, (step, shapes[i])
    assert not a.step_was_skipped() and not b.step_was_skipped()
    if clip is None:
        # single parameters handed over as a backward hook would: the same choice per tensor
        for opt, ps in ((a, ps_a), (b, ps_b)):
            for i in (1, 6, 2):
                opt.step_param(ps[i])
            opt.step()
        torch.cuda.synchronize()
        for i, (x, y) in enumerate(zip(ps_a, ps_b)):
            assert nmis(x.detach(), y.detach()) == 0, shapes[i]
            assert nmis(a.state[x]["ema_squared"], b.state[y]["ema_squared"]) == 0, shapes[i]
            assert a.state[x]["step"] == b.state[y]["step"] == 4


def test_random_sets_step_alike_with_row_sums_inside_the_update_and_in_a_pass_of_their_own():
    """Seeded random parameter sets -- row lengths on both sides of every limit of the row-wise kernel
    (8, 512, 4096, 32768), 1-D to 3-D shapes, bf16 / fp16 parameters, bf16 / fp16 / fp32 states, two groups
    with different centralization (0 included), loss scale, clip, gradients that are missing in some
    steps: an optimizer that sums rows inside the update and one that never does agree bit for bit."""
    lens = [8, 64, 504, 512, 520, 1000, 1024, 4088, 4096, 4104, 8192, 14336, 32768, 32776, 516, 3, 40000]
    for seed in range(40):
        rng = np.random.default_rng(seed)
        shapes = []
        for _ in range(int(rng.integers(3, 14))):
            L = int(rng.choice(lens))
            rows = int(rng.integers(1, max(2, min(40, 400000 // L))))
            kind = rng.integers(0, 4)
            shapes.append((L,) if kind == 0 else (rows, 4, L // 4) if kind == 1 and L % 4 == 0 else (rows, L))
        pdt = [torch.bfloat16, torch.float16][int(rng.integers(0, 2))]
        sdt = [torch.bfloat16, torch.float16, torch.float32][int(rng.integers(0, 3))]
        clip = None if rng.random() < 0.5 else float(rng.choice([0.01, 1.0, 100.0]))
        ls = float(rng.choice([1.0, 8.0, 1024.0]))
        cut = int(rng.integers(1, len(shapes)))
        cens = (float(rng.choice([0.0, 0.3, 1.0])), float(rng.choice([0.5, 1.0])))

        def make(fuse):
            ps, grads = _make_params(shapes, 1000 + seed)
            ps = [torch.nn.Parameter(p.detach().to(pdt)) for p in ps]
            opt = ramtorch_amd.AdamW([{"params": ps[:cut], "centralization": cens[0]},
                                      {"params": ps[cut:], "centralization": cens[1], "lr": 3e-3}],
                                     lr=1e-3, storage_device="cuda", dtype=sdt, seed=seed, loss_scale=ls, max_grad_norm=clip)
            opt.fuse_row_means = fuse
            return ps, grads, opt

        ps_a, grads, a = make(True)
        ps_b, _, b = make(False)
        for step in range(3):
            for x, y, g in zip(ps_a, ps_b, grads):
                if rng.random() < 0.15:
                    x.grad = y.grad = None
                    continue
                x.grad = (g.float() * (ls * (1.0 + step))).to(pdt).cuda()
                y.grad = x.grad.clone()
            a.step(); b.step()
            torch.cuda.synchronize()
            for i, (x, y) in enumerate(zip(ps_a, ps_b)):
                what = (seed, step, shapes[i], pdt, sdt)
                assert nmis(x.detach(), y.detach()) == 0, what
                assert nmis(a.state[x]["ema"], b.state[y]["ema"]) == 0, what
                assert nmis(a.state[x]["ema_squared"], b.state[y]["ema_squared"]) == 0, what
                assert a.state[x]["step"] == b.state[y]["step"], what


def test_frozen_layout_steps_like_the_full_path_and_notices_moved_gradients():
    """assume_static_layout: after the first step the optimizer only checks that parameters and
    gradients are where they were.  Same bits as an optimizer that gathers everything every step,
    through a learning-rate change, a gradient that moves, one that vanishes, and state_dict()."""
    rng = np.random.default_rng(11)
    shapes = [(int(n),) for n in np.floor(np.exp(rng.uniform(0, np.log(3000), 396))).astype(int)] + [(64, 40)] * 4

    def make(**kw):
        ps, grads = _make_params(shapes, 7000)
        for i, (p, g) in enumerate(zip(ps, grads)):
            if i % 11 != 5:                  # some parameters never get a gradient
                p.grad = g.clone()
        return ps, ramtorch_amd.AdamW([{"params": ps[:300]}, {"params": ps[300:], "lr": 3e-4}], lr=1e-3,
                                      storage_device="cuda", seed=9, **kw)

    ps_a, a = make(assume_static_layout=True)
    ps_b, b = make()

    def same():
        torch.cuda.synchronize()
        for x, y in zip(ps_a, ps_b):
            assert nmis(x.detach(), y.detach()) == 0
            assert nmis(a.state[x]["ema"], b.state[y]["ema"]) == 0
            assert nmis(a.state[x]["ema_squared"], b.state[y]["ema_squared"]) == 0

    a.step(); b.step(); same()
    assert a._frozen is not None and a._frozen["pending"] == 0
    for k in range(3):
        for opt in (a, b):
            opt.param_groups[0]["lr"] *= 0.7          # a scheduler at work: re-read every step
        for x, y in zip(ps_a, ps_b):                  # gradients accumulate in place
            if x.grad is not None:
                x.grad.mul_(1.25); y.grad.mul_(1.25)
        a.step(); b.step(); same()
        assert a._frozen is not None and a._frozen["pending"] == k + 1 and a.layout_refreezes == 0
    sd_a, sd_b = a.state_dict(), b.state_dict()       # brings the lagging step counts up to date
    assert [sd_a["state"][i]["step"] for i in sorted(sd_a["state"])] == [sd_b["state"][i]["step"] for i in sorted(sd_b["state"])]
    # ... and the recorded layout stays in use afterwards, with the scalars of the step it really is
    # (bias corrections and step size come from the step count: one taken from before the save would
    # show in every element)
    a.step(); b.step(); same()
    assert a._frozen is not None and a._frozen["pending"] == 1 and a.layout_refreezes == 0
    twin = copy.deepcopy(a)                           # pickling brings the counts up to date as well
    assert [twin.state[p]["step"] for g in twin.param_groups for p in g["params"]] == [b.state[p]["step"] for p in ps_b]
    del twin
    a.step(); b.step(); same()
    assert a._frozen is not None and a._frozen["pending"] == 1 and a.layout_refreezes == 0
    # a state tensor replaced behind the optimizer's back: noticed, full path, same bits as doing it to b
    for opt, ps in ((a, ps_a), (b, ps_b)):
        opt.state[ps[3]]["ema"] = opt.state[ps[3]]["ema"].clone()
    a.step(); b.step(); same()
    assert a.layout_refreezes == 1 and a._frozen is not None
    a.layout_refreezes = 0
    # a gradient moves: caught, the step takes the full path and records the layout again
    for ps in (ps_a, ps_b):
        ps[7].grad = ps[7].grad.clone()
    a.step(); b.step(); same()
    assert a.layout_refreezes == 1 and a._frozen is not None
    a.step(); b.step(); same()
    assert a._frozen["pending"] == 1
    # one vanishes, one appears
    for ps in (ps_a, ps_b):
        ps[8].grad = None
        ps[5].grad = torch.full_like(ps[5], 1e-3)
    a.step(); b.step(); same()
    assert a.layout_refreezes == 2
    a.unfreeze_layout()
    assert [a.state[p]["step"] for p in ps_a] == [b.state[p]["step"] for p in ps_b]
    a.step(); b.step(); same()
    # one parameter stepped on its own while a layout is recorded and its step counts lag
    a.step(); b.step(); same()
    assert a._frozen is not None
    a.step(); b.step(); same()
    assert a._frozen["pending"] >= 1
    for opt, ps in ((a, ps_a), (b, ps_b)):
        opt.step_param(ps[2])
        opt.step()
    same()
    assert [a.state[p]["step"] for p in ps_a] == [b.state[p]["step"] for p in ps_b]


@pytest.mark.parametrize("shape", [(37, 24), (4, 3, 10), (129,)])
def test_reference_noise_mode_with_centralization_is_bit_identical_to_the_reference_step(shape):
    """noise_source="reference" takes the row means with torch's own mean, as adamw.py:179-184 does, so the
    whole step equals the reference's op sequence bit for bit (its own randint noise included)."""
    ps, grads = _make_params([shape], 8100)
    p = ps[0]
    ref_p = p.detach().clone()
    ref_m, ref_v = torch.zeros_like(ref_p), torch.zeros_like(ref_p)
    opt = ramtorch_amd.AdamW([p], storage_device="cuda", centralization=0.5, noise_source="reference", **HP0)
    for step in (1, 2):
        p.grad = (grads[0].float() * (1.0 + 0.3 * step)).bfloat16()
        opt.step()
        torch.cuda.synchronize()
        torch_ops.reference_step_ops(ref_p, p.grad, ref_m, ref_v, step=step, noise=None, centralization=0.5, **HP0)
        assert nmis(p.detach(), ref_p) == 0, f"step {step}"
        assert nmis(opt.state[p]["ema"], ref_m) == 0 and nmis(opt.state[p]["ema_squared"], ref_v) == 0
