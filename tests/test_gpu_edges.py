"""The update kernels at the edges of their work split: arrays that begin at any element, lengths around
units, pieces and rows.  Everything bit for bit against the oracle, and nothing outside the arrays may change.
Needs an MI355X: run with ``-m gpu``.
"""
import numpy as np
import pytest
import torch

import oracle
from ramtorch_amd import _native as N
from ramtorch_amd import functional as F

pytestmark = pytest.mark.gpu

HP0 = dict(lr=1e-4, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01)
_TORCH = {oracle.DT_BF16: torch.bfloat16, oracle.DT_F16: torch.float16, oracle.DT_F32: torch.float32,
          oracle.DT_F64: torch.float64}
_GUARD = 37   # elements of 0xA5 bytes on either side of every array


@pytest.fixture(scope="module")
def handle():
    assert torch.cuda.is_available(), "these tests need the GPU"
    h = N.Handle(0)
    yield h
    torch.cuda.synchronize()
    h.close()


def bits(t):
    t = t.detach().cpu().contiguous()
    return t.view({2: torch.int16, 4: torch.int32, 8: torch.int64}[t.element_size()]).numpy().ravel()


def guarded(a, code, shift):
    """``a`` on the GPU, ``shift`` elements past a 512-byte boundary, between guard bytes."""
    dt = _TORCH[code]
    values = torch.from_numpy((a.view(np.int16) if a.dtype == np.uint16 else a).copy())
    values = values.view(dt) if values.dtype == torch.int16 else values
    whole = torch.empty(256 + shift + a.size + _GUARD, dtype=dt, device="cuda")
    whole.view(torch.uint8).fill_(0xA5)
    view = whole[256 + shift:256 + shift + a.size]
    view.copy_(values)
    return view, whole


def check_guards(whole, shift, n):
    b = whole.view(torch.uint8)
    es = whole.element_size()
    assert bool((b[:(256 + shift) * es] == 0xA5).all()) and bool((b[(256 + shift + n) * es:] == 0xA5).all())


_MIX = {"bf16": (0, 0, 0, 0), "f16": (2, 2, 2, 2), "bf16_f32grad_f32v": (0, 1, 0, 1), "f32_bf16states": (1, 1, 0, 0),
        "f64states": (0, 0, 3, 3)}


@pytest.mark.parametrize("mix", list(_MIX))
@pytest.mark.parametrize("shifts", [(0, 1, 0, 0), (3, 7, 5, 1), (4, 4, 4, 4)])
def test_arrays_may_begin_at_any_element(handle, mix, shifts):
    """Views of a bucket or of a flat buffer: p, g, m and v each begin at an element of their own.  Lengths
    around one and several units of 8192 elements, around pieces of 512 and vectors of 8."""
    codes = _MIX[mix]
    lengths = [1, 7, 8, 9, 511, 513, 2048, 8191, 8192, 8193, 3 * 8192 + 515]
    tensors = []
    for k, n in enumerate(lengths):
        arrays = oracle.synth_inputs(n, 50 + k)
        as_code = [a if c == 0 else oracle.bf16_to_f32(a).astype(
            {1: np.float32, 2: np.float16, 3: np.float64}[c]) for a, c in zip(arrays, codes)]
        as_code = [a.view(np.uint16) if a.dtype == np.float16 else a for a in as_code]
        tensors.append((n, as_code, [guarded(a, c, s) for a, c, s in zip(as_code, codes, shifts)]))
    entries = [F.Entry(p=v[0][0], g=v[1][0], m=v[2][0], v=v[3][0], step=10, scalars_idx=0, tensor_id=k)
               for k, (_, _, v) in enumerate(tensors)]
    F.step_resident(handle, entries, [F.make_scalars(step=10, **HP0)], seed=77, explicit_noise=False)
    torch.cuda.synchronize()
    sc = oracle.scalars_from_hparams(step=10, **HP0)
    for k, (n, a, views) in enumerate(tensors):
        po, mo, vo = a[0].copy(), a[2].copy(), a[3].copy()
        oracle.step_tensor(po, a[1], mo, vo, sc, p_dtype=codes[0], g_dtype=codes[1], m_dtype=codes[2], v_dtype=codes[3],
                           seed=77, step=10, tensor_id=k)
        for name, got, want in zip("pmv", (views[0], views[2], views[3]), (po, mo, vo)):
            w = want.view({2: np.int16, 4: np.int32, 8: np.int64}[want.dtype.itemsize])
            np.testing.assert_array_equal(bits(got[0]), w, err_msg=f"{mix} n={n} {name}")
        for (view, whole), s in zip(views, shifts):
            check_guards(whole, s, n)


@pytest.mark.parametrize("rows,row_len", [(1, 8), (3, 9), (1, 511), (64, 27), (2, 4097), (3, 2731), (9, 1820), (17, 482), (1, 33000)])
def test_centralized_leftovers_take_their_means_in_pieces(handle, rows, row_len):
    """Centralization with row means given, in tensors whose rows end anywhere inside a vector, a piece or a unit
    (bf16, Philox noise: whole units and pieces of 512 both take the centralizing instance)."""
    n = rows * row_len
    p, g, m, v = oracle.synth_inputs(n, 300 + row_len)
    (P, wp), (G, _), (M, wm), (V, wv) = (guarded(a, 0, s) for a, s in zip((p, g, m, v), (0, 1, 0, 0)))
    means = F.row_means(handle, G, rows, row_len)
    e = F.Entry(p=P, g=G, m=M, v=V, step=4, scalars_idx=0, tensor_id=5, row_mean=means, row_len=row_len)
    F.step_resident(handle, [e], [F.make_scalars(step=4, centralization=0.75, **HP0)], seed=3, explicit_noise=False)
    torch.cuda.synchronize()
    np.testing.assert_allclose(means.cpu().numpy(), oracle.row_means(g, rows, row_len), rtol=3e-6, atol=1e-9)
    term = means.cpu().numpy() * np.float32(0.75)
    g32 = (oracle.bf16_to_f32(g).reshape(rows, row_len) - term[:, None]).astype(np.float32).ravel()
    po, mo, vo = p.copy(), m.copy(), v.copy()
    oracle.step_tensor(po, g32, mo, vo, oracle.scalars_from_hparams(step=4, **HP0), g_dtype=oracle.DT_F32, seed=3, step=4, tensor_id=5)
    for got, want in ((P, po), (M, mo), (V, vo)):
        np.testing.assert_array_equal(bits(got), want.view(np.int16))
    for whole in (wp, wm, wv):
        check_guards(whole, 0, n)


def test_scalar_sets_reach_the_kernels_as_arguments_or_through_the_table(handle):
    """One set, as many as travel as kernel arguments, and more, in turn over the same tensors (whole units and
    pieces): the table images have equal lists, and a change of way must not leave one set behind."""
    lens = [8192, 513, 3 * 8192 + 7, 64, 9, 16384]
    cpu = [list(oracle.synth_inputs(n, 600 + k)) for k, n in enumerate(lens)]
    dev = [[torch.from_numpy(a.view(np.int16).copy()).view(torch.bfloat16).cuda() for a in arrays] for arrays in cpu]
    for round_, n_sets in enumerate((1, 1, 4, 5, 5, 6, 4, 2, 3, 5, 1)):
        steps = [100 * (round_ + 1) + k % n_sets for k in range(len(lens))]
        scalars = [F.make_scalars(step=100 * (round_ + 1) + j, **HP0) for j in range(n_sets)]
        F.step_resident(handle, [F.Entry(p=d[0], g=d[1], m=d[2], v=d[3], step=steps[k], scalars_idx=k % n_sets, tensor_id=k)
                                 for k, d in enumerate(dev)], scalars, seed=9, explicit_noise=False)
        for k, a in enumerate(cpu):
            oracle.step_tensor(a[0], a[1], a[2], a[3], oracle.scalars_from_hparams(step=steps[k], **HP0), seed=9,
                               step=steps[k], tensor_id=k)
        for k, (d, a) in enumerate(zip(dev, cpu)):
            for name, got, want in zip("pmv", (d[0], d[2], d[3]), (a[0], a[2], a[3])):
                np.testing.assert_array_equal(bits(got), want.view(np.int16), err_msg=f"round {round_}, {n_sets} sets, tensor {k} {name}")


@pytest.mark.parametrize("mix", ["bf16_f32grad_f32v", "f32_bf16states"])
@pytest.mark.parametrize("rows,row_len", [(2049, 8), (1111, 9), (700, 27), (40, 250), (9, 2731), (3, 8193), (2, 40000)])
def test_centralized_fp32_layouts_take_their_means_in_units(handle, mix, rows, row_len):
    """The layouts with an fp32 array: four elements of a lane in two rows, rows shorter and longer than a half block
    (256), a block (512) and a unit (8192), loss scale and clip on gradient and mean."""
    codes = _MIX[mix]
    n = rows * row_len
    raw = oracle.synth_inputs(n, 700 + row_len)
    arrays = [a if c == 0 else oracle.bf16_to_f32(a) for a, c in zip(raw, codes)]
    (P, wp), (G, _), (M, wm), (V, wv) = (guarded(a, c, s) for a, c, s in zip(arrays, codes, (1, 0, 0, 3)))
    means = F.row_means(handle, G, rows, row_len, 0.5)
    e = F.Entry(p=P, g=G, m=M, v=V, step=4, scalars_idx=0, tensor_id=5, row_mean=means, row_len=row_len)
    clip = torch.tensor([0.75], device="cuda")
    F.step_resident(handle, [e], [F.make_scalars(step=4, centralization=0.75, inv_loss_scale=0.5, **HP0)], seed=3,
                    explicit_noise=False, clip_coef=clip)
    torch.cuda.synchronize()
    # each product and the difference round as in the kernel
    g32 = arrays[1] if codes[1] else oracle.bf16_to_f32(arrays[1])
    g32 = (g32 * np.float32(0.5)) * np.float32(0.75)
    term = (means.cpu().numpy() * np.float32(0.75)) * np.float32(0.75)
    g32 = (g32.reshape(rows, row_len) - term[:, None]).astype(np.float32).ravel()
    po, mo, vo = arrays[0].copy(), arrays[2].copy(), arrays[3].copy()
    oracle.step_tensor(po, g32, mo, vo, oracle.scalars_from_hparams(step=4, **HP0), p_dtype=codes[0], g_dtype=oracle.DT_F32,
                       m_dtype=codes[2], v_dtype=codes[3], seed=3, step=4, tensor_id=5)
    for got, want in ((P, po), (M, mo), (V, vo)):
        np.testing.assert_array_equal(bits(got), want.view({2: np.int16, 4: np.int32}[want.dtype.itemsize]))
    for whole, s in ((wp, 1), (wm, 0), (wv, 3)):
        check_guards(whole, s, n)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 129, 4097])
def test_norm_pass_finds_every_gradient(handle, n):
    """Tables of one, two and three search steps, with gradients that have no whole chunk of 8192 elements, no
    remainder, neither (empty) or both, at either end too.  Each gradient's values lie in a range of its own, so
    that a chunk looked up in the wrong gradient shows; fp32 sums of at most 32 squares a lane: 32 * 2^-24 at most."""
    rng = np.random.default_rng(n)
    sizes = [(8192, 5, 0, 8193, 8192 * 2, 1, 700)[k] for k in rng.integers(0, 7, n)]
    total = sum(sizes)
    flat = torch.randn(total, generator=torch.Generator().manual_seed(n))
    scale = torch.from_numpy(np.repeat(10.0 ** rng.uniform(-3, 0, n), sizes)).float()
    flat = (flat * scale).cuda()
    pick = [torch.float32, torch.bfloat16, torch.float16]
    grads, at = [], 0
    for k, s in enumerate(sizes):
        g = flat[at:at + s].to(pick[k % 3])
        grads.append(g)
        at += s
    want = float(torch.cat([g.float() for g in grads]).double().square().sum()) ** 0.5
    out = F.grad_norm(handle, grads, inv_loss_scale=1.0, max_norm=1.0)
    assert float(out[0]) == pytest.approx(want, rel=32 * 2 ** -24)


@pytest.mark.parametrize("sizes", [(100_000_003, 70_000_000, 8192 * 3 + 5, 30_000_001),   # the cut inside the second
                                   (134_217_728, 8192, 4097), (134_225_920, 20_000, 9)])   # at the first one's end, and one chunk before it
def test_norm_pass_over_more_than_stays_in_the_cache(handle, sizes):
    """Gradients on both sides of the 512 MiB that are loaded to stay, fp32 and 16 bit: each chunk counts once, whichever
    loop takes it.  fp32 sums of at most 32 squares a lane and chunk, in fp64 from chunk to chunk."""
    gen, want, grads = torch.Generator(device="cuda").manual_seed(sizes[1]), 0.0, []
    for k, n in enumerate(sizes):
        g = torch.empty(n, dtype=[torch.float32, torch.bfloat16, torch.float16, torch.float32][k], device="cuda")
        g.normal_(0, 10.0 ** -k, generator=gen)
        grads.append(g)
        want += sum(float(x.double().square().sum()) for x in g.split(1 << 24))
    for _ in range(2):
        out = F.grad_norm(handle, grads, inv_loss_scale=1.0, max_norm=1.0)
        assert float(out[0]) == pytest.approx(want ** 0.5, rel=32 * 2 ** -24)


def test_row_means_over_more_than_stays_in_the_cache(handle):
    """Rows on both sides of the 512 MiB that are loaded to stay, of a wavefront and of a workgroup, many gradients in
    one launch and one on its own.  A lane adds at most row / 64 elements and the lanes' sums in six steps more."""
    gen, jobs = torch.Generator(device="cuda").manual_seed(2), []
    for k, (rows, row, dt) in enumerate([(2001, 33_000, torch.bfloat16), (50_000, 4096, torch.bfloat16), (3, 40_001, torch.float16),
                                         (9000, 4097, torch.float32), (1111, 77, torch.float16), (3000, 33_001, torch.bfloat16)]):
        g = torch.empty(rows, row, dtype=dt, device="cuda").normal_(0, 1, generator=gen)
        jobs.append((F.Entry(p=None, g=g, m=None, v=None, step=1, scalars_idx=0, tensor_id=k), rows, row))
    F.row_means_multi(handle, jobs, 0.5)
    assert sum(e.g.numel() * e.g.element_size() for e, *_ in jobs) > 640 << 20
    single = torch.empty(70_001, 4096, dtype=torch.bfloat16, device="cuda").normal_(0, 1, generator=gen)
    checks = [(e.g, e.row_mean, row) for e, rows, row in jobs]
    checks += [(single, F.row_means(handle, single, 70_001, 4096, 0.5), 4096)]
    long = single.view(-1)[:8000 * 35_001].view(8000, 35_001)
    checks += [(long, F.row_means(handle, long, 8000, 35_001, 0.5), 35_001)]
    for g, mean, row in checks:
        for lo in range(0, len(g), 1024):
            x = g[lo:lo + 1024].double() * 0.5
            bound = (row / 64 + 8) * 2 ** -24 * x.abs().mean(1)
            assert bool(((mean[lo:lo + 1024].double() - x.mean(1)).abs() <= bound).all()), (row, lo)


@pytest.mark.parametrize("mix", ["bf16", "f16", "f16_bf16states"])
@pytest.mark.parametrize("shifts", [(0, 1, 0, 0), (3, 7, 5, 1), (4, 4, 4, 4)])
def test_rows_summed_inside_the_update_may_begin_at_any_element(handle, mix, shifts):
    """The row-wise kernel on views that begin at an element of their own, both instances (rows of up to 4096 elements
    and longer ones) and the limits of its row lengths: the bits of the same update with row means given, over arrays that
    begin at a 512-byte boundary, and nothing outside the arrays changes."""
    codes = {**_MIX, "f16_bf16states": (2, 2, 0, 0)}[mix]
    entries, reference, wholes = [], [], []
    for k, (rows, row) in enumerate([(5, 512), (9, 520), (3, 4096), (6, 4104), (2, 14336), (1, 32768)]):
        n = rows * row
        arrays = oracle.synth_inputs(n, 600 + k)
        arrays = [a if c == 0 else oracle.bf16_to_f32(a).astype(np.float16).view(np.uint16) for a, c in zip(arrays, codes)]
        views = [guarded(a, c, s) for a, c, s in zip(arrays, codes, shifts)]
        plain = [guarded(a, c, 0)[0] for a, c in zip(arrays, codes)]
        wholes += [(w, s, n) for (_, w), s in zip(views, shifts)]
        e = F.Entry(p=views[0][0], g=views[1][0], m=views[2][0], v=views[3][0], step=10, scalars_idx=0, tensor_id=k)
        assert F.rowwise_ok(e, row)
        e.row_len = row
        entries.append(e)
        reference.append(F.Entry(p=plain[0], g=plain[1], m=plain[2], v=plain[3], step=10, scalars_idx=0, tensor_id=k,
                                 row_mean=F.row_means(handle, plain[1], rows, row), row_len=row))
    for lst in (entries, reference):
        F.step_resident(handle, lst, [F.make_scalars(step=10, centralization=0.7, **HP0)], seed=77, explicit_noise=False)
    torch.cuda.synchronize()
    for e, r in zip(entries, reference):
        for name in "pgmv":
            np.testing.assert_array_equal(bits(getattr(e, name)), bits(getattr(r, name)), err_msg=f"rows of {e.row_len} {name}")
    for whole, s, n in wholes:
        check_guards(whole, s, n)
