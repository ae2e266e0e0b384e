"""GPU parity of the chunked tied-head cross-entropy (chunked_lm_loss.py:5-84).

The HIP cross-entropy rows (``mogt_lm_ce_fwd`` / ``mogt_lm_ce_bwd`` through
``mogt_amd.ops``) against the float64 oracle (oracle/lm_loss_oracle.py) on the
same logits, including unaligned rows (strided views), odd vocabularies,
ignored (-100) and out-of-range labels; then chunked_linear_cross_entropy end to
end (loss and both gradients) against the float64 chunked oracle, and the
model's chunked loss paths (model_mogt.py:326-380) against its unchunked loss.
Bars: the rows compute in fp32 from exactly representable inputs, <= 1e-5
normwise; the end-to-end path adds fp32 GEMMs, <= 1e-4; bf16 hidden states
(gradient returned in bf16) <= 2e-2."""
import numpy as np
import pytest
import torch

from conftest import announce, rel_err, to_np
from oracle import lm_loss_oracle as lo

pytestmark = pytest.mark.gpu

ROW_TOL = 1e-5
E2E_TOL = 1e-4
BF16_TOL = 2e-2


def _logits(rows, vocab, dtype, gpu, seed, pad=0):
    g = torch.Generator().manual_seed(seed)
    full = torch.randn(rows, vocab + pad, generator=g) * 4.0
    x = full.to(gpu).to(dtype)
    return x[:, pad // 2: pad // 2 + vocab] if pad else x


def _labels(rows, vocab, gpu, seed, ignore_every=0):
    g = torch.Generator().manual_seed(seed + 1)
    lab = torch.randint(0, vocab, (rows,), generator=g)
    if ignore_every:
        lab[::ignore_every] = -100
    return lab.to(gpu)


CASES = [(1, 1, torch.float32, 0), (3, 7, torch.float32, 0), (64, 129, torch.float32, 3),
         (257, 32000, torch.float32, 0), (33, 50257, torch.float32, 2), (40, 50257, torch.bfloat16, 5),
         (100, 32000, torch.bfloat16, 0), (5, 4095, torch.bfloat16, 3)]


@pytest.mark.parametrize("rows,vocab,dtype,pad", CASES)
def test_ce_rows_forward(gpu, rows, vocab, dtype, pad):
    announce(f"ce rows fwd rows={rows} vocab={vocab} {dtype} pad={pad}")
    from mogt_amd import ops

    x = _logits(rows, vocab, dtype, gpu, seed=rows + vocab, pad=pad)
    lab = _labels(rows, vocab, gpu, seed=rows, ignore_every=4 if rows > 4 else 0)
    loss, lse = ops.lm_ce_forward(x, lab)
    torch.cuda.synchronize()
    ref_loss, ref_lse = lo.ce_rows(to_np(x), lab.cpu().numpy())
    assert loss.dtype == torch.float32 and lse.shape == (rows,)
    assert rel_err(to_np(lse), ref_lse) <= ROW_TOL
    assert rel_err(to_np(loss), ref_loss) <= ROW_TOL
    assert float(loss[lab == -100].abs().sum()) == 0.0


@pytest.mark.parametrize("rows,vocab,dtype,pad", CASES)
def test_ce_rows_backward_in_place(gpu, rows, vocab, dtype, pad):
    announce(f"ce rows bwd rows={rows} vocab={vocab} {dtype} pad={pad}")
    from mogt_amd import ops

    x = _logits(rows, vocab, dtype, gpu, seed=rows * 3 + vocab, pad=pad)
    lab = _labels(rows, vocab, gpu, seed=rows + 7, ignore_every=3 if rows > 3 else 0)
    x_np = to_np(x)
    _, lse = ops.lm_ce_forward(x, lab)
    scale = torch.tensor([0.37], device=gpu)
    out = ops.lm_ce_backward_(x, lab, lse, scale)
    torch.cuda.synchronize()
    assert out.data_ptr() == x.data_ptr()
    ref = lo.ce_rows_grad(x_np, lab.cpu().numpy(), 0.37)
    tol = ROW_TOL if dtype == torch.float32 else 4e-3   # the gradient itself is stored in bf16
    assert rel_err(to_np(x), ref) <= tol
    assert float(x[lab == -100].float().abs().sum()) == 0.0


def test_ce_rows_bad_label_is_nan(gpu):
    from mogt_amd import ops

    x = _logits(4, 50, torch.float32, gpu, seed=1)
    lab = torch.tensor([3, 50, -1, -100], device=gpu)
    loss, lse = ops.lm_ce_forward(x, lab)
    ops.lm_ce_backward_(x, lab, lse, torch.ones(1, device=gpu))
    torch.cuda.synchronize()
    l = loss.cpu()
    assert torch.isfinite(l[0]) and torch.isnan(l[1]) and torch.isnan(l[2]) and l[3] == 0
    assert torch.isnan(x[1]).all() and torch.isnan(x[2]).all() and (x[3] == 0).all()
    assert torch.isfinite(x[0]).all()


def test_ce_rows_argument_errors(gpu):
    from mogt_amd import ops

    x = torch.zeros(4, 10, device=gpu)
    with pytest.raises(ValueError):
        ops.lm_ce_forward(x, torch.zeros(4, dtype=torch.int32, device=gpu))
    with pytest.raises(ValueError):
        ops.lm_ce_forward(x.t(), torch.zeros(10, dtype=torch.int64, device=gpu))
    with pytest.raises(ValueError):
        ops.lm_ce_backward_(x, torch.zeros(4, dtype=torch.int64, device=gpu), torch.zeros(4, device=gpu),
                            torch.ones(2, device=gpu))


@pytest.mark.parametrize("chunk", [1, 64, 333, 10000])
def test_chunked_linear_ce_matches_oracle(gpu, chunk):
    announce(f"chunked linear CE chunk={chunk}")
    from mogt_amd.chunked_lm_loss import chunked_linear_cross_entropy

    g = torch.Generator().manual_seed(chunk)
    B, L, D, V = 2, 300, 64, 1000
    h = torch.randn(B, L, D, generator=g)
    w = torch.randn(V, D, generator=g) * 0.3
    lab = torch.randint(0, V, (B, L), generator=g)
    lab[1, ::17] = -100
    ht = h.to(gpu).requires_grad_()
    wt = w.to(gpu).requires_grad_()
    loss = chunked_linear_cross_entropy(ht, wt, lab.to(gpu), chunk_size=chunk)
    (loss * 2.5).backward()
    torch.cuda.synchronize()
    ref_loss, ref_gh, ref_gw = lo.chunked_linear_ce(h.numpy(), w.numpy(), lab.numpy(), chunk, grad_output=2.5)
    assert abs(float(loss.detach()) - ref_loss) <= E2E_TOL * abs(ref_loss)
    assert rel_err(to_np(ht.grad), ref_gh) <= E2E_TOL
    assert rel_err(to_np(wt.grad), ref_gw) <= E2E_TOL


def test_chunked_linear_ce_bf16_hidden(gpu):
    announce("chunked linear CE bf16 hidden")
    from mogt_amd.chunked_lm_loss import chunked_linear_cross_entropy

    g = torch.Generator().manual_seed(5)
    B, L, D, V = 1, 512, 128, 4096
    h = torch.randn(B, L, D, generator=g).bfloat16()
    w = torch.randn(V, D, generator=g) * 0.1
    lab = torch.randint(0, V, (B, L), generator=g)
    ht = h.to(gpu).requires_grad_()
    wt = w.to(gpu).requires_grad_()
    loss = chunked_linear_cross_entropy(ht, wt, lab.to(gpu), chunk_size=200)
    loss.backward()
    torch.cuda.synchronize()
    ref_loss, ref_gh, ref_gw = lo.chunked_linear_ce(h.float().numpy(), w.numpy(), lab.numpy(), 200)
    assert ht.grad.dtype == torch.bfloat16 and wt.grad.dtype == torch.float32
    assert abs(float(loss.detach()) - ref_loss) <= E2E_TOL * abs(ref_loss)
    assert rel_err(to_np(ht.grad), ref_gh) <= BF16_TOL
    assert rel_err(to_np(wt.grad), ref_gw) <= E2E_TOL


def test_chunked_linear_ce_validation(gpu):
    from mogt_amd.chunked_lm_loss import chunked_linear_cross_entropy

    h = torch.zeros(1, 4, 8, device=gpu)
    w = torch.zeros(10, 8, device=gpu)
    lab = torch.zeros(1, 4, dtype=torch.int64, device=gpu)
    for args, msg in [((h[0], w, lab[0]), "hidden_states"), ((h, w, lab[:, :3]), "labels"),
                      ((h, w[:, :7], lab), "weight")]:
        with pytest.raises(ValueError, match=msg):
            chunked_linear_cross_entropy(*args, chunk_size=2)
    with pytest.raises(ValueError, match="chunk_size"):
        chunked_linear_cross_entropy(h, w, lab, chunk_size=0)


def test_model_chunked_loss_paths(gpu):
    """MOGTForCausalLM.forward (model_mogt.py:350-380): unchunked loss, chunked
    loss with logits, chunked linear CE without logits -- same loss, and the
    linear-CE path's gradients equal the unchunked ones."""
    announce("model chunked loss paths")
    from mogt_amd.model_mogt import MOGTForCausalLM

    torch.manual_seed(3)
    model = MOGTForCausalLM(vocab_size=257, d_model=64, num_layers=1, r=16).to(gpu)
    ids = torch.randint(0, 257, (1, 200), device=gpu)
    labels = torch.randint(0, 257, (1, 200), device=gpu)
    _, l0 = model(ids, labels=labels)
    l0.backward()
    g0 = {k: p.grad.clone() for k, p in model.named_parameters() if p.grad is not None}
    model.zero_grad()
    logits1, l1 = model(ids, labels=labels, loss_chunk_size=64)
    model.zero_grad()
    logits2, l2 = model(ids, labels=labels, return_logits=False, loss_chunk_size=64)
    l2.backward()
    torch.cuda.synchronize()
    assert logits1.shape == (1, 200, 257) and logits2 is None
    l0, l1, l2 = (float(v.detach()) for v in (l0, l1, l2))
    assert abs(l1 - l0) <= 1e-5 * abs(l0)
    assert abs(l2 - l0) <= 1e-5 * abs(l0)
    for k, p in model.named_parameters():
        if k in g0:
            assert rel_err(to_np(p.grad), to_np(g0[k])) <= E2E_TOL, k


def _bf16_or_f32(shape, dtype, seed, std=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std).to(dtype)


def _pieces_of(x):
    from mogt_amd import ops

    return x.unsqueeze(0).contiguous() if x.dtype == torch.bfloat16 else ops.split_pieces(x)


def test_split_pieces_sum_is_exact(gpu):
    """x1 + x2 + x3 == x for every exponent that leaves the last piece normal,
    zero padding, strided rows; non-finite values and the largest floats whole
    in the first piece."""
    announce("split pieces")
    from mogt_amd import ops

    g = torch.Generator().manual_seed(3)
    x = torch.randn(37, 70, generator=g) * torch.exp2(torch.randint(-60, 60, (37, 70), generator=g).float())
    x[0, :6] = torch.tensor([0.0, -0.0, 3.4028235e38, -3.4028235e38, 1.0, 2.0 ** -30])
    p = ops.split_pieces(x.to(gpu)[:, 1:66])
    assert p.shape == (3, 37, 96) and float(p[:, :, 65:].float().abs().sum()) == 0.0
    assert torch.equal(p.double().sum(0)[:, :65].cpu(), x[:, 1:66].double())
    bad = torch.tensor([[float("inf"), float("-inf"), float("nan"), 1.0]], device=gpu)
    q = ops.split_pieces(bad).float().cpu()
    assert torch.equal(q[0, 0, :2], bad[0, :2].cpu()) and torch.isnan(q[0, 0, 2])
    assert float(q[1:, 0, :4].abs().sum()) == 0.0


SPLIT_DT = [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16),
            (torch.float32, torch.float32)]


@pytest.mark.parametrize("da,db", SPLIT_DT)
@pytest.mark.parametrize("M,N,K", [(1, 1, 32), (255, 257, 64), (256, 256, 96), (300, 129, 160), (513, 1001, 768)])
def test_split_gemm_logits_form(gpu, M, N, K, da, db):
    """One to 24 stages, ragged row and column tiles, every piece pair, and the
    accumulating output: within the elementwise bound (K + 8) 2^-24 sum |a b|
    that an fp32 sum of the products has in any order."""
    announce(f"split gemm nt {M} {N} {K} {da} {db}")
    from mogt_amd import ops

    a, b = _bf16_or_f32((M, K), da, 1).to(gpu), _bf16_or_f32((N, K), db, 2).to(gpu)
    out = torch.full((M, -(-N // 4) * 4), 7.0, device=gpu)[:, :N]
    ops.split_gemm_(out, _pieces_of(a), _pieces_of(b), K)
    ref = a.double() @ b.double().t()
    bound = (K + 8) * 2.0 ** -24 * (a.double().abs() @ b.double().abs().t())
    assert bool(((out.double() - ref).abs() <= bound).all())
    ops.split_gemm_(out, _pieces_of(a), _pieces_of(b), K, accumulate=True)
    assert bool(((out.double() - 2 * ref).abs() <= 3 * bound).all())


@pytest.mark.parametrize("db", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,V,D", [(1, 33, 32), (37, 1001, 64), (300, 4096, 96), (257, 10007, 256)])
def test_split_gemm_gradient_forms(gpu, n, V, D, db):
    """The hidden states' gradient (contraction over the vocabulary, ragged, the
    weight K-slow, K slices) and the weight's (both K-slow, contraction over
    the rows), odd sizes included (the last column of a K-slow row is a half
    dword); fp32 and bf16 outputs, run to run equal."""
    announce(f"split gemm gradients {n} {V} {D} {db}")
    from mogt_amd import ops

    g = _bf16_or_f32((n, V), torch.float32, 5).to(gpu)
    x = _bf16_or_f32((V, D), db, 6).to(gpu)
    gp = ops.split_pieces(g)
    dh = torch.empty(n, D, device=gpu)
    ops.split_gemm_(dh, gp, _pieces_of(x), V, k_slow_b=True)
    ref = g.double() @ x.double()
    bound = (V + 8) * 2.0 ** -24 * (g.double().abs() @ x.double().abs())
    assert bool(((dh.double() - ref).abs() <= bound).all())
    half = torch.empty(n, D, device=gpu, dtype=torch.bfloat16)
    ops.split_gemm_(half, gp, _pieces_of(x), V, k_slow_b=True)
    assert torch.equal(half, dh.to(torch.bfloat16))
    h = _bf16_or_f32((n, D), db, 7).to(gpu)
    dw = torch.zeros(V, D, device=gpu)
    ops.split_gemm_(dw, gp, _pieces_of(h), n, k_slow_a=True, k_slow_b=True, accumulate=True)
    ref = g.double().t() @ h.double()
    bound = (n + 8) * 2.0 ** -24 * (g.double().abs().t() @ h.double().abs())
    assert bool(((dw.double() - ref).abs() <= bound).all())
    again = torch.empty(V, D, device=gpu)
    ops.split_gemm_(again, gp, _pieces_of(h), n, k_slow_a=True, k_slow_b=True)
    assert torch.equal(again, dw)


@pytest.mark.parametrize("rows,vocab,dtype,pad", [(3, 7, torch.float32, 0), (64, 129, torch.float32, 3),
                                                  (40, 50257, torch.bfloat16, 5), (33, 4000, torch.bfloat16, 0)])
def test_ce_gradient_pieces_equal_the_block(gpu, rows, vocab, dtype, pad):
    """The pieces sum to lm_ce_grad's fp32 block bit for bit, padding zero."""
    announce(f"ce gradient pieces {rows} {vocab} {dtype} {pad}")
    from mogt_amd import ops

    x = _logits(rows, vocab, dtype, gpu, seed=vocab, pad=pad)
    lab = _labels(rows, vocab, gpu, seed=rows, ignore_every=5)
    _, lse = ops.lm_ce_forward(x, lab)
    scale = torch.tensor([0.37], device=gpu)
    g = ops.lm_ce_grad(x, lab, lse, scale)
    p = ops.lm_ce_grad_pieces(x, lab, lse, scale)
    total = p.double().sum(0)
    # below 2^-110 the last piece leaves bf16's normal range
    assert bool(((total[:, :vocab] - g.double()).abs() <= 2.0 ** -133).all())
    assert float(p[:, :, vocab:].float().abs().sum()) == 0.0


@pytest.mark.parametrize("hd,wd,autocast", [(torch.float32, torch.float32, False), (torch.bfloat16, torch.float32, False),
                                            (torch.float32, torch.bfloat16, False), (torch.float32, torch.float32, True)])
def test_chunked_linear_ce_split_form_matches_library_form(gpu, monkeypatch, hd, wd, autocast):
    """Loss and gradients of the split form against the library form of the same
    call: ragged last chunk, odd vocabulary, ignored labels."""
    announce(f"chunked CE split form {hd} {wd} {autocast}")
    from mogt_amd import chunked_lm_loss as cl

    h = _bf16_or_f32((2, 150, 64), hd, 11).to(gpu).requires_grad_()
    w = _bf16_or_f32((1003, 64), wd, 12, 0.3).to(gpu).requires_grad_()
    lab = _labels(300, 1003, gpu, seed=13, ignore_every=7).view(2, 150)

    def call():
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            loss = cl.chunked_linear_cross_entropy(h, w, lab, chunk_size=128)
        return [loss.detach(), *torch.autograd.grad(loss, [h, w])]

    lib = call()
    monkeypatch.setattr(cl, "SPLIT_MIN_MACS", 0)
    monkeypatch.setattr(cl, "SPLIT_MIN_MACS_AUTOCAST", 0)
    for got, ref, what in zip(call(), lib, ("loss", "dh", "dw")):
        assert got.dtype == ref.dtype and got.shape == ref.shape
        # both fp32 sums in other orders; bf16 gradients one rounding apart
        assert rel_err(to_np(got), to_np(ref)) <= (1e-5 if got.dtype == torch.float32 else 2.0 ** -8), what


@pytest.mark.parametrize("da,db", SPLIT_DT)
@pytest.mark.parametrize("M,V,K", [(1, 3, 32), (5, 129, 64), (257, 1000, 96), (300, 513, 32), (64, 4099, 160)])
def test_split_ce_epilogues_match_the_row_kernels(gpu, da, db, M, V, K):
    """The cross-entropy epilogues against the row kernels on the same product's
    written logits: ragged row and column tiles, a label in every column group
    and at the edges, ignored and bad labels, a row of equal logits and a row of
    NaN."""
    announce(f"split ce {M} {V} {K} {da} {db}")
    from mogt_amd import ops

    a, b = _bf16_or_f32((M, K), da, 21), _bf16_or_f32((V, K), db, 22)
    a[0] = 0.0
    if M > 4:
        a[3, 0] = float("nan")
    a, b = a.to(gpu), b.to(gpu)
    lab = torch.randint(0, V, (M,), generator=torch.Generator().manual_seed(M))
    lab[-1] = V - 1
    if M > 8:
        lab[1], lab[2], lab[4], lab[5], lab[6] = 0, -100, V, -7, V - 1
    lab = lab.to(gpu)
    ap, bp = _pieces_of(a), _pieces_of(b)
    logits = torch.empty(M, ops.split_pad(V), device=gpu)[:, :V]
    ops.split_gemm_(logits, ap, bp, K)
    loss, lse = ops.lm_ce_forward(logits, lab)
    loss2, lse2 = ops.split_ce_forward(ap, bp, K, lab)
    torch.cuda.synchronize()
    # fp32 sums of exponentials in another order: a few ulp of the log-sum-exp
    eps = 4 * 2.0 ** -23 * (1 + lse.abs().nan_to_num(0).max())
    assert torch.equal(torch.isnan(lse), torch.isnan(lse2)) and torch.equal(torch.isnan(loss), torch.isnan(loss2))
    assert bool(((lse - lse2).nan_to_num(0).abs() <= eps).all())
    assert bool(((loss - loss2).nan_to_num(0).abs() <= 2 * eps).all())
    scale = torch.tensor([0.37], device=gpu)
    g = ops.lm_ce_grad_pieces(logits, lab, lse, scale).double().sum(0)
    g2 = ops.split_ce_grad_pieces(ap, bp, K, lab, lse, scale)
    assert float(g2[:, :, V:].float().nan_to_num(1).abs().sum()) == 0.0
    g2 = g2.double().sum(0)
    assert torch.equal(torch.isnan(g), torch.isnan(g2))
    assert bool(((g - g2).nan_to_num(0).abs() <= 2.0 ** -22 * g.nan_to_num(0).abs() + 1e-37).all())


def test_chunked_linear_ce_fused_epilogue_end_to_end(gpu):
    """A head whose logits product fills the GPU (the epilogues are taken), with
    a ragged last chunk that takes the written logits: loss and gradients
    against the library form."""
    announce("chunked CE fused epilogues")
    from mogt_amd import chunked_lm_loss as cl
    from mogt_amd import ops

    N, D, V = 2100, 64, 33000
    assert ops.split_logits_slices(2048, V, D, 1, 3) == 1
    h = _bf16_or_f32((1, N, D), torch.bfloat16, 31).to(gpu).requires_grad_()
    w = _bf16_or_f32((V, D), torch.float32, 32, 0.1).to(gpu).requires_grad_()
    lab = _labels(N, V, gpu, seed=33, ignore_every=9).view(1, N)

    def call(min_macs):
        cl_min, cl.SPLIT_MIN_MACS = cl.SPLIT_MIN_MACS, min_macs
        try:
            loss = cl.chunked_linear_cross_entropy(h, w, lab, chunk_size=2048)
            return [loss.detach(), *torch.autograd.grad(loss, [h, w])]
        finally:
            cl.SPLIT_MIN_MACS = cl_min

    for got, ref in zip(call(0), call(1 << 62)):
        assert rel_err(to_np(got), to_np(ref)) <= (1e-5 if got.dtype == torch.float32 else 2.0 ** -8)


def _fp32_products(a, b):
    """sum_k a b as an fp32 sum of fp32 products has it (infinities, overflow)."""
    return (a.float().cpu()[:, None, :] * b.float().cpu()[None, :, :]).sum(-1)


def _same_specials(got, ref):
    got, ref = got.float().cpu(), ref.float().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.isposinf(got), torch.isposinf(ref)) and torch.equal(torch.isneginf(got), torch.isneginf(ref))


def _specials(a, b):
    """Infinities against pieces that are zero or of the other sign, and products
    past the largest float, in few rows of each operand."""
    inf = float("inf")
    a[0] = 1.0                                  # exact in one piece: its others are zero
    a[1, 0], a[2, 1] = inf, -inf
    b[1, 0], b[2, 3], b[3, 5] = -inf, inf, 0.0
    a[3, 7], b[4, 7], b[5, 7] = 1e30, 1e30, -1e30
    b[6, 0] = 0.0                               # 0 * inf


@pytest.mark.parametrize("da,db", SPLIT_DT)
@pytest.mark.parametrize("M,N,K", [(9, 8, 32), (300, 200, 96)])
def test_split_gemm_infinities_as_in_fp32(gpu, da, db, M, N, K):
    """Infinite and overflowing products come out as fp32 products give them, in
    every piece pair; elements without them within the fp32 bound."""
    announce(f"split gemm infinities {M} {N} {K} {da} {db}")
    from mogt_amd import ops

    a, b = _bf16_or_f32((M, K), da, 41), _bf16_or_f32((N, K), db, 42)
    _specials(a, b)
    a, b = a.to(gpu), b.to(gpu)
    out = torch.empty(M, -(-N // 4) * 4, device=gpu)[:, :N]
    ops.split_gemm_(out, _pieces_of(a), _pieces_of(b), K)
    ref = _fp32_products(a, b)
    _same_specials(out, ref)
    fin = torch.isfinite(ref)
    d64 = (a.double().cpu() @ b.double().cpu().t(), a.double().abs().cpu() @ b.double().abs().cpu().t())
    assert bool(((out.double().cpu() - d64[0]).abs() <= (K + 8) * 2.0 ** -24 * d64[1])[fin].all())


@pytest.mark.parametrize("db", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,V,D", [(37, 1001, 64), (300, 4096, 96)])
def test_split_gemm_gradient_infinities_as_in_fp32(gpu, n, V, D, db):
    announce(f"split gemm gradient infinities {n} {V} {D} {db}")
    from mogt_amd import ops

    g, x, h = _bf16_or_f32((n, V), torch.float32, 43), _bf16_or_f32((V, D), db, 44), _bf16_or_f32((n, D), db, 45)
    inf = float("inf")
    g[0, 0], g[1, 5], g[2, V - 1], g[3, 9] = 0.5, inf, -inf, 1e30   # 0.5: one piece
    x[0, 1], x[V - 1, 2], x[9, 3], x[5, 4] = inf, -inf, 1e30, 0.0
    h[0, 1], h[1, 4], h[3, 3] = -inf, 0.0, 1e30
    gp = ops.split_pieces(g.to(gpu))
    dh = torch.empty(n, D, device=gpu)
    ops.split_gemm_(dh, gp, _pieces_of(x.to(gpu)), V, k_slow_b=True)
    _same_specials(dh, torch.cat([_fp32_products(g[i:i + 8], x.t()) for i in range(0, n, 8)]))
    dw = torch.zeros(V, D, device=gpu)
    ops.split_gemm_(dw, gp, _pieces_of(h.to(gpu)), n, k_slow_a=True, k_slow_b=True, accumulate=True)
    _same_specials(dw, torch.cat([_fp32_products(g.t()[i:i + 64], h.t()) for i in range(0, V, 64)]))


@pytest.mark.parametrize("da,db", SPLIT_DT)
def test_split_ce_epilogues_of_infinite_logits(gpu, da, db):
    """Rows with -inf logits (masked vocabulary rows against a constant feature),
    +inf and NaN logits: the epilogues as the row kernels on the fp32 products."""
    announce(f"split ce infinities {da} {db}")
    from mogt_amd import ops

    M, V, K = 270, 515, 64
    a, b = _bf16_or_f32((M, K), da, 51), _bf16_or_f32((V, K), db, 52)
    a[:, 0] = 1.0
    b[5:400:7, 0] = float("-inf")
    a[260, 1], a[261, 1] = float("inf"), float("nan")
    b[0, 1] = 0.0
    a, b = a.to(gpu), b.to(gpu)
    lab = torch.randint(0, V, (M,), generator=torch.Generator().manual_seed(1)).to(gpu)
    lab[7], lab[8] = 5, 6
    logits = torch.cat([_fp32_products(a[i:i + 16], b) for i in range(0, M, 16)]).to(gpu)
    loss, lse = ops.lm_ce_forward(logits, lab)
    assert int(torch.isfinite(loss).sum()) > 200 and bool(torch.isinf(loss[7]))
    # two fp32 sums of K products, each within (K + 8) 2^-24 sum |a b| of the exact
    # logit: a probability changes by that relative amount
    size = torch.where(torch.isfinite(a), a, 0).abs().double() @ torch.where(torch.isfinite(b), b, 0).abs().double().t()
    tol = ROW_TOL + 2 * (K + 8) * 2.0 ** -24 * float(size.max())
    loss2, lse2 = ops.split_ce_forward(_pieces_of(a), _pieces_of(b), K, lab)
    _same_specials(loss2, loss)
    _same_specials(lse2, lse)
    fin = torch.isfinite(loss)
    assert rel_err(to_np(loss2[fin]), to_np(loss[fin])) <= tol
    scale = torch.tensor([0.37], device=gpu)
    g = ops.lm_ce_grad(logits, lab, lse, scale)
    g2 = ops.split_ce_grad_pieces(_pieces_of(a), _pieces_of(b), K, lab, lse, scale).float().sum(0)[:, :V]
    _same_specials(g2, g)
    fin = torch.isfinite(g)
    assert rel_err(to_np(g2[fin]), to_np(g[fin])) <= tol


@pytest.mark.parametrize("hd", [torch.float32, torch.bfloat16])
def test_chunked_linear_ce_masked_vocabulary(gpu, monkeypatch, hd):
    """Vocabulary rows masked by -inf against a constant hidden feature: the loss
    of the split form is finite as the library form's, the gradients alike."""
    announce(f"chunked CE masked vocabulary {hd}")
    from mogt_amd import chunked_lm_loss as cl

    h, w = _bf16_or_f32((1, 300, 64), hd, 61), _bf16_or_f32((1003, 64), torch.float32, 62, 0.3)
    h[..., 0] = 1.0
    w[10:20, 0] = float("-inf")
    h, w = h.to(gpu).requires_grad_(), w.to(gpu).requires_grad_()
    lab = torch.randint(20, 1003, (1, 300), generator=torch.Generator().manual_seed(5)).to(gpu)

    def call():
        loss = cl.chunked_linear_cross_entropy(h, w, lab, chunk_size=128)
        return [loss.detach(), *torch.autograd.grad(loss, [h, w])]

    lib = call()
    assert bool(torch.isfinite(lib[0])) and bool(torch.isfinite(lib[2]).all())
    monkeypatch.setattr(cl, "SPLIT_MIN_MACS", 0)
    for got, ref in zip(call(), lib):
        _same_specials(got, ref)
        fin = torch.isfinite(ref)
        assert rel_err(to_np(got[fin]), to_np(ref[fin])) <= (1e-5 if got.dtype == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("split", [False, True])
def test_chunked_linear_ce_second_derivative_is_refused(gpu, monkeypatch, split):
    """The gradients are not differentiable again: a second derivative raises
    instead of taking them as constants."""
    announce(f"chunked CE second derivative split={split}")
    from mogt_amd import chunked_lm_loss as cl

    monkeypatch.setattr(cl, "SPLIT_MIN_MACS", 0 if split else 1 << 62)
    h = torch.randn(1, 40, 32, device=gpu, requires_grad=True)
    w = torch.randn(65, 32, device=gpu, requires_grad=True)
    lab = torch.randint(0, 65, (1, 40), device=gpu)
    loss = cl.chunked_linear_cross_entropy(h, w, lab, chunk_size=32)
    gh, gw = torch.autograd.grad(loss, [h, w], create_graph=True)
    for penalty in (gh.square().sum(), gw.square().sum(), loss + gh.square().sum()):
        with pytest.raises(RuntimeError):
            torch.autograd.grad(penalty, [h, w], retain_graph=True)


@pytest.mark.parametrize("hd", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("autocast", [False, True])
def test_chunked_linear_ce_compiled(gpu, monkeypatch, hd, autocast):
    """The split form traced and functionalised into one graph gives the eager
    call's loss and gradients."""
    announce(f"chunked CE compiled {hd} {autocast}")
    from mogt_amd import chunked_lm_loss as cl

    monkeypatch.setattr(cl, "SPLIT_MIN_MACS", 0)
    monkeypatch.setattr(cl, "SPLIT_MIN_MACS_AUTOCAST", 0)
    h = _bf16_or_f32((2, 150, 64), hd, 81).to(gpu).requires_grad_()
    w = _bf16_or_f32((1003, 64), torch.float32, 82, 0.3).to(gpu).requires_grad_()
    lab = _labels(300, 1003, gpu, seed=83, ignore_every=7).view(2, 150)

    def loss(h, w, lab):
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            return cl.chunked_linear_cross_entropy(h, w, lab, chunk_size=128)

    def run(fn):
        value = fn(h, w, lab)
        return [value.detach(), *torch.autograd.grad(value, [h, w])]

    eager = run(loss)
    torch._dynamo.reset()
    for got, ref in zip(run(torch.compile(loss, backend="aot_eager", fullgraph=True)), eager):
        assert got.dtype == ref.dtype and torch.equal(got, ref)


@pytest.mark.parametrize("hd", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [129, 200])
def test_chunked_linear_ce_of_repeated_hidden_states(gpu, monkeypatch, n, hd):
    """Hidden states expanded from one row (row stride 0), with a last chunk of
    one row."""
    announce(f"chunked CE expanded hidden states n={n} {hd}")
    from mogt_amd import chunked_lm_loss as cl

    base = _bf16_or_f32((1, 1, 64), hd, 71).to(gpu)
    w = _bf16_or_f32((1003, 64), torch.float32, 72, 0.3).to(gpu).requires_grad_()
    lab = torch.randint(0, 1003, (1, n), generator=torch.Generator().manual_seed(n)).to(gpu)

    def call():
        loss = cl.chunked_linear_cross_entropy(base.expand(1, n, 64), w, lab, chunk_size=128)
        return [loss.detach(), *torch.autograd.grad(loss, [w])]

    lib = call()
    monkeypatch.setattr(cl, "SPLIT_MIN_MACS", 0)
    for got, ref in zip(call(), lib):
        assert rel_err(to_np(got), to_np(ref)) <= 1e-5


@pytest.mark.parametrize("which", ["hidden", "weight"])
def test_chunked_linear_ce_of_misaligned_bf16(gpu, monkeypatch, which):
    """bf16 operands that start at an odd element."""
    announce(f"chunked CE misaligned {which}")
    from mogt_amd import chunked_lm_loss as cl

    h, w = _bf16_or_f32((1, 200, 64), torch.bfloat16, 91).to(gpu), _bf16_or_f32((1003, 64), torch.bfloat16, 92, 0.3).to(gpu)
    lab = torch.randint(0, 1003, (1, 200), generator=torch.Generator().manual_seed(9)).to(gpu)

    def odd(x):
        return torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].view(x.shape)

    def call(h, w):
        h, w = h.detach().requires_grad_(), w.detach().requires_grad_()
        loss = cl.chunked_linear_cross_entropy(h, w, lab, chunk_size=128)
        return [loss.detach(), *torch.autograd.grad(loss, [h, w])]

    monkeypatch.setattr(cl, "SPLIT_MIN_MACS", 0)
    ref = call(h, w)
    for got, r in zip(call(odd(h) if which == "hidden" else h, odd(w) if which == "weight" else w), ref):
        assert torch.equal(got, r)
