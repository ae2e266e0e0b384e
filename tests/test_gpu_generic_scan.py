"""GPU parity of the generic affine scan (float64 state, ranks above 32, fp16 /
fp64 I/O, host tensors, autograd) through the drop-in ``affine_scan`` /
``triton_scan`` names, against the float64 oracle and the reference's own
sanity checks (sanity_affine_scan.py:19-61, :102-135).

Bars: float64 state, float64 output: max abs error <= 1e-10 (the reference's
own bar between its three scans) and normwise relative error <= 1e-12 against
the oracle; fp32 state: relative error <= 1e-4; bf16 output 2e-2; fp16 output
2e-3."""
import numpy as np
import pytest
import torch

from conftest import announce, rel_err
from mogt_amd import synthetic
from oracle import scan_oracle as so

pytestmark = pytest.mark.gpu

F64_TOL = 1e-12
FP32_TOL = 1e-4


def np64(t):
    return t.detach().double().cpu().numpy()


def _stable(B, L, R, C, seed, dtype=np.float64):
    """U = I + N(0, 0.3^2 / R) rescaled to spectral norm <= 1, V ~ N(0,1)."""
    g = synthetic.rng(seed)
    U = np.eye(R) + (0.3 / np.sqrt(R)) * g.standard_normal((B, L, R, R))
    U /= np.maximum(1.0, np.linalg.norm(U, ord=2, axis=(-2, -1)))[..., None, None]
    V = g.standard_normal((B, L, R, C))
    return U.astype(dtype), V.astype(dtype)


def _torch_seq(U, V, prefix):
    """H_t = U_t H_{t-1} + V_t as a torch loop on the host, so that
    torch.autograd derives its gradients (the reference's backward check,
    sanity_affine_scan.py:102-135)."""
    B, L, R, C = V.shape
    H = torch.zeros(B, R, C, dtype=U.dtype)
    P = torch.eye(R, dtype=U.dtype).expand(B, R, R)
    Hs, Ps = [], []
    for t in range(L):
        H = torch.bmm(U[:, t], H) + V[:, t]
        Hs.append(H)
        if prefix:
            P = torch.bmm(U[:, t], P)
            Ps.append(P)
    return (torch.stack(Ps, 1) if prefix else None), torch.stack(Hs, 1)


def test_reference_sanity_script_fp64_host_tensors(gpu):
    """run_affine_scan_sanity (sanity_affine_scan.py:19-61) as the reference
    writes it: host float64 tensors, state and output float64, the three scans
    with return_prefix=True agreeing within 1e-10; here also against the
    oracle."""
    announce("generic scan: reference sanity script, float64, host tensors")
    from mogt_amd import affine_scan as das

    U, V = synthetic.reference_test_case()
    kw = dict(state_dtype=torch.float64, output_dtype=torch.float64, return_prefix=True)
    U_seq, H_seq = das.affine_scan_sequential(U, V, **kw)
    U_par, H_par = das.affine_scan_doubling(U, V, **kw)
    U_blk, H_blk = das.affine_scan_block_reference(U, V, block_size=5, carry_scan="doubling", **kw)
    for t in (U_seq, H_seq, U_par, H_par, U_blk, H_blk):
        assert t.device.type == "cpu" and t.dtype == torch.float64
    for a, b in ((U_seq, U_par), (H_seq, H_par), (U_seq, U_blk), (H_seq, H_blk)):
        assert float((a - b).abs().max()) <= 1e-10
    P_ref, H_ref = so.affine_scan_sequential(U.numpy(), V.numpy(), return_prefix=True)
    assert np.max(np.abs(H_seq.numpy() - H_ref)) <= 1e-10
    assert np.max(np.abs(U_seq.numpy() - P_ref)) <= 1e-10
    assert rel_err(H_seq.numpy(), H_ref) <= F64_TOL and rel_err(U_seq.numpy(), P_ref) <= F64_TOL


def test_reference_backward_sanity_fp64(gpu):
    """run_affine_backward_sanity (sanity_affine_scan.py:102-135): autograd
    through affine_scan_sequential vs affine_scan_sequential_backward, float64,
    host tensors, bar 1e-10; both also against the oracle's backward."""
    announce("generic scan: reference backward sanity, float64")
    from mogt_amd import affine_scan as das

    U, V = synthetic.reference_test_case(seq_len=9, rank=4, channels=3)
    grad_out = torch.randn_like(V)
    U_ref = U.detach().clone().requires_grad_(True)
    V_ref = V.detach().clone().requires_grad_(True)
    H = das.affine_scan_sequential(U_ref, V_ref, state_dtype=torch.float64, output_dtype=torch.float64)
    gU_auto, gV_auto = torch.autograd.grad(H, (U_ref, V_ref), grad_outputs=grad_out)
    gU, gV = das.affine_scan_sequential_backward(U, V, grad_out, state_dtype=torch.float64)
    assert gU.device.type == "cpu" and gU.dtype == torch.float64
    assert float((gU_auto - gU).abs().max()) <= 1e-10
    assert float((gV_auto - gV).abs().max()) <= 1e-10
    gU_ref, gV_ref = so.affine_scan_sequential_backward(U.numpy(), V.numpy(), grad_out.numpy())
    assert np.max(np.abs(gU.numpy() - gU_ref)) <= 1e-10
    assert np.max(np.abs(gV.numpy() - gV_ref)) <= 1e-10


@pytest.mark.parametrize("B,L,R,C", [(2, 3000, 16, 48), (1, 5000, 4, 3), (3, 700, 24, 5), (1, 17, 1, 1),
                                     (1, 40, 1, 600), (2, 33, 2, 300)])
def test_fp64_state_multichunk(gpu, B, L, R, C):
    """float64 state across many chunks (carry pass and chunk summaries), with
    the prefix product, on the device."""
    announce(f"generic scan fp64 B={B} L={L} R={R} C={C}")
    import mogt_amd.ops as ops

    U, V = _stable(B, L, R, C, seed=L + R)
    P_ref, H_ref = so.affine_scan_sequential(U, V, return_prefix=True)
    Ug, Vg = torch.from_numpy(U).to(gpu), torch.from_numpy(V).to(gpu)
    P, H = ops.affine_scan(Ug, Vg, state_dtype=torch.float64, return_prefix=True)
    H_only = ops.affine_scan(Ug, Vg, state_dtype=torch.float64)
    torch.cuda.synchronize()
    assert H.dtype == torch.float64 and P.dtype == torch.float64
    assert rel_err(np64(H), H_ref) <= F64_TOL
    assert rel_err(np64(P), P_ref) <= F64_TOL
    assert torch.equal(H_only, H)


@pytest.mark.parametrize("R,L,C", [(33, 300, 4), (48, 257, 8), (64, 200, 3), (65, 150, 2), (100, 90, 5),
                                   (130, 40, 3)])
def test_ranks_above_32(gpu, R, L, C):
    """Ranks the matrix-core pipeline does not take: fp32 state (the matrix-core
    chunk kernel up to R = 64, the scalar kernel above), through the hybrid
    drop-in, with the prefix product; float64 state at the same shapes."""
    announce(f"generic scan R={R} L={L} C={C}")
    from mogt_amd import affine_scan as das
    from mogt_amd import triton_scan

    U, V = _stable(1, L, R, C, seed=R)
    P_ref, H_ref = so.affine_scan_sequential(U, V, return_prefix=True)
    U32, V32 = torch.from_numpy(U.astype(np.float32)).to(gpu), torch.from_numpy(V.astype(np.float32)).to(gpu)
    P, H = triton_scan.triton_affine_scan_hybrid(U32, V32, return_prefix=True)
    H2 = triton_scan.triton_affine_scan_hybrid(U32, V32)
    P64, H64 = das.affine_scan_sequential(torch.from_numpy(U).to(gpu), torch.from_numpy(V).to(gpu),
                                          state_dtype=torch.float64, return_prefix=True)
    torch.cuda.synchronize()
    assert H.dtype == torch.float32
    assert rel_err(np64(H), H_ref) <= FP32_TOL and rel_err(np64(P), P_ref) <= FP32_TOL
    assert torch.equal(H, H2)
    assert rel_err(np64(H64), H_ref) <= F64_TOL and rel_err(np64(P64), P_ref) <= F64_TOL


@pytest.mark.parametrize("R", [40, 16])
def test_fused_scan_generic_ranks(gpu, R):
    """triton_fused_scan beyond R = 32 (the generic scan's prefix columns with
    no channels) and a float64 output at R = 16."""
    announce(f"generic fused scan R={R}")
    from mogt_amd import triton_scan

    U, _ = _stable(2, 333, R, 1, seed=5 + R)
    Y_ref = so.fused_scan(U)
    if R > 32:
        Y = triton_scan.triton_fused_scan(torch.from_numpy(U.astype(np.float32)).to(gpu))
        tol = FP32_TOL
    else:
        import mogt_amd.ops as ops
        Y = ops.fused_scan(torch.from_numpy(U.astype(np.float32)).to(gpu), output_dtype=torch.float64)
        tol = FP32_TOL
        assert Y.dtype == torch.float64
    torch.cuda.synchronize()
    assert rel_err(np64(Y), Y_ref) <= tol


@pytest.mark.parametrize("vdt,odt,sdt,tol", [
    (torch.bfloat16, torch.float64, torch.float64, F64_TOL),
    (torch.float16, torch.float16, torch.float64, 2e-3),
    (torch.float64, torch.bfloat16, torch.float64, 2e-2),
    (torch.float64, torch.float32, torch.float32, FP32_TOL),
    (torch.float16, torch.float32, torch.float32, FP32_TOL),
])
def test_io_dtypes(gpu, vdt, odt, sdt, tol):
    """Inputs and outputs in fp16 / bf16 / fp64: V is converted to the state
    dtype on load (V.to(state_dtype), affine_scan.py:36), outputs rounded from
    the state (H_t.to(output_dtype), :52)."""
    announce(f"generic scan V {vdt} out {odt} state {sdt}")
    import mogt_amd.ops as ops

    U, V = _stable(2, 400, 8, 6, seed=11)
    Vt = torch.from_numpy(V).to(vdt)
    P_ref, H_ref = so.affine_scan_sequential(U, Vt.double().numpy(), return_prefix=True)
    Ug = torch.from_numpy(U).to(gpu).to(sdt)
    P, H = ops.affine_scan(Ug, Vt.to(gpu), output_dtype=odt, state_dtype=sdt, return_prefix=True)
    torch.cuda.synchronize()
    assert H.dtype == odt and P.dtype == odt
    if sdt == torch.float32:
        P_ref, H_ref = so.affine_scan_sequential(U.astype(np.float32).astype(np.float64), Vt.double().numpy(),
                                                 return_prefix=True)
    assert rel_err(np64(H.double()), H_ref) <= tol
    assert rel_err(np64(P.double()), P_ref) <= tol


@pytest.mark.parametrize("R,L,C,sdt", [(40, 120, 5, torch.float64), (6, 300, 4, torch.float64),
                                       (12, 150, 7, torch.float32)])
def test_autograd_with_prefix(gpu, R, L, C, sdt):
    """Gradients through both outputs (U_prefix and H) of the differentiable
    drop-in against torch.autograd of a host float64 loop; without the prefix
    against the oracle's backward.  fp32 state (R <= 32) runs on the
    matrix-core pipeline and its autograd."""
    announce(f"generic scan autograd R={R} L={L} C={C} state {sdt}")
    from mogt_amd import affine_scan as das

    U, V = _stable(2, L, R, C, seed=R + C)
    g = synthetic.rng(99)
    dP = torch.from_numpy(g.standard_normal(U.shape))
    dH = torch.from_numpy(g.standard_normal(V.shape))
    Uc = torch.from_numpy(U).requires_grad_(True)
    Vc = torch.from_numpy(V).requires_grad_(True)
    P_c, H_c = _torch_seq(Uc, Vc, True)
    gU_ref, gV_ref = torch.autograd.grad((P_c * dP).sum() + (H_c * dH).sum(), (Uc, Vc))

    tdt = torch.float64 if sdt == torch.float64 else torch.float32
    tol = F64_TOL if sdt == torch.float64 else FP32_TOL
    Ug = torch.from_numpy(U).to(gpu, tdt).requires_grad_(True)
    Vg = torch.from_numpy(V).to(gpu, tdt).requires_grad_(True)
    P, H = das.affine_scan_sequential(Ug, Vg, state_dtype=sdt, return_prefix=True)
    gU, gV = torch.autograd.grad((P * dP.to(gpu, tdt)).sum() + (H * dH.to(gpu, tdt)).sum(), (Ug, Vg))
    torch.cuda.synchronize()
    assert gU.dtype == tdt and gV.dtype == tdt
    assert rel_err(np64(gU.double()), gU_ref.numpy()) <= tol
    assert rel_err(np64(gV.double()), gV_ref.numpy()) <= tol

    gU_o, gV_o = so.affine_scan_sequential_backward(U, V, dH.numpy())
    Ug2 = Ug.detach().requires_grad_(True)
    Vg2 = Vg.detach().requires_grad_(True)
    H2 = das.affine_scan_doubling(Ug2, Vg2, state_dtype=sdt)
    H2.backward(dH.to(gpu, tdt))
    torch.cuda.synchronize()
    assert rel_err(np64(Ug2.grad.double()), gU_o) <= tol
    assert rel_err(np64(Vg2.grad.double()), gV_o) <= tol


def test_hand_backward_fp64_long(gpu):
    """affine_scan_sequential_backward in float64 over many chunks (the
    generic reverse scan with transposed transitions), R = 20."""
    announce("generic reverse scan fp64 L=2500 R=20")
    from mogt_amd import affine_scan as das

    U, V = _stable(2, 2500, 20, 9, seed=3)
    G = synthetic.rng(4).standard_normal(V.shape)
    gU_ref, gV_ref = so.affine_scan_sequential_backward(U, V, G)
    gU, gV = das.affine_scan_sequential_backward(torch.from_numpy(U).to(gpu), torch.from_numpy(V).to(gpu),
                                                 torch.from_numpy(G).to(gpu), state_dtype=torch.float64)
    only_v = das.affine_scan_sequential_backward(torch.from_numpy(U).to(gpu), torch.from_numpy(V).to(gpu),
                                                 torch.from_numpy(G).to(gpu), state_dtype=torch.float64,
                                                 need_grad_u=False)
    torch.cuda.synchronize()
    assert only_v[0] is None and torch.equal(only_v[1], gV)
    assert rel_err(np64(gV), gV_ref) <= F64_TOL
    assert rel_err(np64(gU), gU_ref) <= F64_TOL


def test_generic_argument_errors(gpu):
    from mogt_amd import affine_scan as das
    import mogt_amd.ops as ops

    U = torch.zeros(1, 4, 3, 3, device=gpu)
    V = torch.zeros(1, 4, 3, 2, device=gpu)
    with pytest.raises(ValueError):
        das.affine_scan_sequential(U, V, state_dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        ops.affine_scan(U, V, output_dtype=torch.int32)
    with pytest.raises(ValueError):
        das.affine_scan_sequential(torch.zeros(1, 2, 1025, 1025, device=gpu, dtype=torch.bfloat16),
                                   torch.zeros(1, 2, 1025, 1, device=gpu))
    # empty problems; no channels leaves the prefix product alone (U = 2 I: 2^(t+1) I)
    assert das.affine_scan_sequential(U[:, :0], V[:, :0], state_dtype=torch.float64).shape == (1, 0, 3, 2)
    U2 = (2 * torch.eye(3, device=gpu)).expand(1, 4, 3, 3)
    P, H = das.affine_scan_sequential(U2, V[..., :0], state_dtype=torch.float64, return_prefix=True)
    torch.cuda.synchronize()
    want = torch.stack([2.0 ** (t + 1) * torch.eye(3, dtype=torch.float64) for t in range(4)])[None]
    assert H.shape == (1, 4, 3, 0) and torch.equal(P.cpu(), want)


def test_zz_generic_no_lookback_wait_gave_up(gpu):
    import mogt_amd.ops as ops

    assert ops.workspace_faults() == 0


@pytest.mark.parametrize("R,block", [(40, 1), (40, 7), (64, 64), (100, 33)])
def test_local_scan_ranks_above_32(gpu, R, block):
    """triton_affine_local_scan beyond R = 32 (the generic kernel's block-local
    pass): per-step prefixes and per-block summaries against the oracle's
    local_scan, ragged tail block included."""
    announce(f"generic local scan R={R} block={block}")
    from mogt_amd import triton_scan

    U, V = _stable(2, 155, R, 3, seed=R + block)
    ref = so.local_scan(U, V, block_size=block)
    out = triton_scan.triton_affine_local_scan(torch.from_numpy(U.astype(np.float32)).to(gpu),
                                               torch.from_numpy(V.astype(np.float32)).to(gpu), block_size=block)
    torch.cuda.synchronize()
    for got, want in zip(out, ref):
        assert got.dtype == torch.float32 and tuple(got.shape) == want.shape
        assert rel_err(np64(got), want) <= FP32_TOL


def test_dense_scan_vk_rank_above_32(gpu):
    """dense_scan(A, v=v, k=k) at R = 48: B_t = v_t k_t^T formed as fp32
    products and scanned by the generic kernel, against the oracle."""
    announce("generic dense_scan vk R=48")
    import mogt_amd

    U, _ = _stable(2, 200, 48, 1, seed=48)
    g = synthetic.rng(5)
    v = g.standard_normal((2, 200, 48)).astype(np.float32)
    k = g.standard_normal((2, 200, 20)).astype(np.float32)
    V = (v[..., :, None] * k[..., None, :]).astype(np.float64)
    H_ref = so.affine_scan_sequential(U.astype(np.float32).astype(np.float64), V)
    S = mogt_amd.dense_scan(torch.from_numpy(U.astype(np.float32)).to(gpu), v=torch.from_numpy(v).to(gpu),
                            k=torch.from_numpy(k).to(gpu))
    torch.cuda.synchronize()
    assert S.dtype == torch.float32 and S.shape == (2, 200, 48, 20)
    assert rel_err(np64(S), H_ref) <= FP32_TOL


@pytest.mark.parametrize("sdt,tol", [(torch.float64, F64_TOL), (torch.float32, FP32_TOL)])
def test_hand_backward_rank_above_64(gpu, sdt, tol):
    """The reverse scan with U read transposed from memory (R > 64, not staged
    in LDS), several chunks: affine_scan_sequential_backward against the
    oracle."""
    announce(f"generic reverse scan R=70 L=300 state {sdt}")
    from mogt_amd import affine_scan as das

    U, V = _stable(1, 300, 70, 3, seed=70)
    G = synthetic.rng(8).standard_normal(V.shape)
    tdt = torch.float64 if sdt == torch.float64 else torch.float32
    if sdt == torch.float32:
        U, V, G = (x.astype(np.float32).astype(np.float64) for x in (U, V, G))
    gU_ref, gV_ref = so.affine_scan_sequential_backward(U, V, G)
    gU, gV = das.affine_scan_sequential_backward(torch.from_numpy(U).to(gpu, tdt), torch.from_numpy(V).to(gpu, tdt),
                                                 torch.from_numpy(G).to(gpu, tdt), state_dtype=sdt)
    torch.cuda.synchronize()
    assert gU.dtype == tdt and gV.dtype == tdt
    assert rel_err(np64(gV), gV_ref) <= tol
    assert rel_err(np64(gU), gU_ref) <= tol


def _loop64(U, V, rev=False):
    """H_t = U_t H_{t-1} + V_t (rev: H_t = V_t + U_{t+1}^T H_{t+1}) step by step
    in float64 on the host, and the prefix products."""
    U, V = U.double().cpu(), V.double().cpu()
    B, L, R, C = V.shape
    H, P = torch.empty_like(V), torch.empty_like(U)
    h = torch.zeros(B, R, C, dtype=torch.float64)
    pr = torch.eye(R, dtype=torch.float64).expand(B, R, R)
    for s in range(L):
        t = L - 1 - s if rev else s
        if not rev:
            h = U[:, t] @ h + V[:, t]
            pr = U[:, t] @ pr
            P[:, t] = pr
        else:
            h = V[:, t] + (U[:, t + 1].transpose(-1, -2) @ h if s > 0 else 0)
        H[:, t] = h
    return P, H


@pytest.mark.parametrize("state", [torch.float32, torch.float64])
@pytest.mark.parametrize("B,L,R,C", [(1, 1, 1, 1), (2, 7, 15, 16), (1, 16, 16, 17), (3, 17, 17, 5), (1, 300, 32, 33),
                                     (2, 130, 33, 1), (1, 65, 48, 48), (1, 70, 49, 20), (2, 90, 64, 64),
                                     (1, 2100, 4, 3), (40, 33, 64, 40)])
def test_matrix_core_ranks_match_the_loop(gpu, state, B, L, R, C):
    """Ranks up to 64 on the matrix-core chunk kernel: every row-tile edge (with
    and without 16-byte rows of U), ragged column tiles that hold state and
    prefix columns, one step to several chunks of carries, two tiles per wave
    (40 sequences of 64), forward with prefix, forward alone, and reversed."""
    announce(f"generic mfma {state} {B} {L} {R} {C}")
    from mogt_amd import ops

    g = torch.Generator().manual_seed(L + R)
    U = (0.9 * torch.eye(R, dtype=torch.float64) + 0.3 / R * torch.randn(B, L, R, R, generator=g, dtype=torch.float64))
    V = torch.randn(B, L, R, C, generator=g, dtype=torch.float64)
    Ug, Vg = U.to(state).to(gpu), V.to(state).to(gpu)
    Pr, Hr = _loop64(Ug, Vg)
    tol = 2e-6 if state == torch.float32 else 1e-13
    P, H = torch.ops.mogt.affine_scan_generic(Ug, Vg, state, state, True, False)
    assert rel_err(H.double().cpu().numpy(), Hr.numpy()) <= tol
    assert rel_err(P.double().cpu().numpy(), Pr.numpy()) <= tol
    _, H = torch.ops.mogt.affine_scan_generic(Ug, Vg, state, state, False, False)
    assert rel_err(H.double().cpu().numpy(), Hr.numpy()) <= tol
    _, G = torch.ops.mogt.affine_scan_generic(Ug, Vg, state, state, False, True)
    assert rel_err(G.double().cpu().numpy(), _loop64(Ug, Vg, rev=True)[1].numpy()) <= tol


@pytest.mark.parametrize("B,L,R,C", [(40, 700, 36, 20), (20, 1100, 36, 33), (32, 601, 52, 18), (33, 300, 50, 14),
                                     (64, 250, 64, 2)])
def test_two_tiles_per_wave_match_the_loop(gpu, B, L, R, C):
    """Enough chunks that a wave takes two column tiles: pairs of adjacent
    columns (even C and offsets) and single ones (odd C, or rows of U that are not
    16-byte aligned), ragged last chunks, with the prefix and without."""
    announce(f"generic two tiles per wave {B} {L} {R} {C}")
    g = np.random.default_rng(R * 100 + C)
    U = torch.from_numpy((0.9 * np.eye(R) + 0.3 / R * g.standard_normal((B, L, R, R))).astype(np.float32))
    V = torch.from_numpy(g.standard_normal((B, L, R, C)).astype(np.float32))
    Pr, Hr = _loop64(U, V)
    Ug, Vg = U.to(gpu), V.to(gpu)
    P, H = torch.ops.mogt.affine_scan_generic(Ug, Vg, torch.float32, torch.float32, True, False)
    H1 = torch.ops.mogt.affine_scan_generic(Ug, Vg, torch.float32, torch.float32, False, False)[1]
    torch.cuda.synchronize()
    assert rel_err(P.double().cpu().numpy(), Pr.numpy()) <= FP32_TOL
    assert rel_err(H.double().cpu().numpy(), Hr.numpy()) <= FP32_TOL
    assert rel_err(H1.double().cpu().numpy(), Hr.numpy()) <= FP32_TOL


@pytest.mark.parametrize("state", [torch.float32, torch.float64])
@pytest.mark.parametrize("vdt", [torch.float16, torch.bfloat16, torch.float32, torch.float64])
@pytest.mark.parametrize("odt", [torch.float16, torch.bfloat16, torch.float32, torch.float64])
def test_matrix_core_io_dtypes(gpu, state, vdt, odt):
    """Every input and output type of the general form (ragged last chunk), each
    output rounded once from the state through fp32."""
    announce(f"generic mfma io {state} {vdt} {odt}")
    from mogt_amd import ops

    g = torch.Generator().manual_seed(4)
    B, L, R, C = 2, 45, 20, 18
    U = 0.9 * torch.eye(R) + 0.02 * torch.randn(B, L, R, R, generator=g)
    V = torch.randn(B, L, R, C, generator=g).to(vdt)
    P, H = torch.ops.mogt.affine_scan_generic(U.to(gpu), V.to(gpu), state, odt, True, False)
    Pr, Hr = _loop64(U, V)
    tol = {torch.float16: 2e-3, torch.bfloat16: 1e-2, torch.float32: 1e-6, torch.float64: 1e-6}[odt]
    assert H.dtype == odt and P.dtype == odt
    assert rel_err(H.double().cpu().numpy(), Hr.numpy()) <= tol
    assert rel_err(P.double().cpu().numpy(), Pr.numpy()) <= tol
    wide = torch.ops.mogt.affine_scan_generic(U.to(gpu), V.to(gpu), state, state, True, False)
    assert torch.equal(H, wide[1].float().to(odt) if odt != torch.float64 else wide[1].double())


@pytest.mark.parametrize("vdt", [torch.float16, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("R", [36, 47, 48, 52, 64])
@pytest.mark.parametrize("offset", [0, 1])
def test_wide_ranks_with_other_io_types(gpu, vdt, R, offset):
    """The general form at three and four row tiles: 16-byte loads of U where the
    rank and the pointer allow them (R = 47 and an offset U do not), forward with
    prefix and reversed, over several chunks."""
    announce(f"generic mfma wide io {vdt} R={R} offset {offset}")
    g = torch.Generator().manual_seed(R)
    B, L, C = 2, 75, 18
    U = 0.9 * torch.eye(R) + 0.3 / R * torch.randn(B, L, R, R, generator=g)
    V = torch.randn(B, L, R, C, generator=g).to(vdt)
    flat = torch.zeros(U.numel() + 1, device=gpu)
    Ug = flat[offset:offset + U.numel()].view(U.shape).copy_(U)
    Pr, Hr = _loop64(U, V)
    P, H = torch.ops.mogt.affine_scan_generic(Ug, V.to(gpu), torch.float32, torch.float32, True, False)
    assert rel_err(H.double().cpu().numpy(), Hr.numpy()) <= 2e-6 and rel_err(P.double().cpu().numpy(), Pr.numpy()) <= 2e-6
    _, G = torch.ops.mogt.affine_scan_generic(Ug, V.to(gpu), torch.float32, torch.float32, False, True)
    assert rel_err(G.double().cpu().numpy(), _loop64(U, V, rev=True)[1].numpy()) <= 2e-6


@pytest.mark.parametrize("R,B,L,C,state,vdt", [(1, 16, 70, 1501, torch.float64, torch.float64),
                                               (1, 3, 701, 1000, torch.float32, torch.float16),
                                               (2, 40, 600, 130, torch.float32, torch.float64),
                                               (2, 70, 150, 1000, torch.float64, torch.float32),
                                               (3, 21, 300, 1600, torch.float64, torch.float64),
                                               (4, 9, 1250, 900, torch.float64, torch.float64),
                                               (4, 64, 500, 1000, torch.float32, torch.bfloat16)])
def test_wide_states_of_few_ranks_match_the_loop(gpu, R, B, L, C, state, vdt):
    """Wide states at ranks of 1 to 4 take the scalar kernel (transitions staged
    in LDS): ragged chunks and column tiles, with the prefix, without, reversed."""
    announce(f"generic wide low rank R={R} {B} {L} {C} {state} {vdt}")
    g = torch.Generator().manual_seed(R * L)
    U = (0.8 * torch.eye(R) + 0.2 / R * torch.randn(B, L, R, R, generator=g)).to(state)
    V = torch.randn(B, L, R, C, generator=g).to(vdt)
    Ug, Vg = U.to(gpu), V.to(gpu)
    tol = 2e-6 if state == torch.float32 else 1e-13
    Pr, Hr = _loop64(U, V)
    P, H = torch.ops.mogt.affine_scan_generic(Ug, Vg, state, state, True, False)
    one = torch.ops.mogt.affine_scan_generic(Ug, Vg, state, state, False, False)[1]
    assert rel_err(H.double().cpu().numpy(), Hr.numpy()) <= tol and rel_err(P.double().cpu().numpy(), Pr.numpy()) <= tol
    assert rel_err(one.double().cpu().numpy(), Hr.numpy()) <= tol
    _, G = torch.ops.mogt.affine_scan_generic(Ug, Vg, state, state, False, True)
    assert rel_err(G.double().cpu().numpy(), _loop64(U, V, rev=True)[1].numpy()) <= tol


def test_matrix_core_workspace_covers_both_levels():
    """The workspace the C entry asks for grows with the chunks of both levels
    and is the header alone for one pass (host arithmetic only)."""
    from mogt_amd import _lib

    lib = _lib.load()
    one = lib.mogt_affine_scan_generic_workspace_bytes(1, 16, 16, 48, 0, 2)
    assert one == 256
    n = lib.mogt_affine_scan_generic_workspace_bytes(1, 32768, 16, 48, 0, 2)
    assert n > 256 + 8 * 16 * (64 + 48) * 128
    assert lib.mogt_affine_scan_generic_workspace_bytes(1, 32768, 16, 48, 1, 2) > n


@pytest.mark.parametrize("state", [torch.float32, torch.float64])
@pytest.mark.parametrize("B,L,R,C", [(1, 9, 1, 1), (2, 40, 5, 3), (1, 600, 20, 6), (40, 70, 40, 20), (2, 50, 64, 16)])
def test_infinite_state_keeps_its_sign(gpu, state, B, L, R, C):
    """An infinity entering one column of a rank that does not fill its row tiles
    stays an infinity (positive transitions): the padded rows must not turn it
    into NaN, and the other columns stay as they are."""
    announce(f"generic infinite state {state} {B} {L} {R} {C}")
    g = torch.Generator().manual_seed(R)
    U = ((0.5 + torch.rand(B, L, R, R, generator=g, dtype=torch.float64)) / R).to(state)
    V = torch.rand(B, L, R, C, generator=g, dtype=torch.float64).to(state)
    V[:, L // 3, R // 2, 0] = float("inf")
    for rev in (False, True):
        ref = _loop64(U, V, rev=rev)[1]
        _, H = torch.ops.mogt.affine_scan_generic(U.to(gpu), V.to(gpu), state, state, False, rev)
        H = H.double().cpu()
        inf = torch.isinf(ref)
        assert inf.any() and not torch.isnan(ref).any()
        assert torch.equal(torch.isinf(H), inf) and not torch.isnan(H).any()
        assert bool((H[inf] > 0).all()) and rel_err(H[~inf].numpy(), ref[~inf].numpy()) <= FP32_TOL
