"""GPU parity of the HIP forward and T=1 decode against the FP64 oracle.

Tolerances are the reference's own native gates
(tests/core/test_rebuild_semantics.py:540-597, 870-929 in the reference):
output rtol = atol = 2e-2; C rtol 8e-3 / atol 1.5e-2; S rtol 1e-2 / atol 3e-2;
plus relative-Frobenius bounds stated per test."""
import pytest
import torch

from gpu_common import make_inputs, make_state, max_rel, oracle_of, rel

pytestmark = pytest.mark.gpu


def _native():
    from solvedelta_amd import solvedelta_native
    return solvedelta_native


def _check(out, st, eo, es, tag, frob=1e-2):
    e_out, e_C, e_S = rel(out.float(), eo), rel(st.predictor, es.predictor), rel(st.S, es.S)
    print(f"[{tag}] rel out {e_out:.2e} C {e_C:.2e} S {e_S:.2e} "
          f"max-rel out {max_rel(out.float(), eo):.2e} C {max_rel(st.predictor, es.predictor):.2e} "
          f"S {max_rel(st.S, es.S):.2e}", flush=True)
    torch.testing.assert_close(out.float().cpu(), eo.float(), rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(st.predictor.cpu(), es.predictor.float(), rtol=8e-3, atol=1.5e-2)
    torch.testing.assert_close(st.S.cpu(), es.S.float(), rtol=1e-2, atol=3e-2)
    assert e_out < frob and e_C < frob and e_S < frob


@pytest.mark.parametrize("B,T,H,r,V,seed,decay,with_state", [
    (1, 16, 2, 16, 16, 23, "small", True),
    (1, 64, 2, 16, 16, 3, "softplus", False),
    (2, 130, 2, 32, 24, 4, "softplus", True),
    (1, 256, 1, 128, 128, 5, "softplus", True),
    (1, 19, 2, 16, 16, 6, "small", True),
    (1, 1, 2, 16, 16, 7, "small", True),
    (1, 70, 2, 20, 12, 8, "softplus", True),   # widths not a multiple of 8: element-wise row loads
    (1, 130, 2, 32, 24, 31, "mixed", True),    # wild and ordinary coordinates in one block
    (1, 128, 1, 128, 128, 32, "mixed", True),
])
def test_forward_matches_oracle(B, T, H, r, V, seed, decay, with_state):
    args = make_inputs(B, T, H, r, V, seed=seed, decay=decay)
    state = make_state(B, H, r, V, seed=seed + 100) if with_state else None
    print(f"case B{B} T{T} H{H} r{r} V{V} decay={decay}", flush=True)
    out, st = _native()(*args, initial_state=state, return_final_state=True)
    torch.cuda.synchronize()
    eo, es = oracle_of(args, state)
    _check(out, st, eo, es, f"fwd T{T} r{r}")


def test_forward_gamma_zero_is_gdn2():
    from oracle.sd_oracle import gdn2_oracle
    args = make_inputs(2, 128, 2, 64, 64, seed=11, gamma=0.0)
    out, st = _native()(*args, return_final_state=True)
    d = [a.detach().double().cpu() for a in args]
    eo, eS = gdn2_oracle(d[2], d[3], d[4], d[5], torch.sigmoid(d[6]), torch.sigmoid(d[7]))
    print(f"[gdn2] rel out {rel(out.float(), eo):.2e} S {rel(st.S, eS):.2e}", flush=True)
    assert rel(out.float(), eo) < 1e-2 and rel(st.S, eS) < 1e-2
    assert st.predictor.abs().max().item() == 0.0


def test_forward_extreme_decay_finite():
    args = make_inputs(1, 80, 1, 16, 16, seed=13, decay="extreme")
    state = make_state(1, 1, 16, 16, seed=14, scale=1.0)
    out, st = _native()(*args, initial_state=state, return_final_state=True)
    assert torch.isfinite(out.float()).all() and torch.isfinite(st.predictor).all()
    eo, es = oracle_of(args, state)
    _check(out, st, eo, es, "extreme")


def test_gamma_broadcast_shapes_agree():
    B, T, H, r, V = 1, 70, 2, 16, 16
    outs = []
    for shape in ("BTH", "H", "1H"):
        args = make_inputs(B, T, H, r, V, seed=17, gamma=0.7, gamma_shape=shape)
        outs.append(_native()(*args, return_final_state=True))
    for o, s in outs[1:]:
        assert torch.equal(o, outs[0][0])
        assert torch.equal(s.predictor, outs[0][1].predictor)


def test_strided_views_bitwise_equal_packed():
    """test_rebuild_semantics.py:487-537: strided inputs give bitwise the same result."""
    args = make_inputs(1, 40, 2, 16, 16, seed=19)
    strided = list(args)
    for i in (0, 1, 2, 3, 4, 6, 7):
        x = args[i]
        store = torch.empty(*x.shape[:-1], x.shape[-1] + 7, dtype=x.dtype, device=x.device)
        view = store[..., : x.shape[-1]]
        view.copy_(x)
        strided[i] = view
        assert not view.is_contiguous()
    o1, s1 = _native()(*args, return_final_state=True)
    o2, s2 = _native()(*strided, return_final_state=True)
    o3, s3 = _native()(*args, return_final_state=False)
    assert s3 is None and torch.equal(o1, o3)
    assert torch.equal(o1, o2)
    assert torch.equal(s1.predictor, s2.predictor) and torch.equal(s1.S, s2.S)


def test_aligned_split_continuation():
    """test_rebuild_semantics.py:850-867 (split at a chunk boundary and inside one)."""
    for split in (64, 40):
        args = make_inputs(1, 128, 2, 32, 32, seed=29)
        ow, sw = _native()(*args, return_final_state=True)
        first = [a[:, :split] if a.ndim >= 3 else a for a in args]
        second = [a[:, split:] if a.ndim >= 3 else a for a in args]
        ol, sl = _native()(*first, return_final_state=True)
        orr, sr = _native()(*second, initial_state=sl, return_final_state=True)
        torch.testing.assert_close(ow.float(), torch.cat((ol, orr), 1).float(), rtol=2e-2, atol=2e-2)
        torch.testing.assert_close(sr.predictor, sw.predictor, rtol=8e-3, atol=2e-2)
        torch.testing.assert_close(sr.S, sw.S, rtol=8e-3, atol=2e-2)


@pytest.mark.parametrize("B,H,r,V", [(1, 2, 16, 16), (4, 8, 128, 128), (3, 2, 40, 24)])
def test_decode_step_matches_oracle(B, H, r, V):
    """test_rebuild_semantics.py:900-929 tolerances: out rtol 8e-3 / atol 2e-3,
    states rtol 5e-3 / atol 3e-3."""
    args = make_inputs(B, 1, H, r, V, seed=31)
    state = make_state(B, H, r, V, seed=37)
    with torch.no_grad():
        out, st = _native()(*args, initial_state=state, return_final_state=True)
    torch.cuda.synchronize()
    eo, es = oracle_of(args, state)
    print(f"[decode r{r}] rel out {rel(out.float(), eo):.2e} C {rel(st.predictor, es.predictor):.2e} "
          f"S {rel(st.S, es.S):.2e}", flush=True)
    torch.testing.assert_close(out.float().cpu(), eo.float(), rtol=8e-3, atol=2e-3)
    torch.testing.assert_close(st.predictor.cpu(), es.predictor.float(), rtol=5e-3, atol=3e-3)
    torch.testing.assert_close(st.S.cpu(), es.S.float(), rtol=5e-3, atol=3e-3)


def test_decode_multi_step_matches_oracle():
    """Config-3 style: states advance over several T=1 calls."""
    B, H, r, V, steps = 2, 2, 64, 64, 12
    args = make_inputs(B, steps, H, r, V, seed=41)
    state = make_state(B, H, r, V, seed=43, scale=0.01)
    st = state
    outs = []
    with torch.no_grad():
        for t in range(steps):
            step = [a[:, t:t + 1] if a.ndim >= 3 else a for a in args]
            o, st = _native()(*step, initial_state=st, return_final_state=True)
            outs.append(o)
    eo, es = oracle_of(args, state)
    out = torch.cat(outs, 1)
    print(f"[decode x{steps}] rel out {rel(out.float(), eo):.2e} S {rel(st.S, es.S):.2e}", flush=True)
    assert rel(out.float(), eo) < 1e-2 and rel(st.S, es.S) < 1e-2 and rel(st.predictor, es.predictor) < 1e-2


@pytest.mark.parametrize("B,T,H,r,V,decay,masked", [
    (2, 130, 2, 128, 128, "softplus", False),  # a ragged last chunk
    (1, 64, 1, 40, 100, "mixed", False),       # narrow widths; wild coordinates (d read back)
    (2, 65, 3, 64, 128, "softplus", True),     # token flags
    (1, 17, 2, 160, 144, "softplus", False),   # wide kernels
])
def test_forward_without_gradients_equals_forward_with(B, T, H, r, V, decay, masked):
    """The forward that keeps nothing for a backward gives the training
    forward's output and final states bitwise."""
    from solvedelta_amd import solvedelta_masked_native, solvedelta_native
    args = make_inputs(B, T, H, r, V, seed=T + r, decay=decay, requires_grad=True)
    state = make_state(B, H, r, V, seed=T)
    masks = ()
    if masked:
        g = torch.Generator().manual_seed(T)
        masks = ((torch.rand(B, T, generator=g) > 0.1).cuda(), (torch.rand(B, T, generator=g) < 0.05).cuda())
    fn = solvedelta_masked_native if masked else solvedelta_native
    out, st = fn(*args, *masks, initial_state=state, return_final_state=True)
    assert out.requires_grad
    with torch.no_grad():
        out2, st2 = fn(*args, *masks, initial_state=state, return_final_state=True)
    out3, _ = fn(*[a.detach() for a in args], *masks, initial_state=state)
    assert torch.equal(out, out2) and torch.equal(out, out3)
    assert torch.equal(st.predictor, st2.predictor) and torch.equal(st.S, st2.S)


@pytest.mark.parametrize("H", [2, 140])  # k_prep_c's forms for few and for many chunks
@pytest.mark.parametrize("T,token", [(16, 3), (70, 40), (70, 69)])
def test_predictor_rows_whose_norm_overflows_read_as_zero(T, token, H):
    """u of 3.3e38 along the other tokens' signs: the FP32 sum of squares overflows,
    the inverse norm is 0 and the token's u acts as a zero row, wherever it lies in
    the chunk's Gram blocks; no product of the raw values turns it into NaN."""
    outs = []
    for fill in (3.3e38, 0.0):
        args = make_inputs(4 if T < 64 else 2, T, H, 128, 64, seed=83, decay="small")
        args[0].copy_(args[0].abs())
        args[0][:, token] = fill
        with torch.no_grad():
            out, st = _native()(*args, return_final_state=True)
        outs.append((out, st.predictor, st.S))
    for a, b in zip(*outs):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("H", [64, 65])  # 256 chunks, one per CU; and the first count above
@pytest.mark.parametrize("decay,masked", [("softplus", False), ("mixed", False), ("extreme", False),
                                          ("mixed", True)])
def test_forward_on_both_sides_of_one_chunk_per_cu(H, decay, masked):
    """The two forms of the predictor's chunk preparation at their dividing line,
    a ragged last chunk and wild coordinates among them."""
    from solvedelta_amd import solvedelta_masked_native
    B, T, r, V = 2, 81, 24, 16
    args = make_inputs(B, T, H, r, V, seed=91, decay=decay)
    state = make_state(B, H, r, V, seed=92)
    masks, kw = (), {}
    if masked:
        g = torch.Generator().manual_seed(93)
        masks = (torch.rand(B, T, generator=g) >= 0.2, torch.rand(B, T, generator=g) < 0.1)
        kw = dict(valid_mask=masks[0], reset_mask=masks[1])
    with torch.no_grad():
        fn = solvedelta_masked_native if masked else _native()
        out, st = fn(*args, *(m.cuda() for m in masks), initial_state=state, return_final_state=True)
    eo, es = oracle_of(args, state, **kw)
    _check(out, st, eo, es, f"H{H} {decay} masked={masked}")


@pytest.mark.parametrize("T,r,V,decay,masked", [(81, 24, 16, "mixed", False), (130, 128, 128, "softplus", False),
                                                (65, 65, 80, "extreme", False), (81, 128, 64, "mixed", True)])
def test_a_sequence_is_the_same_alone_and_in_a_large_batch(T, r, V, decay, masked):
    """Rows of a call with more chunks than CUs against calls of one row each with
    fewer: bitwise, gradients and final states included."""
    from solvedelta_amd import solvedelta_masked_native
    B, H = 3, 80  # 160 or 240 chunks a row
    args = make_inputs(B, T, H, r, V, seed=95, decay=decay)
    state = make_state(B, H, r, V, seed=96)
    g = torch.Generator().manual_seed(97)
    masks = (torch.rand(B, T, generator=g) >= 0.2, torch.rand(B, T, generator=g) < 0.1) if masked else ()
    masks = [m.cuda() for m in masks]
    dout = torch.randn(B, T, H, V, generator=g).to(torch.bfloat16).cuda()
    def run(rows):
        a = [x[rows].contiguous().requires_grad_() for x in (*args, *state)]
        fn = solvedelta_masked_native if masked else _native()
        out, st = fn(*a[:9], *(m[rows] for m in masks), initial_state=tuple(a[9:]), return_final_state=True)
        grads = torch.autograd.grad((out, st.S), a, (dout[rows], torch.ones_like(st.S)))
        return [out, st.predictor, st.S, *grads]
    whole = run(slice(0, B))
    for b in range(B):
        for i, (x, y) in enumerate(zip(whole, run(slice(b, b + 1)))):
            assert torch.equal(x[b:b + 1], y), (b, i)
