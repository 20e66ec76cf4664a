"""Shared helpers of the parity tests: seeded inputs and comparison with the oracle."""
import math

import torch

from oracle import fastmax_oracle as O

TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2}   # rel-L2 bars: fp32 1e-5, bf16 2e-2


def make_inputs(bh, nq, nk, d, dtype, device, seed=0, scale=1.0, go_scale=1.0):
    gen = torch.Generator().manual_seed(seed)
    q = (scale * torch.randn(bh, nq, d, generator=gen)).to(dtype)
    k = (scale * torch.randn(bh, nk, d, generator=gen)).to(dtype)
    v = (scale * torch.randn(bh, nk, d, generator=gen)).to(dtype)
    go = (go_scale * torch.randn(bh, nq, d, generator=gen)).to(dtype)
    return tuple(t.to(device) for t in (q, k, v, go))


def rel_err(x, ref, cancel=None):
    """Plain rel-L2 ||x - ref|| / ||ref||, with no floor.

    ``cancel`` is only for a reference that is zero because two terms cancel exactly (dq, dk of a
    single causal token: gh.v and c are the same number): it is the per-element size of the terms that
    cancel, derived from the inputs by the caller (``cancel_scale``).  Only when ||ref|| is below 1e-9 of
    that size (the fp64 oracle's own rounding residue) is the error measured against it instead."""
    x = x.detach().double().cpu(); ref = ref.detach().double().cpu()
    den = float(ref.norm())
    if cancel is not None and den < 1e-9 * cancel * ref.numel() ** 0.5:
        den = cancel * ref.numel() ** 0.5
    if den == 0.0:
        return 0.0 if float((x - ref).norm()) == 0.0 else float("inf")
    return float((x - ref).norm() / den)


def cancel_scale(q, k, v, go, g, tau, a):
    """Per-element size of one of the terms whose difference is dq or dk: f'(s) (dO/g . v) k / tau, from the
    inputs' root-mean-squares (the scores' term with their rms)."""
    rms = lambda t: float(t.detach().double().pow(2).mean().sqrt())
    d = q.shape[-1]
    s = rms(q) * rms(k) * d ** 0.5 / tau
    gmin = max(float(g.detach().double().abs().min()), 1e-300)
    return (abs(a[1]) + 2 * abs(a[2]) * s) * rms(go) * rms(v) * d ** 0.5 * max(rms(q), rms(k)) / (tau * gmin)


def oracle_all(q, k, v, go, *, mask, tau, p, a=(1.0, 1.0, 0.5), block=1024):
    """fp64 closed form on the (already rounded) inputs: o, g, dq, dk, dv."""
    args = [t.detach().cpu().double() for t in (q, k, v, go)]
    if mask or q.shape[1] * k.shape[1] > 1 << 22:
        return O.manual_backward_blocked(*args, mask=mask, tau=tau, p=p, a0=a[0], a1=a[1], a2=a[2], block=block)
    return O.closed_form_forward_backward(*args, mask=mask, tau=tau, p=p, a0=a[0], a1=a[1], a2=a[2])


def check_forward(lib, bh, nq, d, dtype, device, *, mask, p, nk=None, chunk=0, flags=0, tau_mult=8.0,
                  a=(1.0, 1.0, 0.5), seed=0, scale=1.0):
    nk = nk or nq
    q, k, v, go = make_inputs(bh, nq, nk, d, dtype, device, seed, scale)
    tau = tau_mult * math.sqrt(d)
    o, g = lib.forward(q, k, v, mask=mask, inv_tau=1.0 / tau, a0=a[0], a1=a[1], a2=a[2], p=p, chunk=chunk, flags=flags)
    ref = oracle_all(q, k, v, go, mask=mask, tau=tau, p=p, a=a)
    eo, eg = rel_err(o, ref[0]), rel_err(g, ref[1])
    assert eo < TOL[dtype], f"o rel-L2 {eo:.3e}"
    assert eg < TOL[dtype], f"g rel-L2 {eg:.3e}"
    return eo, eg


def check_forward_backward(lib, bh, nq, d, dtype, device, *, mask, p, nk=None, chunk=0, flags=0, tau_mult=8.0,
                           a=(1.0, 1.0, 0.5), seed=0, scale=1.0, saved=False, go_scale=1.0):
    """saved: run the backward on the workspace the forward leaves behind
    (FASTMAX_FLAG_SAVE_FOR_BACKWARD / fastmax_backward_saved).  go_scale: size of the upstream gradient."""
    nk = nk or nq
    q, k, v, go = make_inputs(bh, nq, nk, d, dtype, device, seed, scale, go_scale)
    tau = tau_mult * math.sqrt(d)
    kw = dict(mask=mask, inv_tau=1.0 / tau, a0=a[0], a1=a[1], a2=a[2], p=p, chunk=chunk, flags=flags)
    if saved:
        o, g, ws = lib.forward(q, k, v, save=True, **kw)
        dq, dk, dv = lib.backward(q, k, v, o, g, go, saved=ws, **kw)
    else:
        o, g = lib.forward(q, k, v, **kw)
        dq, dk, dv = lib.backward(q, k, v, o, g, go, **kw)
    ref = oracle_all(q, k, v, go, mask=mask, tau=tau, p=p, a=a)
    cs = cancel_scale(q, k, v, go, ref[1], tau, a)
    errs = {n: rel_err(x, r, cs if n in ("dq", "dk") else None)
            for n, x, r in zip(("o", "g", "dq", "dk", "dv"), (o, g, dq, dk, dv), ref)}
    for n, e in errs.items():
        assert e < TOL[dtype], f"{n} rel-L2 {e:.3e} (all: {errs})"
    return errs


def check_batch_head_strides(lib, b, h, n, d, dtype, device, *, mask, p, chunk=0, seed=0):
    """q, k, v, dO as transposed views of (b, n, h*d) tensors, handed over with batch and head
    strides (FastmaxStrides.heads > 1), outputs written into the same memory order: bit-identical
    to the run on contiguous (b*h, n, d) copies."""
    gen = torch.Generator().manual_seed(seed)
    base = [torch.randn(b, n, h * d, generator=gen).to(dtype).to(device) for _ in range(4)]
    q4, k4, v4, go4 = (x.view(b, n, h, d).transpose(1, 2) for x in base)
    tau = 8.0 * math.sqrt(d)
    kw = dict(mask=mask, inv_tau=1.0 / tau, p=p, chunk=chunk)
    out = torch.empty(b, n, h, d, dtype=dtype, device=device).transpose(1, 2)
    o4, g4, ws = lib.forward(q4, k4, v4, save=True, out=out, **kw)
    q3, k3, v3, go3 = (x.contiguous().view(b * h, n, d) for x in (q4, k4, v4, go4))
    o3, g3, ws3 = lib.forward(q3, k3, v3, save=True, **kw)
    assert torch.equal(o4.contiguous().view(b * h, n, d), o3) and torch.equal(g4.reshape(b * h, n), g3)
    d4 = lib.backward(q4, k4, v4, o4, g4, go4, saved=ws, **kw)
    d3 = lib.backward(q3, k3, v3, o3, g3, go3, saved=ws3, **kw)
    for x4, x3 in zip(d4, d3):
        assert torch.equal(x4.contiguous().view(b * h, n, d), x3)
    return True


def check_norm_fold(lib, bh, nq, d, dtype, device, *, mask, p, nk=None, chunk=0, lim=1.5, tau=1.0, seed=0, saved=True,
                    jacobian=True, scale=1.0):
    """The max-norm normalisation of q and k folded into the kernels (FastmaxNormFold) against the fp64 closed
    form on lim * x / max_n ||x_n||: o, g, and either the gradients with respect to the raw q and k (torch
    autograd through the normalisation: ``jacobian``) or those with respect to the normalised tensors (what the
    reference's extension returns)."""
    nk = nk or nq
    q, k, v, go = make_inputs(bh, nq, nk, d, dtype, device, seed, scale)
    qk, kk = lib.maxnorm_stats(q, k)
    kw = dict(mask=mask, inv_tau=1.0 / tau, p=p, chunk=chunk, norm=(qk, kk, lim, jacobian))
    if saved:
        o, g, ws = lib.forward(q, k, v, save=True, **kw)
        dq, dk, dv = lib.backward(q, k, v, o, g, go, saved=ws, **kw)
    else:
        o, g = lib.forward(q, k, v, **kw)
        dq, dk, dv = lib.backward(q, k, v, o, g, go, **kw)
    qd, kd, vd, gd = (t.detach().cpu().double() for t in (q, k, v, go))
    if jacobian:
        qd.requires_grad_(True); kd.requires_grad_(True); vd.requires_grad_(True)
        oo, gg = O.closed_form_forward(O.normalize_lim(qd, lim), O.normalize_lim(kd, lim), vd, mask=mask, tau=tau, p=p)
        rq, rk, rv = torch.autograd.grad(oo, (qd, kd, vd), gd)
        ref = (oo.detach(), gg.detach(), rq, rk, rv)
    else:
        ref = oracle_all(O.normalize_lim(qd, lim), O.normalize_lim(kd, lim), vd, gd, mask=mask, tau=tau, p=p)
    errs = {n: rel_err(x, r) for n, x, r in zip(("o", "g", "dq", "dk", "dv"), (o, g, dq, dk, dv), ref)}
    for n, e in errs.items():
        assert e < TOL[dtype], f"{n} rel-L2 {e:.3e} (all: {errs})"
    return errs


def check_decode(lib, bh, n, n0, d, dtype, device, *, p, tau_mult=8.0, a=(1.0, 1.0, 0.5), seed=0, four_d=False):
    """Incremental decoding on the persistent moment state: the first n0 tokens are absorbed as a prompt, the
    others go through one step each; every step's o and g against the fp64 closed form of causal attention over
    the whole sequence (the state is fp32, so the bar is the fp32 one for fp32 tensors, the bf16 one for bf16)."""
    q, k, v, _ = make_inputs(bh, n, n, d, dtype, device, seed)
    tau = tau_mult * math.sqrt(d)
    kw = dict(inv_tau=1.0 / tau, p=p, a0=a[0], a1=a[1], a2=a[2])
    if four_d:                                   # (b, h, n, d) views of a (b, n, h*d) layout, two heads per batch
        assert bh % 2 == 0
        q, k, v = (t.view(bh // 2, 2, n, d).transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    state = lib.decode_state(k, **kw)
    if n0:
        lib.decode_absorb(k[..., :n0, :], v[..., :n0, :], state, **kw)
    outs, gs = [], []
    for t in range(n0, n):
        o, g = lib.decode_step(q[..., t:t + 1, :], k[..., t:t + 1, :], v[..., t:t + 1, :], state, **kw)
        outs.append(o); gs.append(g)
    o = torch.cat(outs, dim=-2).reshape(bh, n - n0, d)
    g = torch.cat(gs, dim=-1).reshape(bh, n - n0)
    q3, k3, v3 = (t.reshape(bh, n, d).detach().cpu().double() for t in (q, k, v))
    ro, rg = O.closed_form_forward(q3, k3, v3, mask=True, tau=tau, p=p, a0=a[0], a1=a[1], a2=a[2])
    eo, eg = rel_err(o, ro[:, n0:]), rel_err(g, rg[:, n0:])
    assert eo < TOL[dtype] and eg < TOL[dtype], f"decode o {eo:.3e} g {eg:.3e}"
    return eo, eg


def check_infinite_and_largest_values(lib, bh, n, d, dtype, device, *, flags=0, seed=0, largest=None):
    """One infinite entry, one NaN and one entry at the top of the type's range, in v and in dO: what IEEE arithmetic gives.
    All weights are positive, so an infinite v is an infinite output column, and its neighbours do not change; an infinite
    dO is an infinite column of dv, and the other queries' dq do not change.  The largest entry's key is zero (its weight
    1), so nothing overflows.  Unmasked, plain weights; every other number against the fp64 closed form."""
    q, k, v, go = make_inputs(bh, n, n, d, dtype, device, seed)
    t, f, tau = n - 2, 5, 8.0 * math.sqrt(d)
    k[:, t] = 0.0
    kw = dict(mask=False, inv_tau=1.0 / tau, p=2, flags=flags)
    tol = 1.5 * TOL[dtype] if dtype == torch.bfloat16 else 2e-6
    rest = [i for i in range(d) if i != f]
    ref = oracle_all(q, k, v, go, mask=False, tau=tau, p=2)
    o0, g0 = lib.forward(q, k, v, **kw)
    for x in (float("inf"), float("-inf"), float("nan")):
        w = v.clone(); w[:, t, f] = x
        o, g = lib.forward(q, k, w, **kw)
        same = torch.isnan(o[..., f]) if x != x else o[..., f] == x
        assert bool(same.all()), f"v = {x}: {o[0, :, f]}"
        assert rel_err(o[..., rest], ref[0][..., rest]) < tol and rel_err(g, ref[1]) < tol
        w = go.clone(); w[:, t, f] = x
        dq, dk, dv = lib.backward(q, k, v, o0, g0, w, **kw)
        same = torch.isnan(dv[..., f]) if x != x else dv[..., f] == x
        assert bool(same.all()), f"dO = {x}: {dv[0, :, f]}"
        assert rel_err(dv[..., rest], ref[4][..., rest]) < tol
        others = [i for i in range(n) if i != t]
        assert rel_err(dq[:, others], ref[2][:, others]) < tol
        assert not bool(torch.isfinite(dq[:, t]).any()) and not bool(torch.isfinite(dk).any())
    for x in ((3.0e38, 3.4e38) if largest is None else largest):
        w = v.clone(); w[:, t, f] = x
        o, g = lib.forward(q, k, w, **kw)
        big = oracle_all(q, k, w, go, mask=False, tau=tau, p=2)
        assert rel_err(o[..., f], big[0][..., f]) < tol, f"v = {x}: {o[0, :3, f]}"
        assert rel_err(o[..., rest], big[0][..., rest]) < tol
        w = go.clone(); w[:, t, f] = x
        dq, dk, dv = lib.backward(q, k, v, o0, g0, w, **kw)
        big = oracle_all(q, k, v, w, mask=False, tau=tau, p=2)
        assert rel_err(dv[..., f], big[4][..., f]) < tol and rel_err(dq[:, t], big[2][:, t]) < tol
        assert rel_err(dk.double() / 1e38, big[3] / 1e38) < tol


def check_tiny_values(lib, bh, n, d, dtype, device, *, tol, flags=0, seed=0):
    """One of v, dO, q and k far below 1e-30, at the same bar as ordinary numbers: everything here is linear in v and in dO,
    and dq and dk in the other factor.  (The results stay above fp32's subnormal numbers.)"""
    tau = 8.0 * math.sqrt(d)
    for which, scale in ((2, 3e-36), (3, 1e-34), (0, 1e-35), (1, 1e-35)):
        x = list(make_inputs(bh, n, n, d, torch.float32, device, seed + which, go_scale=1.0 if which == 3 else 1e4))
        x[which] = x[which] * scale
        q, k, v, go = (t.to(dtype) for t in x)
        kw = dict(mask=True, inv_tau=1.0 / tau, p=2, flags=flags)
        o, g = lib.forward(q, k, v, **kw)
        grads = lib.backward(q, k, v, o, g, go, **kw)
        ref = oracle_all(q, k, v, go, mask=True, tau=tau, p=2)
        errs = {m: rel_err(a, b) for m, a, b in zip(("o", "g", "dq", "dk", "dv"), (o, g, *grads), ref)}
        assert max(errs.values()) < tol, f"tiny {'q k v dO'.split()[which]}: {errs}"


def check_upstream_gradients_at_the_ends_of_the_range(lib, bh, n, d, device, *, flags=0, seed=0):
    """bf16 tensors, dO near the smallest and the largest numbers of its type (gradients are linear in dO): dq and dv at the
    bf16 bar.  Small q and large k keep the scores ordinary and dq far enough from the subnormal numbers."""
    tau = 8.0 * math.sqrt(d)
    for go_scale in (2e-37, 3e37):
        q, k, v, go = make_inputs(bh, n, n, d, torch.float32, device, seed, go_scale=go_scale)
        q, k, v, go = (t.bfloat16() for t in (0.02 * q, 50.0 * k, v, go))
        kw = dict(mask=False, inv_tau=1.0 / tau, p=2, flags=flags)
        o, g = lib.forward(q, k, v, **kw)
        dq, _, dv = lib.backward(q, k, v, o, g, go, **kw)
        ref = oracle_all(q, k, v, go, mask=False, tau=tau, p=2)
        eq, ev = rel_err(dq, ref[2]), rel_err(dv, ref[4])
        assert eq < TOL[torch.bfloat16] and ev < TOL[torch.bfloat16], f"dO x {go_scale:g}: dq {eq:.3e}, dv {ev:.3e}"


def check_prompt_at_the_ends_of_the_range(lib, d, dtype, device, n, *, bh=2, seed=0, cases=4):
    """Order-2 sums of a prompt of 64 tokens and more, one token of which has a key of very different features (most of them zero) and
    a value at an end of the range: products k'_a v overflow where k'_a k'_b v do not.  The state is that of the same tokens
    added one after the other: every sum within n 2^-23 of the sizes of its terms (two roundings per term, n of the sums), infinite
    where that one is."""
    inv_tau = 0.125                                            # exact: k' is what is meant
    for t, x, big, small in ((n - 2, 1e38, 8.0, 1e-3), (3, 3e38, 1.25, 1e-30), (40, 1e-37, 2.0, 0.5), (5, 1e25, 1e-10, 1e-25))[:cases]:
        gen = torch.Generator().manual_seed(seed)
        k, v = (torch.randn(bh, n, d, generator=gen) for _ in range(2))
        k[0, t] = 0.0
        k[0, t, 1], k[0, t, d - 1] = big / inv_tau, small / inv_tau
        v[0, t] = 0.5
        v[0, t, 5] = x
        k, v = k.to(dtype).to(device), v.to(dtype).to(device)
        if x < 1.0:
            v[0, :t, 5] = v[0, t + 1:, 5] = 0.0                # nothing beside the tiny terms
        kw = dict(inv_tau=inv_tau, p=2, a0=1.0, a1=1.0, a2=0.5)
        one, want, size = (lib.decode_state(k, **kw) for _ in range(3))
        new = torch.full_like(one, float("nan"))
        lib.decode_absorb(k, v, one, **kw)
        lib.decode_absorb(k, v, new, new=True, **kw)
        for t0 in range(0, n, 48):
            lib.decode_absorb(k[:, t0:t0 + 48], v[:, t0:t0 + 48], want, **kw)
            lib.decode_absorb(k[:, t0:t0 + 48].abs(), v[:, t0:t0 + 48].abs(), size, **kw)
        one, new, want, size = (s.cpu() for s in (one, new, want, size))
        assert torch.equal(one, new) and not bool(torch.isnan(want).any())
        assert torch.equal(torch.isinf(one), torch.isinf(want))
        finite = torch.isfinite(want)
        off = (one[finite].double() - want[finite].double()).abs() / (n * 2.0 ** -23 * size[finite].double()).clamp_min(1e-44)
        assert float(off.max()) <= 1.0, f"v = {x:g}: {float(off.max()):g} of the bound"


def check_ranges_of_two_planes(lib, bh, n, d, device, *, mask=True, seed=0, tol=2e-6):
    """fp32, entries far below the rest of their tensor: a column of v and of dO, a row of k and v, the last queries' dO.  Each result that
    only they reach is held to fp32's bar by itself: the column of o and dv, the first query's o (causal), the last keys' dv."""
    tau = 8.0 * math.sqrt(d)
    kw = dict(mask=mask, inv_tau=1.0 / tau, p=2)
    for which in ("column of v", "column of dO", "first row of v", "last rows of dO"):
        q, k, v, go = make_inputs(bh, n, n, d, torch.float32, device, seed)
        if which == "column of v": v[:, :, 3] *= 1e-9
        if which == "column of dO": go[:, :, 3] *= 1e-9
        if which == "first row of v": v[:, 0] *= 1e-9
        if which == "last rows of dO": go[:, -40:] *= 1e-9
        o, g = lib.forward(q, k, v, **kw)
        dq, dk, dv = lib.backward(q, k, v, o, g, go, **kw)
        ref = oracle_all(q, k, v, go, mask=mask, tau=tau, p=2)
        parts = {"o": (o, ref[0]), "g": (g, ref[1]), "dq": (dq, ref[2]), "dk": (dk, ref[3]), "dv": (dv, ref[4])}
        if which == "column of v": parts["o there"] = (o[..., 3], ref[0][..., 3])
        if which == "column of dO": parts["dv there"] = (dv[..., 3], ref[4][..., 3])
        if which == "first row of v" and mask: parts["o there"] = (o[:, 0], ref[0][:, 0])
        if which == "last rows of dO" and mask: parts["dv there"] = (dv[:, -40:], ref[4][:, -40:])
        for m, (x, r) in parts.items():
            assert rel_err(x, r) < tol, f"{which}: {m} {rel_err(x, r):.3e}"


def check_keys_that_see_small_gradients(lib, bh, n, d, device, *, end, zeros, seed=0, tol=2e-6):
    """fp32, causal: dO is zero in the `zeros` rows up to `end` (tokens left out of a loss) and far smaller behind them, so that the keys of
    those rows see small gradients alone.  Their dk and dv are held to the bar by themselves."""
    tau = 8.0 * math.sqrt(d)
    kw = dict(mask=True, inv_tau=1.0 / tau, p=2)
    rows = slice(end - zeros, end)
    for scale in (1e-5, 1e-9):
        q, k, v, go = make_inputs(bh, n, n, d, torch.float32, device, seed)
        go[:, rows] = 0.0
        go[:, end:] *= scale
        o, g = lib.forward(q, k, v, **kw)
        grads = lib.backward(q, k, v, o, g, go, **kw)
        ref = oracle_all(q, k, v, go, mask=True, tau=tau, p=2)[2:]
        errs = {m: rel_err(x, r) for m, x, r in zip(("dq", "dk", "dv"), grads, ref)}
        errs.update({m + " there": rel_err(x[:, rows], r[:, rows]) for m, x, r in zip(("dk", "dv"), grads[1:], ref[1:])})
        assert max(errs.values()) < tol, f"dO x {scale:g} behind token {end}: {errs}"


def check_small_tensor_against_a_large_one(lib, bh, n, d, device, *, p, seed=0, tol=2e-6, ends=((2e-31, 2e29), (2e29, 2e-31))):
    """fp32: q near one end of the range and k near the other, so that their scores are ordinary numbers."""
    kw = dict(mask=True, inv_tau=1.0, p=p, a2=0.5 if p == 2 else 0.0, flags=2)        # FASTMAX_FLAG_FORCE_DENSE
    for q_scale, k_scale in ends:
        q, k, v, go = make_inputs(bh, n, n, d, torch.float32, device, seed)
        q, k = q * q_scale, k * k_scale
        if p == 1:
            k, q = k.abs(), q.abs()                    # (weights that add up)
        o, g = lib.forward(q, k, v, **kw)
        grads = lib.backward(q, k, v, o, g, go, **kw)
        ref = oracle_all(q, k, v, go, mask=True, tau=1.0, p=p)
        errs = {m: rel_err(x, r) for m, x, r in zip(("o", "g", "dq", "dk", "dv"), (o, g, *grads), ref)}
        assert max(errs.values()) < tol, f"q x {q_scale:g}, k x {k_scale:g}, order {p}: {errs}"


def check_column_of_small_gradients(lib, bh, n, d, device, *, mask, seed=0, tol=2e-6):
    """fp32: a column of dO is zero in the first tokens and dO far smaller behind them, so that this column of dv is made of small
    gradients alone.  It is held to the bar by itself."""
    tau = 8.0 * math.sqrt(d)
    kw = dict(mask=mask, inv_tau=1.0 / tau, p=2, flags=2)      # FASTMAX_FLAG_FORCE_DENSE
    for scale in (1e-8, 1e-12):
        q, k, v, go = make_inputs(bh, n, n, d, torch.float32, device, seed)
        go[:, 64:] *= scale
        go[:, :64, 3] = 0.0
        go[:, :, 7] = 0.0                              # (zero everywhere: not a column of small numbers)
        o, g = lib.forward(q, k, v, **kw)
        grads = lib.backward(q, k, v, o, g, go, **kw)
        ref = oracle_all(q, k, v, go, mask=mask, tau=tau, p=2)[2:]
        errs = {m: rel_err(x, r) for m, x, r in zip(("dq", "dk", "dv"), grads, ref)}
        errs["dv there"] = rel_err(grads[2][..., 3], ref[2][..., 3])
        assert max(errs.values()) < tol and not bool(grads[2][..., 7].any()), f"dO x {scale:g}: {errs}"


def check_numbers_within_two_planes(lib, bh, n, d, device, *, mask, seed=0, tol=2e-6):
    """fp32: a first token with a value near zero and a feature of k far larger than the others, both common in trained models.  What only
    those reach is held to the bar by itself."""
    tau = 8.0 * math.sqrt(d)
    q, k, v, go = make_inputs(bh, n, n, d, torch.float32, device, seed)
    v[:, 0] *= 1e-3
    k[..., 5] *= 300.0
    q[..., 5] /= 300.0
    kw = dict(mask=mask, inv_tau=1.0 / tau, p=2, flags=2)      # FASTMAX_FLAG_FORCE_DENSE
    o, g = lib.forward(q, k, v, **kw)
    grads = lib.backward(q, k, v, o, g, go, **kw)
    ref = oracle_all(q, k, v, go, mask=mask, tau=tau, p=2)
    errs = {m: rel_err(x, r) for m, x, r in zip(("o", "g", "dq", "dk", "dv"), (o, g, *grads), ref)}
    errs["first o"] = rel_err(o[:, 0], ref[0][:, 0])
    errs["other dq"] = rel_err(grads[0][..., :5], ref[2][..., :5])
    errs["dk there"] = rel_err(grads[1][..., 5], ref[3][..., 5])
    assert max(errs.values()) < tol, errs
