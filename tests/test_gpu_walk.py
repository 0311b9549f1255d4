"""The one-pass layer (csrc/ssd_walk.hip) against the oracle where it can go
wrong: one position to a few chunks of 64 with every remainder, each dstate, a
whole head or half of one per workgroup, chains cut into segments (up to 32, a
last one that is shorter; each forced plan is asked for by what it runs), initial
states, the z gate, D per head dim, rising dA_cumsum; and the plan the library
picks by itself.

Tolerance: the bf16 bar of the layer, 2e-2 of the RMS (it holds CB and the
states entering each chunk in bf16, as the other paths do)."""

import contextlib
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import TOL, announce, check, dev, tdtype
from mamba2_jax import _lib as L
from mamba2_jax import configs
from mamba2_jax.kernels import mamba_chunk_scan_combined_fwd
from oracle import ssd_oracle as O

pytestmark = pytest.mark.gpu

# (batch, L, H, G, dstate, chunk, init, z, D per head dim[, head dim]) and, beside a
# whole and half a head per workgroup, the cuts of its chains that the workspace holds:
# {forced plan: (segments, workgroups per head) that it runs}
SHAPES = [
    ((1, 1, 2, 1, 128, 128, False, False, False), {}),
    ((2, 63, 4, 2, 64, 64, True, False, True), {}),
    ((1, 64, 4, 1, 256, 128, True, True, False), {}),
    ((1, 65, 2, 1, 128, 256, False, True, True), {}),
    ((3, 130, 6, 2, 128, 128, True, False, False), {}),
    ((1, 447, 4, 1, 256, 64, False, False, True),
     {"walk_x2": (2, 1), "walk_half_x3": (3, 2), "walk_x5": (4, 1)}),
    ((1, 1000, 5, 1, 64, 128, True, True, True), {"walk_x2": (2, 1), "walk_half_x3": (3, 2)}),
    ((2, 1088, 4, 4, 128, 256, True, False, False), {"walk_x2": (2, 1)}),
    ((1, 65, 4, 2, 128, 256, True, True, False, 32), {}),
    ((2, 700, 6, 1, 64, 128, False, False, True, 32), {"walk_x2": (2, 1)}),
    ((1, 1000, 4, 1, 256, 64, True, False, False, 32), {"walk_x2": (2, 1), "walk_x5": (4, 1)}),
    ((1, 1000, 8, 1, 128, 128, True, False, True),
     {"walk_x2": (2, 1), "walk_half_x3": (3, 2), "walk_x5": (4, 1)}),
    ((2, 901, 4, 1, 128, 64, True, True, False), {"walk_x5": (5, 1), "walk_half_x5": (5, 2)}),
    ((1, 2100, 6, 1, 128, 64, True, False, False, 32), {"walk_x3": (3, 1), "walk_x16": (11, 1)}),
    # as many segments as there are, the last one shorter
    ((1, 4090, 12, 1, 128, 64, True, False, False), {"walk_x32": (32, 1), "walk_half_x32": (32, 2)}),
]


def _inputs(b, Lq, H, G, N, Q, init, z, dhp, P=64, *, seed):
    cfg = configs.SSDConfig("walk", b, Lq, H, G, P, N, Q, "bf16", init_state=init, seed=seed)
    d = configs.make_ssd_inputs(cfg, with_z=z)
    if dhp:
        d["D"] = np.random.default_rng(seed).uniform(0.5, 1.5, (H, P)).astype(np.float32)
    d.pop("seq_idx"), d.pop("cu_seqlens")
    T = tdtype("bf16")
    t = {k: dev(v, T if k in ("x", "dt", "B", "C", "z") else None) for k, v in d.items()}
    return d, t


def _plan(t, chunk, plan=None):
    """(segments, workgroups per head) of the walk that the library runs, (0, 0) where
    it does not."""
    b, Lq, H, P = t["x"].shape
    args = L.SsdCombinedArgs(
        batch=b, seqlen=Lq, nheads=H, headdim=P, ngroups=t["B"].shape[2], dstate=t["B"].shape[3],
        chunk_size=chunk, dtype=L.dtype_code(t["x"], "x"), dt_dtype=L.dtype_code(t["dt"], "dt"),
        dt_softplus=1, dt_min=0.0, dt_max=float("inf"), z=L.ptr(t.get("z")))
    with L.dispatch_override("layer", plan) if plan else contextlib.nullcontext():
        p = L.load_library().m2_ssd_combined_plan(ctypes.byref(args))
    return (p // 2, p % 2 + 1) if p else (0, 0)


def _check_all(t, d, plans, decay_clamp=False, **kw):
    want = O.ssd_combined(io_dtype="bf16", decay_clamp=decay_clamp, **d, **kw)
    for plan in plans:
        announce("walk", plan, _plan(t, kw["chunk_size"], plan))
        if plan is None:
            got = mamba_chunk_scan_combined_fwd(**t, **kw)
        else:
            with L.dispatch_override("layer", plan):
                got = mamba_chunk_scan_combined_fwd(**t, **kw)
        check(got[0], want[0], TOL["bf16"], "out")
        check(got[1], want[1], TOL["bf16"], "final_states")


@pytest.mark.parametrize("shape,cuts", SHAPES, ids=lambda s: "-".join(str(int(v)) for v in s)
                         if isinstance(s, tuple) else f"{len(s)}cuts")
def test_walk_matches_oracle(shape, cuts):
    announce("walk shape", shape)
    d, t = _inputs(*shape, seed=sum(shape[:5]))
    plans = {"walk": (1, 1), "walk_half": (1, 1 if t["x"].shape[3] == 32 else 2), **cuts}
    for plan, runs in plans.items():
        assert _plan(t, shape[5], plan) == runs, plan
    _check_all(t, d, [*plans, None], chunk_size=shape[5], dt_softplus=True, return_final_states=True)


# (shape, plan): long chains, every dstate and head dim, cut or not
LONG = [((1, 8192, 4, 2, 128, 128, True, False, False), "walk_half_x31"),
        ((1, 8192, 4, 2, 128, 128, True, True, False), "walk_x16"),
        ((1, 8192, 4, 2, 128, 128, True, False, False), "walk"),
        ((1, 5000, 3, 1, 256, 128, True, False, False), "walk_x16"),
        ((1, 5000, 3, 1, 256, 128, True, False, False), "walk_half_x3"),
        ((1, 4100, 2, 1, 64, 64, True, False, True), "walk_x32"),
        ((1, 4100, 6, 1, 128, 64, True, False, False, 32), "walk_x16"),
        ((1, 4100, 6, 1, 256, 256, True, False, False, 32), "walk_x2")]


@pytest.mark.parametrize("shape,plan", LONG, ids=lambda v: v if isinstance(v, str) else "-".join(str(int(i)) for i in v))
def test_walk_against_the_other_path(shape, plan):
    """Every row of y and every state row beside the other path's.  Both paths round
    at 2^-9: CB, the state that enters a chunk, and (the other path) C h, none of them
    to the same partial sums, so a row of y may differ by two such roundings, 2^-8, of
    itself or, where its terms cancel, of a typical row; over all rows, whose roundings
    are independent and most of whose value is D x, 1e-4 (2e-5 seen).  The states see
    the rounding of w x alone, 2^-17, in different chunks."""
    announce("walk against", shape, plan)
    d, t = _inputs(*shape, seed=3)
    kw = dict(chunk_size=shape[5], dt_softplus=True, return_final_states=True)
    nseg, parts = _plan(t, shape[5], plan)
    assert nseg > 1 or plan == "walk"
    outs = {}
    for p in ("two_pass", plan):
        with L.dispatch_override("layer", p):
            outs[p] = [v.double() for v in mamba_chunk_scan_combined_fwd(**t, **kw)]
    for what, a, b, tol, all_ in zip(("out", "final"), outs["two_pass"], outs[plan],
                                     (2.0 ** -8, 2.0 ** -16), (1e-4, 2.0 ** -17)):
        an, rms = a.norm(dim=-1), a.norm() / a[..., 0].numel() ** 0.5
        err = (a - b).norm(dim=-1) / (an + rms)
        total = float((a - b).norm() / a.norm())
        print(f"  {what}: worst row {float(err.max()):.2e}, all {total:.2e}", flush=True)
        assert float(err.max()) <= tol and total <= all_


# A > 0: (L, dstate, chunk, head dim, init, z, plan, segments, workgroups per head)
RISING = [
    (300, 128, 64, 64, False, False, "walk", 1, 1),
    (700, 128, 128, 64, False, False, "walk", 1, 1),
    (700, 128, 128, 64, True, False, "walk_half", 1, 2),
    (700, 128, 128, 64, True, False, "walk_x3", 3, 1),
    (705, 64, 128, 64, False, True, "walk_half_x2", 2, 2),
    (640, 64, 256, 64, True, False, "walk", 1, 1),
    (1000, 256, 128, 64, True, False, "walk", 1, 1),
    (1000, 256, 128, 64, False, False, "walk_half_x2", 2, 2),
    (1000, 256, 128, 64, True, True, "walk_x2", 2, 1),
    (1100, 128, 256, 32, False, False, "walk", 1, 1),
    (1100, 128, 256, 32, True, False, "walk_x2", 2, 1),
    (1100, 256, 256, 32, True, False, "walk", 1, 1),
    (1100, 64, 128, 32, True, False, "walk_x2", 2, 1),
]


@pytest.mark.parametrize("case", RISING, ids=lambda c: "-".join(str(v) for v in c))
def test_walk_rising_dA(case):
    """A > 0 (all heads but one): dA_cumsum rises, and the chunk states' weights are
    clamped chunk by chunk of the layer (64, 128 or 256 positions) while the outputs
    are not, whatever the walk's own chunks are.  The other path computes the same: it
    rounds C h to bf16 before exp(dA) and the intra-chunk CB of positions that the walk
    carries in a bf16 state, 2^-9 = 2e-3 of a part of the result; its states hold
    no rounding but that of w x, 2^-17 = 8e-6.  Weights clamped over 64 positions move
    the states by 7e-2 (chunk 128, max over RMS) and more."""
    Lq, N, Q, P, init, z, plan, nseg, parts = case
    announce("rising", case)
    d, t = _inputs(1, Lq, 4, 1, N, Q, init, z, False, P, seed=5)
    d["A"] = np.abs(d["A"] / 500).astype(np.float32)
    d["A"][1] *= -100
    t["A"] = dev(d["A"])
    kw = dict(chunk_size=Q, dt_softplus=True, return_final_states=True)
    assert _plan(t, Q, plan) == (nseg, parts)
    _check_all(t, d, [plan], decay_clamp=True, **dict(kw, chunk_size=Q if P == 32 else min(Q, 128)))
    outs = {}
    for p in ("two_pass", plan):
        with L.dispatch_override("layer", p):
            outs[p] = mamba_chunk_scan_combined_fwd(**t, **kw)
    for what, a, b, tol in zip(("out", "final"), outs["two_pass"], outs[plan], (2e-3, 8e-6)):
        err = float((a.double() - b.double()).norm() / a.double().norm())
        print(f"  {what} against the two passes: {err:.2e}", flush=True)
        assert err <= tol


def test_signed_dt_keeps_the_two_passes():
    """dt' of both signs (no softplus, dt_limit below 0): the clamped decay depends
    on the chunk size, so a forced walk is ignored and chunks of 128 stay 128."""
    d, t = _inputs(1, 512, 8, 2, 128, 128, False, False, False, seed=5)
    t["dt"] = 0.05 * t["dt"]
    t["dt_bias"] = None
    kw = dict(chunk_size=128, dt_limit=(-1.0, float("inf")), return_final_states=True)
    outs = []
    for plan in ("two_pass", "walk"):
        with L.dispatch_override("layer", plan):
            outs.append(mamba_chunk_scan_combined_fwd(**t, **kw))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


def test_walk_large_decay():
    """|dA| past 500 within a chunk: the decay factors underflow, none overflows."""
    d, t = _inputs(1, 700, 4, 1, 128, 128, True, False, False, seed=6)
    d["A"] = (d["A"] * 40).astype(np.float32)
    t["A"] = dev(d["A"])
    assert _plan(t, 128, "walk_half_x3") == (3, 2)
    _check_all(t, d, ["walk", "walk_half_x3"], chunk_size=128, dt_softplus=True,
               return_final_states=True)


@pytest.mark.parametrize("dt32", [False, True])
def test_walk_repeats_bit_identically(dt32):
    """The same call twice, another shape between: identical outputs (the
    workspace holds the other call's data); dt in bf16 and float32."""
    _, t = _inputs(1, 4096, 48, 1, 128, 256, False, False, False, seed=7)
    _, o = _inputs(2, 777, 16, 2, 256, 128, True, False, False, seed=8)
    if dt32:
        t["dt"] = t["dt"].float()
    kw = dict(dt_softplus=True, return_final_states=True)
    a = [v.clone() for v in mamba_chunk_scan_combined_fwd(chunk_size=256, **t, **kw)]
    mamba_chunk_scan_combined_fwd(chunk_size=128, **o, **kw)
    b = mamba_chunk_scan_combined_fwd(chunk_size=256, **t, **kw)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_two_pass_still_matches():
    """The state pass and the scan, which packed sequences take, at a shape the
    walk would take."""
    shape = (1, 1000, 8, 2, 128, 128, True, False, False)
    d, t = _inputs(*shape, seed=9)
    _check_all(t, d, ["two_pass"], chunk_size=128, dt_softplus=True, return_final_states=True)
