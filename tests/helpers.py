"""Shared test helpers: synthetic layers at test sizes and error metrics."""
import numpy as np

import llapis_amd as la
from llapis_amd import IQ2_S, IQ4_NL, Q4_K, Q5_0, LayerSpec

SMALL = LayerSpec(d_model=512, n_ff=96, n_expert=16, top_k=4)
# the benchmark's per-expert shapes with fewer experts (fast to quantise)
FULL16 = LayerSpec(d_model=2816, n_ff=704, n_expert=16, top_k=8)


def rel_l2(a, b):
    a = np.asarray(a, np.float64).ravel()
    b = np.asarray(b, np.float64).ravel()
    den = np.linalg.norm(b)
    return float(np.linalg.norm(a - b) / (den if den > 0 else 1.0))


def all_hot(spec):
    return list(range(spec.n_expert))


_cache = {}


def layer(spec, seed, hot, scales=False, router_bias=None):
    key = (spec.d_model, spec.n_ff, spec.n_expert, spec.top_k, spec.hot_gu_type, spec.hot_dn_type,
           spec.cold_gu_type, spec.cold_dn_type, seed, tuple(hot), scales,
           None if router_bias is None else router_bias.tobytes())
    if key not in _cache:
        _cache[key] = la.make_layer(spec, seed, hot, router_bias=router_bias, scales=scales)
    return _cache[key]


def tokens(seed, T, d):
    return la.synth_normal(seed, T * d).reshape(T, d)


# ------------------------------------------------- the benchmark workloads
# d_model 2816, n_ff 704, 128 experts, top-8 (the benchmark's own layer)
FULL = LayerSpec()


def full_layer(seed):
    """Every expert in both tiers: the hot pool holds expert e in slot e
    (Q4_K/Q5_0, no imatrix) and the cold pool every expert (IQ2_S/IQ4_NL,
    imatrix of ones), all quantised from the same seeded fp32 weights."""
    return layer(FULL, seed, all_hot(FULL))


def with_hot_set(full, hot, router_w=None, router_b=None):
    """A layer over `full`'s quantised experts whose K = len(hot) slots hold
    the experts `hot` (slot s = hot[s]); the cold pool is shared."""
    import copy
    sp = full.spec
    gb, db = sp.gu_bytes(sp.hot_gu_type), sp.dn_bytes(sp.hot_dn_type)
    lay = copy.copy(full)
    lay.residency = la.Residency.from_hot(sp.n_expert, list(hot))
    if hot:
        lay.hot_gu = np.concatenate([full.hot_gu[e * gb:(e + 1) * gb] for e in hot])
        lay.hot_dn = np.concatenate([full.hot_dn[e * db:(e + 1) * db] for e in hot])
    else:
        lay.hot_gu = np.zeros(gb, np.uint8)
        lay.hot_dn = np.zeros(db, np.uint8)
    if router_w is not None:
        lay.router_w = router_w
    lay.router_b = router_b
    return lay


def dual_k57(full, seed, router_seed=None):
    """The dual-precision configuration: K = 57 hot experts, the 57 most
    frequent under a Zipf(s = 1.1) routing prior over a seeded permutation,
    and a router bias alpha * log(prior) tuned so ~85 % of top-8 picks land
    on them.  router_seed: a per-layer router (stack layers)."""
    sp = full.spec
    prior, hot = la.zipf_hot_set(sp.n_expert, 57, seed)
    rw = full.router_w
    if router_seed is not None:
        rw = la.synth_normal(la.seed_for(router_seed, 0, 0), sp.n_expert * sp.d_model, 0.0,
                             0.02).reshape(sp.n_expert, sp.d_model)
    bias, frac = la.tune_router_bias(rw, prior, hot, 0.85, seed + 1)
    lay = with_hot_set(full, hot, rw, bias)
    lay.meta["hot_frac"] = frac
    return lay


def in_workspace_for(dl, n_tokens):
    """dl with its calls in a workspace sized for n_tokens tokens: longer
    prefill calls run in several chunks."""
    import ctypes as C

    import torch
    size = int(la.lib().llapis_moe_ffn_workspace_size(C.byref(dl.desc()), n_tokens))
    ws = torch.zeros(size, dtype=torch.uint8, device=dl.device)
    dl.workspace = lambda T: ws
    return dl


def per_token_rel_l2(got, want):
    return np.array([rel_l2(got[t], want[t]) for t in range(got.shape[0])])


def oracle_mode(act_mode, T):
    """The oracle mode a layer call of T tokens is checked in.  Past 4 tokens
    the prefill path runs on the matrix cores, and in the q8_1 mode it forms
    its sums as ggml-cuda's matrix-core path (mmq) does -- IQ2_S's per-16
    scale exact instead of vecdotq's truncating integer formula, Q5_0 as
    (q - 16) against d8 q instead of the stored sum s8 -- which the oracle's
    ACT_Q8_1_MMA mode restates."""
    from oracle import ACT_Q8_1, ACT_Q8_1_MMA
    return ACT_Q8_1_MMA if act_mode == ACT_Q8_1 and T > 4 else act_mode


def check_layer_bars(got, want, say=print, frac_above=0.01):
    """The layer bar against the oracle: the whole output within relative L2
    5e-4 (the requirement is 1e-3), no token above 3e-3, at most 1 % of the
    tokens above 1e-3 and, with more than 16 tokens, the median token at most
    1e-5.  The integer dots are identical on both sides; the fp32 sums run in
    another order, so a gate_up value can differ in its last bit and
    re-quantise one down activation to the neighbouring q8 integer, which
    moves that pair by ~1e-3 and its token by ~3e-4 (two such flips in one
    token reach ~1e-3).  Measured at 512 tokens: about one token in ten has a
    flip, the median token is ~1e-7.  frac_above: the share of tokens allowed
    above 1e-3 (1 %; q8_1 mode scales every 32-block in fp32 on both
    matvecs, so its fp32 orders differ in more places and it flips about 1.5
    times as often: 2 %)."""
    err = rel_l2(got, want)
    per = per_token_rel_l2(got, want)
    say(f"  rel_l2 = {err:.3e}; tokens: median {np.median(per):.1e} max {per.max():.1e} "
        f"({int((per > 1e-5).sum())} of {per.size} above 1e-5, {int((per > 1e-3).sum())} above 1e-3)")
    assert err <= 5e-4, err
    assert per.max() <= 3e-3, (int(per.argmax()), float(per.max()))
    assert (per > 1e-3).sum() <= int(frac_above * per.size), int((per > 1e-3).sum())
    if per.size > 16:
        assert np.median(per) <= 1e-5
    return per
