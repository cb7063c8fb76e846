"""GPU parity of the Gated-DeltaNet path (conv, L2 norm, recurrence) against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from oracle.ref_np import gdn_seq_f64
from irontimber_amd import ops
from irontimber_amd.synth import gdn_inputs, gdn_step_inputs
from tests.gpu_util import announce, assert_argmax_agrees, dev_f32, host

pytestmark = pytest.mark.gpu
STATE_TOL = 5e-3   # final DeltaNet state
OUT_TOL = 2e-3


@pytest.mark.parametrize("nt,K", [(1, 4), (3, 4), (40, 4), (5, 3), (2, 2), (100, 4)])
def test_conv(dev, nt, K):
    announce(f"conv nt={nt} K={K}")
    d = gdn_inputs(3, nt=nt, nv=8, nk=4)
    w = d["w"][:, :K].copy()
    st0 = d["conv_state"][:K - 1].copy()
    want, wst = oracle.gdn_conv(d["x"], w, st0)
    st = dev_f32(st0, dev)
    got = host(ops.gdn_conv(dev_f32(d["x"], dev), dev_f32(w, dev), st))
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-6)
    np.testing.assert_array_equal(host(st), wst)


@pytest.mark.parametrize("nt,K,nv,nk", [(1, 4, 32, 16), (3, 4, 8, 4), (16, 4, 8, 4), (17, 3, 8, 4), (100, 4, 32, 16),
                                         (1000, 2, 4, 2)])
def test_conv_l2norm_fused(dev, nt, K, nv, nk):
    """The fused conv + L2 entry equals the conv then L2 dispatch pair (the oracle's two passes, and
    the GPU's two kernels), including the carried state."""
    announce(f"conv+l2 nt={nt} K={K} nv={nv} nk={nk}")
    d = gdn_inputs(5, nt=nt, nv=nv, nk=nk)
    w = d["w"][:, :K].copy()
    st0 = d["conv_state"][:K - 1].copy()
    want, wst = oracle.gdn_conv(d["x"], w, st0)
    want = oracle.l2norm_heads(want, 2 * nk, 128)
    st = dev_f32(st0, dev)
    got = host(ops.gdn_conv_l2norm(dev_f32(d["x"], dev), dev_f32(w, dev), st, 2 * nk))
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-6)
    np.testing.assert_array_equal(host(st), wst)
    st2 = dev_f32(st0, dev)
    two = ops.gdn_conv(dev_f32(d["x"], dev), dev_f32(w, dev), st2)
    ops.l2norm_heads(two, 2 * nk, 128)
    np.testing.assert_allclose(got, host(two), rtol=2e-6, atol=1e-7)
    np.testing.assert_array_equal(host(st2), wst)


@pytest.mark.parametrize("d", [128, 256])
def test_l2norm(dev, d):
    x = np.random.default_rng(2).standard_normal((7, 40 * d)).astype(np.float32)
    want = oracle.l2norm_heads(x, 32, d)
    got = host(ops.l2norm_heads(dev_f32(x, dev), 32, d))
    np.testing.assert_allclose(got, want, rtol=1e-6, atol=1e-7)


@pytest.mark.parametrize("nt,nv,nk", [(1, 32, 16), (4, 32, 16), (2, 4, 2), (17, 8, 8), (3, 3, 1), (2, 5, 5)])
def test_step(dev, nt, nv, nk):
    announce(f"gdn_step nt={nt} nv={nv} nk={nk}")
    d = gdn_step_inputs(3, nt, nv=nv, nk=nk)
    want, wst = oracle.gdn_step(d["co"], d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], nv, nk)
    st = dev_f32(d["state"], dev)
    got = host(ops.gdn_step(dev_f32(d["co"], dev), dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev),
                            dev_f32(d["dt"], dev), dev_f32(d["a"], dev), st, nv, nk))
    gst = host(st)
    print(f"out max_abs={np.abs(got - want).max():.3g} state max_abs={np.abs(gst - wst).max():.3g}")
    assert np.abs(got - want).max() <= 1e-5
    assert np.abs(gst - wst).max() <= 1e-5


def test_layer_config4(dev):
    """BASELINE config 4 (seed 3): conv (K=4, rolling state) -> L2 on q/k heads -> one recurrence
    step, 32 V / 16 QK heads, against cpu.rs's layer pass; argmax of a fixed projection agrees."""
    nv, nk, S = 32, 16, 128
    d = gdn_inputs(3, nt=1, nv=nv, nk=nk)
    co_ref = np.zeros((1, d["cd"]), np.float32)
    cst, sst = d["conv_state"].copy(), d["state"].copy()
    out_ref = np.zeros((1, nv * S), np.float32)
    L = oracle.lib()
    P = lambda a: a.ctypes.data
    L.it_ref_gdn_layer(P(d["x"]), d["cd"], P(d["w"]), P(cst), 4, P(d["beta_raw"]), P(d["alpha_raw"]), nv,
                       P(d["dt"]), P(d["a"]), P(sst), P(out_ref), nv * S, P(co_ref), 1, nv, nk, S, 1e-6, 8)
    cs, st = dev_f32(d["conv_state"], dev), dev_f32(d["state"], dev)
    co = ops.gdn_conv(dev_f32(d["x"], dev), dev_f32(d["w"], dev), cs)
    ops.l2norm_heads(co, 2 * nk, S)
    out = host(ops.gdn_step(co, dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev), dev_f32(d["dt"], dev),
                            dev_f32(d["a"], dev), st, nv, nk))
    assert np.abs(out - out_ref).max() <= OUT_TOL
    assert np.abs(host(st) - sst).max() <= STATE_TOL
    np.testing.assert_array_equal(host(cs), cst)
    assert assert_argmax_agrees(out, out_ref) == 0   # no flip


def test_decode_fused_config4(dev):
    """BASELINE config 4 (seed 3) through the one-launch decode layer: against cpu.rs's layer pass
    (conv -> L2 -> recurrence) at the north-star bounds, the new conv state bit-exact, the old conv
    state untouched; argmax of a fixed projection agrees."""
    nv, nk, S = 32, 16, 128
    d = gdn_inputs(3, nt=1, nv=nv, nk=nk)
    co_ref = np.zeros((1, d["cd"]), np.float32)
    cst, sst = d["conv_state"].copy(), d["state"].copy()
    out_ref = np.zeros((1, nv * S), np.float32)
    P = lambda a: a.ctypes.data
    oracle.lib().it_ref_gdn_layer(P(d["x"]), d["cd"], P(d["w"]), P(cst), 4, P(d["beta_raw"]), P(d["alpha_raw"]), nv,
                                  P(d["dt"]), P(d["a"]), P(sst), P(out_ref), nv * S, P(co_ref), 1, nv, nk, S, 1e-6, 8)
    cs_in, st = dev_f32(d["conv_state"], dev), dev_f32(d["state"], dev)
    cs_out = torch.full_like(cs_in, float("nan"))
    out = host(ops.gdn_decode_fused(dev_f32(d["x"], dev), dev_f32(d["w"], dev), cs_in, cs_out, dev_f32(d["beta_raw"], dev),
                                    dev_f32(d["alpha_raw"], dev), dev_f32(d["dt"], dev), dev_f32(d["a"], dev), st, nv, nk))
    assert np.abs(out - out_ref).max() <= OUT_TOL
    assert np.abs(host(st) - sst).max() <= STATE_TOL
    np.testing.assert_array_equal(host(cs_out), cst)
    np.testing.assert_array_equal(host(cs_in), d["conv_state"])
    assert assert_argmax_agrees(out, out_ref) == 0   # no flip


@pytest.mark.parametrize("nt,nv,nk,K", [(1, 32, 16, 4), (2, 32, 16, 4), (4, 8, 4, 3), (3, 4, 2, 2), (1, 8, 8, 4),
                                        (2, 3, 1, 4)])
def test_decode_fused_equals_two_kernels(dev, nt, nv, nk, K):
    """The one-launch layer equals it_gdn_conv_l2norm + it_gdn_step on the same inputs (the q/k
    norms' sums are added in another order: last-bit differences only) and leaves the same conv
    state, bit for bit, in its output buffer."""
    announce(f"gdn fused nt={nt} nv={nv} nk={nk} K={K}")
    d = gdn_inputs(31, nt=nt, nv=nv, nk=nk)
    x, w = dev_f32(d["x"], dev), dev_f32(d["w"][:, :K], dev)
    br, ar = dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev)
    dt, a = dev_f32(d["dt"], dev), dev_f32(d["a"], dev)
    cs0 = d["conv_state"][:K - 1]
    cs, st = dev_f32(cs0, dev), dev_f32(d["state"], dev)
    co = ops.gdn_conv_l2norm(x, w, cs, 2 * nk)
    want = host(ops.gdn_step(co, br, ar, dt, a, st, nv, nk))
    cs_in, cs_out, st2 = dev_f32(cs0, dev), torch.full_like(cs, float("nan")), dev_f32(d["state"], dev)
    got = host(ops.gdn_decode_fused(x, w, cs_in, cs_out, br, ar, dt, a, st2, nv, nk))
    assert np.abs(got - want).max() <= 1e-5
    assert np.abs(host(st2) - host(st)).max() <= 1e-5
    np.testing.assert_array_equal(host(cs_out), host(cs))


@pytest.mark.parametrize("nt,nv,nk,K,ck_after", [(2, 32, 16, 4, 0), (4, 8, 4, 3, 2), (3, 4, 2, 4, 2), (1, 8, 4, 4, 0)])
def test_decode_fused_ckpt_equals_two_kernels(dev, nt, nv, nk, K, ck_after):
    """The MTP verify layer in one launch equals it_gdn_conv_l2norm_ckpt + it_gdn_step_ckpt:
    outputs and final states as in the plain form, the conv checkpoint bit for bit, the state
    checkpoint within last-bit differences."""
    announce(f"gdn fused ckpt nt={nt} nv={nv} nk={nk} K={K} ck_after={ck_after}")
    d = gdn_inputs(37, nt=nt, nv=nv, nk=nk)
    x, w = dev_f32(d["x"], dev), dev_f32(d["w"][:, :K], dev)
    br, ar = dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev)
    dt, a = dev_f32(d["dt"], dev), dev_f32(d["a"], dev)
    cs0 = d["conv_state"][:K - 1]
    cs, st = dev_f32(cs0, dev), dev_f32(d["state"], dev)
    ck_c, ck_s = torch.full_like(cs, float("nan")), torch.full_like(st, float("nan"))
    co = ops.gdn_conv_l2norm(x, w, cs, 2 * nk, ckpt=ck_c, ckpt_after=ck_after)
    want = host(ops.gdn_step(co, br, ar, dt, a, st, nv, nk, ckpt=ck_s, ckpt_after=ck_after))
    cs_in, cs_out, st2 = dev_f32(cs0, dev), torch.full_like(cs, float("nan")), dev_f32(d["state"], dev)
    ck_c2, ck_s2 = torch.full_like(cs, float("nan")), torch.full_like(st, float("nan"))
    got = host(ops.gdn_decode_fused(x, w, cs_in, cs_out, br, ar, dt, a, st2, nv, nk, ckpt_state=ck_s2,
                                    ckpt_conv=ck_c2, ckpt_after=ck_after))
    assert np.abs(got - want).max() <= 1e-5
    assert np.abs(host(st2) - host(st)).max() <= 1e-5
    assert np.abs(host(ck_s2) - host(ck_s)).max() <= 1e-5
    np.testing.assert_array_equal(host(cs_out), host(cs))
    np.testing.assert_array_equal(host(ck_c2), host(ck_c))


@pytest.mark.parametrize("nt,K", [(40, 4), (19, 3)])
def test_conv_l2norm_prompt_equals_token_calls(dev, nt, K):
    """One call over a prompt (the 16-byte, multi-run form) equals nt one-token calls with the conv
    state carried between them (the decode form); the norms' sums differ in order only."""
    announce(f"conv prompt vs tokens nt={nt} K={K}")
    d = gdn_inputs(12, nt=nt, nv=8, nk=4)
    x, w = dev_f32(d["x"], dev), dev_f32(d["w"][:, :K], dev)
    st_a, st_b = dev_f32(d["conv_state"][:K - 1], dev), dev_f32(d["conv_state"][:K - 1], dev)
    whole = host(ops.gdn_conv_l2norm(x, w, st_a, 8))
    steps = np.concatenate([host(ops.gdn_conv_l2norm(x[t:t + 1].contiguous(), w, st_b, 8)) for t in range(nt)])
    assert np.abs(whole - steps).max() <= 1e-6
    np.testing.assert_array_equal(host(st_a), host(st_b))


def test_prefill_equals_fused_decode_steps(dev):
    """GDN prefill over a prompt (conv + L2 in one pass, then the chunk-64 scan) equals the same
    tokens fed one at a time through the one-launch decode layer (conv state alternating between
    two buffers): outputs, final recurrent state and final conv state."""
    nt, nv, nk, S = 70, 8, 4, 128
    d = gdn_inputs(13, nt=nt, nv=nv, nk=nk)
    x, w = dev_f32(d["x"], dev), dev_f32(d["w"], dev)
    br, ar = dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev)
    dt, a = dev_f32(d["dt"], dev), dev_f32(d["a"], dev)
    cs, st = dev_f32(d["conv_state"], dev), dev_f32(d["state"], dev)
    co = ops.gdn_conv_l2norm(x, w, cs, 2 * nk)
    pre = host(ops.gdn_step(co, br, ar, dt, a, st, nv, nk, chunked=True))
    cbuf = [dev_f32(d["conv_state"], dev), torch.empty_like(cs)]
    st2 = dev_f32(d["state"], dev)
    outs = []
    for t in range(nt):
        outs.append(host(ops.gdn_decode_fused(x[t:t + 1].contiguous(), w, cbuf[t & 1], cbuf[(t + 1) & 1],
                                              br[t:t + 1].contiguous(), ar[t:t + 1].contiguous(), dt, a, st2, nv, nk)))
    dec = np.concatenate(outs)
    assert np.abs(pre - dec).max() <= OUT_TOL
    assert np.abs(host(st) - host(st2)).max() <= STATE_TOL
    np.testing.assert_array_equal(host(cs), host(cbuf[nt & 1]))


def test_step_float64_truth(dev):
    d = gdn_step_inputs(4, 6, nv=4, nk=2)
    st = dev_f32(d["state"], dev)
    got = host(ops.gdn_step(dev_f32(d["co"], dev), dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev),
                            dev_f32(d["dt"], dev), dev_f32(d["a"], dev), st, 4, 2))
    o64, s64 = gdn_seq_f64(d["co"], d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], 4, 2)
    np.testing.assert_allclose(got, o64, atol=5e-6)
    np.testing.assert_allclose(host(st), s64, atol=5e-6)


def _chunked(dev, d, nv, nk):
    st = dev_f32(d["state"], dev)
    out = host(ops.gdn_step(dev_f32(d["co"], dev), dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev),
                            dev_f32(d["dt"], dev), dev_f32(d["a"], dev), st, nv, nk, chunked=True))
    return out, host(st)


@pytest.mark.parametrize("nt,nv,nk", [(1, 4, 2), (5, 4, 2), (64, 4, 2), (65, 4, 2), (130, 8, 4), (200, 32, 16),
                                      (64, 4, 4), (1000, 2, 1)])
def test_chunked_matches_float64_recurrence(dev, nt, nv, nk):
    """The chunk-64 WY/UT scan equals the token-sequential recurrence (float64 truth)."""
    announce(f"gdn_chunked nt={nt} nv={nv} nk={nk}")
    d = gdn_step_inputs(5, nt, nv=nv, nk=nk)
    out, st = _chunked(dev, d, nv, nk)
    o64, s64 = gdn_seq_f64(d["co"], d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], nv, nk)
    eo, es = np.abs(out - o64).max(), np.abs(st - s64).max()
    print(f"out max_abs={eo:.3g} state max_abs={es:.3g}")
    assert np.isfinite(out).all() and eo <= OUT_TOL and es <= STATE_TOL



@pytest.mark.parametrize("nt,nv,nk", [(63, 6, 3), (127, 1, 1), (129, 48, 16), (257, 6, 3), (320, 2, 2)])
def test_chunked_and_prefill_more_geometries(dev, nt, nv, nk):
    """More head geometries (one V head; 48 V heads, past the 32 one grid row of the scan holds;
    V heads sharing a q/k head three ways) and chunk counts 1-5 with ragged tails, for both the
    chunked scan from an f32 conv output and the one-call prefill from its f16 one: each against
    the float64 token recurrence on the conv output it consumed."""
    announce(f"gdn chunked + prefill nt={nt} nv={nv} nk={nk}")
    d = gdn_step_inputs(31 + nt, nt, nv=nv, nk=nk)
    out, st = _chunked(dev, d, nv, nk)
    o64, s64 = gdn_seq_f64(d["co"], d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], nv, nk)
    assert np.isfinite(out).all()
    assert np.abs(out - o64).max() <= OUT_TOL and np.abs(st - s64).max() <= STATE_TOL
    d2 = gdn_inputs(41 + nt, nt=nt, nv=nv, nk=nk)
    args = [dev_f32(d2["beta_raw"], dev), dev_f32(d2["alpha_raw"], dev), dev_f32(d2["dt"], dev), dev_f32(d2["a"], dev)]
    cs, st2 = dev_f32(d2["conv_state"], dev), dev_f32(d2["state"], dev)
    co = ops.gdn_conv_l2norm(dev_f32(d2["x"], dev), dev_f32(d2["w"], dev), dev_f32(d2["conv_state"], dev),
                             2 * nk).half().float()
    got = host(ops.gdn_prefill(dev_f32(d2["x"], dev), dev_f32(d2["w"], dev), cs, *args, st2, nv, nk))
    o64, s64 = gdn_seq_f64(host(co), d2["beta_raw"], d2["alpha_raw"], d2["dt"], d2["a"], d2["state"], nv, nk)
    assert np.isfinite(got).all()
    assert np.abs(got - o64).max() <= OUT_TOL and np.abs(host(st2) - s64).max() <= STATE_TOL

def test_chunked_strong_decay_and_zero_beta(dev):
    """Edge cases of the decay/gate: near-total decay (alpha_raw large) and beta ~ 0 on some tokens."""
    nt, nv, nk = 150, 4, 2
    d = gdn_step_inputs(6, nt, nv=nv, nk=nk)
    d["alpha_raw"][10:20] = 30.0
    d["beta_raw"][40:60] = -60.0
    out, st = _chunked(dev, d, nv, nk)
    o64, s64 = gdn_seq_f64(d["co"], d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], nv, nk)
    assert np.abs(out - o64).max() <= OUT_TOL and np.abs(st - s64).max() <= STATE_TOL


def test_chunked_prefill_config5(dev):
    """BASELINE config 5 (seed 4): conv (K=4) -> L2 -> chunk-64 scan over an 8192-token prompt,
    32 V / 16 QK heads, against 8192 sequential steps of the cpu.rs restatement (per-token conv,
    L2 and recurrence); also against the GPU's own token-sequential kernel. Final-state bound
    5e-3, output bound 2e-3, identical argmax of a fixed projection at the last token (the only
    logits a prefill produces), near ties only elsewhere."""
    nv, nk, S, nt = 32, 16, 128, 8192
    d = gdn_inputs(4, nt=nt, nv=nv, nk=nk)
    announce("gdn config5 oracle (cpu)")
    co_ref = np.zeros((nt, d["cd"]), np.float32)
    cst, sst = d["conv_state"].copy(), d["state"].copy()
    out_ref = np.zeros((nt, nv * S), np.float32)
    P = lambda a: a.ctypes.data
    oracle.lib().it_ref_gdn_layer(P(d["x"]), d["cd"], P(d["w"]), P(cst), 4, P(d["beta_raw"]), P(d["alpha_raw"]), nv,
                                  P(d["dt"]), P(d["a"]), P(sst), P(out_ref), nv * S, P(co_ref), nt, nv, nk, S, 1e-6,
                                  oracle.hardware_threads())
    announce("gdn config5 gpu")
    cs = dev_f32(d["conv_state"], dev)
    co = ops.gdn_conv(dev_f32(d["x"], dev), dev_f32(d["w"], dev), cs)
    ops.l2norm_heads(co, 2 * nk, S)
    args = [dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev), dev_f32(d["dt"], dev), dev_f32(d["a"], dev)]
    st = dev_f32(d["state"], dev)
    out = host(ops.gdn_step(co, *args, st, nv, nk, chunked=True))
    gst = host(st)
    eo, es = np.abs(out - out_ref).max(), np.abs(gst - sst).max()
    print(f"config5 chunked vs oracle: out max_abs={eo:.3g} state max_abs={es:.3g}")
    assert eo <= OUT_TOL and es <= STATE_TOL
    np.testing.assert_array_equal(host(cs), cst)
    # the engine takes logits after a prefill only at the prompt's last token (vk/mod.rs:896, `want
    # && last`): that argmax must not move. Over all 8192 tokens, rows may differ only on near
    # ties (oracle top-2 margin within 4 sigma of the measured error); their count is printed.
    assert assert_argmax_agrees(out[-1:], out_ref[-1:]) == 0
    near = assert_argmax_agrees(out, out_ref)
    print(f"config5: {near} near-tie argmax rows of {nt} over the whole prompt")
    st2 = dev_f32(d["state"], dev)
    seq = host(ops.gdn_step(co, *args, st2, nv, nk))
    assert np.abs(seq - out).max() <= OUT_TOL and np.abs(host(st2) - gst).max() <= STATE_TOL


def _z_and_w(seed, nt, nv, S=128):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((nt, nv * S)).astype(np.float32),
            (1 + 0.1 * rng.standard_normal(S)).astype(np.float32))


@pytest.mark.parametrize("nt,nv", [(1, 32), (5, 32), (300, 8)])
def test_gated_rmsnorm(dev, nt, nv):
    """it_gdn_gated_rmsnorm (rmsnorm mode 1, vk/mod.rs:808) against cpu.rs:234-238, in place and
    into a separate buffer."""
    announce(f"gated rmsnorm nt={nt} nv={nv}")
    o = np.random.default_rng(nt).standard_normal((nt, nv * 128)).astype(np.float32)
    z, w = _z_and_w(7, nt, nv)
    want = oracle.gdn_gated_norm(o, z, w, nv)
    od, zd, wd = dev_f32(o, dev), dev_f32(z, dev), dev_f32(w, dev)
    got = host(ops.gdn_gated_rmsnorm(od, zd, wd, nv))
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-6)
    ops.gdn_gated_rmsnorm(od, zd, wd, nv, out=od)
    np.testing.assert_array_equal(host(od), got)


@pytest.mark.parametrize("nt,nv,nk", [(1, 32, 16), (4, 32, 16), (2, 4, 2), (17, 8, 8)])
def test_step_head_kernel_plain(dev, nt, nv, nk):
    """The one-workgroup-per-head recurrence without the epilogue (z = NULL) equals the oracle like
    it_gdn_step does (1e-5), and it_gdn_step within the same bound."""
    announce(f"gdn_step_gated plain nt={nt} nv={nv}")
    d = gdn_step_inputs(3, nt, nv=nv, nk=nk)
    want, wst = oracle.gdn_step(d["co"], d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], nv, nk)
    args = [dev_f32(d[k], dev) for k in ("co", "beta_raw", "alpha_raw", "dt", "a")]
    st = dev_f32(d["state"], dev)
    got = host(ops.gdn_step_gated(*args, st, nv, nk))
    assert np.abs(got - want).max() <= 1e-5 and np.abs(host(st) - wst).max() <= 1e-5
    st2 = dev_f32(d["state"], dev)
    other = host(ops.gdn_step(*args, st2, nv, nk))
    assert np.abs(got - other).max() <= 1e-5


@pytest.mark.parametrize("nt,nv,nk,ck_after", [(1, 32, 16, -1), (4, 32, 16, 0), (2, 32, 16, 0), (9, 8, 4, 5)])
def test_step_gated(dev, nt, nv, nk, ck_after):
    """The recurrence with the gated RMSNorm fused into its output write equals cpu.rs:216-238
    (recurrence then rmsnorm(o)*w*silu(z)); the optional checkpoint is the prefix state."""
    announce(f"gdn_step_gated nt={nt} nv={nv} ck={ck_after}")
    d = gdn_step_inputs(8, nt, nv=nv, nk=nk)
    z, w = _z_and_w(9, nt, nv)
    o_ref, wst = oracle.gdn_step(d["co"], d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], nv, nk)
    want = oracle.gdn_gated_norm(o_ref, z, w, nv)
    args = [dev_f32(d[k], dev) for k in ("co", "beta_raw", "alpha_raw", "dt", "a")]
    st = dev_f32(d["state"], dev)
    ck = torch.full_like(st, float("nan")) if ck_after >= 0 else None
    got = host(ops.gdn_step_gated(*args, st, nv, nk, z=dev_f32(z, dev), norm_w=dev_f32(w, dev), ckpt=ck,
                                  ckpt_after=max(ck_after, 0)))
    e = np.abs(got - want).max()
    print(f"gated out max_abs={e:.3g}")
    assert e <= 1e-4 and np.abs(host(st) - wst).max() <= 1e-5
    if ck is not None:
        st_pre = dev_f32(d["state"], dev)
        n = ck_after + 1
        ops.gdn_step_gated(*[x[:n].contiguous() for x in args[:3]], *args[3:], st_pre, nv, nk)
        np.testing.assert_array_equal(host(ck), host(st_pre))


def test_gated_layer_config4(dev):
    """BASELINE config 4 (seed 3) as the reference's whole GDN decode layer up to the output
    projection: conv + L2 (fused), the recurrence with the fused gated RMSNorm, against cpu.rs
    (layer pass, then the gated norm of cpu.rs:234-238); argmax of a fixed projection agrees."""
    nv, nk, S = 32, 16, 128
    d = gdn_inputs(3, nt=1, nv=nv, nk=nk)
    z, w = _z_and_w(10, 1, nv)
    co_ref = np.zeros((1, d["cd"]), np.float32)
    cst, sst = d["conv_state"].copy(), d["state"].copy()
    out_ref = np.zeros((1, nv * S), np.float32)
    P = lambda a: a.ctypes.data
    oracle.lib().it_ref_gdn_layer(P(d["x"]), d["cd"], P(d["w"]), P(cst), 4, P(d["beta_raw"]), P(d["alpha_raw"]), nv,
                                  P(d["dt"]), P(d["a"]), P(sst), P(out_ref), nv * S, P(co_ref), 1, nv, nk, S, 1e-6, 8)
    want = oracle.gdn_gated_norm(out_ref, z, w, nv)
    cs, st = dev_f32(d["conv_state"], dev), dev_f32(d["state"], dev)
    co = ops.gdn_conv_l2norm(dev_f32(d["x"], dev), dev_f32(d["w"], dev), cs, 2 * nk)
    out = host(ops.gdn_step_gated(co, dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev), dev_f32(d["dt"], dev),
                                  dev_f32(d["a"], dev), st, nv, nk, z=dev_f32(z, dev), norm_w=dev_f32(w, dev)))
    assert np.abs(out - want).max() <= OUT_TOL
    assert np.abs(host(st) - sst).max() <= STATE_TOL
    np.testing.assert_array_equal(host(cs), cst)
    assert_argmax_agrees(out, want)


def test_conv_kparity_geometry(dev):
    """The reference's kernel-parity conv case (src/vk/kparity.rs:32: cd 1000, 5 tokens, K 4, input
    rows at arena 0 with stride 1000, weights at params 0, state at arena 2M), on the harness's own
    xorshift inputs (kparity.rs:13, 59-62): a channel count that is not a multiple of 4 or 128. The
    GPU conv matches the oracle within 1e-6 and leaves the rolling state bit-exact; a second call
    continues from that state."""
    MB = 1 << 20
    arena, params = oracle.kparity_draws(5 << 20, 1 << 16)
    params = params.copy()
    params[16:20] = -np.abs(params[16:20]) - 0.1     # set before every case (kparity.rs:63)
    cd, nt, K = 1000, 5, 4
    x = arena[:nt * cd].reshape(nt, cd)
    w = params[:cd * K].reshape(cd, K)
    st0 = arena[2 * MB:2 * MB + (K - 1) * cd].reshape(K - 1, cd)
    announce("gdn conv kparity cd=1000 nt=5 K=4")
    want, wst = oracle.gdn_conv(x, w, st0)
    st = dev_f32(st0, dev)
    got = host(ops.gdn_conv(dev_f32(x, dev), dev_f32(w, dev), st))
    print(f"kparity conv max_abs={np.abs(got - want).max():.3g}")
    assert np.abs(got - want).max() <= 1e-6
    np.testing.assert_array_equal(host(st), wst)
    x2 = arena[MB:MB + 3 * cd].reshape(3, cd)
    want2, wst2 = oracle.gdn_conv(x2, w, wst)
    got2 = host(ops.gdn_conv(dev_f32(x2, dev), dev_f32(w, dev), st))
    assert np.abs(got2 - want2).max() <= 1e-6
    np.testing.assert_array_equal(host(st), wst2)


@pytest.mark.parametrize("nt,nv,nk,K", [(1, 4, 2, 4), (5, 4, 2, 3), (64, 8, 4, 4), (65, 4, 2, 2), (200, 32, 16, 4),
                                        (130, 8, 8, 4)])
def test_prefill_one_call_equals_f16_conv_output_two_calls(dev, nt, nv, nk, K):
    """it_gdn_prefill (conv + L2 kept as f16, then the chunk-64 scan) equals, bit for bit, the two
    f32 calls it_gdn_conv_l2norm + it_gdn_chunked fed with that conv output rounded to f16 (RNE):
    the f16 prep's single hi x hi product is the three-term hi/lo form with exact zero lo terms.
    Conv state identical; outputs also within the GDN bars of the float64 recurrence."""
    announce(f"gdn prefill one call nt={nt} nv={nv} nk={nk} K={K}")
    d = gdn_inputs(17 + nt, nt=nt, nv=nv, nk=nk, K=K)
    x, w = dev_f32(d["x"], dev), dev_f32(d["w"], dev)
    args = [dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev), dev_f32(d["dt"], dev), dev_f32(d["a"], dev)]
    cs1, st1 = dev_f32(d["conv_state"], dev), dev_f32(d["state"], dev)
    got = host(ops.gdn_prefill(x, w, cs1, *args, st1, nv, nk))
    cs2, st2 = dev_f32(d["conv_state"], dev), dev_f32(d["state"], dev)
    co = ops.gdn_conv_l2norm(x, w, cs2, 2 * nk).half().float()
    want = host(ops.gdn_step(co, *args, st2, nv, nk, chunked=True))
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(host(st1), host(st2))
    np.testing.assert_array_equal(host(cs1), host(cs2))
    o64, s64 = gdn_seq_f64(host(co), d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], nv, nk)
    assert np.abs(got - o64).max() <= OUT_TOL and np.abs(host(st1) - s64).max() <= STATE_TOL


def test_prefill_one_call_config5(dev):
    """BASELINE config 5 (seed 4, f16 activations) through it_gdn_prefill: against 8192 sequential
    steps of the cpu.rs restatement on the f32 layer input, the output and final-state bars,
    the conv state bit-exact, and the last token's argmax identical."""
    nv, nk, S, nt = 32, 16, 128, 8192
    d = gdn_inputs(4, nt=nt, nv=nv, nk=nk)
    announce("gdn config5 one-call oracle (cpu)")
    co_ref = np.zeros((nt, d["cd"]), np.float32)
    cst, sst = d["conv_state"].copy(), d["state"].copy()
    out_ref = np.zeros((nt, nv * S), np.float32)
    P = lambda a: a.ctypes.data
    oracle.lib().it_ref_gdn_layer(P(d["x"]), d["cd"], P(d["w"]), P(cst), 4, P(d["beta_raw"]), P(d["alpha_raw"]), nv,
                                  P(d["dt"]), P(d["a"]), P(sst), P(out_ref), nv * S, P(co_ref), nt, nv, nk, S, 1e-6,
                                  oracle.hardware_threads())
    announce("gdn config5 one call gpu")
    cs, st = dev_f32(d["conv_state"], dev), dev_f32(d["state"], dev)
    args = [dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev), dev_f32(d["dt"], dev), dev_f32(d["a"], dev)]
    out = host(ops.gdn_prefill(dev_f32(d["x"], dev), dev_f32(d["w"], dev), cs, *args, st, nv, nk))
    eo, es = np.abs(out - out_ref).max(), np.abs(host(st) - sst).max()
    print(f"config5 one call vs oracle: out max_abs={eo:.3g} state max_abs={es:.3g}")
    assert eo <= OUT_TOL and es <= STATE_TOL
    np.testing.assert_array_equal(host(cs), cst)
    assert assert_argmax_agrees(out[-1:], out_ref[-1:]) == 0
    near = assert_argmax_agrees(out, out_ref)
    print(f"config5 one call: {near} near-tie argmax rows of {nt} over the whole prompt")


@pytest.mark.parametrize("nt,nv,nk,K", [(17, 8, 4, 4), (18, 8, 4, 3), (19, 4, 2, 2), (24, 8, 4, 4), (67, 48, 16, 4),
                                        (1029, 32, 16, 4), (665, 40, 8, 2), (2405, 40, 8, 4), (2400, 40, 8, 3)])
def test_conv_runs_and_prefill_conv_state(dev, nt, nv, nk, K):
    """The prompt conv at the edges of its 4-token runs, of its 8-token runs (above 4.5 * 2^20 values, 2^23 at 8192
    channels) and of its 16-token runs (above 2^24): against the oracle; and the conv state that the one-call prefill leaves is the layer input's
    last K-1 rows. Taps off by a float: the same to rounding."""
    announce(f"conv runs nt={nt} nv={nv} K={K}")
    d = gdn_inputs(51 + nt, nt=nt, nv=nv, nk=nk)
    w, st0 = d["w"][:, :K].copy(), d["conv_state"][:K - 1].copy()
    want, wst = oracle.gdn_conv(d["x"], w, st0)
    want = oracle.l2norm_heads(want, 2 * nk, 128)
    x, wd = dev_f32(d["x"], dev), dev_f32(w, dev)
    st = dev_f32(st0, dev)
    got = host(ops.gdn_conv_l2norm(x, wd, st, 2 * nk))
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-6)
    np.testing.assert_array_equal(host(st), wst)
    off = torch.empty(w.size + 1, device=dev)[1:].view(w.shape)
    off.copy_(wd)
    st = dev_f32(st0, dev)
    np.testing.assert_allclose(host(ops.gdn_conv_l2norm(x, off, st, 2 * nk)), got, rtol=2e-6, atol=1e-7)
    st = dev_f32(st0, dev)
    ops.gdn_prefill(x, wd, st, dev_f32(d["beta_raw"], dev), dev_f32(d["alpha_raw"], dev), dev_f32(d["dt"], dev),
                    dev_f32(d["a"], dev), dev_f32(d["state"], dev), nv, nk)
    np.testing.assert_array_equal(host(st), wst)


@pytest.mark.parametrize("nt,nv,nk,K", [(17, 8, 4, 4), (24, 8, 4, 3), (67, 32, 16, 2), (1029, 32, 16, 4)])
def test_conv_taps_at_any_float(dev, nt, nv, nk, K):
    """Taps one to three floats off a 16-byte boundary run the prompt conv in the same form: the same bits."""
    announce(f"conv taps nt={nt} nv={nv} K={K}")
    d = gdn_inputs(91 + nt, nt=nt, nv=nv, nk=nk)
    x, w = dev_f32(d["x"], dev), dev_f32(d["w"][:, :K].copy(), dev)
    runs = []
    for off in range(4):
        wd = torch.empty(w.numel() + off, device=dev)[off:].view(w.shape)
        wd.copy_(w)
        runs.append(host(ops.gdn_conv_l2norm(x, wd, dev_f32(d["conv_state"][:K - 1].copy(), dev), 2 * nk)))
    for got in runs[1:]:
        np.testing.assert_array_equal(got, runs[0])


@pytest.mark.parametrize("nt,K,ck_after", [(17, 4, 0), (40, 4, 1), (40, 3, 16), (1029, 4, 1028)])
def test_conv_checkpoint_at_any_float(dev, nt, K, ck_after):
    """A prompt conv with a checkpoint gives the same bits wherever the checkpoint buffer starts, and the
    checkpoint is the last K-1 inputs up to that token."""
    announce(f"conv ckpt nt={nt} K={K} after={ck_after}")
    nv, nk = (32, 16) if nt > 1000 else (8, 4)
    d = gdn_inputs(95 + nt, nt=nt, nv=nv, nk=nk)
    st0 = d["conv_state"][:K - 1].copy()
    x, w = dev_f32(d["x"], dev), dev_f32(d["w"][:, :K].copy(), dev)
    want = np.concatenate([st0, d["x"]])[ck_after + 1:ck_after + K]
    runs = []
    for off in range(2):
        ck = torch.empty(st0.size + off, device=dev)[off:].view(st0.shape)
        st = dev_f32(st0, dev)
        runs.append(host(ops.gdn_conv_l2norm(x, w, st, 2 * nk, ckpt=ck, ckpt_after=ck_after)))
        np.testing.assert_array_equal(host(ck), want)
        np.testing.assert_array_equal(host(st), d["x"][nt - (K - 1):])
    np.testing.assert_array_equal(runs[1], runs[0])


@pytest.mark.parametrize("nt,nv,nk", [(64, 40, 8), (65, 48, 16), (128, 64, 16), (193, 72, 24), (257, 33, 11)])
def test_scan_column_blocks(dev, nt, nv, nk):
    """Head counts whose scan takes 32 state columns a workgroup (more than 32 V heads), with one to five
    chunks, whole and ragged, and head counts that leave an XCD short: the chunked scan and the
    one-call prefill against the float64 recurrence on the conv output each consumed."""
    announce(f"scan column blocks nt={nt} nv={nv} nk={nk}")
    d = gdn_step_inputs(71 + nt, nt, nv=nv, nk=nk)
    out, st = _chunked(dev, d, nv, nk)
    o64, s64 = gdn_seq_f64(d["co"], d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], nv, nk)
    assert np.abs(out - o64).max() <= OUT_TOL and np.abs(st - s64).max() <= STATE_TOL
    d = gdn_inputs(81 + nt, nt=nt, nv=nv, nk=nk)
    x, w = dev_f32(d["x"], dev), dev_f32(d["w"], dev)
    co = ops.gdn_conv_l2norm(x, w, dev_f32(d["conv_state"], dev), 2 * nk).half().float()
    st = dev_f32(d["state"], dev)
    got = host(ops.gdn_prefill(x, w, dev_f32(d["conv_state"], dev), dev_f32(d["beta_raw"], dev),
                               dev_f32(d["alpha_raw"], dev), dev_f32(d["dt"], dev), dev_f32(d["a"], dev), st, nv, nk))
    o64, s64 = gdn_seq_f64(host(co), d["beta_raw"], d["alpha_raw"], d["dt"], d["a"], d["state"], nv, nk)
    assert np.abs(got - o64).max() <= OUT_TOL and np.abs(host(st) - s64).max() <= STATE_TOL
