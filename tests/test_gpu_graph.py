"""Decode steps captured in a HIP graph and replayed (the use the
allocation-free entry point serves, and how bench.py issues its engine-order
figures).

Layer chain: each layer's output is the next one's input, two tokens per
graph (so every layer's ring epoch alternates as in eager use).  A twin set
of layers runs the same tokens eagerly through omh_gdn_decode_dev.  The
graph is replayed three times with eager work and synchronisations in
between, and every replay's outputs, and the final states, must equal the
eager run's bit for bit (same kernels, same data)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from overhang_amd import gdn, hip, synth
from overhang_amd.dims import CFG1, Q35B
from tests.tol import assert_close

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("d,B,int8,nl", [(Q35B, 1, True, 3), (CFG1, 6, False, 4)], ids=["35b-int8-B1", "cfg1-B6"])
def test_graph_replays_equal_eager_decode(d, B, int8, nl):
    seed = 6100 + B
    w = synth.layer_weights(d, seed, gnorm_std=0.1)
    conv0, S0 = synth.states(d, seed, B=B)
    base = 3400 + 20 * int8
    A = [gdn.GdnLayer(base + l, d, w, max_seqs=B, int8=int8) for l in range(nl)]
    E = [gdn.GdnLayer(base + 10 + l, d, w, max_seqs=B, int8=int8) for l in range(nl)]
    for L in A + E:
        for s in range(B):
            L.set_state(s, conv0[s], S0[s])
    st = hip.Stream()
    nbytes = B * d.hidden * 4
    xs = [hip.Buffer.from_numpy(synth.normal(seed + t, synth.S_X, (B, d.hidden))) for t in range(2)]
    ga = [[hip.Buffer(nbytes) for _ in range(nl)] for _ in range(2)]
    ea = [[hip.Buffer(nbytes) for _ in range(nl)] for _ in range(2)]

    def run(layers, outs, call):
        for t in range(2):
            for l in range(nl):
                call(layers[l].li, B, xs[t] if l == 0 else outs[t][l - 1], outs[t][l], stream=st)

    g = hip.Graph(st, lambda: run(A, ga, gdn.decode_noalloc_dev))
    try:
        assert g.nodes >= 2 * nl
        for rep in range(3):
            g.launch()
            st.synchronize()
            run(E, ea, gdn.decode_dev)                    # eager work between replays
            st.synchronize()
            for t in range(2):
                for l in range(nl):
                    a = ga[t][l].numpy((B, d.hidden))
                    e = ea[t][l].numpy((B, d.hidden))
                    assert np.isfinite(e).all()
                    np.testing.assert_array_equal(a, e, err_msg=f"replay {rep} token {t} layer {l}")
        for l in range(nl):
            for s in range(B):
                c1, S1 = A[l].get_state(s)
                c2, S2 = E[l].get_state(s)
                assert np.array_equal(c1, c2) and np.array_equal(S1, S2), f"layer {l} seq {s} state"
    finally:
        g.close()
        for L in A + E:
            L.free()


def _attn(li, D, H, KV, hd, rot, max_t, pos, rng):
    """An fp32 attention layer behind a seeded cache of pos rows."""
    w = {"W_" + n: rng.normal(0, 0.02, s).astype(np.float32)
         for n, s in {"q": (2 * H * hd, D), "k": (KV * hd, D), "v": (KV * hd, D), "o": (D, H * hd)}.items()}
    w.update(q_norm=np.zeros(hd, np.float32), k_norm=np.zeros(hd, np.float32))
    L = gdn.AttnLayer(li, D, H, KV, hd, rot, 1e7, 1e-6, max_t, w)
    L.cache_set(0, 0, pos, *(rng.normal(0, 1, (KV, pos, hd)).astype(np.float32) for _ in range(2)))
    return L


def captured_step_outlives_later_steps(warm, pos, T, later):
    """A step captured after one step of `warm` tokens from position 0 (which
    keeps no partials, or those of one split), then eager steps whose splits
    take more room: replays in between equal the eager step bit for bit, so
    the partials have not moved and the capture has planned as an eager call."""
    D = 2048
    L = _attn(3500, D, 16, 2, 256, 64, 4096, 4096, np.random.default_rng(47))
    st = hip.Stream()
    try:
        x = hip.Buffer.from_numpy(np.random.default_rng(48).normal(0, 1, (warm, D)).astype(np.float32))
        out, eager = (hip.Buffer(warm * D * 4) for _ in range(2))
        gdn.attn_forward_dev(L.li, 0, 0, warm, x, out, st)
        st.synchronize()
        g = hip.Graph(st, lambda: gdn.attn_forward_dev(L.li, 0, pos, T, x, out, st))
        try:
            for p, t in [(pos, T)] + later:
                gdn.attn_forward_dev(L.li, 0, p, t, x, eager, st)
                st.synchronize()
                gdn.attn_forward_dev(L.li, 0, pos, T, x, eager, st)
                st.synchronize()
                ref = eager.numpy((T, D)).copy()
                for rep in range(2):
                    out.upload(np.zeros((T, D), np.float32))
                    g.launch()
                    st.synchronize()
                    np.testing.assert_array_equal(out.numpy((T, D)), ref, err_msg=f"replay {rep} after T {t} at {p}")
                assert np.isfinite(ref).all()
        finally:
            g.close()
    finally:
        L.free()


def captured_flash_step_before_any_eager_one():
    """The first flash step of a process, captured: there is no room for
    partials and a capture cannot allocate, so it runs unsplit, and replays
    the same after an eager step has split its keys.  (A wider layer's step
    of 63 tokens, on the split kernel, has made the other scratch.)"""
    rng = np.random.default_rng(49)
    W = _attn(3501, 2048, 16, 2, 256, 64, 64, 1, rng)
    D, pos, T = 1024, 2000, 64
    L = _attn(3502, D, 8, 2, 128, 64, pos + T, pos, rng)
    st = hip.Stream()
    try:
        x = hip.Buffer.from_numpy(rng.normal(0, 1, (63, 2048)).astype(np.float32))
        out, eager = (hip.Buffer(63 * 2048 * 4) for _ in range(2))
        gdn.attn_forward_dev(W.li, 0, 0, 63, x, out, st)
        st.synchronize()
        g = hip.Graph(st, lambda: gdn.attn_forward_dev(L.li, 0, pos, T, x, out, st))
        try:
            got = []
            for rep in range(4):
                g.launch()
                st.synchronize()
                got.append(out.numpy((T, D)).copy())
                if rep == 1:
                    gdn.attn_forward_dev(L.li, 0, pos, T, x, eager, st)
                    st.synchronize()
        finally:
            g.close()
        ref = eager.numpy((T, D))
        assert not np.array_equal(got[0], ref), "the capture was to run unsplit, the eager step split"
        for rep, o in enumerate(got):
            np.testing.assert_array_equal(o, got[0], err_msg=f"replay {rep}")
            assert_close(o, ref, atol=2e-5, rtol=2e-4, what=f"replay {rep}")
    finally:
        W.free()
        L.free()


@pytest.mark.parametrize("call", ["captured_step_outlives_later_steps(4096, 3072, 1024, [(3763, 333), (0, 1023), (0, 449)])",
                                  "captured_step_outlives_later_steps(63, 3000, 40, [(4000, 5), (4000, 63), (4095, 1)])",
                                  "captured_flash_step_before_any_eager_one()"], ids=["prompt", "few-tokens", "no-room"])
def test_captured_attention_steps(call):
    """In a process of its own: scratch is process-wide and only grows, so
    after other tests there would be room from the start."""
    r = subprocess.run([sys.executable, "-c", f"from tests import test_gpu_graph as t; t.{call}; print('done')"],
                       capture_output=True, text=True, timeout=100, cwd=ROOT)
    assert r.returncode == 0 and "done" in r.stdout, r.stderr[-2000:]
