"""GPU parity of deltanet::chunked_prefill (the chunked gated-DeltaNet prefill) against the
oracle (oracle/deltanet_chunked.py, float64): out and new_state within the path's 2e-3
relative bar, measured as Frobenius and elementwise (tests/_util.py).

Cases: the reference test's heads (V_HEADS = 12 per core, contrib/qwen3.6-27b/kernels/tests/
test_deltanet_chunked_v2.py:17-60, model gates), the 27B model's 48 v-heads (also at a 4096-token
prompt, first and last head against the oracle at 1e-4), a 16379-token prompt (256 chunks), the
C entry point's workspace check, lengths that are
and are not multiples of the chunk, a single token, the reference's chunk sizes in the [C, C]
constants (16 and 64: the kernel chunks by 64 either way), identical pad rows (where the
reference's doubling-product inverse blows up, test_doubling_pad_stability.py:1-19), and the
HF vectors of tests/golden/deltanet_chunked_hf.npz.
"""
import os

import numpy as np
import pytest
import torch

from _util import assert_rel_close
from oracle import deltanet_chunked as oc

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden",
                      "deltanet_chunked_hf.npz")


def _inputs(Hv, S, seed, pad_from=None):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((Hv * S, 128)).astype(np.float32)
    k = rng.standard_normal((Hv * S, 128)).astype(np.float32)
    v = rng.standard_normal((Hv * S, 128)).astype(np.float32)
    A_log = rng.standard_normal(Hv)
    dt = rng.standard_normal(Hv) * 0.1
    a = rng.standard_normal((Hv, S))
    g = (-np.exp(A_log)[:, None] * np.log1p(np.exp(a + dt[:, None]))).reshape(-1, 1)
    beta = 1.0 / (1.0 + np.exp(-rng.standard_normal((Hv * S, 1))))
    state = (rng.standard_normal((Hv * 128, 128)) * 0.05).astype(np.float32)
    if pad_from is not None:
        for arr in (q, k, v):
            a3 = arr.reshape(Hv, S, 128)
            a3[:, pad_from:] = a3[:, pad_from:pad_from + 1]
        for arr in (g, beta):
            a2 = arr.reshape(Hv, S)
            a2[:, pad_from:] = a2[:, pad_from:pad_from + 1]
    return state, q, k, v, g.astype(np.float32), beta.astype(np.float32)


def _run(ops, args, C):
    m = [torch.from_numpy(x).cuda() for x in oc.constants(C)]
    t = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in args]
    out, ns = ops.deltanet.chunked_prefill(*t, *m)
    torch.cuda.synchronize()
    return out.cpu().numpy(), ns.cpu().numpy()


@pytest.mark.parametrize("S", [1, 63, 64, 193])
def test_column_block_widths_agree(ops, S):
    """33 heads run in 32-column blocks, up to 32 in 16-column blocks; a head's results are the
    same bits in both (the blocks' columns are independent and summed alike)."""
    Hv = 33
    args = _inputs(Hv, S, seed=S)
    out, ns = _run(ops, args, 64)
    for n in (1, 9, 32):
        o, s = _run(ops, [a[:a.shape[0] // Hv * n] for a in args], 64)
        assert np.array_equal(o, out[:n * S]) and np.array_equal(s, ns[:n * 128])


@pytest.mark.parametrize("Hv,S,C,seed", [(12, 64, 64, 0), (12, 200, 16, 1), (48, 130, 64, 2),
                                         (4, 1, 64, 3), (3, 1000, 64, 4), (2, 63, 16, 5)])
def test_chunked_prefill_matches_oracle(ops, Hv, S, C, seed):
    args = _inputs(Hv, S, seed)
    out, ns = _run(ops, args, C)
    ro, rs = oc.chunked_prefill(*args, 64)
    assert_rel_close(out, ro, name="out")
    assert_rel_close(ns, rs, name="new_state")


def test_full_size_heads_match_oracle(ops):
    """The 27B layer's width at a 4096-token prompt (48 v-heads x 64 chunks): the first and the
    last head against the float64 oracle, at the op's 2e-3 bar and at 1e-4 (the split bf16
    products keep the result fp32-class over all 64 chunks)."""
    Hv, S = 48, 4096
    g = torch.Generator(device="cuda").manual_seed(11)
    st = torch.randn(Hv * 128, 128, generator=g, device="cuda") * 0.05
    q, k, v = (torch.randn(Hv * S, 128, generator=g, device="cuda") for _ in range(3))
    a_log = torch.randn(Hv, 1, generator=g, device="cuda")
    dt = torch.randn(Hv, 1, generator=g, device="cuda") * 0.1
    a_in = torch.randn(Hv, S, generator=g, device="cuda")
    gate = (-torch.exp(a_log) * torch.nn.functional.softplus(a_in + dt)).reshape(-1, 1)
    beta = torch.sigmoid(torch.randn(Hv * S, 1, generator=g, device="cuda"))
    m = [torch.from_numpy(x).cuda() for x in oc.constants(64)]
    out, ns = ops.deltanet.chunked_prefill(st, q, k, v, gate, beta, *m)
    torch.cuda.synchronize()
    for h in (0, Hv - 1):
        rows, srows = slice(h * S, (h + 1) * S), slice(h * 128, (h + 1) * 128)
        args = [x[rows].cpu().numpy() for x in (q, k, v, gate, beta)]
        ro, rs = oc.chunked_prefill(st[srows].cpu().numpy(), *args, 64)
        o, s_ = out[rows].cpu().numpy(), ns[srows].cpu().numpy()
        assert_rel_close(o, ro, name=f"head {h} out")
        assert_rel_close(s_, rs, name=f"head {h} new_state")
        assert np.abs(o - ro).max() <= 1e-4 * np.abs(ro).max(), f"head {h} out"
        assert np.abs(s_ - rs).max() <= 1e-4 * np.abs(rs).max(), f"head {h} new_state"


def test_long_prompt_matches_oracle(ops):
    """16384 tokens (256 chunks, with a partial last one) on 2 heads: the state carried through
    the whole scan stays within 1e-4 of the float64 oracle."""
    args = _inputs(2, 16384 - 5, 12)
    out, ns = _run(ops, args, 64)
    ro, rs = oc.chunked_prefill(*args, 64)
    assert_rel_close(out, ro, name="out")
    assert_rel_close(ns, rs, name="new_state")
    assert np.abs(ns - rs).max() <= 1e-4 * np.abs(rs).max()


def test_c_abi_rejects_small_workspace(ops):
    """npn_deltanet_chunked_prefill checks its workspace before launching anything."""
    import npn_native
    Hv, S = 2, 130
    t = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in _inputs(Hv, S, 13)]
    out = torch.empty(Hv * S, 128, device="cuda")
    ns = torch.empty(Hv * 128, 128, device="cuda")
    n_ws = npn_native.query("npn_deltanet_chunked_workspace_size", Hv, S)
    assert n_ws == Hv * 3 * 34048
    ws = torch.empty(n_ws, dtype=torch.uint8, device="cuda")
    with pytest.raises(RuntimeError, match="status 4"):
        npn_native.call("npn_deltanet_chunked_prefill", *t, out, ns, Hv, S, ws, n_ws - 16,
                        npn_native.stream_of(out))
    npn_native.call("npn_deltanet_chunked_prefill", *t, out, ns, Hv, S, ws, n_ws,
                    npn_native.stream_of(out))
    torch.cuda.synchronize()
    ro, rs = oc.chunked_prefill(*[x.cpu().numpy() for x in t], 64)
    assert_rel_close(out.cpu().numpy(), ro, name="out")
    assert_rel_close(ns.cpu().numpy(), rs, name="new_state")


def test_identical_pad_rows(ops):
    args = _inputs(2, 192, 6, pad_from=15)
    out, ns = _run(ops, args, 64)
    assert np.all(np.isfinite(ns)) and np.all(np.isfinite(out))
    ro, rs = oc.recurrent(*args)
    assert_rel_close(out, ro, name="out")
    assert_rel_close(ns, rs, name="new_state")


def test_hf_vectors(ops):
    z = np.load(GOLDEN)
    for c in sorted({k.split("_")[0] for k in z.files}):
        f = lambda n: z[f"{c}_{n}"]
        out, ns = _run(ops, (f("state"), f("q"), f("k"), f("v"), f("g"), f("beta")), int(f("C")))
        assert_rel_close(out, f("out"), name=f"{c} out")
        assert_rel_close(ns, f("new_state"), name=f"{c} new_state")


def test_rejects_bad_shapes(ops):
    args = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in _inputs(2, 10, 7)]
    m = [torch.from_numpy(x).cuda() for x in oc.constants(16)]
    with pytest.raises(RuntimeError):
        ops.deltanet.chunked_prefill(args[0][:200], *args[1:], *m)       # state rows % 128
    with pytest.raises(RuntimeError):
        ops.deltanet.chunked_prefill(*args, m[0][:, :8], m[1], m[2])      # constants not [C, C]
