"""GPU parity of the forward kernels at the edges of their dispatch, against the fp64 oracle.

The layer scan takes 16-, 32- or 64-column workgroups and either applies the gated norm itself
or leaves it to the epilogue kernel, by the number of sequences x value heads x columns; the
prep gives a key head's value heads to one workgroup or to several, by the number of chunks.
The suite's small shapes all take the first of each.  Tolerances as in
tests/test_gpu_layer.py and tests/test_gpu_prefill.py, whose inputs these reuse.
"""
import numpy as np
import pytest

from omegalax_amd import workloads as W

import test_gpu_layer as layer
import test_gpu_prefill as core

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ROWS = ("mixed_qkv", "z", "a", "b")


def check_rows(B, T, dims, rows, seed):
    """A batch on the GPU, the given rows of it (rows are independent) against the oracle."""
    d = W.layer_inputs(B, T, **dims, seed=seed)
    S0 = (0.02 * np.random.default_rng(seed).standard_normal(
        (B, dims["Hv"], dims["dk"], dims["dv"]))).astype(np.float32)
    out, S, conv = layer.gpu_prefill(W.to_device(d), dims, None, S0)
    for n in rows:
        one = {k: (v[n:n + 1] if k in ROWS else v) for k, v in d.items()}
        ref, S_ref, conv_ref = layer.ref_prefill(one, dims, None, S0[n:n + 1])
        assert layer.rel(layer.np_(out[n:n + 1]), ref) < layer.BF16_TOL
        assert layer.rel(layer.np_(S[n:n + 1]), S_ref) < layer.STATE_TOL
        assert np.array_equal(layer.np_(conv[n:n + 1]), conv_ref)


@pytest.mark.parametrize("T", [1, 64, 65, 129, 200, 257, 385, 640])
@pytest.mark.parametrize("B,Hk,Hv,dv", [
    (1, 1, 2, 128),    # 16-column workgroups
    (16, 2, 4, 128),   # 32-column, 256 workgroups
])
def test_layer_scan_pipeline_depth(B, Hk, Hv, dv, T):
    """Sequences of one to ten chunks: the exchange and finalizing wavefronts run up to four
    chunks behind the scan and drain it after the last one."""
    layer.say(f"layer scan depth B={B} Hv={Hv} T={T}")
    check_rows(B, T, dict(Hk=Hk, dk=128, Hv=Hv, dv=dv), (0, B - 1), 8000 + T)


@pytest.mark.parametrize("B,Hk,Hv,dk,dv", [
    (8, 1, 4, 128, 256),    # 32-column workgroups, eight to a value head
    (9, 1, 4, 128, 256),    # 64-column, less than one round
    (10, 1, 4, 128, 128),   # 32-column, less than one round
    (33, 1, 4, 128, 128),   # 64-column, past one round, groups not a multiple of eight
    (40, 1, 4, 128, 128),   # 64-column, past one round
    (24, 1, 3, 128, 256),   # 64-column, four to a value head, past one round
    (40, 2, 4, 128, 64),    # one workgroup to a value head
    (40, 1, 4, 64, 128),    # dk = 64
])
def test_layer_scan_at_every_workgroup_width(B, Hk, Hv, dk, dv):
    layer.say(f"layer scan widths B={B} Hk={Hk} Hv={Hv} dk={dk} dv={dv}")
    check_rows(B, 460, dict(Hk=Hk, dk=dk, Hv=Hv, dv=dv), (0, B // 2, B - 1), 8100 + B + dv)


@pytest.mark.parametrize("N", [
    10,   # 16-column workgroups past one round of the chip: the epilogue kernel
    24,   # 32-column, past one round
    25,   # the same, groups not a multiple of eight: the epilogue kernel
    40,   # 64-column, past one round
])
def test_layer_scan_of_packed_sequences_past_one_round(N):
    """Packed sequences, some of them empty, from their own states, longest first."""
    layer.say(f"layer scan: {N} packed sequences")
    dims = dict(Hk=1, dk=128, Hv=4, dv=128)
    rng = np.random.default_rng(8200 + N)
    lens = rng.integers(0, 1200, size=N)
    lens[[0, 7, N - 1]] = 0
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    d = W.layer_inputs(1, int(cu[-1]), **dims, seed=8201 + N)
    S0 = (0.02 * rng.standard_normal((N, 4, 128, 128))).astype(np.float32)
    out, S, conv = layer.gpu_prefill(W.to_device(d), dims, cu, S0)
    ref, S_ref, conv_ref = layer.ref_prefill(d, dims, cu, S0)
    assert layer.rel(layer.np_(out), ref) < layer.BF16_TOL
    assert layer.rel(layer.np_(S), S_ref) < layer.STATE_TOL
    assert np.array_equal(layer.np_(conv), conv_ref)


@pytest.mark.parametrize("Hv", [16, 24])
def test_packed_layer_rows_of_one_block_a_head_equal_the_batch(Hv):
    """dv = 64, more workgroups than CUs, eight chunks a sequence or more: the batch takes the
    fused scan, packed rows of 16 heads the epilogue kernel, of 24 the fused scan; bit for bit."""
    B, T = 24, 520
    layer.say(f"layer scan: one block a head, Hv={Hv}")
    dims = dict(Hk=8, dk=128, Hv=Hv, dv=64)
    d = W.layer_inputs(B, T, **dims, seed=8250 + Hv)
    S0 = (0.02 * np.random.default_rng(8250).standard_normal((B, Hv, 128, 64))).astype(np.float32)
    batch = layer.gpu_prefill(W.to_device(d), dims, None, S0)
    row = {k: (v.reshape(1, B * T, *v.shape[2:]) if k in ROWS else v) for k, v in d.items()}
    packed = layer.gpu_prefill(W.to_device(row), dims, np.arange(B + 1, dtype=np.int32) * T, S0)
    for a, b in zip(batch, packed):
        assert torch.equal(a.reshape(b.shape), b)


def test_layer_of_no_tokens_keeps_the_states():
    """T = 0 over more workgroups than the chip holds: no chunk to prepare, states copied."""
    layer.say("layer T=0")
    dims = dict(Hk=1, dk=128, Hv=4, dv=128)
    d = W.layer_inputs(40, 1, **dims, seed=8300)
    t = W.to_device({k: (v[:, :0] if k in ROWS else v) for k, v in d.items()})
    S0 = np.random.default_rng(8301).standard_normal((40, 4, 128, 128)).astype(np.float32)
    _, S, _ = layer.gpu_prefill(t, dims, None, S0)
    assert np.array_equal(layer.np_(S), S0)


@pytest.mark.parametrize("B,T,Hk,Hv,dtype", [
    (1, 70, 1, 1, "bf16"), (1, 70, 1, 4, "bf16"),   # one part; one value head to a part
    (1, 130, 1, 8, "bf16"), (1, 130, 1, 6, "f32"),
    (80, 300, 1, 6, "bf16"),                        # 400 chunks: two value heads to a part or more
    (40, 300, 1, 6, "f32"),
    (80, 300, 2, 4, "bf16"),                        # 800 chunk tasks
])
def test_prep_split_over_value_heads(B, T, Hk, Hv, dtype):
    core.say(f"prep split B={B} T={T} Hk={Hk} Hv={Hv} {dtype}")
    args = core.make(8400 + T + Hv, B, T, Hk, Hv, 64, 64, dtype)
    o, S = core.run_gpu(*args, dtype)
    for n in (0, B - 1):
        ro, rs = core.run_ref(*(x[n:n + 1] for x in args), dtype)
        tol = core.BF16_TOL if dtype == "bf16" else core.F32_OUT_TOL
        assert core.rel(o[n:n + 1], ro) < tol
        assert core.rel(S[n:n + 1], rs) < core.STATE_TOL


@pytest.mark.parametrize("B,T,Hk,Hv", [(1, 70, 1, 1), (1, 70, 2, 8), (1, 130, 1, 6), (70, 300, 1, 6)])
def test_layer_prep_split_over_value_heads(B, T, Hk, Hv):
    layer.say(f"layer prep split B={B} T={T} Hk={Hk} Hv={Hv}")
    check_rows(B, T, dict(Hk=Hk, dk=64, Hv=Hv, dv=64), (0, B - 1), 8500 + T + Hv)


@pytest.mark.parametrize("B,T,Hk,Hv", [
    (40, 1, 8, 16), (40, 63, 8, 16), (40, 64, 8, 16),   # one chunk a sequence
    (30, 150, 16, 64),                                  # three chunks: with them
    (12, 460, 16, 64),                                  # eight, records past 84 MiB, shared K and Q rows
    (9, 65, 16, 16),                                    # with loader wavefronts, for comparison
])
@pytest.mark.parametrize("path", ["core", "layer", "layer packed"])
def test_scan_of_64_columns_with_and_without_loader_wavefronts(B, T, Hk, Hv, path):
    """dk = 64, bf16: a sequence of the batch against the oracle, and bit for bit against the
    call of that sequence alone, whose 16-column workgroups have loader wavefronts."""
    layer.say(f"staging {path} B={B} T={T} Hk={Hk} Hv={Hv}")
    dims = dict(Hk=Hk, dk=64, Hv=Hv, dv=64)
    if path == "core":
        args = core.make(8600 + T + Hv, B, T, Hk, Hv, 64, 64, "bf16")
        o, S = core.run_gpu(*args, "bf16")
        one = [x[B - 1:] for x in args]
        o1, S1 = core.run_gpu(*one, "bf16")
        assert np.array_equal(o[B - 1:], o1) and np.array_equal(S[B - 1:], S1)
        ro, rs = core.run_ref(*one, "bf16")
        assert core.rel(o1, ro) < core.BF16_TOL and core.rel(S1, rs) < core.STATE_TOL
        return
    d = W.layer_inputs(B, T, **dims, seed=8600 + T + Hv)
    S0 = (0.02 * np.random.default_rng(T).standard_normal((B, Hv, 64, 64))).astype(np.float32)
    one = {k: (v[B - 1:] if k in ROWS else v) for k, v in d.items()}
    cu = None
    if path == "layer packed":
        d = {k: (v.reshape(1, B * T, *v.shape[2:]) if k in ROWS else v) for k, v in d.items()}
        cu = np.arange(B + 1, dtype=np.int32) * T
    got = [layer.np_(x) for x in layer.gpu_prefill(W.to_device(d), dims, cu, S0)]
    got[0] = got[0].reshape(B, T, -1)
    alone = [layer.np_(x) for x in layer.gpu_prefill(W.to_device(one), dims, None, S0[B - 1:])]
    for a, b in zip(got, alone):
        assert np.array_equal(a[B - 1:].reshape(b.shape), b)
    ref, S_ref, conv_ref = layer.ref_prefill(one, dims, None, S0[B - 1:])
    assert layer.rel(alone[0], ref) < layer.BF16_TOL and layer.rel(alone[1], S_ref) < layer.STATE_TOL
    assert np.array_equal(alone[2], conv_ref)


# more 64-column workgroups than the chip has CUs, eight chunks a sequence or more: the fused
# scan's workgroups take their places by ticket and wait for the other blocks of their head
TICKETED = dict(Hk=2, dk=128, Hv=8, dv=128)


def ticketed(B, T, seed):
    d = W.layer_inputs(B, T, **TICKETED, seed=seed)
    rng = np.random.default_rng(seed)
    S0 = (0.02 * rng.standard_normal((B, 8, 128, 128))).astype(np.float32)
    return d, W.to_device(d), S0


def test_ticketed_layer_scan_replays_under_graph_capture():
    """The tickets start from zero in every replay: fresh inputs copied into the captured
    buffers, with eager calls and synchronisations in between, equal the eager call and, on two
    sequences, the scan of one round, which takes no tickets."""
    B, T = 24, 520
    layer.say(f"ticketed layer scan under capture B={B} T={T}")
    _, t, S0 = ticketed(B, T, 8700)
    layer.gpu_prefill(t, TICKETED, None, S0)
    from omegalax_amd import gdn_prefill
    names = ("mixed_qkv", "z", "a", "b", "conv_w", "A_log", "dt_bias", "norm_w")
    state = torch.from_numpy(S0).cuda()
    kw = dict(num_k_heads=2, head_k_dim=128, num_v_heads=8, head_v_dim=128, output_final_state=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = gdn_prefill(*(t[n] for n in names), initial_state=state, **kw)
    for rep in range(4):
        d2, t2, S2 = ticketed(B, T, 8710 + rep)
        for n in names:
            t[n].copy_(t2[n])
        state.copy_(torch.from_numpy(S2))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        want = layer.gpu_prefill(t2, TICKETED, None, S2)
        for a, b in zip(out, want):
            assert torch.isfinite(a.float()).all() and torch.equal(a, b)
        few = {n: (t2[n][:2].contiguous() if n in ROWS else t2[n]) for n in names}
        for a, b in zip(out, layer.gpu_prefill(few, TICKETED, None, S2[:2])):
            assert torch.equal(a[:2], b)


def test_ticketed_layer_scans_beside_each_other_and_other_work():
    """Two streams of ticketed scans and a third of matrix products share the CUs: waiting
    workgroups, at most three of each eighth of a grid, leave room for the ones they wait for."""
    B, T = 40, 520
    layer.say(f"ticketed layer scans on two streams B={B} T={T}")
    from omegalax_amd import gdn_prefill
    names = ("mixed_qkv", "z", "a", "b", "conv_w", "A_log", "dt_bias", "norm_w")
    kw = dict(num_k_heads=2, head_k_dim=128, num_v_heads=8, head_v_dim=128, output_final_state=True)
    ins = [ticketed(B, T, 8720 + i)[1] for i in range(2)]
    want = [gdn_prefill(*(t[n] for n in names), **kw) for t in ins]
    x = torch.randn(4096, 4096, device="cuda").bfloat16()
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(6):
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                got[i].append(gdn_prefill(*(ins[i][n] for n in names), **kw))
        with torch.cuda.stream(streams[2]):
            for _ in range(4):
                y = x @ x
    torch.cuda.synchronize()
    for i in range(2):
        for res in got[i]:
            for a, b in zip(res, want[i]):
                assert torch.equal(a, b)
