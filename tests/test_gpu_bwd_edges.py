"""GPU parity of the backward kernels at the edges of their tiles, against the fp64 oracle.

The gradient kernel works on 16-token row blocks of 64-token chunks and forms dbeta without
dividing by beta (beta = 0 is a padding token's gate); the layer tail's conv adjoint gives a
wavefront 16 tokens and masks the taps at every sequence start.  Tolerances as in
tests/test_gpu_bwd.py and tests/test_gpu_layer_bwd.py, whose inputs these reuse.
"""
import numpy as np
import pytest

from oracle import gdn_oracle as O

import test_gpu_bwd as core
import test_gpu_layer_bwd as layer

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,dk,dv,dtype", [
    (15, 128, 128, "bf16"), (16, 128, 64, "bf16"), (17, 64, 128, "bf16"), (63, 128, 128, "bf16"),
    (65, 128, 128, "bf16"), (79, 64, 64, "bf16"), (17, 64, 64, "f32"), (65, 32, 64, "f32"),
])
def test_core_backward_at_row_block_edges(T, dk, dv, dtype):
    core.say(f"bwd edges T={T} dk={dk} dv={dv} {dtype}")
    args = core.make(7000 + T + dk, 2, T, 2, 4, dk, dv, dtype)
    core.check(core.run_gpu(*args, dtype), core.run_ref(*args, dtype), dtype)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_core_backward_with_zero_and_one_beta(dtype):
    """dbeta of a token with beta = 0 is its derivative, not 0 / 0."""
    core.say(f"bwd beta in {{0, 1}} {dtype}")
    args = list(core.make(7100, 1, 90, 1, 2, 64, 64, dtype))
    beta = args[4]
    beta[:, ::3] = 0.0
    beta[:, 1::3] = 1.0
    got = core.run_gpu(*args, dtype)
    assert all(np.isfinite(x).all() for x in got)
    core.check(got, core.run_ref(*args, dtype), dtype)


@pytest.mark.parametrize("dk", [64, 32])
def test_core_backward_of_fast_decay_keeps_the_diagonal(dk):
    """Gates summing to -3,800 in a chunk leave Gamma its unit diagonal alone, so dq is one
    product chain of four split operands (dO, V_new, dP, K) of relative error 2^-17 each: 2^-16
    together, in quadrature.  A diagonal off by the rounding of G gives 4e-5 and more."""
    core.say(f"bwd fast decay dk={dk}")
    args = list(core.make(7150 + dk, 2, 192, 1, 2, dk, 64, "f32"))
    args[3] = (-60 - np.random.default_rng(7150).uniform(0, 1, args[3].shape)).astype(np.float32)
    got, ref = core.run_gpu(*args, "f32"), core.run_ref(*args, "f32")
    assert all(np.isfinite(x).all() for x in got)
    core.check(got, ref, "f32", skip=("dg",))  # dg is a difference of sums that are all but equal
    err = np.linalg.norm(got[0] - ref[0]) / np.linalg.norm(ref[0])
    assert err < 2.0 ** -16, err


@pytest.mark.parametrize("dk", [128, 64])
def test_bf16_backward_of_fast_decay_keeps_the_diagonal(dk):
    """The same for the reverse scan's P, which bf16 inputs form there: with Gamma's unit
    diagonal alone dbeta_i is scale (q_i . k_i) (dO_i . v_i), P and dO split to 2^-17 each and
    v exact.  q and k rows hold 64 entries of +-1, so that their normalised rows are exact."""
    core.say(f"bwd fast decay bf16 dk={dk}")
    args = list(core.make(7160 + dk, 2, 192, 1, 2, dk, 64, "bf16"))
    for n in (0, 1):
        args[n] = np.sign(args[n])
        args[n][..., 64:] = 0
    args[3] = (-60 - np.random.default_rng(7160).uniform(0, 1, args[3].shape)).astype(np.float32)
    got, ref = core.run_gpu(*args, "bf16"), core.run_ref(*args, "bf16")
    assert all(np.isfinite(x).all() for x in got)
    core.check(got, ref, "bf16", skip=("dg",))  # dg is a difference of sums that are all but equal
    err = np.linalg.norm(got[4] - ref[4]) / np.linalg.norm(ref[4])
    core.say(f"  dbeta {err:.2e}")
    assert err < 2.0 ** -16, err


@pytest.mark.parametrize("dk,dtype", [(128, "bf16"), (64, "bf16"), (64, "f32")])
def test_packed_documents_of_one_length_agree_with_the_batch(dk, dtype):
    """Three documents of one length, packed, take the widths of the batch of three and give
    its gradients bit for bit (24 heads: more 16-column workgroups than the chip has CUs)."""
    core.say(f"bwd packed widths dk={dk} {dtype}")
    N, T, Hk, Hv = 3, 150, 8, 24
    args = core.make(7180 + dk, N, T, Hk, Hv, dk, 64 if dk == 64 else 128, dtype)
    batch = core.run_gpu(*args, dtype)
    row = [x.reshape(1, N * T, *x.shape[2:]) for x in args[:5]] + [args[5], args[6].reshape(1, N * T, *args[6].shape[2:]), args[7]]
    packed = core.run_gpu(*row, dtype, np.arange(N + 1, dtype=np.int32) * T)
    for a, b in zip(batch, packed):
        assert np.array_equal(a.reshape(b.shape), b)


@pytest.mark.parametrize("T,dk,dv,dtype", [(64, 64, 64, "f32"), (40, 32, 128, "f32"),
                                           (64, 128, 128, "bf16"), (40, 64, 64, "bf16")])
def test_gate_gradient_takes_the_state_in_fp32(T, dk, dv, dtype):
    """Without decay, writes (beta = 0) or a cotangent of o, dg is the sum of dS * S.  Every
    entry of S is 1 + 2^-9 + 2^-17, whose last bit two bf16 parts do not hold: 2^-17 of the
    sum.  In fp32 a lane's products and sums are exact, and the ten additions over lanes and
    wavefronts leave at most 10 * 2^-24."""
    core.say(f"bwd dg from the state T={T} dk={dk} dv={dv} {dtype}")
    q, k, v, g, beta, S0, do, dht = core.make(7170 + T + dk, 1, T, 1, 2, dk, dv, dtype)
    S0[:] = 1 + 2.0 ** -9 + 2.0 ** -17
    dht[:] = 0.5
    args = (q, k, v, 0 * g, 0 * beta, S0, 0 * do, dht)
    got, ref = core.run_gpu(*args, dtype), core.run_ref(*args, dtype)
    core.check(got, ref, dtype, skip=("dq",))  # zero
    err = core.rel(got[3], ref[3])
    core.say(f"  dg {err:.2e}")
    assert err < 10 * 2.0 ** -24, err


@pytest.mark.parametrize("lens,Hk,Hv,dk,dv", [
    ([1], 1, 1, 64, 64),                              # one token; 192 channels (not a multiple of 256)
    ([40], 1, 1, 64, 64),                             # the same over three wavefronts' rows, each with a first one
    ([2, 1, 1, 3], 1, 2, 64, 64),                     # sequences shorter than the conv window
    ([15, 1, 2, 14, 17, 15], 1, 1, 64, 128),          # starts on both sides of 16-token edges
    ([62, 1, 1, 3, 64, 0, 5], 2, 4, 128, 128),        # starts around a 64-token edge, one empty
    ([0, 0, 17, 0, 0, 0, 30] + [0] * 40, 1, 2, 64, 64),  # empty ones everywhere, the row filled up with them
])
def test_layer_backward_at_conv_edges(lens, Hk, Hv, dk, dv):
    layer.say(f"layer bwd edges lens={lens}")
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    dims = dict(Hk=Hk, dk=dk, Hv=Hv, dv=dv)
    d = layer.make(7200 + len(lens), 1, int(cu[-1]), Hk, Hv, dk, dv, N=len(lens))
    layer.check(layer.run_gpu(d, dims, cu=cu), layer.run_ref(d, dims, cu=cu))


@pytest.mark.parametrize("B,T", [(3, 16), (2, 19), (5, 1)])
def test_layer_backward_of_batch_rows_at_conv_edges(B, T):
    layer.say(f"layer bwd edges B={B} T={T}")
    dims = dict(Hk=1, dk=64, Hv=2, dv=64)
    d = layer.make(7300 + T, B, T, 1, 2, 64, 64)
    layer.check(layer.run_gpu(d, dims), layer.run_ref(d, dims))


@pytest.mark.parametrize("B,Hk,Hv,dk,dv,dtype", [
    (1, 2, 4, 64, 64, "f32"), (8, 8, 16, 64, 64, "f32"),      # 16- and 32-column workgroups
    (8, 8, 16, 64, 64, "bf16"), (8, 16, 32, 64, 64, "bf16"),  # 32- and 64-column
    (4, 8, 16, 128, 128, "bf16"), (8, 8, 16, 128, 128, "bf16"),
])
def test_scans_at_every_workgroup_width(B, Hk, Hv, dk, dv, dtype):
    """Sequences x value heads x dv / 16 chooses the scans' 16-, 32- or 64-column workgroups;
    the suite's small shapes all take the narrowest."""
    from omegalax_amd import chunk_gated_delta_rule
    core.say(f"scan widths B={B} Hk={Hk} Hv={Hv} dk={dk} dv={dv} {dtype}")
    T = 150
    q, k, v, g, beta, S0, do, dht = args = core.make(7400 + B + Hv + dk, B, T, Hk, Hv, dk, dv, dtype)
    got = core.run_gpu(*args, dtype)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    o, fs = chunk_gated_delta_rule(core.dev(q, tdt), core.dev(k, tdt), core.dev(v, tdt), core.dev(g),
                                   core.dev(beta), initial_state=core.dev(S0), output_final_state=True)
    # the last batch row against the oracle (rows are independent)
    row = [x[-1:] for x in args]
    core.check([x[-1:] for x in got], core.run_ref(*row, dtype), dtype)
    act = O.round_bf16 if dtype == "bf16" else (lambda x: x)
    ro, rs = O.chunk_gated_delta_rule(*row[:5], initial_state=row[5], output_final_state=True, act_round=act)
    assert core.rel(core.np_(o[-1:]), ro) < (core.BF16_TOL if dtype == "bf16" else core.F32_TOL)
    assert core.rel(core.np_(fs[-1:]), rs) < core.F32_TOL
