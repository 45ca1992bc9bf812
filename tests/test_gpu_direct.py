"""The one-launch attention form (attn_direct_kernel), taken for short contexts,
at the edges of its tiles (32 keys), waves (4), token pairs and value slices
(16 / 8 / 4 value blocks from 1 / 65 / 129 tokens on), against the oracle and
the split forms.  Tolerances are those of every parity test (gpu_util)."""
import numpy as np
import pytest
import torch

from moe_infer_amd import Cache, attn_decode, attn_prefill, attn_step, attn_step_proj, attn_verify
from oracle import oracle as O

from .conftest import f16
from .gpu_util import announce, assert_close, dev, host
from .test_gpu_rope import oracle_rows

pytestmark = pytest.mark.gpu
H, G, D = 16, 2, 256


def causal_case(past, n, call, groups=G, scale=None, poison=True):
    rng = np.random.default_rng(past * 1000 + n)
    heads = 8 * groups
    rows = past + n
    k, v = f16(rng, rows, groups * D), f16(rng, rows, groups * D)
    if scale is not None:
        k = (k.astype(np.float32) * scale(np.arange(rows))[:, None]).astype(np.float16)
    q, g = f16(rng, n, heads, D), f16(rng, n, heads, D)
    c = Cache(num_layers=1, num_q_heads=heads, num_kv_heads=groups, capacity=rows + 40)
    full = np.full((c.capacity, groups * D), np.nan, np.float16)  # stale rows hold anything
    full[:past] = k[:past]
    c.upload(0, full, full)
    if past:
        c.upload(0, k[:past], v[:past])
    announce(f"direct past={past} n={n} groups={groups}")
    out = call(c, 0, dev(q), dev(k[past:]), dev(v[past:]), past, gate=dev(g))
    ref = O.causal(q, k, v, past, gate=g) if groups == G else None
    kc, vc = c.download(0, rows=n, row0=past)
    np.testing.assert_array_equal(kc, k[past:])
    np.testing.assert_array_equal(vc, v[past:])
    c.close()
    return out, ref


def step(c, layer, q, k, v, past, gate):
    return attn_step(c, layer, q.reshape(-1), k, v, past, gate=gate.reshape(-1))


@pytest.mark.parametrize("past", [0, 1, 30, 31, 32, 127, 128, 1023, 1024])
def test_step(past):
    out, ref = causal_case(past, 1, step)
    assert_close(out, ref.reshape(-1), f"step past={past}")


@pytest.mark.parametrize("past,n", [(0, 2), (31, 3), (500, 4), (1260, 4), (1261, 4), (97, 5),
                                    (1720, 16), (300, 40),
                                    # groups of four tokens in one split launch, then the wide pass
                                    (1721, 16), (1501, 5), (1800, 6), (4000, 9), (3001, 7), (20475, 5),
                                    (20476, 5)])
def test_verify(past, n):
    out, ref = causal_case(past, n, attn_verify)
    assert_close(out, ref, f"verify past={past} n={n}")


@pytest.mark.parametrize("past,n", [(0, 17), (0, 64), (7, 65), (100, 128), (33, 129), (0, 333),
                                    (700, 299), (3000, 30), (3183, 17), (500, 511)])
def test_prefill(past, n):
    out, ref = causal_case(past, n, attn_prefill)
    assert_close(out, ref, f"prefill past={past} n={n}")


def test_rising_scores_move_the_reference_max():
    """Keys that grow with their row: every tile moves the reference max and
    rescales what was summed."""
    out, ref = causal_case(600, 3, attn_verify, scale=lambda r: 0.1 + r / 60.0)
    assert_close(out, ref, "rising scores")


@pytest.mark.parametrize("groups", [1, 4])
def test_other_head_counts_against_the_groups_apart(groups):
    """Eight query heads and their KV head do not depend on the others."""
    out, _ = causal_case(200, 5, attn_verify, groups=groups)
    rng = np.random.default_rng(200 * 1000 + 5)
    k, v = f16(rng, 205, groups * D), f16(rng, 205, groups * D)
    q, g = f16(rng, 5, 8 * groups, D), f16(rng, 5, 8 * groups, D)
    got = host(out).reshape(5, groups, 8, D)
    for i in range(0, groups, 2):
        lo, hi = i, min(i + 2, groups)
        pick = lambda a: np.concatenate([a.reshape(-1, groups, D)[:, j % groups] for j in (lo, hi - 1)], 1)
        heads = lambda a: np.concatenate([a.reshape(5, groups, 8, D)[:, j] for j in (lo, hi - 1)], 1)
        ref = O.causal(heads(q), pick(k), pick(v), 200, gate=heads(g)).reshape(5, 2, 8, D)
        assert_close(got[:, lo], ref[:, 0], f"groups={groups} head {lo}")
        assert_close(got[:, hi - 1], ref[:, 1], f"groups={groups} head {hi - 1}")


@pytest.mark.parametrize("rot", [0, 64, 128, 192, 256])
@pytest.mark.parametrize("pos", [0, 45])
def test_step_from_projections(rot, pos):
    rng = np.random.default_rng(rot + pos)
    qp = (rng.standard_normal((1, H, 2 * D)) * 3).astype(np.float32)
    kp = rng.standard_normal((1, G, D)).astype(np.float32)
    vp = rng.standard_normal((1, G, D)).astype(np.float32)
    w = torch.from_numpy((1 + 0.2 * rng.standard_normal(D)).astype(np.float32)).bfloat16()
    k, v = f16(rng, pos + 1, G * D), f16(rng, pos + 1, G * D)
    c = Cache(num_layers=1, capacity=256)
    if pos:
        c.upload(0, k[:pos], v[:pos])
    announce(f"direct proj pos={pos} rot={rot}")
    up = lambda a: torch.from_numpy(a).cuda()
    out = attn_step_proj(c, 0, up(qp), up(kp), up(vp), w.cuda(), w.cuda(), pos, rotary_dim=rot)
    qr, kr = oracle_rows(qp, kp, w, w, pos, rot)
    k[pos], v[pos] = kr.reshape(-1), vp.reshape(-1)
    ref = O.sigmoid_gate(O.decode(qr[0].astype(np.float16), k, v, pos + 1).reshape(-1),
                         qp[0, :, D:].reshape(-1))
    # outputs reach |v| ~ 4, where an f16 ulp is 2^-8
    assert_close(out.reshape(-1), ref, f"proj pos={pos} rot={rot}", atol=2.0 ** -8)


@pytest.mark.parametrize("n", [1, 6])
def test_same_as_the_split_forms(monkeypatch, n):
    """The routes differ in the order of their f32 sums and in which f16
    weights round: two f16 ulps of the largest output (below 1)."""
    rng = np.random.default_rng(n)
    rows = 700
    k, v = f16(rng, rows, G * D), f16(rng, rows, G * D)
    q, g = f16(rng, n, H, D), f16(rng, n, H, D)
    c = Cache(num_layers=1, capacity=rows)
    c.upload(0, k, v)
    c.set_pos(rows)
    call = ((lambda: attn_decode(c, 0, dev(q[0]), rows, gate=dev(g[0]))) if n == 1 else
            (lambda: attn_verify(c, 0, dev(q), None, None, rows - n, gate=dev(g))))
    one = host(call())
    monkeypatch.setenv("MI_ATTN_DECODE_MERGE", "0")
    monkeypatch.setenv("MI_ATTN_VERIFY_WIDE", "0")
    assert_close(one, host(call()), f"direct against split n={n}", atol=2.0 ** -10)


@pytest.mark.parametrize("past,n", [(516, 1), (1000, 1), (1000, 12), (3100, 24),
                                    (4300, 16), (6100, 12)])  # token groups, two tiles a wave
def test_weights_of_the_split_forms(monkeypatch, past, n):
    """Both forms take a tile's f16 weights against the tile's own max, so the
    weights are the same numbers but for a rounding of the exponent (2^-22 of a
    weight, 2^-11 apart: a few in ten thousand) and the f32 sums differ in their
    order only (1e-6 of an output, whose f16 values are 5e-4 to 1e-3 apart): few
    outputs round to another f16 value (0.3 %).  With weights against a running
    max a third to a half of them do, and the error against 64 bits is 3 to 10 % larger."""
    rng = np.random.default_rng(past + n)
    rows = past + n
    k, v = f16(rng, rows, G * D), f16(rng, rows, G * D)
    q, g = f16(rng, n, H, D), f16(rng, n, H, D)
    c = Cache(num_layers=1, capacity=rows)
    c.upload(0, k, v)
    c.set_pos(rows)
    announce(f"weights past={past} n={n}")
    call = ((lambda: attn_decode(c, 0, dev(q[0]), rows, gate=dev(g[0]))) if n == 1 else
            (lambda: attn_verify(c, 0, dev(q), None, None, past, gate=dev(g))))
    one = host(call())
    monkeypatch.setenv("MI_ATTN_DECODE_MERGE", "0")
    monkeypatch.setenv("MI_ATTN_VERIFY_WIDE", "0")
    other = host(call())
    share = float(np.mean(one != other))
    print(f"[parity] weights past={past} n={n}: {share:.4f} of the outputs differ", flush=True)
    assert share <= 0.1


@pytest.mark.parametrize("call,past,n", [
    (step, 0, 1), (step, 300, 1), (step, 5000, 1), (attn_verify, 40, 2), (attn_verify, 300, 4),
    (attn_verify, 300, 9), (attn_verify, 5000, 9), (attn_verify, 100, 40), (attn_prefill, 0, 17),
    (attn_prefill, 300, 64), (attn_prefill, 0, 100), (attn_prefill, 50, 333),
    (attn_prefill, 0, 1100), (attn_prefill, 3000, 100)])
@pytest.mark.parametrize("buffer", ["q", "gate"])
def test_output_in_the_buffer_of_an_input(call, past, n, buffer):
    """The output may take the place of the queries or of the gate, at any
    length: the calls that would run in one launch, where workgroups share
    their queries, go to the forms that write the output when all are read."""
    rng = np.random.default_rng(past + n)
    rows = past + n
    k, v = f16(rng, rows, G * D), f16(rng, rows, G * D)
    q, g = dev(f16(rng, n, H, D)), dev(f16(rng, n, H, D))
    c = Cache(num_layers=1, capacity=rows)
    if past:
        c.upload(0, k[:past], v[:past])
    announce(f"out in {buffer} {call.__name__} past={past} n={n}")
    args = (c, 0, q, dev(k[past:]), dev(v[past:]), past)
    ref = host(call(*args, gate=g)).reshape(n, H, D)
    out = q if buffer == "q" else g
    f = attn_step if call is step else call
    args = (c, 0, q.view(-1) if call is step else q) + args[3:]
    got = f(*args, gate=g.view(-1) if call is step else g,
            out=out.view(-1) if call is step else out)
    assert got.data_ptr() == out.data_ptr()
    # two forms of the same sums: an f16 ulp of outputs below 4
    assert_close(host(out).reshape(n, H, D), ref, f"out in {buffer}", atol=2.0 ** -9)


@pytest.mark.parametrize("past", [0, 300])
@pytest.mark.parametrize("buffer", ["k", "v"])
def test_output_over_the_new_rows(past, buffer):
    """The same for the new K / V rows, which every workgroup of a head reads
    when the launch appends them."""
    rng = np.random.default_rng(past)
    n = 16
    rows = past + n
    k, v = f16(rng, rows, G * D), f16(rng, rows, G * D)
    q = dev(f16(rng, n, H, D))
    c = Cache(num_layers=1, capacity=rows)
    if past:
        c.upload(0, k[:past], v[:past])
    announce(f"out over {buffer} past={past}")
    ref = host(attn_verify(c, 0, q, dev(k[past:]), dev(v[past:]), past))
    buf = torch.empty(n * H * D, dtype=torch.float16, device="cuda")
    new = buf[:n * G * D]
    new.copy_(dev((k if buffer == "k" else v)[past:]).view(-1))
    pair = (new, dev(v[past:])) if buffer == "k" else (dev(k[past:]), new)
    got = attn_verify(c, 0, q, *pair, past, out=buf.view(n, H, D))
    assert_close(got, ref, f"out over {buffer}", atol=2.0 ** -9)
    kc, vc = c.download(0, rows=n, row0=past)
    np.testing.assert_array_equal(kc, k[past:])
    np.testing.assert_array_equal(vc, v[past:])


@pytest.mark.parametrize("past,n", [(999, 513), (480, 640), (1030, 1024),
                                    (777, 777), (9000, 49), (12500, 40), (30000, 17)])
def test_split_k_with_row_blocks_of_different_length(monkeypatch, past, n):
    """The split-K prefill where the blocks of 16 tokens see different numbers
    of chunks (last chunks of more blocks than fit one at 480 + 640 and 777 +
    777 rows), in each order of its workgroups: against the prefill grid (the bound of that comparison in
    test_gpu_prefill) and, at rows on both sides of a block, the oracle."""
    rng = np.random.default_rng(past + n)
    rows = past + n
    k, v = f16(rng, rows, G * D), f16(rng, rows, G * D)
    q, g = f16(rng, n, H, D), f16(rng, n, H, D)
    c = Cache(num_layers=1, capacity=rows)
    c.upload(0, k[:past], v[:past])
    announce(f"split-K rows past={past} n={n}")
    args = (c, 0, dev(q), dev(k[past:]), dev(v[past:]), past)
    out = host(attn_prefill(*args, gate=dev(g)))
    monkeypatch.setenv("MI_ATTN_PREFILL_SPLIT", "0")
    assert_close(out, host(attn_prefill(*args, gate=dev(g))), "split-K against the grid", atol=1e-3)
    for i in (0, 15, 16, n // 2, n - 1):
        ref = O.decode(q[i], k[:past + i + 1], v[:past + i + 1], past + i + 1, gate=g[i])
        assert_close(out[i].reshape(-1), ref.reshape(-1), f"split-K row {i}")
