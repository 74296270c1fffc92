"""Expert selection of several tokens (kq_hip_moe_execute_quantized): the
candidates' exact chains must give the CPU's ids in the CPU's order, whatever
lies near the selection's edge."""
import numpy as np
import pytest

import kq_hip
import kq_oracle
import kq_synth as S
from test_gpu_moe import ROLES, near_tie

from conftest import assert_close, oracle_threads

import exact

pytestmark = pytest.mark.gpu

I = 256  # intermediate size


@pytest.fixture(scope="module")
def ctx():
    c = kq_hip.Context(0)
    yield c
    c.close()


def run(ctx, w, H, E, K, x):
    T = x.shape[0]
    cfg = kq_hip.MoeConfig(H, E, K, I, I)
    n = cfg.scratch_bytes(T)
    bufs = {k: ctx.upload(v) for k, v in w.items()}
    rest = scratch, dx, dout, dids = (ctx.alloc(n), ctx.upload(x), ctx.alloc(T * H * 4),
                                      ctx.alloc(T * K * 4))
    try:
        ctx.moe_execute(cfg, kq_hip.moe_weights(bufs), dx, T, dout, dids, scratch, n)
        return (ctx.download(dout, np.float32, T * H).reshape(T, H),
                ctx.download(dids, np.uint32, T * K).reshape(T, K))
    finally:
        for b in list(bufs.values()) + list(rest):
            b.close()
        cfg.close()


def oracle_ids(H, E, K, router, x):
    dims = dict(hidden=H, experts=E, top_k=K, inter=1, shared_inter=1)
    return np.stack([kq_oracle.moe_route(dims, (kq_oracle.F32, router), r)[2] for r in x])


PATTERNS = ["random", "duplicates", "triples", "zero", "near-tie", "quantised"]


@pytest.mark.parametrize("H,E,K,T,pattern", [
    (*shape, p) for shape in ((256, 24, 3, 2), (512, 64, 12, 19), (1024, 130, 8, 67),
                              (2048, 512, 10, 33), (2560, 512, 10, 201), (256, 1000, 32, 130),
                              (512, 600, 10, 900), (1024, 24, 3, 2), (1024, 1000, 32, 130))
    for p in PATTERNS] + [(2560, 512, 10, 1281, "random"), (1024, 512, 10, 1300, "zero"),
                          (2048, 600, 10, 900, "triples")])
def test_ids_exact(ctx, H, E, K, T, pattern):
    # from 1,024 columns or 524,288 logits on the candidate route, the chains
    # of every expert below: one and more tokens per tile
    # of the approximate logits (64 x 64, and 64 x 256 from 40 of those on: 900
    # and 1,281 tokens), expert counts off the tiles and above 512, up to 32
    # selected; tokens of zeros, of tiny and of large activations (whose lower
    # probabilities underflow) among the others
    key = S.stream_key(S.W_MOE, 60, H + E, K)
    w = S.moe_weights(S.W_MOE + 60, H, E, I, I)
    router = S.normal_f32(key, E * H, 0.02).reshape(E, H)
    x = S.normal_f32(key ^ 1, T * H).reshape(T, H)
    rng = np.random.default_rng(E + T)
    if pattern == "duplicates":
        # equal logits inside and across the selection's edge
        router[rng.integers(0, E, E // 3)] = router[rng.integers(0, E, E // 3)]
    elif pattern == "triples":
        # equal logits across the edge of every token, few enough to decide
        router[1::3] = router[0::3][: len(router[1::3])]
        router[2::3] = router[0::3][: len(router[2::3])]
        router = router[rng.permutation(E)]
    elif pattern == "zero":
        router[:] = 0.0
    elif pattern == "quantised":
        # logits on a coarse grid: many exact ties
        router = np.rint(router * 40).astype(np.float32)
        x = np.sign(np.rint(x)).astype(np.float32)
    elif pattern == "near-tie":
        c = rng.choice([0.0, 1e-4, 1e-3, 0.02, 0.3], T)
        x = np.stack([near_tie(router, x[t], K, c[t]) for t in range(T)])
    if T > 6:
        x[1] = 0.0
        x[3] *= np.float32(1e-30)
        x[4] *= np.float32(1e6)
        x[5] *= np.float32(3e4)
    w["router"] = router.reshape(-1)
    _, ids = run(ctx, w, H, E, K, x)
    want = oracle_ids(H, E, K, router, x)
    bad = np.flatnonzero((ids != want).any(axis=1))
    assert bad.size == 0, (bad[:5], ids[bad[:2]], want[bad[:2]])


@pytest.mark.parametrize("H", [512, 1024])
def test_output_with_ties(ctx, H):
    # the layer's output where some tokens tie: weights and combine order are
    # those of the ids
    E, K, T = 48, 5, 40
    w = S.moe_weights(S.W_MOE + 61, H, E, I, I)
    r = w["router"].reshape(E, H)
    r[7] = r[30]
    r[11] = r[12]
    x = S.normal_f32(S.stream_key(S.W_MOE, 61), T * H).reshape(T, H)
    out, ids = run(ctx, w, H, E, K, x)
    dims = dict(hidden=H, experts=E, top_k=K, inter=I, shared_inter=I)
    ref, tr = kq_oracle.moe_execute(dims, {k: (t, w[k]) for k, t in ROLES.items()}, x, trace=True,
                                    threads=oracle_threads())
    assert np.array_equal(ids, tr["selected_ids"])
    assert_close(out, ref, exact=exact.moe(dims, ROLES, w, x, ids))


@pytest.mark.parametrize("H", [512, 1024])
@pytest.mark.parametrize("where", ["activation", "router", "overflow"])
def test_fails_closed(ctx, where, H):
    E, K, T = 64, 6, 21
    w = S.moe_weights(S.W_MOE + 62, H, E, I, I)
    x = S.normal_f32(S.stream_key(S.W_MOE, 62), T * H).reshape(T, H)
    good = run(ctx, w, H, E, K, x)
    bad_w, bad_x = dict(w), x.copy()
    if where == "activation":
        bad_x[20, H - 1] = np.inf
    else:
        r = w["router"].copy().reshape(E, H)
        r[63, 0] = np.nan if where == "router" else 1.0
        if where == "overflow":  # a logit past binary32
            r[5, :] = 3e37
            bad_x[3, :] = 100.0
        bad_w["router"] = r.reshape(-1)
    with pytest.raises(kq_hip.KqError) as e:
        run(ctx, bad_w, H, E, K, bad_x)
    assert e.value.name == "NUMERIC_DOMAIN"
    again = run(ctx, w, H, E, K, x)
    assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(good, again))
