"""cwen_model_prefill (many positions per sweep over the weights) against
blocks of 16 through cwen_model_forward: the bar is bit equality of everything
that follows -- logits of a ragged block, of verify cycles that keep one
position of eight (so the conv history and a replayed prefix are read), and
of a second prompt part on top.

Sizes: prompts of two blocks, past one 64-position tile, ragged against it,
and past one workspace of 1024 positions; matrices whose rows are all split
over K, whole, and whole with a split remainder; every weight format that a
layer takes.
"""
import numpy as np
import pytest

from cwen_amd import synth

pytestmark = pytest.mark.gpu

SMALL = dict(n_layers=4, d_model=1024, d_ffn=2048, vocab=4096, n_head=4, n_kv_head=2, head_dim=256,
             n_rot_pairs=32, n_rot=64, gdn_nkh=2, gdn_nvh=4, gdn_dk=128, full_interval=4, max_ctx=1600,
             rope_theta=1e7, rms_eps=1e-6)
# 32-position tiles against 16-query attention groups of 6 heads; q/k/v heads as at the 27B shape
WIDE = dict(SMALL, d_model=5120, d_ffn=17408, vocab=2048, n_head=24, n_kv_head=4, gdn_nkh=16, gdn_nvh=48)
ODD = dict(SMALL, d_model=1536, d_ffn=1024, n_head=6, n_kv_head=1, gdn_nkh=4, gdn_nvh=12, full_interval=2)
# a context at which the attention's scores are made in several batches
LONG = dict(SMALL, n_layers=2, d_model=512, d_ffn=512, n_head=24, n_kv_head=4, full_interval=2, max_ctx=6400)


@pytest.fixture(scope="module")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cwen_amd import gpu
    yield gpu
    torch.cuda.synchronize()


def _after(m, cfg, toks):
    """Logits of what follows a prompt: a ragged block, two verify cycles that
    reject every draft, a serial step."""
    out = []
    m.forward(toks[:5])
    out.append(m.logits(5))
    for i in (5, 13):
        k, _ = m.verify(toks[i:i + 8])
        out += [m.logits(8), np.array([k])]
    m.verify(toks[21:22])
    out.append(m.logits(1))
    return out


def _same(a, b, what):
    for i, (x, y) in enumerate(zip(a, b)):
        assert np.isfinite(x).all()
        assert np.array_equal(x, y), (what, i, float(np.abs(x.astype(np.float64) - y).max()))


def _compare(gpu, m, cfg, n, n2=0, ragged=0):
    """n2: positions of a second prompt part; ragged: positions between the
    two, so that the second starts off any 16 or 32."""
    toks = synth.rng(9, n).integers(0, cfg["vocab"], n + ragged + n2 + 32).astype(np.int32)
    got = {}
    for how in ("blocks", "prefill"):
        m.reset()
        for a, b in ((0, n), (n, n + ragged), (n + ragged, n + ragged + n2)):
            if b - a == ragged:
                if ragged:
                    m.forward(toks[a:b], want_argmax=False)
            elif how == "prefill":
                m.prefill(toks[a:b])
            else:
                for i in range(a, b, 16):
                    m.forward(toks[i:i + 16], want_argmax=False)
            assert m.pos == b - 1
        got[how] = _after(m, cfg, toks[n + ragged + n2:])
    _same(got["prefill"], got["blocks"], (n, n2))


@pytest.mark.parametrize("name,n,n2", [("small", 32, 0), ("small", 48, 160), ("small", 1056, 32), ("odd", 80, 0),
                                       ("odd", 1024, 64), ("wide", 32, 0), ("wide", 336, 48), ("long", 6144, 80)])
def test_prefill_equals_blocks(gpu, name, n, n2):
    cfg = {"small": SMALL, "odd": ODD, "wide": WIDE, "long": LONG}[name]
    print(f"prefill {name}: {n} + {n2} positions", flush=True)
    ctx = gpu.Context(0)
    m = gpu.Model(ctx, **cfg)
    m.synth(3)
    _compare(gpu, m, cfg, n, n2)
    if n2:
        _compare(gpu, m, cfg, n, n2, ragged=5)
    m.free()


@pytest.mark.parametrize("streams", [1, 4])
@pytest.mark.parametrize("types", [("q8_0", "q6_k"), ("q5_k", "q4_1"), ("q4_0", "q8_0")])
def test_prefill_formats(gpu, types, streams):
    """ssm_out / wo and ffn_down in each format the layers take, in the products'
    two forms: one row stream per wave (1024 rows, 176 positions: at most 3 tiles
    of positions x 16 row blocks x 4 pieces), and four (2048 x 2048 at 528 positions:
    9 x 8 x 4 pieces, more workgroups than CUs; the last tile has 16 positions)."""
    print(f"prefill formats {types}, {streams} streams", flush=True)
    ctx = gpu.Context(0)
    cfg, n = (SMALL, 176) if streams == 1 else (dict(SMALL, d_model=2048, n_head=8, gdn_nkh=4, gdn_nvh=16), 528)
    m = gpu.Model(ctx, **cfg)
    tid = {"q8_0": gpu.T_Q8_0, "q6_k": gpu.T_Q6_K, "q5_k": gpu.T_Q5_K, "q4_1": gpu.T_Q4_1, "q4_0": gpu.T_Q4_0}
    gen = {"q8_0": synth.q8_0, "q6_k": synth.q6_k, "q5_k": synth.q5_k, "q4_1": synth.q4_1, "q4_0": synth.q4_gguf}
    for l, t, ty, data, sc, ne0, ne1 in synth.model_tensors(cfg, seed=4):
        if t in (gpu.SSM_OUT, gpu.ATTN_OUTPUT, gpu.FFN_DOWN):
            f = types[t == gpu.FFN_DOWN]
            ty, data, sc = tid[f], gen[f](5, ne1, ne0, key=100 * l + t), None
        m.set(l, t, ty, data, sc, ne0, ne1)
    _compare(gpu, m, cfg, n)
    m.free()


def test_prefill_after_a_weight_is_replaced(gpu):
    """The workspace of an earlier prompt part does not bound the pieces of K
    of a weight set later: ffn_down 4096 x 8192 takes 4 pieces as Q8_0 and,
    small enough for a workgroup per row group, 6 as Q4_0; no other matrix of
    this model needs as much room."""
    cfg = dict(SMALL, n_layers=2, d_model=4096, d_ffn=8192, vocab=1024, full_interval=2)
    H, I = cfg["d_model"], cfg["d_ffn"]
    ctx = gpu.Context(0)
    m = gpu.Model(ctx, **cfg)
    m.synth(3)
    for ty, data in ((gpu.T_Q8_0, synth.q8_0(6, H, I)), (gpu.T_Q4_0, synth.q4_gguf(6, H, I)), (gpu.T_Q8_0, synth.q8_0(7, H, I))):
        print(f"prefill with ffn_down of type {ty}", flush=True)
        for l in range(cfg["n_layers"]):
            m.set(l, gpu.FFN_DOWN, ty, data, None, I, H)
        _compare(gpu, m, cfg, 48)
    m.free()


def test_prefill_refuses(gpu):
    ctx = gpu.Context(0)
    m = gpu.Model(ctx, **SMALL)
    m.synth(3)
    m.reset()
    for bad in (np.zeros(17, np.int32), np.full(32, SMALL["vocab"], np.int32), np.zeros(1616, np.int32)):
        with pytest.raises(gpu.CwenError) as e:
            m.prefill(bad)
        assert e.value.rc == -1 and m.pos == -1
    m.prefill(np.zeros(1600, np.int32))          # the whole cache
    assert m.pos == 1599
    m.free()
