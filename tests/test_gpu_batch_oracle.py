"""Batched decode (t2r_decode_batch) against the CPU restatement, row by row: each slot's cache holds the
oracle's prefill of a prompt of its own length, one batched step runs every slot at its position, and
every row's logits and new KV row equal OracleModel.forward on that slot's cache. The shapes reach every
instantiation of the grouped-query attention kernel (k_attn_gqa<hd/16, OPT, GW>): head dims 64 and 128,
groups of 2, 3 and 4 query heads, with and without the HF options, K and V per channel among them, at one
query head a workgroup (few rows) and at two (four-head groups of more than 256 heads over all rows)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def shape(name):
    import t2r_amd.config as C
    # hd 128 with four-head groups (no measured config has it): C3's shape with 4 KV heads, 4 layers
    g4 = C.C3.with_(name="c3-g4", kv_heads=4, layers=4, prompt_len=64)
    table = {
        "c4-llama3.2-1b": C.C4,                                            # hd 64, G 4: <4, false, 1>
        "c2-smollm2-135m": C.C2,                                           # hd 64, G 3: <4, false, 1>
        "c3-qwen3-0.6b": C.C3,                                             # hd 128, G 2: <8, false, 1>
        "c3-g4": g4,                                                       # hd 128, G 4: <8, false, 1>
        "c4-llama3.2-1b-hf": C.hf_options(C.C4),                           # <4, true, 1>: qsum, K per channel
        "c3-g4-hf": C.hf_options(g4),                                      # <8, true, 1>
        "c2-kv": C.C2.with_(name="c2-kv", kv_channel="kv", layers=6),      # <4, true, 1>: K and V per channel
        "c4-v": C.C4.with_(name="c4-v", kv_channel="v", attn_norm="qsum", layers=4),   # <4, true, 1>: V per channel
    }
    return table[name]


@pytest.mark.parametrize("name,lens", [("c4-llama3.2-1b", [5, 37, 70, 100]), ("c2-smollm2-135m", [3, 40, 66]),
                                       ("c3-qwen3-0.6b", [9, 50]), ("c3-g4", [7, 33, 64]),
                                       ("c4-llama3.2-1b-hf", [6, 45]), ("c3-g4-hf", [12, 40]),
                                       ("c2-kv", [4, 31, 57]), ("c4-v", [8, 65])])
def test_decode_batch_rows_vs_oracle(name, lens):
    import torch
    from oracle import OracleModel
    from t2r_amd import weights as W
    from t2r_amd.model import ResidentModel
    import t2r_amd.config as C
    cfg = shape(name)
    # the measured configs' recorded KV scales; the others calibrated on 32 prompt tokens (per channel
    # where the config says)
    kv = None if cfg.name in C.CONFIGS else W.calibrate_kv(cfg, tokens=cfg.prompt()[:32])
    qm = W.QuantModel(cfg, kv_scales=kv)
    om = OracleModel(qm)
    B = len(lens)
    rng = np.random.default_rng(31)
    prompts = [rng.integers(0, cfg.vocab, n).tolist() for n in lens]
    nxt = [int(rng.integers(0, cfg.vocab)) for _ in lens]
    rm = ResidentModel(qm, max_rows=B)
    kc, vc = rm.batch_caches(B)
    want, rows = [], []
    for b, p in enumerate(prompts):
        om.reset()
        om.prefill(p)
        kc[b].copy_(torch.from_numpy(om.kc))
        vc[b].copy_(torch.from_numpy(om.vc))
        want.append(om.forward(nxt[b], lens[b]))
        rows.append((om.kc[:, lens[b]].copy(), om.vc[:, lens[b]].copy()))
    print(f"{name}: B = {B} at positions {lens}", flush=True)
    got = rm.decode_batch(nxt, lens, kc, vc).cpu().numpy()
    for b in range(B):
        assert np.array_equal(got[b].view(np.uint32), want[b].view(np.uint32)), f"{name} row {b} at {lens[b]}"
        assert np.array_equal(kc[b, :, lens[b]].cpu().numpy(), rows[b][0]), f"K row {b}"
        assert np.array_equal(vc[b, :, lens[b]].cpu().numpy(), rows[b][1]), f"V row {b}"
    rm.close()


def small(name, hd, seq=2048, **kw):
    """Four-head groups at C4's heads (32, 8 KV heads) or, at head dim 128, 16 and 4; small elsewhere."""
    import t2r_amd.config as C
    h = 32 if hd == 64 else 16
    cfg = C.ModelConfig(name, dim=256, hidden=256, layers=2, heads=h, kv_heads=h // 4, head_dim=hd, vocab=512, seq_len=seq,
                        theta=5e5, qk_norm=hd == 128, weight_std=None, gain_std=0.1, emb_scale=4.0, seed_w=61, seed_p=62,
                        prompt_len=32)
    return (C.hf_options(cfg) if kw.pop("hf", False) else cfg).with_(**kw).validate()


# rows H on both sides of 256, and the kernel each runs; the caches hold random int8 rows, the positions lie at
# the ends of 32-key tiles, 1024-key passes and the cache
@pytest.mark.parametrize("hd,kw,B,kernel", [
    (64, {}, 8, "k_attn_gqa<4, false, 1>"), (64, {}, 9, "k_attn_gqa<4, false, 2>"), (64, dict(D=8), 19, "k_attn_gqa<4, false, 2>"),
    (64, dict(hf=True), 8, "k_attn_gqa<4, true, 1>"), (64, dict(hf=True), 9, "k_attn_gqa<4, true, 2>"),
    (64, dict(kv_channel="kv"), 10, "k_attn_gqa<4, true, 2>"), (64, dict(kv_channel="v", attn_norm="qsum"), 11, "k_attn_gqa<4, true, 2>"),
    (64, dict(seq=8192), 9, "k_attn_gqa<4, false, 2>"),
    (128, {}, 16, "k_attn_gqa<8, false, 1>"), (128, {}, 17, "k_attn_gqa<8, false, 2>"),
    (128, dict(hf=True), 17, "k_attn_gqa<8, true, 2>"), (128, dict(kv_channel="kv", D=8), 18, "k_attn_gqa<8, true, 2>"),
    (128, dict(seq=8192, hf=True), 17, "k_attn_gqa<8, true, 2>")])
def test_decode_batch_group_split(kernels, hd, kw, B, kernel):
    import torch
    from oracle import OracleModel
    from t2r_amd import weights as W
    from t2r_amd.model import ResidentModel
    cfg = small(f"small-g4-{hd}", hd, **kw)
    S = cfg.seq_len
    qm = W.QuantModel(cfg, kv_scales=W.calibrate_kv(cfg, tokens=cfg.prompt()[:32]))
    om, rm = OracleModel(qm), ResidentModel(qm, max_rows=B)
    rng = np.random.default_rng(17 + B)
    pos = ([S - 1, 0, 1024, 31, 1023, 32, 1500, 1, 63] + rng.integers(2, S - 1, B).tolist())[:B]
    toks = rng.integers(0, cfg.vocab, B).tolist()
    kc, vc = rm.batch_caches(B)
    want, rows = [], []
    for b, p in enumerate(pos):
        for t, o in ((kc, om.kc), (vc, om.vc)):
            o[:, :p] = np.clip(np.rint(rng.standard_normal((cfg.layers, p, cfg.kv_dim)) * 28), -127, 127)
            t[b, :, :p].copy_(torch.from_numpy(o[:, :p].astype(np.int8)))
        want.append(om.forward(toks[b], p))
        rows.append((om.kc[:, p].copy(), om.vc[:, p].copy()))
    print(f"{cfg.name} {kw}: B = {B} at positions {pos}", flush=True)
    got = rm.decode_batch(toks, pos, kc, vc).cpu().numpy()
    for b, p in enumerate(pos):
        assert np.array_equal(got[b].view(np.uint32), want[b].view(np.uint32)), f"row {b} at {p}"
        assert np.array_equal(kc[b, :, p].cpu().numpy(), rows[b][0]), f"K row {b}"
        assert np.array_equal(vc[b, :, p].cpu().numpy(), rows[b][1]), f"V row {b}"
    ran = kernels(lambda: rm.decode_batch(toks, pos, kc, vc))
    assert not ran or kernel in ran, ran
    rm.close()
