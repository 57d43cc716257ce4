"""What a user of this framework has it do, as cases that can be timed and checked: the DSA attention layer of a
serving engine in decode and in chunked prefill, its indexer, cache writes, absorbed projections and host-offloaded
rows, each through the entry point that the engine calls.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the inputs, caches and handles that the engine holds before the call
    run(state)           one call and its outputs
    work(case)           bytes and operations that the call cannot do without
    tolerance(case)      by how much the outputs of two correct implementations may differ
    exact(case, seed)    the outputs in 64 bits by plain torch (None: no such value)
"""
import math

import torch

from arcagi2_flashnext_dots3_amd import dsa, kernels, mla_fp8, shard_indexer, sparse_offload

SM = 192 ** -0.5          # softmax scale of the 128 + 64 wide MLA heads
BS = 64                   # positions per cache block
KV_SCALE = 0.25           # per-tensor scale of the fp8 (576-byte) cache
DEV = "cuda"
CHUNK = 1 << 17           # rows generated at a time


# ---------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # one user's token: launches and latency
        dict(name="decode_1", kind="attn", tokens=1, per_req=1, heads=128, ctx=4096, topk=2048, row=656),
        # a tensor-parallel rank (32 of 128 heads) over the per-tensor fp8 cache, an ordinary batch
        dict(name="decode_tp4_fp8", kind="attn", tokens=24, per_req=1, heads=32, ctx=20000, topk=2048, row=576),
        # the full decode batch on one GPU (the benchmark's default shape)
        dict(name="decode_64", kind="attn", tokens=64, per_req=1, heads=128, ctx=32768, topk=2048, row=656),
        # a prefill chunk of one long request
        dict(name="prefill", kind="attn", tokens=2048, per_req=2048, heads=128, ctx=16384, topk=2048, row=656),
        # a prefill chunk over the per-tensor fp8 cache holding several prompts, ragged, the first rows under topk
        dict(name="prefill_fp8", kind="attn", tokens=1455, per_req=485, heads=128, ctx=3001, topk=2048, row=576),
        # the indexer of a few users: paged key cache, logits, then the selection
        dict(name="index_paged_4", kind="index", path="paged", rows=4, per_req=1, ctx=16000, topk=2048, f16out=False),
        # the indexer of the full decode batch at the longest context (the benchmark's second indexer shape)
        dict(name="index_64", kind="index", path="shard", rows=64, per_req=1, ctx=131072, topk=2048, f16out=False),
        # the indexer of a prefill chunk over the request's gathered keys
        dict(name="index_prefill", kind="index", path="flat", rows=2048, per_req=2048, ctx=16384, topk=2048,
             f16out=False),
        # the cache writes of a prefill chunk: KV rows and indexer keys to random slots
        dict(name="cache_write", kind="write", tokens=8192, row=656),
        # the absorbed matmuls either side of the attention, full decode batch
        dict(name="projections_64", kind="proj", tokens=64, heads=128),
        # decode over host-resident compact rows behind an HBM hot set of a quarter of them
        dict(name="offload_32", kind="offload", tokens=32, heads=128, rows=262144, topk=2048, host="e2m2"),
        # one whole decode step of a layer: projections, cache writes, indexer, attention
        dict(name="layer_8", kind="layer", tokens=8, heads=128, ctx=12000, topk=2048),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "index", "index", "index", "write", "proj",
                       "offload", "layer"])
    topk = rng.choice([512, 1024, 2048, 2048, 2048])
    heads = rng.choice([16, 32, 64, 128, 128])
    if kind == "decode":
        per = rng.choice([1, 1, 1, 2, 3])                    # speculative tokens of a request
        req = max(1, _logu(rng, 1, 64) // per)
        return dict(kind="attn", tokens=req * per, per_req=per, heads=heads,
                    ctx=_logu(rng, 600, min(65536, 2097152 // req)), topk=topk, row=rng.choice([656, 656, 576]))
    if kind == "prefill":
        req = rng.choice([1, 1, 2, 4])
        per = _logu(rng, 128, 2048) // req
        return dict(kind="attn", tokens=req * per, per_req=per, heads=heads, ctx=per + _logu(rng, 1, 14000),
                    topk=topk, row=rng.choice([656, 576]))
    if kind == "index":
        path = rng.choice(["shard", "paged", "flat"])
        if path == "flat":
            req = rng.choice([1, 1, 2, 4])
            per = _logu(rng, 64, 2048) // req
            return dict(kind="index", path=path, rows=req * per, per_req=per,
                        ctx=(per * req + _logu(rng, 1, 14000)) // req, topk=topk, f16out=False)
        per = rng.choice([1, 1, 2])
        req = max(1, _logu(rng, 1, 64) // per)
        return dict(kind="index", path=path, rows=req * per, per_req=per, ctx=_logu(rng, 700, 131072), topk=topk,
                    f16out=path == "shard" and rng.random() < 0.4)
    if kind == "write":
        return dict(kind="write", tokens=_logu(rng, 1, 8192), row=rng.choice([656, 576]))
    if kind == "proj":
        return dict(kind="proj", tokens=_logu(rng, 1, 2048), heads=heads)
    if kind == "offload":
        return dict(kind="offload", tokens=_logu(rng, 1, 32), heads=heads, rows=rng.randrange(60000, 262144),
                    topk=topk, host=rng.choice(["e2m2", "row656"]))
    return dict(kind="layer", tokens=_logu(rng, 1, 32), heads=heads, ctx=_logu(rng, 2100, 24000), topk=topk)


# ---------------------------------------------------------------------------------------------- inputs from the seed
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).to(torch.bfloat16)


def _rows(seed, n, width):
    """n rows of N(0, 1) in bf16 (latent ‖ rope, or indexer keys), CHUNK at a time."""
    g = _gen(seed)
    for r0 in range(0, n, CHUNK):
        yield r0, _randn(g, min(CHUNK, n - r0), width)


def _requests(case, n):
    """Per token: its request, and the number of positions it sees. Decode requests are ragged (0.6 to 1 of ctx);
    the tokens of a request are its last per_req positions."""
    per = case["per_req"]
    req = torch.arange(n, device=DEV) // per
    nreq = -(-n // per)
    span = 1.0 - 0.4 * (torch.arange(nreq, device=DEV) % 7) / 7.0
    last = (case["ctx"] * span).long().clamp(min=min(per, case["ctx"])) if per < 64 else torch.full(
        (nreq,), case["ctx"], device=DEV)
    seen = last[req] - per + 1 + torch.arange(n, device=DEV) % per
    return req.to(torch.int32), seen.clamp(min=1).to(torch.int32), nreq


def _blocks(g, nreq, ctx):
    nb = -(-ctx // BS)
    return torch.randperm(nreq * nb, generator=g, device=DEV).view(nreq, nb).to(torch.int32)


def _selection(g, seen, topk, ctx):
    """Distinct positions below each token's count in the indexer's order, -1 where it sees fewer than topk."""
    out = torch.full((seen.shape[0], topk), -1, dtype=torch.int32, device=DEV)
    k = min(topk, ctx)
    for t0 in range(0, seen.shape[0], 256):
        s = seen[t0:t0 + 256, None]
        score = torch.rand(s.shape[0], ctx, generator=g, device=DEV)
        score.masked_fill_(torch.arange(ctx, device=DEV)[None] >= s, -1.0)
        v, i = score.topk(k, dim=1)
        out[t0:t0 + 256, :k] = torch.where(v >= 0, i, -1).to(torch.int32)
    return out


class _Layer:                                                # what forward_mqa reads of the engine's layer object
    _k_scale_float = KV_SCALE


def _attn_inputs(case, seed):
    g = _gen(seed)
    T = case["tokens"]
    req, seen, nreq = _requests(case, T)
    bt = _blocks(g, nreq, case["ctx"])
    return dict(q=_randn(g, T, case["heads"], 576), req=req, seen=seen, bt=bt,
                sel=_selection(g, seen, case["topk"], case["ctx"]))


def _impl(heads, buffer):
    return dsa.PortableSparseImpl(heads, 576, SM, 1, None, None, "fp8", None, "decoder", None,
                                  topk_indices_buffer=buffer, offload=False)


def _metadata(case, req, seen, bt, slots):
    T, dev = case["tokens"], req.device
    per = case.get("per_req", 1)
    start = torch.arange(0, T + per, per, device=dev, dtype=torch.int32).clamp(max=T)
    cam = dsa.CommonAttentionMetadata(query_start_loc=start, num_reqs=bt.shape[0], num_actual_tokens=T,
                                      max_query_len=per, max_seq_len=case["ctx"], slot_mapping=slots,
                                      block_table_tensor=bt, seq_lens=None)
    return dsa.PortableXPUBuilder(BS, case["topk"], T, dev).build(0, cam)


def _prepare_attn(case, seed):
    x = _attn_inputs(case, seed)
    impl = _impl(case["heads"], x["sel"])
    cache = torch.zeros(x["bt"].numel(), BS, case["row"], dtype=torch.uint8, device=DEV)
    for r0, kv in _rows(seed + 1, x["bt"].numel() * BS, 576):
        slots = torch.arange(r0, r0 + kv.shape[0], device=DEV)
        impl.do_kv_cache_update(kv[:, :512], kv[:, None, 512:], cache, slots, "fp8", KV_SCALE)
    md = _metadata(case, x["req"], x["seen"], x["bt"], None)
    return lambda: impl.forward_mqa(x["q"], cache, md, _Layer if case["row"] == 576 else None)[0]


def _index_inputs(case, seed):
    g = _gen(seed)
    n = case["rows"]
    req, seen, nreq = _requests(case, n)
    return dict(q=_randn(g, n, 64, 128), w=torch.rand(n, 64, generator=g, device=DEV), req=req, seen=seen,
                bt=_blocks(g, nreq, case["ctx"]))


def _prepare_index(case, seed):
    x = _index_inputs(case, seed)
    q, w, bt, ctx, K = x["q"], x["w"], x["bt"], case["ctx"], case["topk"]
    if case["path"] == "flat":                               # the requests' keys gathered one after another
        nreq = bt.shape[0]
        codes, scales = [], []
        for _, k in _rows(seed + 1, nreq * ctx, 128):
            c, s = _quant(k, 128, 1e-4)
            codes.append(c)
            scales.append(s)
        kv = (torch.cat(codes), torch.cat(scales).view(-1))
        ks = x["req"] * ctx
        ke = (ks + x["seen"]).to(torch.int32)

        def flat():
            lg = kernels.mqa_logits(q, kv, w, ks, ke)
            return lg, kernels.topk(lg, ke, K)
        return flat
    cache = torch.zeros(bt.numel(), BS, 132, dtype=torch.uint8, device=DEV)
    store = shard_indexer.ShardStore(cache, 1, 0, f16out=case["f16out"])
    for r0, k in _rows(seed + 1, bt.numel() * BS, 128):
        slots = torch.arange(r0, r0 + k.shape[0], device=DEV)
        if case["path"] == "paged":
            kernels.index_key_write_shuffle(k, slots, cache)
        else:
            store.write(k, slots, False)
    if case["path"] == "paged":
        per = case["per_req"]
        lens = x["seen"].view(-1, per)
        q4 = q.view(-1, per, 64, 128)

        def paged():
            lg = kernels.paged_mqa_logits(q4, cache, w, lens, bt, ctx)
            return lg, kernels.topk(lg, x["seen"], K)
        return paged
    out = torch.empty(case["rows"], K, dtype=torch.int32, device=DEV)
    return lambda: shard_indexer.sharded_topk(store, q, w, bt, x["req"], x["seen"], ctx, out, K)


def _write_inputs(case, seed):
    g = _gen(seed)
    n = case["tokens"]
    R = -(-2 * n // BS) * BS
    return _randn(g, n, 576), _randn(g, n, 128), torch.randperm(R, generator=g, device=DEV)[:n], R


def _prepare_write(case, seed):
    kv, k, slots, R = _write_inputs(case, seed)
    impl = _impl(128, None)
    cache = torch.zeros(R // BS, BS, case["row"], dtype=torch.uint8, device=DEV)
    keys = torch.zeros(R // BS, BS, 132, dtype=torch.uint8, device=DEV)
    store = shard_indexer.ShardStore(keys, 1, 0)
    lat, pe = kv[:, :512], kv[:, None, 512:]

    def write():
        impl.do_kv_cache_update(lat, pe, cache, slots, "fp8", KV_SCALE)
        store.write(k, slots, False)
        return cache, keys
    return write


def _weights(g, heads):
    """kv_b_proj's absorbed halves as block-scaled fp8: (codes, scales, scale over k) of W_UK_T and of W_UV."""
    def code(*shape):
        return (torch.randn(*shape, generator=g, device=DEV) * 64).to(torch.float8_e4m3fn).view(torch.uint8)

    def scale(*shape):
        return (0.5 + torch.rand(*shape, generator=g, device=DEV)) / 2048
    uk = (code(heads, 512, 128), scale(heads, 1, 4).expand(heads, 128, 4).contiguous(), False)
    uv = (code(heads, 128, 512), scale(heads, 1, 4).expand(heads, 128, 4).contiguous(), True)
    return uk, uv


def _proj_inputs(case, seed):
    g = _gen(seed)
    T, H = case["tokens"], case["heads"]
    uk, uv = _weights(g, H)
    return dict(q_nope=_randn(g, T, H, 128), q_pe=_randn(g, T, H, 64), o=_randn(g, T, H, 512), uk=uk, uv=uv)


def _prepare_proj(case, seed):
    x = _proj_inputs(case, seed)
    y = torch.empty(case["tokens"], case["heads"], 128, dtype=torch.bfloat16, device=DEV)

    def proj():
        q = mla_fp8.build_query(x["q_nope"], x["q_pe"], x["uk"])
        mla_fp8.bmm_fp8(x["o"].transpose(0, 1), x["uv"], y.transpose(0, 1))
        return q, y
    return proj


def _offload_inputs(case, seed):
    g = _gen(seed)
    T, R = case["tokens"], case["rows"]
    p = torch.arange(1, R + 1, device=DEV, dtype=torch.float32).pow(-1.1)      # Zipf(1.1) over a random row order
    order = torch.randperm(R, generator=g, device=DEV)
    draws = torch.log(p) - torch.log(-torch.log(torch.rand(T, R, generator=g, device=DEV).clamp(1e-9, 1 - 1e-7)))
    idx = order[draws.topk(min(case["topk"], R), dim=1).indices].to(torch.int32)
    return dict(q=_randn(g, T, case["heads"], 576), idx=idx, hot=order[:R // 4])


def _prepare_offload(case, seed):
    x = _offload_inputs(case, seed)
    scale = KV_SCALE if case["host"] == "e2m2" else 1.0
    off = sparse_offload.LayerOffload(case["rows"], DEV, cache_rows=case["rows"] // 4, row_fmt=case["host"])
    for r0, kv in _rows(seed + 1, case["rows"], 576):
        off.store(kv[:, :512], kv[:, 512:], torch.arange(r0, r0 + kv.shape[0], device=DEV), scale)
    off.set_hot_rows(x["hot"])
    return lambda: off.attend(x["q"], x["idx"], SM, scale)


def _layer_inputs(case, seed):
    g = _gen(seed)
    x = _proj_inputs(case, seed + 2)
    T = case["tokens"]
    one = dict(case, per_req=1)
    req, seen, nreq = _requests(one, T)
    bt = _blocks(g, nreq, case["ctx"])
    pos = (seen - 1).long()
    slots = bt[req.long(), pos // BS].long() * BS + pos % BS
    x.update(req=req, seen=seen, bt=bt, slots=slots, kv=_randn(g, T, 576), k=_randn(g, T, 128),
             iq=_randn(g, T, 64, 128), iw=torch.rand(T, 64, generator=g, device=DEV))
    return x


def _prepare_layer(case, seed):
    x = _layer_inputs(case, seed)
    T, H, K = case["tokens"], case["heads"], case["topk"]
    top = torch.empty(T, K, dtype=torch.int32, device=DEV)
    impl = _impl(H, top)
    cache = torch.zeros(x["bt"].numel(), BS, 656, dtype=torch.uint8, device=DEV)
    keys = torch.zeros(x["bt"].numel(), BS, 132, dtype=torch.uint8, device=DEV)
    store = shard_indexer.ShardStore(keys, 1, 0)
    for r0, kv in _rows(seed + 1, x["bt"].numel() * BS, 704):
        slots = torch.arange(r0, r0 + kv.shape[0], device=DEV)
        impl.do_kv_cache_update(kv[:, :512], kv[:, None, 512:576], cache, slots, "fp8_ds_mla", None)
        store.write(kv[:, 576:], slots, False)
    md = _metadata(case, x["req"], x["seen"], x["bt"], x["slots"])
    lat, pe = x["kv"][:, :512], x["kv"][:, None, 512:]

    def step():
        store.write(x["k"], x["slots"], False)
        impl.do_kv_cache_update(lat, pe, cache, x["slots"], "fp8_ds_mla", None)
        shard_indexer.sharded_topk(store, x["iq"], x["iw"], x["bt"], x["req"], x["seen"], case["ctx"], top, K)
        q = mla_fp8.build_query(x["q_nope"], x["q_pe"], x["uk"])
        o, _ = impl.forward_mqa(q, cache, md)
        y = mla_fp8.bmm_fp8(o.transpose(0, 1), x["uv"])
        return y, o, top
    return step


_PREPARE = dict(attn=_prepare_attn, index=_prepare_index, write=_prepare_write, proj=_prepare_proj,
                offload=_prepare_offload, layer=_prepare_layer)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state()


# ---------------------------------------------------------------------------------------------- work and tolerance
def _counts(case, n):
    """(positions seen by all tokens, rows selected by all tokens, distinct context rows) without a GPU."""
    per = case.get("per_req", 1)
    seen = chosen = rows = 0
    for r in range(-(-n // per)):
        last = case["ctx"] if per >= 64 else max(int(case["ctx"] * (1 - 0.4 * (r % 7) / 7)), min(per, case["ctx"]))
        rows += last
        for j in range(per):
            s = max(1, last - per + 1 + j)
            seen += s
            chosen += min(s, case["topk"])
    return seen, chosen, rows


def work(case):
    kind = case["kind"]
    if kind == "attn":
        T, H = case["tokens"], case["heads"]
        _, chosen, rows = _counts(case, T)
        return dict(bytes=min(chosen, rows) * case["row"] + T * H * (1152 + 1024) + T * case["topk"] * 4,
                    flops=chosen * H * 2 * (576 + 512))
    if kind == "index":
        n = case["rows"]
        seen, _, rows = _counts(case, n)
        whole = case["path"] != "shard"                      # the logits come back as well
        cols = rows if case["path"] == "flat" else case["ctx"]
        return dict(bytes=rows * 132 + n * 64 * (256 + 4) + n * case["topk"] * 4 + (n * cols * 4 if whole else 0),
                    flops=seen * 64 * 128 * 2)
    if kind == "write":
        return dict(bytes=case["tokens"] * (1152 + 256 + 8 + case["row"] + 132), flops=0)
    if kind == "proj":
        T, H = case["tokens"], case["heads"]
        return dict(bytes=H * 2 * (65536 + 2048) + T * H * 2 * (128 + 64 + 576 + 512 + 128),
                    flops=T * H * 2 * 2 * 128 * 512)
    if kind == "offload":
        T, H, K = case["tokens"], case["heads"], case["topk"]
        return dict(bytes=T * K * (400 if case["host"] == "e2m2" else 656) + T * H * (1152 + 1024) + T * K * 4,
                    flops=T * K * H * 2 * (576 + 512))
    T, H = case["tokens"], case["heads"]
    seen, chosen, _ = _counts(case, T)
    return dict(bytes=seen * 132 + chosen * 656 + H * 2 * (65536 + 2048) + T * H * 2 * (192 + 128 + 512),
                flops=seen * 16384 + chosen * H * 2 * (576 + 512) + T * H * 2 * 2 * 128 * 512)


def tolerance(case):
    kind = case["kind"]
    if kind == "write":
        return "exact"
    if kind == "index":                # fp32 logits; positions whose logits are a rounding apart may swap
        return dict(rel=1e-5, max=1e-4, differ=0.01)
    if kind == "layer":                # a row at the selection's edge may be another one
        return dict(rel=0.02, max=0.5, differ=0.01)
    return dict(rel=0.01, max=0.1)     # bf16 outputs


# ---------------------------------------------------------------------------------------------- 64-bit results
def _quant(x, group, floor):
    """e4m3 codes (uint8) and fp32 scales of bf16 rows, one scale per `group` values: indexer keys and KV rows."""
    v = x.float().view(x.shape[0], -1, group)
    s = _div(v.abs().amax(2).clamp(min=floor), 448.0)
    return (v / s[..., None]).to(torch.float8_e4m3fn).view(torch.uint8).view(x.shape), s


def _div(x, by):
    """x / by rounded once (torch multiplies by the reciprocal when it divides by a number)."""
    return x / torch.full_like(x, by)


def _kept656(kv):
    c, s = _quant(kv[:, :512], 128, 448e-12)
    return torch.cat([(c.view(torch.float8_e4m3fn).float().view(-1, 4, 128) * s[..., None]).view(-1, 512),
                      kv[:, 512:].float()], 1)


def _kept576(kv):
    return (kv.float() / KV_SCALE).clamp(-448, 448).to(torch.float8_e4m3fn).float() * KV_SCALE


def _kept400(kv):
    """Latent values on the e2m2 grid with a power-of-two scale per 32, the rope in e4m3."""
    x = (kv[:, :512].float() / KV_SCALE).clamp(-448, 448).view(-1, 16, 32)
    m, e = torch.frexp(_div(x.abs().amax(2), 7.0))
    k = torch.where(m == 0.5, e - 1, e).clamp(-126, 127)
    unit = torch.exp2(k.float())[..., None]
    y = x.abs() / unit
    step = torch.where(y < 2, 0.25, torch.where(y < 4, 0.5, 1.0))
    y = (torch.floor(y / step + 0.5) * step).clamp(max=7.0)
    return torch.cat([(torch.sign(x) * y * unit).view(-1, 512) * KV_SCALE, _kept576(kv[:, 512:])], 1)


def _attend64(q, rows, idx):
    """q [T, H, 576], rows [R, 576] fp32 (kept values), idx [T, K] rows or -1 -> [T, H, 512] in 64 bits."""
    out = torch.zeros(q.shape[0], q.shape[1], 512, dtype=torch.float64, device=DEV)
    step = max(1, 65536 // idx.shape[1])
    for t0 in range(0, q.shape[0], step):
        i = idx[t0:t0 + step].long()
        kv = rows[i.clamp(min=0)].double()
        s = torch.bmm(q[t0:t0 + step].double(), kv.transpose(1, 2).contiguous()) * SM
        s.masked_fill_((i < 0)[:, None], -math.inf)
        out[t0:t0 + step] = torch.bmm(torch.softmax(s, 2), kv[..., :512].contiguous())
    return out


def _paged_rows(sel, req, bt):
    blk = bt[req.long()[:, None], sel.clamp(min=0).long() // BS].long()
    return torch.where(sel >= 0, blk * BS + sel.clamp(min=0) % BS, -1)


def _logits64(q, w, keys, seen, first, ncol, base=0):
    """First key row of each query row's request -> [rows, ncol] in 64 bits, -inf beyond its positions; column
    base[row] + j is position j."""
    out = torch.full((q.shape[0], ncol), -math.inf, dtype=torch.float64, device=DEV)
    seen, first = seen.tolist(), first.tolist()
    base = [0] * len(seen) if isinstance(base, int) else base.tolist()
    for r in range(q.shape[0]):
        k = keys(r, first[r], seen[r]).double()
        s = torch.relu(q[r].double() @ k.t())
        out[r, base[r]:base[r] + seen[r]] = w[r].double() @ s
    return out


def _kept_keys(k):
    c, s = _quant(k, 128, 1e-4)
    return c.view(torch.float8_e4m3fn).float() * s


def _scaled64(f):
    """The bf16 weights that codes and scales stand for, [N, J, K] in 64 bits."""
    codes, scales, over_k = f
    c = codes.view(torch.float8_e4m3fn).float()
    s = scales.repeat_interleave(128, 2) if over_k else scales.transpose(1, 2).repeat_interleave(128, 1)
    return (c * s).to(torch.bfloat16).double()


def _project64(x):
    q = torch.einsum("thk,hjk->thj", x["q_nope"].double(), _scaled64(x["uk"]))
    return torch.cat([q, x["q_pe"].double()], 2)


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn":
        x = _attn_inputs(case, seed)
        keep = _kept656 if case["row"] == 656 else _kept576
        rows = torch.empty(x["bt"].numel() * BS, 576, device=DEV)
        for r0, kv in _rows(seed + 1, rows.shape[0], 576):
            rows[r0:r0 + kv.shape[0]] = keep(kv)
        return _attend64(x["q"], rows, _paged_rows(x["sel"], x["req"], x["bt"]))
    if kind == "index":
        if case["path"] == "shard":                          # positions only
            return None
        x = _index_inputs(case, seed)
        n = x["bt"].numel() * BS if case["path"] == "paged" else x["bt"].shape[0] * case["ctx"]
        keys = torch.cat([_kept_keys(k) for _, k in _rows(seed + 1, n, 128)])
        req = x["req"].long()
        if case["path"] == "flat":
            first = req * case["ctx"]
            lg = _logits64(x["q"], x["w"], lambda r, f, s: keys[f:f + s], x["seen"], first, n, first)
        else:
            blocks = keys.view(-1, BS, 128)

            def of(r, f, s):
                return blocks[x["bt"][f].long()].view(-1, 128)[:s]
            lg = _logits64(x["q"], x["w"], of, x["seen"], req, case["ctx"])
        return lg, None
    if kind == "write":
        return None
    if kind == "proj":
        x = _proj_inputs(case, seed)
        return _project64(x), torch.einsum("thk,hjk->thj", x["o"].double(), _scaled64(x["uv"]))
    if kind == "offload":
        x = _offload_inputs(case, seed)
        keep = _kept400 if case["host"] == "e2m2" else _kept656
        rows = torch.cat([keep(kv) for _, kv in _rows(seed + 1, case["rows"], 576)])
        return _attend64(x["q"], rows, x["idx"])
    x = _layer_inputs(case, seed)
    kv = torch.cat([c for _, c in _rows(seed + 1, x["bt"].numel() * BS, 704)])
    kv[x["slots"]] = torch.cat([x["kv"], x["k"]], 1)
    keys = _kept_keys(kv[:, 576:].contiguous()).view(-1, BS, 128)
    lg = _logits64(x["iq"], x["iw"], lambda r, f, s: keys[x["bt"][f].long()].view(-1, 128)[:s], x["seen"],
                   x["req"].long(), case["ctx"])
    v, sel = lg.topk(min(case["topk"], case["ctx"]), dim=1)
    sel = torch.where(v > -math.inf, sel, -1)
    o = _attend64(_project64(x), _kept656(kv[:, :576]), _paged_rows(sel, x["req"], x["bt"]))
    return torch.einsum("thk,hjk->htj", o, _scaled64(x["uv"])), o, None
