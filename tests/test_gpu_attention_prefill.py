"""GPU parity of the 128-head prefill kernel (fwd_kernel, both row formats) against the fp64 oracle at the edges of its
range: launches just past the rule that selects it, partial head groups, ragged row lists (no row, one row, a tile and
one row, 2048 rows), invalid entries, fp32 partials, a prior partial, row scales that rise tile after tile. Output bar:
1e-2 plus half a bf16 ulp (fp32 partials: 1e-2); lse within 1e-3."""
import numpy as np
import pytest
import torch

from oracle import spmla_ref as ref
from tests.helpers import attn_excess, make_pool_576, make_pool_656, make_q

pytestmark = pytest.mark.gpu
SM = 192 ** -0.5


def _pool(fmt, R, kv_scale):
    return make_pool_576(R, seed=3, kv_scale=kv_scale) if fmt == 576 else make_pool_656(R, seed=3)[0]


@pytest.mark.parametrize("fmt", [656, 576])
@pytest.mark.parametrize("T,H,K,form", [
    (256, 128, 70, "plain"),           # K <= 512: three tiles, the last of 6 rows
    (256, 112, 2048, "counts"),        # the longest lists; ragged counts; heads past H in the last block
    (250, 256, 512, "invalid"),        # two full head groups
    (400, 224, 96, "counts"),          # the second group has 96 heads
    (120, 128, 1024, "partials"),      # two splits as fp32 partials
    (256, 128, 160, "prior"),          # the output merged with a prior partial (Row656)
    (256, 128, 256, "rising"),         # rows in the order of their magnitude, 2^-18 .. 2^9 (Row656)
])
def test_prefill_kernel_vs_oracle(dev, fmt, T, H, K, form):
    from arcagi2_flashnext_dots3_amd import kernels
    if fmt == 576 and form in ("prior", "rising"):
        pytest.skip("Row656 only")
    print(f"[prefill] fmt={fmt} T={T} H={H} K={K} {form}", flush=True)
    R, kv = 4096, 0.5 if fmt == 576 else 1.0
    g = torch.Generator().manual_seed(K + T)
    if form == "rising":
        mag = torch.exp2(torch.linspace(-18, 9, R))[:, None]
        from tests.helpers import bf16_bits
        pool = np.zeros((R, 656), dtype=np.uint8)
        ref.cache_write_656(bf16_bits(torch.randn(R, 512, generator=g) * mag), bf16_bits(torch.randn(R, 64, generator=g)),
                            np.arange(R), pool)
        idx = torch.sort(torch.randint(0, R, (T, K), generator=g), 1)[0].to(torch.int32)
    else:
        pool = _pool(fmt, R, kv)
        idx = torch.randint(0, R, (T, K), generator=g).to(torch.int32)
    q = make_q(T, H, seed=T + H, scale=2 ** -9 if form == "rising" else 1.0)
    kcount = None
    if form == "counts":
        kcount = torch.randint(0, K + 1, (T,), generator=g).to(torch.int32)
        kcount[:8] = torch.tensor([0, 1, 31, 32, 33, 64, K - 1, K], dtype=torch.int32)
    if form == "invalid":
        idx[torch.rand(T, K, generator=g) < 0.1] = -1
        idx[1, 5::7] = R + 11
        idx[2, :] = -1
    some = np.unique(np.r_[0:8, np.arange(0, T, 37), T - 1])      # tokens compared
    qd, pd, xd = q.to(dev), torch.from_numpy(pool).to(dev), idx.to(dev)
    kc = None if kcount is None else kcount.to(dev)
    qn, xn = q[some].float().numpy(), idx[some].numpy()
    if form == "partials":
        kernels_out, lses = kernels.attend_partial(qd, pd, xd, SM, kv, split=2)
        torch.cuda.synchronize()
        for s in range(2):
            o_ref, l_ref = ref.attention(qn, pool, xn[:, s * K // 2:(s + 1) * K // 2], SM, kv, fmt=fmt)
            assert np.abs(kernels_out[s].cpu().numpy()[some] - o_ref).max() <= 1e-2
            assert np.abs(lses[s].cpu().numpy()[some] - l_ref).max() <= 1e-3
        return
    if form == "prior":
        px = torch.randint(0, R, (T, 64), generator=g).to(torch.int32)
        po, pl = ref.attention(q.float().numpy()[some], pool, px[some].numpy(), SM, kv)
        o1, l1 = torch.zeros(T, H, 512), torch.full((T, H), -np.inf)
        o1[some], l1[some] = torch.from_numpy(po).float(), torch.from_numpy(pl).float()
        out, lse = kernels.attend_merge(qd, pd, xd, SM, kv, o1.to(dev), l1.to(dev))
        xn = np.concatenate([xn, px[some].numpy()], 1)
    else:
        out, lse = kernels.attend(qd, pd, xd, SM, kv, split=1, kcount=kc)
    torch.cuda.synchronize()
    o_ref, l_ref = ref.attention(qn, pool, xn, SM, kv, kcount=None if kcount is None else kcount[some].numpy(), fmt=fmt)
    o, l = out.float().cpu().numpy()[some], lse.cpu().numpy()[some]
    fin = np.isfinite(l_ref)
    assert np.array_equal(fin, np.isfinite(l))
    assert np.all(o[~fin] == 0)
    assert np.abs(l[fin] - l_ref[fin]).max() <= 1e-3
    # "rising": outputs up to 1e3; P' rounded to f16 and the bf16 output: 2^-8 of the token's largest value
    tol = 1e-2 if form != "rising" else 2 ** -8 * np.abs(o_ref).max()
    assert attn_excess(o, o_ref, tol) <= 0


@pytest.mark.parametrize("fmt", [656, 576])
@pytest.mark.parametrize("T,H,K,bs,pad", [
    (3, 32, 2048, 64, 0),              # splits merged in the kernel
    (5, 128, 40, 1, 0),                # one tile and eight rows, one row per block
    (130, 64, 200, 16, 3),             # unsplit, a padded block stride
    (256, 128, 300, 128, 0),           # the 128-head kernel
    (256, 128, 2048, 64, 1),
])
def test_paged_rows_formed_in_the_kernel(dev, fmt, T, H, K, bs, pad):
    """attend_paged against attend over rows_from_topk: the same bits, with entries of -1, positions past the table and
    negative table entries, from strided views."""
    from arcagi2_flashnext_dots3_amd import kernels
    print(f"[paged attention] fmt={fmt} T={T} H={H} K={K} bs={bs} pad={pad}", flush=True)
    g = torch.Generator().manual_seed(T + K + bs)
    nreq, cols, stride = 3, max(2, 1024 // bs), bs + pad
    nblk = nreq * cols
    pool = torch.from_numpy(_pool(fmt, nblk * stride, 1.0)).to(dev)
    table = torch.randperm(nblk, generator=g).view(nreq, cols).to(torch.int32)
    table[1, cols // 2] = -1
    table = torch.nn.functional.pad(table, (0, 5), value=-7).to(dev)[:, :cols]
    pos = torch.randint(0, cols * bs, (T, K + 9), generator=g).to(torch.int32)
    pos[torch.rand(T, K + 9, generator=g) < 0.05] = -1
    pos[0, :3] = torch.tensor([cols * bs, cols * bs + bs, 2 ** 31 - 1], dtype=torch.int32)
    pos[min(2, T - 1), :] = -1
    pos = pos.to(dev)[:, :K]
    req = torch.randint(0, nreq, (T,), generator=g).to(torch.int32).to(dev)
    q = make_q(T, H, seed=K).to(dev)
    rows = kernels.rows_from_topk(pos, req, table, bs, stride_rows=stride)
    a, _ = kernels.attend(q, pool, rows, SM, 0.7)
    b = kernels.attend_paged(q, pool, pos, req, table, bs, stride, SM, 0.7, row_bytes=fmt)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    assert kernels.attend_paged(q, pool, pos, req, table, 48, 48, SM, row_bytes=fmt) is None


@pytest.mark.parametrize("fmt", [656, 576])
@pytest.mark.parametrize("T,K", [(3, 2048), (5, 40), (256, 300)])    # merged splits, unsplit, the 128-head kernel
def test_paged_padding_tokens_of_no_request(dev, fmt, T, K):
    """Tokens without a position in the table may have any request id: the same bits as attend over rows_from_topk."""
    from arcagi2_flashnext_dots3_amd import kernels
    print(f"[paged attention] padding fmt={fmt} T={T} K={K}", flush=True)
    g = torch.Generator().manual_seed(T + K)
    bs, nreq, cols, H = 64, 2, 12, 128
    pool = torch.from_numpy(_pool(fmt, nreq * cols * bs, 1.0)).to(dev)
    table = torch.randperm(nreq * cols, generator=g).view(nreq, cols).to(torch.int32).to(dev)
    pos = torch.randint(0, cols * bs, (T, K), generator=g).to(torch.int32)
    req = torch.randint(0, nreq, (T,), generator=g).to(torch.int32)
    pos[1], req[1] = -1, -1
    pos[T - 1], req[T - 1] = cols * bs, 2 ** 31 - 1
    pos, req, q = pos.to(dev), req.to(dev), make_q(T, H, seed=K).to(dev)
    a, _ = kernels.attend(q, pool, kernels.rows_from_topk(pos, req, table, bs), SM, 0.7)
    b = kernels.attend_paged(q, pool, pos, req, table, bs, bs, SM, 0.7, row_bytes=fmt)
    torch.cuda.synchronize()
    assert torch.equal(a, b) and not a[1].any() and not a[T - 1].any()
