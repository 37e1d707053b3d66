"""GPU parity of single kernels at the sizes where their tiles, rings and splits begin and end,
against the CPU oracle with the tolerances of test_gpu_attention.py."""

import numpy as np
import pytest
import torch

from hackaton_amd import attention as att
from hackaton_amd import workloads as wl
from oracle import attention_oracle as orc
from tests.test_gpu_attention import SCALE, TOL, banner, oracle

pytestmark = pytest.mark.gpu


EDGES = [[1, 31, 32, 33], [63, 64, 65], [95, 96, 97, 127], [128, 129, 160, 161], [255, 256, 257],
         [383, 385]]
LONG_LIST = 7 * 256  # (tile, head) pairs from which the many-item forward runs its 32-key tiles


def _many_item_forward(q, k, v, lengths, scale=SCALE):
    """out and lse of va_fwd_kernel(VA_FWD_MANY) on the GPU tensors, from NaN-filled outputs."""
    (n, hq, _), hkv = q.shape, k.shape[1]
    plan = att._plan(att._cu_seqlens(lengths, q.device), hq, hkv)
    out = torch.full_like(q, float("nan"))
    lse = torch.full((hq, n), float("nan"), dtype=torch.float32, device=q.device)
    att.check(att.lib().va_fwd_kernel(att._lib.VA_FWD_MANY, q.data_ptr(), k.data_ptr(),
                                      v.data_ptr(), out.data_ptr(), lse.data_ptr(),
                                      plan.fwd_items.data_ptr(), plan.n_fwd, n, hq, hkv, 128,
                                      scale, 0 if q.dtype == torch.float16 else 1, att._stream()),
              "va_fwd_kernel")
    torch.cuda.synchronize()
    return out, lse


@pytest.mark.parametrize("lengths", EDGES)
@pytest.mark.parametrize("hq,hkv,dtype", [(3, 1, torch.float16), (14, 2, torch.bfloat16)])
def test_many_item_forward_at_tile_and_ring_edges(lengths, hq, hkv, dtype):
    """One, two, three and more 64-key tiles through the two stages of a short list (two work-groups
    a CU), with full and partial last tiles and strips, documents before and after each other in
    one packed array."""
    banner("many-item forward edges", lengths, hq, hkv, dtype)
    q, k, v, do = wl.make_inputs(lengths, hq, hkv, dtype, seed=sum(lengths))
    out, lse = _many_item_forward(q.cuda(), k.cuda(), v.cuda(), lengths)
    o_ref, lse_ref = oracle(q, k, v, do, lengths)[:2]
    assert float(np.max(np.abs(out.cpu().float().numpy() - o_ref))) <= TOL[dtype]["o"]
    assert float(np.max(np.abs(lse.cpu().numpy() - lse_ref))) <= TOL[dtype]["lse"]


@pytest.mark.parametrize("hq,hkv,dtype", [(96, 8, torch.float16), (98, 14, torch.bfloat16)])
def test_many_item_forward_edges_in_a_long_list(hq, hkv, dtype):
    """The same documents in one batch with heads enough for the 32-key tiles in a ring of three
    stages, three work-groups a CU: one, two, three and more tiles, each end of the ring."""
    lengths = sum(EDGES, [])
    assert -(-sum(lengths) // 128) * hq >= LONG_LIST
    banner("many-item forward edges, long list", hq, hkv, dtype)
    q, k, v, _ = wl.make_inputs(lengths, hq, hkv, dtype, seed=hq)
    out, lse = _many_item_forward(q.cuda(), k.cuda(), v.cuda(), lengths)
    o_ref, lse_ref = orc.attention_forward(*(t.double().numpy() for t in (q, k, v)),
                                           orc.cu_seqlens_from_lengths(lengths), SCALE)
    assert float(np.max(np.abs(out.cpu().float().numpy() - o_ref))) <= TOL[dtype]["o"]
    assert float(np.max(np.abs(lse.cpu().numpy() - lse_ref))) <= TOL[dtype]["lse"]


def _two_key_documents(dtype, hq, hkv, first):
    """Documents of 200 tokens in which a query sees a key of score 0 (key 0), with `first` one
    of 9 (key 70) and, 8 keys into the next 32, one of 5 to 7.5 more, in log2 units; every other key
    lies 60 or more below. Returns lengths, q, k, v and the two late keys' positions."""
    lengths = [200] * 5 + [24]
    n = sum(lengths)
    start = np.repeat(np.cumsum([0] + lengths[:-1]), lengths)
    at = torch.from_numpy(np.arange(n) - start)
    last = 40 if first is None else 104
    rise = torch.linspace(5.0, 7.5, hkv * len(lengths)).view(len(lengths), hkv)
    rise = torch.repeat_interleave(rise, torch.tensor(lengths), dim=0)
    score = torch.full((n, hkv), -60.0)
    score[at == 0] = 0.0
    if first is not None:
        score[at == first] = 9.0
        rise = rise + 9.0
    score[at == last] = rise[at == last]
    k = torch.zeros(n, hkv, 128)
    k[:, :, 0] = score
    q = torch.zeros(n, hq, 128)
    q[:, :, 0] = 1.0
    return lengths, at, q.to(dtype), k.to(dtype), torch.randn(n, hkv, 128).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("first", [None, 70])
@pytest.mark.parametrize("long_list", [False, True])
def test_many_item_forward_keeps_the_largest_weight_exact(long_list, first, dtype):
    """The reference maximum moves freely over a document's first 64 keys and over the 64 keys where
    it moved last, so the largest weight there is 1 and rounds to nothing: lse is within the
    rounding of the weights below it. A maximum that stays at the first 32 keys' leaves the
    largest weight at 2^5 to 2^7.5, rounded to 16 bits, which shows in lse.

    Bound: the other weight is at most 2^-5 of the largest and its rounding u = 2^-9 (bf16) or
    2^-12 (fp16) of it; fp32 sums, exponentials and logarithms of values below 24: 8 ulp of 16."""
    hq, hkv = (224, 28) if long_list else (28, 28)
    lengths, at, q, k, v = _two_key_documents(dtype, hq, hkv, first)
    assert (-(-sum(lengths) // 128) * hq >= LONG_LIST) == long_list
    banner("largest weight", long_list, first, dtype)
    scale = float(np.float32(np.log(2.0)))  # scores are in log2 units
    _, lse = _many_item_forward(q.cuda(), k.cuda(), v.cuda(), lengths, scale)
    late = (at >= (40 if first is None else 104)).numpy()
    s = torch.repeat_interleave(k[:, :, 0].double(), hq // hkv, dim=1).t().numpy() * scale
    ref, start = np.empty_like(s), 0
    for length in lengths:
        rows = slice(start, start + length)
        ref[:, rows] = np.logaddexp.accumulate(s[:, rows], axis=1)
        start += length
    u = 2.0 ** -12 if dtype == torch.float16 else 2.0 ** -9
    bound = 2.0 ** -5 * u + 8 * 2.0 ** -20
    assert float(np.max(np.abs(lse.cpu().double().numpy() - ref)[:, late])) <= bound


def test_graph_with_host_lengths_outlives_the_plan_caches():
    """A training step captured with host lengths, its autograd nodes gone, replays its own work lists
    after 40 other batches have gone through the plan caches and the allocator."""
    banner("captured plan")
    lengths, hq, hkv = [200, 77, 31], 12, 2
    dev = torch.device("cuda")
    q, k, v, do = (t.to(dev) for t in wl.make_inputs(lengths, hq, hkv, torch.float16, seed=3))
    leaves = [t.requires_grad_() for t in (q, k, v)]
    do = do.reshape(sum(lengths), -1)

    def step():
        out = att.varlen_attention(*leaves, lengths, SCALE)
        return (out.detach(), *torch.autograd.grad(out, leaves, do))

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        eager = [t.clone() for t in step()]
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    plan = att._plan(att._cu_seqlens(lengths, dev), hq, hkv)
    addresses = {plan.fwd_items.data_ptr(), plan.bwd_items.data_ptr()}
    del plan
    others = []
    for i in range(40):
        cu = att._cu_seqlens([150 + i, 60], dev)
        other = att._plan(cu, hq, hkv)
        others += [other.fwd_items, other.bwd_items, torch.full_like(other.fwd_items, -1)]
    assert not addresses & {t.data_ptr() for t in others}
    for _ in range(2):
        for t in captured:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(captured, eager):
            assert torch.equal(x, y)
    del graph, captured
    att.release_captured_plans()


def _positions(batch, seq, n, seed):
    """n distinct rows of a (batch, seq) batch in random order: (b_idx, t_idx) int32, on the GPU."""
    rows = torch.from_numpy(np.random.default_rng(seed).permutation(batch * seq)[:n])
    return (rows // seq).to(torch.int32).cuda(), (rows % seq).to(torch.int32).cuda()


@pytest.mark.parametrize("batch,seq,n,heads,dim,dtype", [
    (1, 1, 1, 1, 8, torch.float16), (3, 7, 5, 2, 128, torch.float16),
    (2, 65, 130, 12, 128, torch.bfloat16), (4, 33, 64, 5, 128, torch.float32),
    (2, 9, 11, 28, 128, torch.float16), (2, 17, 20, 3, 24, torch.float32),
    (3, 5, 0, 2, 128, torch.float16)])
def test_row_packing_writes_every_row(batch, seq, n, heads, dim, dtype):
    """pack_rows and its backward at row widths of one chunk, of a power of two and of neither, with
    rows in any order; the backward's row map scratch and output hold anything before (here NaN, and
    a map that names no token, a wrong one for every row, or none of the batch's), and the plain
    scatter of va_pack_rows."""
    banner("row packing", batch, seq, n, heads, dim, dtype)
    b, t = _positions(batch, seq, n, seed=n)
    attn = torch.randn(batch, heads, seq, dim, device="cuda").to(dtype)
    grad = torch.randn(n, heads * dim, device="cuda").to(dtype)
    out = att.pack_rows(attn, b, t)
    assert torch.equal(out, attn[b.long(), :, t.long()].reshape(n, heads * dim))
    ref = torch.zeros(batch, heads, seq, dim, dtype=dtype, device="cuda")
    ref[b.long(), :, t.long()] = grad.view(n, heads, dim)
    for fill in (-1, 0, n - 1, 1 << 30):
        got = torch.full_like(ref, float("nan"))
        row_map = torch.full((batch * seq,), fill, dtype=torch.int32, device="cuda")
        att.check(att.lib().va_unpack_rows(grad.data_ptr(), got.data_ptr(), b.data_ptr(),
                                           t.data_ptr(), row_map.data_ptr(), n, batch, heads, seq,
                                           dim, grad.element_size(), att._stream()),
                  "va_unpack_rows")
        torch.cuda.synchronize()
        assert torch.equal(got, ref), fill
    got = torch.zeros_like(ref)  # va_pack_rows' own scatter, into a cleared buffer
    att.check(att.lib().va_pack_rows(grad.data_ptr(), got.data_ptr(), b.data_ptr(), t.data_ptr(), n,
                                     heads, seq, dim, grad.element_size(), 1, att._stream()),
              "va_pack_rows")
    torch.cuda.synchronize()
    assert torch.equal(got, ref)


def test_row_packing_past_2_26_rows():
    """pack_rows and its backward where one wave per row passes the 2^32 threads of a launch's first
    dimension: 2^26 and a few rows of 16 bytes, the last tokens and rows among them."""
    n = (1 << 26) + 6
    batch, seq, dim = 2, (1 << 25) + 70, 8
    banner("row packing past 2^26 rows", n, batch, seq)
    skip = batch * seq - n  # padded rows without a token
    rows = torch.arange(skip, batch * seq, device="cuda")
    b, t = (rows // seq).to(torch.int32), (rows % seq).to(torch.int32)
    gen = torch.Generator(device="cuda").manual_seed(1)
    attn = torch.randint(-99, 99, (batch, 1, seq, dim), generator=gen, device="cuda").half()
    attn.requires_grad_()
    out = att.pack_rows(attn, b, t)
    assert torch.equal(out.detach(), attn.detach().view(-1, dim)[skip:])
    grad = torch.randint(1, 99, (n, dim), generator=gen, device="cuda").half()
    back = torch.autograd.grad(out, attn, grad)[0].view(-1, dim)
    assert torch.equal(back[skip:], grad) and not back[:skip].any()


@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("batch,seq,n,heads,kv_heads,in_dtype", [
    (1, 1, 1, 1, 1, torch.float16), (3, 7, 5, 4, 2, torch.bfloat16),
    (2, 65, 130, 12, 2, torch.float32), (2, 9, 11, 28, 4, torch.float16),
    (3, 5, 0, 2, 1, torch.float16)])
def test_padded_rotation_matches_the_packed_one(batch, seq, n, heads, kv_heads, in_dtype,
                                                out_dtype):
    """va_rope_fwd_padded writes the packed rotation's rows, bit for bit, where tokens lie and zeros
    elsewhere, for rows in any order, into outputs that hold NaN and over a row map that names
    no token, a wrong token for every row, or none of the batch's; qkv_rotate(padded=True) and
    va_rope_fwd's padded layout into zeroed outputs give the same."""
    banner("padded rotation", batch, seq, n, heads, kv_heads, in_dtype, out_dtype)
    b, t = _positions(batch, seq, n, seed=n + 1)
    q = torch.randn(n, heads * 128, device="cuda").to(in_dtype)
    k, v = (torch.randn(n, kv_heads * 128, device="cuda").to(in_dtype) for _ in range(2))
    cos, sin = (torch.randn(batch, seq, 128, device="cuda") for _ in range(2))
    refs = []
    for rows in att.rope_forward(q, k, v, cos, sin, b, t, heads, kv_heads, out_dtype, expand=True):
        ref = torch.zeros(batch, heads, seq, 128, dtype=out_dtype, device="cuda")
        ref[b.long(), :, t.long()] = rows
        refs.append(ref)
    inputs = [x.data_ptr() for x in (q, k, v, cos, sin)] + [seq * 128, 128, b.data_ptr(),
                                                            t.data_ptr()]
    dtypes = [att._DTYPES[in_dtype], att._DTYPES[out_dtype]]
    for fill in (-1, 0, n - 1, 1 << 30):
        got = [torch.full_like(ref, float("nan")) for ref in refs]
        row_map = torch.full((batch * seq,), fill, dtype=torch.int32, device="cuda")
        att.check(att.lib().va_rope_fwd_padded(*inputs, row_map.data_ptr(),
                                               *(x.data_ptr() for x in got), n, batch, heads,
                                               kv_heads, 128, seq, *dtypes, att._stream()),
                  "va_rope_fwd_padded")
        torch.cuda.synchronize()
        assert all(torch.equal(x, ref) for x, ref in zip(got, refs)), fill
    got = [torch.zeros_like(ref) for ref in refs]
    att.check(att.lib().va_rope_fwd(*inputs, *(x.data_ptr() for x in got), n, heads, kv_heads, 128,
                                    seq, *dtypes, att._lib.VA_LAYOUT_PADDED, 1, att._stream()),
              "va_rope_fwd")
    torch.cuda.synchronize()
    assert all(torch.equal(x, ref) for x, ref in zip(got, refs))
    if out_dtype == torch.float16:
        got = att.qkv_rotate(q, k, v, cos, sin, b, t, batch, seq, heads, kv_heads, True)
        assert all(torch.equal(x, ref) for x, ref in zip(got, refs))


@pytest.mark.parametrize("heads,kv_heads", [(4, 2), (2, 2)])
def test_padded_rotation_without_expansion_is_refused(heads, kv_heads):
    """rope_forward into the padded layout repeats key/value heads or raises; it does not expand what
    it was told not to."""
    b, t = _positions(2, 5, 3, seed=0)
    q = torch.randn(3, heads * 128, device="cuda").half()
    k, v = (torch.randn(3, kv_heads * 128, device="cuda").half() for _ in range(2))
    cos = torch.ones(1, 5, 128, device="cuda")
    with pytest.raises(att._lib.VarlenAttnError) as e:
        att.rope_forward(q, k, v, cos, cos, b, t, heads, kv_heads, torch.float16,
                         att._lib.VA_LAYOUT_PADDED, False, 2, 5)
    assert e.value.code == att._lib.VA_EINVAL
