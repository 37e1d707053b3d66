"""GPU parity of single kernels at the sizes where their tiles, rings and splits begin and end,
against the CPU oracle with the tolerances of test_gpu_attention.py."""

import numpy as np
import pytest
import torch

from hackaton_amd import attention as att
from hackaton_amd import workloads as wl
from tests.test_gpu_attention import SCALE, TOL, banner, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [[1, 31, 32, 33], [63, 64, 65], [95, 96, 97, 127],
                                     [128, 129, 160, 161], [255, 256, 257], [383, 385]])
@pytest.mark.parametrize("hq,hkv,dtype", [(3, 1, torch.float16), (14, 2, torch.bfloat16)])
def test_many_item_forward_at_tile_and_ring_edges(lengths, hq, hkv, dtype):
    """One, two, three and more 32-key tiles through the three-stage ring, with full and partial
    last tiles and strips, documents before and after each other in one packed array."""
    banner("many-item forward edges", lengths, hq, hkv, dtype)
    q, k, v, do = wl.make_inputs(lengths, hq, hkv, dtype, seed=sum(lengths))
    n, dev = sum(lengths), torch.device("cuda")
    plan = att._plan(att._cu_seqlens(lengths, dev), hq, hkv)
    qd, kd, vd = (t.to(dev) for t in (q, k, v))
    out = torch.full_like(qd, float("nan"))
    lse = torch.full((hq, n), float("nan"), dtype=torch.float32, device=dev)
    att.check(att.lib().va_fwd_kernel(att._lib.VA_FWD_MANY, qd.data_ptr(), kd.data_ptr(),
                                      vd.data_ptr(), out.data_ptr(), lse.data_ptr(),
                                      plan.fwd_items.data_ptr(), plan.n_fwd, n, hq, hkv, 128,
                                      SCALE, 0 if dtype == torch.float16 else 1, att._stream()),
              "va_fwd_kernel")
    torch.cuda.synchronize()
    o_ref, lse_ref = oracle(q, k, v, do, lengths)[:2]
    assert float(np.max(np.abs(out.cpu().float().numpy() - o_ref))) <= TOL[dtype]["o"]
    assert float(np.max(np.abs(lse.cpu().numpy() - lse_ref))) <= TOL[dtype]["lse"]


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
    rows in any order; the backward's row map scratch and output hold anything before (here a map
    that names a wrong token for every row)."""
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


@pytest.mark.parametrize("batch,seq,n,heads,kv_heads,in_dtype", [
    (1, 1, 1, 1, 1, torch.float16), (3, 7, 5, 4, 2, torch.bfloat16),
    (2, 65, 130, 12, 2, torch.float32), (2, 9, 11, 28, 4, torch.float16),
    (3, 5, 0, 2, 1, torch.float16)])
def test_padded_rotation_matches_the_packed_one(batch, seq, n, heads, kv_heads, in_dtype):
    """qkv_rotate(padded=True) holds the packed rotation's rows, bit for bit, where tokens lie and
    zeros elsewhere, for rows in any order and outputs from memory that held other values."""
    banner("padded rotation", batch, seq, n, heads, kv_heads, in_dtype)
    b, t = _positions(batch, seq, n, seed=n + 1)
    q = torch.randn(n, heads * 128, device="cuda").to(in_dtype)
    k, v = (torch.randn(n, kv_heads * 128, device="cuda").to(in_dtype) for _ in range(2))
    cos, sin = torch.randn(batch, seq, 128, device="cuda"), torch.randn(batch, seq, 128, device="cuda")
    packed = att.qkv_rotate(q, k, v, cos, sin, b, t, batch, seq, heads, kv_heads)
    junk = torch.full((4 * batch * heads * seq * 128,), float("nan"), device="cuda").half()
    del junk  # the allocator hands its memory out again
    padded = att.qkv_rotate(q, k, v, cos, sin, b, t, batch, seq, heads, kv_heads, True)
    for rows, got in zip(packed, padded):
        ref = torch.zeros(batch, heads, seq, 128, dtype=torch.float16, device="cuda")
        ref[b.long(), :, t.long()] = rows
        assert torch.equal(got, ref)
