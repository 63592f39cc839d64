"""Launches that move more than the last-level cache holds (256 MB) run some kernels with another
number of waves per SIMD than launches that fit it: the same tensors in one launch of each size give
the same params, codes and scales bit for bit."""
import pytest
import torch

import mdq_hip

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
N = 2_650_003          # elements a tensor: 8 of them move 297 MB or more, 2 of them 148 MB or less
CODES = {4: (torch.uint8, None), 8: (torch.int8, torch.uint8), 16: (torch.int16, torch.uint16), 32: (torch.int32, torch.uint32)}
SIGNED = {torch.uint16: torch.int16, torch.uint32: torch.int32}


def rand_bytes(n, gen):
    return torch.randint(0, 256, (n,), dtype=torch.uint8, device=DEV, generator=gen)


def codes(bits, n, gen):
    mdt, vdt = CODES[bits]
    m = rand_bytes(n * mdt.itemsize, gen).view(mdt)
    return m, torch.empty(0, dtype=torch.uint8, device=DEV) if vdt is None else rand_bytes(n * vdt.itemsize, gen).view(vdt)


def state(bits, B, grad, count, views, gen):
    """``count`` tensors' entries; with ``views`` params and grads lie back to back at odd offsets."""
    total = count * (N if views else -(-N // 64) * 64) + 64
    p = torch.randn(total, device=DEV, generator=gen) * 0.02
    g = (torch.randn(total, device=DEV, generator=gen) * 1e-3).to(grad)
    out, nb = [], -(-N // B)
    for k in range(count):
        o = k * N + 1 if views else k * (-(-N // 64) * 64)
        m, v = codes(bits, N, gen)
        r = torch.rand(3, nb, device=DEV, generator=gen)
        out.append(mdq_hip.TensorState(p[o:o + N], g[o:o + N], m, v, r[0] * 1e-4 / 2 ** (bits - 1), r[1] / 2 ** bits + 1e-12,
                                       -14.0 - r[2], 7, bits, 1e-3, 0.9, 0.999, 1e-8, 0.01, k))
    return out


def copy(entries, views):
    """The same values, params as views of one buffer again."""
    base = entries[0].p.storage_offset()
    end = entries[-1].p.storage_offset() + N
    flat = torch.as_strided(entries[0].p, (end,), (1,), 0).clone()
    assert views == bool(base)
    return [mdq_hip.TensorState(flat[e.p.storage_offset():e.p.storage_offset() + N], e.grad, e.exp_avg.clone(), e.exp_avg_sq.clone(),
                                e.scale_m.clone(), e.scale_v.clone(), e.v_min.clone(), e.step, e.bits, e.lr, e.beta1, e.beta2, e.eps,
                                e.weight_decay, e.tensor_id) for e in entries]


def assert_same(a, b):
    for x, y in zip(a, b):
        for k in ("p", "exp_avg", "exp_avg_sq", "scale_m", "scale_v", "v_min"):
            s, t = getattr(x, k), getattr(y, k)
            s, t = (u.view(torch.int32) if u.dtype == torch.float32 else u.view(SIGNED.get(u.dtype, u.dtype)) for u in (s, t))
            assert torch.equal(s, t), f"tensor {x.tensor_id}: {k}"


@pytest.mark.parametrize("bits,B,grad,rounding,views", [
    (4, 1024, torch.float32, "nearest", False), (4, 1024, torch.float32, "stochastic", False),
    (8, 1024, torch.float32, "nearest", False), (16, 1024, torch.float32, "nearest", True),
    (32, 1024, torch.bfloat16, "nearest", False), (32, 1024, torch.float32, "nearest", True),
    (8, 64, torch.float32, "nearest", True), (8, 16, torch.float32, "nearest", True)])
def test_one_large_launch_equals_small_ones(bits, B, grad, rounding, views):
    print(f"case: large and small launches bits={bits} B={B} {grad} {rounding} views={views}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(bits * B)
    whole = state(bits, B, grad, 8, views, gen)
    parts = copy(whole, views)
    mdq_hip.multi_tensor_step(whole, B, rounding=rounding, seed=3)
    for k in range(0, 8, 2):
        mdq_hip.multi_tensor_step(parts[k:k + 2], B, rounding=rounding, seed=3)
    assert_same(whole, parts)


@pytest.mark.parametrize("grad", [torch.float32, torch.float16])
def test_one_large_storage_change_equals_small_ones(grad):
    print(f"case: large and small storage changes {grad}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(11)
    whole = state(32, 128, grad, 8, False, gen)
    for e in whole:
        e.bits = 4
        e.scale_m *= 2.0 ** 28
        e.scale_v *= 2.0 ** 28
    parts = copy(whole, False)
    outs = [[mdq_hip.empty_codes(e.exp_avg, mdq_hip.STORE_P4) for e in whole] for _ in range(2)]
    mdq_hip.multi_tensor_restore(whole, outs[0], 128)
    for k in range(0, 8, 2):
        mdq_hip.multi_tensor_restore(parts[k:k + 2], outs[1][k:k + 2], 128)
    for es, os in zip((whole, parts), outs):
        for e, (m, v) in zip(es, os):
            e.exp_avg, e.exp_avg_sq = m, v
    assert_same(whole, parts)


@pytest.mark.parametrize("bits,B,grad,n", [(4, 1024, torch.float32, 20_000_003), (16, 256, torch.bfloat16, 15_000_000),
                                           (32, 1024, torch.float32, 10_000_001)])
def test_one_large_tensor_equals_its_pieces(bits, B, grad, n):
    """One tensor in a call of its own, and the same as block-aligned pieces, each in a call of its own."""
    print(f"case: one large tensor and its pieces bits={bits} B={B} {grad}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(n)
    nb = -(-n // B)
    m, v = codes(bits, n, gen)
    r = torch.rand(3, nb, device=DEV, generator=gen)
    whole = mdq_hip.TensorState(torch.randn(n, device=DEV, generator=gen) * 0.02,
                                (torch.randn(n, device=DEV, generator=gen) * 1e-3).to(grad), m, v, r[0] * 1e-4 / 2 ** (bits - 1),
                                r[1] / 2 ** bits + 1e-12, -14.0 - r[2], 7, bits, 1e-3, 0.9, 0.999, 1e-8, 0.01, 0)
    split = mdq_hip.TensorState(*(t.clone() for t in (whole.p, whole.grad, m, v, whole.scale_m, whole.scale_v, whole.v_min)),
                                7, bits, 1e-3, 0.9, 0.999, 1e-8, 0.01, 0)
    mdq_hip.multi_tensor_step([whole], B)
    for rank in range(4):
        mdq_hip.multi_tensor_step(mdq_hip.shard_states([split], B, 4, rank), B)
    assert_same([whole], [split])
