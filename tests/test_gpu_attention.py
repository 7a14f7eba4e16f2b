"""GPU causal grouped-query attention (neko_hip_attention) against the oracle's restatement of
cpu::attention (cpu_ops.cpp:544-575), which tests/test_oracle.py pins bit-exact to the compiled
reference and to a float64 softmax.

No canonical summation order exists -- the reference's CPU loop and its shader (attention.comp) sum
in different orders -- so the bar is a tolerance, written below: |gpu - oracle| <= TOL * (1 + |oracle|)
with TOL = 2e-6 for f32 outputs (the reference's own self-test allows 2e-3), and f16 outputs within
half an f16 ulp of the oracle's f32 result plus that bar. Shapes: the reference self-test case, the Qwen3-4B
decode (one token over 4096 and 40000 cached positions: the keys split over many workgroups and
merged) and a 256-token prefill, GPT-2 heads, head sizes 6 / 40 / 96 / 256 (the per-half and masked
loads), groups of 3, 8 and 16 query heads per kv head, strided and unaligned q / out rows, f16
activations, infinities, extreme scores, graph capture, and the argument checks. Heads of 64 and 128 run
on the matrix cores where that is estimated to be faster, the rest on the vector path.
"""
import numpy as np
import pytest
import torch

from nekochat_amd import NekoError, ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 2e-6


def _case(msg):
    print(f"[case] {msg}", flush=True)


def _inputs(T, H, KV, hd, pos0, dev, seed, q_extra=0, dtype=torch.float32):
    g = torch.Generator(device="cpu").manual_seed(seed)
    q = torch.randn((T, H * hd + q_extra), generator=g, dtype=torch.float32)
    kc = torch.randn((pos0 + T, KV * hd), generator=g, dtype=torch.float32).half()
    vc = torch.randn((pos0 + T, KV * hd), generator=g, dtype=torch.float32).half()
    if dtype == torch.float16:
        q = q.half()
    return q.to(dev), kc.to(dev), vc.to(dev)


def _oracle(q, kc, vc, H, KV, hd, pos0):
    qf = q.float().cpu().numpy()
    return O.attention(qf, kc.cpu().view(torch.int16).numpy().view(np.uint16),
                       vc.cpu().view(torch.int16).numpy().view(np.uint16), H, KV, hd, pos0)


def _check_f32(got, want, what):
    got = got.cpu().numpy()
    err = np.abs(got - want) / (1.0 + np.abs(want))
    worst = float(err.max())
    print(f"{what}: worst |gpu - oracle| / (1 + |oracle|) = {worst:.3e}", flush=True)
    assert np.isfinite(got).all(), what
    assert worst <= TOL, f"{what}: {worst:.3e} > {TOL}"


@pytest.mark.parametrize("T,H,KV,hd,pos0", [
    (3, 4, 2, 64, 1030),    # the reference self-test case (compute.cpp:262-283)
    (1, 32, 8, 128, 4095),  # Qwen3-4B decode, 4096 cached positions: 32 key splits
    (4, 32, 8, 128, 2000),  # four-sequence decode step
    (256, 32, 8, 128, 0),   # Qwen3-4B prefill of 256 tokens: eight row tiles per kv head
    (64, 12, 12, 64, 0),    # GPT-2 small: one query head per kv head
    (8, 8, 2, 256, 100),    # head size 256, one query head per work item
    (512, 8, 2, 256, 0),    # head size 256, four query heads per work item
    (5, 6, 2, 96, 70),      # head size 96: dimensions past hd masked
    (3, 4, 2, 6, 9),        # head size 6: per-half loads, one query head per work item
    (512, 4, 2, 6, 0),      # head size 6, two query heads per work item
    (7, 12, 4, 64, 200),    # three query heads per kv head
    (2, 16, 2, 128, 3000),  # eight query heads per kv head
    (1, 16, 2, 128, 40000),  # 128 key splits
    (1, 32, 8, 128, 40000),  # long context: 32, of ten tiles
    (1, 4, 1, 128, 100000),  # one kv head: 256
])
def test_attention_f32(dev, T, H, KV, hd, pos0):
    _case(f"attention f32 T={T} H={H} KV={KV} hd={hd} pos0={pos0}")
    q, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=T * 131 + hd + pos0)
    out = ops.attention(q, kc, vc, H, KV, hd, pos0)
    torch.cuda.synchronize()
    _check_f32(out, _oracle(q, kc, vc, H, KV, hd, pos0), f"attention T={T} H={H} KV={KV} hd={hd} pos0={pos0}")


def test_attention_strided_rows(dev):
    """q as the first columns of qkv rows (the models' layout) and out rows wider than n_head*hd."""
    _case("attention strided q / out rows")
    T, H, KV, hd, pos0 = 9, 8, 2, 64, 33
    qkv, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=7, q_extra=2 * KV * hd)
    q = qkv[:, : H * hd]
    out_full = torch.full((T, H * hd + 40), 7.0, dtype=torch.float32, device=dev)
    out = out_full[:, : H * hd]
    ops.attention(q, kc, vc, H, KV, hd, pos0, out=out)
    torch.cuda.synchronize()
    _check_f32(out, _oracle(q, kc, vc, H, KV, hd, pos0), "attention strided")
    assert torch.all(out_full[:, H * hd:] == 7.0), "columns past n_head*hd were written"


def test_attention_f16(dev):
    """f16 q and out: the oracle's f32 result of the same (f16-valued) q, within half an f16 ulp (the
    rounding) plus the f32 bar above."""
    _case("attention f16")
    T, H, KV, hd, pos0 = 16, 32, 8, 128, 500
    q, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=11, dtype=torch.float16)
    out = ops.attention(q, kc, vc, H, KV, hd, pos0)
    torch.cuda.synchronize()
    want = _oracle(q, kc, vc, H, KV, hd, pos0)
    got = out.float().cpu().numpy()
    half_ulp = np.spacing(np.abs(want).astype(np.float16)).astype(np.float32) / 2
    excess = np.abs(got - want) - half_ulp - TOL * (1.0 + np.abs(want))
    print(f"attention f16: worst excess over half an ulp + bar = {excess.max():.3e}", flush=True)
    assert (excess <= 0).all()


def test_attention_scale_and_single_key(dev):
    """Position 0 sees one key: out = v_0 exactly, whatever q or the scale. A zero scale weights every
    key alike: out = the mean of the v rows."""
    _case("attention single key / zero scale")
    H, KV, hd = 4, 2, 64
    q, kc, vc = _inputs(1, H, KV, hd, 0, dev, seed=3)
    out = ops.attention(q, kc, vc, H, KV, hd, 0, scale=0.37)
    torch.cuda.synchronize()
    want = torch.cat([vc[0, (h // 2) * hd:(h // 2 + 1) * hd] for h in range(H)]).float()
    assert torch.equal(out[0], want)
    T, pos0 = 2, 300
    q, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=4)
    out = ops.attention(q, kc, vc, H, KV, hd, pos0, scale=0.0)
    torch.cuda.synchronize()
    v = vc.double().cpu()
    for t in range(T):
        mean = v[: pos0 + t + 1].mean(0)
        want = torch.cat([mean[(h // 2) * hd:(h // 2 + 1) * hd] for h in range(H)])
        assert torch.allclose(out[t].double().cpu(), want, rtol=0, atol=1e-5)


# The matrix-core path (rows = tokens x query heads per kv head, 32 to a wave): one, two or four row groups
# per workgroup and key tiles of 128 or 64, at their edges, split over the keys and not; then short rows.
@pytest.mark.parametrize("T,H,KV,hd,pos0", [
    (8, 256, 64, 128, 119),  # 32 rows, 127 keys: one row group, the key tile short of one
    (8, 128, 32, 128, 119),  # the same of half the heads: the vector path
    (8, 256, 64, 64, 121),   # 129 keys: one past a tile
    (16, 128, 32, 128, 48),  # 64 rows, 64 keys: two row groups
    (17, 256, 64, 128, 100),  # 68 rows: four row groups, the third with 4 rows, the last empty
    (17, 64, 16, 128, 100),  # a quarter of the heads: the vector path
    (32, 64, 16, 64, 33),    # 128 rows, 65 keys
    (33, 16, 4, 128, 640),   # 132 rows: a second row tile of 4 rows, keys split
    (43, 6, 2, 128, 515),    # three heads per kv head: tokens straddle waves and row tiles
    (129, 12, 12, 64, 0),    # one head per kv head
    (300, 16, 1, 128, 1),    # sixteen heads per kv head, splits empty for the first rows
    (32, 8, 1, 128, 203),    # 256 rows of one kv head: the vector path
    (50, 32, 32, 128, 0),    # as much work in 1600 items: the matrix cores
    (1, 8, 2, 128, 128),     # below: a head's whole row by eight waves; 129 keys, five waves with a step
    (2, 8, 2, 128, 254),     # 256 keys: every wave's step full
    (1, 8, 2, 128, 256),     # 257 keys: split again
    (1, 6, 6, 64, 511),      # 512 keys of 64 dimensions
    (3, 4, 2, 40, 400),      # dimensions past 40 masked
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_attention_row_and_key_tiles(dev, T, H, KV, hd, pos0, dtype):
    """q rows of very different sizes (each is scaled by its own power of two). The scores' f32 rounding
    weighs on the weights by its absolute size, so q is kept to scores of a few units and the bar is
    the one above; f16 outputs as in test_attention_f16."""
    _case(f"attention tiles T={T} H={H} KV={KV} hd={hd} pos0={pos0} {dtype}")
    q, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=T + hd)
    q *= 2.0 ** torch.randint(-12, 1, (T, 1), generator=torch.Generator().manual_seed(1)).to(dev)
    q = q.to(dtype)
    out = ops.attention(q, kc, vc, H, KV, hd, pos0)
    torch.cuda.synchronize()
    want = _oracle(q, kc, vc, H, KV, hd, pos0)
    half_ulp = 0 if dtype == torch.float32 else np.spacing(np.abs(want).astype(np.float16)).astype(np.float32) / 2
    excess = np.abs(out.float().cpu().numpy() - want) - half_ulp - TOL * (1.0 + np.abs(want))
    print(f"worst excess {excess.max():.3e}", flush=True)
    assert (excess <= 0).all()


@pytest.mark.parametrize("T,pos0", [(3, 200), (2, 9000), (12, 2000), (40, 75), (40, 900)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_attention_infinities(dev, T, pos0, dtype):
    """A key of score -inf weighs nothing; an infinite or NaN v row reaches the tokens that see it and no
    earlier one, and a negative scale turns the scores round: as the oracle has it."""
    _case(f"attention infinities T={T} pos0={pos0} {dtype}")
    H, KV, hd = 8, 2, 128
    q, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=T + pos0)
    q = q.abs().to(dtype)
    kc[5] = -float("inf")
    vc[pos0 + T // 2, 3] = float("nan")
    vc[pos0 + T - 1, 7] = float("inf")
    out = ops.attention(q, kc, vc, H, KV, hd, pos0)
    torch.cuda.synchronize()
    want, got = _oracle(q, kc, vc, H, KV, hd, pos0), out.float().cpu().numpy()
    assert np.isfinite(want[0, hd:]).all() and np.isnan(want[-1, 3])
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    bar = 5e-4 if dtype == torch.float16 else TOL  # an f16 rounding: 2^-11
    assert (np.abs(got - want)[ok] <= bar * (1 + np.abs(want[ok]))).all()
    kc[5] = 1.0
    vc = torch.nan_to_num(vc, nan=0.0, posinf=0.0)
    a = ops.attention(q, kc, vc, H, KV, hd, pos0, scale=-0.1)
    b = ops.attention(-q, kc, vc, H, KV, hd, pos0, scale=0.1)
    assert torch.equal(a, b)


@pytest.mark.parametrize("T,H,KV,hd,pos0", [(1, 32, 8, 128, 4095), (70, 8, 2, 64, 900)])
@pytest.mark.parametrize("warm", [False, True])
def test_attention_captured(dev, T, H, KV, hd, pos0, warm):
    """Under graph capture the workspace cannot grow: a fresh context's matrix-core call takes as many key
    splits as fit (here one); after an eager call it takes the same splits. Replays follow their inputs."""
    _case(f"attention captured T={T} H={H} KV={KV} hd={hd} pos0={pos0} warm={warm}")
    from nekochat_amd._lib import lib
    ctx = ops.Context(dev.index)
    q, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=T + pos0)
    out, eager = torch.zeros_like(q), torch.zeros_like(q)
    scale = 1.0 / hd ** 0.5

    def call(o):
        assert lib.neko_hip_set_stream(ctx.handle, torch.cuda.current_stream().cuda_stream or None) == 0
        return lib.neko_hip_attention(ctx.handle, q.data_ptr(), q.stride(0), kc.data_ptr(), vc.data_ptr(), o.data_ptr(),
                                      o.stride(0), T, H, KV, hd, pos0, scale, ops.DT_F32)

    if warm:
        assert call(eager) == 0
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        rc = call(out)
    assert rc == 0, lib.neko_hip_last_error(ctx.handle).decode()
    for k in range(3):
        q.mul_(0.75)
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        _check_f32(out, _oracle(q, kc, vc, H, KV, hd, pos0), f"replay {k}")
        if warm:
            assert call(eager) == 0
            torch.cuda.synchronize()
            assert torch.equal(out, eager)
    assert lib.neko_hip_set_stream(ctx.handle, None) == 0
    ctx.close()


@pytest.mark.parametrize("T,H,KV,hd,pos0,n", [
    (1, 8, 2, 128, 200, 100),      # one workgroup per head: three waves see only such keys
    (1, 8, 2, 96, 9000, 3000),     # whole splits
    (300, 8, 2, 96, 0, 70),        # no splits: the first 70 tokens see nothing else
    (12, 8, 2, 128, 2000, 200),    # the matrix cores: some waves and splits see only such keys
    (2, 8, 2, 128, 9000, 3000),    # whole splits
    (40, 8, 2, 64, 900, 130),
    (43, 6, 2, 128, 515, 150),     # rows done again: three heads of a token, across waves and row tiles
    (129, 12, 12, 64, 0, 70),      # one head each
    (70, 16, 1, 128, 400, 130),    # sixteen: items of four
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("low", [-float("inf"), float("nan")])
def test_attention_infinite_prefix(dev, T, H, KV, hd, pos0, n, dtype, low):
    """The first n keys score -inf (weight 0, and NaN for a token that sees only such) or NaN, whole steps, waves
    and splits of them: as the oracle has it."""
    _case(f"attention infinite prefix T={T} H={H} KV={KV} hd={hd} pos0={pos0} n={n} {dtype} {low}")
    q, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=T + pos0)
    q = q.abs().to(dtype)
    kc[:n] = low
    out = ops.attention(q, kc, vc, H, KV, hd, pos0)
    torch.cuda.synchronize()
    want, got = _oracle(q, kc, vc, H, KV, hd, pos0), out.float().cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = np.isfinite(want)
    bar = 5e-4 if dtype == torch.float16 else TOL
    assert (np.abs(got - want)[ok] <= bar * (1 + np.abs(want[ok]))).all()


@pytest.mark.parametrize("T,H,KV,hd,pos0", [(1, 32, 8, 128, 5000), (24, 16, 8, 128, 600), (130, 16, 4, 64, 300)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("size", [-1e4, -1e8, -2e9, -1e12, -1e30, 1e8, 2e9, 1e12, 1e30])
def test_attention_extreme_scores(dev, T, H, KV, hd, pos0, dtype, size):
    """Scores of about 10 times `size` (f32 q of that size, or an f16 q under such a scale), apart by more than
    any weight survives: only the keys of the largest weigh, all alike."""
    _case(f"attention extreme scores T={T} H={H} KV={KV} hd={hd} pos0={pos0} {dtype} {size}")
    _, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=T + pos0)
    level = torch.arange(pos0 + T, device=dev) % 7
    kc[:] = (1.0 + level / 8.0)[:, None].half()
    heads = (1.0 + torch.arange(H, device=dev) / 64.0).repeat_interleave(hd).repeat(T, 1)
    heads = heads if size > 0 else -heads
    if dtype == torch.float32:
        out = ops.attention(heads * abs(size), kc, vc, H, KV, hd, pos0)
    else:
        out = ops.attention(heads.half(), kc, vc, H, KV, hd, pos0, scale=abs(size) / hd ** 0.5)
    torch.cuda.synchronize()
    v = vc.double().cpu()
    for t in (0, T // 2, T - 1):
        want = v[: pos0 + t + 1][(level[: pos0 + t + 1] == (0 if size < 0 else 6)).cpu()].mean(0)
        want = torch.cat([want[(h // (H // KV)) * hd:(h // (H // KV) + 1) * hd] for h in range(H)])
        bar = TOL if dtype == torch.float32 else 5e-4  # an f16 rounding: 2^-11
        assert ((out[t].double().cpu() - want).abs() <= bar * (1 + want.abs())).all()


@pytest.mark.parametrize("gap", [14.0, 18.0, 21.0, 22.0, 26.0])
@pytest.mark.parametrize("H,KV,keys,hd", [(32, 8, 32768, 128), (16, 4, 32768, 64), (520, 520, 8192, 64),
                                           (260, 260, 8192, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_attention_dominant_key(dev, H, KV, keys, hd, gap, dtype):
    """One key `gap` nats above all others, its v zero and theirs of mean 1: the output is their weights' sum.
    Every kv head holds the same, so that few (keys split) and many (not) share a reference in 64 bits. The
    bar: the f32 bar, relative here, and a weight's rounding of 2^-39 of the largest for every key."""
    _case(f"attention dominant key H={H} KV={KV} keys={keys} hd={hd} gap={gap} {dtype}")
    g = torch.Generator().manual_seed(int(gap) + hd)
    k, v = 0.25 * torch.randn((keys, hd), generator=g), 1.0 + 0.25 * torch.randn((keys, hd), generator=g)
    q = 0.25 * torch.randn((1, hd), generator=g)
    sink = keys // 3
    k[:, 0] = 0.0
    k[sink] = v[sink] = 0.0
    k[sink, 0], q[0, 0] = 8.0, gap * hd ** 0.5 / 8.0
    k, v, q = k.half(), v.half(), q.to(dtype)
    s = (k.double() @ q[0].double()) / hd ** 0.5
    want = torch.softmax(s, 0) @ v.double()
    out = ops.attention(q.to(dev).repeat(1, H), k.to(dev).repeat(1, KV), v.to(dev).repeat(1, KV), H, KV, hd, keys - 1)
    torch.cuda.synchronize()
    err = (out.double().cpu().reshape(H, hd) - want).abs()
    if dtype == torch.float16:
        err -= torch.from_numpy(np.spacing(np.abs(want.numpy()).astype(np.float16)).astype(np.float64)) / 2
    print(f"worst error {err.max():.3e} of {want.abs().max():.3e}", flush=True)
    assert (err <= TOL * want.abs() + keys * 2.0 ** -39).all()


@pytest.mark.parametrize("T,H,KV,hd,pos0", [
    (9, 32, 8, 128, 700), (33, 16, 4, 128, 640), (130, 12, 12, 64, 20), (40, 12, 4, 64, 1500),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("off,pad", [(0, 40), (1, 0), (0, 1), (1, 7)])
def test_attention_mfma_layouts(dev, T, H, KV, hd, pos0, dtype, off, pad):
    """The matrix-core path over q and out rows that are padded, off 16-byte alignment by one element, or of an odd
    stride (element loads and stores); nothing beside the out rows is written."""
    _case(f"attention layouts T={T} H={H} KV={KV} hd={hd} pos0={pos0} {dtype} off={off} pad={pad}")
    q, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=T + pos0)
    W = H * hd
    qfull = torch.full((off + T * (W + pad),), float("nan"), dtype=dtype, device=dev)
    qs = qfull[off:].view(T, W + pad)[:, :W]
    qs.copy_(q)
    ofull = torch.full((off + T * (W + pad) + 8,), 7.0, dtype=dtype, device=dev)
    o = ofull[off:-8].view(T, W + pad)
    ops.attention(qs, kc, vc, H, KV, hd, pos0, out=o[:, :W])
    torch.cuda.synchronize()
    want = _oracle(qs.contiguous(), kc, vc, H, KV, hd, pos0)
    half_ulp = 0 if dtype == torch.float32 else np.spacing(np.abs(want).astype(np.float16)).astype(np.float32) / 2
    excess = np.abs(o[:, :W].float().cpu().numpy() - want) - half_ulp - TOL * (1.0 + np.abs(want))
    assert (excess <= 0).all()
    assert bool((o[:, W:] == 7.0).all()) and bool((ofull[:off] == 7.0).all()) and bool((ofull[-8:] == 7.0).all())


@pytest.mark.parametrize("T,H,KV,hd,pos0", [(1, 32, 8, 128, 5000), (130, 12, 12, 64, 20)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_attention_mfma_zero_scale(dev, T, H, KV, hd, pos0, dtype):
    """A zero scale on the matrix cores: the mean of the v rows, splits and prompts."""
    _case(f"attention zero scale T={T} H={H} KV={KV} hd={hd} pos0={pos0} {dtype}")
    q, kc, vc = _inputs(T, H, KV, hd, pos0, dev, seed=T)
    out = ops.attention(q.to(dtype), kc, vc, H, KV, hd, pos0, scale=0.0)
    torch.cuda.synchronize()
    mean = vc.double().cumsum(0)[pos0:] / torch.arange(pos0 + 1, pos0 + T + 1, device=dev)[:, None]
    want = mean.reshape(T, KV, 1, hd).expand(T, KV, H // KV, hd).reshape(T, H * hd)
    bar = TOL if dtype == torch.float32 else 5e-4  # an f16 rounding: 2^-11
    assert bool(((out.double() - want).abs() <= bar * (1 + want.abs())).all())


@pytest.mark.parametrize("H,KV,hd,pos0", [
    (1, 1, 96, 40000),    # 313 splits, each item one query head
    (2, 1, 256, 30000),   # 469
    (4, 1, 96, 100000),   # 782 splits of items of four query heads (38 MB of K and V)
    (16, 2, 256, 40000),  # two blocks of four
])
def test_attention_vector_splits(dev, H, KV, hd, pos0):
    """Head sizes of the vector path at long decode: splits past 256, which the merge's threads take several of,
    and items of four query heads with split keys."""
    _case(f"attention vector splits H={H} KV={KV} hd={hd} pos0={pos0}")
    q, kc, vc = _inputs(1, H, KV, hd, pos0, dev, seed=hd + pos0)
    out = ops.attention(q, kc, vc, H, KV, hd, pos0)
    torch.cuda.synchronize()
    _check_f32(out, _oracle(q, kc, vc, H, KV, hd, pos0), f"attention H={H} KV={KV} hd={hd} pos0={pos0}")


def test_attention_argument_checks(dev):
    _case("attention argument checks")
    q, kc, vc = _inputs(2, 4, 2, 64, 5, dev, seed=5)
    assert ops.attention(q[:0], kc, vc, 4, 2, 64, 5).shape == (0, 256)  # no tokens: nothing to do
    with pytest.raises(NekoError):
        ops.attention(q, kc, vc, 3, 2, 64, 5)  # n_head not a multiple of n_kv
    with pytest.raises(NekoError):
        ops.attention(q, kc[:6], vc, 4, 2, 64, 5)  # caches shorter than pos0 + T
    qo, kco, vco = _inputs(2, 4, 2, 63, 5, dev, seed=6)
    with pytest.raises(NekoError):
        ops.attention(qo, kco, vco, 4, 2, 63, 5)  # odd head size
    with pytest.raises(NekoError):
        ops.attention(q, kc, vc, 4, 2, 64, 5, out=q)  # out over q
