"""GPU parity of the quantized kernels (wl_dequant, wl_gemv, wl_linear, wl_gemv_batch, wl_gemv_combine) against the
CPU oracle. Dequantized weights must be bit-exact; products within the normwise bound 2e-3 (fp32 accumulation), or
4e-3 for wl_linear, whose output is rounded to bf16 (up to 2^-8 relative, less in the norm) as the reference's bf16
F.linear is."""
import os

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from gguf import synth
from oracle import moe_ref
from oracle import quants_ref as q

pytestmark = pytest.mark.gpu
TOL = 2e-3
GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "known_blocks.npz")


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("name", ["Q4_K", "Q6_K"])
def test_dequant_known_blocks(hip, name):
    g = np.load(GOLDEN)
    blocks, values = g[name.lower() + "_blocks"], g[name.lower() + "_values"]
    out = hip.dequantize_gpu(dev(blocks), name, (len(blocks), 256), torch.float32).cpu().numpy()
    np.testing.assert_array_equal(out, values)


@pytest.mark.parametrize("name,rows,k", [("Q4_K", 512, 2048), ("Q6_K", 2048, 512), ("Q4_K", 3, 256),
                                         ("Q6_K", 5, 768), ("Q4_K", 7, 2560)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_dequant_bit_exact(hip, name, rows, k, dtype):
    print(f"[dequant] {name} {rows}x{k} {dtype}", flush=True)
    rng = np.random.default_rng(rows * 7 + k)
    w = synth.matrix(rng, name, rows, k)
    expect = q.dequantize(w, name, (rows, k), dtype)
    got = hip.dequantize_gpu(dev(w), name, (rows, k), torch.bfloat16 if dtype == "bf16" else torch.float32)
    got = got.cpu()
    got = got.view(torch.int16).numpy().view(np.uint16) if dtype == "bf16" else got.numpy()
    np.testing.assert_array_equal(got.view(np.uint16 if dtype == "bf16" else np.uint32),
                                  expect.view(np.uint16 if dtype == "bf16" else np.uint32))


@pytest.mark.parametrize("name", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("pad", [0, 96])
def test_dequant_nonfinite_and_strided(hip, name, pad):
    """bf16 values are the fp32 ones rounded to nearest even, NaN as 0x7FC0, also where a block's scale is infinite or
    NaN (the lanes that leave the packed conversion), with dense rows and with padding between them."""
    rows, k = 5, 768
    w = synth.matrix(np.random.default_rng(77), name, rows, k).reshape(rows, -1)
    per, at = (144, 0) if name == "Q4_K" else (210, 208)
    for r, bits in ((1, 0x7C00), (2, 0xFC00), (3, 0x7E01)):  # inf, -inf, NaN with a payload, in block r - 1 of row r
        w[r, per * (r - 1) + at:per * (r - 1) + at + 2] = np.frombuffer(np.uint16(bits).tobytes(), np.uint8)
    stride = w.shape[1] + pad
    padded = np.zeros((rows, stride), np.uint8)
    padded[:, :w.shape[1]] = w
    raw = dev(padded)
    out = {}
    for code, dtype in ((hip.DTYPE_F32, torch.float32), (hip.DTYPE_BF16, torch.bfloat16)):
        out[code] = torch.empty(rows, k, dtype=dtype, device="cuda")
        assert hip.library().wl_dequant(hip.TYPE_IDS[name], raw.data_ptr(), rows, k, stride, code, out[code].data_ptr(),
                                        torch.cuda.current_stream().cuda_stream) == 0
    f = out[hip.DTYPE_F32].cpu().numpy()
    ok = np.isfinite(f)
    assert not ok.all() and ok[0].all() and ok[4].all()
    u = f.view(np.uint32).astype(np.uint64)
    want = np.where(np.isnan(f), 0x7FC0, (u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    np.testing.assert_array_equal(out[hip.DTYPE_BF16].cpu().view(torch.int16).numpy().view(np.uint16), want)


def test_gemv_config0(hip):
    """The 512x2048 Q4_K GEMV (seed 0)."""
    case = synth.gemv_case(0)
    expect = case["x"] @ q.dequantize_matrix(case["w"], "Q4_K", 512, 2048).T
    got = hip.gemv(dev(case["w"]), "Q4_K", (512, 2048), dev(case["x"])).cpu().numpy()
    err = moe_ref.rel_err(got, expect)
    print(f"[gemv c0] rel err {err:.2e}", flush=True)
    assert err < TOL


@pytest.mark.parametrize("name,rows,k,tokens", [
    ("Q4_K", 1024, 2048, 1), ("Q4_K", 512, 2048, 3), ("Q4_K", 512, 2048, 8), ("Q4_K", 100, 2048, 11),
    ("Q6_K", 2048, 512, 1), ("Q6_K", 2048, 512, 5), ("Q6_K", 33, 256, 2), ("Q6_K", 17, 768, 1),
    ("Q4_K", 64, 512, 4), ("Q4_K", 9, 1024, 1), ("Q6_K", 40, 2560, 3), ("Q4_K", 5, 4096, 2)])
def test_gemv_shapes(hip, name, rows, k, tokens):
    print(f"[gemv] {name} {rows}x{k} T={tokens}", flush=True)
    case = synth.gemv_case(rows + k + tokens, rows, k, name, tokens)
    w32 = q.dequantize_matrix(case["w"], name, rows, k).astype(np.float64)
    expect = case["x"].astype(np.float64) @ w32.T
    got = hip.gemv(dev(case["w"]), name, (rows, k), dev(case["x"])).cpu().numpy()
    assert moe_ref.rel_err(got, expect) < TOL


@pytest.mark.parametrize("name,rows,k", [
    ("Q4_K", 1, 256), ("Q6_K", 37, 512), ("Q4_K", 130, 768), ("Q6_K", 31, 1024), ("Q4_K", 97, 2048),
    ("Q6_K", 65, 2560), ("Q4_K", 33, 4096), ("Q6_K", 21, 6400), ("Q4_K", 4201, 2048), ("Q6_K", 16500, 2048)])
@pytest.mark.parametrize("tokens", [1, 2, 7, 8])
def test_gemv_forms(hip, name, rows, k, tokens):
    """Every split of the GEMV (blocks per row 1 .. 25 over lanes, wavefronts and the K loop; 1, 2 and 4 rows per lane
    group; a last workgroup with missing rows) in fp32, and bf16 in and out: the kernel's fp32 sums on the same values,
    rounded once. Bound: 2 roundings per product and add of the longest chain (under 64 of them, errors of either sign)
    over sum |w x|, and bf16's half ulp."""
    rng = np.random.default_rng(rows + 3 * k + tokens)
    w = synth.matrix(rng, name, rows, k)
    w64 = q.dequantize_matrix(w, name, rows, k).astype(np.float64)
    xb = torch.from_numpy(rng.standard_normal((tokens, k)).astype(np.float32)).to(torch.bfloat16)
    x64 = xb.double().numpy()
    expect, size = x64 @ w64.T, np.abs(x64) @ np.abs(w64).T
    # the runs' unsigned form (a * q, b apart) makes terms up to a few times |w x|
    bound = 64 * 2.0 ** -24 * 4 * size + 1e-30
    raw = dev(w).reshape(-1)
    got = hip.gemv(raw, name, (rows, k), xb.cuda().float())
    assert (np.abs(got.cpu().double().numpy() - expect) <= bound).all()
    y = F.linear(xb.cuda(), hip.GGMLWeight(raw, name, (rows, k)))
    assert y.dtype == torch.bfloat16 and torch.equal(y, got.to(torch.bfloat16))
    odd = torch.empty(tokens * k + 1, dtype=torch.bfloat16, device="cuda")[1:].view(tokens, k).copy_(xb)
    assert torch.equal(F.linear(odd, hip.GGMLWeight(raw, name, (rows, k))), y)  # x off a 16-byte boundary


@pytest.mark.parametrize("name,rows,k", [("Q4_K", 512, 2048), ("Q6_K", 512, 2048), ("Q4_K", 40, 4096),
                                         ("Q6_K", 24, 8704)])
@pytest.mark.parametrize("tokens", [1, 8])
def test_gemv_small_x(hip, name, rows, k, tokens):
    """x 2^-110 gives y 2^-110 bit for bit: scaling by a power of two rounds the same while nothing is subnormal. x holds
    all 24 bits and |x| is in [2^-6, 4), so every product and sum of a run is a multiple of 2^-139, a normal number or an
    exact subnormal; a kernel that scales the products down further loses their low bits."""
    rng = np.random.default_rng(rows + k + tokens)
    raw = dev(synth.matrix(rng, name, rows, k)).reshape(-1)
    x = rng.uniform(2.0 ** -6, 4.0, (tokens, k)) * rng.choice((-1.0, 1.0), (tokens, k))
    x = torch.from_numpy(x.astype(np.float32)).cuda()
    y = hip.gemv(raw, name, (rows, k), x)
    assert torch.equal(hip.gemv(raw, name, (rows, k), x * 2.0 ** -110), y * 2.0 ** -110)


@pytest.mark.parametrize("name,rows,k", [
    ("Q4_K", 33, 256), ("Q6_K", 37, 512), ("Q4_K", 130, 768), ("Q6_K", 31, 1024), ("Q4_K", 65, 1280), ("Q6_K", 70, 1792),
    ("Q4_K", 4096, 2048), ("Q6_K", 2100, 2048), ("Q4_K", 4096, 2560), ("Q6_K", 1030, 4096), ("Q4_K", 8201, 2304),
    ("Q6_K", 700, 2816), ("Q6_K", 600, 4352), ("Q6_K", 130, 8192), ("Q4_K", 2050, 8448), ("Q4_K", 300, 8704),
    ("Q6_K", 17, 33024)])
@pytest.mark.parametrize("tokens", [1, 3, 8])
def test_gemv_sums_as_batch(hip, name, rows, k, tokens):
    """gemv's bits are gemv_batch's for each token, whatever the split: blocks over lanes, over wavefronts (one round and
    more, the last one short), 1, 2 and 4 rows per lane group, missing rows. fp32 in and out, and the two mixed forms:
    bf16 x gives the bits of its fp32 values, bf16 y is y rounded once."""
    rng = np.random.default_rng(rows + k + tokens)
    raw = dev(synth.matrix(rng, name, rows, k)).reshape(-1)
    xb = torch.from_numpy(rng.standard_normal((tokens, k)).astype(np.float32)).cuda().to(torch.bfloat16)
    x = xb.float()
    y = hip.gemv(raw, name, (rows, k), x)
    alone = torch.zeros(1, rows, device="cuda")
    for t in range(tokens):
        hip.gemv_batch(raw, name, (rows, k), x[t], [0], [0], alone)
        assert torch.equal(y[t], alone[0]), t
    for xin, in_code, out_code, out in ((xb, hip.DTYPE_BF16, hip.DTYPE_F32, torch.empty_like(y)),
                                        (x, hip.DTYPE_F32, hip.DTYPE_BF16, torch.empty_like(y, dtype=torch.bfloat16))):
        assert hip.library().wl_gemv_dtype(hip.TYPE_IDS[name], raw.data_ptr(), rows, k, hip.row_bytes(name, k),
                                           xin.data_ptr(), in_code, tokens, out.data_ptr(), out_code,
                                           torch.cuda.current_stream().cuda_stream) == 0
        assert torch.equal(out, y.to(out.dtype))


@pytest.mark.parametrize("name,k", [("Q4_K", 768), ("Q6_K", 2048), ("Q4_K", 4096)])
def test_gemv_strided_and_nonfinite(hip, name, k):
    """Rows with padding between them give the dense rows' bits; an infinity or a NaN in one token's x reaches that
    token's outputs alone, as in the dense product, in fp32 and in bf16."""
    rows, tokens, pad = 45, 5, 48
    w = synth.matrix(np.random.default_rng(k), name, rows, k).reshape(rows, -1)
    padded = np.full((rows, w.shape[1] + pad), 0xFF, np.uint8)
    padded[:, :w.shape[1]] = w
    raw, strided = dev(w).reshape(-1), dev(padded)
    x = torch.from_numpy(np.random.default_rng(k + 1).standard_normal((tokens, k)).astype(np.float32)).cuda()
    y = hip.gemv(raw, name, (rows, k), x)
    out = torch.empty_like(y)
    assert hip.library().wl_gemv(hip.TYPE_IDS[name], strided.data_ptr(), rows, k, strided.shape[1], x.data_ptr(), tokens,
                                 out.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out, y)
    x[1, 5], x[3, k - 1] = float("inf"), float("nan")
    clean = [0, 2, 4]
    for xin in (x, x.to(torch.bfloat16)):
        bad = F.linear(xin, hip.GGMLWeight(raw, name, (rows, k)))
        ref = hip.gemv(raw, name, (rows, k), xin.float())
        assert not torch.isfinite(bad[1]).any() and torch.isnan(bad[3]).all() and torch.isfinite(bad[clean]).all()
        assert torch.equal(bad[clean], ref[clean].to(bad.dtype))
    assert torch.equal(hip.gemv(raw, name, (rows, k), x)[clean], y[clean])


def test_gemv_batch_and_combine(hip):
    """gate_up of 4 experts in one launch (gemv_batch), then down + weighted sum (gemv_combine), as
    Engine.batched_decode_experts drives them (engines/base.py:492-532)."""
    rng = np.random.default_rng(21)
    E, H, I = 6, 2048, 512
    gu = synth.matrix(rng, "Q4_K", 2 * I, H, count=E).reshape(E, -1)
    dn = synth.matrix(rng, "Q6_K", H, I, count=E).reshape(E, -1)
    x = rng.standard_normal(H).astype(np.float32)
    picks = [4, 1, 5, 2]
    gu_d, dn_d = dev(gu), dev(dn)
    out = torch.zeros(len(picks), 2 * I, dtype=torch.float32, device="cuda")
    hip.gemv_batch(gu_d, "Q4_K", (2 * I, H), dev(x), [e * gu.shape[1] for e in picks], [3, 0, 1, 2], out)
    out = out.cpu().numpy()
    for pos, e in zip([3, 0, 1, 2], picks):
        expect = q.dequantize_matrix(gu[e], "Q4_K", 2 * I, H) @ x
        assert moe_ref.rel_err(out[pos], expect) < TOL
    h = rng.standard_normal((len(picks), I)).astype(np.float32)
    weights = rng.random(8).astype(np.float32)
    perm = [6, 0, 3, 1]
    y = hip.gemv_combine(dn_d, "Q6_K", (H, I), dev(h), [e * dn.shape[1] for e in picks], dev(weights), perm)
    expect = sum(weights[perm[i]] * (q.dequantize_matrix(dn[e], "Q6_K", H, I).astype(np.float64) @ h[i])
                 for i, e in enumerate(picks))
    assert moe_ref.rel_err(y.cpu().numpy()[0], expect) < TOL


def test_ggml_weight_linear(hip):
    rng = np.random.default_rng(4)
    w = synth.matrix(rng, "Q4_K", 256, 1024)
    weight = hip.GGMLWeight(dev(w).reshape(-1), "Q4_K", (256, 1024))
    dense = torch.from_numpy(q.dequantize_matrix(w, "Q4_K", 256, 1024)).double()
    for tokens in (1, 8, 20):  # 20 > MAX_TOKENS: dequantize to bf16 + torch matmul, as gguf/metal.py:407
        x = torch.randn(tokens, 1024, generator=torch.Generator().manual_seed(tokens))
        y = F.linear(x.cuda(), weight)
        assert y.dtype == x.dtype and y.shape == (tokens, 256)
        expect = (x.double() @ dense.T).numpy()
        assert moe_ref.rel_err(y.cpu().numpy(), expect) < (TOL if tokens <= 8 else 2e-2)
    base, offset = weight.location()
    assert offset == 0 and base.numel() == w.size


def test_ggml_weight_linear_routes(hip):
    """Above MAX_TOKENS: with keep_dense (the default) the bf16 values are dequantized once and kept, and each call is
    the reference's bf16 F.linear on them (gguf/metal.py:407), bit for bit; with keep_dense False each call
    dequantizes to a temporary and runs the same F.linear, nothing kept, also bit for bit."""
    rng = np.random.default_rng(14)
    w = synth.matrix(rng, "Q6_K", 512, 2048)
    weight = hip.GGMLWeight(dev(w).reshape(-1), "Q6_K", (512, 2048))
    x = torch.randn(70, 2048, generator=torch.Generator().manual_seed(15)).cuda()
    want = F.linear(x.to(torch.bfloat16), hip.dequantize_gpu(weight.raw, "Q6_K", (512, 2048))).float()
    y = F.linear(x, weight)
    kept = weight.dense()
    assert torch.equal(y, want)
    assert torch.equal(F.linear(x, weight), want) and weight.dense() is kept  # dequantized once
    dense = torch.from_numpy(q.dequantize_matrix(w, "Q6_K", 512, 2048))
    assert torch.equal(kept.float().cpu(), dense.to(torch.bfloat16).float())  # the blocks' values, rounded to bf16
    weight.drop_dense()
    weight.keep_dense = False
    y2 = F.linear(x, weight)
    assert weight._dense is None
    assert torch.equal(y2, want)


@pytest.mark.parametrize("name", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("rows,k", [(256, 256), (512, 2048), (2048, 512)])
@pytest.mark.parametrize("tokens", [9, 20, 64, 65, 130, 300])
def test_linear_mfma(hip, name, rows, k, tokens):
    """wl_linear against bf16(x) . bf16(dequantized W)^T in fp64 at few rows: one round of the CUs, so the K-split kernels
    (and 64-token tiles for one block a row), the last token tile partial."""
    rng = np.random.default_rng(rows + k + tokens)
    w = synth.matrix(rng, name, rows, k)
    x = rng.standard_normal((tokens, k)).astype(np.float32)
    y = hip.linear_mfma(dev(w).reshape(-1), name, (rows, k), torch.from_numpy(x).cuda())
    assert y.dtype == torch.bfloat16 and y.shape == (tokens, rows)
    wb = q.round_bf16(q.dequantize_matrix(w, name, rows, k)).astype(np.float64)
    ref = q.round_bf16(x).astype(np.float64) @ wb.T
    err = moe_ref.rel_err(y.float().cpu().numpy(), ref)
    assert err < 4e-3, err


@pytest.mark.parametrize("name,rows,k,tokens", [
    ("Q4_K", 256, 768, 9), ("Q6_K", 768, 1280, 65), ("Q4_K", 2304, 2048, 200), ("Q6_K", 256, 1024, 449),  # K 4 ways
    ("Q6_K", 512, 512, 17), ("Q4_K", 768, 512, 500), ("Q6_K", 2048, 1280, 700),                           # K 2 ways
    ("Q4_K", 4096, 256, 130), ("Q4_K", 4096, 768, 640),                                               # 64-token tiles
    ("Q6_K", 4096, 1280, 1000), ("Q6_K", 4096, 512, 1300)])                                          # 128-token tiles
def test_linear_mfma_forms(hip, name, rows, k, tokens):
    """Each kernel of wl_linear at its edges: block counts that do not divide into the K split, fewer than 8 token
    tiles and 8 or more, row slabs that do not fill the 8 XCDs, a last tile of 1, 8, 17 and 64 tokens. Bound: bf16's
    half ulp on the output (up to 2^-8 of its value) plus the fp32 sums' rounding (k 2^-24 of sum |w x|)."""
    rng = np.random.default_rng(rows + k + tokens)
    w = synth.matrix(rng, name, rows, k)
    x = rng.standard_normal((tokens, k)).astype(np.float32)
    y = hip.linear_mfma(dev(w).reshape(-1), name, (rows, k), torch.from_numpy(x).cuda()).float().cpu().numpy()
    wb = q.round_bf16(q.dequantize_matrix(w, name, rows, k)).astype(np.float64)
    xb = q.round_bf16(x).astype(np.float64)
    ref, size = xb @ wb.T, np.abs(xb) @ np.abs(wb).T
    assert (np.abs(y - ref) <= 2.0 ** -8 * np.abs(ref) + k * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("name,rows,k,tokens", [
    ("Q6_K", 4096, 1536, 1000), ("Q6_K", 1280, 768, 700),           # 64-token tiles, an even and an odd number of blocks
    ("Q4_K", 4096, 2048, 1290), ("Q6_K", 4096, 2048, 1300), ("Q4_K", 2048, 1280, 2900), ("Q6_K", 4096, 2304, 1370),
    ("Q4_K", 8192, 1024, 570), ("Q6_K", 3072, 256, 1100), ("Q6_K", 16384, 768, 400), ("Q4_K", 16384, 1280, 390)])
def test_linear_mfma_large_tiles(hip, name, rows, k, tokens):
    """wl_linear's 128-token tiles (but for the first two), with 1 to 9 blocks a row: double-buffered, and in phases for a
    last tile of 10 to 64 tokens (10, 20, 84, 90, 58, 76, 16, 6); 8 tiles and more, and fewer (dealt by row slabs). The
    bound is test_linear_mfma_forms'."""
    rng = np.random.default_rng(rows + k + tokens)
    w = synth.matrix(rng, name, rows, k)
    x = rng.standard_normal((tokens, k)).astype(np.float32)
    y = hip.linear_mfma(dev(w).reshape(-1), name, (rows, k), torch.from_numpy(x).cuda()).float().cpu().numpy()
    wb = q.round_bf16(q.dequantize_matrix(w, name, rows, k)).astype(np.float64)
    xb = q.round_bf16(x).astype(np.float64)
    ref, size = xb @ wb.T, np.abs(xb) @ np.abs(wb).T
    assert (np.abs(y - ref) <= 2.0 ** -8 * np.abs(ref) + k * 2.0 ** -24 * size).all()


def test_linear_mfma_rejects(hip):
    w = torch.zeros(255 * 144, dtype=torch.uint8, device="cuda")
    x = torch.zeros(16, 256, device="cuda")
    with pytest.raises(ValueError):  # rows not a multiple of 256
        hip.linear_mfma(w, "Q4_K", (255, 256), x)


def test_errors_raise(hip):
    w = torch.zeros(144, dtype=torch.uint8, device="cuda")
    with pytest.raises(NotImplementedError):
        hip.dequantize_gpu(w, "Q5_K", (1, 256))
    with pytest.raises(ValueError):
        hip.gemv(w, "Q4_K", (1, 100), torch.zeros(1, 100, device="cuda"))
