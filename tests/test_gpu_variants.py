"""GPU parity of the kernel variants that the entry points select by shape
and operand alignment and that the configuration-shaped tests do not reach:

- FP8: the general kernel for every segment count (K up to 1024, 2048, 3072,
  aligned and unaligned rows); the fused SwiGLU and the multi-matrix launch on
  the vector tile kernels for every K and token group; the matrix-core kernel
  with four row blocks per wave at K = 1024 and 2048 and the fused SwiGLU with
  two; the RMSNorm-folded GEMV for every token group, K and residual choice,
  with the GEMV on the vector units or on the matrix cores;
- MXFP4: the dense general kernel for two to four blocks per lane, aligned and
  unaligned; the routed layer's general stage-A and stage-B kernels, which take
  over when scale rows, the activation or W2 are not 16-byte aligned, for one
  and two blocks per lane; the router GEMV at K = 8192;
- RMSNorm: hidden 6144 (16 waves with a quarter of the threads past the row)
  and the scalar forward path.

Every case is checked against the oracle (max rel err <= 1e-2, cosine >=
0.9999); where two launches must agree, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import mx
from runtime import moe, synth
from runtime import fp8_e4m3_gemv_binding as fp8b
from runtime import mxfp4_gemv_binding as mxb
from runtime import mxfp4_grouped_gemv_binding as gb
from runtime import rmsnorm_fuse_binding as rb
from tests.gpu_util import announce, assert_close, dev_bf16, dev_f32, dev_u8, host_bits

pytestmark = pytest.mark.gpu


def _at_offset(t: torch.Tensor, nbytes: int) -> torch.Tensor:
    """A contiguous copy of t whose data starts nbytes past a 256-byte boundary."""
    n = t.numel() * t.element_size()
    buf = torch.zeros(n + 256, dtype=torch.uint8, device=t.device)
    v = buf[nbytes:nbytes + n]
    v.copy_(t.contiguous().reshape(-1).view(torch.uint8))
    out = v.view(t.dtype).view(t.shape)
    assert out.data_ptr() % 16 == nbytes % 16
    return out


def _fp8_uniform(seed: int, N: int, K: int):
    """E4M3 codes uniform over the non-NaN bytes and tile scales 2^-14 .. 2^-10:
    a quick stand-in for large weight matrices (any code is a valid weight)."""
    rng = np.random.default_rng(seed)
    w = rng.integers(0, 256, (N, K), dtype=np.uint8)
    w[(w & 0x7F) == 0x7F] ^= 1
    s = rng.integers(113, 118, ((N + 127) // 128, K // 128), dtype=np.uint8)
    return w, s


def _x1(xd, T):
    return xd if T > 1 else xd[0]


# ---------------------------------------------------------------- FP8 -------

@pytest.mark.parametrize("N,K,T,odd_stride", [(77, 1024, 2, True), (90, 1536, 1, False), (90, 1536, 3, True),
                                              (70, 2560, 2, False), (70, 3072, 1, True)])
def test_fp8_general_kernel_segments(device, N, K, T, odd_stride):
    """The general kernel with one, two and three 1 KiB chunks per lane, on
    aligned and on odd-stride (unaligned) weight rows."""
    announce(f"fp8_e4m3_gemv general N={N} K={K} T={T} odd_stride={odd_stride}")
    w, s = synth.fp8_weight(20000 + N + K + T, N, K)
    x = synth.normal_bf16(20100 + T, (T, K))
    if odd_stride:
        buf = torch.zeros(N, K + 1, dtype=torch.uint8, device=device)
        buf[:, :K] = dev_u8(w, device)
        tw = buf[:, :K]
    else:
        tw = dev_u8(w, device)
    y = fp8b.fp8_e4m3_gemv(tw, dev_u8(s, device), _x1(dev_bf16(x, device), T))
    assert_close(host_bits(y).reshape(T, N), mx.fp8_gemv(x, w, s), f"fp8 general N={N} K={K} T={T}")


@pytest.mark.parametrize("K", [1024, 2048, 4096])
@pytest.mark.parametrize("T", [1, 2, 3, 8])
def test_fp8_swiglu_vector_tiles(device, K, T):
    """The fused SwiGLU on the vector tile kernel (300 rows: below the
    matrix-core rule) for every K up to 4096 and token group 1, 2, 4, 8."""
    N = 300
    announce(f"fp8_e4m3_swiglu_gemv vector N={N} K={K} T={T}")
    w1, s1 = synth.fp8_weight(20200 + K, N, K)
    w3, s3 = synth.fp8_weight(20300 + K, N, K)
    x = mx.bf16_round(24 * mx.bf16_to_f32(synth.normal_bf16(20400 + T, (T, K))))
    act = fp8b.fp8_e4m3_swiglu_gemv(dev_u8(w1, device), dev_u8(s1, device), dev_u8(w3, device), dev_u8(s3, device),
                                    _x1(dev_bf16(x, device), T), 10.0, True)
    assert_close(host_bits(act).reshape(T, N), mx.fp8_swiglu(x, w1, s1, w3, s3, 10.0, True),
                 f"fp8 swiglu vector K={K} T={T}")


def test_fp8_vector_tile_k1024_eight_tokens(device):
    N, K, T = 600, 1024, 6
    announce(f"fp8_e4m3_gemv vector tile N={N} K={K} T={T}")
    w, s = synth.fp8_weight(20500, N, K)
    x = synth.normal_bf16(20501, (T, K))
    y = fp8b.fp8_e4m3_gemv(dev_u8(w, device), dev_u8(s, device), dev_bf16(x, device))
    assert_close(host_bits(y).reshape(T, N), mx.fp8_gemv(x, w, s), "fp8 K=1024 T=6")


@pytest.mark.parametrize("K,T,shapes", [(1024, 1, [300, 200]), (1024, 2, [300, 200]), (1024, 3, [300, 200]),
                                        (1024, 8, [300, 200]), (1024, 12, [300, 200]),
                                        (2048, 1, [300, 200]), (2048, 2, [300, 200]), (2048, 3, [300, 200]),
                                        (2048, 8, [300, 200]), (2048, 12, [300, 200]),
                                        (4096, 2, [300, 200]), (4096, 8, [300, 200]), (4096, 12, [300, 200]),
                                        (8192, 1, [300, 200]),
                                        (1024, 4, [2048, 2048]), (2048, 5, [2048, 2048])])
def test_fp8_multi_launch_variants(device, K, T, shapes):
    """The multi-matrix launch for every K and token group on the vector
    kernels, and on the matrix cores at K = 1024 and 2048: each output has the
    bits of fp8_e4m3_gemv on its matrix alone and matches the oracle."""
    announce(f"fp8_e4m3_gemv_multi N={shapes} K={K} T={T}")
    mats, dmats = [], []
    for i, N in enumerate(shapes):
        w, s = synth.fp8_weight(20600 + 10 * i + K, N, K)
        mats.append((w, s))
        dmats.append((dev_u8(w, device), dev_u8(s, device)))
    x = synth.normal_bf16(20700 + T, (T, K))
    xin = _x1(dev_bf16(x, device), T)
    ys = fp8b.fp8_e4m3_gemv_multi(dmats, xin)
    for (w, s), (tw, ts), y, N in zip(mats, dmats, ys, shapes):
        got = host_bits(y).reshape(T, N)
        single = host_bits(fp8b.fp8_e4m3_gemv(tw, ts, xin)).reshape(T, N)
        assert np.array_equal(got, single), f"N={N}: multi launch differs from the single launch"
        assert_close(got, mx.fp8_gemv(x, w, s), f"multi N={N} K={K} T={T}")


@pytest.mark.parametrize("N,K", [(65536, 1024), (32768, 2048)])
def test_fp8_matrix_core_four_row_blocks_short_k(device, N, K):
    """Four 16-row blocks per wave at K = 1024 and 2048 (T = 8): the shapes at
    which the row-block rule first takes four."""
    T = 8
    announce(f"fp8_e4m3_gemv matrix cores N={N} K={K} T={T}")
    w, s = _fp8_uniform(20800 + K, N, K)
    x = synth.normal_bf16(20801, (T, K))
    y = fp8b.fp8_e4m3_gemv(dev_u8(w, device), dev_u8(s, device), dev_bf16(x, device))
    assert_close(host_bits(y).reshape(T, N), mx.fp8_gemv(x, w, s), f"fp8 R=4 N={N} K={K}")


@pytest.mark.parametrize("N,K", [(16384, 1024), (8192, 4096)])
def test_fp8_swiglu_matrix_core_two_row_blocks(device, N, K):
    """The fused SwiGLU with two 16-row blocks per wave (T = 8)."""
    T = 8
    announce(f"fp8_e4m3_swiglu_gemv matrix cores N={N} K={K} T={T}")
    w1, s1 = _fp8_uniform(20900 + K, N, K)
    w3, s3 = _fp8_uniform(20950 + K, N, K)
    x = synth.normal_bf16(20901, (T, K))
    act = fp8b.fp8_e4m3_swiglu_gemv(dev_u8(w1, device), dev_u8(s1, device), dev_u8(w3, device), dev_u8(s3, device),
                                    dev_bf16(x, device), 10.0, False)
    assert_close(host_bits(act).reshape(T, N), mx.fp8_swiglu(x, w1, s1, w3, s3, 10.0, False),
                 f"fp8 swiglu R=2 N={N} K={K}")


@pytest.mark.parametrize("K", [2048, 4096])
@pytest.mark.parametrize("T,N", [(1, 300), (2, 300), (3, 300), (4, 4096)])
@pytest.mark.parametrize("resid", [True, False])
def test_fp8_rmsnorm_gemv_variants(device, K, T, N, resid):
    """RMSNorm folded into the GEMV for token groups 1, 2 and 4, with and
    without the residual, the GEMV on the vector units (300 rows) or, at
    T = 4 and 4096 rows, on the matrix cores after the norm in one workgroup:
    x_norm and new_residual match the oracle (new_residual bit for bit), y
    has fp8_e4m3_gemv's bits on x_norm and matches the oracle."""
    announce(f"fp8_e4m3_rmsnorm_gemv N={N} K={K} T={T} residual={resid}")
    w, s = synth.fp8_weight(21000 + N + K, N, K)
    h = synth.normal_bf16(21001 + T, (T, K))
    r = synth.normal_bf16(21002 + T, (T, K), 0.0, 0.5)
    g = synth.normal_bf16(21003, (K,), 1.0, 0.1)
    tw, ts = dev_u8(w, device), dev_u8(s, device)
    hd, rd, gd = dev_bf16(h, device), dev_bf16(r, device), dev_bf16(g, device)
    y, xn, nr = fp8b.fp8_e4m3_rmsnorm_gemv(tw, ts, _x1(hd, T), gd, _x1(rd, T) if resid else None)
    if resid:
        oracle_xn, oracle_nr = mx.rmsnorm_residual(h, r, g)
        assert np.array_equal(host_bits(nr).reshape(T, K), oracle_nr), "new_residual bits"
    else:
        oracle_xn = mx.rmsnorm(h, g)
    assert_close(host_bits(xn).reshape(T, K), oracle_xn, "x_norm vs oracle")
    ref_y = fp8b.fp8_e4m3_gemv(tw, ts, xn.reshape(T, K) if T > 1 else xn.reshape(K))
    assert np.array_equal(host_bits(y).reshape(T, N), host_bits(ref_y).reshape(T, N)), "y bits"
    assert_close(host_bits(y).reshape(T, N), mx.fp8_gemv(oracle_xn, w, s), "y vs oracle")


# ------------------------------------------------------------ dense MXFP4 ---

@pytest.mark.parametrize("K,unaligned", [(3072, False), (3072, True), (6144, True), (7168, False), (8192, True)])
def test_mxfp4_gemv_general_kernel(device, K, unaligned):
    """The general dense kernel with two, three and four MX blocks per lane
    (K off the tile set, or unaligned rows and activation at any K)."""
    N = 50
    announce(f"mxfp4_gemv_m1 general N={N} K={K} unaligned={unaligned}")
    p, s = synth.mxfp4_weight(21100 + K, N, K)
    x = synth.normal_bf16(21101 + K, (K,))
    ref = mx.mxfp4_gemv(x, p[0], s[0])
    ts = dev_u8(s[0], device)
    if unaligned:
        odd_p = np.zeros((N, K // 2 + 1 + 7), np.uint8)
        odd_p[:, 1:1 + K // 2] = p[0]
        to = dev_u8(odd_p, device)
        xb = dev_bf16(np.concatenate([[0], x]).astype(np.uint16), device)
        y = mxb.mxfp4_gemv(to[:, 1:1 + K // 2], ts, xb[1:])
    else:
        y = mxb.mxfp4_gemv(dev_u8(p[0], device), ts, dev_bf16(x, device))
    assert_close(host_bits(y), ref, f"mxfp4 general K={K}")


# ------------------------------------------------------------- routed MoE ---

def _host_expert_fn(weights):
    cache = {}

    def fn(e):
        if e not in cache:
            cache[e] = tuple((m["packed"][e].cpu().numpy(), m["scale"][e].cpu().numpy())
                             for m in (weights.W1, weights.W3, weights.W2))
        return cache[e]

    return fn


@pytest.mark.parametrize("K,H", [(2048, 2048), (4096, 2048), (2048, 4096)])
@pytest.mark.parametrize("variant", ["scales_offset", "x_offset", "w2_offset"])
def test_moe_general_kernels(device, K, H, variant):
    """The routed layer when an operand is not 16-byte aligned, which moves it
    off the one-token and multi-token kernels onto the general ones: scale
    tensors 2 bytes past a boundary (the checked-alignment fast kernels), the
    activation 2 bytes past (stage A's unaligned loads), W2 1 byte past (stage
    B's unaligned loads); for one and two MX blocks per lane in stage A (K)
    and stage B (hidden), one and three tokens, and the drop-in."""
    E, O, topk = 8, 256, 2
    announce(f"mxfp4 routed general kernels {variant} K={K} H={H}")
    w = moe.make_moe_weights(21200 + K + H, E, K, H, O, device)
    fn = _host_expert_fn(w)
    mats = {m: dict(getattr(w, m)) for m in ("W1", "W3", "W2")}
    if variant == "scales_offset":
        for m in mats:
            mats[m]["scale"] = _at_offset(mats[m]["scale"], 2)
    if variant == "w2_offset":
        mats["W2"]["packed"] = _at_offset(mats["W2"]["packed"], 1)
    for T in (1, 3):
        x = synth.normal_bf16(21300 + T, (T, K))
        xd = dev_bf16(x, device)
        if variant == "x_offset":
            xd = _at_offset(xd, 2)
        ids, wt = mx.route_sigmoid_topk(synth.gating_logits(21400 + T, T, E), topk)
        out = host_bits(gb.mxfp4_moe_grouped_gemv(xd, mats["W1"], mats["W3"], mats["W2"],
                                                  torch.from_numpy(ids).to(device), dev_f32(wt, device)))
        assert_close(out, mx.moe_layer(x, fn, ids, wt, O, n_experts=E), f"{variant} T={T}")
        if T == 1:
            sub = {m: {"packed": mats[m]["packed"][:4], "scale": mats[m]["scale"][:4]} for m in mats}
            r = np.linspace(0.1, 0.4, 4).astype(np.float32)
            got = host_bits(gb.mxfp4_grouped_gemv(sub["W1"], sub["W3"], sub["W2"], None, xd[0], dev_f32(r, device)))
            ref = mx.moe_layer(x, fn, np.arange(4, dtype=np.int32)[None, :], r[None, :], O)
            assert_close(got, ref[0], f"{variant} drop-in")
    del w, mats
    torch.cuda.empty_cache()


def test_router_logits_longest_rows(device):
    """The router GEMV at K = 8192 (16 pieces of a row per lane)."""
    T, E, K = 2, 64, 8192
    announce(f"mxfp4_moe_router_logits T={T} E={E} K={K}")
    x = synth.normal_bf16(21500, (T, K))
    wg = synth.normal_bf16(21501, (E, K), 0.0, 0.02)
    got = gb.router_logits(dev_bf16(x, device), dev_bf16(wg, device)).cpu().numpy()
    ref = mx.router_logits(x, wg)
    bound = (np.abs(mx.bf16_to_f32(x)).astype(np.float64) @ np.abs(mx.bf16_to_f32(wg)).astype(np.float64).T) * 2e-6
    assert np.all(np.abs(got.astype(np.float64) - ref) <= bound + 1e-30)


# ---------------------------------------------------------------- RMSNorm ---

def test_rmsnorm_partial_block_and_scalar_forward(device):
    """hidden = 6144 (768 pieces in a 1,024-thread block: the last 256 threads
    hold no piece) through both entries, and the forward entry on its scalar
    path (hidden not a multiple of 8)."""
    for H, T in ((6144, 3), (4001, 2)):
        announce(f"rmsnorm H={H} T={T}")
        h = synth.normal_bf16(21600 + H, (T, H))
        r = synth.normal_bf16(21601 + H, (T, H), 0.0, 0.5)
        g = synth.normal_bf16(21602 + H, (H,), 1.0, 0.1)
        hd, rd, gd = dev_bf16(h, device), dev_bf16(r, device), dev_bf16(g, device)
        assert_close(host_bits(rb.rmsnorm_fuse_fwd(hd, gd)), mx.rmsnorm(h, g), f"rmsnorm fwd H={H}")
        y, nr = rb.rmsnorm_fuse_residual_add(hd, rd, gd)
        ry, rnr = mx.rmsnorm_residual(h, r, g)
        assert np.array_equal(host_bits(nr), rnr)
        assert_close(host_bits(y), ry, f"rmsnorm residual H={H}")


def _fp8_vector_tiles_far_apart_rows(device, K, Ts, seed):
    """Token rows just far enough apart that the T rows span more than 2^31
    bytes: the matrix-core kernels read the activation rows through one buffer
    of at most 2^31 bytes, so these calls stay on the vector tile kernels
    (single matrix, fused SwiGLU, multi-matrix, fp32 tile scales), called
    through the C ABI with the row stride. Each against the oracle; the
    multi-matrix and fp32-scale outputs bit for bit against the single GEMV."""
    import ctypes
    from runtime import _lib as rl

    lib = fp8b._load_lib()
    N = 300
    x = synth.normal_bf16(seed, (max(Ts), K))
    x = mx.bf16_round(8 * mx.bf16_to_f32(x))
    xd = dev_bf16(x, device)
    w1, s1 = synth.fp8_weight(seed + 1, N, K)
    w3, s3 = synth.fp8_weight(seed + 2, N, K)
    w2, s2 = synth.fp8_weight(seed + 3, 200, K)
    d1, e1, d3, e3 = dev_u8(w1, device), dev_u8(s1, device), dev_u8(w3, device), dev_u8(s3, device)
    d2, e2 = dev_u8(w2, device), dev_u8(s2, device)
    sf = torch.from_numpy(np.ldexp(np.float32(1.0), s1.astype(np.int32) - 127).astype(np.float32)).to(device)
    st = ctypes.c_void_p(rl.stream_ptr(device))
    for T in Ts:
        stride = (2**30 // (T - 1) // 8 + 1) * 8            # (T - 1) * stride * 2 bytes > 2^31
        assert ((T - 1) * stride + K) * 2 > 2**31 - 1
        announce(f"fp8 K={K} T={T} rows {stride} elements apart")
        xbuf = torch.zeros((T - 1) * stride + K, dtype=torch.bfloat16, device=device)
        for t in range(T):
            xbuf[t * stride:t * stride + K] = xd[t]
        y = torch.empty(T, N, dtype=torch.bfloat16, device=device)
        rc = lib.fp8_e4m3_gemv(rl.vp(xbuf), stride, rl.vp(d1), rl.vp(e1), K, N, T, K, K // 128, rl.vp(y), N, st)
        assert rc == 0
        single = host_bits(y)
        assert_close(single, mx.fp8_gemv(x[:T], w1, s1), f"fp8 far rows K={K} T={T}")
        act = torch.empty(T, N, dtype=torch.bfloat16, device=device)
        rc = lib.fp8_e4m3_swiglu_gemv(rl.vp(xbuf), stride, rl.vp(d1), rl.vp(e1), rl.vp(d3), rl.vp(e3), K, N, T,
                                      K, K // 128, 10.0, 1, rl.vp(act), N, st)
        assert rc == 0
        assert_close(host_bits(act), mx.fp8_swiglu(x[:T], w1, s1, w3, s3, 10.0, True),
                     f"swiglu far rows K={K} T={T}")
        ya = torch.empty(T, N, dtype=torch.bfloat16, device=device)
        yb = torch.empty(T, 200, dtype=torch.bfloat16, device=device)
        PA, IA, LA = ctypes.c_void_p * 2, ctypes.c_int * 2, ctypes.c_int64 * 2
        rc = lib.fp8_e4m3_gemv_multi(rl.vp(xbuf), stride, K, T, 2, PA(d1.data_ptr(), d2.data_ptr()),
                                     PA(e1.data_ptr(), e2.data_ptr()), IA(N, 200), LA(K, K), LA(K // 128, K // 128),
                                     PA(ya.data_ptr(), yb.data_ptr()), LA(N, 200), st)
        assert rc == 0
        assert np.array_equal(host_bits(ya), single), "multi launch differs from the single launch"
        assert_close(host_bits(yb), mx.fp8_gemv(x[:T], w2, s2), f"multi far rows K={K} T={T}")
        # the fp32-scale entry on the same vector tiles: scales 2^(b-127) give the E8M0 bits
        yf = torch.empty(T, N, dtype=torch.bfloat16, device=device)
        rc = lib.fp8_e4m3_gemv_f32s(rl.vp(xbuf), stride, rl.vp(d1), rl.vp(sf), K, N, T, K, K // 128, rl.vp(yf), N, st)
        assert rc == 0
        assert np.array_equal(host_bits(yf), single), "fp32-scale entry differs from the E8M0 entry"
        del xbuf
        torch.cuda.empty_cache()


def test_fp8_k8192_vector_tiles_far_apart_rows(device):
    """K = 8192 on the vector tile kernels (token groups of 2 and 4, two
    k-slices per thread): every other shape with T >= 2 at this K takes the
    matrix cores."""
    _fp8_vector_tiles_far_apart_rows(device, 8192, (2, 4), 21700)


@pytest.mark.parametrize("K", [1024, 2048])
def test_fp8_short_rows_vector_tiles_far_apart_rows(device, K):
    """K = 1024 and 2048 with 5 .. 16 tokens on the vector tile kernels (token
    groups of 8 and 16; the fused SwiGLU in groups of 8 and a last group of
    1): every other shape with T >= 5 at these K takes the matrix cores."""
    _fp8_vector_tiles_far_apart_rows(device, K, (5, 9, 16), 21710 + K)


# ------------------------------------------------------- prefill, wide tiles ---

_TILE_EDGES = [1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 127, 128, 129, 192, 257]


def _pairs_with_counts(counts, topk, seed):
    """ids [T, topk] in which expert e is listed counts[e] times; -1 fills up."""
    rng = np.random.default_rng(seed)
    flat = np.repeat(np.arange(len(counts)), counts)
    T = -(-len(flat) // topk)
    flat = np.concatenate([flat, np.full(T * topk - len(flat), -1)])
    return rng.permutation(flat).astype(np.int32).reshape(T, topk)


@pytest.mark.parametrize("K,H,O,counts,topk", [
    (512, 2048, 64, _TILE_EDGES, 2),               # every tile size; one macro-step pair in stage A, a quarter-full row block
    (1536, 2560, 320, _TILE_EDGES[::2], 3),        # 3 and 5 x 512: the four-deep weight ring ends mid-way
    (2560, 3072, 576, _TILE_EDGES[1::2], 1),
    (4096, 2048, 256, [1, 16, 40, 64, 100, 128, 900], 2),
    (1024, 8192, 192, [20, 60, 120, 130], 2),
    (1024, 512, 1024, [3, 70, 1100, 129, 2900], 2),  # one macro-step pair in stage B
])
def test_prefill_wide_tiles_equal_small_tiles(device, K, H, O, counts, topk):
    """Chunks of many pairs, 12 or more per expert, run on the wide tiles. The same
    chunk with more (unrouted) experts in the tensors runs on the 64 x 64 tiles:
    same weights, k order, sums and rounding, so the same bits. Special scale
    bytes (0xFF and 0) are among the blocks."""
    E = len(counts)
    ids = _pairs_with_counts(counts, topk, 9000 + K + O)
    T = ids.shape[0]
    E_all = T * topk // 12 + 1
    announce(f"mxfp4_moe_prefill wide tiles K={K} H={H} O={O} T={T} topk={topk} E={E} / {E_all}")
    wide_rule = gb._load_lib().mxfp4_moe_prefill_wide
    assert wide_rule(T, topk, E, K, H, O) and not wide_rule(T, topk, E_all, K, H, O) and E_all >= E
    rng = np.random.default_rng(9001 + K)
    mats = []
    for m, (rows, cols) in enumerate(((H, K), (H, K), (O, H))):
        p, s = synth.mxfp4_weight(9010 + 2 * m + K, rows, cols, E)
        u = rng.random(s.shape)
        s[u < 0.01] = 0xFF
        s[(u >= 0.01) & (u < 0.02)] = 0
        pd = torch.zeros((E_all,) + p.shape[1:], dtype=torch.uint8, device=device)
        sd = torch.zeros((E_all,) + s.shape[1:], dtype=torch.uint8, device=device)
        pd[:E], sd[:E] = dev_u8(p, device), dev_u8(s, device)
        mats.append((p, s, {"packed": pd, "scale": sd}))
    x = synth.normal_bf16(9020 + T, (T, K))
    w = (rng.random((T, topk)) + 0.1).astype(np.float32)
    xd, idd, wd = dev_bf16(x, device), torch.from_numpy(ids).to(device), dev_f32(w, device)
    few = [{k: v[:E] for k, v in d.items()} for _, _, d in mats]
    wide = host_bits(gb.mxfp4_moe_prefill(xd, *few, idd, wd))
    small = host_bits(gb.mxfp4_moe_prefill(xd, *(d for _, _, d in mats), idd, wd))
    assert np.array_equal(wide, small)
    # scale rows that are not 16-byte aligned keep the 64 x 64 tiles
    off = [{"packed": d["packed"], "scale": _at_offset(d["scale"], 4)} for d in few]
    assert np.array_equal(host_bits(gb.mxfp4_moe_prefill(xd, *off, idd, wd)), wide)
    if K == 512:
        def fn(e):
            return tuple((p[e], s[e]) for p, s, _ in mats)

        assert_close(wide, mx.moe_layer(x, fn, ids, w, O, n_experts=E), f"prefill wide tiles K={K} H={H} O={O}")


@pytest.mark.parametrize("T,topk,E", [(8193, 1, 5), (1500, 6, 600), (16384, 16, 64), (5000, 13, 1024)])
def test_prefill_routing_of_large_chunks(device, T, topk, E):
    """More than 8192 (token, k) entries are routed by several workgroups in two
    launches. A token's row does not depend on the other tokens of the chunk, so
    the chunk has to give the bits of its 512-token pieces, which one workgroup
    routes (ids out of range and duplicates included)."""
    K, H, O = 512, 512, 64
    announce(f"mxfp4_moe_prefill routing T={T} topk={topk} E={E}")
    mats = []
    for m, (rows, cols) in enumerate(((H, K), (H, K), (O, H))):
        p, s = synth.mxfp4_weight(9100 + 2 * m + E, rows, cols, min(E, 16))
        reps = -(-E // p.shape[0])
        mats.append({"packed": dev_u8(np.tile(p, (reps, 1, 1))[:E], device),
                     "scale": dev_u8(np.tile(s, (reps, 1, 1))[:E], device)})
    g = torch.Generator(device=device).manual_seed(9200 + T)
    x = torch.randn((T, K), generator=g, device=device).to(torch.bfloat16)
    ids = torch.randint(-1, E + 1, (T, topk), generator=g, device=device, dtype=torch.int32)
    ids[: T // 3] = ids[: T // 3].remainder(7)     # a few hot experts
    w = torch.rand((T, topk), generator=g, device=device)
    whole = gb.mxfp4_moe_prefill(x, *mats, ids, w)
    for t0 in range(0, T, 512):
        part = gb.mxfp4_moe_prefill(x[t0:t0 + 512].contiguous(), *mats, ids[t0:t0 + 512].contiguous(),
                                    w[t0:t0 + 512].contiguous())
        assert torch.equal(part.view(torch.int16), whole[t0:t0 + 512].view(torch.int16)), t0


@pytest.mark.parametrize("topk", [1, 2, 3, 4, 5, 8, 9, 16])
def test_prefill_combine_of_every_topk(device, topk):
    """The combine keeps 1, 2, 4 or 8 rows in flight: against the oracle, with ids
    out of range (a token without any among them) and duplicates."""
    T, E, K, H, O = 19, 8, 512, 512, 1088
    announce(f"mxfp4_moe_prefill combine topk={topk} T={T} O={O}")
    host = [synth.mxfp4_weight(9120 + 2 * m, rows, cols, E) for m, (rows, cols) in enumerate(((H, K), (H, K), (O, H)))]
    rng = np.random.default_rng(9130 + topk)
    ids = rng.integers(-1, E + 1, (T, topk)).astype(np.int32)
    ids[3], ids[7] = -1, 5
    w = (rng.random((T, topk)) + 0.1).astype(np.float32)
    x = synth.normal_bf16(9131, (T, K))
    mats = [{"packed": dev_u8(p, device), "scale": dev_u8(s, device)} for p, s in host]
    out = host_bits(gb.mxfp4_moe_prefill(dev_bf16(x, device), *mats, torch.from_numpy(ids).to(device), dev_f32(w, device)))
    assert not out[3].any()

    def fn(e):
        return tuple((p[e], s[e]) for p, s in host)

    assert_close(out, mx.moe_layer(x, fn, ids, w, O, n_experts=E), f"combine topk={topk}")


# ------------------------------------------------- routing of larger batches ---

@pytest.mark.parametrize("K", [1000, 4096])
def test_router_logits_token_groups(device, K):
    """The router GEMV takes four tokens per workgroup: a token's logits have the
    bits of a one-token call, whatever its place in the group."""
    E, T = 37, 64
    announce(f"router_logits token groups E={E} K={K}")
    g = torch.Generator(device=device).manual_seed(9300 + K)
    x = torch.randn((T, K), generator=g, device=device).to(torch.bfloat16)
    W = (torch.randn((E, K), generator=g, device=device) * 0.02).to(torch.bfloat16)
    one = torch.cat([gb.router_logits(x[t:t + 1].contiguous(), W) for t in range(T)])
    for n in (1, 3, 4, 5, 8, 17, 63, 64):
        assert torch.equal(gb.router_logits(x[:n].contiguous(), W), one[:n]), n


@pytest.mark.parametrize("outputs", ["both", "none", "ids", "weights"])
@pytest.mark.parametrize("T", [16, 17, 20, 21, 64])
def test_layer_gating_of_larger_batches(device, T, outputs):
    """Above 20 tokens the logits are ranked in a launch of its own, whose picks
    pass through the requested outputs or through the pair tables: the layer has
    to equal the layer on the caller's routing, bit for bit."""
    E, K, H, O, topk = 40, 512, 256, 128, 8
    announce(f"mxfp4_moe_layer gating T={T} outputs={outputs}")
    W1, W3, W2 = ({"packed": dev_u8(p, device), "scale": dev_u8(s, device)}
                  for p, s in (synth.mxfp4_weight(9400 + 2 * m, r, c, E)
                               for m, (r, c) in enumerate(((H, K), (H, K), (O, H)))))
    x = dev_bf16(synth.normal_bf16(9410, (T, K)), device)
    logits = dev_f32(synth.gating_logits(9411 + T, T, E), device)
    ids, w = gb.route_sigmoid_topk(logits, topk)
    want = gb.mxfp4_moe_grouped_gemv(x, W1, W3, W2, ids, w)
    io = torch.full_like(ids, -7) if outputs in ("both", "ids") else None
    wo = torch.full_like(w, -7.0) if outputs in ("both", "weights") else None
    got = gb.mxfp4_moe_layer(x, logits, W1, W3, W2, topk, ids_out=io, weights_out=wo)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert io is None or torch.equal(io, ids)
    assert wo is None or torch.equal(wo, w)


@pytest.mark.parametrize("outputs", ["both", "none", "ids", "weights"])
@pytest.mark.parametrize("T", [16, 17, 64])
def test_dispatch_gating_of_larger_batches(device, T, outputs):
    """The routed dispatch ranks the square-root scores in a launch of its own
    above 16 tokens: it has to equal the layer on the routing of
    router_logits + route_topk, bit for bit."""
    E, K, H, O, topk = 200, 512, 256, 128, 6
    announce(f"mxfp4_moe_routed_dispatch gating T={T} outputs={outputs}")
    W1, W3, W2 = ({"packed": dev_u8(p, device), "scale": dev_u8(s, device)}
                  for p, s in (synth.mxfp4_weight(9420 + 2 * m, r, c, E)
                               for m, (r, c) in enumerate(((H, K), (H, K), (O, H)))))
    x = dev_bf16(synth.normal_bf16(9430, (T, K)), device)
    wg = dev_bf16(synth.normal_bf16(9431 + T, (E, K), 0.05), device)
    ids, w = gb.route_topk(gb.router_logits(x, wg), topk, gb.SCORE_SQRT_SOFTPLUS, 1.5)
    want = gb.mxfp4_moe_grouped_gemv(x, W1, W3, W2, ids, w)
    io = torch.full_like(ids, -7) if outputs in ("both", "ids") else None
    wo = torch.full_like(w, -7.0) if outputs in ("both", "weights") else None
    got = gb.mxfp4_moe_routed_dispatch(x, wg, W1, W3, W2, topk, ids_out=io, weights_out=wo)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert io is None or torch.equal(io, ids)
    assert wo is None or torch.equal(wo, w)


@pytest.mark.parametrize("T", [1, 2])
def test_moe_scales_end_with_their_allocation(device, T):
    """K = 3072 has 96 blocks a row, read two per lane: lanes 48 to 63 have none,
    and past the last row of the last expert their scale bytes would lie outside
    the tensor, which here fills its allocation (12 MiB) to the last byte."""
    E, K, H, O = 32, 3072, 4096, 64
    announce(f"mxfp4_moe_grouped_gemv scales at the end of their allocation T={T} K={K} H={H}")
    used = [0, 9, E - 1]
    mats, host = [], []
    for m, (rows, cols) in enumerate(((H, K), (H, K), (O, H))):
        p, s = synth.mxfp4_weight(9500 + 2 * m, rows, cols, len(used))
        pd = torch.zeros((E, rows, cols // 2), dtype=torch.uint8, device=device)
        sd = torch.zeros((E, rows, cols // 32), dtype=torch.uint8, device=device)
        for i, e in enumerate(used):
            pd[e], sd[e] = dev_u8(p[i], device), dev_u8(s[i], device)
        mats.append({"packed": pd, "scale": sd})
        host.append((p, s))
    assert mats[0]["scale"].numel() == 12 << 20
    x = synth.normal_bf16(9510 + T, (T, K))
    ids = np.tile(np.array(used, dtype=np.int32), (T, 1))
    w = (np.random.default_rng(9511).random((T, len(used))) + 0.1).astype(np.float32)
    out = gb.mxfp4_moe_grouped_gemv(dev_bf16(x, device), *mats, torch.from_numpy(ids).to(device), dev_f32(w, device))

    def fn(e):
        return tuple((p[used.index(e)], s[used.index(e)]) for p, s in host)

    assert_close(host_bits(out), mx.moe_layer(x, fn, ids, w, O, n_experts=E), f"scales at the end T={T}")


def _decode_stages(*shape):
    """Stages of a decode batch (T, topk, experts, K, hidden, out_dim) that run on
    the matrix cores: bit 0 A, bit 1 B."""
    return gb._load_lib().mxfp4_moe_decode_stages(*shape)


# T, topk, experts, K, hidden, out_dim, skew (every token lists expert 1 first),
# stages on the matrix cores (1: A, 2: B)
DECODE_MFMA = [
    (2, 8, 8, 1024, 2048, 400, False, 1),     # too few pairs for stage B
    (2, 16, 64, 3072, 1536, 64, False, 1),    # K between 2048 and 4096: fewer pairs per expert suffice
    (6, 8, 8, 1024, 256, 16, False, 2),       # too little work for stage A; one wave per slot, eight sets, one row tile
    (16, 8, 8, 1024, 512, 48, True, 3),       # four sets of slots
    (13, 4, 8, 1024, 1024, 48, True, 3),      # two sets
    (17, 3, 12, 2048, 768, 400, True, 3),     # six waves, two sets; 17 pairs on one expert
    (12, 8, 64, 1024, 1024, 384, False, 2),   # fewer pairs per expert than stage A takes
    (33, 2, 9, 512, 1280, 3072, True, 2),     # K too short for stage A; five waves; 16 rows per workgroup; 33 pairs
    (48, 2, 8, 2560, 1024, 4112, True, 3),    # 257 row tiles
    (24, 8, 16, 2048, 2048, 2048, False, 3),  # eight waves, the most row tiles of 8
    (64, 4, 30, 4096, 2048, 3088, True, 3),   # the largest batch, 193 row tiles
    (64, 16, 3, 1024, 256, 32, True, 3),      # duplicates in every token: 64 pairs per expert
]


@pytest.mark.parametrize("T,topk,E,K,H,O,skew,stages", DECODE_MFMA)
def test_decode_batches_on_matrix_cores(device, T, topk, E, K, H, O, skew, stages):
    """Decode batches whose stages run on the matrix cores, with ids out of
    range and duplicates, E8M0 bytes 0 and 0xFF: against the oracle and the
    general kernels (scales at an odd address), which add in another order and
    round M to bf16 from sums that differ in the last bits; bit-equal replays."""
    announce(f"decode batches on matrix cores T={T} topk={topk} E={E} K={K} H={H} O={O} skew={skew}")
    assert _decode_stages(T, topk, E, K, H, O) == stages
    host = []
    for m, (rows, cols) in enumerate(((H, K), (H, K), (O, H))):
        p, s = synth.mxfp4_weight(9600 + 5 * m + T, rows, cols, E)
        s = s.copy()
        s[:, ::7, ::5] = 0xFF
        s[:, 3::11, 1::6] = 0
        host.append((p, s))
    x = synth.normal_bf16(9620 + T, (T, K))
    rng = np.random.default_rng(9630 + T)
    ids = rng.integers(0, E, (T, topk)).astype(np.int32)
    if skew:
        ids[:, 0] = 1
    ids[T - 1, 0] = -1
    ids[T // 2, topk - 1] = E + 3
    w = (rng.random((T, topk)) + 0.1).astype(np.float32)
    xd, idd, wd = dev_bf16(x, device), torch.from_numpy(ids).to(device), dev_f32(w, device)
    mats = [{"packed": dev_u8(p, device), "scale": dev_u8(s, device)} for p, s in host]
    gen = [{"packed": m["packed"], "scale": _at_offset(m["scale"], 1)} for m in mats]
    out = gb.mxfp4_moe_grouped_gemv(xd, *mats, idd, wd)

    def fn(e):
        return tuple((p[e], s[e]) for p, s in host)

    assert_close(host_bits(out), mx.moe_layer(x, fn, ids, w, O, n_experts=E), "oracle")
    assert_close(host_bits(out), host_bits(gb.mxfp4_moe_grouped_gemv(xd, *gen, idd, wd)), "general kernels",
                 cos_tol=0.99999)
    graph, res = torch.cuda.CUDAGraph(), torch.empty_like(out)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        gb.mxfp4_moe_grouped_gemv(xd, *mats, idd, wd, out=res)
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            gb.mxfp4_moe_grouped_gemv(xd, *mats, idd, wd, out=res)
    for _ in range(3):
        res.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host_bits(res), host_bits(out))
        assert np.array_equal(host_bits(gb.mxfp4_moe_grouped_gemv(xd, *mats, idd, wd)), host_bits(out))
    # no routed expert at all
    none = torch.full_like(idd, -1)
    assert not host_bits(gb.mxfp4_moe_grouped_gemv(xd, *mats, none, wd)).any()


@pytest.mark.parametrize("big", [0, 1])
def test_decode_batches_largest_scales(device, big):
    """Scales up to 2^127 in W1 or W3 and in W2, against activations of 2^-124,
    so that M is about 2^-120: 6 * 2^127 is no bf16 (the oracle's weights
    overflow), and the results are ordinary numbers, which the general kernels
    give."""
    T, topk, E, K, H, O = 16, 8, 16, 1024, 512, 128
    announce(f"decode batches largest scales T={T} E={E} K={K} H={H} O={O} big={big}")
    assert _decode_stages(T, topk, E, K, H, O) == 3
    mats = []
    for m, (rows, cols) in enumerate(((H, K), (H, K), (O, H))):
        p, s = synth.mxfp4_weight(9650 + 2 * m, rows, cols, E)
        if m in (big, 2):
            s = (s.astype(np.int32) + 254 - int(s.max())).astype(np.uint8)
            assert s.max() == 254
        mats.append({"packed": dev_u8(p, device), "scale": dev_u8(s, device)})
    gen = [{"packed": m["packed"], "scale": _at_offset(m["scale"], 1)} for m in mats]
    x = mx.bf16_round(mx.bf16_to_f32(synth.normal_bf16(9660, (T, K))) * np.float32(2.0 ** -124))
    rng = np.random.default_rng(9661)
    ids = np.stack([rng.permutation(E)[:topk] for _ in range(T)]).astype(np.int32)
    w = (rng.random((T, topk)) + 0.1).astype(np.float32)
    args = torch.from_numpy(ids).to(device), dev_f32(w, device)
    out = gb.mxfp4_moe_grouped_gemv(dev_bf16(x, device), *mats, *args)
    assert_close(host_bits(out), host_bits(gb.mxfp4_moe_grouped_gemv(dev_bf16(x, device), *gen, *args)),
                 "largest scales", cos_tol=0.99999)


def _one_hot_rows(E, n, cols, device):
    """MXFP4 [E, n, cols] whose row o is 1.0 at column o and 0 elsewhere."""
    p = np.zeros((E, n, cols // 2), dtype=np.uint8)
    o = np.arange(n)
    p[:, o, o // 2] = np.where(o % 2, 0x20, 0x02)
    return {"packed": dev_u8(p, device), "scale": dev_u8(np.full((E, n, cols // 32), 127, np.uint8), device)}


def _codes(g, shape, device):
    return torch.randint(0, 16, shape, dtype=torch.uint8, generator=g, device=device)


def _packed(codes):
    return (codes[..., 0::2] | (codes[..., 1::2] << 4)).contiguous()


@pytest.mark.parametrize("K", [2048, 2560, 4096])
@pytest.mark.parametrize("T,E", [(64, 8), (48, 16), (24, 32)])
def test_decode_stage_a_sums_as_exact_as_general(device, K, T, E):
    """Every W3 row ends in its first half again, blocks and codes permuted and
    with the other sign, and so does x: W3 x is zero, and M is the rounding of
    the sums (W2 rows are unit vectors, so the layer returns M). Its rms must not
    exceed the general kernels'. One permutation of the blocks is one draw of
    which partial sums cancel early, which moves either figure by up to 10% at
    these K: measured 0.70 to 0.94 of the general kernels' (four chains of MFMAs
    over K, two above 48 tokens: 1.2 to 1.95)."""
    H, topk = 1024, 8
    announce(f"decode stage A sums K={K} T={T} E={E}")
    assert _decode_stages(T, topk, E, K, H, H) & 1
    g = torch.Generator(device=device).manual_seed(9700 + K + T)
    nb = K // 64
    bp = torch.randperm(nb, generator=g, device=device)
    ep = torch.stack([torch.randperm(32, generator=g, device=device) for _ in range(nb)])
    perm = (bp[:, None] * 32 + ep).flatten()
    c3 = _codes(g, (E, H, K // 2), device)
    s3 = torch.randint(119, 126, (E, H, nb), dtype=torch.uint8, generator=g, device=device)
    W3 = {"packed": _packed(torch.cat((c3, (c3 ^ 8)[..., perm]), -1)),
          "scale": torch.cat((s3, s3[..., bp]), -1).contiguous()}
    # W1 x = 64 in every row: silu(64) is 64
    c1 = torch.zeros((E, H, K), dtype=torch.uint8, device=device)
    c1[..., 0] = 2
    W1 = {"packed": _packed(c1), "scale": torch.full((E, H, K // 32), 133, dtype=torch.uint8, device=device)}
    x = torch.randn((T, K // 2), generator=g, device=device).to(torch.bfloat16)
    x[:, 0] = 1.0
    x = torch.cat((x, x[:, perm]), -1).contiguous()
    ids = torch.stack([torch.randperm(E, generator=g, device=device)[:topk] for _ in range(T)]).int()
    w = torch.zeros((T, topk), device=device)
    w[:, 0] = 1.0
    W2 = _one_hot_rows(E, H, H, device)

    def rms(mats):
        out = gb.mxfp4_moe_grouped_gemv(x, *mats, W2, ids, w)
        return float(out.double().pow(2).mean().sqrt())

    ours = rms([W1, W3])
    general = rms([{"packed": m["packed"], "scale": _at_offset(m["scale"], 1)} for m in (W1, W3)])
    print(f"  rms {ours:.4e}, general kernels {general:.4e}", flush=True)
    assert 0 < ours <= general


def test_decode_rows_independent_of_neighbours(device):
    """On the matrix cores a token's M row has the same bits whatever the number
    of tokens on its expert (1 to 4 blocks of 16): the layer returns M."""
    K, H, E = 2048, 2048, 4
    announce(f"decode rows against their neighbours K={K} H={H}")
    mats = [{"packed": dev_u8(p, device), "scale": dev_u8(s, device)}
            for p, s in (synth.mxfp4_weight(9720 + 2 * m, H, K, E) for m in range(2))]
    mats.append(_one_hot_rows(E, H, H, device))
    x = dev_bf16(synth.normal_bf16(9730, (64, K)), device)
    out = {}
    for n in (16, 32, 48, 64):
        assert _decode_stages(n, 1, E, K, H, H) & 1
        ids = torch.full((n, 1), 2, dtype=torch.int32, device=device)
        out[n] = gb.mxfp4_moe_grouped_gemv(x[:n].contiguous(), *mats, ids, torch.ones((n, 1), device=device))
    for n in (16, 32, 48):
        assert torch.equal(out[n].view(torch.int16), out[64][:n].view(torch.int16)), n


def test_decode_overflow_stays_infinite(device):
    """Sums beyond fp32 give the infinities of the general kernels, no NaN."""
    T, E, K, H, O = 24, 2, 1024, 2048, 64
    announce(f"decode overflow T={T} K={K} H={H}")
    assert _decode_stages(T, 1, E, K, H, O) & 1
    g = torch.Generator(device=device).manual_seed(9740)

    def positive(rows, cols, byte):
        return {"packed": _packed(torch.randint(1, 8, (E, rows, cols), dtype=torch.uint8, generator=g, device=device)),
                "scale": torch.full((E, rows, cols // 32), byte, dtype=torch.uint8, device=device)}

    W1, W3, W2 = positive(H, K, 250), positive(H, K, 127), positive(O, H, 120)
    x = torch.rand((T, K), generator=g, device=device).add_(0.5).to(torch.bfloat16)
    x[::2] *= 2.0 ** -120                          # every second token stays finite
    ids = torch.zeros((T, 1), dtype=torch.int32, device=device)
    w = torch.ones((T, 1), device=device)
    out = gb.mxfp4_moe_grouped_gemv(x, W1, W3, W2, ids, w)
    gen = [{"packed": m["packed"], "scale": _at_offset(m["scale"], 1)} for m in (W1, W3, W2)]
    want = gb.mxfp4_moe_grouped_gemv(x, *gen, ids, w)
    assert torch.equal(torch.isposinf(out), torch.isposinf(want)) and not out.isnan().any()
    assert torch.isposinf(out[1::2]).all() and torch.isfinite(out[::2]).all()
    assert_close(host_bits(out[::2].contiguous()), host_bits(want[::2].contiguous()), "finite tokens", cos_tol=0.99999)


def test_decode_stage_b_adds_waves_in_double(device):
    """Stage B's waves take 256 k each: sums of 2^24, 1 and -2^24 from three of
    them have to give the 1, which fp32 sums in wave order lose."""
    T, E, K, H, O = 64, 2, 2048, 2048, 4096
    announce(f"decode stage B sums of the waves T={T} H={H} O={O}")
    assert _decode_stages(T, 1, E, K, H, O) & 2
    W1 = np.zeros((E, H, K // 2), np.uint8)
    W1[..., 0] = 0x02                              # W1 x = x[0] = 128, and so is its silu
    W2 = np.zeros((E, O, H // 2), np.uint8)
    x = np.zeros((T, K), np.float32)
    x[:, 0] = 128.0
    for i, v in ((1, 2.0 ** 17), (257, 2.0 ** -7), (513, -2.0 ** 17)):
        W2[..., i // 2] = 0x20
        x[:, i] = v                                # M[i] = 128 x[i]
    mats = [{"packed": dev_u8(W1, device), "scale": dev_u8(np.full((E, H, K // 32), 127), device)},
            _one_hot_rows(E, H, K, device),
            {"packed": dev_u8(W2, device), "scale": dev_u8(np.full((E, O, H // 32), 127), device)}]
    ids = torch.zeros((T, 1), dtype=torch.int32, device=device)
    xd = torch.from_numpy(x).to(torch.bfloat16).to(device)
    out = gb.mxfp4_moe_grouped_gemv(xd, *mats, ids, torch.ones((T, 1), device=device))
    assert torch.equal(out, torch.ones_like(out))


@pytest.mark.parametrize("K,H", [(1024, 2048), (2048, 1024), (4096, 2048), (3072, 1280)])
@pytest.mark.parametrize("small", [0, 1, 2])
def test_decode_batches_smallest_scales(device, small, K, H):
    """All scale bytes of one matrix 0 or 1 (2^-127, 2^-126), with activations or
    other scales that make the result an ordinary number: the weights are exact
    on the matrix cores too, so the general kernels give it up to the rounding of
    sums and M. One expert of W2 has no such byte."""
    T, topk, E, O = 33, 8, 16, 192
    announce(f"decode batches smallest scales K={K} H={H} matrix {small}")
    assert _decode_stages(T, topk, E, K, H, O) == 3
    rng = np.random.default_rng(9750 + K)
    mats = []
    for m, (rows, cols) in enumerate(((H, K), (H, K), (O, H))):
        p, s = synth.mxfp4_weight(9760 + 2 * m, rows, cols, E)
        if m == small:
            s = rng.integers(0, 2, s.shape).astype(np.uint8)
            if m == 2:
                s[3] = rng.integers(2, 4, s[3].shape)
        elif m == 1 and small == 2:
            s = (s + 100).astype(np.uint8)         # M about 2^100
        mats.append({"packed": dev_u8(p, device), "scale": dev_u8(s, device)})
    scale = 1.0 if small == 2 else 2.0 ** 100      # the other of W1 x and W3 x about 2^100
    x = mx.bf16_round(mx.bf16_to_f32(synth.normal_bf16(9770, (T, K))) * np.float32(scale))
    ids = np.stack([rng.permutation(E)[:topk] for _ in range(T)]).astype(np.int32)
    ids[:, 0] = 1                                  # 33 pairs on one expert
    w = (rng.random((T, topk)) + 0.1).astype(np.float32)
    args = torch.from_numpy(ids).to(device), dev_f32(w, device)
    gen = [{"packed": m["packed"], "scale": _at_offset(m["scale"], 1)} for m in mats]
    out = gb.mxfp4_moe_grouped_gemv(dev_bf16(x, device), *mats, *args)
    want = host_bits(gb.mxfp4_moe_grouped_gemv(dev_bf16(x, device), *gen, *args))
    assert np.median(np.abs(mx.bf16_to_f32(want))) > 2.0 ** -100
    assert_close(host_bits(out), want, "smallest scales", cos_tol=0.99999)
