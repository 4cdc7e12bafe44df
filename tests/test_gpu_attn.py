"""Attention (ggml_flash_attn_ext over an f16 KV cache) against the oracle: one row within 1e-3, several rows within 1e-5
and no further from float64 than the per-row kernel."""

import numpy as np
import pytest
import torch

from conftest import to_np

pytestmark = pytest.mark.gpu
TOL = 1e-3


def _case(orc, H, Hkv, Sq, n_kv, D, ctx, seed, causal=True):
    q = orc.normal((H, Sq, D), seed=seed)
    kc = orc.fp32_to_fp16(orc.normal((Hkv, ctx, D), seed=seed + 1))
    vc = orc.fp32_to_fp16(orc.normal((Hkv, ctx, D), seed=seed + 2))
    pos = n_kv - Sq + np.arange(Sq)
    mask = np.where((np.arange(n_kv)[None] <= pos[:, None]) | (not causal), 0.0, -np.inf).astype(np.float32)
    return q, kc, vc, orc.fp32_to_fp16(mask)


def _run(gops, q, kc, vc, m16, n_kv, scale):
    tq = torch.from_numpy(q).cuda()
    tk = torch.from_numpy(kc.view(np.float16)).cuda()
    tv = torch.from_numpy(vc.view(np.float16)).cuda()
    tm = None if m16 is None else torch.from_numpy(m16.view(np.float16)).cuda()
    return to_np(gops.flash_attn_ext(tq, tk, tv, tm, scale, n_kv=n_kv))


@pytest.mark.parametrize("n_kv", [1, 17, 512, 4096, 32768])
def test_decode_llama_heads(gops, orc, n_kv):
    """32 query heads on 8 KV heads, d=128, one query at the last position (every key visible)."""
    H, Hkv, D = 32, 8, 128
    q, kc, vc, m16 = _case(orc, H, Hkv, 1, n_kv, D, n_kv, seed=40)
    out = _run(gops, q, kc, vc, m16, n_kv, 1 / np.sqrt(D))
    ref = orc.flash_attn_ext(q, kc, vc, m16, 1 / np.sqrt(D))
    assert orc.parity(out, ref) < TOL


def test_cache_view_and_masked_tail(gops, orc):
    """K/V are the first n_kv rows of a longer cache; keys past the position are -inf."""
    H, Hkv, D, ctx, n_kv, Sq = 32, 8, 128, 2048, 768, 3
    q, kc, vc, m16 = _case(orc, H, Hkv, Sq, n_kv, D, ctx, seed=41)
    m16 = m16.copy()
    m16[:, 700:] = orc.fp32_to_fp16(np.array([-np.inf], np.float32))[0]
    out = _run(gops, q, kc, vc, m16, n_kv, 0.088)
    ref = orc.flash_attn_ext(q, kc[:, :n_kv], vc[:, :n_kv], m16, 0.088)
    assert orc.parity(out, ref) < TOL


@pytest.mark.parametrize("H,Hkv,D", [(4, 4, 64), (8, 2, 128), (16, 2, 256), (6, 3, 128)])
def test_head_layouts(gops, orc, H, Hkv, D):
    q, kc, vc, m16 = _case(orc, H, Hkv, 2, 300, D, 300, seed=42)
    out = _run(gops, q, kc, vc, m16, 300, 0.1)
    assert orc.parity(out, orc.flash_attn_ext(q, kc, vc, m16, 0.1)) < TOL


def test_no_mask_and_fully_masked_row(gops, orc):
    q, kc, vc, _ = _case(orc, 4, 2, 2, 50, 128, 50, seed=43)
    out = _run(gops, q, kc, vc, None, 50, 0.125)
    assert orc.parity(out, orc.flash_attn_ext(q, kc, vc, None, 0.125)) < TOL
    mask = np.zeros((2, 50), np.float32)
    mask[1] = -np.inf
    m16 = orc.fp32_to_fp16(mask)
    out = _run(gops, q, kc, vc, m16, 50, 0.125)
    assert np.isfinite(out).all() and not out[1].any()
    assert orc.parity(out, orc.flash_attn_ext(q, kc, vc, m16, 0.125)) < TOL


def test_prefill_rows(gops, orc):
    H, Hkv, D, Sq = 32, 8, 128, 64
    q, kc, vc, m16 = _case(orc, H, Hkv, Sq, 512, D, 512, seed=44)
    out = _run(gops, q, kc, vc, m16, 512, 1 / np.sqrt(D))
    assert orc.parity(out, orc.flash_attn_ext(q, kc, vc, m16, 1 / np.sqrt(D))) < TOL


@pytest.mark.parametrize("n_kv", [1, 17, 129, 700, 1024, 1500, 2048, 2049, 4096, 32768])
@pytest.mark.parametrize("H,Hkv,D", [(32, 8, 128), (8, 8, 128), (8, 4, 64), (16, 4, 64), (64, 8, 128), (16, 2, 64)])
def test_decode_kernel_no_mask(gops, orc, n_kv, H, Hkv, D):
    """One query row: up to 2048 keys the lane-group kernel (splits of 64 keys at D = 128, 128 at
    D = 64, at most 512 / H of them, 4, 8 or 16 wavefronts each), beyond it the matrix-core kernel
    (16-key blocks per wavefront, Q·Kᵀ and Vᵀ·P on MFMA, online softmax per head, wavefronts merged
    in LDS); splits merged by k_attn_merge. Against the oracle within 1e-3, 1 to 8 query heads per
    KV head. 17 keys leave most wavefronts without a key; 129 gives three splits of 43 keys; 1500
    ends inside a 16-key block; 2048 / 2049 are the last lane-group and first matrix-core
    lengths."""
    q, kc, vc, _ = _case(orc, H, Hkv, 1, n_kv, D, n_kv, seed=45)
    out = _run(gops, q, kc, vc, None, n_kv, 1 / np.sqrt(D))
    ref = orc.flash_attn_ext(q, kc, vc, None, 1 / np.sqrt(D))
    assert orc.parity(out, ref) < TOL


@pytest.mark.parametrize("H,Hkv", [(32, 8), (16, 2)])
def test_decode_row_with_holes_in_the_mask(gops, orc, H, Hkv):
    """One query row with an f16 mask that drops keys inside blocks and whole blocks, and adds
    finite biases to others: the decode kernel's mask path against the oracle."""
    D, n_kv = 128, 1000
    q, kc, vc, _ = _case(orc, H, Hkv, 1, n_kv, D, n_kv, seed=46)
    mask = (orc.normal((1, n_kv), seed=47) * 0.5).astype(np.float32)
    mask[0, 3:9] = -np.inf
    mask[0, 64:160] = -np.inf
    mask[0, 997] = -np.inf
    m16 = orc.fp32_to_fp16(mask)
    out = _run(gops, q, kc, vc, m16, n_kv, 1 / np.sqrt(D))
    assert orc.parity(out, orc.flash_attn_ext(q, kc, vc, m16, 1 / np.sqrt(D))) < TOL


@pytest.mark.parametrize("H,Hkv,D", [(4, 4, 64), (14, 2, 64), (8, 2, 128), (12, 4, 128), (16, 2, 128)])
@pytest.mark.parametrize("Sq,n_kv", [(2, 2), (5, 67), (9, 64), (17, 300), (65, 65), (129, 256), (200, 1111)])
@pytest.mark.parametrize("masked", [True, False])
def test_prompt_rows(gops, orc, H, Hkv, D, Sq, n_kv, masked):
    """Prompt attention on the matrix cores: 1, 2 and 4 row groups (up to 32, up to 64, more rows of a KV
    head), partial row tiles and key blocks, heads per KV head that do not divide a tile, one and
    several key splits; causal masks whose blocks are empty, full and partial, and no mask. f32 sums over
    n_kv keys, weights to 22 bits or an absolute 2^-40 of the largest: about 2^-21 sqrt(n_kv) of the largest value together,
    which 1e-5 holds with room."""
    q, kc, vc, m16 = _case(orc, H, Hkv, Sq, n_kv, D, n_kv + 5, seed=50)
    out = _run(gops, q, kc, vc, m16 if masked else None, n_kv, D ** -0.5)
    ref = orc.flash_attn_ext(q, kc[:, :n_kv], vc[:, :n_kv], m16 if masked else None, D ** -0.5)
    assert orc.parity(out, ref) < 1e-5


def test_prompt_rows_mask_values(gops, orc):
    """Finite mask values (added to the scores), -inf keys scattered through blocks, a row that sees no key
    (zeros), rows whose first visible key is far in, a mask with a wider row stride; scores spread over
    a hundred powers of two (the reference exponent moves block by block)."""
    H, Hkv, D, Sq, n_kv = 8, 2, 128, 33, 523
    q, kc, vc, _ = _case(orc, H, Hkv, Sq, n_kv, D, n_kv, seed=51)
    rng = np.random.default_rng(3)
    m = rng.standard_normal((Sq, n_kv)).astype(np.float32) * 2
    m[rng.random((Sq, n_kv)) < 0.3] = -np.inf
    m[4] = -np.inf
    m[7, :500] = -np.inf
    m[8] += np.linspace(-40, 30, n_kv)
    m16 = orc.fp32_to_fp16(m)
    wide = np.zeros((Sq, n_kv + 13), np.uint16)
    wide[:, :n_kv] = m16
    out = to_np(gops.flash_attn_ext(torch.from_numpy(q).cuda(), torch.from_numpy(kc.view(np.float16)).cuda(),
                                    torch.from_numpy(vc.view(np.float16)).cuda(),
                                    torch.from_numpy(wide.view(np.float16)).cuda(), 0.3, n_kv=n_kv))
    ref = orc.flash_attn_ext(q, kc, vc, m16, 0.3)
    assert np.all(out.reshape(Sq, -1)[4] == 0.0)
    assert orc.parity(out, ref) < 1e-5


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("n_kv", [64, 67, 300])
@pytest.mark.parametrize("masked", [True, False])
@pytest.mark.parametrize("scale", [0.0, -0.0, 1e-40, 2.0 ** -61, -(2.0 ** -60), -0.1, 1e5, -3e6, 7e7, 2.0 ** 31,
                                   -(2.0 ** 45), 2.0 ** 60, -(2.0 ** 61), 2.0 ** 100])
def test_prompt_rows_scales(gops, orc, D, n_kv, masked, scale):
    """Every finite scale over several query rows: 0 gives the mean of the visible values, tiny ones too; negative
    ones; huge ones the value of the best key. Whole-number q and k make the dot products exact, so the best keys (ties among
    them) are the same ones in every order of the sums."""
    H, Hkv, Sq = 8, 2, 9
    rng = np.random.default_rng(n_kv)
    q = rng.integers(-3, 4, (H, Sq, D)).astype(np.float32)
    kc = orc.fp32_to_fp16(rng.integers(-3, 4, (Hkv, n_kv, D)).astype(np.float32))
    _, _, vc, m16 = _case(orc, H, Hkv, Sq, n_kv, D, n_kv, seed=52)
    m16 = m16 if masked else None
    out = _run(gops, q, kc, vc, m16, n_kv, scale)
    assert orc.parity(out, orc.flash_attn_ext(q, kc, vc, m16, scale)) < 1e-5


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("n_kv", [2048, 2049, 2111, 4160])
@pytest.mark.parametrize("what", ["causal", "far", "border", "scattered"])
def test_prompt_rows_mask_block_words(gops, orc, D, n_kv, what):
    """Masks of more than 2048 keys over several row tiles: a word of the mask's block bits holds 32 blocks of 64 keys.
    Causal masks; tiles that see nothing of the first word, or nothing at all; visible keys only on both sides of the
    word's border; and single visible blocks far apart."""
    H, Hkv, Sq = 8, 2, 100
    q, kc, vc, m16 = _case(orc, H, Hkv, Sq, n_kv, D, n_kv + 3, seed=55)
    if what != "causal":
        m = np.full((Sq, n_kv), -np.inf, np.float32)
        if what == "far":
            m[:32, n_kv - 40:] = 0  # the first tile of 128 (query, head) rows; the second sees nothing
            m[64:, :5] = 0
        elif what == "border":
            m[:, 2048 - 70:2048 - 60] = 0
            m[:, 2047:2050] = 0
        else:
            m[np.arange(Sq), (np.arange(Sq) * 61) % n_kv] = 0
            m[:, n_kv - 1] = 0
        m16 = orc.fp32_to_fp16(m)
    out = _run(gops, q, kc, vc, m16, n_kv, D ** -0.5)
    assert orc.parity(out, orc.flash_attn_ext(q, kc[:, :n_kv], vc[:, :n_kv], m16, D ** -0.5)) < 1e-5


@pytest.mark.parametrize("H,Hkv,D,Sq,n_kv", [(8, 2, 64, 5, 300), (8, 2, 128, 13, 700), (8, 2, 128, 70, 2200), (14, 2, 64, 3, 9000)])
@pytest.mark.parametrize("masked", [True, False])
def test_prompt_rows_interleaved_cache(gops, orc, H, Hkv, D, Sq, n_kv, masked):
    """K and V rows farther apart than D ([ctx, Hkv, D + pad] caches viewed as [Hkv, ctx, D], K and V of different pads), q
    rows in both orders; at 9000 keys more than 32 splits meet in the merge."""
    q, kc, vc, m16 = _case(orc, H, Hkv, Sq, n_kv, D, n_kv, seed=56)

    def view(c, pad):
        t = torch.zeros((n_kv, Hkv, D + pad), dtype=torch.float16, device="cuda")
        t[:, :, :D] = torch.from_numpy(c.view(np.float16)).cuda().transpose(0, 1)
        return t[:, :, :D].transpose(0, 1)

    tq = torch.from_numpy(q).cuda()
    tm = torch.from_numpy(m16.view(np.float16)).cuda() if masked else None
    ref = orc.flash_attn_ext(q, kc, vc, m16 if masked else None, 0.1)
    for qq in (tq, tq.transpose(0, 1).contiguous().transpose(0, 1)):
        out = to_np(gops.flash_attn_ext(qq, view(kc, 8), view(vc, 24), tm, 0.1, n_kv=n_kv))
        assert orc.parity(out, ref) < 1e-5


def _same_with_infinities(out, ref, tol):
    for kind in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(kind(out), kind(ref)), kind.__name__
    f = np.isfinite(ref)
    assert np.max(np.abs(out[f] - ref[f])) < tol * max(1.0, np.max(np.abs(ref[f])))


@pytest.mark.parametrize("H,Hkv,D,Sq", [(8, 2, 64, 5), (8, 2, 128, 5), (8, 2, 128, 13), (8, 2, 64, 70), (8, 2, 128, 70)])
@pytest.mark.parametrize("n_kv", [96, 1000])
@pytest.mark.parametrize("masked", [True, False])
def test_prompt_rows_infinite_values(gops, orc, H, Hkv, D, Sq, n_kv, masked):
    """A V value that overflowed f16: every row that sees its key with any weight (e^-40 of the largest, too) gets that
    infinity in its dim, a NaN where both signs meet, and no other dim or row changes; a key that a row does not see
    does not count. A NaN in V alike."""
    q, kc, vc, m16 = _case(orc, H, Hkv, Sq, n_kv, D, n_kv, seed=53)
    m = np.zeros((Sq, n_kv), np.float32)
    m[:, n_kv - Sq:] = np.where(np.arange(Sq)[None] <= np.arange(Sq)[:, None], 0, -np.inf)
    m[:, 20] = -40
    vc = vc.copy()
    vc[0, 7, 3], vc[0, 20, 11], vc[0, n_kv - 2, 3] = 0x7C00, 0xFC00, 0xFC00  # +inf; -inf at the weight e^-40; -inf late
    vc[1, 40, 30] = 0x7E00  # NaN
    m16 = orc.fp32_to_fp16(m) if masked else None
    out = _run(gops, q, kc, vc, m16, n_kv, D ** -0.5)
    _same_with_infinities(out, orc.flash_attn_ext(q, kc, vc, m16, D ** -0.5), 1e-5)


def _error2(gops, q, kc, vc, m16, n_kv, scale):
    """The squared 2-norm of the error against float64, of the prompt kernel and of the per-row kernel (which takes heads
    of 256: the same values beside zeros)."""
    H, Sq, D = q.shape
    G = H // kc.shape[0]
    f16 = lambda a: a.view(np.float16).astype(np.float64)  # noqa: E731
    k, v = f16(kc)[:, :n_kv], f16(vc)[:, :n_kv]
    ref = np.empty((Sq, H, D))
    for h in range(H):
        s = q[h].astype(np.float16).astype(np.float64) @ k[h // G].T * float(np.float32(scale)) + f16(m16)
        p = np.exp(s - s.max(1, keepdims=True))
        ref[:, h] = p @ v[h // G] / p.sum(1, keepdims=True)
    wide = lambda a: np.concatenate([a, np.zeros((*a.shape[:2], 256 - D), a.dtype)], 2)  # noqa: E731
    out = _run(gops, q, kc, vc, m16, n_kv, scale).reshape(Sq, H, D)
    rows = _run(gops, wide(q), wide(kc), wide(vc), m16, n_kv, scale).reshape(Sq, H, 256)[:, :, :D]
    return np.sum((out - ref) ** 2), np.sum((rows - ref) ** 2)


@pytest.mark.parametrize("H,Hkv,D,Sq,n_kv", [(4, 4, 128, 13, 16), (14, 2, 64, 79, 107), (8, 4, 128, 79, 297), (4, 4, 64, 20, 3000),
                                             (8, 1, 128, 5, 21504), (2, 2, 128, 29, 14510), (8, 2, 128, 70, 5000)])
def test_prompt_rows_precision(gops, orc, H, Hkv, D, Sq, n_kv):
    """The matrix cores' sums and the split weights are no further from float64 than the per-row kernel's f32 sums (5 %:
    how far the ratio of two errors of a few thousand values moves with the inputs)."""
    e = np.zeros(2)
    for seed in (60, 70, 80):
        q, kc, vc, m16 = _case(orc, H, Hkv, Sq, n_kv, D, n_kv, seed=seed)
        e += _error2(gops, q, kc, vc, m16, n_kv, D ** -0.5)
    assert np.sqrt(e[0] / e[1]) < 1.05


@pytest.mark.parametrize("H,Hkv,D,Sq,n_kv", [(8, 2, 128, 5, 700), (8, 2, 128, 33, 523)])
def test_prompt_rows_precision_large_scores(gops, orc, H, Hkv, D, Sq, n_kv):
    """The same for scores of up to 13 over several splits, whose maxima are no powers of two."""
    e = np.zeros(2)
    for seed in (60, 70, 80, 90):
        q, kc, vc, m16 = _case(orc, H, Hkv, Sq, n_kv, D, n_kv, seed=seed)
        e += _error2(gops, q, kc, vc, m16, n_kv, 0.3)
    assert np.sqrt(e[0] / e[1]) < 1.05


@pytest.mark.parametrize("H,Hkv,D,Sq,n_kv", [(8, 2, 128, 5, 700), (8, 2, 128, 33, 523), (14, 2, 64, 129, 257), (8, 2, 128, 30, 90)])
@pytest.mark.parametrize("what", ["added", "distance", "lowest", "thousand"])
def test_prompt_rows_precision_mask_values(gops, orc, H, Hkv, D, Sq, n_kv, what):
    """The same for finite mask values: N(0, 2), a distance penalty, the type's lowest value on every key of half of the rows
    (their weights come from scores rounded at 65504 in both kernels), and 1000."""
    e = np.zeros(2)
    for seed in (60, 70, 80, 90):
        q, kc, vc, m16 = _case(orc, H, Hkv, Sq, n_kv, D, n_kv, seed=seed)
        m = m16.view(np.float16).astype(np.float32)
        if what == "added":
            m += 2 * orc.normal((Sq, n_kv), seed=seed + 5)
        elif what == "distance":
            m -= np.abs(np.arange(n_kv)[None] - (n_kv - Sq + np.arange(Sq)[:, None])) / 32
        elif what == "lowest":
            m[::2] = -65504
        else:
            m += 1000
        m16 = orc.fp32_to_fp16(m)
        e += _error2(gops, q, kc, vc, m16, n_kv, D ** -0.5)
    assert np.sqrt(e[0] / e[1]) < 1.05


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("Sq", [1, 2, 40])
def test_more_than_8_heads_per_kv_head_refused(gops, orc, D, Sq):
    """The C API's bound (include/gcq.h), for one query row and several, with and without a mask."""
    q, kc, vc, m16 = _case(orc, 9, 1, Sq, 70, D, 70, seed=54)
    for m in (m16, None):
        with pytest.raises(Exception, match="8 query heads"):
            _run(gops, q, kc, vc, m, 70, 0.1)
