"""Exact token batches bit for bit against the C oracle. Products of up to 16384
outputs run on the one-wave-per-row kernels (SIZES); larger ones on the tiles
of k3_exact.hip (TILES: every dense form, partial row blocks, rows shorter than
a stage and longer than the staged scales, several rounds of the persistent
grid). Both with aligned and unaligned tensors; the grouped form in every tile
shape; and denormal, infinite and signed-zero inputs on each."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import _oracle as O  # noqa: E402
import _ops as ops  # noqa: E402
from moonshine_amd import layer as L  # noqa: E402
from moonshine_amd.synth import ACT_SITU, Config, f32_to_bf16_bits, make_inputs  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cuda():
    return torch.device("cuda:0")


def bf16(rng, shape):
    return f32_to_bf16_bits(rng.normal(0, 1, shape).astype(np.float32))


def at_offset(a, off, cuda):
    """The array's bytes on the device, `off` bytes past a 16-byte boundary."""
    raw = np.ascontiguousarray(a).view(np.uint8).reshape(-1)
    buf = torch.zeros(raw.size + 32, dtype=torch.uint8, device=cuda)
    buf[off:off + raw.size] = torch.from_numpy(raw).to(cuda)
    return buf[off:]


SIZES = [(2, 64, 512), (3, 1, 32), (4, 33, 64), (5, 65, 288), (8, 63, 544), (9, 130, 1024),
         (16, 32, 3584), (17, 96, 8192), (33, 31, 8224), (2, 40, 16512), (64, 7, 256)]


# 16-row tiles (few works); 64-row tiles of one, two and four quads of tokens
TILES = [(17, 1025, 288), (130, 129, 544), (512, 33, 128), (8, 4001, 8224), (64, 1050, 16512),
         (2, 12321, 288), (4, 8225, 32), (3, 40000, 64), (3, 20011, 8224),
         (7, 4161, 1024), (5, 6111, 64), (8, 8191, 8256),
         (33, 2753, 544), (16, 8255, 96), (40, 3001, 8224), (64, 16500, 64), (9, 8200, 512)]


@pytest.mark.parametrize("T,rows,cols", SIZES + TILES)
def test_mxfp4_batches(cuda, T, rows, cols):
    rng = np.random.default_rng(T * 7919 + rows * 31 + cols)
    p = rng.integers(0, 256, (rows, cols // 2), dtype=np.uint8)
    s = rng.integers(118, 130, (rows, cols // 32), dtype=np.uint8)
    x = bf16(rng, (T, cols))
    out = torch.zeros((T, rows), dtype=torch.int16, device=cuda)
    dx = torch.from_numpy(x.view(np.int16)).to(cuda)
    want, _ = O.mxfp4_gemm(p, s, x, rows, cols)
    for poff, soff in ((0, 0), (8, 1)):
        assert ops.k3_rocm_mxfp4_gemm_bf16(out, at_offset(p, poff, cuda), at_offset(s, soff, cuda),
                                           dx, T, rows, cols)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy().view(np.uint16), want)
        out.zero_()


@pytest.mark.parametrize("T,rows,cols",
                         [(T, r, (c + 127) // 128 * 128) for T, r, c in SIZES + TILES])
def test_q8_batches(cuda, T, rows, cols):
    rng = np.random.default_rng(T * 104729 + rows * 17 + cols)
    q = rng.integers(-127, 128, (rows, cols)).astype(np.int8)
    s = rng.uniform(1e-3, 1e-2, (rows, cols // 128)).astype(np.float32)
    x = bf16(rng, (T, cols))
    out = torch.zeros((T, rows), dtype=torch.int16, device=cuda)
    dx = torch.from_numpy(x.view(np.int16)).to(cuda)
    want = O.q8_gemm(q, s, x)[0]
    for qoff, soff in ((0, 0), (8, 4)):
        assert ops.k3_rocm_q8_128_gemm_bf16(out, at_offset(q, qoff, cuda),
                                            at_offset(s, soff, cuda), dx, T, rows, cols)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy().view(np.uint16), want)
        out.zero_()


def odd_inputs(rng, shape):
    """Tokens of ordinary values, of bf16 denormals, with -0 and with infinities, in turn."""
    x = bf16(rng, shape)
    x[1::4] = rng.integers(1, 0x80, x[1::4].shape) | (rng.integers(0, 2, x[1::4].shape) << 15)
    x[2::4][rng.random(x[2::4].shape) < 0.5] = 0x8000
    x[3::4, ::29] = np.array([0x7F80, 0xFF80], np.uint16)[rng.integers(0, 2, x[3::4, ::29].shape)]
    return x


def equal_or_both_nan(got, want):
    nan = ((got & 0x7FFF) > 0x7F80) & ((want & 0x7FFF) > 0x7F80)
    np.testing.assert_array_equal(np.where(nan, 0, got), np.where(nan, 0, want))
    return nan


@pytest.mark.parametrize("T,rows,cols", [(17, 1025, 288), (4, 8225, 96), (7, 4161, 512),
                                         (33, 2753, 544)])
def test_dense_tiles_extremes(cuda, T, rows, cols):
    """E8M0 bytes 0, 1, 254 and 255 among ordinary ones, and for both formats
    scales that bring denormal sums back into range."""
    rng = np.random.default_rng(T + rows)
    p = rng.integers(0, 256, (rows, cols // 2), dtype=np.uint8)
    s = rng.integers(118, 130, (rows, cols // 32), dtype=np.uint8)
    s[::3] += 100                      # denormal tokens end up in the normal range
    s[1::3][rng.random(s[1::3].shape) < 0.1] = 0
    s[1::3][rng.random(s[1::3].shape) < 0.1] = 1
    s[5], s[8, 0], s[11] = 254, 255, 0
    x = odd_inputs(rng, (T, cols))
    dx = torch.from_numpy(x.view(np.int16)).to(cuda)
    out = torch.zeros((T, rows), dtype=torch.int16, device=cuda)
    assert ops.k3_rocm_mxfp4_gemm_bf16(out, at_offset(p, 0, cuda), at_offset(s, 0, cuda), dx, T,
                                       rows, cols)
    torch.cuda.synchronize()
    want, _ = O.mxfp4_gemm(p, s, x, rows, cols)
    assert not equal_or_both_nan(out.cpu().numpy().view(np.uint16), want)[1::4, ::3].any()
    c8 = (cols + 127) // 128 * 128
    q = rng.integers(-127, 128, (rows, c8)).astype(np.int8)
    f = rng.uniform(1e-3, 1e-2, (rows, c8 // 128)).astype(np.float32)
    f[::3] *= np.float32(1e30)
    f[1::3, 0] = np.float32(1e-41)
    x = odd_inputs(rng, (T, c8))
    dx = torch.from_numpy(x.view(np.int16)).to(cuda)
    assert ops.k3_rocm_q8_128_gemm_bf16(out, at_offset(q, 0, cuda), at_offset(f, 0, cuda), dx, T,
                                        rows, c8)
    torch.cuda.synchronize()
    want = O.q8_gemm(q, f, x)[0]
    assert not equal_or_both_nan(out.cpu().numpy().view(np.uint16), want)[1::4].any()


def routes(counts, T, k):
    """ids [T, k] in which expert e has counts[e] tokens (spread over the
    batch); the other slots take k more experts, one per slot."""
    ids = np.tile(np.arange(k, dtype=np.uint32) + len(counts), (T, 1))
    free = np.zeros(T, np.int64)
    for e in np.argsort(-np.asarray(counts), kind="stable"):
        for t in np.argsort(free, kind="stable")[:counts[e]]:
            ids[t, free[t]] = e
            free[t] += 1
    return ids


# every light tile (1 .. 8 rows), the heavy ones and their remainders
COUNTS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 16, 17, 21, 24, 33, 38, 40, 0, 40]


@pytest.mark.parametrize("hidden,ffn,act", [(96, 160, 1), (576, 1056, ACT_SITU), (512, 32, 1),
                                            (8224, 544, 1)])
@pytest.mark.parametrize("shift", [0, 4])
def test_grouped_tiles(cuda, hidden, ffn, act, shift):
    T, k, E = 40, 12, len(COUNTS) + 12
    cfg = Config("tiles", T, hidden, E, k, ffn, scale=1.5, activation=act, seed=hidden + ffn)
    inputs = make_inputs(cfg)
    store = L.ExpertStore(E, hidden, ffn, seed=cfg.seed, device=cuda, misalign=shift)
    moe = L.build_layer(cfg, inputs, device=cuda, store=store)
    ids = routes(COUNTS, T, k)
    w = np.random.default_rng(5).uniform(0.01, 0.3, (T, k)).astype(np.float32)
    x, r = L.bf16_tensor(inputs.hidden, cuda), L.bf16_tensor(inputs.residual, cuda)
    out = moe.experts_only(x, torch.from_numpy(ids.view(np.int32)).to(cuda),
                           torch.from_numpy(w).to(cuda), residual=r)
    torch.cuda.synchronize()
    want = O.layer(cfg, inputs, {e: store.host_expert(e) for e in range(E)}, ids=ids, weights=w)
    np.testing.assert_array_equal(L.bf16_bits(out), want["output"])


@pytest.mark.parametrize("act", [1, ACT_SITU])
def test_grouped_tiles_extremes(cuda, act):
    """The same inputs through the grouped tiles: the down products' tokens are
    the activations of denormal, signed-zero and infinite rows."""
    from types import SimpleNamespace
    T, k, H, F = 40, 12, 288, 96
    E = len(COUNTS) + 12
    cfg = Config("odd", T, H, E, k, F, scale=1.5, activation=act, seed=3)
    inputs = make_inputs(cfg)
    rng = np.random.default_rng(17 + act)
    inputs.hidden[:] = odd_inputs(rng, (T, H))
    host, table, keep = {}, np.zeros((E, 6), np.int64), []
    for e in range(E):
        host[e] = []
        for j, (r, c) in enumerate(((F, H), (H, F), (F, H))):
            s = rng.integers(118, 130, (r, c // 32), dtype=np.uint8)
            s[::2] += 70
            s[1::4, 0] = rng.integers(0, 2, s[1::4, 0].shape)
            host[e] += [rng.integers(0, 256, (r, c // 2), dtype=np.uint8), s]
        keep.append([torch.from_numpy(t).to(cuda) for t in host[e]])
        table[e] = [t.data_ptr() for t in keep[e]]
    tab = torch.from_numpy(table).to(cuda)
    moe = L.RoutedMoE(cfg, tab, None, SimpleNamespace(table=tab))
    ids = routes(COUNTS, T, k)
    w = rng.uniform(0.01, 0.3, (T, k)).astype(np.float32)
    x, r = L.bf16_tensor(inputs.hidden, cuda), L.bf16_tensor(inputs.residual, cuda)
    out = moe.experts_only(x, torch.from_numpy(ids.view(np.int32)).to(cuda),
                           torch.from_numpy(w).to(cuda), residual=r)
    torch.cuda.synchronize()
    want = O.layer(cfg, inputs, host, ids=ids, weights=w)
    nan = equal_or_both_nan(L.bf16_bits(out), want["output"])
    assert not nan[1::4].any() and (want["expert_out"][1::4] & 0x7FFF).any()
