"""The exact batch kernels (k3_exact.hip) at the edges of their tiles, bit for
bit against the C oracle: token tiles of one row to several quads, partial
row blocks, rows shorter than a stage and longer than the staged scales,
unaligned tensors, and every tile shape of the grouped form."""
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


@pytest.mark.parametrize("T,rows,cols", SIZES)
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


@pytest.mark.parametrize("T,rows,cols", [(T, r, (c + 127) // 128 * 128) for T, r, c in SIZES])
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
