"""The GPU Tiled-CSL encoder must produce the reference's bits: it is compared with the CPU
oracle, with the committed outputs of the reference's own encoder (tests/golden/), and with
the product's host encoder."""
import hashlib
import json
import os
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _torch():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return torch


def _encode(spmm, A):
    torch = _torch()
    d_A = torch.from_numpy(np.ascontiguousarray(A).view(np.int16).copy()).cuda().view(torch.float16)
    print(f"[gpu case] device encode {A.shape}", flush=True)
    d_items, d_offsets = spmm.encode_on_device(d_A)
    torch.cuda.synchronize()
    return d_items, d_offsets


def _compare(spmm, oracle, A):
    """Device encoder against the CPU oracle (the checker) and against the product's host encoder."""
    d_items, d_offsets = _encode(spmm, A)
    got_items, got_offsets = d_items.cpu().numpy().view(np.uint32), d_offsets.cpu().numpy()
    o_items, o_offsets = oracle.encode(A)
    assert np.array_equal(got_offsets, o_offsets)
    assert np.array_equal(got_items, o_items)
    items, offsets = spmm.InitSparseMatrixA_API(A)
    assert np.array_equal(got_offsets, offsets)
    assert np.array_equal(got_items, items)
    return d_items, d_offsets


def test_device_encoder_matches_reference_golden_small(spmm):
    """Full arrays written by the reference's own encoder (tests/golden/make_golden.py)."""
    z = np.load(os.path.join(GOLD, "encoder_small.npz"))
    names = sorted({k.rsplit(".", 1)[0] for k in z.files})
    assert len(names) >= 10
    for n in names:
        d_items, d_offsets = _encode(spmm, z[n + ".A"])
        assert np.array_equal(d_offsets.cpu().numpy(), z[n + ".offsets"]), n
        assert np.array_equal(d_items.cpu().numpy().view(np.uint32), z[n + ".items"]), n


def test_device_encoder_matches_reference_golden_large(spmm):
    """SHA-256 of the reference encoder's output on larger seeded matrices."""
    with open(os.path.join(GOLD, "encoder_large.json")) as f:
        cases = json.load(f)
    for c in cases:
        A = spmm.synth_weights(c["M"], c["K"], c["sparsity"], c["row_skewed"], seed=c["seed"])
        assert hashlib.sha256(A.tobytes()).hexdigest() == c["input_sha256"]
        d_items, d_offsets = _encode(spmm, A)
        assert hashlib.sha256(d_items.cpu().numpy().tobytes()).hexdigest() == c["items_sha256"]
        assert hashlib.sha256(d_offsets.cpu().numpy().tobytes()).hexdigest() == c["offsets_sha256"]


def test_device_split_pack_matches_reference_golden(spmm, oracle):
    """The GPU's 2:4 split against the committed outputs of the reference's decompose()
    (tests/golden/decompose_small.npz).  The device entry point takes M % 128 == 0 and K % 128 == 0,
    so each case sits in the top left corner of an otherwise zero matrix of that shape (groups of
    four never cross a row, so the expected parts are the golden ones in the same corner).  The
    records are read back with the oracle's reader of the record layout."""
    torch = _torch()
    z = np.load(os.path.join(GOLD, "decompose_small.npz"))
    names = sorted({k.rsplit(".", 1)[0] for k in z.files})
    assert len(names) >= 7
    for n in names:
        A, A1, A2 = z[n + ".A"], z[n + ".A1"], z[n + ".A2"]
        m, k = A.shape
        M, K = -(-m // 128) * 128, -(-k // 128) * 128
        big = np.zeros((M, K), dtype=np.uint16)
        big[:m, :k] = A.view(np.uint16)
        want1 = np.zeros((M, K), dtype=np.uint16)
        want1[:m, :k] = A1.view(np.uint16)
        want2 = np.zeros((M, K), dtype=np.uint16)
        want2[:m, :k] = A2.view(np.uint16)
        d_A = torch.from_numpy(big.view(np.int16).copy()).to("cuda:0").view(torch.float16)
        print(f"[gpu case] device split+pack of golden case {n}", flush=True)
        packed, residual = spmm.split_pack_on_device(d_A)
        torch.cuda.synchronize()
        assert np.array_equal(residual.cpu().numpy().view(np.uint16), want2), n
        assert np.array_equal(oracle.a24_unpack(packed.cpu().numpy(), M, K).view(np.uint16), want1), n


@pytest.mark.parametrize("M,K,sparsity,skew", [
    (128, 64, 0.8, False), (256, 192, 0.5, False), (1024, 1024, 0.8, False), (1024, 1024, 0.9, True),
    (512, 512, 0.0, False), (512, 512, 0.999, False), (384, 64 * 5, 0.3, True),
])
def test_device_encoder_matches_oracle(spmm, oracle, M, K, sparsity, skew):
    _compare(spmm, oracle, spmm.synth_weights(M, K, sparsity, skew, seed=M + K))


@pytest.mark.parametrize("M,K,sparsity,passes", [(128, 64, 0.516, {1, 2}), (256, 64 * 9, 0.515, {1, 2}), (128, 64 * 8, 0.03, {2}),
                                                 (256, 64 * 17, 0.27, {2}), (256, 64 * 9, 0.01, {3})])
def test_device_encoder_edges(spmm, oracle, M, K, sparsity, passes):
    """Tiles around the 3968 words that the GPU encoder emits in one pass (48.4 % dense) and beyond, in two
    (31 groups of 128 words each, and a tail) and in three; spans of eight tiles, whole and with a rest of one; pads
    of every number."""
    A = spmm.synth_weights(M, K, sparsity, False, seed=M + K)
    words = -(-(A != 0).reshape(M // 128, 128, K // 64, 64).sum((1, 3)).ravel() // 4) * 4
    assert {1 if w <= 3968 else -(-(int(w) // 128) // 31) for w in words} <= passes
    if passes == {3}:
        assert (words % 128 > 0).all()
    _compare(spmm, oracle, A)


def test_device_encoder_special_tiles(spmm, oracle):
    """All-zero tiles, a fully dense tile, single elements, and the values the reference treats specially."""
    rng = np.random.default_rng(7)
    A = np.zeros((512, 256), dtype=np.float16)
    A[0:128, 0:64] = rng.standard_normal((128, 64)).astype(np.float16) + np.float16(3)  # dense tile (no zeros)
    A[128 + 5, 64 + 9] = 1.5                               # a single element: three pads
    A[256:384, 128:192][::7, ::5] = -2.0                   # regular pattern
    bits = A.view(np.uint16)
    bits[384 + 1, 192 + 1] = 0x8000                        # -0: dropped
    bits[384 + 2, 192 + 2] = 0x7e00                        # NaN: dropped (fabs(NaN) > 0 is false)
    bits[384 + 3, 192 + 3] = 0x7c00                        # +inf: kept
    bits[384 + 4, 192 + 4] = 0x0001                        # smallest subnormal: kept
    bits[384 + 5, 192 + 5] = 0xfc00                        # -inf: kept
    _compare(spmm, oracle, A)


def test_device_encoded_weight_feeds_the_product(spmm, oracle):
    torch = _torch()
    M, K, N = 512, 1024, 16
    A = spmm.synth_weights(M, K, 0.8, False, seed=5)
    B = spmm.synth_activations(N, K, seed=6)
    d_items, d_offsets = _compare(spmm, oracle, A)
    d_B = torch.from_numpy(B.view(np.int16).copy()).cuda()
    d_C = torch.full((N, M), float("nan"), dtype=torch.float16, device="cuda")
    spmm.SpMM_SplitK_API(None, None, d_items, d_offsets, d_B, d_C, M, N, K, None, 1)
    torch.cuda.synchronize()
    ref = oracle.gemm_f32(A, B)
    err = np.abs(d_C.cpu().numpy().astype(np.float32) - ref)
    assert (err <= 1e-2 + 1e-2 * np.abs(ref)).all()


def test_device_encoder_full_size(spmm):
    """OPT-30B FFN1: bit equality on 25088 tiles, and the time of the two device passes."""
    torch = _torch()
    M, K = 28672, 7168
    A = spmm.synth_weights(M, K, 0.8, False, seed=1234)
    t0 = time.perf_counter()
    items, offsets = spmm.InitSparseMatrixA_API(A)
    t_host = time.perf_counter() - t0
    d_A = torch.from_numpy(A.view(np.int16)).cuda().view(torch.float16)
    spmm.encode_on_device(d_A)  # warm up
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    d_items, d_offsets = spmm.encode_on_device(d_A)
    torch.cuda.synchronize()
    t_dev = time.perf_counter() - t0
    print(f"[gpu case] full-size encode: host {t_host * 1e3:.1f} ms, device {t_dev * 1e3:.2f} ms", flush=True)
    assert np.array_equal(d_offsets.cpu().numpy(), offsets)
    assert np.array_equal(d_items.cpu().numpy().view(np.uint32), items)


def test_device_encoder_rejects_bad_shapes(spmm):
    torch = _torch()
    z = torch.zeros(1024, dtype=torch.int32, device="cuda")
    lib = spmm.load_library()
    assert lib.SpMM_DeviceEncodeOffsets(None, z.data_ptr(), 100, 64, z.data_ptr()) != 0
    assert lib.SpMM_DeviceEncodeOffsets(None, z.data_ptr(), 128, 60, z.data_ptr()) != 0
    assert lib.SpMM_DeviceEncodeOffsets(None, None, 128, 64, z.data_ptr()) != 0
    assert lib.SpMM_DeviceEncodeItems(None, z.data_ptr(), 128, 64, None, z.data_ptr()) != 0


@pytest.mark.parametrize("at", [1, 2, 5])
def test_device_encoder_of_a_matrix_at_any_element(spmm, oracle, at):
    """A contiguous view that begins at any element of a larger buffer: the wide loads ask for no alignment."""
    torch = _torch()
    M, K = 256, 64 * 9
    A = spmm.synth_weights(M, K, 0.7, False, seed=at)
    flat = torch.zeros(M * K + 16, dtype=torch.float16, device="cuda:0")
    view = flat[at:at + M * K].view(M, K)
    view.copy_(torch.from_numpy(A.view(np.int16).copy()).cuda().view(torch.float16))
    print(f"[gpu case] device encode at element {at}", flush=True)
    d_items, d_offsets = spmm.encode_on_device(view)
    torch.cuda.synchronize()
    items, offsets = oracle.encode(A)
    assert np.array_equal(d_offsets.cpu().numpy(), offsets)
    assert np.array_equal(d_items.cpu().numpy().view(np.uint32), items)


def test_device_encoder_with_offsets_of_another_matrix(spmm):
    """The second step of the encoding, given offsets of a matrix that has fewer words in some tiles and more in others:
    tiles whose counts agree get their words, the room of all others and what lies behind stay as they were."""
    import ctypes

    torch = _torch()
    M, K = 512, 64 * 11
    dev = torch.device("cuda:0")
    A = torch.from_numpy(spmm.synth_weights(M, K, 0.8, False, seed=8).view(np.int16).copy()).to(dev).view(torch.float16)
    items, offsets = spmm.encode_on_device(A)
    kind = (torch.arange(M // 128 * (K // 64), device=dev) % 4).view(M // 128, K // 64)  # 0: emptied, 1: dense, else its own
    spread = kind.repeat_interleave(128, 0).repeat_interleave(64, 1)
    other = torch.where(spread == 0, torch.zeros_like(A), torch.where(spread == 1, torch.ones_like(A), A)).contiguous()
    mark, total = 0x5A5A5A5A, items.numel()
    out = torch.full((total + 16384,), mark, dtype=torch.int32, device=dev)
    print("[gpu case] device encode with foreign offsets", flush=True)
    rc = spmm.load_library().SpMM_DeviceEncodeItems(
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream or None), ctypes.c_void_p(other.data_ptr()), M, K,
        ctypes.c_void_p(offsets.data_ptr()), ctypes.c_void_p(out.data_ptr()))
    assert rc == 0
    torch.cuda.synchronize()
    keep = np.repeat((kind.view(-1) > 1).cpu().numpy(), 4 * np.diff(offsets.cpu().numpy()[:-1]))
    want, got = items.cpu().numpy(), out.cpu().numpy()
    assert np.array_equal(got[:total], np.where(keep, want, mark)) and (got[total:] == mark).all()


@pytest.mark.parametrize("heights", ["one", "few", "full", "staggered"])
@pytest.mark.parametrize("extra", [0, 1, 2, 3])
def test_device_encoder_uneven_banks(spmm, oracle, heights, extra):
    """Levels: tiles whose words lie in one bank (256 of them: the tallest there is, with pads on the empty banks),
    in a few, all full, and 32 different heights of odd and even distances, with 0 to 3 words more for the pads; NaN and
    signed zeros (not kept) everywhere else."""
    rng = np.random.default_rng(extra)
    M, K = 256, 64 * 5
    want = {"one": [256] + [0] * 31, "few": [0, 0, 255, 0, 1, 128] + [0] * 25 + [2], "full": [256] * 32,
            "staggered": [(7 * b * b) % 257 for b in range(32)]}[heights]
    column = ((np.arange(64) ^ ((np.arange(128)[:, None] & 7) << 3)) >> 1)  # the bank of (row, column)
    A = np.where(rng.random((M, K)) < 0.5, 0x8000, 0x7E01).astype(np.uint16)
    for r in range(0, M, 128):
        for c in range(0, K, 64):
            tile = np.ascontiguousarray(A[r:r + 128, c:c + 64])
            order = rng.permutation(32)
            for b in range(32):
                at = np.flatnonzero(column.ravel() == order[b])
                n = min(want[b] + (extra if b == 4 else 0), 256)
                tile.ravel()[rng.choice(at, size=n, replace=False)] = rng.choice([0x0001, 0x8001, 0x7C00, 0xFC00, 0x3C00], size=n)
            A[r:r + 128, c:c + 64] = tile
    _compare(spmm, oracle, A.view(np.float16))


@pytest.mark.parametrize("K", [(1 << 27) - 64, 1 << 27, (1 << 27) + 64])
def test_device_encoder_rows_of_a_quarter_gigabyte(spmm, oracle, K):
    """Sixteen rows of 2^27 columns are 2^32 bytes: tiles of odd and even row groups at the matrix's start, end and
    in between, all other tiles empty, each against the oracle on the tile alone."""
    torch = _torch()
    M, tiles = 128, K // 64
    if torch.cuda.mem_get_info()[0] < 2 * M * K + (4 << 30):
        pytest.skip("needs 36 GiB of device memory")
    rng = np.random.default_rng(K % 1000)
    at = sorted({0, 1, tiles // 2, tiles - 2, tiles - 1, *rng.integers(0, tiles, 20).tolist()})
    A = rng.standard_normal((M, 64 * len(at))).astype(np.float16)
    A[rng.random(A.shape) < 0.8] = 0
    A[64:] = np.where(rng.random((64, A.shape[1])) < 0.5, A[64:], np.float16(0))  # row groups of different densities
    d_A = torch.zeros((M, K), dtype=torch.float16, device="cuda:0")
    for i, t in enumerate(at):
        d_A[:, 64 * t:64 * t + 64] = torch.from_numpy(A[:, 64 * i:64 * i + 64].copy()).cuda()
    print(f"[gpu case] device encode {M} x {K}", flush=True)
    d_items, d_offsets = spmm.encode_on_device(d_A)
    torch.cuda.synchronize()
    del d_A
    torch.cuda.empty_cache()
    counts = np.zeros(tiles, dtype=np.int64)
    words = []
    for i, t in enumerate(at):
        items, offsets = oracle.encode(A[:, 64 * i:64 * i + 64])
        counts[t] = offsets[-1]
        words.append(items[:4 * offsets[-1]])
    offsets = d_offsets.cpu().numpy()
    assert offsets[0] == 0 and np.array_equal(np.diff(offsets), np.append(counts, 0))
    assert np.array_equal(d_items.cpu().numpy().view(np.uint32), np.concatenate(words))
