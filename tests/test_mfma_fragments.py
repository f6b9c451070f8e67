"""The matrix fragments that plans of the matrix-core kernels upload: put back together by the
operand layout of the matrix instructions (lane l holds A[l % 16][Q (l / 16) + q]), high plus
low halves must be the DFT matrix, and the product with a line its DFT."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "emu")


@pytest.mark.parametrize("split", [0, 1])
@pytest.mark.parametrize("S", [-1, 1])
def test_fragments_are_the_dft_matrix(S, split):
    subprocess.run(["make", "-s", "-C", EMU, "libfft3d_emu.so"], check=True)
    lib = ctypes.CDLL(os.path.join(EMU, "libfft3d_emu.so"))
    lib.emu_frag.argtypes = [ctypes.c_int] * 3 + [ctypes.POINTER(ctypes.c_int)] * 3 + [
        ctypes.c_void_p, ctypes.c_size_t]
    # Each half is off by half a unit of its last place: the high one by 2^-9 (bf16) or 2^-12
    # (fp16) of an entry of at most 1, the low one by the same share of that, or half of fp16's
    # smallest step, 2^-25; and the entries are float32 themselves.
    bound = (2.0 ** -18, 2.0 ** -24 + 2.0 ** -25)[split] + 2.0 ** -25
    forms = 0
    for k in range(32):
        n, kw, fold = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
        buf = np.zeros(1 << 16, dtype=np.uint8)
        size = lib.emu_frag(S, split, k, n, kw, fold, buf.ctypes.data, buf.nbytes)
        if size == -1:
            break
        assert size > 0
        forms += 1
        n, kw, fold, Q = n.value, kw.value, fold.value, kw.value // 4
        h = buf[:size].view(np.uint16)
        v = (h.astype(np.uint32) << 16).view(np.float32) if split == 0 else h.view(np.float16)
        v = v.astype(np.float64).reshape(-1, 2, 64, Q).sum(axis=1)          # tile, lane, q
        tiles = np.zeros((v.shape[0], 16, kw))
        for lane in range(64):
            tiles[:, lane % 16, Q * (lane // 16):Q * (lane // 16) + Q] = v[:, lane]
        rng = np.random.default_rng(k)
        x = rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)
        want = np.fft.fft(x) if S < 0 else np.fft.ifft(x) * n
        pairs = lambda z: np.stack([z.real, z.imag], axis=-1).ravel()       # noqa: E731
        if fold:
            a, b = x[1:9] + x[:8:-1], x[1:9] - x[:8:-1]
            p, m = (t @ pairs(np.concatenate([a, b])) for t in tiles)
            got = np.concatenate([[x.sum()], x[0] + p[::2] + 1j * p[1::2],
                                  (x[0] + m[::2] + 1j * m[1::2])[::-1]])
        else:
            tm, tk = (2 * n + 15) // 16, (2 * n + kw - 1) // kw
            A = tiles.reshape(tm, tk, 16, kw).transpose(0, 2, 1, 3).reshape(16 * tm, kw * tk)
            assert not A[2 * n:].any() and not A[:, 2 * n:].any()
            y = A[:2 * n, :2 * n] @ pairs(x)
            got = y[::2] + 1j * y[1::2]
        # 2n entries a row, |x| parts at most 2 after the fold, real and imaginary outputs
        assert np.max(np.abs(got - want)) <= bound * 2 * n * 2 * np.sqrt(2), (n, kw, fold)
    assert forms == 9
