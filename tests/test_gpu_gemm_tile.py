"""The 64 x 64-tile GEMM of many rows against the 16-row one (GPU).

Both form the same sums in the same order, so a product of many rows has to be the same bits
as the same rows taken a few at a time, which go to the 16-row tiles: at the first sizes that
the large tiles take, with 1 row and with all 64 in the last tile, from row-major operands and
(in a prefill) from the matrix-core order with each epilogue.
"""
import numpy as np
import pytest

from mosship import HipLLM, lib
from mosship import moss_format as mf

pytestmark = pytest.mark.gpu


def _weights(torch, rows, cols, seed):
    rng = np.random.default_rng(seed)
    q = rng.integers(-127, 128, size=(rows, cols), dtype=np.int8)
    d = (np.abs(rng.standard_normal((rows, cols // 32))) * 0.02 / 127).astype(np.float16)
    return torch.from_numpy(mf.pack_q8x4(q, d).reshape(-1)).cuda()


@pytest.mark.parametrize("rows,cols,m", [(3072, 768, 449), (3072, 768, 512), (2304, 768, 1000), (1536, 256, 1023)])
def test_rows_do_not_depend_on_their_number(torch_gpu, rows, cols, m):
    torch = torch_gpu
    print(f"gemm rows={rows} cols={cols} m={m}", flush=True)
    w = _weights(torch, rows, cols, rows + m)
    x = torch.randn(m, cols, generator=torch.Generator("cuda").manual_seed(m), device="cuda")
    y, want = torch.empty(m, rows, device="cuda"), torch.empty(m, rows, device="cuda")
    lib.gemm_q8x4(w, rows, cols, x, m, y)
    for a in range(0, m, 48):
        b = min(m, a + 48)
        lib.gemm_q8x4(w, rows, cols, x[a:b], b - a, want[a:b])
    assert torch.equal(y, want)
    # an output that 16-byte stores may not touch takes the 16-row tiles and gives the same
    odd = torch.empty(m * rows + 1, device="cuda")
    lib.gemm_q8x4(w, rows, cols, x, m, odd[1:])
    assert torch.equal(odd[1:].view(m, rows), want)


@pytest.mark.parametrize("rows,cols,m", [(3072, 768, 641), (3072, 768, 704), (2304, 768, 961), (4096, 512, 513)])
def test_w8a8_rows_do_not_depend_on_their_number(torch_gpu, rows, cols, m):
    torch = torch_gpu
    print(f"gemm w8a8 rows={rows} cols={cols} m={m}", flush=True)
    w = _weights(torch, rows, cols, rows + m)
    x = torch.randn(m, cols, generator=torch.Generator("cuda").manual_seed(m), device="cuda")
    q = torch.empty(m, cols, device="cuda", dtype=torch.int8)
    d = torch.empty(m, cols // 32, device="cuda")
    lib.quantize_rows(x, m, cols, q, d)
    y, want = torch.empty(m, rows, device="cuda"), torch.empty(m, rows, device="cuda")
    lib.gemm_q8x4_w8a8(w, rows, cols, q, d, m, y)
    for a in range(0, m, 48):
        b = min(m, a + 48)
        lib.gemm_q8x4_w8a8(w, rows, cols, q[a:b], d[a:b], b - a, want[a:b])
    assert torch.equal(y, want)


@pytest.mark.parametrize("a16", [False, True])
@pytest.mark.parametrize("kv32", [False, True])
def test_long_prompt_is_its_pieces(torch_gpu, golden_model, a16, kv32):
    """A prompt of 961 rows (its last tile holds one) in one call and in three of 352 and 353
    (the same fc_out split, no large tiles): the same keys,
    values and hidden state."""
    print(f"a16={a16} kv32={kv32}", flush=True)
    blob, _ = golden_model
    n, rng = 961, np.random.default_rng(5)
    rows = mf.text_rows(rng.integers(0, mf.VOCAB, n))
    rows[n // 4:n // 2, 0] = mf.SLOT
    rows[n // 4:n // 2, 1:] = rng.integers(0, 1024, (n // 2 - n // 4, 16))
    m = HipLLM(blob, max_ctx=1024, kv_fp32=kv32, prefill_a16=a16)
    m.prefill(rows)
    whole = (*m.kv_export(n), m.hidden())
    m.reset()
    for at, end in ((0, 352), (352, 704), (608, n)):
        m.prefill(rows[at:end], start=at)
    pieces = (*m.kv_export(n), m.hidden())
    m.close()
    for w, p in zip(whole, pieces):
        assert np.array_equal(w, p)


@pytest.mark.parametrize("m,cols", [(1, 256), (3, 768), (640, 3072)])
def test_quantised_rows_do_not_depend_on_alignment(torch_gpu, m, cols):
    """Rows that 16-byte loads and 4-byte stores may touch, and the same ones off by a value: the same
    bytes and scales, with a block of zeros, of infinities and of NaN among them."""
    torch = torch_gpu
    x = torch.randn(m, cols, generator=torch.Generator("cuda").manual_seed(m), device="cuda")
    x[0, 32:64] = 0.0
    x[0, 70] = float("inf")
    x[-1, 130] = float("nan")
    odd = torch.empty(m * cols + 1, device="cuda")
    odd[1:] = x.view(-1)
    out = []
    for src, off in ((x, 0), (odd[1:], 1)):
        q = torch.empty(m * cols + off, device="cuda", dtype=torch.int8)
        d = torch.empty(m, cols // 32, device="cuda")
        lib.quantize_rows(src, m, cols, q[off:], d)
        out.append((q[off:].clone(), d))
    assert torch.equal(out[0][0], out[1][0])
    assert torch.equal(out[0][1].nan_to_num(7.0), out[1][1].nan_to_num(7.0))
