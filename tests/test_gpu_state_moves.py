"""The one-launch moves of a model's state (GPU): import, export, snapshot and restore, and the
admission to a batch stream, at the edges of a page and in every pair of cache types."""
import numpy as np
import pytest

from mosship import HipBatch, HipLLM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src32,dst32", [(False, False), (False, True), (True, False), (True, True)])
def test_state_moves(torch_gpu, golden_model, src32, dst32):
    blob, _ = golden_model
    m = HipLLM(blob, max_ctx=256, kv_fp32=src32)
    b = HipBatch(m, 3, 256, kv_fp32=dst32)
    rng = np.random.default_rng(3)
    for i, n in enumerate((200, 1, 63, 64, 65, 256, 0)):
        print(f"src32 {src32} dst32 {dst32} n {n}", flush=True)
        k, v = (rng.standard_normal((12, n, 768), dtype=np.float32) for _ in range(2))
        hidden = rng.standard_normal(768, dtype=np.float32)
        m.kv_import(k, v, hidden)
        held = (lambda x: x) if src32 else (lambda x: x.astype(np.float16).astype(np.float32))
        got = m.kv_export(n)
        assert np.array_equal(got[0], held(k)) and np.array_equal(got[1], held(v))
        assert np.array_equal(m.hidden(), hidden)
        if n:
            m.snapshot_prefix()
            m.kv_import(rng.standard_normal(k.shape, dtype=np.float32), v + 1, hidden)
            m.restore_prefix()
            got = m.kv_export(n)
            assert np.array_equal(got[0], held(k)) and np.array_equal(got[1], held(v))
        b.admit(i % 3, m)
        assert b.position(i % 3) == n and np.array_equal(b.hidden(i % 3), hidden)
        if n:
            got = b.kv_export(i % 3, n)
            want = (held(x) if dst32 else held(x).astype(np.float16).astype(np.float32) for x in (k, v))
            assert all(np.array_equal(g, w) for g, w in zip(got, want))
    b.close()
    m.close()


def test_moves_in_passes_keep_little(torch_gpu, golden_model):
    """Import and export of more positions than the staging buffer holds at once: every layer's
    K and V at the last size of one pass (227 positions), the first of two, five planes a pass and
    one plane larger than the buffer.  What the model keeps afterwards is at most the buffer's 16 MiB
    (and one page of the allocator)."""
    blob, _ = golden_model
    m = HipLLM(blob, max_ctx=5632)
    rng = np.random.default_rng(4)

    def used():
        torch_gpu.cuda.synchronize()
        free, total = torch_gpu.cuda.mem_get_info()
        return total - free

    start = used()
    for n in (1, 227, 228, 1024, 5600):
        print(f"n {n}", flush=True)
        k, v = (rng.integers(-2048, 2049, (12, n, 768)).astype(np.float32) for _ in range(2))  # exact in fp16
        m.kv_import(k, v, np.zeros(768, np.float32))
        got = m.kv_export(n)
        assert np.array_equal(got[0], k) and np.array_equal(got[1], v)
        assert used() - start <= (16 << 20) + (2 << 20), n
    m.close()
