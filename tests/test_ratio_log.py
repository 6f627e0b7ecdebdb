"""The sparsity ratio that every operator call logs: the number the call returns, whatever thread, stream and size it comes from,
and also after a call whose line could not be written."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(n, seed):
    from anchor_attn.synthetic import make_qkv
    return [x.cuda() for x in make_qkv(n, 4, 2, head_dim=64, n_stripes=16 + 8 * seed, seed=seed)[:3]]


@pytest.fixture
def log_file(monkeypatch, tmp_path):
    from my_utils import Logger
    path = tmp_path / "sub" / "ratio.log"
    monkeypatch.setattr(Logger, "enabled", True)
    monkeypatch.setattr(Logger, "log_file_path", str(path))
    return path


def _logged(path):
    return [line.split("anchor sparse_ratio:")[1] for line in path.read_text().splitlines()]


def test_logged_ratio_is_the_returned_one(monkeypatch, log_file, capsys):
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn, anchor_attn_without_anchor
    from my_utils import Logger
    want = []
    for n_big, block in ((1, 32), (3, 32), (2, 16), (1, 32)):  # (a single big block: written by stage 1)
        q, k, v = _inputs(n_big * block * 16, n_big)
        ratio = anchor_attn(q, k, v, block_size=block)[1]
        assert ratio.shape == () and ratio.dtype == torch.float32 and ratio.is_cuda
        assert float(ratio) == float(anchor_attn_without_anchor(q, k, v, block_size=block)[1])
        want.append(str(float(ratio)))
    assert _logged(log_file) == want and want[1] != want[2] != "0.0"
    # a line that cannot be written, then one that can
    monkeypatch.setattr(Logger, "log_file_path", str(log_file.parent))
    q, k, v = _inputs(1536, 5)
    anchor_attn(q, k, v, block_size=32)
    assert "Unable to write" in capsys.readouterr().out
    monkeypatch.setattr(Logger, "log_file_path", str(log_file))
    q, k, v = _inputs(512, 1)
    assert float(anchor_attn(q, k, v, block_size=32)[1]) == 0.0 and _logged(log_file)[-1] == "0.0"
    # another default type: the ratio has it, and is logged from the tensor
    torch.set_default_dtype(torch.float64)
    try:
        q, k, v = [x.bfloat16() for x in _inputs(1536, 3)]
        ratio = anchor_attn(q, k, v, block_size=32)[1]
    finally:
        torch.set_default_dtype(torch.float32)
    assert ratio.dtype == torch.float64 and _logged(log_file)[-1] == str(float(ratio))


def test_threads_and_streams_log_their_own(log_file):
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn
    ratios, failures = [], []

    def work(seed):
        try:
            q, k, v = _inputs(1536, seed)
            torch.cuda.synchronize()
            with torch.cuda.stream(torch.cuda.Stream()):
                mine = [float(anchor_attn(q, k, v, block_size=32)[1]) for _ in range(5)]
            assert len(set(mine)) == 1
            ratios.extend(mine)
        except Exception as e:  # noqa: BLE001 - reported by the main thread
            failures.append(e)
    threads = [threading.Thread(target=work, args=(seed,)) for seed in (1, 3, 5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
    assert sorted(_logged(log_file)) == sorted(str(r) for r in ratios) and len(set(ratios)) == 3


def test_a_call_that_is_left_early_does_not_reach_the_next_ones_line(monkeypatch, log_file):
    from anchor_attn.src.ops import anchor_attn_v4 as v4
    first, second = _inputs(1536, 1), _inputs(1536, 5)
    want = [float(v4.anchor_attn(*x, block_size=32)[1]) for x in (first, second)]
    assert want[0] != want[1]
    a = torch.randn(8192, 8192, device="cuda").bfloat16()
    b = torch.empty_like(a)

    def interrupted(*args):
        raise KeyboardInterrupt
    for _ in range(3):
        for _ in range(40):  # (keeps the stream busy until the second call waits)
            torch.mm(a, a, out=b)
        with monkeypatch.context() as m:
            m.setattr(v4, "_log_ratio", interrupted)
            with pytest.raises(KeyboardInterrupt):
                v4.anchor_attn(*first, block_size=32)
        assert float(v4.anchor_attn(*second, block_size=32)[1]) == want[1]
        assert _logged(log_file)[-1] == str(want[1])
    with pytest.raises(Exception, match="workspace|unsupported|head"):
        v4.anchor_attn(*[x[..., :32].contiguous() for x in first], block_size=32)  # (refused before any launch)
    torch.cuda.synchronize()
    with pytest.raises(Exception):
        v4.anchor_attn(*[x[..., :32].contiguous() for x in first], block_size=32)
    assert len(v4._left_words) <= 1  # (what is done is given back)
    v4.anchor_attn(*first, block_size=32)
    assert _logged(log_file)[-1] == str(want[0])


@pytest.mark.parametrize("raises", [False, True])
def test_a_logger_in_the_place_of_the_own_one_gets_the_line(monkeypatch, log_file, raises):
    import my_utils
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn
    lines = []

    class Other:
        enabled = True

        @staticmethod
        def log(message):
            lines.append(message)
            if raises:
                raise RuntimeError("no room")
    monkeypatch.setattr(my_utils, "Logger", Other)
    q, k, v = _inputs(1536, 3)
    if raises:
        with pytest.raises(RuntimeError, match="no room"):
            anchor_attn(q, k, v, block_size=32)
    else:
        lines.append(f"anchor sparse_ratio:{float(anchor_attn(q, k, v, block_size=32)[1])}")
        assert lines[0] == lines[1]
    assert isinstance(lines[0], str) and lines[0].startswith("anchor sparse_ratio:0.")
