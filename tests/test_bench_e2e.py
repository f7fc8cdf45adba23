"""bench.py's end-to-end section: "tokens_identical" is true only where every
pair of token streams was compared."""
import json
import sys

import pytest

from conftest import load

bench = load("bench.py", "bench")


def program(path, tokens):
    """An executable that prints what the end-to-end programs print last."""
    line = json.dumps({"tokens": tokens, "decode_tok_s": 1.0, "prefetch_misses": 0})
    path.write_text(f"#!{sys.executable}\nprint({line!r})\n")
    path.chmod(0o755)
    return str(path)


@pytest.mark.parametrize("gpu,cpu,want", [(None, None, None), ([1, 2], None, None), (None, [1, 2], None),
                                          ([1, 2], [1, 2], True), ([1, 3], [1, 2], False)])
def test_tokens_identical(tmp_path, monkeypatch, gpu, cpu, want):
    for name, tokens in (("E2E_GPU", gpu), ("E2E_CPU", cpu)):
        path = tmp_path / name
        monkeypatch.setattr(bench, name, str(path) if tokens is None else program(path, tokens))
    out = bench.e2e(prompt=1, gen=1)
    assert out["tokens_identical"] is want
    assert ("not built" in out.values()) == (gpu is None or cpu is None)
