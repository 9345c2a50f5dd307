"""The native word tokenizer (csrc/runtime/word_tokenizer.h) against the Python one, text by text: hashes, white space, characters past
ASCII, truncation, words longer than a block of the hash, batches that fill and do not fill its lanes."""
import random

import pytest
import torch

from distributed_llm_amd.models import minilm

pytestmark = pytest.mark.skipif(minilm._runtime is None, reason="native runtime not built")
TOK = minilm._HashWordTokenizer(30522)


def _same(texts, max_len=256):
    got, want = TOK.pack(texts, max_len), minilm._pack([TOK.encode(t, max_len) for t in texts])
    assert torch.equal(got[0], want[0]) and got[1:] == want[1:]


@pytest.mark.parametrize("n", [1, 7, 8, 9, 40])
def test_any_text(n):
    r = random.Random(n)
    near = "abcXYZ019 .,?!-_\t\n\x0b\x0c\r\x1b\x1c\x1f\x00\x7f'"
    far = near + "éßİ \u0085中ſK"
    for _ in range(60):
        _same(["".join(r.choice(near if r.random() < 0.8 else far) for _ in range(r.choice([0, 1, 5, 40, 400]))) for _ in range(n)],
              r.choice([2, 3, 10, 256]))


@pytest.mark.parametrize("n", [1, 127, 128, 129, 255, 256, 257, 1000])
def test_long_words(n):
    _same(["a" * n, "b " + "Q7" * n + "?", "x"])


def test_short_limits_and_other_types():
    _same(["one two", ""], 1)
    with pytest.raises(AttributeError):
        TOK.pack([None], 256)
