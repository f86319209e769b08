"""The native byte-level BPE against the Python one that defines it."""

from __future__ import annotations

import copy
import pickle
import random

import pytest

from quickstart_streaming_agents_amd.models.tokenizer import BpeTokenizer
from quickstart_streaming_agents_amd.ops import have_ext

pytestmark = pytest.mark.skipif(not have_ext(), reason="extension not built")

PIECES = list("abzAZ059 '\n\t\r.,;!-_$\u00e9\u4e2d\U0001f600\u00a0\u3000\u2003"
              "\x85\x1c\x1f\x0b\x0c\x00\u1680\u200b\ufeff\u2029\u202f\u205f") + [
    "'s", "'re", "'ll", "'m", "'d", "'S", "<|finish|>", "<|tool_1|>", "<|",
    "|>", "  ", "\n ", "the", "window ", "ing", "x" * 70, "streaming"]


@pytest.mark.parametrize("vocab", [272, 300, 1024, 30_522])
def test_same_tokens(vocab):
    tok, r = BpeTokenizer(vocab), random.Random(vocab)
    for _ in range(3000):
        text = "".join(r.choices(PIECES, k=r.randint(0, 14)))
        for bos in (True, False):
            assert tok.encode(text, bos) == tok._encode(text, bos), repr(text)
        assert tok.decode(tok.encode(text)) == tok.decode(
            tok._encode(text, True))


def test_every_character_beside_others():
    """White space is what a str pattern's \\s matches."""
    tok = BpeTokenizer(30_522)
    for i in range(0, 0x110000, 7):
        if not 0xD800 <= i < 0xE000:
            text = f"a {chr(i)}b{chr(i)}  {chr(i)}"
            assert tok.encode(text) == tok._encode(text, True), hex(i)
    for i in list(range(0x3100)) + [0xFEFF, 0xFFFD, 0x10FFFF]:
        text = f"a {chr(i)}b{chr(i)} {chr(i)}"
        assert tok.encode(text) == tok._encode(text, True), hex(i)


def test_batches_and_what_is_refused():
    tok = BpeTokenizer(30_522)
    texts = ["", "one window", None, "claims " * 700, "<|eot|>"]
    ids, lens = tok.encode_batch(texts, 512)
    want = [tok._encode(t, True)[:512] for t in texts]
    assert lens.tolist() == [len(x) for x in want]
    assert ids.tolist() == sum(want, [])
    tok._native, native = None, (ids, lens)
    ids, lens = tok.encode_batch(texts, 512)
    assert (ids == native[0]).all() and (lens == native[1]).all()
    tok = BpeTokenizer(30_522)
    with pytest.raises(UnicodeEncodeError):
        tok.encode("\ud800")


def test_more_words_than_are_kept():
    tok = BpeTokenizer(1024)
    words = [f"w{i}x" for i in range(70_000)]
    tok.encode_batch(words, 99)
    for w in words[::997] + words[-3:]:
        assert tok.encode(w) == tok._encode(w, True)


def test_copies_and_pickles():
    """A tokenizer goes to other processes and is copied like any object."""
    tok = BpeTokenizer(1024)
    for other in (copy.deepcopy(tok), copy.copy(tok),
                  pickle.loads(pickle.dumps(tok))):
        assert other._native is not None
        assert other.encode("a window<|finish|> of 12") == \
            tok.encode("a window<|finish|> of 12")
