"""The native byte-level BPE against the Python one that defines it."""

from __future__ import annotations

import copy
import json
import pickle
import random
import time

import pytest

from quickstart_streaming_agents_amd.models import tokenizer
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


@pytest.mark.parametrize("n", [47, 48, 49, 64, 65, 200, 900])
def test_long_words(n):
    """Above some 48 bytes pairs are merged from a heap, in the same order."""
    for vocab in (300, 1024, 30_522):
        tok, r = BpeTokenizer(vocab), random.Random(n)
        for letters in ("ab", "aeinorst", "abcdefghijklmnopqrstuvwxyz"):
            for size in (n, n + r.randint(1, 40)):
                word = "".join(r.choices(letters, k=size))
                want = tok._encode(word, True)
                assert tok.encode(word) == want
                assert tok.encode(word) == want           # and as it is kept
        word = "streaming" * (n // 9 + 1)
        assert tok.encode(word + " " + word) == tok._encode(
            word + " " + word, True)


def test_long_words_take_no_square_of_their_length():
    """20,000 letters were 1.2 s each time; now once some 10 ms."""
    tok, r = BpeTokenizer(30_522), random.Random(1)
    word = "".join(r.choices("abcdefghijklmnopqrstuvwxyz", k=20_000))
    t = time.perf_counter()
    for _ in range(50):
        ids = tok.encode(word)
    assert time.perf_counter() - t < 5
    assert tok.decode(ids) == word


def test_a_batch_reads_no_further_than_it_keeps():
    tok = BpeTokenizer(30_522)
    text = "one window " * 50_000 + "<|finish|>"
    t = time.perf_counter()
    for _ in range(200):
        ids, lens = tok.encode_batch([text, "a<|finish|>b"], 3)
    assert time.perf_counter() - t < 5
    assert ids.tolist() == tok._encode(text[:100], True)[:3] + \
        tok._encode("a<|finish|>b", True)[:3] and lens.tolist() == [3, 3]
    with pytest.raises(UnicodeEncodeError):
        tok.encode_batch([text + "\ud800"], 3)


@pytest.mark.parametrize("specials", [{}, {"": 3}, {"<|eot|>": 2}])
def test_vocabularies_of_other_specials(specials, tmp_path):
    with open(tokenizer._VOCAB_PATH) as f:
        vocab = dict(json.load(f), specials=specials)
    path = tmp_path / "vocab.json"
    path.write_text(json.dumps(vocab))
    tok = BpeTokenizer(1024, str(path))
    for text in ("one window<|eot|> of 12", "", "a"):
        assert tok.encode(text) == tok._encode(text, True)
        ids, _ = tok.encode_batch([text], 99)
        assert ids.tolist() == tok._encode(text, True)
