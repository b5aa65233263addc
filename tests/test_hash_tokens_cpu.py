"""The native rows of token ids (csrc/runtime/hash_tokens.cpp) are the ones that the Python tokenizer finds."""
import random

import pytest

from shai_amd import native
from shai_amd.tokenizers import HashTokenizer

TEXTS = ["", " ", "a", "A photo, of a_cat!", "x" * 300, "\x1c\x1fa\x00b\x7f\t\n", "don't -- stop", "café au lait", "你好 world",
         "50%  off now", "end."]


def _texts(seed, ascii_only):
    rng = random.Random(seed)
    alphabet = "abzAZ019_ \t\n\x0b\x1d.,!'-" + ("" if ascii_only else "éİ 你")
    return ["".join(rng.choice(alphabet) for _ in range(rng.randint(0, 60))) for _ in range(rng.randint(1, 9))]


@pytest.mark.skipif(not native.runtime_available(), reason="runtime library is not built")
@pytest.mark.parametrize("bos,eos", [(None, None), (None, 1), (49406, 49407), (300, None)])
@pytest.mark.parametrize("length", [1, 2, 7, 77])
@pytest.mark.parametrize("padding", ["max_length", "longest"])
def test_rows(bos, eos, length, padding, monkeypatch):
    tok = HashTokenizer(49408, bos, eos, 0, 77)
    batches = [TEXTS] + [[t] for t in TEXTS] + [_texts(s, s % 3 > 0) for s in range(40)]
    got = [tok(b, max_length=length, padding=padding) for b in batches]
    monkeypatch.setattr(HashTokenizer, "_native", lambda *a: None)
    for b, g in zip(batches, got):
        want = tok(b, max_length=length, padding=padding)
        for name in ("input_ids", "attention_mask"):
            assert g[name].dtype == want[name].dtype and g[name].shape == want[name].shape and bool((g[name] == want[name]).all()), (b, name)


# whatever is iterated over once, as before
def test_any_iterable():
    tok = HashTokenizer(1000, None, 1, 0, 16)
    want = tok(["a b", "c"])["input_ids"]
    assert bool((tok(t for t in ("a b", "c"))["input_ids"] == want).all()) and bool((tok(("a b", "c"))["input_ids"] == want).all())


# a word whose id is the first token's stays the row's beginning; special strings and rows that may not be cut go the Python way
def test_first_token_and_specials():
    probe = HashTokenizer(1000, None, None, 0, 16)
    bos = probe.encode("hello")[0]
    tok = HashTokenizer(1000, bos, None, 0, 16)
    assert tok(["hello you"])["attention_mask"].sum().item() == 2 and tok(["you"])["attention_mask"].sum().item() == 2
    special = HashTokenizer(1000, None, None, 0, 16, specials={"<|image|>": 999})
    assert special(["a <|image|>"])["input_ids"][0, :2].tolist() == [probe.encode("a")[0], 999]
    with pytest.raises(RuntimeError):
        probe(["a " * 20], max_length=4, truncation=False)


# ids that are made another way, by a derived class or on the object, are those of the batch too
@pytest.mark.parametrize("name", ["encode", "_words", "_tok"])
def test_other_ids(name):
    class Other(HashTokenizer):
        pass
    other = {"encode": lambda self, text, add_special_tokens=True: [7, 7], "_words": lambda self, text: [7, 7], "_tok": lambda self, w: 7}[name]
    setattr(Other, name, other)
    tok, own = Other(1000, None, None, 0, 4), HashTokenizer(1000, None, None, 0, 4)
    setattr(own, name, other.__get__(own))
    assert tok(["a b"])["input_ids"].tolist() == own(["a b"])["input_ids"].tolist() == [[7, 7, 0, 0]]
