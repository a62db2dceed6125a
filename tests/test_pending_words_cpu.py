"""The completion words of calls that are waited for later."""

import threading

import pytest
import torch

from fast_compressai.coders import gaans


# words made in one mode are handed to a call in the other
@pytest.mark.parametrize("first,then", [(True, False), (False, True), (True, True)])
def test_words_serve_calls_in_and_out_of_inference_mode(monkeypatch, first, then):
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory, **k: empty(*a, **k))  # no GPU here
    st = gaans._StreamState.__new__(gaans._StreamState)
    st.slots, st.lock = [], threading.Lock()
    with torch.inference_mode(first):
        words = st.slot()
    words.view[:] = 7  # as a kernel leaves them
    st.give_back(words)
    with torch.inference_mode(then):
        again = st.slot()
        assert again is words and again.tensor.tolist() == [0, 0, 0, 0]
