"""HF (multi-byte BPE) tokenizer support: byte-exact token_bytes mapping
and token-level format="json" enforcement over the byte automaton
(engine/constraints.py::mask_logits_token_level) (not for
the byte tokenizer alone)."""

import json

import pytest
import torch

from gridllm_amd.engine.constraints import (JsonByteConstraint,
                                            mask_logits_token_level)


@pytest.fixture(scope="module")
def hf_tok(tmp_path_factory):
    from tokenizers import (Tokenizer, decoders, models, pre_tokenizers,
                            trainers)
    tok = Tokenizer(models.BPE())
    tok.pre_tokenizer = pre_tokenizers.ByteLevel(add_prefix_space=False)
    tok.decoder = decoders.ByteLevel()
    tr = trainers.BpeTrainer(
        vocab_size=400, special_tokens=["<|end_of_text|>"],
        initial_alphabet=pre_tokenizers.ByteLevel.alphabet())
    tok.train_from_iterator(
        ['{"a": 1, "b": [true, false, null], "c": "hi"}',
         'hello world {"nested": {"x": 2.5e3}}'] * 20, tr)
    path = str(tmp_path_factory.mktemp("tok") / "tokenizer.json")
    tok.save(path)
    from gridllm_amd.engine.tokenizer import HFTokenizer
    return HFTokenizer(path)


def test_token_bytes_roundtrip(hf_tok):
    for txt in ['{"key": [1, true, "vé"]}', "hello wörld",
                '{"a": -1.5e-3, "b": "\\n"}']:
        ids = hf_tok.encode(txt)
        bs = b"".join(hf_tok.token_bytes(i) or b"" for i in ids)
        assert bs == txt.encode("utf-8"), txt


def test_byte_fallback_covers_json_alphabet(hf_tok):
    for b in b'{}[]",: 0123456789.-+eEtrufalsn':
        assert hf_tok.byte_token_id(b) is not None, chr(b)


def test_special_token_not_representable(hf_tok):
    assert hf_tok.token_bytes(hf_tok.eos_id) in (None, b"")


def test_token_level_json_enforcement(hf_tok):
    """Greedy decode over RANDOM logits with the token-level mask must
    produce a complete JSON document once EOS is chosen."""
    v = hf_tok.vocab_size
    g = torch.Generator().manual_seed(6)
    for trial in range(5):
        c = JsonByteConstraint()
        out = b""
        for _ in range(400):
            logits = torch.randn(v, generator=g)
            mask_logits_token_level(logits, c, hf_tok, hf_tok.eos_id)
            tok = int(logits.argmax())
            if tok == hf_tok.eos_id:
                break
            bs = hf_tok.token_bytes(tok)
            assert bs, tok                       # masked tokens never win
            for by in bs:                        # byte-wise: the automaton
                assert by in c.allowed()[0], \
                    (bs, out[-40:])              # advances WITHIN a token
                c.push(by)
            out += bs
        else:
            pytest.fail(f"no EOS within 400 steps: {out[:80]!r}")
        # string contents may carry automaton-legal non-UTF8 bytes (same
        # property as the byte tokenizer) — decode like the engine does
        json.loads(out.decode("utf-8", errors="replace"))


def test_engine_with_hf_tokenizer_enforces_json(hf_tok):
    """End-to-end: an engine whose tokenizer is the HF one produces valid
    JSON under format=json (or ends by length). The tiny spec's vocab
    (512) exceeds the HF vocab — the mask skips unmappable ids."""
    from gridllm_amd.config import EngineConfig
    from gridllm_amd.engine import InferenceEngine
    from gridllm_amd.models.registry import get_spec
    spec = get_spec("tiny")
    if spec.vocab < hf_tok.vocab_size:
        pytest.skip("tiny vocab smaller than HF tokenizer")
    eng = InferenceEngine(EngineConfig(
        model="tiny", device="cpu", dtype="fp32", max_seq_len=128,
        max_batch_size=2, use_hipgraph=False, seed=3))
    eng.tokenizer = hf_tok
    res = eng.generate("make json", {"temperature": 1.0, "seed": 11,
                                     "format": "json", "num_predict": 80})
    if res.done_reason != "length":
        json.loads(res.text.encode("utf-8", errors="replace")
                   .decode("utf-8", errors="replace"))


def test_hf_stream_decoder_matches_full_decode(hf_tok):
    """Span-wise streaming decode (O(tail) per token, not O(history))
    reassembles exactly the full decode for byte-level BPE — including
    code points split across tokens."""
    for txt in ['{"key": "vérité ✓"}', "héllo wörld ünïcode",
                "plain ascii text here", "日本語 mixed ascii"]:
        ids = hf_tok.encode(txt)
        dec = hf_tok.decode_stream()
        out = []
        for i in ids:
            out.append(dec.push(i))
        out.append(dec.flush())
        assert "".join(out) == hf_tok.decode(ids), txt


def test_engine_hf_tokenizer_with_schema(hf_tok):
    """Schema constraint through the token-level mask path."""
    from gridllm_amd.config import EngineConfig
    from gridllm_amd.engine import InferenceEngine
    from gridllm_amd.models.registry import get_spec
    if get_spec("tiny").vocab < hf_tok.vocab_size:
        pytest.skip("tiny vocab smaller than HF tokenizer")
    eng = InferenceEngine(EngineConfig(
        model="tiny", device="cpu", dtype="fp32", max_seq_len=256,
        max_batch_size=2, use_hipgraph=False, seed=3))
    eng.tokenizer = hf_tok
    schema = {"type": "object",
              "properties": {"mode": {"enum": ["a", "b"]}},
              "required": ["mode"], "additionalProperties": False}
    res = eng.generate("x", {"temperature": 1.0, "seed": 9,
                             "format": schema, "num_predict": 60})
    if res.done_reason != "length":
        assert json.loads(res.text) in ({"mode": "a"}, {"mode": "b"})


def test_hf_stream_decoder_bounded_holdback(hf_tok):
    """A token stream whose decode ALWAYS ends mid-codepoint (possible
    with random/adversarial byte-fragment tokens) must not silence the
    stream for the whole generation: the decoder emits (with replacement
    chars) after at most MAX_HOLD held tokens."""
    from gridllm_amd.engine.tokenizer import HFStreamDecoder
    # find a token whose bytes END with a dangling UTF-8 lead byte
    frag = None
    for i in range(hf_tok.vocab_size):
        bs = hf_tok.token_bytes(i)
        if bs and hf_tok._tok.decode([i]).endswith("�"):
            frag = i
            break
    if frag is None:
        pytest.skip("no dangling-lead token in this vocab")
    dec = hf_tok.decode_stream()
    emitted, max_gap, gap = [], 0, 0
    for _ in range(100):
        piece = dec.push(frag)
        gap = gap + 1 if not piece else 0
        max_gap = max(max_gap, gap)
        emitted.append(piece)
    assert any(emitted), "stream stayed silent for 100 tokens"
    assert max_gap < HFStreamDecoder.MAX_HOLD + 1
