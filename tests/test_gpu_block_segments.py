"""Segments of a packed block, found on the device once for all layers, against counting them on the host."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _block(template, lens, first_id=1):
    ids = [-2] * template
    for i, n in enumerate(lens):
        ids += [first_id + i] * n
    return torch.tensor([ids], dtype=torch.int64, device="cuda")


@pytest.mark.parametrize("template,lens", [(3, [1]), (0, [5, 1, 7]), (2, []), (1, [1023, 1]), (3, [64] * 31), (3, [1, 2] * 3000), (0, [40000, 1, 3]),
                                           (1024, [1, 1024, 2048]), (7, [1] * 4094), (6, [1] * 4096), (3, [65536, 1, 63, 70000, 2])])
def test_segments(template, lens):
    from msa_amd import ops
    print(f"[case] segments {template} + {len(lens)}", flush=True)
    ids = _block(template, lens)
    g = torch.Generator(device="cuda").manual_seed(len(lens))
    mask = torch.randint(0, 3, ids.shape, generator=g, device="cuda")
    pos = torch.randint(0, 1 << 40, ids.shape, generator=g, device="cuda") if template % 2 else torch.randint(0, 9000, ids.shape, generator=g, device="cuda")
    b = ops.BlockSegments(ids, mask, pos).read()
    seg = ([template] if template else []) + lens
    assert b.n_template == template and b.doc_lens == lens and b.lens == seg and not b.bad
    assert b.mask_sum == int(mask.sum()) and b.last_position == min(int(pos.max()), (1 << 31) - 1)
    cu = torch.tensor([0] + seg).cumsum(0)
    assert b.cu.dtype == torch.int32 and b.cu.tolist() == cu.tolist() and b.start.tolist() == cu[:-1].tolist() and b.len.tolist() == seg
    if lens:
        t, want = b.table(16), ops.chunk_table(lens, 16, first_token=template)
        for name in ("doc_start", "doc_chunk_off", "chunk_start", "chunk_len", "chunk_doc", "n_chunks"):
            assert torch.equal(getattr(t, name), getattr(want, name)), name
        assert b.table(16) is t


@pytest.mark.parametrize("ids", [[-2, -2, 1, 1, 0, 2], [1, 1, -2, 2], [-2, 3, -1]])
def test_ids_that_are_no_document(ids):
    from msa_amd import ops
    assert ops.BlockSegments(torch.tensor([ids], device="cuda"), None, None).read().bad


def _model():
    from msa_amd.config import MSAConfig
    from msa_amd.model import MSAForCausalLM
    torch.manual_seed(3)
    cfg = MSAConfig(num_hidden_layers=3, hidden_size=256, intermediate_size=512, vocab_size=500, num_attention_heads=4, num_key_value_heads=2,
                    max_position_embeddings=700)
    cfg.msa_config.router_layer_idx = "1,2"
    return MSAForCausalLM(cfg).init_random(0.05).cuda().bfloat16().eval()


def test_encoding_is_what_each_layer_by_itself_makes_of_it(monkeypatch):
    from msa_amd.model import MSAModel, encode_block
    from msa_amd.prefill import Document, prepare_block_inputs
    model = _model()
    docs = [Document(doc_id=i, input_ids=[(7 * i + j) % 500 for j in range(n)]) for i, n in enumerate((130, 64, 1, 333))]
    block = prepare_block_inputs(docs, [1, 2, 3], model.config.msa_config.pooling_kernel_size)
    a = encode_block(model, block, "cuda")
    assert "block_segments" not in a.meta and a.meta["q_lens_host"] == [531]
    monkeypatch.setattr(MSAModel, "_block_segments", lambda self, *args: None)
    b = encode_block(model, block, "cuda")
    assert b.meta["q_lens_host"] == [531]
    for i in (1, 2):
        assert torch.equal(a.key_cache[i], b.key_cache[i]) and torch.equal(a.value_cache[i], b.value_cache[i])
        assert torch.equal(a.router_key_cache[i], b.router_key_cache[i])
        assert torch.equal(a.cache_kwargs[i]["pooled_doc_ids"], b.cache_kwargs[i]["pooled_doc_ids"])
    for i in range(3):
        assert torch.equal(a.cache_kwargs[i]["template_prefix_kcache"], b.cache_kwargs[i]["template_prefix_kcache"])


@pytest.mark.parametrize("wrong", ["mask", "ids", "position"])
def test_blocks_that_are_refused(wrong):
    from msa_amd.model import encode_block
    from msa_amd.prefill import Document, prepare_block_inputs
    model = _model()
    block = prepare_block_inputs([Document(doc_id=1, input_ids=list(range(100)))], [1, 2, 3], model.config.msa_config.pooling_kernel_size)
    if wrong == "mask":
        block.doc_attention_mask[0, 5] = 0
    elif wrong == "ids":
        block.doc_ids[0, 50] = 0
    else:
        block.position_ids[0, 7] = 700
    with pytest.raises(ValueError, match="position 700 is beyond" if wrong == "position" else "stage 1 expects"):
        encode_block(model, block, "cuda")
