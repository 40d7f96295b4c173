"""A request's float32 logits do not depend on the requests beside it."""

import pytest
import torch

pytestmark = pytest.mark.gpu

CONFIG = {
    "architectures": ["LlamaForCausalLM"], "num_hidden_layers": 3, "hidden_size": 256, "num_attention_heads": 4, "num_key_value_heads": 2,
    "head_dim": 64, "intermediate_size": 512, "vocab_size": 512, "rope_theta": 10000.0, "rms_norm_eps": 1e-5, "tie_word_embeddings": False,
    "max_position_embeddings": 512,
}


def test_decoding_alone_and_beside_others_gives_the_same_bits():
    """1 to 9 requests: through the kernels of up to 4, up to 8 and more rows."""
    from mini_infer_amd import ModelRunner, StepEntry
    from mini_infer_amd.models import architecture_for

    arch = architecture_for(CONFIG)
    parsed = arch.parse_config(CONFIG)
    model = arch.make_model(parsed, torch.float32, "cuda:0")
    generator = torch.Generator(device="cuda").manual_seed(0)
    specs = model.param_specs()
    model.load_params(lambda name: torch.randn(specs[name].shape, generator=generator, device="cuda") * (1.0 if len(specs[name].shape) == 1 else 0.05))
    tokens = torch.randint(0, 512, (9, 45), generator=torch.Generator().manual_seed(1)).tolist()
    alone = None
    for beside in (1, 2, 4, 5, 8, 9):
        runner = ModelRunner(model, parsed, num_blocks=64, block_size=16, max_concurrent=9)
        for i in range(beside):
            runner.step([StepEntry(i, tokens[i][:40], [])])
        made = [runner.step([StepEntry(i, [tokens[i][40 + step]], [0]) for i in range(beside)])[0].clone() for step in range(3)]
        alone = alone or made
        assert all(torch.equal(a, b) for a, b in zip(alone, made)), beside
