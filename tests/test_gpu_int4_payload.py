"""Packed INT4 buckets: the code words are produced in their place in the payload, also where the 8-byte shape records in
front of them leave that place off a 16-byte boundary."""

from argparse import Namespace

import pytest
import torch

from miles_amd import _lib

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("group", [32, 128])
def test_int4_codes_are_written_in_place(symmetric, group):
    from miles_amd.weight_update.updater import WeightUpdater
    from oracle import mq_oracle as oracle

    hidden, ffn, experts = 384, 136, 5          # ffn x hidden / group scales: 2-byte sizes that are no multiple of 16
    if group == 128:
        ffn = 256
    args = Namespace(hidden_size=hidden, num_attention_heads=4, num_query_groups=2, kv_channels=128, vocab_size=64, num_layers=1,
                     update_weight_buffer_size=1 << 20, q_lora_rank=None)
    cfg = {"quant_method": "compressed-tensors", "format": "pack-quantized", "config_groups": {"group_0": {"weights": {
        "group_size": group, "symmetric": symmetric, "num_bits": 4, "type": "int"}}}}
    g = torch.Generator().manual_seed(group)
    host = {}
    for e in range(experts):        # gate and up only: their codes have any number of rows
        host[f"module.module.decoder.layers.0.mlp.experts.linear_fc1.weight{e}"] = (torch.randn(2 * ffn, hidden, generator=g) * 0.02).bfloat16()
    names = {f"model.layers.0.mlp.experts.{e}.{p}_proj" for e in range(experts) for p in ("gate", "up")}
    dev = {k: v.to(DEV) for k, v in host.items()}
    got = []
    upd = WeightUpdater(args, weights_getter=lambda: dev, model_name="kimi_k2", quantization_config=cfg, send_bucket=got.append,
                        packed_weight_basenames=names, packed_buckets=True)
    for rep in range(2):            # recorded, then replayed into overwritten payloads
        got.clear()
        upd.update_weights()
        torch.cuda.synchronize()
        places = set()
        for bucket in got:
            for meta, (name, t) in zip(bucket.get_metadata(), bucket):
                expert, kind = int(name.split(".")[5]), name.split(".")[6]
                w = host[f"module.module.decoder.layers.0.mlp.experts.linear_fc1.weight{expert}"].chunk(2)[kind == "up_proj"].contiguous()
                packed, scale, zero = oracle.pack_layer(w, group, symmetric)
                want = {"weight_packed": packed, "weight_scale": scale, "weight_zero_point": zero,
                        "weight_shape": torch.tensor(w.shape, dtype=torch.int32)}[name.split(".")[-1]]
                assert torch.equal(t.cpu().contiguous().view(torch.uint8), want.contiguous().view(torch.uint8)), f"{name}, sync {rep}"
                if name.endswith("weight_packed"):
                    places.add(meta.start_idx % 16)
            bucket.flat.fill_(0x5A)
        assert places - {0}, "the shapes of this test put some codes off a 16-byte boundary"
    records = upd._plan.batch.records
    assert {r[8] for r in records if r[0] == _lib.JOB_COPY} == {8}, "only the shape records are copied in"
