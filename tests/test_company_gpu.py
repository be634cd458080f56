"""What a request is answered on the GPU does not depend on which others are served beside it: to the bit, at the width whose
products take tiles of several sizes by the rows there are."""

import dataclasses

import numpy as np
import pytest
import torch

import bench
from iron_amd.applications import pegilix, pudinex, pufuzen, tilarax
from iron_amd.lm import Sampler
from iron_amd.lm.batched import Entry

pytestmark = pytest.mark.gpu

FAMILIES = {"pegilix": (bench.pegilix_config, pegilix.Pegilix, pegilix.shapes), "pufuzen": (bench.pufuzen_config, pufuzen.Pufuzen, pufuzen.shapes),
            "tilarax": (bench.tilarax_config, tilarax.Tilarax, tilarax.shapes), "pudinex": (bench.pudinex_config, pudinex.Pudinex, pudinex.shapes)}


@pytest.mark.parametrize("name", FAMILIES)
def test_a_request_is_answered_the_same_in_any_company(cuda, name):
    make, family, shapes = FAMILIES[name]
    config = make(2048, slots=4, chunk=1024)
    config = dataclasses.replace(config, layers=config.layers[:4], vocab_size=2048)
    weights = bench.random_weights(torch, shapes(config), cuda)
    for n, w in weights.items():
        if n.endswith("lower"):   # a fading memory's least share, below one
            w.mul_(0.5)
    model = family(config, weights)
    model.load_versions()
    try:
        # (rows on both sides of each line between two tiles, alone and together; a prompt longer than a portion)
        rng = np.random.default_rng(1)
        prompts = [rng.integers(0, config.vocab_size, n).tolist() for n in (96, 301, 17, 520)]
        logits = []
        for p in prompts:
            logits.append(model.batch.step([Entry("alone", p, [0, len(p) - 1])])[0])
            model.batch.end("alone")
        assert all(np.isfinite(rows).all() for rows in logits)
        for order in ((0, 1, 2, 3), (3, 2, 1, 0), (1, 2)):
            got = model.batch.step([Entry(i, prompts[i], [0, len(prompts[i]) - 1]) for i in order])
            for i, rows in zip(order, got):
                assert np.array_equal(rows, logits[i]), (order, i)
                model.batch.end(i)
        prompts.append(rng.integers(0, config.vocab_size, 1100).tolist())
        alone = [model.generate(p, 12) for p in prompts]
        assert model.generate_batch(prompts, 12) == alone
        assert model.generate_batch(prompts[::-1], 12) == alone[::-1]
        draws = [Sampler(0.9, 40, seed=i) for i in range(5)]
        drawn = model.generate_batch(prompts, 12, draws)
        assert drawn == [model.generate(p, 12, Sampler(0.9, 40, seed=i)) for i, p in enumerate(prompts)]
    finally:
        model.release()
