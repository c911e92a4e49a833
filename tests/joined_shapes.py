"""Vepelix and Pukatar configurations whose shared experts have the experts' sizes and bounds, at sizes that rows in bf16 and the wide tiles take."""
from tests import pukatar_shapes as P, vepelix_shapes as V

SHAPES = {
    "vepelix": {"architecture": "Vepelix", "vocab": 96, "width": 128, "norm": {"eps": 1e-6}, "loop": {"start": 1, "stop": 2, "times": 2},
                "layers": [V.layer(V.parallel(4, 2, 32, 32, V.rotation(1000.0, 16), 40, 2, 64, 32, 6.0, (1.0, 0.8)), V.moe(4, 2, 64, 64)),
                           V.layer(V.latent(4, 16, 16, 16, 32, 24), V.moe(7, 3, 128, 128)),
                           V.layer(V.latent(2, 32, 8, 32, 24, 16), V.dense(192, 1.0)),
                           V.layer(V.latent(2, 16, 8, 16, 16, 8), V.moe(5, 1, 64, 96))],      # (one that stays outside, between its neighbours' buffers)
                "ranks": {0: 16}},
    "pukatar": {"architecture": "Pukatar", "vocab": 96, "width": 128, "norm": {"eps": 1e-6}, "loop": {"start": 1, "stop": 2, "times": 2},
                "layers": [P.layer(P.delta(4, 2, 32, 32, 4), P.moe(4, 2, 64, 1.1, (64, 1.1))),
                           P.layer(P.attn(4, 2, 32, 32, (1000.0, 16), (40, 3)), P.moe(7, 3, 128, 0.9, (128, 0.9))),
                           P.layer(P.attn(2, 2, 16, 32), P.dense(192)),
                           P.layer(P.delta(2, 1, 64, 32, 3), P.moe(5, 1, 64, 0.8, (64, 1.4)))],
                "ranks": {0: (16, 8), 3: (8, 24)}},
}


def use(monkeypatch, design):
    """Puts the configuration among the design's own under the name "joined"."""
    monkeypatch.setitem((V if design == "vepelix" else P).SHAPES, "joined", SHAPES[design])
