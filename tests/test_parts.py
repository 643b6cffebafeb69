"""Parts without a GPU: how they hand work to each other."""
from types import SimpleNamespace

import pytest
import torch

from infinilm_amd import kernels
from infinilm_amd.config.spec import PartSpec
from infinilm_amd.parts.attention import GQAttention
from infinilm_amd.parts.base import BuildContext, ResidualStream
from infinilm_amd.parts.norm import RMSNorm
from infinilm_amd.parts.rotary import NoPositionEncoding, RotaryEmbedding

CTX = BuildContext(torch.bfloat16, torch.device("cpu"))


class OwnNorm(RMSNorm):
    def forward(self, stream, frag=False):
        return super().forward(stream, frag) * 2


class OwnAttention(GQAttention):
    def forward(self, x, batch, cache_view, tail=None):
        return super().forward(x * 2, batch, cache_view, tail)


class OwnEncoding(RotaryEmbedding):
    def project_encode_store(self, x, proj, batch, view, nh, nkv, d):
        return super().project_encode_store(x * 2, proj, batch, view, nh, nkv, d)


@pytest.mark.parametrize("norm,mixer,encoding,taken", [(RMSNorm, GQAttention, RotaryEmbedding, True), (OwnNorm, GQAttention, RotaryEmbedding, False),
                                                       (RMSNorm, OwnAttention, RotaryEmbedding, False), (RMSNorm, GQAttention, OwnEncoding, False),
                                                       (RMSNorm, GQAttention, NoPositionEncoding, False)])
def test_rows_formed_by_the_projection_pass_no_override_by(monkeypatch, norm, mixer, encoding, taken):
    """A norm, a mixer or an encoding made from those that hand the norm's rows to the projection, with a method of its own where the
    rows would go through: the method is called, as at any number of rows."""
    n = norm(64, 1e-6, CTX)
    m = mixer(64, 2, 1, 32, False, False, 1.0, 0, PartSpec("rotary", {"head_dim": 32, "rotary_dim": 32, "max_positions": 8, "theta": 1e4, "scaling": None}), CTX)
    m.position = RotaryEmbedding(32, 32, 8, 1e4, None, CTX) if encoding is RotaryEmbedding else encoding(CTX) if encoding is NoPositionEncoding \
        else encoding(32, 32, 8, 1e4, None, CTX)
    monkeypatch.setattr(m.position, "check", lambda batch: None)
    q, new = torch.zeros(1, 64), torch.ones(1, 64)
    monkeypatch.setattr(kernels, "qkv_rope_sum", lambda *a: (q, new))
    stream = ResidualStream(torch.zeros(1, 64))
    stream.push(torch.zeros(2, 1, 64), 1.0)
    pending = n.pending(stream)
    got = None if pending is None else m.project_pending(pending, SimpleNamespace(positions=None), SimpleNamespace(k=None, v=None, slots=None))
    assert (got is q) == taken and (stream.residual is new) == taken and (stream.pending is None) == taken
