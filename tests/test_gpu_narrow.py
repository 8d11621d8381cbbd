"""The narrow chunked prefill (16 state rows per workgroup, taken where the
launch leaves CUs idle) against the wide one (32 rows): the same sequence run
alone and as part of a batch too large for the narrow form.  Both form the
same numbers from the same operands, so outputs and final states are equal
bit for bit; the wide form and the narrow one are also held to the f64 oracle
by the other prefill tests."""
import pytest
import torch

import rhizome_amd

pytestmark = pytest.mark.gpu
H = 2


def _batch(n, T, dk, dv, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=gen, device="cuda")

    q, k = normal(n, T, H, dk), normal(n, T, H, dk)
    q, k = q / q.norm(dim=-1, keepdim=True) * dk ** 0.5, k / k.norm(dim=-1, keepdim=True)
    g = -torch.nn.functional.softplus(normal(n, T, H) - 2.0)
    return dict(q=q.bfloat16(), k=k.bfloat16(), v=normal(n, T, H, dv).bfloat16(), g=g,
                beta=torch.sigmoid(normal(n, T, H)), initial_state=normal(n, H, dv, dk))


def _check(b, reruns=0):
    n, T, _, dk = b["q"].shape
    dv = b["v"].shape[-1]
    assert H * ((dv + 15) // 16) <= 256 < n * H * ((dv + 15) // 16)  # one sequence narrow, the batch wide
    rhizome_amd.exact_reruns()
    o, fin = rhizome_amd.prefill(**{x: t[:1].contiguous() for x, t in b.items()})
    assert rhizome_amd.exact_reruns() == reruns
    wo, wfin = rhizome_amd.prefill(**b)
    assert rhizome_amd.exact_reruns() == reruns
    assert torch.equal(o[0], wo[0]) and torch.equal(fin[0], wfin[0])
    lengths = torch.tensor([0, T, T], dtype=torch.int32, device="cuda")  # packed, an empty sequence after it
    po, pfin = rhizome_amd.prefill(*(b[x][0] for x in ("q", "k", "v", "g", "beta")), cu_seqlens=lengths,
                                   initial_state=b["initial_state"][:2].contiguous())
    assert torch.equal(po, o[0]) and torch.equal(pfin[0], fin[0])
    assert torch.equal(pfin[1], b["initial_state"][1])
    rhizome_amd.exact_reruns()
    assert rhizome_amd.sync_timeouts() == 0


@pytest.mark.parametrize("T", [1, 63, 64, 65, 129, 320])
@pytest.mark.parametrize("dk,dv", [(8, 8), (32, 16), (64, 24), (64, 64), (128, 40), (128, 128)])
def test_equals_wide(T, dk, dv):
    _check(_batch(140 if dv <= 16 else 70, T, dk, dv, seed=T + dk + dv))


@pytest.mark.parametrize("dv", [16, 48])
def test_reset_inside_a_chunk(dv):
    b = _batch(140, 150, 128, dv, seed=dv)
    b["g"][:, 70] = float("-inf")
    b["g"][:, 90, 1] = -100.0
    _check(b)


@pytest.mark.parametrize("dv", [8, 40])
def test_exact_rerun(dv):
    """A key outside the fp16 path's domain: the tiles of its head rerun, counted per 32 rows."""
    b = _batch(140, 100, 64, dv, seed=dv)
    b["k"][0, 50, 1] *= 4
    _check(b, reruns=(dv + 31) // 32)
