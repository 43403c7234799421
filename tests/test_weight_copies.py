"""The working copies of weights (``ops/_prep.py``) follow their source: a weight whose storage was given back and replaced by
another one at the same address is another weight."""

import pytest
import torch

from oracle import svdq_oracle as O


def _replace_at_the_same_address(p: torch.Tensor, fill: torch.Tensor) -> bool:
    """Free ``p``'s storage the way sharding and offloading code does, and give ``p`` the first new tensor of its size that
    gets the block.  ``False`` where the allocator hands the block out elsewhere."""
    address = p.data_ptr()
    p.untyped_storage().resize_(0)
    tried = []
    for _ in range(64):
        other = torch.empty_like(fill)
        if other.data_ptr() == address:
            other.copy_(fill)
            p.data = other
            return True
        tried.append(other)
    return False


def test_a_freed_source_is_not_taken_for_its_successor():
    from nunchaku_rocm_amd.ops import _prep

    handed_out_again = 0
    for elements in [256 << i for i in range(16)]:  # up to 32 MB: small blocks and mapped ones, by the allocator's mood
        p = torch.nn.Parameter(torch.zeros(elements), requires_grad=False)
        src = _prep._source_of(p)
        assert _prep._same_source(src, p)
        if _replace_at_the_same_address(p, torch.ones(elements)):
            handed_out_again += 1
            assert not _prep._same_source(src, p)
    if not handed_out_again:
        pytest.skip("the allocator did not hand any block out again")


def test_what_makes_a_source_another():
    from nunchaku_rocm_amd.ops import _prep

    base = torch.arange(48.0)
    t = base[8:24].view(4, 4)
    src = _prep._source_of(t)
    assert _prep._same_source(src, t) and _prep._same_source(src, base[8:24].view(4, 4))
    assert not _prep._same_source(src, base[9:25].view(4, 4))  # another offset
    assert not _prep._same_source(src, t.t())  # another order
    assert not _prep._same_source(src, base[8:24].view(2, 8))  # another shape
    assert not _prep._same_source(src, base.clone()[8:24].view(4, 4))  # another storage
    base.add_(1)
    assert not _prep._same_source(src, t)  # written to


@pytest.mark.gpu
def test_module_after_its_weights_moved_through_a_freed_block(dev):
    from nunchaku_rocm_amd.linear import SVDQW4A4Linear

    K, N = 512, 256
    one, two = (O.make_svdq_linear(K, N, seed=s, dtype=torch.bfloat16) for s in (1, 2))
    names = ("qweight", "wscales", "smooth_factor", "proj_down", "proj_up", "bias")
    mods = []
    for lin in (one, two):
        mod = SVDQW4A4Linear(K, N, rank=32, torch_dtype=torch.bfloat16, device=dev).requires_grad_(False)
        for name in names:
            getattr(mod, name).data.copy_(lin[name])
        mods.append(mod)
    x = O.make_activations(40, K, seed=3, dtype=torch.bfloat16).to(dev)[None]
    with torch.no_grad():
        want = mods[1](x)
        assert not torch.equal(mods[0](x), want)
        moved = [_replace_at_the_same_address(getattr(mods[0], name), getattr(mods[1], name).data) for name in names]
        if not all(moved):
            pytest.skip("the allocator did not hand the blocks out again")
        assert torch.equal(mods[0](x), want)
