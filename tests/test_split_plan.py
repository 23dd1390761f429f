"""What the split-x product runs for a call (eff_split_plan): decided on the host
from the shape, the type and the options alone, so checked without a device."""
import pytest

# what a context holds for the k slices of the LDS-shared tiles: the tiles'
# counters and the sums of 640 workgroups of 64 tokens x 128 rows
SLICE_BUFFER = (1 << 18) + 640 * 64 * 128 * 4

ROWS = [1, 130, 513, 1024, 2048, 4096, 8192, 14336, 32768]
TOKENS = [33, 64, 65, 129, 300, 512, 1000, 2048, 5000]


@pytest.mark.parametrize("tname", ["Q4_K", "Q2_K", "Q6_K", "IQ2_XXS"])
def test_shared_tiles_never_need_more_than_their_buffer(eff, tname):
    """The slices' buffer is made once and never replaced (a recording may read
    it), so no plan of the shared tiles may need more: neither an automatic one
    nor one of a forced slice count, which then runs the other kernel."""
    seen, turned_away = 0, 0
    for rows in ROWS:
        for k in (256, 2048, 4096, 8192, 14336):
            for tokens in TOKENS:
                auto = eff.split_plan(tname, rows, k, tokens)
                for slices in (0, 1, 2, 3, 8, 16, 64):
                    p = eff.split_plan(tname, rows, k, tokens, 0, slices)
                    if p["shared"]:
                        assert p["slice_bytes"] <= SLICE_BUFFER, (rows, k, tokens, slices)
                        seen += p["slices"] > 1
                    elif auto["shared"]:
                        assert p["rows"] in (32, 64)
                        turned_away += 1
                    if slices:
                        assert p["slices"] == min(slices, k // 256)
    assert seen > 100 and turned_away > 50
    # 512 tiles in 8 slices: 134 MB
    if tname == "Q4_K":
        assert not eff.split_plan("Q4_K", 8192, 2048, 512, 0, 8)["shared"]
        assert eff.split_plan("Q4_K", 8192, 2048, 512)["shared"]


def test_split_plan_errors(eff):
    for bad in (("Q4_K", 0, 256, 64), ("Q4_K", 64, 300, 64), ("Q4_K", 64, 256, 64, 4)):
        with pytest.raises(eff.EffError):
            eff.split_plan(*bad)
    for none in (("Q4_K", 64, 256, 1), ("Q8_0", 64, 288, 64)):
        with pytest.raises(eff.NotApplicable):
            eff.split_plan(*none)


def test_preparations_of_x(eff):
    """x is prepared inside the product at up to 8 tokens of an automatic call with
    few workgroups times k, and by a launch of its own everywhere else."""
    for tname, rows, k, tokens, own in [("Q8_0", 2048, 8192, 8, 0), ("Q8_0R", 1024, 8192, 5, 0),
                                        ("Q6_K", 2048, 8192, 8, 0), ("Q6_K", 4096, 14336, 8, 1),
                                        ("Q8_0", 2048, 8192, 9, 1), ("Q2_K", 8192, 2048, 6, 0),
                                        ("IQ2_XXS", 65536, 2048, 5, 1), ("Q4_K", 4096, 4608, 8, 1),
                                        ("Q4_K", 8192, 2048, 512, 1)]:
        assert eff.split_plan(tname, rows, k, tokens)["prepares_x"] == own, (tname, rows, k, tokens)
        assert eff.split_plan(tname, rows, k, tokens, 1)["prepares_x"] == 1
