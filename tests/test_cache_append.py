"""The host side of appending a token to the steady zone (CPU): what is refused, and which rows take which way."""
import pytest
import torch

from retrievalattention_amd.cache_hub import retroinfer_cache


def _cache(monkeypatch, rows, filled, **attributes):
    """A cache of one layer, one sequence and two KV heads, with only what the append looks at."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    c = object.__new__(retroinfer_cache)
    zone = lambda: [torch.zeros(1, 2, rows, 128, dtype=torch.bfloat16)]
    c.__dict__.update(dict(
        layer_num=1, context=filled, static_pattern_start=4, static_pattern_end=64, static_pattern_total=filled,
        device_positions=False, steady_zone_keys=zone(), steady_zone_values=zone(), _row_shape=(1, 1, 2, 128)), **attributes)
    return c


@pytest.mark.parametrize("device_positions", [False, True])
def test_full_steady_zone_refuses_a_token(monkeypatch, device_positions):
    c = _cache(monkeypatch, 70, 69, device_positions=device_positions, steady_pos_dev=torch.tensor([69]))
    row = torch.ones(1, 1, 2, 128, dtype=torch.bfloat16)
    c.decode_update_kv_cache(row, row, 0)
    assert c.static_pattern_total == 70 and bool((c.steady_zone_keys[0][:, :, 69] == 1).all())
    c.steady_pos_dev.fill_(3)      # (a position inside the zone: the host counter alone has to refuse)
    with pytest.raises(IndexError):
        c.decode_update_kv_cache(2 * row, row, 0)
    assert c.static_pattern_total == 70 and not c.steady_zone_keys[0][:, :, :69].any()


def test_replayed_token_without_a_row_is_reported(monkeypatch):
    c = _cache(monkeypatch, 70, 69, device_positions=True)
    c.token_replayed()             # the zone's last row
    with pytest.raises(IndexError, match="zone is full"):
        c.token_replayed()
    assert c.context == 70 and c.static_pattern_total == 70
