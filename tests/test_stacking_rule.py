"""Whether a world's partitions may be stacked goes by what their plans answer now, not by what they answered once."""


def test_a_schedule_that_turns_out_impossible_no_longer_keeps_partitions_apart():
    from super_gnn_amd.aggregator import _Product

    class Plan:
        band, asked = 1, 0

        def schedule(self, F):
            self.asked += 1
            return {"band": self.band}

    plan = Plan()
    product = _Product([plan])
    assert product.takes_bands(64) and product.takes_bands(64)
    plan.band = 0                      # its first product has found the columns out of order
    assert not product.takes_bands(64)
    asked = plan.asked
    assert not product.takes_bands(64) and plan.asked == asked     # a no is kept
    assert not product.takes_bands(128) and plan.asked == asked + 1
