"""The launch rule of the sequential-sum linears (fh_seq.hpp, rows_per_lane), restated
for the tests that must reach each of its instances."""


def rows_per_lane(cols, tiles, m, cus=256):
    """Rows of x per lane for `tiles` tiles of `cols` columns and m rows."""
    def blocks(tm):
        return tiles * -(-m // (256 // cols * tm))

    def cost(tm):
        return -(-blocks(tm) // cus) * (20 * tm + 3)

    tm = 1
    for t in (2, 4):
        if blocks(t) >= 2 * cus and cost(t) < cost(tm):
            tm = t
    return tm
