// The Hilbert curve by which points are put in an order that keeps neighbours together.
#pragma once

// Place of the cell (x, y, z) of a 16^3 grid along a Hilbert curve (J. Skilling, "Programming the
// Hilbert curve", AIP Conference Proceedings 707, 2004).
constexpr unsigned tk_hilbert(unsigned x, unsigned y, unsigned z)
{
    unsigned c[3] = {x, y, z};
    for (unsigned q = 8u; q > 1u; q >>= 1) {
        for (int a = 0; a < 3; ++a) {
            const bool flip = (c[a] & q) != 0u;
            const unsigned swap = flip ? 0u : (c[0] ^ c[a]) & (q - 1u);
            c[0] ^= flip ? q - 1u : swap;
            c[a] ^= swap;
        }
    }
    c[1] ^= c[0];
    c[2] ^= c[1];
    unsigned gray = 0u;
    for (unsigned q = 8u; q > 1u; q >>= 1)
        gray ^= (c[2] & q) != 0u ? q - 1u : 0u;
    unsigned place = 0u;
    for (int b = 3; b >= 0; --b)
        for (int a = 0; a < 3; ++a)
            place = 2u * place + (((c[a] ^ gray) >> b) & 1u);
    return place;
}
