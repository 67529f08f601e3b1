// The code of a block's column list (lal_csrmv_info::d_list), in plain C++: the
// analysis writes it, the list kernel reads it, and a host test runs both.
#pragma once

namespace lal
{
    // A list holds its block's distinct columns, ascending, as the low 16 bits of
    // their offsets from the smallest; `near` of its `len` offsets are below 65536.
    // From entry `split` on they are 65536 further than stored.  A list of odd
    // length holds its last column once more, as entry len: without far entries
    // the split lies behind that one too, so that it decodes to a column of the
    // block whatever other blocks of the matrix hold.
    constexpr int list_split(int len, int near)
    {
        return near < len ? near : len + 1;
    }
    constexpr unsigned list_offset(unsigned stored, unsigned entry, unsigned split)
    {
        return stored + (entry >= split ? 65536u : 0u);
    }
}
