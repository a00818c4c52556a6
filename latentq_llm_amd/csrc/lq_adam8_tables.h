// Whether an optimizer step on blocks of 2048 looks stored moments up in tables of the block's codes (lq_adam8.hip). Host arithmetic.
#pragma once

// The tables are for busy vector ALUs and take a workgroup of one block, two waves; without them two blocks share a workgroup of
// four. us without / with tables, by blocks to a compute unit:
//                       up to 2      3            5            6            7            9            10           11           14
//   stochastic rounding 5.7 / 6.6    7.0 / 6.4    8.8 / 8.2    9.2 / 9.7    10.7 / 10.0  13.0 / 12.0  13.2 / 13.6  14.8 / 13.9  17.0 / 15.7
//   int4 + residual                  8.9 / 8.7    11.6 / 11.2  11.9 / 13.4  14.6 / 13.7  17.6 / 16.7  17.9 / 18.9  20.4 / 19.0  23.4 / 21.5
// Up to two nothing is bound but the chain that the tables lengthen. A unit's four SIMDs are even with four workgroups of two waves;
// two more of them take as long as four more would (six as long as eight), where three workgroups of four waves are even. From 14 on
// units take blocks as others finish and that no longer shows: tables are 2 to 9 % faster at each number looked at, to 34.
constexpr bool adam8_tables(long long blocks, long long cus) {
    const long long each = (blocks + cus - 1) / cus;
    return each > 2 && each != 6 && each != 10;
}
