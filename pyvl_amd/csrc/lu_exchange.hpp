// Which rows a sub-block's interchanges move, and through which words (panel_kernel, lu.hip).
// Plain constexpr functions: the kernel and the CPU model of its exchange use the same ones.
#pragma once

namespace pvl
{
// Pivot row t of a sub-block at positions j0 .. j0 + kb - 1 becomes the row that stood at position
// `from` when the sub-block began.  Wave t & 3 of a group overwrites the positions j0 + t and, below
// the sub-block, `from`, with no barrier since the publishing; so the row at a position is
// published by that wave alone: the row at `from` below the sub-block, or staying in place, in
// row[0][t] (up), the row at j0 + t that leaves its place in row[1][t] (down).  A row that moves inside the
// sub-block is published once, by the wave of the pivot row that it was, and read from there.
struct RowMove
{
    bool up, down;
    int buf, idx; // row[buf][idx] holds the new pivot row
};
constexpr RowMove row_move(int t, int from, int j0, int kb)
{
    const bool stays = from == j0 + t, inside = from < j0 + kb && !stays;
    return inside ? RowMove{false, true, 1, from - j0} : RowMove{true, !stays, 0, t};
}
} // namespace pvl
