// What a workgroup of ir_expand_dw_i8 makes and how its waves walk over their pixels: index arithmetic that the kernel and a check on
// the host share.
#pragma once

#include "thip_kernels.h"

namespace thip {

constexpr int kIrChunk = 32;           // channels of a workgroup
constexpr int kIrPitch = kIrChunk / 2;  // bytes of a cell in LDS, in each of two planes

struct IrStrip {
    int images;               // more than one only where a strip is a whole image
    int oy0, rows;            // its output rows
    int iyFirst, iyLo;        // the first input row under its windows, and the first of them inside the image
    int cellRows, imageRows;  // rows of cells, and rows of pixels, of one image
    int pixels;
};

// Rows of cells of an image whose strip has `rows` output rows.  Images that share a workgroup are one dense matrix of pixels, so all their
// rows are made, also one below the last window (stride 2 over an even height without padding): they all have cells.
__host__ __device__ inline int irCellRows(const IrExpandDwArgs &p, int images, int rows) {
    const int windows = (rows - 1) * p.S + 3, all = p.PT + p.H;
    return images > 1 && windows < all ? all : windows;
}

// Strip `strip` of the images from `n` on.
__host__ __device__ inline IrStrip irStrip(const IrExpandDwArgs &p, int n, int strip) {
    IrStrip s;
    s.images = p.N - n < p.images ? p.N - n : p.images;
    s.oy0 = strip * p.stripRows;
    s.rows = p.OH - s.oy0 < p.stripRows ? p.OH - s.oy0 : p.stripRows;
    s.iyFirst = s.oy0 * p.S - p.PT;
    s.cellRows = irCellRows(p, p.images, s.rows);
    s.iyLo = s.iyFirst < 0 ? 0 : s.iyFirst;
    const int iyHi = s.iyFirst + s.cellRows < p.H ? s.iyFirst + s.cellRows : p.H;
    s.imageRows = iyHi - s.iyLo;
    s.pixels = s.images * s.imageRows * p.W;
    return s;
}

inline size_t irLds(int images, int cellRows, int cellCols) { return (size_t)images * cellRows * cellCols * kIrPitch * 2; }

// The bytes of LDS that a launch asks for: the cells, and the rows below the strip that lanes of the last segment read where the segments
// make more rows than it has.
inline size_t irLaunchLds(const IrExpandDwArgs &a) {
    const int rows = irCellRows(a, a.images, a.stripRows), read = (a.segments * a.segmentRows - 1) * a.S + 3;
    return irLds(a.images, rows, a.cellCols) + (read > rows ? (size_t)(read - rows) * a.cellCols * kIrPitch : 0);
}

// The rows of results that every lane walks down, those of the strip's highest segment.
__host__ __device__ inline int irWalkedRows(const IrExpandDwArgs &p, const IrStrip &s) { return s.rows < p.segmentRows ? s.rows : p.segmentRows; }

// A lane's column of results, of segment `seg` of image `image`.
struct IrColumn {
    int oy, left;  // its first row, and the rows that it stores
    int first;     // where the first cell under its first window starts, bytes from the plane's start
};

// S: p.S, which the kernel knows when it is compiled.  Lanes without rows (an item that the strip does not have, a segment below its last
// row) read those of the first column.
__host__ __device__ inline IrColumn irColumn(const IrExpandDwArgs &p, const IrStrip &s, int S, bool item, int image, int seg, int ox) {
    const int count = irWalkedRows(p, s), rowBytes = p.cellCols * kIrPitch;
    IrColumn c;
    c.oy = seg * p.segmentRows;
    c.left = s.rows - c.oy < count ? s.rows - c.oy : count;
    if (!item || c.left < 0) c.left = 0;
    c.first = c.left > 0 ? image * s.cellRows * rowBytes + c.oy * S * rowBytes + ox * S * kIrPitch : 0;
    return c;
}

// A wave's next tile lies 128 pixels on.  Where its pixels are (the row and column of the cell, the cell, the first run) is
// advanced by a constant and put right where a row or an image ends, without the divisions and products that say it for any pixel:
// vector instructions are most of the launch. With dot products behind it, those of 256 images, millions of waves': the first
// layer 47.4 -> 40.9, 112x112x16 -> 96 52.9 -> 49.5.
struct IrWalk {
    int column, row, at;  // at: bytes, of the cell from `cells` or of the first run from x
};

// Pixel m: row r of the strip's images one below the other, which lies in image `image`.
__host__ __device__ inline IrWalk irWalkFrom(const IrExpandDwArgs &p, int m, int r, int image, int imageStep, int rowStep, int columnStep, int first) {
    IrWalk k;
    k.column = m - r * p.W;
    k.row = r - image * p.H;
    k.at = first + image * imageStep + k.row * rowStep + k.column * columnStep;
    return k;
}

__host__ __device__ inline void irWalkOn(const IrExpandDwArgs &p, IrWalk &k, int imageStep, int rowStep, int columnStep) {
    k.column += p.stepColumns;
    k.row += p.stepRows;
    k.at += p.stepImages * imageStep + p.stepRows * rowStep + p.stepColumns * columnStep;
    const bool wrap = k.column >= p.W;
    k.column -= wrap ? p.W : 0;
    k.row += wrap ? 1 : 0;
    k.at += wrap ? rowStep - p.W * columnStep : 0;
    if (p.images > 1) {
        const bool next = k.row >= p.H;
        k.row -= next ? p.H : 0;
        k.at += next ? imageStep - p.H * rowStep : 0;
    }
}

// Whether pixel m, `cell` on its walk over the cells, has a cell.
__host__ __device__ inline bool irHasCell(const IrExpandDwArgs &p, const IrStrip &s, int m, const IrWalk &cell) {
    return m < s.pixels && cell.column + p.PL < p.cellCols;
}

}  // namespace thip
