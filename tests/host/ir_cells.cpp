// The index arithmetic of ir_expand_dw_i8 on the host: every cell that a window reads is written once, by its own pixel, and nothing
// else is written; the walk over the runs of a first layer names the runs of the same pixel; every result is made once, from its own window,
// and no lane reads LDS that the launch does not ask for.
// Arguments: N H W K C OH OW S PT PL, and for a first layer CKH CS CPT CPL IH IW IC KW behind them.  Prints the images per workgroup.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <vector>

#include "thip_inverted_residual.h"

using namespace thip;

static int fail(const char *what, int a, int b, int c) {
    printf("%s (%d, %d, %d)\n", what, a, b, c);
    return 1;
}

int main(int argc, char **argv) {
    if (argc != 11 && argc != 19) return 2;
    int v[18] = {0};
    for (int i = 1; i < argc; i++) v[i - 1] = atoi(argv[i]);
    IrExpandDwArgs p;
    memset(&p, 0, sizeof(p));
    static int8_t *const somewhere = (int8_t *)0x1000000;
    p.x = p.wexp = p.out = somewhere;
    p.bias1 = p.scale1 = p.wdw = p.bias2 = p.scale2 = (const int32_t *)somewhere;
    p.N = v[0]; p.H = v[1]; p.W = v[2]; p.K = v[3]; p.C = v[4]; p.OH = v[5]; p.OW = v[6]; p.S = v[7]; p.PT = v[8]; p.PL = v[9];
    p.Kp = (p.K + 63) / 64 * 64;
    p.Np = (p.C + 63) / 64 * 64;
    p.CKH = v[10]; p.CS = v[11]; p.CPT = v[12]; p.CPL = v[13]; p.IH = v[14]; p.IW = v[15]; p.IC = v[16];
    p.runBytes = v[17] * p.IC;
    p.xBytes = (int64_t)p.N * p.IH * p.IW * p.IC;
    if (p.CKH) p.Kp = 64;
    const IrExpandDwArgs asked = p;
    if (!planIrExpandDw(&p)) return fail("refused", 0, 0, 0);
    // what a program has chosen before its launches: the same layout, and none that does not fit
    IrExpandDwArgs chosen = asked, again = asked;
    if (!(irExpandDwTime(&chosen) < 1e9)) return fail("no time", 0, 0, 0);
    again.images = chosen.images;
    again.stripRows = chosen.stripRows;
    if (!planIrExpandDw(&again) || memcmp(&again, &p, sizeof(p)) != 0) return fail("another layout", chosen.images, chosen.stripRows, 0);
    const int wrong[][2] = {{13, p.OH}, {p.N + 1, p.OH}, {1, 0}, {0, 1}, {-1, 1}, {1, p.OH + 1}, {2, p.OH - 1}};
    for (auto &w : wrong) {
        again = asked;
        again.images = w[0];
        again.stripRows = w[1];
        if (planIrExpandDw(&again)) return fail("taken", w[0], w[1], 0);
    }
    const bool runs = p.CKH > 0;
    const int rowBytes = p.cellCols * kIrPitch;
    for (int n = 0; n < p.N; n += p.images) {
        for (int strip = 0; strip < p.strips; strip++) {
            const IrStrip s = irStrip(p, n, strip);
            const int imageBytes = s.cellRows * rowBytes;
            std::vector<int> writer((size_t)s.images * s.cellRows * p.cellCols, -1);  // the pixel that wrote a cell
            for (int wave = 0; wave < 4; wave++) {
                for (int fr = 0; fr < 32; fr++) {
                    const int first = wave * 32 + fr, r = first / p.W, image = p.images > 1 ? r / p.H : 0;
                    IrWalk cell = irWalkFrom(p, first, r, image, imageBytes, rowBytes, kIrPitch, (s.iyLo - s.iyFirst) * rowBytes + p.PL * kIrPitch);
                    const int in = p.IH * p.IW * p.IC, inRow = p.CS * p.IW * p.IC, inColumn = p.CS * p.IC;
                    IrWalk run = irWalkFrom(p, first, r, image, in, inRow, inColumn, ((s.iyLo * p.CS - p.CPT) * p.IW - p.CPL) * p.IC);
                    for (int m = first; m < s.pixels; m += 128) {
                        // pixel m of the strip's dense rows, which are consecutive in memory from row iyLo of the first image on
                        const int row = m / p.W + s.iyLo, im = p.images > 1 ? row / p.H : 0, iy = row - im * p.H, ix = m % p.W;
                        if (runs && run.at != im * in + ((iy * p.CS - p.CPT) * p.IW + ix * p.CS - p.CPL) * p.IC) return fail("the run of another pixel", n, strip, m);
                        if (runs && (run.row + s.iyLo != iy || run.column != ix)) return fail("another pixel", n, strip, m);
                        if (irHasCell(p, s, m, cell)) {
                            if (cell.at < 0 || cell.at % kIrPitch != 0 || (size_t)(cell.at / kIrPitch) >= writer.size()) return fail("a write outside the cells", n, strip, m);
                            if (writer[cell.at / kIrPitch] >= 0) return fail("a cell written twice", n, strip, m);
                            writer[cell.at / kIrPitch] = (im * p.H + iy) * p.W + ix;
                        }
                        irWalkOn(p, cell, imageBytes, rowBytes, kIrPitch);
                        irWalkOn(p, run, in, inRow, inColumn);
                    }
                }
            }
            for (int im = 0; im < s.images; im++) {
                for (int y = 0; y < s.cellRows; y++) {
                    for (int x = 0; x < p.cellCols; x++) {
                        const int iy = s.iyFirst + y, ix = x - p.PL, inside = iy >= 0 && iy < p.H && ix >= 0 && ix < p.W;
                        if (writer[((size_t)im * s.cellRows + y) * p.cellCols + x] != (inside ? (im * p.H + iy) * p.W + ix : -1)) return fail("a cell of another pixel, or of none", n + im, iy, ix);
                    }
                }
            }
        }
    }
    // the depthwise half: the loop of a wave over items of 16 columns
    const size_t lds = irLaunchLds(p);
    for (int n = 0; n < p.N; n += p.images) {
        for (int strip = 0; strip < p.strips; strip++) {
            const IrStrip s = irStrip(p, n, strip);
            const int imageBytes = s.cellRows * rowBytes, items = p.OW * p.segments * s.images, walked = irWalkedRows(p, s);
            const size_t planeBytes = (size_t)s.images * imageBytes;
            std::vector<char> made((size_t)s.images * s.rows * p.OW, 0);
            for (int first = 0; first < items; first += 16) {
                for (int item = first; item < first + 16; item++) {
                    const int ox = p.segments * p.images > 1 ? item % p.OW : item, seg = p.segments * p.images > 1 ? item / p.OW % p.segments : 0;
                    const int image = p.images > 1 ? item / p.OW / p.segments : 0;
                    const IrColumn c = irColumn(p, s, p.S, item < items, image, seg, ox);
                    // rows (walked - 1) * S + 3 deep, three cells wide, in both planes
                    const size_t end = (size_t)c.first + (size_t)((walked - 1) * p.S + 2) * rowBytes + 3 * kIrPitch + planeBytes;
                    if (c.first < 0 || end > lds) return fail("a read behind the launch's LDS", n, strip, item);
                    if (c.left < 0 || c.left > walked || (c.left > 0 && (image >= s.images || ox >= p.OW || c.oy + c.left > s.rows))) return fail("a result outside the strip", n, strip, item);
                    for (int r = 0; r < c.left; r++) {
                        if (c.first + r * p.S * rowBytes != image * imageBytes + (c.oy + r) * p.S * rowBytes + ox * p.S * kIrPitch) return fail("another window", n, strip, item);
                        if ((c.oy + r) * p.S + 2 >= s.cellRows || ox * p.S + 2 >= p.cellCols) return fail("a window behind the cells", n, strip, item);
                        char &m = made[((size_t)image * s.rows + c.oy + r) * p.OW + ox];
                        if (m++) return fail("a result made twice", n, strip, item);
                    }
                }
            }
            for (size_t i = 0; i < made.size(); i++) {
                if (!made[i]) return fail("a result that nobody makes", n, strip, (int)i);
            }
        }
    }
    printf("%d\n", p.images);
    return 0;
}
