// The planner's choices that go by the shape of a call and not by a rule: which of several forms of a kernel is
// fastest changes from one l_max to the next (row lengths, channels per wave and workgroups per CU all change
// with it), so the measured winner is written down here, one row per range of l_max, next to the figures of
// the sweep that decided it. Everything else in sphx_plan.cpp follows from LDS sizes and lane counts.
// Plain C++.
#ifndef SPHX_PLAN_SHAPES_HPP
#define SPHX_PLAN_SHAPES_HPP

namespace sphx {

// values_kernel (kind 0) and the lane kernels of the fused product (kind 1) on an MI355X.
//   pack    values: channels a wave evaluates side by side (1, 2, 4, 8); tiles of 64 / pack points
//   alone   one workgroup per CU with all of its LDS instead of two with half each
//   waves   the product, alone on its CU: waves of the workgroup (0: as many as there are channels)
//   floor   the product: tiles shrink in steps of four points down to this size and halve from there
struct ShapeRow {
    int kind, elem, l_from, l_to;
    unsigned pack;
    bool alone;
    int waves;
    unsigned floor;
    const char* measured;
    unsigned long long points_from = 0, points_below = ~0ull; // calls of so many points
};

constexpr ShapeRow kShapeRows[] = {
    // values, float32. 1.2 GB of values, us, with one / two / four / eight channels side by side / pairs_kernel. More
    // workgroups on a CU hide more of one another's loads, tables and flush, fewer points in one make more of its
    // waves wait for a point's tables: four channels are ahead where the rows of 16 points leave room for three
    // workgroups and those of 32 for two at most, eight channels where only two of 16 points fit. (l_max = 16
    // from 1 000 000 points, 28, 32, and float64 22 and 23 below 32 768 points keep the plans that
    // tests/test_library_abi.py states.)
    {0, 4, 12, 15, 2, false, 0, 32, "191 179 187 244 -, 189 181 192 - -, 187 182 188 - -, 206 205 221 - -; 200 000 points 42.0 39.1"},
    {0, 4, 16, 16, 2, false, 0, 32, "199 188 189 - -", 0, 1000000},
    {0, 4, 17, 21, 4, false, 0, 32, "205 196 190 - -, 207 207 192 218 -, 247 237 207 241 -, 242 202 199 - -, 237 209 195 - -"},
    {0, 4, 22, 22, 2, false, 0, 32, "249 198 210 216 -"},
    {0, 4, 23, 25, 4, false, 0, 32, "280 347 227 264 -, 267 287 208 221 266, 286 299 203 226 245"},
    {0, 4, 26, 26, 4, false, 0, 32, "291 277 247 221 239; 20 000 points - 21.6 19.9 18.9"},
    {0, 4, 27, 27, 8, false, 0, 32, "344 313 277 234 255"},
    {0, 4, 29, 31, 4, false, 0, 32, "310 272 227 234 220, 356 251 222 235 225, 357 296 252 252 222"},
    {0, 4, 32, 32, 2, false, 0, 32, "356 239 221 271 229"},
    {0, 4, 33, 33, 4, false, 0, 32, "361 360 343 260 260"},
    // values, float64, the same columns
    {0, 8, 8, 9, 2, false, 0, 32, "214 180 204 - -, 199 201 217 331 -; 200 000 points 30.5 26.5, 37.1 31.7"},
    {0, 8, 14, 15, 2, false, 0, 32, "203 191 194 - -, 219 198 238 250 -"},
    {0, 8, 16, 17, 4, false, 0, 32, "221 274 204 226 -, 230 277 208 258 -"},
    {0, 8, 18, 18, 8, false, 0, 32, "221 239 243 221 -; 100 000 points 65 66 68 61"},
    {0, 8, 19, 21, 4, false, 0, 32, "284 259 240 267 221, 290 232 218 230 217, 308 239 218 241 281"},
    {0, 8, 22, 22, 4, false, 0, 32, "287 220 227 266 279; 100 000 points - 89 89 102 103", 32768},
    {0, 8, 23, 23, 8, false, 0, 32, "299 299 349 274 324", 32768},
    {0, 8, 24, 24, 8, false, 0, 32, "293 293 314 237 244; 20 000 points - 33.8 33.0 31.0"},
    {0, 8, 25, 32, 4, false, 0, 32, "20 000 points, l_max = 26 - - 36 36, recursion kernel 39, 32 - - 46 66, 49"},
    // the product, float64. 200 000 points (400 000 to l_max = 16), us: tiles in half of LDS / one workgroup per
    // CU with 8 / with up to 12 waves; from l_max = 21 with tiles of 28, 24, 20 points before they halve
    {1, 8, 17, 17, 1, true, 12, 32, "289 228 214"},
    {1, 8, 18, 18, 1, true, 12, 32, "299 261 240"},
    {1, 8, 19, 19, 1, true, 12, 32, "315 290 272"},
    {1, 8, 25, 25, 1, true, 8, 16, "660 598 602"},
    {1, 8, 26, 26, 1, true, 12, 16, "675 719 661"},
    // the product, float32, the same columns (l_max = 21, 31: sixteen waves 162, 423)
    {1, 4, 25, 25, 1, true, 12, 32, "335 274 255"},
    {1, 4, 26, 26, 1, true, 12, 32, "340 294 276"},
    {1, 4, 27, 27, 1, true, 8, 32, "348 289 313"},
    {1, 4, 28, 28, 1, true, 8, 32, "356 318 342"},
    {1, 4, 29, 29, 1, true, 12, 32, "385 404 370"},
    {1, 4, 30, 30, 1, true, 8, 32, "397 381 422"},
    {1, 4, 31, 31, 1, true, 16, 32, "477 436 442"},
    {1, 4, 32, 32, 1, true, 8, 32, "500 470 645"},
    {1, 4, 35, 35, 1, true, 12, 16, "789 692 642"},
    {1, 4, 36, 36, 1, true, 12, 16, "807 678 667"},
    {1, 4, 37, 37, 1, true, 8, 16, "820 718 792"},
    {1, 4, 38, 40, 1, true, 8, 32, "874 852 851 (l_max = 40)"},
    {1, 4, 43, 43, 1, true, 8, 16, "909 866 868"},
};

// The row for a shape, or nullptr: then one channel per wave, two workgroups per CU where they fit.
inline const ShapeRow* shape_row(int kind, int elem, int l_max, unsigned long long n_samples) {
    for (const ShapeRow& row : kShapeRows) {
        if (row.kind == kind && row.elem == elem && l_max >= row.l_from && l_max <= row.l_to &&
            n_samples >= row.points_from && n_samples < row.points_below) {
            return &row;
        }
    }
    return nullptr;
}

// recursion_kernel and pairs_kernel: the shapes at which the waves that flush a tile run at raised priority
// (s_setprio) while other waves prepare the next tile. The flush and the preparation end at the same barrier;
// whichever of them a tile waits for gains or loses by it, and which one that is changes from one l_max to the
// next with the tile and the rounds of the sequence lanes. Measured at 1.2 GB of output after 0.3 s of the same
// launches (settled clocks; `python -m sphericart_amd.tune` is the measurement), on two boxes: percent gained on either
// box (the same sign on both at nearly every l_max, and the same in short bursts on two other boxes; the rows are
// the shapes that gained 3 % or more on both, elsewhere the priority costs up to 10 %). The gain holds from
// 50 000 points up in pairs_kernel (2 to 13 % at 50 000, 100 000, 200 000 and 400 000 points) and from 50 000
// down to 20 000 in recursion_kernel (1 to 11 %); the planner asks for 32 and 4 tiles per workgroup. Whether the
// priority is 1, 2 or 3 makes no difference.
struct PriorityRow {
    int mode, elem;
    bool normalized;
    int l_from, l_to;
    unsigned priorities;     // 1: the flushing waves at raised priority
    unsigned sequence_waves; // recursion_kernel: this many instead of the planner's rule (0: the rule)
    const char* measured;
};

constexpr PriorityRow kFlushPriorityRows[] = {
    // gradients, float32
    {1, 4, true, 31, 31, 1, 0, "+4 / +8 (l_max = 32, cfg5: between -3 and +6 from run to run at 50 000 to 800 000 points, left alone)"},
    {1, 4, true, 34, 35, 1, 0, "+8 / +8, +14 / +14"},
    {1, 4, false, 11, 14, 1, 0, "+10 / +8, +7 / +7, +5 / +5, +6 / +5"},
    {1, 4, false, 16, 16, 1, 0, "+5 / +5"},
    {1, 4, false, 23, 23, 1, 0, "+5 / +6"},
    {1, 4, false, 29, 29, 1, 0, "+12 / +10"},
    {1, 4, false, 33, 34, 1, 0, "+14 / +12, +10 / +9"},
    // gradients, float64
    {1, 8, true, 23, 24, 1, 0, "+5 / +7, +8 / +5"},
    {1, 8, true, 31, 32, 1, 0, "+7 / +6, +9 / +10"},
    {1, 8, false, 19, 19, 1, 0, "+11 / +11"},
    {1, 8, false, 21, 21, 1, 0, "+13 / +12"},
    {1, 8, false, 25, 25, 1, 0, "+8 / +8"},
    {1, 8, false, 30, 31, 1, 0, "+12 / +14, +6 / +4"},
    // second derivatives, float32, solid (normalised: 0 to +3 at l_max = 5-28 on both boxes, -1 to -2 on a third)
    {2, 4, false, 5, 6, 1, 0, "+13 / +13, +11 / +12"},
    {2, 4, false, 8, 8, 1, 0, "+11 / +9"},
    {2, 4, false, 10, 14, 1, 0, "+14 / +14, +10 / +12, +10 / +8, +4 / +3, +7 / +6"},
    {2, 4, false, 27, 28, 1, 0, "+6 / +5, +12 / +12"},
    // second derivatives, float64, solid
    {2, 8, false, 19, 19, 1, 0, "+5 / +5"},
    {2, 8, false, 22, 22, 1, 0, "+5 / +5"},
    {2, 8, false, 24, 24, 1, 0, "+6 / +5"},
    // With another number of sequence waves than the rule's (four for gradients in float32, three in float64, three or
    // two for solid second derivatives in float32). Every setting measured after 0.4 s of its own launches, median
    // of three turns, us per 1.2 GB: the rule without priority / this row, on one box, then on another.
    {1, 4, false, 8, 8, 1, 3, "221 / 197, 222 / 195"},
    {1, 4, false, 9, 9, 0, 2, "221 / 205, 222 / 205"},
    {1, 4, false, 10, 10, 1, 3, "230 / 202, 231 / 200"},
    {1, 8, false, 11, 11, 1, 4, "211 / 204, 210 / 203"},
    {1, 8, false, 13, 13, 1, 4, "217 / 209, 216 / 207"},
    {1, 8, false, 15, 16, 1, 4, "218 / 208 and 220 / 212, 216 / 205 and 219 / 213"},
    {2, 4, false, 4, 4, 0, 8, "215 / 199, 217 / 199"},
    {2, 4, false, 18, 19, 1, 4, "214 / 206 and 216 / 207, 211 / 205 and 215 / 206"},
    {2, 4, false, 21, 21, 1, 4, "219 / 207, 218 / 206"},
    {2, 8, false, 23, 23, 1, 2, "240 / 217, 239 / 218 (the rule: three)"},
    // pairs_kernel with gradients, where the planner's estimate gives four sequence waves in float32 and two or three in
    // float64: the rule with the priority where a row above had it / this row; one turn, then the median of three
    {1, 4, false, 30, 30, 0, 3, "223 / 214, 223 / 211"},
    {1, 4, false, 31, 31, 0, 3, "233 / 205, 233 / 204"},
    {1, 4, false, 32, 32, 1, 3, "220 / 204, 217 / 205"},
    {1, 4, false, 35, 35, 0, 3, "240 / 210, 241 / 211"},
    {1, 8, false, 20, 20, 1, 2, "225 / 204, 225 / 204"},
    {1, 8, false, 23, 23, 1, 2, "239 / 221, 237 / 225"},
    {1, 8, false, 26, 27, 1, 4, "228 / 205 and 239 / 230, 229 / 206 and 240 / 231"},
    {1, 8, false, 28, 29, 1, 2, "227 / 208 and 244 / 225, 227 / 208 and 244 / 228"},
};

inline const PriorityRow* priority_row(int mode, int elem, bool normalized, int l_max) {
    for (const PriorityRow& row : kFlushPriorityRows) {
        if (row.mode == mode && row.elem == elem && row.normalized == normalized && l_max >= row.l_from &&
            l_max <= row.l_to) {
            return &row;
        }
    }
    return nullptr;
}

// gradients_fixed_kernel and hessians_fixed_kernel, calls of more points than one round of workgroups takes: points per tile and waves, by the
// first row that matches (tile 0: the kernels that follow in make_plan, whatever the number of rounds). A unit of work costs a wave the same however many
// of its 32 points the tile has, so tiles are as large as leaves LDS for two or three workgroups; which of those, and
// whether one workgroup of sixteen waves with 32 points is ahead, goes by the rounds and by how the runs of the tiles lie in
// HBM. us, what ran before / tile of points x waves, normalised unless it says otherwise.
struct FixedRow {
    int mode; // derivatives: 1, 2
    int elem, l_from, l_to;
    unsigned long long points_from;
    int harmonics; // 0 solid, 1 normalised, -1 both
    unsigned tile, waves;
    const char* measured;
    unsigned long long points_below = ~0ull;
};

constexpr FixedRow kFixedRows[] = {
    {1, 4, 7, 8, 500000, 0, 0, 0, "solid, 1.2 GB, l_max = 7 196 / 24x8 206, 8 201 / 32x16 205 (250 000 points 60.5 57.3)"},
    {1, 4, 9, 9, 400000, 0, 0, 0, "solid, 1.2 GB 202 / 32x16 208 (250 000 76.3 71.1)"},
    {1, 4, 11, 12, 400000, 0, 0, 0, "solid, 1.2 GB, 11 203 / 24x8 205, 12 207 / 16x8 209 (200 000 89 81, 108 97)"},
    {1, 4, 7, 7, 0, -1, 24, 8, "50 000 points 16.3 / 20x8 11.6 24x8 11.7 32x8 11.9, 1.2 GB 209 / 205 186 203"},
    {1, 4, 8, 8, 0, -1, 32, 16, "50 000 20.1 / 20x8 13.6 32x8 13.7 32x16 13.9, 1.2 GB 202 / 196 207 190"},
    {1, 4, 9, 9, 0, -1, 32, 16, "50 000 25.0 / 16x8 17.0 32x8 17.2 32x16 16.2, 1.2 GB 208 / 215 212 188"},
    {1, 4, 10, 10, 400000, 0, 0, 0, "solid, 400 000 133 / 20x8 144 28x16 138 32x16 137"},
    {1, 4, 10, 10, 1000000, 1, 0, 0, "(tests/test_planner_host_only.py states the plan of 1 000 000 points; 1.2 GB 222 / 204)"},
    {1, 4, 10, 10, 0, -1, 32, 16, "50 000 26.8 / 16x8 20.1 32x8 19.2 32x16 19.0, 200 000 80 / 32x16 69, 28x16 71"},
    {1, 4, 11, 11, 0, -1, 24, 8, "100 000 52.2 / 24x8 43.4 28x8 43.3 32x8 44.0, 1.2 GB 214 / 191 204 209"},
    {1, 4, 13, 13, 131072, 0, 0, 0, "solid, 200 000 112 / 16x8 113 20x8 115, 1.2 GB 208 / 212 216"},
    {1, 4, 12, 13, 0, -1, 16, 8, "l_max = 12, 100 000 60.5 / 16x8 49.5 20x8 51.0, 1.2 GB 210 / 188 202; 13, 61.8 / 59.0 58.8, 217 / 193 193"},
    {1, 4, 14, 16, 0, -1, 16, 8, "14, 50 000 45.1 / 16x8 35.4 20x8 37.5 32x16 38.5, 1.2 GB 210 / 32x8 199 16x8 200; 16, 50 000 49.7 / 43.7 - 46.3"},
    {1, 4, 17, 18, 65536, 1, 28, 8, "17, 100 000 98.6 / 12x8 101.7 28x8 97.5, 1.2 GB 223 / 226 207; 18, 111 / 111 104, 218 / 221 208"},
    {1, 4, 17, 18, 0, -1, 12, 8, "17, 25 000 34.7 / 12x8 28.9 28x8 31.6; solid, 1.2 GB 209 / 190 217; 18, 35.1 / 30.7 34.8, 224 / 208 213"},
    {1, 8, 7, 7, 400000, 0, 0, 0, "solid, 1.2 GB 203 / 20x8 206"},
    {1, 8, 7, 7, 131072, -1, 20, 8, "250 000 94.1 / 20x8 79.8 32x8 88.9"},
    {1, 8, 7, 7, 0, -1, 32, 8, "50 000 25.4 / 16x8 21.0 20x8 21.2 32x8 20.3, 100 000 42.1 / - 38.6 37.6"},
    {1, 8, 8, 9, 65536, 0, 32, 16, "solid, 100 000 53.9 / 20x8 49.7 24x8 48.0 32x16 45.6, 1.2 GB 210 / 215 209 191; 9, 65.6 / 59.2 59.4 57.1, 211 / 207 210 202"},
    {1, 8, 8, 9, 0, -1, 20, 8, "8, 100 000 53.9 / 20x8 45.3 24x8 48.1 32x16 49.5, 1.2 GB 207 / 193 203 205; 9, 68.7 / 57.3 58.6 60.9, 221 / 196 207 207"},
    {1, 8, 10, 10, 131072, 0, 24, 8, "solid, 1.2 GB 204 / 20x8 210 24x8 198 32x16 207"},
    {1, 8, 10, 10, 65536, -1, 32, 16, "100 000 78.0 / 20x8 72.2 32x16 69.6, 1.2 GB 224 / 194 195"},
    {1, 8, 10, 10, 0, -1, 20, 8, "50 000 44.4 / 16x8 38.3 20x8 38.1 32x16 39.8"},
    {1, 8, 11, 11, 131072, 0, 0, 0, "solid, 200 000 159 / 16x8 164 32x16 162"},
    {1, 8, 11, 11, 65536, -1, 32, 16, "200 000 179 / 16x8 160 32x16 155"},
    {1, 8, 11, 11, 0, -1, 16, 8, "50 000 57.0 / 16x8 43.6 32x16 46.6"},
    {1, 8, 12, 12, 131072, 0, 12, 8, "solid, 1.2 GB 210 / 12x8 205 28x8 211"},
    {1, 8, 12, 12, 65536, -1, 28, 8, "100 000 108 / 12x8 98.7 28x8 98.9, 1.2 GB 223 / 216 201"},
    {1, 8, 13, 13, 131072, 0, 0, 0, "solid, 1.2 GB 208 / 12x8 210 24x8 212"},
    {1, 8, 13, 13, 65536, -1, 24, 8, "100 000 127 / 12x8 116 24x8 113, 1.2 GB 232 / 220 203"},
    {1, 8, 12, 13, 0, -1, 12, 8, "12, 50 000 62.0 / 12x8 52.2 28x8 54.9; 13, 69.9 / 61.2 24x8 63.9"},
    {1, 8, 14, 14, 0, 1, 8, 8, "6 000 18.4 / 8x8 15.1 16x8 15.8, 12 000 26.6 / 25.2, 15 000 30.7 / 31.3, 50 000 78 / 78", 14000},
    {1, 8, 15, 15, 0, 1, 8, 8, "12 000 32.2 / 27.7, 15 000 38.3 / 34.2, 30 000 59.2 / 59.2", 16384},
    {1, 8, 14, 15, 0, 0, 8, 8, "solid, 14, 12 000 25.6 / 8x8 20.7 20x8 23.5, 30 000 49.6 / 43.4 45.8; 15, 30 000 56.6 / 48.2", 32768},
    {1, 8, 16, 16, 0, 1, 16, 8, "200 28.6 / 8.1, 4 000 16.7 / 16x8 12.1, 12 000 31.5 / 32.4", 4097},
    {1, 8, 16, 16, 0, 0, 16, 8, "solid, 4 000 15.2 / 10.7, 12 000 30.5 / 16x8 28.8, 30 000 61.4 / 60.8", 16384},
    {1, 8, 17, 18, 0, 1, 12, 8, "17, 1 000 16.6 / 9.1, 4 000 22.3 / 12x8 18.1, 12 000 38.0 / 39.2; 18, 25.6 / 19.3", 5000},
    {1, 8, 19, 19, 0, 1, 12, 8, "1 100 19.6 / 10.6, 2 500 19.3 / 12.9, 4 000 25.7 / 22.0, 4 096 21.2 / 22.4", 3073},
    {1, 8, 17, 19, 0, 0, 12, 8, "solid, 17, 4 000 17.9 / 15.3, 7 000 25.2 / 23.6, 12 500 36.7 / 37.9; 18, 7 000 25.9 / 25.4, 12 500 36.9 / 40.3; 19, 31.1 / 27.8, 42.8 / 45.1", 8192},
    {1, 8, 20, 20, 0, 1, 8, 8, "1 100 20.2 / 11.0, 2 500 25.4 / 22.9, 4 000 26.5 / 8x8 23.6, 4 096 21.6 / 23.9, 4 900 26.4 / 31.5", 3073},
    {1, 8, 20, 20, 0, 0, 8, 8, "solid, 2 500 24.6 / 19.7, 4 000 25.9 / 20.0, 4 900 24.6 / 26.1", 4097},
    {1, 4, 19, 19, 0, 1, 12, 8, "4 000 13.3 / 9.0, 12 000 25.0 / 8x8 20.9 12x8 18.5, 30 000 45.3 / 43.6 39.5", 65536},
    {1, 4, 19, 19, 0, 0, 8, 8, "solid, 12 000 24.2 / 8x8 17.9 12x8 19.0, 30 000 43.8 / 37.0 39.8", 65536},
    {1, 4, 20, 24, 0, 1, 8, 8, "20, 4 000 13.6 / 9.5, 12 000 25.5 / 8x8 23.9 16x8 25.2; 22, 31.2 / 27.6 29.4; 24, 33.2 / 31.5 33.9, 30 000 64 / 68", 16384},
    {1, 4, 20, 24, 0, 0, 8, 8, "solid, 20, 12 000 24.7 / 8x8 20.2 16x8 23.2, 30 000 47.1 / 42.1; 24, 31.8 / 26.6 30.8, 61.0 / 55.9", 32768},
    // second derivatives
    {2, 4, 2, 2, 500000, -1, 0, 0, "1.2 GB 217 / 24x8 266 32x8 215-221 32x16 321; solid 200 / 32x8 201-204"},
    {2, 4, 2, 2, 0, -1, 32, 8, "30 000 7.5 / 24x8 6.6 32x8 5.4 32x16 7.2, 300 000 34.4 / 32x8 26.9"},
    {2, 4, 3, 3, 131072, 1, 28, 8, "1.2 GB 291 / 24x8 200 28x8 189 32x8 210"},
    {2, 4, 3, 3, 131072, 0, 24, 16, "solid, 1.2 GB 248 / 12x8 191 24x16 178 28x16 195"},
    {2, 4, 3, 3, 0, -1, 32, 8, "30 000 9.3 / 24x8 6.6 32x8 6.2; solid 8.8 / 5.9 5.9"},
    {2, 4, 4, 4, 400000, -1, 0, 0, "1.2 GB 205 / 32x8 209 32x16 209; solid 203 / 24x16 205 32x16 207"},
    {2, 4, 4, 4, 0, -1, 32, 16, "30 000 12.8 / 24x8 9.3 32x8 9.8 32x16 9.4; solid 13.1 / 9.2 8.5 8.4"},
    {2, 4, 5, 5, 500000, 1, 0, 0, "(tests/test_planner_host_only.py states the plan of 500 000 points; 1.2 GB 212 / 28x16 203)"},
    {2, 4, 5, 5, 400000, 0, 0, 0, "solid, 1.2 GB 206 / 16x16 204-207 32x16 210"},
    {2, 4, 5, 5, 0, -1, 32, 16, "30 000 17.1 / 24x8 12.6 32x8 12.7 32x16 12.5; solid 17.7 / 11.9 11.8 11.6, 1.2 GB 207 / 8x8 196 16x16 204 32x8 209"},
    {2, 4, 6, 6, 0, 1, 24, 8, "30 000 25.5 / 20x8 16.8 24x8 18.9 32x8 16.7, 1.2 GB 223 / 207 200 212"},
    {2, 4, 6, 6, 65536, 0, 16, 16, "solid, 1.2 GB 210 / 16x8 213 16x16 186 28x16 211"},
    {2, 4, 6, 6, 0, 0, 32, 16, "solid, 30 000 24.1 / 16x16 16.0 32x8 15.8 32x16 15.5"},
    {2, 4, 7, 7, 0, 1, 20, 8, "30 000 33.1 / 16x8 21.7 20x8 21.2 24x8 21.4, 1.2 GB 234 / 218 207 213"},
    {2, 4, 7, 7, 0, 0, 12, 16, "solid, 30 000 31.1 / 12x16 19.8 20x16 19.7, 1.2 GB 208 / 191 -"},
    {2, 4, 8, 8, 65536, 1, 32, 8, "1.2 GB 236 / 16x8 228 32x8 217"},
    {2, 4, 8, 8, 65536, 0, 20, 16, "solid, 1.2 GB 207 / 20x8 201 20x16 201 28x16 203"},
    {2, 4, 8, 8, 0, 1, 16, 8, "30 000 35.0 / 12x8 29.7 16x8 27.7 32x8 31.8"},
    {2, 4, 8, 8, 0, 0, 16, 16, "solid, 30 000 31.3 / 16x8 26.1 16x16 24.9 32x16 25.1"},
    {2, 4, 9, 10, 250000, 0, 0, 0, "(tests/test_planner_host_only.py states the plans of 300 000 points)"},
    {2, 4, 9, 9, 65536, 1, 28, 8, "1.2 GB 244 / 24x8 225 28x8 225"},
    {2, 4, 9, 9, 65536, 0, 16, 16, "solid, 1.2 GB 210 / 8x16 204 16x8 196 16x16 197"},
    {2, 4, 9, 9, 0, 0, 8, 16, "solid, 30 000 37.9 / 8x16 30.2 12x16 31.6 24x8 31.3"},
    {2, 4, 9, 10, 0, 1, 12, 8, "9, 30 000 44.5 / 12x8 37.6 24x16 38.7; 10, 51.0 / 43.8 47.3", 65536},
    {2, 4, 10, 10, 65536, 1, 24, 16, "1.2 GB 249 / 24x8 236 24x16 234"},
    {2, 4, 10, 10, 65536, 0, 16, 16, "solid, 1.2 GB 208 / 16x8 202 16x16 196"},
    {2, 4, 10, 10, 0, 0, 24, 16, "solid, 30 000 43.7 / 12x8 39.7 24x8 38.7 24x16 38.2"},
    {2, 4, 11, 11, 131072, 1, 20, 8, "1.2 GB 252 / 16x8 266 20x8 237 24x8 252"},
    {2, 4, 11, 11, 0, 1, 20, 8, "2 500 12.2 / 9.1, 10 000 28.6 / 8x8 25.8 20x8 22.5, 16 000 36.0 / 38.1, 30 000 55.6 / 55.5", 12288},
    {2, 4, 12, 13, 0, 1, 0, 0, "300 points, 12 9.0 / 9.8, 13 9.6 / 11.3; 500 9.3 / 8.8, level", 768},
    {2, 4, 12, 12, 0, 1, 8, 8, "2 500 12.7 / 10.5, 7 000 23.2 / 24.8, 10 000 30.6 / 30.1", 4097},
    {2, 4, 13, 13, 0, 1, 8, 8, "2 500 13.2 / 11.7, 7 000 29.8 / 28.4, 9 000 31.1 / 34.6, 10 000 37.8 / 35.5, 16 000 45.4 / 52.6", 7169},
    {2, 4, 11, 13, 0, 0, 8, 8, "solid, 11, 10 000 24.2 / 17.0, 30 000 47.6 / 8x8 39.9 20x8 44.5, 1.2 GB 210 / 193; 12, 54.2 / 50.4, 210 / 198; 13, 65.5 / 54.7, 215 / 193"},
    {2, 8, 7, 7, 0, 1, 0, 0, "300 points 9.5 / 11.0", 1024},
    {2, 8, 9, 10, 0, 0, 0, 0, "solid, 300 points, 9 7.7 / 7.8, 10 8.5 / 9.5", 1024},
    {2, 8, 2, 2, 0, 1, 32, 8, "30 000 11.8 / 24x8 8.9 32x8 7.7 32x16 10.5, 1.2 GB 255 / 241 208 -"},
    {2, 8, 2, 2, 0, 0, 32, 16, "solid, 30 000 11.6 / 32x8 6.5 32x16 6.6, 1.2 GB 251 / 212 189"},
    {2, 8, 3, 3, 131072, 1, 28, 8, "1.2 GB 266 / 24x8 189 28x8 182 32x8 204"},
    {2, 8, 3, 3, 65536, 0, 16, 16, "solid, 1.2 GB 248 / 16x16 186 28x16 202"},
    {2, 8, 3, 3, 0, 1, 24, 8, "30 000 19.7 / 20x8 11.1 24x8 10.7 32x8 10.7"},
    {2, 8, 3, 3, 0, 0, 32, 16, "solid, 30 000 15.3 / 12x8 10.4 32x8 10.6 32x16 10.4"},
    {2, 8, 4, 5, 0, 1, 20, 8, "4, 30 000 26.7 / 16x8 17.4 20x8 17.2 24x8 17.9, 1.2 GB 236 / 210 199 205; 5, 36.7 / 24.6 23.3 -, 249 / 216 201 -"},
    {2, 8, 4, 4, 65536, 0, 20, 16, "solid, 1.2 GB 209 / 8x8 190 20x16 190 24x16 202"},
    {2, 8, 4, 4, 0, 0, 24, 8, "solid, 30 000 22.6 / 16x8 15.9 24x8 15.8 32x16 16.1"},
    {2, 8, 5, 5, 65536, 0, 16, 16, "solid, 1.2 GB 213 / 8x8 201 16x16 188 20x16 202"},
    {2, 8, 5, 5, 0, 0, 24, 16, "solid, 30 000 30.1 / 12x8 22.7 24x16 22.2 32x8 22.6"},
    {2, 8, 6, 6, 0, 1, 16, 8, "30 000 44.2 / 12x8 33.4 16x8 30.4 32x16 35.2, 1.2 GB 255 / - 205 207"},
    {2, 8, 6, 6, 65536, 0, 16, 16, "solid, 1.2 GB 222 / 8x8 206 16x16 189 28x16 204"},
    {2, 8, 6, 6, 0, 0, 32, 8, "solid, 30 000 36.7 / 16x16 30.4 32x8 29.3 32x16 29.5"},
    {2, 8, 7, 7, 65536, 1, 24, 8, "1.2 GB 264 / 12x8 236 20x8 234 24x8 219"},
    {2, 8, 7, 7, 65536, 0, 16, 8, "solid, 1.2 GB 222 / 8x8 197 16x8 192 16x16 194"},
    {2, 8, 7, 7, 0, 1, 12, 8, "30 000 60.2 / 12x8 42.6 24x8 46.2"},
    {2, 8, 7, 8, 0, 0, 8, 8, "solid, 7, 30 000 49.5 / 8x8 39.0 24x8 39.4; 8, 58.9 / 49.0 16x16 51.0, 1.2 GB 225 / 199 208"},
    {2, 8, 9, 9, 0, 0, 12, 16, "solid, 30 000 69.2 / 12x8 65.6 12x16 63.9, 1.2 GB 230 / 207 200"},
    {2, 8, 10, 10, 65536, 0, 12, 16, "solid, 1.2 GB 223 / 12x8 216 12x16 209"},
    {2, 8, 10, 10, 0, 0, 12, 16, "solid, 5 000 20.7 / 12x8 19.3 12x16 18.8 (30 000 78.0 / 78 and more)", 8192},
};

} // namespace sphx

#endif
