// LDS of a backbone layer launch (bb_chain.hip), in floats from its start: where each stage combines its waves' partial sums.  Plain C++.
//   o_proj | gate_up | down_proj, and the last stage (qkv or head) over the first of them: down_proj's barrier stands behind their readers.
// A workgroup that has gate_up columns and no o_proj / down_proj rows passes no barrier between gate_up's reads and the last stage's writes.  The last
// stage then either stays inside o_proj's area, which such a workgroup does not use, or lies behind all three.
#pragma once

constexpr int BB_WAVES = 8;
constexpr int bb_area(int tiles) { return BB_WAVES * tiles * 256 + BB_WAVES * 64; }      // 16 x 16 sums of every wave and tile + row statistics

struct BbAreas {
    int o, gate_up, down, last, total;
    // tiles of a workgroup in each stage; barrier: whoever runs gate_up runs down_proj
    constexpr BbAreas(int o_tiles, int gu_tiles, int last_tiles, bool barrier)
        : o(0), gate_up(bb_area(o_tiles)), down(gate_up + bb_area(gu_tiles)),
          last(barrier || last_tiles <= o_tiles ? 0 : down + bb_area(o_tiles)),
          total(last == 0 ? down + bb_area(o_tiles) : last + bb_area(last_tiles)) {}
};

// ROWS: the launch's split of its stages (bb_flow_kernel, bb_flow_small_kernel)
constexpr BbAreas bb_areas_wide(int rows) {
    return rows == 64 ? BbAreas(2, 12, 4, true) : rows == 32 ? BbAreas(1, 6, 2, true) : BbAreas(1, 3, 1, false);
}
constexpr BbAreas bb_areas_small(int rows) {
    return rows == 16 ? BbAreas(1, 2, 1, false) : rows == 32 ? BbAreas(1, 6, 2, false) : BbAreas(1, 6, 4, true);
}
