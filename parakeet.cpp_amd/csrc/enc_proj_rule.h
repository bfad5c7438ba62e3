// enc_proj_rule.h -- which enc_proj kernel a call takes (host code only; the kernels: pk_device.h).
#pragma once

namespace pkhost {

// At most this many rows: the narrow kernel (one wave per 16x16 block; measured faster up to 256
// rows, slower from 750 on).
constexpr long long kNarrowRows = 256;
// At least this many rows: the wide kernel (128 x 320 tiles) where wide_fills holds, the 64 x 64 tiles
// otherwise.  us, 64 x 64 / wide, D = 1024, J = 640, q8_0, f16 and f32 weights: 8,192 rows 47 / 47,
// 43 / 43, 57 / 58; 16,384 rows 89 / 51, 83 / 48, 106 / 64.
constexpr long long kWideRows = 10240;
constexpr int kTileEdge = 64, kWideTileRows = 128, kWideTileCols = 320;

// A compute unit holds one wide workgroup, so they run in waves of n_cu, and a wave takes the same
// time however much of its tiles lies past the last row or column.  Full, it covers as much as
// 10 n_cu of the 64 x 64 tiles; it takes about as long as 5 n_cu of them.  So: wide where its waves
// are more than half full.  us, 64 x 64 / wide, D = 1024, q8_0: 65,536 rows J = 64 57 / 93, J = 128
// 98 / 94, J = 256 177 / 104, J = 384 273 / 185; 10,240 rows J = 320 40 / 46, J = 640 63 / 47,
// J = 1024 85 / 88; 16,640 rows J = 384 70 / 86, J = 640 102 / 88, J = 1024 159 / 127.
inline bool wide_fills(long long rows, int J, int n_cu) {
    const auto up = [](long long n, long long d) { return (n + d - 1) / d; };
    const long long tiles = up(rows, kTileEdge) * up(J, kTileEdge),
                    waves = up(up(rows, kWideTileRows) * up(J, kWideTileCols), n_cu);
    return tiles > 5 * (long long)n_cu * waves;
}

// 'n' narrow, 't' 64 x 64 tiles, 'w' wide.
inline char enc_proj_kernel_for(long long rows, int J, int n_cu) {
    if (rows <= kNarrowRows) return 'n';
    return rows >= kWideRows && wide_fills(rows, J, n_cu) ? 'w' : 't';
}

}  // namespace pkhost
