// Host-side geometry of the row-register kernels: elements per lane and row,
// rows per lane, how lanes are laid over a strip and how many channels a wave
// walks.
#include <algorithm>
#include <cmath>

#include "ddf_rows_taprow.h"

namespace ddf {

int tune_int(const char *name, int fallback);

namespace {

constexpr int kRowsStages = 3;   // channels in flight per wave of k_rows (rows::kStages)
constexpr int kMaxRowLanes = 32;  // lanes per image row before the row is cut into segments

unsigned magic_of(int d) { return d == 1 ? 0u : (unsigned)((0x100000000ull + d - 1) / d); }

// Lanes over a strip: lpr = W / vx lanes per image row, rg row groups of R rows
// per wave, strips of even height.  Where it costs no row group, every image
// row is followed by an idle lane (lane pitch lpr + 1): its loads return zero,
// which is exactly what the neighbour shift must bring in at the row ends.
// Rows vx does not divide (the TAIL kernels, which are built padded): ceil(W / vx) lanes,
// always followed by the idle one.
void lay_out_lanes(RowsGeom *t, int H, int W, int vx, int R, bool padded = false) {
    t->segs = t->seg_out = 0;
    t->segs_magic = 0;
    t->tail = W % vx;
    t->shift = 0;
    const int vectors = (W + vx - 1) / vx;
    if (vectors > kMaxRowLanes) {
        // an image row is longer than the lanes of a wave take: even segments of at
        // most 62 vectors, each with a vector of its neighbours on either side
        t->segs = (vectors + kWave - 3) / (kWave - 2);
        t->seg_out = (vectors + t->segs - 1) / t->segs;
        t->segs_magic = magic_of(t->segs);
        t->lpr = t->lp = t->seg_out + 2;
        t->lp_magic = magic_of(t->lp);
        t->rg = 1;
        t->rps = R;
        t->nstrips = ((H + R - 1) / R) * t->segs;
        return;
    }
    t->lpr = vectors;
    const int row_units = (H + R - 1) / R;                  // lane-sized row groups of the plane
    const int fit_plain = std::min(kWave / t->lpr, row_units);
    const int fit_padded = std::min((kWave + 1) / (t->lpr + 1), row_units);
    auto strips_with = [&](int fit) { return fit > 0 ? (row_units + fit - 1) / fit : 1 << 30; };
    const bool pad = padded || t->tail > 0 || (fit_padded > 0 && strips_with(fit_padded) <= strips_with(fit_plain) &&
                                     tune_int("DDF_TUNE_ROWS_PAD", 1) != 0);
    t->lp = t->lpr + (pad ? 1 : 0);
    t->lp_magic = magic_of(t->lp);
    const int rg_max = pad ? fit_padded : fit_plain;
    t->nstrips = (row_units + rg_max - 1) / rg_max;
    t->rg = (row_units + t->nstrips - 1) / t->nstrips;      // even strips
    t->rps = t->rg * R;
    t->run = t->rg * t->lp;
    t->halo = 0;
}

// Channels per wave of k_rows: enough waves to fill the machine (and to even out
// its SIMDs), walks long enough to amortise the spatial-filter registers.  The
// kernels walk whole rounds of `nst` channels, so the count is a multiple of
// that.  `plane`: pixels of a result plane; `min_walk`: shortest walk worth the
// prologue (0: two rounds).
bool cut_channels_forward(RowsGeom &t, int64_t N, int C, int nst, int64_t plane, int min_walk = 0) {
    const int64_t base = N * t.nstrips;
    const int target = tune_int("DDF_TUNE_ROWS_WAVES", 8192);
    const int64_t want_split = std::max<int64_t>(1, (target + base - 1) / base);
    int cpw = (int)(C / want_split);
    // Small planes (up to 32 x 32) walk more rounds where that still leaves a wave per
    // SIMD: the spatial taps a wave loads first are paid for once per walk.  Measured with
    // operands that really come from memory (fp16 and fp32, batches of 8 to 256): planes
    // up to 16 x 16 want walks of 12 channels once those leave a thousand waves (10-15 %
    // over walks of 6) and of 24 once those leave some three thousand (7-9 % more); planes
    // up to 32 x 32 want the longest of 18, 12 and 9 that leaves a thousand (6-11 % over
    // 12 at 28 x 28).  Larger planes and small batches lose by longer walks.
    auto waves_with = [&](int rnds) { return base * ((C + rnds * nst - 1) / (rnds * nst)); };
    int rounds = 2;
    if (plane <= 256) {
        if (waves_with(8) >= 2816) rounds = 8;
        else if (waves_with(4) >= 1024) rounds = 4;
    } else if (plane <= 1024) {
        if (waves_with(6) >= 1024) rounds = 6;
        else if (waves_with(4) >= 1024) rounds = 4;
        else if (waves_with(3) >= 900) rounds = 3;
    }
    const int min_cpw = tune_int("DDF_TUNE_ROWS_MIN_CPW", std::max(rounds * nst, (min_walk + nst - 1) / nst * nst));
    cpw = std::max(cpw / nst * nst, min_cpw);
    const int forced = tune_int("DDF_TUNE_ROWS_CPW", 0);
    if (forced) cpw = forced;
    t.cpw = std::max(1, std::min(cpw, C));
    t.cpb = t.cpw;
    t.csplit = (C + t.cpw - 1) / t.cpw;
    // (single-wave workgroups spread over the machine faster: what counts for the
    // smallest launches)
    t.wpb = std::max(1, std::min(tune_int("DDF_TUNE_ROWS_WPB", plane <= 256 ? 1 : 2), rows::kMaxWpb));
    const int64_t nwork = base * t.csplit;
    if (nwork > (1 << 30)) return false;
    // magic-number division of the work id is exact while id * divisor < 2^32
    if (nwork * std::max(t.csplit, t.nstrips) >= (1ll << 32)) return false;
    t.csplit_magic = magic_of(t.csplit);
    t.nstrips_magic = magic_of(t.nstrips);
    const int64_t ngroups = (nwork + t.wpb - 1) / t.wpb;
    t.xcd_per = (unsigned)((ngroups + rows::kXcd - 1) / rows::kXcd);
    t.nwork = (int)nwork;
    return true;
}

// Channels per wave of k_rows_filters: the four waves of a workgroup cover cpb =
// 4 * cpw channels; enough workgroups to fill the machine, as few channel splits
// (dSF partial sums through the workspace) as that allows.
bool cut_channels_filters(RowsGeom &t, int64_t N, int C) {
    const int64_t base = N * t.nstrips;
    const int target = tune_int("DDF_TUNE_ROWSF_WAVES", 2048);
    const int64_t want_split = std::max<int64_t>(1, (target + base * rows::kFilterWaves - 1) /
                                                        (base * rows::kFilterWaves));
    // Channels per wave for `split` channel ranges: whole rounds of the kernel's channel
    // pipeline and whole dCF flush groups.
    auto cpw_of = [&](int64_t split) {
        const int cpb = (int)((C + split - 1) / split);
        int w = (cpb + rows::kFilterWaves - 1) / rows::kFilterWaves;
        w = (w + rows::kFlushChannels - 1) / rows::kFlushChannels * rows::kFlushChannels;
        return std::max(w, tune_int("DDF_TUNE_ROWSF_MIN_CPW", 2 * rows::kFlushChannels));
    };
    // One split fewer where that turns a ragged second round of waves into a single round
    // of longer walks (rounds of `target` resident waves times channels per wave is what
    // the launch takes): 32 x 128 x 56 x 56 at stride 2 runs 1 792 waves of 16 channels
    // 5 % faster than 2 688 of 12.
    auto cost_of = [&](int w) {
        const int64_t waves = base * rows::kFilterWaves * ((C + (int64_t)w * rows::kFilterWaves - 1) / ((int64_t)w * rows::kFilterWaves));
        return ((waves + target - 1) / target) * w;
    };
    int cpw = cpw_of(want_split);
    if (want_split > 1 && cost_of(cpw_of(want_split - 1)) < cost_of(cpw)) cpw = cpw_of(want_split - 1);
    const int forced = tune_int("DDF_TUNE_ROWSF_CPW", 0);
    if (forced) cpw = std::min(forced, C);
    t.cpw = std::max(1, cpw);
    t.cpb = t.cpw * rows::kFilterWaves;
    t.csplit = (C + t.cpb - 1) / t.cpb;
    t.wpb = 1;
    const int64_t nwork = base * t.csplit;
    if (nwork > (1 << 30)) return false;
    if (nwork * std::max(t.csplit, t.nstrips) >= (1ll << 32)) return false;
    t.csplit_magic = magic_of(t.csplit);
    t.nstrips_magic = magic_of(t.nstrips);
    t.xcd_per = (unsigned)((nwork + rows::kXcd - 1) / rows::kXcd);
    t.nwork = (int)nwork;
    return true;
}

// Stride 2 (3 x 3, fp16 / fp32): lanes over the result plane, one row per lane,
// vx result pixels per lane from feature vectors of 2 * vx elements.  Rows of
// the feature plane must keep those vectors aligned (W a multiple of 2 * vx) and
// a result row must fit the lanes of a wave.  filters: the cut of
// k_rows_filters, else of k_rows.
bool stride2_geometry(const Problem &p, int dtype, bool filters, int max_vx, RowsGeom *g,
                      int *vx_out, int *r_out) {
    if (!(p.s == 2 && p.k == 3 && p.d == 1)) return false;
    if (dtype != DDF_F16 && dtype != DDF_F32) return false;
    if (p.N <= 0 || p.C <= 0 || p.Ho <= 0 || p.Wo <= 0) return false;
    if (p.H > 16384 || p.W > 16384 || p.C > (1 << 24) || p.N > (1 << 24)) return false;
    const int esz = dtype == DDF_F16 ? 2 : 4;
    const int H = (int)p.H, W = (int)p.W, Ho = (int)p.Ho, Wo = (int)p.Wo, C = (int)p.C;
    if ((int64_t)H * W * 8 >= (1ll << 31)) return false;   // byte offsets inside a plane are 32-bit
    // A lane's feature vectors are 2 * vx elements: 16 bytes at most, so that one load
    // or store instruction covers its rows without gaps.  (Vectors of 32 bytes go out as
    // two instructions that each touch every other 16 bytes: measured 7 % slower forward,
    // 9 % backward and 55 % for the feature gradient alone at 32 x 128 x 56 x 56 fp32.)
    int vx = 0;
    for (int cand = 8 / esz; cand >= 1; cand /= 2) {
        if (cand > tune_int("DDF_TUNE_ROWS_VX", 16) || cand > max_vx) continue;
        if (W % (2 * cand) != 0) continue;
        vx = cand;
        break;
    }
    if (vx == 0 || Wo / vx > kMaxRowLanes) return false;
    RowsGeom t{};
    t.C = C; t.H = Ho; t.W = Wo; t.Hi = H; t.Wi = W;
    lay_out_lanes(&t, Ho, Wo, vx, 1);
    if (filters ? !cut_channels_filters(t, p.N, C)
                : !cut_channels_forward(t, p.N, C, kRowsStages, (int64_t)Ho * Wo))
        return false;
    *g = t;
    *vx_out = vx;
    *r_out = 1;
    return true;
}

// Lanes and channel walk of k_rows for vx elements and R rows per lane.
bool rows_cut(const Problem &p, int vx, int R, RowsGeom *g, int *vx_out, int *r_out) {
    const int H = (int)p.H, W = (int)p.W, C = (int)p.C;
    RowsGeom t{};
    t.C = C; t.H = t.Hi = H; t.W = t.Wi = W;
    lay_out_lanes(&t, H, W, vx, R);

    // (25 spatial taps per pixel to load before the walk: 32 pixel-channels per lane at least)
    if (!cut_channels_forward(t, p.N, C, p.k == 5 ? 2 : kRowsStages, (int64_t)H * W, p.k == 5 ? 32 / vx : 0))
        return false;
    *g = t;
    *vx_out = vx;
    *r_out = R;
    return true;
}

// The plane as one run of lanes (RowsGeom::halo) instead of strips of whole rows, in vectors of vx
// and R rows per lane; false where that takes no strip less.  (Whether the forward pass and the
// feature gradient take it: rows_layout_cost.)  A strip of whole rows leaves up to
// half of a wave's lanes idle (38 vectors of a 300-pixel row, 26 of a 101-pixel one); a run
// leaves two, and one per row.  Forward, strips -> run: fp16 8 x 64 x 200 x 300 39.7 -> 34.9 us,
// 5 x 5 at 8 x 64 x 90 x 100 18.8 -> 15.9, 3 x 77 x 140 x 190 12.1 -> 11.0; fp32 8 x 64 x 100 x
// 150 17.0 -> 15.9, 12 x 144 x 80 x 87 27.2 -> 25.5; the feature gradient alone at 8 x 128 x 64 x
// 88 with dilation 2 12.9 -> 11.6.  Launches that are over in a few microseconds keep the strips
// (the run is not laid out for them): they wait for memory, whatever their lanes do.
bool lay_out_run(const Problem &p, int vx, int R, const RowsGeom &rows, RowsGeom *g) {
    if (tune_int("DDF_TUNE_ROWS_RUN", 1) == 0) return false;
    RowsGeom t{};
    t.C = (int)p.C; t.H = t.Hi = (int)p.H; t.W = t.Wi = (int)p.W;
    t.tail = rows.tail;
    t.shift = rows.shift;
    t.lpr = (t.W + vx - 1) / vx;
    t.lp = t.lpr + 1;
    t.lp_magic = magic_of(t.lp);
    t.rg = 1;
    t.rps = R;
    t.run = kWave - 2;
    t.halo = 1;
    const int64_t slots = (int64_t)((t.H + R - 1) / R) * t.lp;
    if (slots * t.lp >= (1ll << 32) || slots >= (1ll << 30)) return false;    // (divisions by multiplication; see magic_div)
    t.nstrips = (int)((slots + t.run - 1) / t.run);
    if (t.nstrips >= rows.nstrips) return false;
    *g = t;
    return true;
}
bool rows_run_geometry(const Problem &p, int vx, int R, const RowsGeom &rows, RowsGeom *g) {
    return lay_out_run(p, vx, R, rows, g) &&
           cut_channels_forward(*g, p.N, g->C, p.k == 5 ? 2 : kRowsStages, p.H * p.W, p.k == 5 ? 32 / vx : 0);
}

// Channels split as for another cut of the same problem; `items`: waves or workgroups per strip
// and channel range.
void cut_channels_like(RowsGeom &t, const RowsGeom &g, int64_t items) {
    t.cpw = g.cpw;
    t.cpb = g.cpb;
    t.csplit = g.csplit;
    t.wpb = g.wpb;
    t.csplit_magic = g.csplit_magic;
    t.nstrips_magic = magic_of(t.nstrips);
    t.nwork = (int)(items * t.nstrips * t.csplit);
    const int64_t ngroups = (t.nwork + t.wpb - 1) / t.wpb;
    t.xcd_per = (unsigned)((ngroups + rows::kXcd - 1) / rows::kXcd);
}

// What the ragged-row variants cover.  (Planes of at most 64 pixels that the exact vectors do
// not cover belong to the kernel that packs several of them into a workgroup.)
bool ragged_shape(const Problem &p, int dtype, int vx) {
    if (dtype != DDF_F16 && dtype != DDF_F32) return false;
    if (p.s != 1 || p.N <= 0 || p.C <= 0 || p.H <= 0 || p.W <= vx || p.W % vx == 0) return false;
    if (p.H > 16384 || p.W > 16384 || p.C > (1 << 24) || p.N > (1 << 24)) return false;
    return p.H * p.W > 64 && (int64_t)p.H * p.W * 8 < (1ll << 31) && tune_int("DDF_TUNE_RAGGED", 1) != 0;
}

constexpr int64_t kCus = 256, kSimds = 4 * kCus;

// Channels per wave of k_rows_taprow_filters (one wave per filter row).
bool cut_channels_taprow(RowsGeom &t, const Problem &p) {
    const int flush = p.k <= 4 ? rows::taprow_flush_channels<3>() : rows::taprow_flush_channels<5>();
    const int C = (int)p.C, target = tune_int("DDF_TUNE_TAPROW_WAVES", 2048);
    const int64_t base = p.N * t.nstrips;
    const int64_t want_split = std::max<int64_t>(1, (target + base * p.k - 1) / (base * p.k));
    int cpw = (int)((C + want_split - 1) / want_split);
    cpw = (cpw + flush - 1) / flush * flush;   // whole flush groups (and pipeline rounds)
    cpw = std::max(cpw, tune_int("DDF_TUNE_TAPROW_MIN_CPW", 2 * flush));
    const int forced = tune_int("DDF_TUNE_TAPROW_CPW", 0);
    if (forced) cpw = forced;
    t.cpw = std::max(1, std::min(cpw, C));
    t.cpb = t.cpw;
    t.csplit = (C + t.cpw - 1) / t.cpw;
    t.wpb = rows::kTaprowWaves;
    const int64_t nwork = base * t.csplit * p.k;   // one wave per filter row
    if (nwork > (1 << 30)) return false;
    if (nwork * std::max(t.csplit, t.nstrips) >= (1ll << 32)) return false;
    t.csplit_magic = magic_of(t.csplit);
    t.nstrips_magic = magic_of(t.nstrips);
    const int64_t ngroups = (nwork + t.wpb - 1) / t.wpb;
    t.xcd_per = (unsigned)((ngroups + rows::kXcd - 1) / rows::kXcd);
    t.nwork = (int)nwork;
    return true;
}

// Stride 2 with any sizes: 16-byte feature vectors, rows cut into segments where they are
// long, the last vector of a row cut short (LaneStride2Ragged).  whole: the lanes cover the
// feature plane (every feature pixel's gradient is written), not only the result plane.
bool stride2_ragged_geometry(const Problem &p, int dtype, bool filters, bool whole, RowsGeom *g, int *vx_out,
                             int *r_out) {
    if (!(p.s == 2 && p.k == 3 && p.d == 1)) return false;
    if (dtype != DDF_F16 && dtype != DDF_F32) return false;
    const int vx = dtype == DDF_F16 ? 4 : 2;
    if (p.N <= 0 || p.C <= 0 || p.Ho <= 0 || p.Wo <= vx) return false;   // (an odd tail loads one pixel to its left)
    if (p.H > 16384 || p.W > 16384 || p.C > (1 << 24) || p.N > (1 << 24)) return false;
    if (p.H * p.W * 8 >= (1ll << 31) || tune_int("DDF_TUNE_RAGGED", 1) == 0) return false;
    RowsGeom t{};
    t.ch = (int)(whole ? (p.H + 1) / 2 : p.Ho);
    t.cw = (int)(whole ? (p.W + 1) / 2 : p.Wo);
    lay_out_lanes(&t, t.ch, t.cw, vx, 1, true);
    t.C = (int)p.C; t.H = (int)p.Ho; t.W = (int)p.Wo; t.Hi = (int)p.H; t.Wi = (int)p.W;
    t.tail = t.W % vx;
    t.shift = dtype == DDF_F16 ? t.tail & 1 : 0;
    if (filters ? !cut_channels_filters(t, p.N, t.C)
                : !cut_channels_forward(t, p.N, t.C, kRowsStages, (int64_t)t.H * t.W))
        return false;
    *g = t;
    *vx_out = vx;
    *r_out = 1;
    return true;
}

// What a launch of k_rows takes, for choosing between two cuts of a problem: the instructions
// of a wave - some 40 per channel and 16 per pixel of a lane (25 taps: 45), the spatial taps
// before the walk as much as three channels - times its waves per SIMD, of which it takes two
// or three to keep one busy.  Ragged vectors cost more than their masks: unaligned accesses
// touch a cache line more.
double rows_cost(const RowsGeom &g, bool ragged, int k, int esz, int vx, int r, double odd_tail = 1.5,
                 double busy = 2.5) {
    const double per_wave = (g.cpw + 3.0) * (40 + (k == 5 ? 45 : 16) * vx * r);
    const double over = !ragged ? 1.0 : g.shift ? odd_tail : esz == 2 ? 1.05 : 1.15;
    return per_wave * over * std::max(busy, (double)g.nwork / kSimds);
}

// For choosing between whole rows and a run of lanes: the same beside the memory the launch moves
// (an instruction of a wave takes 1.1 ns, in which a large copy moves 5.8 kB), as two sides of a
// right angle.  Whole rows end on memory lines, or in one that the next strip shares; a run ends
// anywhere, and lanes of two rows end in two lines per strip, whose parts two compute units read
// and store (32 x 256 x 112 x 112 fp32: 13.5 % more cache accesses, 5 % more requests to L2, 360 000 of
// 6.8 million writes to memory shorter than 64 bytes).  In a launch that waits for memory that costs
// more than idle lanes do: 3 x 3, strips -> run, fp32 32 x 256 x 112 x 112 168.6 -> 194.8 us (28 strips
// -> 27), 32 x 256 x 224 x 224 727 -> 806 (112 -> 103), 32 x 192 x 139 x 145 252 -> 284 (70 -> 43); fp16
// 51 x 170 x 108 x 162 172 -> 191 (27 -> 20).  Lanes of one row: 22 x 456 x 100 x 72 fp32 130.6 -> 138.9, elsewhere within 2 %.  Rows in
// several segments end inside lines as well (fp32 12 x 112 x 238 x 331 252 -> 236, 238 strips -> 162;
// 8 x 64 x 200 x 300 68.8 -> 66.0), and what fits L2 is put together there (3 x 56 x 221 x 133 15.2
// -> 13.1, 111 -> 63).  Vectors of less than 16 bytes ask more often for the same (8 x 64 x 100 x 150
// fp16: 11.7 us in strips of 16-byte vectors, 12.3 in a run of 8-byte ones); those of an odd tail,
// which start at odd elements, are dearer the longer they are.  The shares are fitted over 2738 calls
// between 0.6 and 1600 MB: their choices are 0.6 % over the best one's time on average, counting
// instructions alone 3.5 %, whole rows throughout 4.9 %.  25 taps never wait for memory.
double rows_layout_cost(const Problem &p, const RowsGeom &g, int esz, int vx, int r) {
    const bool wide = vx * esz >= 16;
    const double instructions = rows_cost(g, g.tail > 0, p.k, esz, vx, r, !wide ? 1.2 : p.d == 1 ? 1.8 : 1.5, 2.0);
    if (p.k == 5) return instructions;
    // (64 bytes: what a write to memory holds)
    const bool on_lines = g.segs <= 1 || (g.seg_out * vx * esz % 64 == 0 && p.W * esz % 64 == 0);
    const double parted = g.halo ? (r == 2 ? 0.35 : 0.02) : on_lines ? 0.0 : 0.3;
    const double bytes = 2.0 * p.N * p.C * p.H * p.W * esz, beyond_l2 = std::max(0.0, 1 - 30e6 / bytes);
    const double memory = bytes / 5800 * ((wide ? 1.1 : esz == 2 ? 1.2 : 1.4) + parted * beyond_l2);
    return std::sqrt(instructions * instructions + memory * memory);
}

// The same for k_rows_filters: some 60 instructions per channel and 50 per pixel of a lane;
// two loads per channel leave a single wave per SIMD busy enough.
double rows_filters_cost(const RowsGeom &g, bool ragged, int vx, int r) {
    const double waves = (double)g.nwork * rows::kFilterWaves;
    return (g.cpw + 3.0) * (60 + 50 * vx * r) * (ragged ? 1.1 : 1.0) * std::max(1.0, waves / kSimds);
}

// The same in whole workgroups per CU.
double rows_filters_steps(const RowsGeom &g, bool ragged, int vx, int r) {
    return (g.cpw + 3.0) * (60 + 50 * vx * r) * (ragged ? 1.1 : 1.0) * ((g.nwork + kCus - 1) / kCus);
}

// And of k_rows_taprow_filters (some 40 instructions per channel and 25 per pixel of a lane) in
// whole waves per SIMD.
double taprow_steps(const RowsGeom &g, int vx) {
    return (g.cpw + 3.0) * (40 + 25 * vx) * (g.tail > 0 ? 1.1 : 1.0) * ((g.nwork + kSimds - 1) / kSimds);
}

}  // namespace

// Instantiated (elements per lane and row, rows per lane) per element size.
bool rows_variant_built(int esz, int vx, int r) {
    if (esz == 2) return (r == 1 && (vx == 8 || vx == 4 || vx == 2 || vx == 1)) || (r == 2 && (vx == 8 || vx == 4 || vx == 2));
    if (esz == 4) return (r == 1 && (vx == 4 || vx == 2 || vx == 1)) || (r == 2 && (vx == 2 || vx == 4));
    return false;
}

// (stride 2: the forward pass only)
bool rows_shape_built(int k, int d, int s) {
    return (s == 1 && (k == 3 || k == 5) && (d == 1 || d == 2)) || (s == 2 && k == 3 && d == 1);
}

bool rows_geometry(const Problem &p, int dtype, int max_vx, RowsGeom *g, int *vx_out, int *r_out) {
    if (!rows_shape_built(p.k, p.d, p.s)) return false;
    if (p.s == 2) return max_vx <= 0 && stride2_geometry(p, dtype, false, 16, g, vx_out, r_out);
    if (p.N <= 0 || p.C <= 0 || p.H <= 0 || p.W <= 0) return false;
    if (p.H > 16384 || p.W > 16384 || p.C > (1 << 24) || p.N > (1 << 24)) return false;
    const int esz = dtype == DDF_F16 ? 2 : dtype == DDF_F32 ? 4 : 8;
    const int H = (int)p.H, W = (int)p.W;
    const int hx = p.r * p.d;
    if ((int64_t)H * W * esz >= (1ll << 31)) return false;   // byte offsets inside a plane are 32-bit
    // widest vector the row length allows, at most 32 lanes per image row
    int vx = 0;
    for (int cand = 16 / esz; cand >= 1; cand /= 2) {
        if (max_vx > 0 && cand > max_vx) continue;
        if (cand > tune_int("DDF_TUNE_ROWS_VX", 16)) continue;
        if (W % cand != 0 || cand < hx) continue;
        vx = cand;
        break;
    }
    if (vx == 0) return false;
    // One row per lane keeps the registers low enough for 4-5 waves per SIMD,
    // which is what the larger planes want.  Small planes whose rows are a few
    // two-pixel vectors (14 x 14, 30 x 30) take two rows per lane: fewer strips
    // per plane, and the shorter prologue matters more there.
    // (fp16 rows of a few 4-pixel vectors as well - 28 x 28: 8-byte accesses, and half the
    // loads and neighbour shifts per pixel: 10 % faster)
    int R = ((vx == 2 || (esz == 2 && vx == 4)) && H % 2 == 0 && H * W <= 1024) ? 2 : 1;
    // Large planes stream from HBM and a lane's halo rows come in through the
    // L1 once more per row group: two rows per lane of full 16-byte vectors read
    // four rows for two instead of three for one (built for 3x3 without dilation).
    if (vx * esz == 16 && p.k == 3 && p.d == 1 && H * W >= 112 * 112) R = 2;
    R = tune_int("DDF_TUNE_ROWS_R", R);
    if (p.k == 5) {   // 25 taps: built for one row per lane and vectors of four pixels or more
        R = 1;
        if (vx < 4) return false;
    }
    if (!rows_variant_built(esz, vx, R)) return false;

    return rows_cut(p, vx, R, g, vx_out, r_out);
}

// Vectors of vx elements over rows they do not divide (Ragged in ddf_rows.h).
bool rows_ragged_geometry(const Problem &p, int dtype, int vx, RowsGeom *g, int *r) {
    const int esz = dtype == DDF_F16 ? 2 : 4;
    if (!ragged_shape(p, dtype, vx) || !rows_shape_built(p.k, p.d, p.s)) return false;
    // (two rows per lane: see rows_geometry)
    const int R = vx * esz == 16 && p.k == 3 && p.d == 1 && p.H * p.W >= 112 * 112 ? 2 : 1;
    int tvx;
    if (!rows_cut(p, vx, R, g, &tvx, r)) return false;
    g->shift = esz == 2 ? g->tail & 1 : 0;
    return true;
}

bool rows_plan(const Problem &p, int dtype, RowsGeom *g, int *vx, int *r, bool backward) {
    // (stride 2: the exact cut writes feature rows 2y and 2y + 1 per result row)
    const bool exact = (p.s != 2 || !backward || p.H % 2 == 0) && rows_geometry(p, dtype, 0, g, vx, r);
    if (dtype != DDF_F16 && dtype != DDF_F32) return exact;
    // Which cut: fitted over 80 sizes.  Forward at 12 x 144 x 80 x 87 fp32 28.1 -> 19.9 us, fp16
    // 26.1 -> 22.1 (odd rows: taps combined in fp32 on either); 5 x 5 at 2 x 48 x 135 x 166,
    // which only the LDS-tile kernels covered, 45 -> 11.3.  Small launches keep vectors that
    // divide their rows: 4 x 256 x 25 x 38 fp16 takes 5.2 us in vectors of two and 6.7 in eight.
    const int esz = dtype == DDF_F16 ? 2 : 4;
    double best = exact ? rows_cost(*g, false, p.k, esz, *vx, *r) : 1e30;
    bool found = exact;
    RowsGeom t; int tvx, tr;
    auto consider = [&](bool ragged) {
        const double c = rows_cost(t, ragged, p.k, esz, tvx, tr);
        if (c >= best) return;
        best = c;
        found = true;
        *g = t;
        *vx = tvx;
        *r = tr;
    };
    if (p.s == 2) {
        if (stride2_ragged_geometry(p, dtype, false, backward, &t, &tvx, &tr)) consider(true);
        return found;
    }
    // (what the shortest ragged walk takes: small launches are decided without laying it out)
    if (best <= (std::min<int64_t>(p.C, 2 * kRowsStages) + 3.0) * (40 + (p.k == 5 ? 45 : 16) * 4) * 2.5) return true;
    const RowsGeom whole = *g;
    const int exact_vx = *vx, exact_r = *r;
    for (tvx = 16 / esz; tvx >= 4; tvx /= 2)
        if (rows_ragged_geometry(p, dtype, tvx, &t, &tr)) consider(true);
    if (!found) return false;
    // The plane as one run of lanes; 3 x 3 taps with no less than half the pixels per lane (fp16
    // 12 x 72 x 245 x 369 100 us with sixteen, 118 with four)
    // (ragged rows take operands at any address: such a launch stays one, as a run or not)
    const bool rows_ragged = g->tail > 0;
    const int pixels = *vx * *r;
    best = rows_layout_cost(p, *g, esz, *vx, *r);
    auto consider_run = [&](int rvx, int rr) {
        if (p.k == 3 && rvx * rr * 2 < pixels) return;
        const double c = rows_layout_cost(p, t, esz, rvx, rr);
        if (c >= best) return;
        best = c;
        *g = t;
        *vx = rvx;
        *r = rr;
    };
    if (exact && !rows_ragged && rows_run_geometry(p, exact_vx, exact_r, whole, &t)) consider_run(exact_vx, exact_r);
    for (tvx = 16 / esz; tvx >= 4; tvx /= 2) {
        RowsGeom rows;
        if (rows_ragged_geometry(p, dtype, tvx, &rows, &tr) && rows_run_geometry(p, tvx, tr, rows, &t)) consider_run(tvx, tr);
    }
    return true;
}

// Instantiated (elements per lane and row, rows per lane) of k_rows_filters;
// fused: of the variant that also writes the feature gradient.
bool rows_filters_variant_built(int esz, int vx, int r, bool fused) {
    if (esz != 2 && esz != 4) return false;
    if (vx == 1) return r == 1;   // odd row lengths: one pixel per lane
    if (fused) return (vx == 2 && r == 2) || (vx == 4 && r == 1);
    return r == 1 && (vx == 4 || vx == 2);
}

bool rows_filters_geometry(const Problem &p, int dtype, bool fused, RowsGeom *g, int *vx_out,
                           int *r_out) {
    // (stride 2, one launch for the whole backward pass: every feature row must be some
    // lane's 2y or 2y + 1, so the height is even; the width already is)
    if (p.s == 2)
        return (!fused || (p.H % 2 == 0 && tune_int("DDF_TUNE_ROWSF_FUSED", 1) != 0)) &&
               stride2_geometry(p, dtype, true, 16, g, vx_out, r_out);
    if (!(p.s == 1 && p.k == 3 && (p.d == 1 || p.d == 2))) return false;
    if (p.N <= 0 || p.C <= 0 || p.H <= 0 || p.W <= 0) return false;
    if (p.H > 16384 || p.W > 16384 || p.C > (1 << 24) || p.N > (1 << 24)) return false;
    const int esz = dtype == DDF_F16 ? 2 : dtype == DDF_F32 ? 4 : 8;
    const int H = (int)p.H, W = (int)p.W, C = (int)p.C;
    const int hx = p.r * p.d;
    if ((int64_t)H * W * 8 >= (1ll << 31)) return false;   // byte offsets inside a plane are 32-bit
    // One launch for the whole backward pass: dO, CF and SF are read once.  It is
    // the faster route at every plane size measured (7 x 7 to 200 x 300).
    if (fused && (H * W > tune_int("DDF_TUNE_ROWSF_FUSED_PLANE", 1 << 30) ||
                  tune_int("DDF_TUNE_ROWSF_FUSED", 1) == 0))
        return false;
    int vx = 0, R = 1;
    for (int cand = std::min(16 / esz, 4); cand >= 1; cand /= 2) {
        if (cand > tune_int("DDF_TUNE_ROWSF_VX", 16)) continue;
        if (W % cand != 0 || cand < hx) continue;
        // two rows per lane where a row is a few 2-pixel vectors (14 x 14: one strip per plane)
        const int r = (fused && cand == 2 && H % 2 == 0 && p.d == 1) ? 2 : 1;
        if (!rows_filters_variant_built(esz, cand, r, fused)) continue;
        vx = cand;
        R = r;
        break;
    }
    if (vx == 0) return false;

    RowsGeom t{};
    t.C = C; t.H = t.Hi = H; t.W = t.Wi = W;
    lay_out_lanes(&t, H, W, vx, R);

    if (!cut_channels_filters(t, p.N, C)) return false;
    *g = t;
    *vx_out = vx;
    *r_out = R;
    return true;
}

bool rows_filters_plan(const Problem &p, int dtype, bool fused, RowsGeom *g, int *vx, int *r) {
    const bool exact = rows_filters_geometry(p, dtype, fused, g, vx, r);
    if (fused && tune_int("DDF_TUNE_ROWSF_FUSED", 1) == 0) return exact;
    RowsGeom t{};
    // All gradients at 12 x 144 x 80 x 87 fp32: 63 -> 42 us; 3 x 3 with dilation 2 at 4 x 64 x
    // 60 x 131, which only the LDS-tile kernels covered, 178 -> 18.5; 2 x 256 x 25 x 38 keeps
    // single pixels, 11.3 us against 12.6.
    bool found = exact;
    double best = exact ? rows_filters_cost(*g, false, *vx, *r) : 1e30;
    auto consider = [&](bool ragged, int tvx, int tr) {
        const double c = rows_filters_cost(t, ragged, tvx, tr);
        if (c >= best) return;
        best = c;
        found = true;
        *g = t;
        *vx = tvx;
        *r = tr;
    };
    if (p.s == 2) {
        int tvx, tr;
        if (stride2_ragged_geometry(p, dtype, true, fused, &t, &tvx, &tr)) consider(true, tvx, tr);
        return found;
    }
    const RowsGeom whole = *g;
    const int exact_vx = *vx, exact_r = *r;
    const bool any_tail = p.k == 3 && (p.d == 1 || p.d == 2) && ragged_shape(p, dtype, 4);
    RowsGeom rows{};
    if (any_tail) {
        rows.C = (int)p.C; rows.H = rows.Hi = (int)p.H; rows.W = rows.Wi = (int)p.W;
        lay_out_lanes(&rows, rows.H, rows.W, 4, 1);
        rows.shift = dtype == DDF_F16 ? rows.tail & 1 : 0;
        t = rows;
        if (cut_channels_filters(t, p.N, t.C)) consider(true, 4, 1);
    }
    // The plane as one run of lanes, with the channels split as before if that leaves a workgroup
    // per CU: where it takes three tenths of the strips away, or leaves the fullest CU fewer
    // workgroups to walk.  (A CU holds
    // two: 360 of them at 12 x 144 x 80 x 87 take what 480 do, and 4 % more.)  All gradients,
    // strips -> run: fp16 8 x 64 x 200 x 300 106 -> 75 us, 1 x 128 x 180 x 260 34.0 -> 25.8; fp32
    // 4 x 64 x 200 x 300 71 -> 58, 8 x 64 x 100 x 150 47 -> 39, 2 x 100 x 130 x 140 32.1 -> 22.5.
    // Strips of fp32 vectors that end with a line part none of dX's and the features' lines, which
    // such launches wait for where the features are larger than the L2s: there a run has to take a
    // quarter of the strips away.  (8 x 96 x 72 x 96 fits: 29.8 us as rows, 24.2 as a run.  32 x 256 x
    // 224 x 224, 203 strips for 224: 1161 us as rows, 1206 as a run; 4 x 128 x 445 x 448 323 and
    // 333; 16 x 64 x 88 x 176, 63 for 88: 63.1 and 52.8.  In fp16, at the vector ALU's bound, 16 x
    // 192 x 221 x 224 takes 328 and 319.)  (A ragged cut stays one: see rows_plan.)
    if (!found) return false;
    const RowsGeom strips = *g;
    best = rows_filters_steps(strips, strips.tail > 0, *vx, *r);
    const bool on_lines = dtype == DDF_F32 && strips.tail == 0 && p.W * 4 % 64 == 0 &&
                          p.N * p.C * p.H * p.W * 4 > 32 << 20 &&
                          (strips.segs <= 1 || strips.seg_out * *vx * 4 % 64 == 0);
    auto consider_run = [&](bool ragged, int tvx, int tr) {
        cut_channels_like(t, strips, p.N);
        if (t.nwork < kCus && !cut_channels_filters(t, p.N, t.C)) return;   // (too few workgroups)
        const double c = rows_filters_steps(t, ragged, tvx, tr);
        if (c > best || (c == best && t.nstrips * 10 > strips.nstrips * 7)) return;
        if (on_lines && t.nstrips * 4 > strips.nstrips * 3) return;
        best = c;
        *g = t;
        *vx = tvx;
        *r = tr;
    };
    if (exact && strips.tail == 0 && lay_out_run(p, exact_vx, exact_r, whole, &t)) consider_run(false, exact_vx, exact_r);
    if (any_tail && lay_out_run(p, 4, 1, rows, &t)) consider_run(true, 4, 1);
    return true;
}

// Built: 5 x 5 filters (and, as a tuning alternative, 3 x 3 without dilation).
bool rows_taprow_shape_built(int k, int d, int s) {
    if (s != 1) return false;
    if (k == 5) return d == 1 || d == 2;
    return k == 3 && d == 1 && tune_int("DDF_TUNE_TAPROW_K3", 0) != 0;
}

bool rows_taprow_geometry(const Problem &p, int dtype, RowsGeom *g, int *vx_out, int *r_out) {
    if (!rows_taprow_shape_built(p.k, p.d, p.s)) return false;
    if (p.N <= 0 || p.C <= 0 || p.H <= 0 || p.W <= 0) return false;
    if (p.H > 16384 || p.W > 16384 || p.C > (1 << 24) || p.N > (1 << 24)) return false;
    if (dtype != DDF_F16 && dtype != DDF_F32) return false;
    const int esz = dtype == DDF_F16 ? 2 : 4;
    const int H = (int)p.H, W = (int)p.W, C = (int)p.C;
    const int hx = p.r * p.d;
    if ((int64_t)H * W * 8 >= (1ll << 31)) return false;   // byte offsets inside a plane are 32-bit
    // Widest vector that still leaves enough workgroups; below that, channel
    // splits (dSF partial sums through the workspace) make up the number.
    const int target = tune_int("DDF_TUNE_TAPROW_WAVES", 2048);
    RowsGeom t{};
    int vx = 0;
    for (int cand = 16 / esz; cand * esz >= 4; cand /= 2) {
        if (cand > tune_int("DDF_TUNE_TAPROW_VX", 16)) continue;
        if (W % cand != 0 || cand < hx || cand < 2) continue;
        RowsGeom c{};
        c.C = C; c.H = c.Hi = H; c.W = c.Wi = W;
        lay_out_lanes(&c, H, W, cand, 1);
        t = c;
        vx = cand;
        if (p.N * c.nstrips * p.k >= target) break;
    }
    if (vx == 0) return false;
    if (!cut_channels_taprow(t, p)) return false;
    *g = t;
    *vx_out = vx;
    *r_out = 1;
    return true;
}

bool rows_taprow_plan(const Problem &p, int dtype, RowsGeom *g, int *vx, int *r) {
    const bool exact = rows_taprow_geometry(p, dtype, g, vx, r);
    if (p.k != 5 || (p.d != 1 && p.d != 2)) return exact;
    bool found = exact;
    // 16-byte vectors, or 8-byte ones of fp16 where those of 16 leave too few workgroups
    for (int cand = dtype == DDF_F16 ? 8 : 4; cand >= 4; cand /= 2) {
        if (!ragged_shape(p, dtype, cand)) continue;
        RowsGeom t{};
        t.C = (int)p.C; t.H = t.Hi = (int)p.H; t.W = t.Wi = (int)p.W;
        lay_out_lanes(&t, (int)p.H, (int)p.W, cand, 1);
        if (cand > 4 && p.N * t.nstrips * p.k < 2048) continue;
        // (most lanes idle - rows a little too long for one strip of a small plane: the tile
        // kernel is as fast)
        if (!exact && p.H * p.W * 2 < (int64_t)t.nstrips * kWave * cand) continue;
        t.shift = dtype == DDF_F16 ? t.tail & 1 : 0;
        if (!cut_channels_taprow(t, p)) continue;
        // (as rows_plan; some 40 instructions per channel and 25 per pixel of a lane.  All
        // gradients at 2 x 48 x 135 x 166 fp32, 5 x 5: 1056 -> 36 us.)
        if (exact && (int64_t)t.nstrips * (40 + 25 * cand) * 11 >= (int64_t)g->nstrips * (40 + 25 * *vx) * 10)
            break;
        *g = t;
        *vx = cand;
        *r = 1;
        found = true;
        break;
    }
    if (!found) return false;
    // The plane as one run of lanes (a ragged cut stays one: see rows_plan), the channels split as
    // before or anew.  Ragged rows are not split for it: their partial sums are stored value by
    // value (4 x 64 x 113 x 150 fp32 29 us, in two channel ranges 36).  Filter gradients, strips ->
    // run: fp32 8 x 64 x 90 x 100 40.5 -> 28.6 us, 2 x 96 x 140 x 301 48.7 -> 41.0, 4 x 128 x 60 x
    // 131 37.7 -> 29.9; fp16 8 x 64 x 200 x 304 162 -> 108.
    const RowsGeom strips = *g;
    RowsGeom rows{}, t{};
    rows.C = (int)p.C; rows.H = rows.Hi = (int)p.H; rows.W = rows.Wi = (int)p.W;
    double best = taprow_steps(strips, *vx);
    for (int cand = dtype == DDF_F16 ? 8 : 4; cand >= std::max(2, p.r * p.d); cand /= 2) {
        const bool ragged = p.W % cand != 0;
        if (ragged ? cand < 4 || !ragged_shape(p, dtype, cand) : strips.tail > 0) continue;
        lay_out_lanes(&rows, rows.H, rows.W, cand, 1);
        if (cand > 4 && p.N * rows.nstrips * p.k < 2048) continue;
        rows.shift = dtype == DDF_F16 ? rows.tail & 1 : 0;
        if (!lay_out_run(p, cand, 1, rows, &t)) continue;
        for (int anew = 0; anew < 2; ++anew) {
            if (anew && ragged && strips.csplit == 1 && t.nwork >= kSimds) break;
            if (!anew) cut_channels_like(t, strips, p.N * p.k);
            else if (!cut_channels_taprow(t, p)) break;
            const double c = taprow_steps(t, cand);
            if (c >= best) continue;
            best = c;
            *g = t;
            *vx = cand;
        }
    }
    return true;
}

bool rows_taprow_backward_plan(const Problem &p, int dtype, RowsGeom *g, RowsGeom *gx, int *vxf, int *vx) {
    int r, r_dx;
    if (p.k != 5 || p.s != 1 || (p.d != 1 && p.d != 2) || (dtype != DDF_F16 && dtype != DDF_F32) ||
        tune_int("DDF_TUNE_ROWS", 1) == 0 || !rows_taprow_plan(p, dtype, g, vxf, &r) ||
        !rows_plan(p, dtype, gx, vx, &r_dx, true))
        return false;
    // (the two walks are built with one PAD and one TAIL: a plane that they would lay out differently takes two launches)
    if (r != 1 || r_dx != 1 || gx->tail != g->tail || gx->shift != g->shift || rows_shift_in_as_is(*gx) != rows_shift_in_as_is(*g) ||
        !rows::taprow_backward_built(dtype == DDF_F16 ? 2 : 4, p.d, *vxf, *vx, rows::taprow_backward_pad(*g), rows::taprow_backward_tail(*g)))
        return false;
    gx->wpb = rows::kTaprowWaves;
    gx->xcd_per = (unsigned)cdiv(cdiv(gx->nwork, gx->wpb), rows::kXcd);
    return true;
}

bool rows_cover_backward(const Problem &p, int dtype) {
    RowsGeom g; int vx, r;
    return rows_plan(p, dtype, &g, &vx, &r, true) &&
           (rows_taprow_plan(p, dtype, &g, &vx, &r) ||
            rows_filters_plan(p, dtype, false, &g, &vx, &r));
}

bool rows_cover_stride2_filters(const Problem &p, int dtype) {
    RowsGeom g; int vx, r;
    return p.s == 2 && rows_filters_plan(p, dtype, false, &g, &vx, &r);
}

size_t rows_filters_workspace(const Problem &p, int dtype, unsigned need) {
    if (!(need & (DDF_NEED_DCF | DDF_NEED_DSF))) return 0;
    const size_t asz = dtype == DDF_F64 ? 8 : 4;
    size_t most = 0;
    // (room for either cut of the problem: which one runs also depends on pointer alignment)
    for (int cut = 0; cut < 3; ++cut) {
        RowsGeom g; int vx, r;
        if (cut == 1 && !(need & DDF_NEED_DX)) continue;
        if (cut < 2 ? !rows_filters_plan(p, dtype, cut != 0, &g, &vx, &r)
                    : !rows_taprow_plan(p, dtype, &g, &vx, &r))
            continue;
        size_t bytes = 0;
        if ((need & DDF_NEED_DSF) && g.csplit > 1)
            bytes += ((size_t)p.N * g.csplit * p.kk * p.Ho * p.Wo * asz + 255) / 256 * 256;
        if ((need & DDF_NEED_DCF) && g.nstrips > 1)
            bytes += ((size_t)p.N * p.C * g.nstrips * p.kk * asz + 255) / 256 * 256;
        most = std::max(most, bytes);
    }
    return most;
}

}  // namespace ddf
