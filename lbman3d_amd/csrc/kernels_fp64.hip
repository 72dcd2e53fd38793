// kernels_fp64.hip — FP64 instantiation of the step kernels. Built with
// -ffp-contract=off so that, with the operand order kept in physics.hpp,
// results reproduce the reference CPU arithmetic bit for bit.
#include "step_kernels.hpp"
#define LBM_FUSED_BODY_ONLY
#include "fused_step.hpp"

namespace lbm {
template void launch_qstep<double>(const Fields<double>&, const BCDesc<double>&, const Phys<double>&, hipStream_t);
template void launch_force_lbm<double, false>(const Fields<double>&, const BCDesc<double>&, const Phys<double>&, int, int, hipStream_t);
template void launch_stream_only<double>(const Fields<double>&, const BCDesc<double>&, int, double*, hipStream_t);
template void launch_diagnostics<double>(const Fields<double>&, const BCDesc<double>&, const Phys<double>&, long,
                                         double*, double*, int, double*, hipStream_t);
template void launch_order_director<double>(const Fields<double>&, long, long, double*, double*, hipStream_t);

// FP64 tile catalogue of the fused step (fused64_kernel): the two column shapes
// with chunk_planes' chunk length, which are what tuning chooses from, then the
// same with a fixed length. Callers that hold a schedule number keep one: the
// catalogue had seven entries before these shapes replaced the first pipeline's.
struct Tile64 {
    bool wide;     // 32x8 columns, else 16x16
    int planes;    // length of the z chunks; 0: by chunk_planes
    const char* name;
};
constexpr Tile64 kTiles64[] = {
    {true, 0, "fp64:32x8"},       {false, 0, "fp64:16x16"},       {false, 64, "fp64:16x16x64"}, {false, 32, "fp64:16x16x32"},
    {true, 64, "fp64:32x8x64"},   {true, 128, "fp64:32x8x128"},   {true, 32, "fp64:32x8x32"},
};
constexpr int kNumTiles64 = sizeof(kTiles64) / sizeof(kTiles64[0]);

int fused64_tile_count() { return kNumTiles64; }
int fused64_tuned_count() { return 2; }
const char* fused64_tile_name(int tile) { return (tile >= 0 && tile < kNumTiles64) ? kTiles64[tile].name : "?"; }

// Length of the z chunks of a grid of `columns` column tiles: a chunk costs its
// planes and two more, and the chunks run in rounds of two blocks per CU, so
// that one block too many costs a whole round (150x130x100 on 32x8 tiles: 595
// chunks of 16 planes in two rounds, 329 us; 510 of 17 in one, 270 us). Of 32,
// 64 and 128 planes for every grid, no one comes within 5 % of this choice
// everywhere (192^3: 664 us here, 741, 708 and 1262; 224x224x200: 942, 1072, 1357
// and 1357). The limit of 64 costs up to 1 % where longer chunks would fill
// their rounds as well (256^3: 1.555 ms with 64 planes, 1.54 with 128).
static int chunk_planes(int columns, int nz) {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    const long slots = 2L * std::max(1, cus);
    long best = 1L << 62;
    int planes = std::min(nz, 64);
    for (int n = (nz + 63) / 64; n <= nz; ++n) {
        const int zc = (nz + n - 1) / n;
        const long chunks = (long)columns * ((nz + zc - 1) / zc);
        const long cost = (chunks + slots - 1) / slots * (zc + 2);
        if (cost < best) {
            best = cost;
            planes = zc;
        }
        if (chunks > 8 * slots) break;
    }
    return planes;
}

template <int TX, int TY>
static void launch_tile64(const Fields<double>& f, const BCDesc<double>& bc, const Phys<double>& k, int planes,
                          int pull, int aux, hipStream_t s) {
    const int ntx = (bc.n[0] + TX - 1) / TX, nty = (bc.n[1] + TY - 1) / TY;
    const int zc = planes ? std::min(planes, bc.n[2]) : chunk_planes(ntx * nty, bc.n[2]), nzc = (bc.n[2] + zc - 1) / zc;
    const int grid = (ntx * nty * nzc + 7) / 8 * 8;
    bool walls = false;
    for (int face = 0; face < 6; ++face)
        walls = walls || bc.qkind[face] != QB_PERIODIC || bc.ukind[face] != UB_PERIODIC;
    auto go = [&](auto masked, auto adv, auto nt) {
        hipLaunchKernelGGL((fused64_kernel<TX, TY, decltype(masked)::value, decltype(adv)::value, decltype(nt)::value>),
                           dim3(grid), dim3(TX * TY), 0, s, f, bc, k, pull, aux, ntx, nty, nzc, zc);
    };
    // Rows of whole 64-byte pieces are stored past the L2 (they leave it before
    // they are read again): 32x8 tiles at 128, 136, 152 and 168 x 128 x 128
    // take 200, 257, 266 and 303 us so and 207, 262, 274 and 312 us with plain
    // stores. In other rows a tile begins inside a piece, which then reaches
    // memory in two parts; plain stores let the L2 put it together: 130, 131,
    // 140 and 150 x 128 x 128 306, 321, 291 and 326 -> 270, 273, 271 and 283 us.
    const bool nt = bc.n[0] % 8 == 0;
    auto with_nt = [&](auto masked, auto adv) {
        if (nt) go(masked, adv, std::true_type{});
        else go(masked, adv, std::false_type{});
    };
    auto with_adv = [&](auto masked) {
        if (k.advection) with_nt(masked, std::integral_constant<int, 1>{});
        else with_nt(masked, std::integral_constant<int, 0>{});
    };
    if (walls) {
        with_adv(std::true_type{});
        launch_shells(f, bc, k, pull, aux, s);
    } else {
        with_adv(std::false_type{});
    }
}

void launch_fused_step_f64(const Fields<double>& f, const BCDesc<double>& bc, const Phys<double>& k, int tile,
                           int pull, int aux, hipStream_t s) {
    const Tile64& t = kTiles64[tile];
    if (t.wide) launch_tile64<32, 8>(f, bc, k, t.planes, pull, aux, s);
    else launch_tile64<16, 16>(f, bc, k, t.planes, pull, aux, s);
}
}  // namespace lbm
