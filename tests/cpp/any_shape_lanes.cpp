// any_shape_lanes IN OUT -- one step of the any-shape kernels on the CPU, lane
// by lane (lanes/hip/hip_runtime.h), by the walks and the workgroup sizes that
// the library takes.  Built with the address and undefined-behaviour checks,
// all arrays of their exact size.  Test infrastructure.
//
// IN:  int32 kind (0 advection, 1 adjoint, 2 Euler), rank, extents[3], leaves,
//      direction of the sweep, leaf count the split of a leaf is chosen for;
//      then keys, face records, relations, the kind's constants and fields.
// OUT: the result's fields (and the adjoint's velocity sums, Euler's dt).
#include "kernels_adjoint.hpp"
#include "kernels_euler.hpp"

#include <fstream>
#include <type_traits>

using namespace amrhip;

namespace
{

std::ifstream g_in;
std::ofstream g_out;

template <class T>
std::vector<T> take(size_t count)
{
    std::vector<T> v(count);
    g_in.read(reinterpret_cast<char*>(v.data()), static_cast<std::streamsize>(count * sizeof(T)));
    if (!g_in) std::abort();
    return v;
}

template <class T>
void give(std::vector<T> const& v)
{
    g_out.write(reinterpret_cast<const char*>(v.data()), static_cast<std::streamsize>(v.size() * sizeof(T)));
}

// f with nt as a constant, one of those listed.
template <int... NT, class Fn>
bool with_threads(int nt, Fn&& f)
{
    return ((nt == NT ? (f(std::integral_constant<int, NT>{}), true) : false) || ...);
}

template <int R>
struct job
{
    int32_t                ext[3];
    uint32_t               n, reverse, count;
    launch_box<R>          B;
    launch_box<R, true>    small;
    std::vector<uint64_t>  keys;
    std::vector<face_link> links;
    std::vector<uint32_t>  metas;
    size_t                 cells;

    explicit job(std::vector<int32_t> const& head)
        : ext{ head[2], head[3], head[4] }, n(static_cast<uint32_t>(head[5])), reverse(static_cast<uint32_t>(head[6])),
          count(static_cast<uint32_t>(head[7])), B(launch_box<R>::of(ext)), small(launch_box<R, true>::of(ext)),
          keys(take<uint64_t>(n)), links(take<face_link>(n * 2 * R)), metas(take<uint32_t>(n * 2 * R)),
          cells(static_cast<size_t>(n) * static_cast<size_t>(B.ni()))
    {
    }

    size_t tile_bytes(int fields) const
    {
        return static_cast<size_t>(fields) * static_cast<size_t>(box_tile<R>::cells(B)) * sizeof(double);
    }

    void advection()
    {
        step_params prm{};
        const auto  c = take<double>(6 + kMaxLevels * 3);
        for (int d = 0; d < 3; ++d) prm.vel[d] = c[d], prm.hs[d] = c[3 + d];
        std::memcpy(prm.dtdx, &c[6], sizeof(prm.dtdx));
        const auto          u = take<double>(cells);
        std::vector<double> un(cells);
        box_walk            W{};
        const int           nt = tile_bytes(1) <= kBoxTileBytes ? box_walk_for<R>(B, W) : 0;
        const bool          tile = with_threads<64, 128, 256, 512>(nt, [&](auto threads) {
            constexpr int NT = decltype(threads)::value;
            lanes::launch(k_step_box_tile<R, NT, 4, FROM_LAUNCH>, xcd_grid(n), NT, tile_bytes(1), u.data(), un.data(),
                          keys.data(), links.data(), metas.data(), n, walk_of(n, reverse), small, W, prm,
                          static_cast<const step_params*>(nullptr), static_cast<const uint32_t*>(nullptr));
        });
        if (!tile)
            lanes::launch(k_step_box<R, 256, FROM_LAUNCH>, xcd_grid(n), 256, 0, u.data(), un.data(), keys.data(),
                          links.data(), metas.data(), n, walk_of(n, reverse), B, prm,
                          static_cast<const step_params*>(nullptr), static_cast<const uint32_t*>(nullptr));
        give(un);
    }

    void adjoint()
    {
        adjoint_params prm{};
        const auto     c = take<double>(kMaxLevels * 3 + 9);
        std::memcpy(&prm, c.data(), sizeof(prm));
        const auto          lam = take<double>(cells), u = take<double>(cells);
        std::vector<double> out(cells), sums(static_cast<size_t>(n) * 3);
        if (tile_bytes(2) <= kBoxTileBytes)
            lanes::launch(k_adj_step_box_tile<R, 256>, xcd_grid(n), 256, tile_bytes(2), lam.data(), u.data(),
                          keys.data(), links.data(), metas.data(), &prm, out.data(), n, walk_of(n, reverse), small,
                          sums.data());
        else
            lanes::launch(k_adj_step_box<R, 256>, n, 256, 0, B, lam.data(), u.data(), keys.data(), links.data(),
                          metas.data(), &prm, out.data(), sums.data(), n);
        give(out);
        give(sums);
    }

    void euler()
    {
        euler_params prm{};
        const auto   c = take<double>(2 + kMaxLevels * 3);
        prm.gamma      = c[0];
        prm.cfl        = c[1];
        std::memcpy(prm.cs, &c[2], sizeof(prm.cs));
        prm.remaining = 1.7976931348623157e308;
        const auto              u = take<double>(cells * (R + 2));
        std::vector<double>     un(cells * (R + 2));
        std::vector<euler_slot> ring(kEulerSlots);
        auto                    clear = [&](uint32_t slot) { lanes::launch(k_euler_clear, 1, 64, 0, &ring[slot]); };
        for (uint32_t s = 0; s < kEulerSlots; ++s) clear(s);
        prm.next  = 0;
        prm.clear = 1;
        lanes::launch(k_euler_dt_box<R, 256>, xcd_grid(n), 256, 0, B, u.data(), cells, keys.data(), prm, ring.data(), n);
        // the first of two steps: it folds the second one's minimum
        prm.next_dt = 1;
        prm.first   = 1;
        prm.next    = 1;
        prm.clear   = 2;
        euler_walk W{};
        const int  nt     = euler_walk_for<R>(ext, count, W);
        const bool layers = with_threads<64, 128, 192, 256, 512>(nt, [&](auto threads) {
            constexpr int  NT    = decltype(threads)::value;
            const uint64_t items = static_cast<uint64_t>(n) * W.groups;
            const size_t   lds   = static_cast<size_t>(euler_layer_lds<R>(B, W)) * sizeof(double);
            lanes::launch(k_euler_step_layers<R, NT>, xcd_grid(items), NT, lds, u.data(), un.data(), cells, keys.data(),
                          links.data(), metas.data(), n, walk_of(items, reverse), small, W, prm, ring.data());
        });
        if (!layers)
            lanes::launch(k_euler_step_box<R, 256>, xcd_grid(n), 256, 0, u.data(), un.data(), cells, keys.data(),
                          links.data(), metas.data(), n, walk_of(n, reverse), B, prm, ring.data());
        give(un);
        double next = __longlong_as_double(static_cast<long long>(kEulerNoMinimum));
        for (auto const& p : ring[1].min) next = std::min(next, __longlong_as_double(static_cast<long long>(p.bits)));
        give(std::vector<double>{ ring[1].sums.acc, prm.cfl * next, static_cast<double>(layers ? W.layers : 0),
                                  static_cast<double>(layers ? W.segs : 0) });
    }
};

template <int R>
void run(std::vector<int32_t> const& head)
{
    job<R> j(head);
    switch (head[0])
    {
        case 0: j.advection(); break;
        case 1: j.adjoint(); break;
        default: j.euler();
    }
}

} // namespace

int main(int argc, char** argv)
{
    if (argc != 3) return 2;
    g_in.open(argv[1], std::ios::binary);
    g_out.open(argv[2], std::ios::binary);
    const auto head = take<int32_t>(8);
    if (head[1] == 2)
        run<2>(head);
    else
        run<3>(head);
    return g_out.flush() ? 0 : 1;
}
