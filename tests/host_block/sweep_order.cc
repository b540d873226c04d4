// One force sweep of a disturbed Sedov cube, block by block on the CPU, with
// the threads of a block in several orders (hip/hip_runtime.h here):
//   sweep_order KIND NX TX TY NZ      KIND: sweep or planes
// The nodes it moves have to be the same bits in every order.
// SOURCE: the kernel source; LULESH_FUSED, HOST_BLOCK_MIXED: the form.
#include <hip/hip_runtime.h>

#include SOURCE
#include "lulesh_setup.cpp"

using namespace lulesh;

#ifdef HOST_BLOCK_MIXED
using Fields = DevFieldsMixed;
#else
using Fields = DevFields;
#endif

namespace {

// a value in [0, 1) of each i
double noise(uint64_t i)
{
    i = (i ^ (i >> 30)) * 0xbf58476d1ce4e5b9ull;
    i = (i ^ (i >> 27)) * 0x94d049bb133111ebull;
    return double((i ^ (i >> 31)) >> 11) * 0x1.0p-53;
}

struct Cube {
    HostMesh m;
    std::vector<char> arena;
    Fields f{};
    DevScalars *s = nullptr;

    explicit Cube(int nx)
    {
        MeshConfig cfg;
        cfg.nx = nx;
        m = build_mesh(cfg);
#ifdef HOST_BLOCK_MIXED
        arena.resize(domain_arena_bytes_mixed(m));
        carve_domain_mixed(arena.data(), m, f, &s);
        upload_mesh_mixed(m, f, nullptr);
#else
        arena.resize(domain_arena_bytes(m));
        carve_domain(arena.data(), m, f, &s);
        upload_mesh(m, f, nullptr);
#endif
        s[0] = s[1] = initial_scalars(m, 1.0e-2, 100);
        const double h = 1.125 / nx;
        double *const pos[3] = {f.x[0], f.y[0], f.z[0]};
        double *const vel[3] = {f.xd[0], f.yd[0], f.zd[0]};
        for (int t = 0; t < 3; ++t) {
            for (int64_t n = 0; n < m.num_node; ++n) {
                const uint64_t i = uint64_t(n) * 8 + uint64_t(t);
                pos[t][n] += 0.1 * h * (noise(i) - 0.5);
                vel[t][n] = 100.0 * (noise(i + 4) - 0.5);
            }
        }
        for (int64_t e = 0; e < m.num_elem; ++e) {
            f.p[e] = 1.0e6 * noise(uint64_t(e) + 1);
            f.q[e] = 1.0e5 * noise(uint64_t(e) + 2);
            f.ss[e] = 1.0e3 * noise(uint64_t(e) + 3);
        }
    }
};

}  // namespace

int main(int argc, char **argv)
{
    if (argc != 6) return 2;
    const std::string kind = argv[1];
    const int nx = std::atoi(argv[2]);
    const SweepShape shape = {std::atoi(argv[3]), std::atoi(argv[4]), std::atoi(argv[5]),
                              SWEEP_WAVES};
    std::vector<double> first;
    int differing = 0;
    using host_block::Order;
    for (Order o : {Order::ascending, Order::descending, Order::waves_descending}) {
        host_block::order = o;
        Cube c(nx);
        const PhysParams prm = make_params(2);
        hipError_t rc = hipErrorInvalidValue;
#ifdef HOST_BLOCK_MIXED
        if (kind == "sweep") rc = launch_force_sweep_mixed(shape, c.f, c.s, c.s + 1, prm, nullptr);
#elif defined(LULESH_FUSED)
        if (kind == "sweep") rc = fused::launch_force_sweep(shape, c.f, c.s, c.s + 1, prm, nullptr);
#else
        if (kind == "sweep") rc = launch_force_sweep(shape, c.f, c.s, c.s + 1, prm, nullptr);
        if (kind == "planes") rc = launch_force_planes(c.f, c.s, c.s + 1, prm, nullptr);
#endif
        if (rc != hipSuccess || c.s[1].error != 0 || c.s[1].cycle != 1) {
            std::printf("not run: %d, error %d\n", rc, c.s[1].error);
            return 2;
        }
        std::vector<double> out;
        double moved = 0.0;
        for (const double *a : {c.f.x[1], c.f.y[1], c.f.z[1], c.f.xd[1], c.f.yd[1], c.f.zd[1]}) {
            out.insert(out.end(), a, a + c.m.num_node);
        }
        for (int64_t n = 0; n < c.m.num_node; ++n) {
            moved += std::fabs(c.f.xd[1][n] - c.f.xd[0][n]);
        }
        if (!(moved > 0.0)) {
            std::printf("nothing moved\n");
            return 2;
        }
        if (first.empty()) first = out;
        for (size_t i = 0; i < out.size(); ++i) {
            differing += std::memcmp(&out[i], &first[i], sizeof(double)) != 0 ? 1 : 0;
        }
    }
    std::printf("%d values differ\n", differing);
    return differing == 0 ? 0 : 1;
}
