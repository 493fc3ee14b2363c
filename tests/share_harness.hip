// Host build of PlaneShare (mist_device.h) beside the reference's computePLIC2VF arithmetic, for
// tests/test_plane_share.py.
#include "../ns_multiphase_amd/csrc/mist_device.h"

using namespace mist;

extern "C" {

double h_deviation(double R, double hmin) { return share_deviation(R, hmin); }

// The share of m = (m1, m2, m3) (any order, sum 1) at offset a.
double h_share(const double* m, double a) { return PlaneShare(m[0], m[1], m[2])(a); }

// For the plane n.x = D in the neighbourhood of cell (i, j, k) of a unit N[0] x N[1] x N[2] mesh:
// out[2 nb] computePLIC2VF of neighbour nb with the reference's sub-tets (fourteen case bodies on
// the snapped distances), out[2 nb + 1] as k_elvira forms it from the plane's offset in the cell.
void h_neighbours(const int* N, const int* c, const double* n, double D, double* out) {
    double x[3][4], xm[3], h[3];
    for (int a = 0; a < 3; ++a) {
        for (int o = 0; o < 4; ++o) x[a][o] = (double)(c[a] - 1 + o) / (double)N[a];
        xm[a] = 0.5 * (x[a][1] + x[a][2]);
        h[a] = 1.0 / (double)N[a];
    }
    const NeighbourShare share(n[0], n[1], n[2], D, h[0], h[1], h[2], xm[0], xm[1], xm[2]);
    const double vol = (h[0] * h[1]) * h[2];
    for (int nb = 0; nb < 27; ++nb) {
        const int o[3] = {nb % 3, (nb / 3) % 3, nb / 9};
        const bool even = ((c[0] + o[0] + c[1] + o[1] + c[2] + o[2] - 3) % 2) == 0;
        const double ts = even ? 1.0 : -1.0;
        double ref = 0.0;
        for (int t = 0; t < 5; ++t) {
            V3 P[4];
            double d[4];
            for (int v = 0; v < 4; ++v) {
                const int q = vert_corner((CutTab::tet5[t] >> (4 * v)) & 15, even);
                P[v] = V3{x[0][o[0] + (q & 1)], x[1][o[1] + ((q >> 1) & 1)], x[2][o[2] + (q >> 2)]};
                d[v] = ((n[0] * P[v].x + n[1] * P[v].y) + n[2] * P[v].z) - D;
            }
            const int cs = d2case_snap(d);
            cut_dispatch<false>(cs, P, d, [&](double v) { ref += (ts * v) / vol; }, [](double) {});
        }
        out[2 * nb] = ref;
        out[2 * nb + 1] = share(share.row(o[1], o[2]), o[0]);
    }
}
}
