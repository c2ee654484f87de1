// Node-wise actions of the UFEM NavierStokes solver (gfx950), SoA fields.
//   LinearizeU    u_adv = 2.1875 u - 2.1875 u1 + 1.3125 u2 - 0.3125 u3   (ns_implementation/NavierStokes.cpp:105)
//   UpdateActions u3 = u2; u2 = u1; u1 = u; u += du; p += dp              (NavierStokes.cpp:172-180)
// Evaluated left to right without contraction into fused multiply-adds, as in the reference expression.
#include "internal.hpp"

namespace cf3hip {

namespace {

#pragma clang fp contract(off)

// the components of a field history, one launch for all of them (blockIdx.y): on small meshes a launch costs
// its latency (linearise + assemble on 32^2 x 2 triangles 28.0 -> 26.5 us, on 23^3 x 6 FP32 tetrahedra
// 36.0 -> 33.4 us)
struct History {
  double *u[3], *u1[3], *u2[3], *u3[3], *ua[3];
};

__global__ void k_linearize(uint32_t n, History h)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const int d = blockIdx.y;
  if(i >= n) return;
  h.ua[d][i] = 2.1875 * h.u[d][i] - 2.1875 * h.u1[d][i] + 1.3125 * h.u2[d][i] - 0.3125 * h.u3[d][i];
}

// blockIdx.y = dim: the pressure.  p2m (null: identity) gives the block row of mesh node i under periodic links
__global__ void k_update(uint32_t n, int dim, History h, double* __restrict__ p, const double* __restrict__ sol,
                         const uint32_t* __restrict__ p2m)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const int d = blockIdx.y;
  if(i >= n) return;
  const uint64_t row = p2m ? p2m[i] : i;
  const double inc = sol[row * (dim + 1) + d];
  if(d == dim) {
    p[i] += inc;
    return;
  }
  h.u3[d][i] = h.u2[d][i];
  h.u2[d][i] = h.u1[d][i];
  h.u1[d][i] = h.u[d][i];
  h.u[d][i] += inc;
}

History history(Fields& F)
{
  History h = {};
  for(int d = 0; d < F.mesh->dim; ++d) {
    h.u[d] = F.u[d].as<double>();
    h.u1[d] = F.u1[d].as<double>();
    h.u2[d] = F.u2[d].as<double>();
    h.u3[d] = F.u3[d].as<double>();
    h.ua[d] = F.uadv[d].as<double>();
  }
  return h;
}

}  // namespace

void ns_linearize(Fields& F)
{
  const Mesh& M = *F.mesh;
  Context& c = *M.ctx;
  hipLaunchKernelGGL(k_linearize, dim3(grid_for(M.n_nodes, 256), M.dim), dim3(256), 0, c.stream, M.n_nodes, history(F));
  HIP_OK(hipGetLastError());
}

void ns_update(Lss& L, Fields& F)
{
  const Mesh& M = *F.mesh;
  Context& c = *M.ctx;
  if(L.neq != M.dim + 1 || (L.periodic ? L.mesh != F.mesh : L.n_nodes != M.n_nodes))
    CF3_THROW(CF3HIP_ERR_INVALID_ARG, "system does not match the fields");
  const uint32_t* p2m = L.periodic ? L.p2m.as<uint32_t>() : nullptr;
  hipLaunchKernelGGL(k_update, dim3(grid_for(M.n_nodes, 256), M.dim + 1), dim3(256), 0, c.stream, M.n_nodes, M.dim,
                     history(F), F.p.as<double>(), L.sol.as<double>(), p2m);
  HIP_OK(hipGetLastError());
}

}  // namespace cf3hip
