// vgpu_create for the CPU build: with CPU_HIP_SEPARATE=1 the context keeps its
// corrections in launches of their own, as grids do that are too large for the
// in-line form.
#include "vgpu_internal.h"

struct vgpu_ctx : public vgpu::Ctx {};
extern "C" int vgpu_create_library(const vgpu_grid_desc *g, vgpu_prec prec, int device, vgpu_ctx **out);
extern "C" int vgpu_create(const vgpu_grid_desc *g, vgpu_prec prec, int device, vgpu_ctx **out)
{
  const int r = vgpu_create_library(g, prec, device, out);
  const char *s = getenv("CPU_HIP_SEPARATE");
  if (r == 0 && s && s[0] == '1') (*out)->inl = false;
  return r;
}
