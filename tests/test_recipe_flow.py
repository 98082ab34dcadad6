"""build_recipe_flow and validate_flow_order on hand-made input, in a program of
the library's own host sources: recipes with a hazard have no dataflow form,
values that nothing reads before they are overwritten are left out, and the
order check sees the circle around a missing leaf."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "samurai_amd", "csrc", "host")

PROGRAM = r"""
#include "programs.hpp"
#include <cstdio>
using namespace smr;

struct One
{
    int64_t dst;
    int op;
    std::vector<int64_t> src;
};

// the levels finest first, as the update runs them
static RecipeFlow flow(const std::vector<std::vector<One>>& levels, int64_t nref)
{
    std::vector<Recipes> r(MAXL);
    std::vector<const Recipes*> p;
    for (size_t k = 0; k < levels.size(); ++k)
    {
        for (const One& o : levels[k])
        {
            r[size_t(MAXL) - 1 - k].push(o.dst, o.op, o.src.data(), int(o.src.size()));
        }
    }
    for (const Recipes& x : r)
    {
        p.push_back(&x);
    }
    return build_recipe_flow(p, nref);
}

static int bad = 0;
static void expect(bool ok, const char* what)
{
    if (!ok)
    {
        std::printf("FAILED: %s\n", what);
        ++bad;
    }
}

int main()
{
    for (int round = 0; round < 3; ++round) // the scratch is kept between calls
    {
        RecipeFlow f = flow({{{4, RECIPE_COPY, {0}}, {5, RECIPE_COPY, {4}}}, {{6, RECIPE_DIRICHLET, {1}}}}, 8);
        expect(f.ok && f.rec.size() == 12 && f.level[0] == 3 && f.level[MAXL - 1] == 2, "a chain of recipes");
        expect(!flow({{{4, RECIPE_COPY, {5}}, {5, RECIPE_COPY, {0}}}}, 8).ok, "read, then written");
        expect(!flow({{{4, RECIPE_COPY, {5}}}, {{5, RECIPE_COPY, {0}}}}, 8).ok, "read on one level, written on the next");
        expect(!flow({{{4, RECIPE_COPY, {0}}, {5, RECIPE_COPY, {4}}, {4, RECIPE_COPY, {1}}}}, 8).ok, "written, read, written again");
        f = flow({{{4, RECIPE_COPY, {0}}}, {{4, RECIPE_COPY, {1}}, {5, RECIPE_COPY, {4}}}}, 8);
        expect(f.ok && f.rec.size() == 8 && f.level[MAXL] == 0 && f.level[MAXL - 1] == 0 && f.level[0] == 2 && f.rec[2] == 1,
               "overwritten unread: the first one leaves");
        f = flow({{{4, RECIPE_COPY_NO_BC, {5}}, {5, RECIPE_COPY, {0}}}}, 8);
        expect(f.ok && f.rec.size() == 4, "recipes of fields without a B.C. do not count");
        expect(!flow({{{4, RECIPE_COPY, {0}}}}, kFlowSlots + 1).ok, "more slots than the scratch");
    }
    for (int dim = 2; dim <= 3; ++dim)
    {
        for (int s = 0; s <= 1; ++s)
        {
            MeshConfig c;
            c.dim       = dim;
            c.min_level = 1;
            c.max_level = 3;
            c.pred_s    = s;
            // the first cell of level 1 refined twice
            std::vector<std::vector<std::array<int32_t, 4>>> q(MAXL);
            for (int l = 1; l <= 3; ++l)
            {
                for (int k = l < 3 ? 1 : 0; k < 1 << dim; ++k)
                {
                    q[size_t(l)].push_back({(k >> 1) & 1, k >> 2, k & 1, (k & 1) + 1});
                }
            }
            for (int hole = 0; hole <= 1; ++hole)
            {
                if (hole)
                {
                    q[3].pop_back();
                }
                auto copy    = q;
                CellArray ca = empty_cell_array(dim);
                for (int l = 0; l < MAXL; ++l)
                {
                    ca[size_t(l)] = from_runs(dim, l, copy[size_t(l)]);
                }
                MRMeshData m = build_mesh(c, ca);
                m.tiles      = tiles_box(m, false);
                expect(m.tiles == !hole, "tiles_box");
                m.tiles = true; // as if it did
                expect(validate_flow_order(m, build_ghost_program(m)).empty() == !hole, "validate_flow_order");
            }
        }
    }
    return bad;
}
"""


def test_hand_made_recipes_and_meshes(tmp_path):
    src, exe = tmp_path / "recipe_flow.cpp", tmp_path / "recipe_flow"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", f"-I{HOST}", str(src), *(os.path.join(HOST, f) for f in ("interval_set.cpp", "mr_mesh.cpp", "programs.cpp")),
                    "-o", str(exe)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
