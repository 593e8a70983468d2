/*
 * Worlds for the tests that call the engine ABI directly (test_engine_calls.py), made through alis.h:
 * cubes with 8-cell CPML, TF/SF boxes side by side along x or a point dipole, a gold sphere.
 */
#include "alis.h"
#include "../alis_amd/host/internal.h"

/* sphere: its radius in 4 cells, 0 for none; percent: the boxes' edges, of the domain's. */
world ec_boxes(int cells, int boxes, int sphere, int percent)
{
	const float half = 0.01f * percent;
	const float dx = 10, e = dx * (cells - 18) / 2;
	dom D = {{-e, e}, {-e, e}, {-e, e}};
	res R = {5, {dx}, {1240}};
	sur S = {{PML}, {PML}, {PML}, {8}};
	world W = createWorld(D, R, S, "");
	matter Gold = {{1.5}, {{9, 0.07}, {2.6, 0.3, 0.5}, {3.5, 0.6, 0.8}}};
	const float r = 4 * sphere * dx;
	object Sphere = {Ball, {{-r, r}, {-r, r}, {-r, r}}};
	if (sphere) putObjects(W, Gold, Sphere, Air);
	for (int b = 0; b < boxes; b++) {
		const float x = -0.8f * e + 1.6f * e * b / boxes;
		dom T = {{x, x + 2 * half * e / boxes}, {-half * e, half * e}, {-half * e, half * e}};
		planewave(W, T, Ppol, 0, 0, Pulse, 600, 400);
	}
	if (!boxes) pointDipole(W, Ez, 0, 0, 0, Pulse, 600, 240);
	return W;
}

/* A focused beam: a source with a phase per cell, of `steps` steps. */
world ec_beam(int cells, int steps)
{
	world W = ec_boxes(cells, 0, 0, 60);
	removeSources(W);
	focusedBeam(W, W->Dom, Ex, 0, 0, 0, 180, Sine, 600, 3, 1.5);
	for (source S = W->SE; S; S = S->S) S->N = steps;
	return W;
}

world ec_world(int cells, int boxes, int sphere) { return ec_boxes(cells, boxes, sphere, 60); }
void ec_step(world W, int n) { for (int s = 0; s < n; s++) updateE(W), updateH(W); }
void ec_free(world W) { deleteWorld(W); }
alis_dev_world *ec_device(world W) { return W->dev; }
alis_dev_world *ec_aux(world W, int n)
{
	tfsf S = W->S;
	while (n--) S = S->S;
	return S->W->dev;
}

/* W's device worlds belong to the caller from here on. */
void ec_disown(world W)
{
	W->dev = 0;
	for (tfsf S = W->S; S; S = S->S) S->W->dev = 0;
}

/* Commit W with the box of its dispersive object reaching `below` cells under the grid. */
int ec_commit_below(world W, int below)
{
	alis_dev_world_desc d;
	alis_dev_world *D;
	describeWorld(W, &d);
	alis_dev_ade *o = (alis_dev_ade *)d.obj;
	o->k0 = d.kMIN - below;
	for (int c = 0; c < 3; c++) {
		o->fill[c] = makeField(o->i0, o->i1, o->j0, o->j1, o->k0, o->k1);
		for (int p = 0; p < o->nk; p++)
			for (int m = 0; m <= d.complexField; m++) {
				o->J[m][c][p] = makeField(o->i0, o->i1, o->j0, o->j1, o->k0, o->k1);
				o->K[m][c][p] = makeField(o->i0, o->i1, o->j0, o->j1, o->k0, o->k1);
			}
	}
	const int rc = alis_dev_commit(&d, 0, 1, &D);
	freeWorldDesc(&d);
	if (!rc) alis_dev_release(D);
	return rc;
}

/* The real part of one field array of W as alis_dev_read_field gives it: the values, or 0 for too small a
 * buffer. */
long ec_field(world W, int h, int axis, double *out, long room)
{
	const long n = (long)(W->iNUM + 2) * (W->jNUM + 2) * (W->kNUM + 2);
	if (n > room) return 0;
	alisFatal("read", alis_dev_read_field(W->dev, h, 0, axis, out));
	return n;
}

/* W[0..n-1] together. */
void ec_step_many(world *W, int n, int steps) { for (int s = 0; s < steps; s++) updateWorldsE(W, n), updateWorldsH(W, n); }

/* cells x cells x 4 nodes, periodic, with a uniform source over the whole upper plane and a dipole: more
 * cells of strips and sources in one launch than the chip holds wavefronts' lanes, from 725 cells on. */
world ec_plane(int cells)
{
	const float dx = 10, e = dx * cells / 2;
	dom D = {{-e, e}, {-e, e}, {0, 3 * dx}};
	res R = {5, {dx}, {1240}};
	sur S = {{PBC}, {PBC}, {PBC}};
	world W = createWorld(D, R, S, "");
	focusedBeam(W, W->Dom, Ex, 0, 0, 0, 0, Sine, 600, 3);
	pointDipole(W, Ez, 3 * dx, -5 * dx, dx, Pulse, 600, 240);
	return W;
}

/* Overlapping dispersive objects of one, three and two poles around a point dipole, 10 scale cells wide. */
world ec_objects(int cells, int scale)
{
	world W = ec_boxes(cells, 0, 0, 60);
	matter Gold = {{1.5}, {{9, 0.07}, {2.6, 0.3, 0.5}, {3.5, 0.6, 0.8}}}, Metal = {{1}, {{9, 0.07}}}, Glass = {{2}, {{2.6, 0.3, 0.5}, {3.1, 0.2, 0.4}}};
	const float s = scale;
	object A = {Box, {{-83 * s, 21 * s}, {-55 * s, 47 * s}, {-71 * s, 33 * s}}}, B = {Ball, {{-50 * s, 60 * s}, {-50 * s, 60 * s}, {-47 * s, 63 * s}}},
	       C = {Box, {{-15 * s, 75 * s}, {-90 * s, 25 * s}, {-15 * s, 95 * s}}};
	putObjects(W, Metal, A, Gold, B, Glass, C, Air);
	return W;
}

/* n worlds stepped together, or one by one (together 0), their currents read after every third step. */
void ec_step_read(world *W, int n, int steps, int together)
{
	for (int s = 0; s < steps; s++) {
		if (together) updateWorldsE(W, n), updateWorldsH(W, n);
		else for (int a = 0; a < n; a++) updateE(W[a]), updateH(W[a]);
		if (s % 3 == 2) alisFatal("sync", alis_dev_sync(W[s % n]->dev, 0, -1, 0, -1, 0, -1));
	}
}
