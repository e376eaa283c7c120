// Chip-resident time loop, FDORDER 8, viscoelastic P/SV.
#define DN_F 4
#define DN_GROUP 2
#include "dn_resident_inst.inc"
